/*
 * vt_gemm_rows.hip - the backbone's prefill products of up to 64 rows, and the K cuts of the codec's (vt_gemm_rows_kernel).
 */
#include "vt_gemm_tiles.h"

/* ---- the backbone: column strips of 288 or 96, the rows of a K cut shared by a workgroup -----------------------
 * With so few rows the product is a weight stream: what counts is that every CU has an equal share of the weights, and
 * moves little else.  A workgroup owns a strip of columns over a K cut, so that strips times cuts make one item per CU:
 * gate|up 64 strips of 288 in 4 cuts, q|k|v 64 of 96 in 4, output and down 32 of 96 in 8, and its rows are those of a quarter
 * or an eighth of K.  At 37 rows a CU moves 565 / 270 / 180 / 405 KB (gate|up, q|k|v, output, down; weights and rows); with
 * 64 columns over half or all of K, where every wave fetches rows of its own (vt_gemm_rows_kernel), 983 / 442 / 295 / 531.
 * Nine waves: KW = 1, a block of 32 columns each; KW = 3, three blocks with a third of the K steps each, whose sums are added
 * through LDS.  The hi and the lo plane of 16 rows are the 32 rows of one matrix instruction, and their sums are added at the
 * end: ceil(rows / 16) instructions per 32 columns and 16 k.  The weights go from memory into the B operand registers, D steps
 * ahead (with twice as many the registers spill, and at 6 rows, where they do not, it gains nothing).  The rows pass through three
 * LDS buffers of three K steps, written by buffer loads (lane i of a request brings 16 bytes of row i/8 to place i, the piece
 * i%8 ^ row%8 of its 128-byte line, so that eight lanes reading one piece of eight rows meet all banks).  Three arrays, so that
 * the compiler knows that reading one need not wait for the others; the number of requests per wave is fixed (what is
 * past the end brings zeros, what a wave has no part in goes to a spare kilobyte), so the waits count exactly.
 * Row-major weights (a caller's own, FRAG false): the same, a lane's 16 bytes from its own row, a line's four requests behind one
 * another; their last strip may have one or two blocks of columns.
 * us per launch inside a prefill of 37 rows, q|k|v / output / gate|up / down: 13.0 / 11.6 / 23.5 / 15.8, on the 64-column tiles
 * 15.2 / 11.1 / 29.9 / 17.4; whole prefills of 6 / 24 / 37 / 64 rows 1829 / 2199 / 2473 / 2763 -> 1785 / 1994 / 2340 / 2737. */
#define GS_WAVES 9
#define GS_CHUNK 3                        /* K steps per buffer */

template <int N> struct gs_int { static constexpr int v = N; };

template <int NP, int KW, bool FRAG>
__global__ void __launch_bounds__(64 * GS_WAVES)
vt_gemm_strip_kernel(float *C, int ldc, size_t plane_stride, const uint16_t *Ahi, const uint16_t *Alo, const uint16_t *Wf, int M, int N, int K,
                     vt_divisor strips, gm_cuts cuts) {
    constexpr int MG = (NP + 1) / 2, CB = GS_WAVES / KW, STEP = MG * 4096, BUF = GS_CHUNK * STEP;
    constexpr int SPW = GS_CHUNK / KW, D = 3;                                /* a wave's steps per chunk; steps ahead */
    constexpr int ND = (2 * GS_CHUNK * NP + GS_WAVES - 1) / GS_WAVES;        /* requests of rows per wave and chunk */
    __shared__ __attribute__((aligned(16))) unsigned char buf0[BUF + 1024], buf1[BUF + 1024], buf2[BUF + 1024];
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int cb = wave / KW, kw = wave % KW;
    /* slot id lands on XCD id % 8: an XCD takes a run of items, strip fastest, i.e. few cuts, whose rows its L2 then holds */
    const int id = (int)blockIdx.x, items = strips.d * cuts.n, li = (items & 7) == 0 ? (id & 7) * (items >> 3) + (id >> 3) : id;
    const int cut = vt_div(li, strips), strip = li - cut * strips.d;
    const int ns = cuts.steps + (cut < cuts.longer ? 1 : 0), s0 = cut * cuts.steps + min(cut, cuts.longer);
    const int chunks = (ns + GS_CHUNK - 1) / GS_CHUNK;

    const int a_voff = (lane >> 3) * K * 2 + ((lane & 7) ^ (lane >> 3)) * 16;
    auto fetch_a = [&](unsigned char *buf, int chunk) {
#pragma unroll
        for (int i = 0; i < ND; i++) {
            const int idx = wave + GS_WAVES * i, step = idx / (2 * NP), plane = idx / NP % 2, grp = idx % NP, k = chunk * GS_CHUNK + step;
            const bool mine = idx < 2 * GS_CHUNK * NP, live = mine && k < ns;
            const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc((void *)(plane ? Alo : Ahi), 0, live ? M * K * 2 : 0, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(d, (__attribute__((address_space(3))) void *)(buf + (mine ? step * STEP + (grp >> 1) * 4096 + plane * 2048 + (grp & 1) * 1024 : BUF)), 16,
                                                     a_voff + grp * 16 * K, live ? (s0 + k) * 128 : 0, 0, 0);
        }
    };
    const unsigned char *w = (const unsigned char *)Wf + (size_t)(strip * CB + cb) * 64 * K;
    const int w_voff = (lane & 31) * K * 2 + (lane >> 5) * 64;               /* row-major weights: a lane's own row */
    const bool here = FRAG || (strip * CB + cb) * 32 < N;                    /* of these the last strip may have less than its columns */
    u32x4 ring[D][4];
    auto request = [&](u32x4 (&r)[4], int i) {                               /* this wave's i-th step */
        const int k = i * KW + kw;
        const bool live = k < ns && here;
        const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc((void *)w, 0, live ? 64 * K : 0, 0x00020000);
#pragma unroll
        for (int j = 0; j < 4; j++) r[j] = FRAG ? gr_ld_nt(d, lane * 16 + 1024 * j, live ? (s0 + k) * 4096 : 0) : gm_ldb(d, w_voff + 16 * j, live ? (s0 + k) * 128 : 0);
    };
    f32x16 acc[MG];
#pragma unroll
    for (int a = 0; a < MG; a++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[a][v] = 0.f;
    int f_off[4];
#pragma unroll
    for (int j = 0; j < 4; j++) f_off[j] = (lane & 31) * 128 + ((4 * (lane >> 5) + j) ^ (lane & 7)) * 16;
    auto multiply = [&](const unsigned char *buf, int step, const u32x4 (&r)[4]) {
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int a = 0; a < MG; a++)
                acc[a] = gm_bf16::mfma(*reinterpret_cast<const u32x4 *>(buf + step * STEP + a * 4096 + f_off[j]), r[j], acc[a]);
    };
    /* chunk c: behind the requests for its rows this wave has made at least `after` others (vmcnt(after)); `next` takes the rows of
     * chunk c + 2, which every wave has read as those of chunk c - 1 when all have met here.  (A bare barrier:
     * __syncthreads() waits for all rows on their way, those of chunk c + 1 too.  What a wave has read from LDS it has multiplied by then,
     * and the empty statements keep requests and reads on their side of it.) */
    auto body = [&](int c, const unsigned char *rows, unsigned char *next, auto slot, auto after) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0f70 | (decltype(after)::v & 15) | (decltype(after)::v >> 4 << 14));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        fetch_a(next, c + 2);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < SPW; j++) {
            const int at = (decltype(slot)::v + j) % D;
            multiply(rows, KW == 1 ? j : kw, ring[at]);
            request(ring[at], c * SPW + j + D);
            asm volatile("" ::: "memory");
        }
    };
    fetch_a(buf0, 0);
    fetch_a(buf1, 1);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < D; i++) request(ring[i], i);
    asm volatile("" ::: "memory");
    /* Behind the requests for chunk c's rows stand at least the ND for chunk c + 1's and, KW = 1, one chunk's (D steps) of weights; KW = 3, two
     * chunks' (a step each; three steps at chunk 0, of which the first is multiplied right away).  So one count holds for every chunk, and the
     * code is there once per buffer instead of twice (what runs once comes from memory: 9.0 -> 6.3 KB of code for gate|up at 37 rows). */
    typedef gs_int<ND + 4 * (KW == 1 ? D : D - 1)> after;
    for (int c = 0;; c += 3) {
        body(c, buf0, buf2, gs_int<0>(), after());
        if (c + 1 >= chunks) break;
        body(c + 1, buf1, buf0, gs_int<SPW>(), after());
        if (c + 2 >= chunks) break;
        body(c + 2, buf2, buf1, gs_int<2 * SPW>(), after());
        if (c + 3 >= chunks) break;
    }

    /* accumulator element v of lane l: row 8*(v/4) + 4*(l/32) + v%4 of the 16 (v < 8: hi, then lo), column l%32 */
    const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(C + (size_t)cut * plane_stride, 0, here ? M * ldc * 4 : 0, 0x00020000);
    const int out_at = 4 * (lane >> 5) * ldc * 4 + (strip * (32 * CB) + 32 * cb + (lane & 31)) * 4;
    auto store = [&](int qd, const f32x4 &x) {
        const f32x4 q[1] = {x};
        const int none[1] = {};
        gm_store_quad<gm_bf16, 1>(out, out_at + 8 * qd * ldc * 4, ldc * 4, q, i32x4{}, none);
    };
    auto quad = [&](int qd) {
        const f32x16 &p = acc[qd / 2];
        const int v = 4 * (qd % 2);
        return f32x4{__fadd_rn(p[v], p[v + 8]), __fadd_rn(p[v + 1], p[v + 9]), __fadd_rn(p[v + 2], p[v + 10]), __fadd_rn(p[v + 3], p[v + 11])};
    };
    __builtin_amdgcn_s_waitcnt(0x0f70);                                      /* nothing arrives in the buffers any more */
    if constexpr (KW == 1) {
#pragma unroll
        for (int qd = 0; qd < NP; qd++) store(qd, quad(qd));
    } else {
        /* parked over the buffers; added in the order of the waves */
        __syncthreads();
        constexpr int HERE = BUF / (1024 * NP) < GS_WAVES ? BUF / (1024 * NP) : GS_WAVES;        /* waves that park in the first buffer */
        auto park = [&](int wv, int qd) {
            return reinterpret_cast<f32x4 *>((wv < HERE ? buf0 + wv * (1024 * NP) : buf1 + (wv - HERE) * (1024 * NP)) + qd * 1024 + lane * 16);
        };
#pragma unroll
        for (int qd = 0; qd < NP; qd++) *park(wave, qd) = quad(qd);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < (NP + KW - 1) / KW; i++) {
            const int qd = kw + KW * i;
            if (qd < NP) {
                f32x4 x = *park(cb * KW, qd);
#pragma unroll
                for (int r = 1; r < KW; r++) {
                    const f32x4 y = *park(cb * KW + r, qd);
                    x = f32x4{__fadd_rn(x.x, y.x), __fadd_rn(x.y, y.y), __fadd_rn(x.z, y.z), __fadd_rn(x.w, y.w)};
                }
                store(qd, x);
            }
        }
    }
}

template <int NP, int KW, bool FRAG>
static void gs_launch(float *d_C, int ldc, size_t plane_stride, const uint16_t *d_Ahi, const uint16_t *d_Alo, const uint16_t *d_Wf, int M, int N, int K, int cuts) {
    const int tn = 32 * GS_WAVES / KW, strips = (N + tn - 1) / tn;
    hipLaunchKernelGGL((vt_gemm_strip_kernel<NP, KW, FRAG>), dim3(strips * cuts), dim3(64 * GS_WAVES), 0, g_vt.stream, d_C, ldc, plane_stride, d_Ahi, d_Alo, d_Wf, M, N, K,
                       vt_divisor_of(strips, strips * cuts), gm_cuts_of(K, cuts));
}

void vt_launch_gemm_few_rows(float *d_C, int ldc, size_t plane_stride, const uint16_t *d_Ahi, const uint16_t *d_Alo,
                             const uint16_t *d_Wf, int M, int N, int K, const vt_gemm_plan &pl) {
    typedef void (*fn)(float *, int, size_t, const uint16_t *, const uint16_t *, const uint16_t *, int, int, int, int);
#define GS_BY_ROWS(KW, FRAG) {gs_launch<1, KW, FRAG>, gs_launch<2, KW, FRAG>, gs_launch<3, KW, FRAG>, gs_launch<4, KW, FRAG>, gs_launch<5, KW, FRAG>, gs_launch<6, KW, FRAG>, \
                              gs_launch<7, KW, FRAG>, gs_launch<8, KW, FRAG>}
    static const fn launch[3][8] = {GS_BY_ROWS(1, true), GS_BY_ROWS(3, true), GS_BY_ROWS(3, false)};
    launch[pl.tn == GS_WIDE ? 0 : pl.row_major ? 2 : 1][(M + 7) / 8 - 1](d_C, ldc, plane_stride, d_Ahi, d_Alo, d_Wf, M, N, K, pl.cuts);
}

/*
 * vt_gemm_rows.hip - the matrix product of vt_gemm.hip for few rows (a short prompt): C[M,N] = X[M,K] W[N,K]^T
 * with M <= 64, weights in fragment order, activations as (hi, lo) bf16 planes, fp32 accumulation.
 *
 * With so few rows the product is a weight stream: at 64 rows a CU needs 1024 of the 2900 cycles in which its
 * share of HBM delivers 32 KB of weights.  What counts is that every CU has a share, and an equal one.  A tile
 * of vt_gemm_wide_kernel is 256 columns wide, so gate|up has 72 of them for 256 CUs, and the other products
 * can only give more CUs something to do by cutting K into many planes.  Here a workgroup owns 64 columns and
 * its waves share K among themselves: wave w takes the 64-wide K steps w, w + NW, ... of the workgroup's range,
 * keeps its own sums for all rows, and the waves' sums are added through LDS at the end (in wave order: the
 * result does not depend on timing).  288 gate|up tiles (256 whole and the last 32 in 8 K cuts), 96 q|k|v tiles
 * in 2 cuts, 48 output and down tiles in 4 and 5 then fill the chip with at most 5 planes.
 *
 * No two waves work on the same K step, so nobody shares anything before the end: a wave stages its own
 * activation rows through its own piece of LDS (one stage; the LDS serves a wave's accesses in order, so the
 * rows of the next step are written over those of this one behind its last reads) and there is no barrier in
 * the K loop.  The weights of a step go straight into the B operand registers, two steps ahead.  Every request
 * goes through a buffer descriptor whose size says whether there is anything to load: steps past a wave's last
 * one and rows past M ask for nothing, without a branch (behind a branch the compiler would wait for all
 * outstanding loads).
 *
 * What bounds it, from 26 layers in rotation: the stream plus about 4 us of launch, first latency, sums and
 * stores, plus the activation rows, which every workgroup reads for itself at about 50 KB/us per CU (1.3 us per
 * 8 rows in the gate|up product; that is why the passes over the rows are a template argument and the kernel is
 * not used beyond 64 rows, where rows shared through LDS cost less).  us per launch, q|k|v / output / gate|up /
 * down: 10.0 / 7.7 / 22.2 / 11.9 at 6 rows, 14.5 / 10.4 / 29.6 / 16.5 at 37, 15.5 / 11.5 / 34.1 / 18.8 at 64;
 * vt_gemm_wide_kernel takes 21.7 / 16.8 / 62.1 / 27.9 at 37.
 */
#include "vt_state.h"
#include "vt_gemm.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define GR_TN 64
#define GR_ROWB 144                       /* bytes per staged row: 64 bf16 + 16 (fragment reads cover all banks) */

struct gr_part {
    float *C;                             /* `splits` planes of [M, ldc], plane_stride floats apart */
    const uint16_t *Wf;                   /* fragment-order weights of the part's first column */
    size_t plane_stride;
    int ldc, n_tiles, splits;
    uint16_t *h_hi, *h_lo;                /* gate|up (paired column order): planes of SiLU(gate) * up instead of C */
    int ldh;
};
struct gr_plan { gr_part part[2]; int n_parts; };

struct gr_bregs { u32x4 v[2][4]; };       /* weights of one K step: [column block][16-wide slice] */

__device__ __forceinline__ u32x4 gr_ld(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
}
__device__ __forceinline__ u32x4 gr_ld_nt(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 2 /* non-temporal: weights are read once */);
}

/* One workgroup's piece of a product: a 64-column tile over one K cut */
struct gr_item {
    const unsigned char *w;               /* weights of the tile */
    int part, nt, sp, s0, n;              /* n: this wave's K steps s0 + wave + 8 i */
};

template <int NW>
__device__ __forceinline__ gr_item gr_item_at(const gr_plan &plan, int part, int id, int K, int wave) {
    const gr_part &P = plan.part[part];
    /* slot id lands on XCD id % 8: an XCD takes a run of items, N tile fastest, i.e. few K cuts: the slice of
     * the planes that its L2 has to fetch is that of its cuts */
    const int items = P.n_tiles * P.splits;
    const int li = (items & 7) == 0 ? (id & 7) * (items >> 3) + (id >> 3) : id;
    gr_item it;
    it.part = part;
    it.nt = li % P.n_tiles;
    it.sp = li / P.n_tiles;
    const int steps = K / 64, q = steps / P.splits, rem = steps % P.splits;
    const int ns = q + (it.sp < rem ? 1 : 0);
    it.s0 = it.sp * q + min(it.sp, rem);
    it.n = ns > wave ? (ns - wave + NW - 1) / NW : 0;
    it.w = (const unsigned char *)(P.Wf + (size_t)it.nt * GR_TN * K);
    return it;
}

/* NP passes of 8 rows: M <= 8 NP; NW waves */
template <int NP, int NW>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW / 4, NW / 4)))
vt_gemm_rows_kernel(gr_plan plan, const uint16_t *Ahi, const uint16_t *Alo, int M, int K) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    constexpr int MB = (NP + 3) / 4;                                         /* blocks of 32 rows */
    constexpr int PLANE = 32 * MB * GR_ROWB;
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int blk_bytes = 64 * K;                                            /* 32 columns x K x 2 bytes */
    const int a_bytes = M * K * 2;
    unsigned char *mine = lds + wave * (2 * PLANE);
    const int lr = lane >> 3, lc = lane & 7;                                 /* staging: row lr + 8 p, 16-byte chunk lc */
    const int a_voff = (lr * K + lc * 8) * 2, a_pass = 16 * K;               /* byte distance of two passes */
    const int st_off = lr * GR_ROWB + lc * 16;
    const int fa_off = (lane & 31) * GR_ROWB + (lane >> 5) * 64;

    u32x4 ra_hi[NP], ra_lo[NP];
    auto fetch_a = [&](const gr_item &it, int i) {
        const int soff = i < it.n ? (it.s0 + wave + NW * i) * 128 : 0;
        const __amdgpu_buffer_rsrc_t h = __builtin_amdgcn_make_buffer_rsrc((void *)Ahi, 0, i < it.n ? a_bytes : 0, 0x00020000);
        const __amdgpu_buffer_rsrc_t l = __builtin_amdgcn_make_buffer_rsrc((void *)Alo, 0, i < it.n ? a_bytes : 0, 0x00020000);
#pragma unroll
        for (int p = 0; p < NP; p++) {
            ra_hi[p] = gr_ld(h, a_voff + p * a_pass, soff);
            ra_lo[p] = gr_ld(l, a_voff + p * a_pass, soff);
        }
    };
    auto fetch_b_slice = [&](const gr_item &it, gr_bregs &r, int i, int j) {
        const int soff = i < it.n ? (it.s0 + wave + NW * i) * 4096 : 0;
        const __amdgpu_buffer_rsrc_t w = __builtin_amdgcn_make_buffer_rsrc((void *)it.w, 0, i < it.n ? 2 * blk_bytes : 0, 0x00020000);
        r.v[0][j] = gr_ld_nt(w, lane * 16 + 1024 * j, soff);
        r.v[1][j] = gr_ld_nt(w, lane * 16 + 1024 * j, soff + blk_bytes);
    };
    auto store_a = [&]() {
#pragma unroll
        for (int p = 0; p < NP; p++) {
            *reinterpret_cast<u32x4 *>(mine + st_off + 8 * p * GR_ROWB) = ra_hi[p];
            *reinterpret_cast<u32x4 *>(mine + PLANE + st_off + 8 * p * GR_ROWB) = ra_lo[p];
        }
    };
    struct frags { bf16x8 hi[MB], lo[MB]; };
    auto read_frags = [&](frags &f, int ks) {
#pragma unroll
        for (int a = 0; a < MB; a++) {
            f.hi[a] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(mine + fa_off + 32 * a * GR_ROWB + 16 * ks));
            f.lo[a] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(mine + PLANE + fa_off + 32 * a * GR_ROWB + 16 * ks));
        }
    };
    f32x16 acc[MB][2];
    auto mma = [&](const frags &f, const gr_bregs &rb, int ks) {
        const bf16x8 b0 = __builtin_bit_cast(bf16x8, rb.v[0][ks]), b1 = __builtin_bit_cast(bf16x8, rb.v[1][ks]);
#pragma unroll
        for (int a = 0; a < MB; a++) {
            acc[a][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.lo[a], b0, acc[a][0], 0, 0, 0);
            acc[a][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.lo[a], b1, acc[a][1], 0, 0, 0);
        }
#pragma unroll
        for (int a = 0; a < MB; a++) {
            acc[a][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.hi[a], b0, acc[a][0], 0, 0, 0);
            acc[a][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.hi[a], b1, acc[a][1], 0, 0, 0);
        }
    };
    gr_bregs b0, b1;
    frags f0, f1;
    /* the first requests of an item: the rows of step 0, the weights of steps 0 and 1 */
    auto begin = [&](const gr_item &it) {
        fetch_a(it, 0);
#pragma unroll
        for (int j = 0; j < 4; j++) fetch_b_slice(it, b0, 0, j);
#pragma unroll
        for (int j = 0; j < 4; j++) fetch_b_slice(it, b1, 1, j);
        __builtin_amdgcn_sched_barrier(0);
    };
    /* step i: the stage holds its rows, f0 their slice 0; ra holds the rows of step i + 1.  A slice's weight
     * registers are requested again (step i + 2) as soon as the slice has been multiplied. */
    auto step = [&](const gr_item &it, int i, gr_bregs &cur) {
        read_frags(f1, 1);
        mma(f0, cur, 0);
        __builtin_amdgcn_sched_barrier(0);
        fetch_b_slice(it, cur, i + 2, 0);
        read_frags(f0, 2);
        mma(f1, cur, 1);
        __builtin_amdgcn_sched_barrier(0);
        fetch_b_slice(it, cur, i + 2, 1);
        read_frags(f1, 3);
        mma(f0, cur, 2);
        __builtin_amdgcn_sched_barrier(0);
        fetch_b_slice(it, cur, i + 2, 2);
        store_a();
        fetch_a(it, i + 2);
        read_frags(f0, 0);
        mma(f1, cur, 3);
        __builtin_amdgcn_sched_barrier(0);
        fetch_b_slice(it, cur, i + 2, 3);
    };
    auto multiply = [&](const gr_item &it) {
#pragma unroll
        for (int a = 0; a < MB; a++)
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[a][b][v] = 0.f;
        store_a();
        fetch_a(it, 1);
        __builtin_amdgcn_sched_barrier(0);
        read_frags(f0, 0);
        for (int i = 0; i < it.n; i += 2) {
            step(it, i, b0);
            step(it, i + 1, b1);          /* past the last one: zeros times zeros */
        }
    };
    /* the waves' sums: parked as quads of accumulator elements over each wave's own stage, added in wave order */
    auto finish = [&](const gr_item &it) {
        const gr_part &P = plan.part[it.part];
        float *park = reinterpret_cast<float *>(mine);
#pragma unroll
        for (int a = 0; a < MB; a++)
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int vq = 0; vq < 4; vq++)
                    *reinterpret_cast<f32x4 *>(park + (((a * 4 + vq) * 2 + b) * 64 + lane) * 4) =
                        f32x4{acc[a][b][4 * vq], acc[a][b][4 * vq + 1], acc[a][b][4 * vq + 2], acc[a][b][4 * vq + 3]};
        __syncthreads();
        /* wave w finishes the quads w, w + NW, ...: rows 8 q + 4 (lane / 32) + 0..3, column lane % 32 of both blocks */
#pragma unroll
        for (int qd = wave; qd < NP; qd += NW) {
            f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int w = 0; w < NW; w++)
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    const f32x4 v = *reinterpret_cast<const f32x4 *>(lds + w * (2 * PLANE) + ((qd * 2 + b) * 64 + lane) * 16);
                    s[b].x = __fadd_rn(s[b].x, v.x); s[b].y = __fadd_rn(s[b].y, v.y);
                    s[b].z = __fadd_rn(s[b].z, v.z); s[b].w = __fadd_rn(s[b].w, v.w);
                }
            const int row0 = 8 * qd + 4 * (lane >> 5), c = lane & 31;
            if (P.h_hi) {
                const vt_h_quad h = vt_silu_mul_quad(s[0], s[1]);                /* voxtral_tts_llm.c:346-350 */
                const size_t at = (size_t)(row0 + h.row) * P.ldh + it.nt * (GR_TN / 2) + (c & ~1);
#pragma unroll
                for (int r = 0; r < 2; r++)
                    if (row0 + h.row + r < M) {
                        *reinterpret_cast<unsigned *>(P.h_hi + at + (size_t)r * P.ldh) = h.hi[r];
                        *reinterpret_cast<unsigned *>(P.h_lo + at + (size_t)r * P.ldh) = h.lo[r];
                    }
            } else {
                float *Cs = P.C + (size_t)it.sp * P.plane_stride + it.nt * GR_TN + c;
#pragma unroll
                for (int v = 0; v < 4; v++)
                    if (row0 + v < M) {
                        Cs[(size_t)(row0 + v) * P.ldc] = s[0][v];
                        Cs[(size_t)(row0 + v) * P.ldc + 32] = s[1][v];
                    }
            }
        }
    };

    /* items blockIdx.x, + gridDim.x, ... of each part in turn; the first requests of the next item go out in
     * front of the sums of this one */
    int part = 0, id = (int)blockIdx.x;
    gr_item it = gr_item_at<NW>(plan, 0, id, K, wave);
    begin(it);
    for (;;) {
        multiply(it);
        id += (int)gridDim.x;
        while (part < plan.n_parts && id >= plan.part[part].n_tiles * plan.part[part].splits) {
            part++;
            id = (int)blockIdx.x;
        }
        if (part >= plan.n_parts) break;
        const gr_item nx = gr_item_at<NW>(plan, part, id, K, wave);
        begin(nx);
        finish(it);
        __syncthreads();                  /* the next item stages over the parked sums */
        it = nx;
    }
    finish(it);
}

int vt_gemm_rows_ok(int M, int N, int K) { return M >= 1 && M <= 64 && N % GR_TN == 0 && K % 64 == 0; }

/* Waves of a workgroup: 8 while the registers of a wave (sums, two sets of weights, staged rows) fit two waves
 * per SIMD; beyond 40 rows they spill (64 rows, gate|up: 63 us against 34 with 4 waves). */
#define GR_ROWS_8_WAVES 40
static int gr_waves(int M) { return M <= GR_ROWS_8_WAVES ? 8 : 4; }

template <int NP>
static int gr_launch_np(const gr_plan &plan, int grid, const uint16_t *d_Ahi, const uint16_t *d_Alo, int M, int K) {
    constexpr int NW = 8 * NP <= GR_ROWS_8_WAVES ? 8 : 4;
    static int attr_set = 0;
    const int lds = NW * 2 * 32 * ((NP + 3) / 4) * GR_ROWB;
    if (!attr_set) {
        if (vt_check(hipFuncSetAttribute((const void *)vt_gemm_rows_kernel<NP, NW>, hipFuncAttributeMaxDynamicSharedMemorySize, lds), "product LDS size"))
            return -1;
        attr_set = 1;
    }
    hipLaunchKernelGGL((vt_gemm_rows_kernel<NP, NW>), dim3(grid), dim3(64 * NW), lds, g_vt.stream, plan, d_Ahi, d_Alo, M, K);
    return 0;
}

static void gr_launch(const gr_plan &plan, const uint16_t *d_Ahi, const uint16_t *d_Alo, int M, int K) {
    static int (*const launch[8])(const gr_plan &, int, const uint16_t *, const uint16_t *, int, int) = {
        gr_launch_np<1>, gr_launch_np<2>, gr_launch_np<3>, gr_launch_np<4>, gr_launch_np<5>, gr_launch_np<6>, gr_launch_np<7>, gr_launch_np<8>};
    const int items = plan.part[0].n_tiles * plan.part[0].splits;     /* every workgroup takes an item of the first part */
    launch[(M + 7) / 8 - 1](plan, items < g_vt.n_cu ? items : g_vt.n_cu, d_Ahi, d_Alo, M, K);
}

int vt_gemm_rows_cuts(int M, int N, int K, int most) {
    /* of the cut counts that leave every CU at most one item, the fewest planes among those with the fewest
     * K steps on the busiest wave */
    const int tiles = N / GR_TN, steps = K / 64, nw = gr_waves(M);
    int best = 1, best_cost = steps;
    for (int c = 1; c <= most && tiles * c <= g_vt.n_cu; c++) {
        const int cost = ((steps + c - 1) / c + nw - 1) / nw;
        if (c == 1 || cost < best_cost) { best = c; best_cost = cost; }
    }
    return best;
}

void vt_launch_gemm_rows(float *d_C, int ldc, size_t plane_stride, const uint16_t *d_Ahi, const uint16_t *d_Alo,
                         const uint16_t *d_Wf, int M, int N, int K, int splits) {
    gr_plan plan = {};
    plan.n_parts = 1;
    plan.part[0] = gr_part{d_C, d_Wf, plane_stride, ldc, N / GR_TN, splits, NULL, NULL, 0};
    gr_launch(plan, d_Ahi, d_Alo, M, K);
}

void vt_launch_gemm_rows_swiglu(uint16_t *d_hhi, uint16_t *d_hlo, int ldh, float *d_tail, const uint16_t *d_Ahi,
                                const uint16_t *d_Alo, const uint16_t *d_Wf, int M, int n_main, int n_tail, int K, int tail_splits) {
    gr_plan plan = {};
    if (n_main > 0) plan.part[plan.n_parts++] = gr_part{NULL, d_Wf, 0, 0, n_main / GR_TN, 1, d_hhi, d_hlo, ldh};
    if (n_tail > 0)
        plan.part[plan.n_parts++] = gr_part{d_tail, d_Wf + (size_t)n_main * K, (size_t)M * n_tail, n_tail, n_tail / GR_TN, tail_splits, NULL, NULL, 0};
    gr_launch(plan, d_Ahi, d_Alo, M, K);
}

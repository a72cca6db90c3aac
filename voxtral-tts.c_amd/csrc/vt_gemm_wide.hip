/*
 * vt_gemm_wide.hip - the matrix product of vt_gemm.hip for the backbone's prefill, more than 64 rows:
 * C[M,N] = X[M,K] W[N,K]^T on (hi, lo) bf16 activation planes and fragment-order weights, fp32 accumulation.
 * Also the plans of the backbone's products: which tile, and which columns in how many K cuts.
 *
 * A wave owns MB x 32 rows (MB 3 or 4) x 64 columns: the weights of its 64 columns are nobody else's among the
 * waves that work on the same K step, so they go from global memory straight into the B operand registers, and
 * only the activation planes pass through the LDS: 8 KB of fragment reads per 16 matrix instructions, half
 * the LDS bandwidth (a 64 x 64 wave tile with both operands in LDS, vt_gemm_mfma_kernel, needs three quarters).
 * One workgroup of four waves per CU (a wave may then use the whole register file of its SIMD: up to 128
 * accumulator registers, two sets of weight registers, two sets of fragments), in one of two shapes:
 *   CW = 4: four waves side by side, tile MB*32 x 256; the planes of one K step serve four waves;
 *   CW = 2: two waves side by side and two K steps at a time, tile MB*32 x 128; the two halves of K are added
 *           through LDS at the end.  Half the tile, for row counts whose 256-column tiles do not deal out over
 *           the CUs, at the price of twice the plane traffic (L2 and LDS stores) per matrix instruction.
 * Two LDS stages: the planes of the next step are written while this one is multiplied, one barrier per step;
 * the global loads of the step after that are in flight meanwhile (every request unconditional, through
 * descriptors whose size says whether there is anything to load, so the waits count exactly).
 * The k order inside a matrix instruction is free as long as both operands agree: lane group g (lane / 32)
 * takes k = 32 g + 8 ks .. + 8 of the 64-wide step in slice ks.
 * A lane's operand is 8 consecutive k of ONE weight row, and the 32 lanes of a group are 32 different rows:
 * read from the row-major matrix, every load instruction touches 32 lines 6 KB apart, and the CU's address
 * pipeline, not the matrix cores, sets the pace (measured: 434 against 518 TFLOP/s).  The backbone therefore
 * keeps a second copy of its matrices in fragment order, written once at upload by vt_frag_layout_kernel:
 * every load is then 1 KB of consecutive bytes.
 *
 * A launch has at most one workgroup per CU, which walks its items: first whole tiles, as many rounds of them
 * as every CU can take part in, then the tiles that are left as K cuts, so many that every CU gets one.  The
 * first requests of an item go out in front of the stores of the one before it.  Only the columns of the cut
 * tiles have more than one partial plane; whoever reads the result is told from which column on (vt_gemm_plan).
 */
#include "vt_state.h"
#include "vt_gemm.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define GW_ROWB 144                       /* bytes per staged row: 64 bf16 + 16 (fragment reads cover all banks) */

/* One set of equal items: tiles of n_tiles x (row tiles), K in `splits` cuts */
struct gw_part {
    float *C;                             /* `splits` planes of [M, ldc], plane_stride floats apart */
    const uint16_t *Wf;                   /* fragment-order weights of the set's first column */
    size_t plane_stride;
    int ldc, n_tiles, splits;
    /* gate|up product in the paired column order (vt_launch_frag_layout with pair = 1): instead of C, the
     * (hi, lo) planes of SiLU(gate) * up, row pitch ldh */
    uint16_t *h_hi, *h_lo;
    int ldh;
};
struct gw_list { gw_part part[2]; int n_parts, m_tiles; };

struct gw_item {
    const unsigned char *w;               /* weights of the tile's first column */
    int part, mt, nt, sp, s0, ns;         /* this cut's K steps: s0 .. s0 + ns - 1 (64 wide) */
};

struct gw_bregs { u32x4 v[2][4]; };       /* weights of one K step: [column block][16-wide slice] */

template <int TN>
__device__ __forceinline__ gw_item gw_item_at(const gw_list &list, int part, int id, int K) {
    const gw_part &P = list.part[part];
    /* Slot id lands on XCD id % 8.  An XCD takes a run of consecutive items, row tile fastest, then N tile,
     * then K cut: the row tiles of a (K cut, N tile) pair share its weights, the N tiles of a K cut share the
     * activation planes of that cut, and both leave the memory side once per XCD instead of once per workgroup. */
    const int items = list.m_tiles * P.n_tiles * P.splits, x = id & 7, run = items >> 3, rem = items & 7;
    const int li = x * run + min(x, rem) + (id >> 3);
    gw_item it;
    it.part = part;
    it.mt = li % list.m_tiles;
    const int ci = li / list.m_tiles;
    it.nt = ci % P.n_tiles;
    it.sp = ci / P.n_tiles;
    const int steps = K / 64, q = steps / P.splits, r = steps % P.splits;
    it.ns = q + (it.sp < r ? 1 : 0);
    it.s0 = it.sp * q + min(it.sp, r);
    it.w = (const unsigned char *)(P.Wf + (size_t)it.nt * TN * K);
    return it;
}

__device__ __forceinline__ u32x4 gw_ld(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
}

template <int MB, int CW>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
vt_gemm_wide_kernel(gw_list list, const uint16_t *Ahi, const uint16_t *Alo, int M, int K) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    constexpr int KW = 4 / CW, TM = 32 * MB, TN = 64 * CW;
    constexpr int NP = 4 * MB / CW;                        /* staging passes over a plane, 8 * CW rows each */
    constexpr int PLANE = TM * GW_ROWB, GROUP = 2 * PLANE, STAGE = KW * GROUP;
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int cw = wave % CW, kw = wave / CW;              /* column block of the tile; which of the KW K steps */
    const int tg = (int)threadIdx.x - kw * 64 * CW;
    const int lr = tg >> 3, lc = tg & 7;                   /* staging: row lr + 8 CW p, 16-byte chunk lc */
    const int a_voff = (lr * K + lc * 8) * 2, a_pass = 16 * CW * K, blk_bytes = 64 * K;
    const int st_off = kw * GROUP + lr * GW_ROWB + lc * 16;
    const int fa_off = kw * GROUP + (lane & 31) * GW_ROWB + (lane >> 5) * 64;

    struct aregs { u32x4 hi[NP], lo[NP]; };                /* staged rows of one K step, both planes */
    /* rows past M and steps past the cut's end: beyond the descriptor's size, nothing is loaded (zeros) */
    auto fetch_a = [&](const gw_item &it, const uint16_t *plane, u32x4 (&r)[NP], int i) {
        const int s = KW * i + kw, rows = min(M - it.mt * TM, TM);
        const bool live = s < it.ns;
        const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc((void *)(plane + (size_t)it.mt * TM * K), 0, live ? rows * K * 2 : 0, 0x00020000);
        const int soff = live ? (it.s0 + s) * 128 : 0;
#pragma unroll
        for (int p = 0; p < NP; p++) r[p] = gw_ld(d, a_voff + p * a_pass, soff);
    };
    auto fetch_b_slice = [&](const gw_item &it, gw_bregs &r, int i, int j) {
        const int s = KW * i + kw;
        const bool live = s < it.ns;
        const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc((void *)(it.w + (size_t)cw * 2 * blk_bytes), 0, live ? 2 * blk_bytes : 0, 0x00020000);
        const int soff = live ? (it.s0 + s) * 4096 : 0;
        r.v[0][j] = gw_ld(d, lane * 16 + 1024 * j, soff);
        r.v[1][j] = gw_ld(d, lane * 16 + 1024 * j, soff + (live ? blk_bytes : 0));
    };
    auto store_a = [&](const u32x4 (&r)[NP], int at) {
#pragma unroll
        for (int p = 0; p < NP; p++) *reinterpret_cast<u32x4 *>(lds + at + st_off + 8 * CW * p * GW_ROWB) = r[p];
    };
    struct frags { bf16x8 hi[MB], lo[MB]; };
    auto read_frags = [&](frags &f, int stage, int ks) {
        const unsigned char *base = lds + stage * STAGE + fa_off + ks * 16;
#pragma unroll
        for (int a = 0; a < MB; a++) {
            f.hi[a] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(base + 32 * a * GW_ROWB));
            f.lo[a] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(base + PLANE + 32 * a * GW_ROWB));
        }
    };
    f32x16 acc[MB][2];
    auto mma = [&](const frags &f, const gw_bregs &rb, int ks) {
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

    /* One step: stage `stage` holds the planes of step i and `cur` its weights; ra holds the planes of step
     * i + 1 (requested two steps ago: with one step between request and store, the step takes as long as a load,
     * 1.2 us, whatever the tile); f0 already holds the fragments of slice 0.  Four regions of 4 MB matrix
     * instructions each; the other instructions of a region (the fragment reads of the next slice, in the first
     * two also the LDS stores of a plane of step i + 1 and its requests of step i + 3, in all but the first the
     * two weight requests that refill the slice just used) are dealt out between the matrix instructions, one
     * after every second, so that the matrix pipe never waits for a block of them to issue.  The step's one
     * barrier stands in front of the last region: by then every wave has issued (and waited for) its stores
     * into the other stage and its last reads of this one, so the first fragments of step i + 1 are read under
     * the last matrix instructions of step i. */
    gw_bregs b0, b1;
    aregs ra0, ra1;                       /* the rows of even and of odd steps */
    frags f0, f1;
#define GW_FENCE() __builtin_amdgcn_sched_barrier(0)
#define GW_MFMA2() __builtin_amdgcn_sched_group_barrier(0x008, 2, 0)
#define GW_DSR1() __builtin_amdgcn_sched_group_barrier(0x100, 1, 0)
#define GW_DSW1() __builtin_amdgcn_sched_group_barrier(0x200, 1, 0)
#define GW_VMR1() __builtin_amdgcn_sched_group_barrier(0x020, 1, 0)
    auto step = [&](const gw_item &it, int i, int stage, gw_bregs &cur, aregs &ra) {
        const int other = (stage ^ 1) * STAGE;
        GW_FENCE();
        store_a(ra.hi, other);
        fetch_a(it, Ahi, ra.hi, i + 3);
        read_frags(f1, stage, 1);
        mma(f0, cur, 0);
#pragma unroll
        for (int k = 0; k < 2 * MB; k++) { GW_MFMA2(); GW_DSR1(); if (k < NP) { GW_DSW1(); GW_VMR1(); } }
        GW_FENCE();
        store_a(ra.lo, other + PLANE);
        fetch_a(it, Alo, ra.lo, i + 3);
        fetch_b_slice(it, cur, i + 2, 0);
        read_frags(f0, stage, 2);
        mma(f1, cur, 1);
#pragma unroll
        for (int k = 0; k < 2 * MB; k++) { GW_MFMA2(); GW_DSR1(); if (k < NP) { GW_DSW1(); GW_VMR1(); } if (k < 2) GW_VMR1(); }
        GW_FENCE();
        fetch_b_slice(it, cur, i + 2, 1);
        read_frags(f1, stage, 3);
        mma(f0, cur, 2);
#pragma unroll
        for (int k = 0; k < 2 * MB; k++) { GW_MFMA2(); GW_DSR1(); if (k < 2) GW_VMR1(); }
        GW_FENCE();
        __syncthreads();
        GW_FENCE();
        fetch_b_slice(it, cur, i + 2, 2);
        read_frags(f0, stage ^ 1, 0);
        mma(f1, cur, 3);
#pragma unroll
        for (int k = 0; k < 2 * MB; k++) { GW_MFMA2(); GW_DSR1(); if (k < 2) GW_VMR1(); }
        GW_FENCE();
        fetch_b_slice(it, cur, i + 2, 3);
    };
    /* the first requests of an item: the planes and weights of steps 0 and 1 */
    auto begin = [&](const gw_item &it) {
        fetch_a(it, Ahi, ra0.hi, 0);
        fetch_a(it, Alo, ra0.lo, 0);
#pragma unroll
        for (int j = 0; j < 4; j++) fetch_b_slice(it, b0, 0, j);
        fetch_a(it, Ahi, ra1.hi, 1);
        fetch_a(it, Alo, ra1.lo, 1);
#pragma unroll
        for (int j = 0; j < 4; j++) fetch_b_slice(it, b1, 1, j);
        GW_FENCE();
    };
    auto multiply = [&](const gw_item &it) {
#pragma unroll
        for (int a = 0; a < MB; a++)
#pragma unroll
            for (int b = 0; b < 2; b++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[a][b][v] = 0.f;
        store_a(ra0.hi, 0);
        store_a(ra0.lo, PLANE);
        fetch_a(it, Ahi, ra0.hi, 2);
        fetch_a(it, Alo, ra0.lo, 2);
        GW_FENCE();
        __syncthreads();
        read_frags(f0, 0, 0);
        const int n = (it.ns + KW - 1) / KW;
        int i = 0;
        for (; i + 1 < n; i += 2) {
            step(it, i, 0, b0, ra1);
            step(it, i + 1, 1, b1, ra0);
        }
        if (i < n) step(it, i, 0, b0, ra1);
    };
#undef GW_MFMA2
#undef GW_DSR1
#undef GW_DSW1
#undef GW_VMR1
#undef GW_FENCE

    /* accumulator element v of lane l: row 8*(v/4) + 4*(l/32) + v%4, column l%32; quad (a, vq) holds v = 4 vq .. + 3 */
    auto emit = [&](const gw_part &P, const gw_item &it, int a, int vq, const f32x4 &q0, const f32x4 &q1) {
        const int row0 = it.mt * TM + 32 * a + 8 * vq + 4 * (lane >> 5), c = lane & 31;
        if (P.h_hi) {
            /* a wave's two column blocks are the gates and the ups of the same 32 h columns (voxtral_tts_llm.c:346-350) */
            const vt_h_quad h = vt_silu_mul_quad(q0, q1);
            const size_t at = (size_t)(row0 + h.row) * P.ldh + it.nt * (TN / 2) + 32 * cw + (c & ~1);
#pragma unroll
            for (int r = 0; r < 2; r++)
                if (row0 + h.row + r < M) {
                    *reinterpret_cast<unsigned *>(P.h_hi + at + (size_t)r * P.ldh) = h.hi[r];
                    *reinterpret_cast<unsigned *>(P.h_lo + at + (size_t)r * P.ldh) = h.lo[r];
                }
        } else {
            float *Cs = P.C + (size_t)it.sp * P.plane_stride + it.nt * TN + 64 * cw + c;
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (row0 + v < M) {
                    Cs[(size_t)(row0 + v) * P.ldc] = q0[v];
                    Cs[(size_t)(row0 + v) * P.ldc + 32] = q1[v];
                }
        }
    };
    auto quad = [&](int a, int b, int vq) { return f32x4{acc[a][b][4 * vq], acc[a][b][4 * vq + 1], acc[a][b][4 * vq + 2], acc[a][b][4 * vq + 3]}; };
    auto finish = [&](const gw_item &it) {
        const gw_part &P = list.part[it.part];
        if constexpr (KW == 1) {
#pragma unroll
            for (int a = 0; a < MB; a++)
#pragma unroll
                for (int vq = 0; vq < 4; vq++) emit(P, it, a, vq, quad(a, 0, vq), quad(a, 1, vq));
        } else {
            /* the two waves of a column block hold the sums over the even and the odd K steps: each parks the half
             * of its quads that the other one finishes */
            float *park = reinterpret_cast<float *>(lds) + (size_t)wave * (MB * 4 * 256);
            const float *theirs = reinterpret_cast<const float *>(lds) + (size_t)(wave ^ CW) * (MB * 4 * 256);
            __syncthreads();
#pragma unroll
            for (int a = 0; a < MB; a++)
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int b = 0; b < 2; b++)
                        *reinterpret_cast<f32x4 *>(park + (((a * 2 + h) * 2 + b) * 64 + lane) * 4) = kw == 0 ? quad(a, b, 2 + h) : quad(a, b, h);
            __syncthreads();
#pragma unroll
            for (int a = 0; a < MB; a++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    f32x4 q[2];
#pragma unroll
                    for (int b = 0; b < 2; b++) {
                        const f32x4 o = *reinterpret_cast<const f32x4 *>(theirs + (((a * 2 + h) * 2 + b) * 64 + lane) * 4);
                        const f32x4 m = kw == 0 ? quad(a, b, h) : quad(a, b, 2 + h);
                        q[b] = f32x4{__fadd_rn(m.x, o.x), __fadd_rn(m.y, o.y), __fadd_rn(m.z, o.z), __fadd_rn(m.w, o.w)};
                    }
                    emit(P, it, a, kw == 0 ? h : 2 + h, q[0], q[1]);
                }
        }
    };

    int part = 0, id = (int)blockIdx.x;
    gw_item it = gw_item_at<TN>(list, 0, id, K);
    begin(it);
    for (;;) {
        multiply(it);
        id += (int)gridDim.x;
        while (part < list.n_parts && id >= list.m_tiles * list.part[part].n_tiles * list.part[part].splits) {
            part++;
            id = (int)blockIdx.x;
        }
        if (part >= list.n_parts) break;
        const gw_item nx = gw_item_at<TN>(list, part, id, K);
        begin(nx);
        finish(it);
        __syncthreads();                  /* the next item stages over what this one read */
        it = nx;
    }
    finish(it);
}

/* ---- plans and launches ---------------------------------------------------------------------------- */

/* What a product is expected to take, in us, for the choice between tiles and cuts.  A round of items takes as
 * long as the operands of its steps need to arrive (1.3 / 1.05 us for the 128 / 96 x 256 tile, 2.0 / 1.6 for the
 * 128-column ones, which move 1.5 times the bytes per matrix instruction) and 1.5 us for sums and stores, but no
 * less than the card's power limit lets the matrix cores of its items run (about 1.12 PFLOP/s executed, padding
 * included); a launch takes 5 us; cut planes are written and read once more.  Measured against every tile and
 * cut count at 65 .. 1531 rows: the plan taken is within 5 % of the fastest. */
static float gw_rounds(int items, float item_us, float item_flops) {
    const float power = item_flops / 1.12e9f;
    const int full = items / g_vt.n_cu, rem = items % g_vt.n_cu;
    return full * fmaxf(item_us, g_vt.n_cu * power) + (rem ? fmaxf(item_us, rem * power) : 0.f);
}

static float gw_cost(int M, int N, int K, int mb, int cw, int n_main, int cuts, int swiglu) {
    const int kw = 4 / cw, mt = (M + 32 * mb - 1) / (32 * mb);
    const float t_step = cw == 4 ? (mb == 4 ? 1.30f : 1.05f) : (mb == 4 ? 2.0f : 1.6f);
    const float tile_flops = 4.f * (32 * mb) * (64 * cw) * (float)K;
    const int rest = N / (64 * cw) - n_main;
    float t = 5.f + gw_rounds(mt * n_main, (float)((K / 64 + kw - 1) / kw) * t_step + 1.5f, tile_flops);
    if (rest) {
        t += gw_rounds(mt * rest * cuts, (float)((K / 64 + cuts * kw - 1) / (cuts * kw)) * t_step + 1.5f, tile_flops / cuts);
        if (cuts > 1 || swiglu) t += 1.2f * cuts * M * (float)(rest * 64 * cw) * 4.f / 4.5e6f + (swiglu ? 4.5f : 0.f);
    }
    return t;
}

vt_gemm_plan vt_gemm_frag_plan(int M, int N, int K, int swiglu) {
    vt_gemm_plan best = {0, 1, 0, 1};
    if (vt_gemm_rows_ok(M, N, K)) {
        if (swiglu) {
            best.col0 = N / 64 / g_vt.n_cu * g_vt.n_cu * 64;
            const int rest = (N - best.col0) / 64;
            while (rest && best.cuts < VT_MAX_CUTS && (best.cuts + 1) * rest <= g_vt.n_cu) best.cuts++;
        } else {
            best.cuts = vt_gemm_rows_cuts(M, N, K, VT_MAX_CUTS);
        }
        return best;
    }
    float best_cost = 0.f;
    for (int mb = 3; mb <= 4; mb++)
        for (int cw = 2; cw <= 4; cw += 2) {
            const int mt = (M + 32 * mb - 1) / (32 * mb), nt = N / (64 * cw);
            /* whole tiles: as many as make full rounds over the CUs, or one round fewer, or all */
            const int full = mt * nt / g_vt.n_cu;
            for (int pick = 0; pick < 3; pick++) {
                int n_main = pick == 2 ? nt : (full - pick) * g_vt.n_cu / mt;
                if (n_main < 0 || n_main > nt) continue;
                for (int cuts = 1; cuts <= VT_MAX_CUTS && cuts <= K / 64; cuts++) {
                    if (n_main == nt && cuts > 1) break;
                    if (swiglu && n_main < nt && cuts == 1) continue;
                    const float c = gw_cost(M, N, K, mb, cw, n_main, cuts, swiglu);
                    if (best_cost == 0.f || c < best_cost) {
                        best_cost = c;
                        best = vt_gemm_plan{mb, cw, n_main * 64 * cw, n_main == nt ? 1 : cuts};
                    }
                }
            }
        }
    return best;
}

template <int MB, int CW>
static void gw_launch(const gw_list &list, const uint16_t *d_Ahi, const uint16_t *d_Alo, int M, int K) {
    constexpr int LDS = 2 * (4 / CW) * 2 * 32 * MB * GW_ROWB;
    static int attr_set = 0;
    if (!attr_set) {
        if (vt_check(hipFuncSetAttribute((const void *)vt_gemm_wide_kernel<MB, CW>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS), "product LDS size"))
            return;
        attr_set = 1;
    }
    const int items = list.m_tiles * list.part[0].n_tiles * list.part[0].splits;      /* every workgroup takes an item of the first part */
    hipLaunchKernelGGL((vt_gemm_wide_kernel<MB, CW>), dim3(items < g_vt.n_cu ? items : g_vt.n_cu), dim3(256), LDS, g_vt.stream, list, d_Ahi, d_Alo, M, K);
}

static void gw_run(const vt_gemm_plan &pl, gw_part whole, gw_part cut, const uint16_t *d_Ahi, const uint16_t *d_Alo, int M, int N, int K) {
    gw_list list = {};
    list.m_tiles = (M + 32 * pl.mb - 1) / (32 * pl.mb);
    whole.n_tiles = pl.col0 / (64 * pl.cw);
    whole.splits = 1;
    cut.n_tiles = (N - pl.col0) / (64 * pl.cw);
    cut.splits = pl.cuts;
    if (whole.n_tiles) list.part[list.n_parts++] = whole;
    if (cut.n_tiles) list.part[list.n_parts++] = cut;
    if (pl.mb == 4 && pl.cw == 4) gw_launch<4, 4>(list, d_Ahi, d_Alo, M, K);
    else if (pl.mb == 4) gw_launch<4, 2>(list, d_Ahi, d_Alo, M, K);
    else if (pl.cw == 4) gw_launch<3, 4>(list, d_Ahi, d_Alo, M, K);
    else gw_launch<3, 2>(list, d_Ahi, d_Alo, M, K);
}

void vt_launch_gemm_frag(float *d_C, int ldc, size_t plane_stride, const uint16_t *d_Ahi, const uint16_t *d_Alo,
                         const uint16_t *d_Wf, int M, int N, int K, const vt_gemm_plan &pl) {
    if (pl.mb == 0) { vt_launch_gemm_rows(d_C, ldc, plane_stride, d_Ahi, d_Alo, d_Wf, M, N, K, pl.cuts); return; }
    gw_run(pl, gw_part{d_C, d_Wf, plane_stride, ldc, 0, 0, NULL, NULL, 0},
           gw_part{d_C + pl.col0, d_Wf + (size_t)pl.col0 * K, plane_stride, ldc, 0, 0, NULL, NULL, 0}, d_Ahi, d_Alo, M, N, K);
}

void vt_launch_gemm_frag_swiglu(uint16_t *d_hhi, uint16_t *d_hlo, int ldh, float *d_tail, const uint16_t *d_Ahi,
                                const uint16_t *d_Alo, const uint16_t *d_Wf, int M, int N, int K, const vt_gemm_plan &pl) {
    const int tail = N - pl.col0;
    if (pl.mb == 0)
        vt_launch_gemm_rows_swiglu(d_hhi, d_hlo, ldh, d_tail, d_Ahi, d_Alo, d_Wf, M, pl.col0, tail, K, pl.cuts);
    else
        gw_run(pl, gw_part{NULL, d_Wf, 0, 0, 0, 0, d_hhi, d_hlo, ldh},
               gw_part{d_tail, d_Wf + (size_t)pl.col0 * K, (size_t)M * tail, tail, 0, 0, NULL, NULL, 0}, d_Ahi, d_Alo, M, N, K);
    if (tail) vt_launch_swiglu_pair_tail(d_hhi, d_hlo, ldh, pl.col0 / 2, d_tail, pl.cuts, (size_t)M * tail, M, tail);
}

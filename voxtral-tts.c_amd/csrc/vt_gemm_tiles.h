/*
 * vt_gemm_tiles.h - the tile kernels of the sequence-level products C[M,N] = X[M,K] W[N,K]^T on the matrix cores,
 * fp32 accumulation: vt_gemm_wide_kernel, for weights in fragment order (vt_launch_frag_layout) or, with FRAG false, row-major
 * ones, and, for few rows and fragment order, vt_gemm_rows_kernel.  Both are templates over the number format (gm_bf16, gm_f16x2 below).
 */
#ifndef VT_GEMM_TILES_H
#define VT_GEMM_TILES_H

#include "vt_state.h"
#include "vt_gemm.h"
#include "vt_requests.h"

#include <type_traits>

typedef __bf16 gm_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 gm_f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

/* K in n cuts, of `steps` steps of 64 each and one more in the first `longer` of them */
struct gm_cuts { int n, steps, longer; };
static inline gm_cuts gm_cuts_of(int K, int n) { return gm_cuts{n, K / 64 / n, K / 64 % n}; }

#define GM_STAGE_ROW 144                  /* bytes per staged row: 64 elements of 2 bytes + 16 (fragment reads cover all banks) */

/* The backbone: bf16 weights as they are, fp32 activations as two bf16 planes (hi, lo) */
struct gm_bf16 {
    static constexpr int WP = 1;          /* weight planes */
    static constexpr bool SCALED = false;
    static __device__ __forceinline__ f32x16 mfma(const u32x4 &x, const u32x4 &w, const f32x16 &c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(gm_bf16x8, x), __builtin_bit_cast(gm_bf16x8, w), c, 0, 0, 0);
    }
};
/* The codec: fp32 weights and activations as two fp16 planes each (vt_split_f16x2), rows of both scaled by powers of
 * two so that the planes stay in range; x w = hi hi + hi lo + lo hi (lo lo is at most 2^-22 of the product).  The lo
 * planes are kept 2^6 larger, for small values in rows with a large one, and meet hi times 2^-6, made in registers
 * beside the matrix instructions.  (Dealt out between them by number, as the memory instructions are, it costs 3.5 %
 * of a decode instead of 2; in front of them 2.5.)  The scaling is undone on the sums by its exponents, one per row
 * and one per column. */
struct gm_f16x2 {
    static constexpr int WP = 2;
    static constexpr bool SCALED = true;
    static __device__ __forceinline__ f32x16 mfma(const u32x4 &x, const u32x4 &w, const f32x16 &c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(gm_f16x8, x), __builtin_bit_cast(gm_f16x8, w), c, 0, 0, 0);
    }
};

template <int WP, int NB> struct gm_weights { u32x4 v[WP][NB][4]; };      /* one 64-wide K step: [plane][block of 32 columns][16-wide slice] */
template <int MB> struct gm_frags { u32x4 hi[MB], lo[MB]; };      /* one 16-wide slice of MB blocks of 32 rows, both planes */
template <int MB> struct gm_paired { u32x4 v[MB]; };      /* of MB groups of 16 rows, lanes 0..15 (of 32) their hi, 16..31 their lo plane */

/* A request through a descriptor: one whose size is 0, and a byte offset beyond the size, load nothing (zeros) */
__device__ __forceinline__ u32x4 gm_ldb(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
}

__device__ __forceinline__ u32x4 gm_down(const u32x4 &hi) {
    return __builtin_bit_cast(u32x4, __builtin_bit_cast(gm_f16x8, hi) * (_Float16)(1.0f / (1 << VT_F16_LO_EXP)));
}

/* One slice, MB or MB NB independent sums between two products into the same one.  One weight plane: column block by column block, so that the
 * weights' operand stays the same for 2 MB products in a row, which draws less power than row block by row block (the card's clock under load
 * follows it): 3072 x 9216 at 4096 rows on tiles of 96 x 384 / 128 x 192 / 128 x 384 428 / 376 / 321 -> 417 / 363 / 319 us; the backbone's
 * planned products 1 % faster from 1000 rows on, 0.3 % below.  Two: plane by plane (column block by column block is 0.5 % slower over the codec's products). */
template <class T, int MB, int NB>
__device__ __forceinline__ void gm_multiply(f32x16 (&acc)[MB][NB], const gm_frags<MB> &f, const gm_weights<T::WP, NB> &w, int ks) {
    if constexpr (T::WP == 2) {
#pragma unroll
        for (int a = 0; a < MB; a++)
#pragma unroll
            for (int b = 0; b < NB; b++) acc[a][b] = T::mfma(f.hi[a], w.v[0][b][ks], acc[a][b]);
        u32x4 wd[NB];
#pragma unroll
        for (int b = 0; b < NB; b++) wd[b] = gm_down(w.v[0][b][ks]);
#pragma unroll
        for (int a = 0; a < MB; a++)
#pragma unroll
            for (int b = 0; b < NB; b++) acc[a][b] = T::mfma(f.lo[a], wd[b], acc[a][b]);
#pragma unroll
        for (int a = 0; a < MB; a++) {
            const u32x4 d = gm_down(f.hi[a]);
#pragma unroll
            for (int b = 0; b < NB; b++) acc[a][b] = T::mfma(d, w.v[1][b][ks], acc[a][b]);
        }
    } else {
        /* the small products first */
#pragma unroll
        for (int b = 0; b < NB; b++) {
#pragma unroll
            for (int a = 0; a < MB; a++) acc[a][b] = T::mfma(f.lo[a], w.v[0][b][ks], acc[a][b]);
#pragma unroll
            for (int a = 0; a < MB; a++) acc[a][b] = T::mfma(f.hi[a], w.v[0][b][ks], acc[a][b]);
        }
    }
}

/* the same for paired planes: the sums of both planes' products stand apart, 16 rows above 16 */
template <class T, int MB, int NB>
__device__ __forceinline__ void gm_multiply(f32x16 (&acc)[MB][NB], const gm_paired<MB> &f, const gm_weights<T::WP, NB> &w, int ks) {
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int a = 0; a < MB; a++) acc[a][b] = T::mfma(f.v[a], w.v[0][b][ks], acc[a][b]);
}

/* Results leave through a descriptor whose size is that of the rows that exist: a row past them is dropped by the range check, with
 * no branch and no address beyond one addition per row (the row is in the vector offset, which the check counts in any case).
 * `at`: byte offset of row 0 of the quad, in the first of NB columns 32 apart. */
template <class T, int NB>
__device__ __forceinline__ void gm_store_quad(__amdgpu_buffer_rsrc_t C, int at, int row_bytes, const f32x4 (&q)[NB], const i32x4 &er, const int (&ec)[NB]) {
#pragma unroll
    for (int v = 0; v < 4; v++)
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const float x = T::SCALED ? __builtin_amdgcn_ldexpf(q[b][v], -ec[b] - er[v]) : q[b][v];
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), C, at + v * row_bytes + 128 * b, 0, 0);
        }
}

/* ---- more than 64 rows ---------------------------------------------------------------------------------
 * A wave owns 80 to 128 rows (gw_shape) x 64 or 96 columns: the weights of its columns are nobody else's among the
 * waves that work on the same K step, so they go from global memory straight into the B operand registers, and
 * only the activation planes pass through the LDS: 8 KB of fragment reads per 16 matrix instructions, half
 * the LDS bandwidth (a 64 x 64 wave tile with both operands in LDS, vt_gemm_mfma_kernel, needs three quarters).
 * One workgroup of four waves per CU (a wave may then use the whole register file of its SIMD: up to 128
 * accumulator registers, 192 with 96 columns, in paired tiles 160 (80 x 256), 224 (112 x 256) and 240 (80 rows, 96 columns); two sets of weight
 * registers, two sets of fragments.  With 96 columns and in the paired tiles all 512 are about used up: 112 x 256 spills 12 and 80 x 384 one,
 * which their times in vt_gemm_plans.h hold), in one of these shapes:
 *   CW = 4: four waves side by side, tiles x 256 (NB = 2 blocks of 32 columns per wave) or x 384 (NB = 3); the planes of one K
 *           step serve four waves.  With 384 columns a fragment read from LDS serves 3 blocks instead of 2: a third less LDS traffic
 *           per matrix instruction, which is time and, under the card's power limit, clock: executed TFLOP/s at 4096 rows of
 *           3072 x 9216 1146 with 128 x 256, 1253 with 128 x 192, 1420 with 128 x 384, of 6144 x 3072 1234 / 1153 / 1346 (96 x 512: 989,
 *           spilled; 64 x 512 1234 and 160 x 384 1159 on a box 5 % slower).  In prefills of 1531 rows, q|k|v / gate|up 101 / 280 -> 87 / 259 us;
 *   CW = 2: two waves side by side and two K steps at a time, tiles x 128 (NB = 2 blocks of 32 columns per wave) or
 *           x 192 (NB = 3); the two halves of K are added through LDS at the end.  For row counts whose 256-column
 *           tiles do not deal out over the CUs, at the price of more plane traffic (L2 and LDS stores) per matrix
 *           instruction: operand bytes per cycle of matrix instructions 32 (128 x 256), 37 (128 x 192), 47 (128 x 128).
 *           With 192 columns a step is half as long again, and the planes of 128 rows are requested one step ahead.
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
 * as every CU can take part in, then the tiles that are left as K cuts, of which a CU gets one or none.  The
 * first requests of an item go out in front of the stores of the one before it.  Only the columns of the cut
 * tiles have more than one partial plane; whoever reads the result is told from which column on (vt_gemm_plan).
 */

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
    const int *row_exp, *col_exp;         /* T::SCALED: exponents of the rows and of the set's columns */
    /* gw_add: */
    int items;
    vt_divisor by_n_tiles;
    gm_cuts cuts;
};
struct gw_list { gw_part part[2]; int n_parts, m_tiles; vt_divisor by_m_tiles; };
static inline void gw_add(gw_list &list, const gw_part &p, int M, int tm, int K) {
    if (!p.n_tiles) return;
    gw_part &q = list.part[list.n_parts++];
    q = p;
    list.m_tiles = (M + tm - 1) / tm;
    q.items = list.m_tiles * p.n_tiles * p.splits;
    list.by_m_tiles = vt_divisor_of(list.m_tiles, q.items > list.part[0].items ? q.items : list.part[0].items);
    q.by_n_tiles = vt_divisor_of(p.n_tiles, p.n_tiles * (long long)p.splits);
    q.cuts = gm_cuts_of(K, p.splits);
}

struct gw_item {
    const unsigned char *w;               /* weights of the tile's first column */
    int part, mt, nt, sp, s0, ns;         /* this cut's K steps: s0 .. s0 + ns - 1 (64 wide) */
};

template <int TN, int WP>
__device__ __forceinline__ gw_item gw_item_at(const gw_list &list, int part, int id, int K) {
    const gw_part &P = list.part[part];
    /* Slot id lands on XCD id % 8.  An XCD takes a run of consecutive items, row tile fastest, then N tile,
     * then K cut: the row tiles of a (K cut, N tile) pair share its weights, the N tiles of a K cut share the
     * activation planes of that cut, and both leave the memory side once per XCD instead of once per workgroup. */
    const int x = id & 7, run = P.items >> 3, rem = P.items & 7;
    const int li = x * run + min(x, rem) + (id >> 3);
    gw_item it;
    it.part = part;
    const int ci = vt_div(li, list.by_m_tiles);
    it.mt = li - ci * list.m_tiles;
    it.sp = vt_div(ci, P.by_n_tiles);
    it.nt = ci - it.sp * P.n_tiles;
    it.ns = P.cuts.steps + (it.sp < P.cuts.longer ? 1 : 0);
    it.s0 = it.sp * P.cuts.steps + min(it.sp, P.cuts.longer);
    it.w = (const unsigned char *)(P.Wf + (size_t)it.nt * TN * K * WP);
    return it;
}

/* A tile's shape.  PAIR false: MB blocks of 32 rows.  PAIR true (WP 1): MB groups of 16, hi and lo plane of a group the 32 rows of one matrix
 * instruction: row counts between, for twice the accumulator registers per row. */
template <int MB, int CW, bool PAIR> struct gw_shape {
    static constexpr int TM = (PAIR ? 16 : 32) * MB;
    static constexpr int NP = (TM + 8 * CW - 1) / (8 * CW);                  /* staging passes over a plane, 8 * CW rows each */
    static constexpr int PLANE = NP * 8 * CW * GM_STAGE_ROW, STAGE = 4 / CW * 2 * PLANE;
};

/* FRAG false: row-major weights (WP 1), a caller's own: the same operands, a lane's 16 bytes of each slice from its own row */
template <class T, int MB, int CW, int NB, bool FRAG = true, bool PAIR = false>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
vt_gemm_wide_kernel(gw_list list, const uint16_t *Ahi, const uint16_t *Alo, int M, int K) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    typedef gw_shape<MB, CW, PAIR> shape;
    constexpr int WP = T::WP, KW = 4 / CW, TM = shape::TM, TN = 32 * NB * CW, NP = shape::NP;
    constexpr int READS = PAIR ? MB : 2 * MB;              /* fragment reads of a slice */
    constexpr int AHEAD = MB * NB > (PAIR ? 14 : 9) ? 1 : 2;       /* steps between the request of a step's planes and their store (registers) */
    /* The first requests of an item go out in front of the stores of the one before it, where registers for both are left (where
     * they were not, a launch's first loads were spilled one by one, each behind a wait: 5 us). */
    constexpr bool EARLY = CW == 4 || MB == 3;
    constexpr int PLANE = shape::PLANE, GROUP = 2 * PLANE, STAGE = shape::STAGE;
    int *tile_exp = reinterpret_cast<int *>(lds + 2 * STAGE);      /* T::SCALED: the exponents of the tile's rows */
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int cw = wave % CW, kw = wave / CW;              /* column block of the tile; which of the KW K steps */
    const int tg = (int)threadIdx.x - kw * 64 * CW;
    const int lr = tg >> 3, lc = tg & 7;                   /* staging: row lr + 8 CW p, 16-byte chunk lc */
    const int a_voff = (lr * K + lc * 8) * 2, a_pass = 16 * CW * K, blk_bytes = 64 * K * WP;
    const int st_off = kw * GROUP + lr * GM_STAGE_ROW + lc * 16;
    const int fa_off = kw * GROUP + (PAIR ? (lane & 15) * GM_STAGE_ROW + (lane >> 4 & 1) * PLANE : (lane & 31) * GM_STAGE_ROW) + (lane >> 5) * 64;

    const int w_voff = FRAG ? lane * 16 : (lane & 31) * K * 2 + (lane >> 5) * 64;

    struct aregs { u32x4 hi[NP], lo[NP]; };                /* staged rows of one K step, both planes */
    /* rows past M and steps past the cut's end: beyond the descriptor's size, nothing is loaded (zeros) */
    auto fetch_a = [&](const gw_item &it, const uint16_t *plane, u32x4 (&r)[NP], int i) {
        const int s = KW * i + kw, rows = min(M - it.mt * TM, TM);
        const bool live = s < it.ns;
        const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc((void *)(plane + (size_t)it.mt * TM * K), 0, live ? rows * K * 2 : 0, 0x00020000);
        const int soff = live ? (it.s0 + s) * 128 : 0;
#pragma unroll
        for (int p = 0; p < NP; p++) r[p] = gm_ldb(d, a_voff + p * a_pass, soff);
    };
    auto fetch_b_slice = [&](const gw_item &it, gm_weights<WP, NB> &r, int i, int j) {
        const int s = KW * i + kw;
        const bool live = s < it.ns;
        const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc((void *)(it.w + (size_t)cw * NB * blk_bytes), 0, live ? NB * blk_bytes : 0, 0x00020000);
        const int soff = live ? (it.s0 + s) * (FRAG ? 4096 * WP : 128) : 0;
#pragma unroll
        for (int p = 0; p < WP; p++)
#pragma unroll
            for (int b = 0; b < NB; b++) r.v[p][b][j] = gm_ldb(d, w_voff + (FRAG ? 1024 : 16) * j, soff + 4096 * p + (live ? b * blk_bytes : 0));
    };
    auto store_a = [&](const u32x4 (&r)[NP], int at) {
#pragma unroll
        for (int p = 0; p < NP; p++) *reinterpret_cast<u32x4 *>(lds + at + st_off + 8 * CW * p * GM_STAGE_ROW) = r[p];
    };
    typedef typename std::conditional<PAIR, gm_paired<MB>, gm_frags<MB>>::type frags;
    auto read_frags = [&](frags &f, int stage, int ks) {
        const unsigned char *base = lds + stage * STAGE + fa_off + ks * 16;
#pragma unroll
        for (int a = 0; a < MB; a++) {
            if constexpr (PAIR) {
                f.v[a] = *reinterpret_cast<const u32x4 *>(base + 16 * a * GM_STAGE_ROW);
            } else {
                f.hi[a] = *reinterpret_cast<const u32x4 *>(base + 32 * a * GM_STAGE_ROW);
                f.lo[a] = *reinterpret_cast<const u32x4 *>(base + PLANE + 32 * a * GM_STAGE_ROW);
            }
        }
    };
    f32x16 acc[MB][NB];
    auto mma = [&](const frags &f, const gm_weights<WP, NB> &w, int ks) { gm_multiply<T, MB, NB>(acc, f, w, ks); };

    /* One step: stage `stage` holds the planes of step i and `cur` its weights; ra holds the planes of step
     * i + 1 (requested two steps ago: with one step between request and store, the step takes as long as a load,
     * 1.2 us, whatever the tile); f0 already holds the fragments of slice 0.  Four regions of 2 MB NB (PAIR: MB NB; 3 MB NB with
     * two weight planes) matrix instructions each; the other instructions of a region (the fragment reads of the next slice, in the first
     * two also the LDS stores of a plane of step i + 1 and its requests of step i + 3, in all but the first the
     * weight requests that refill the slice just used) are dealt out between the matrix instructions, one
     * after every second or third, so that the matrix pipe never waits for a block of them to issue.  The step's one
     * barrier stands in front of the last region: by then every wave has issued (and waited for) its stores
     * into the other stage and its last reads of this one, so the first fragments of step i + 1 are read under
     * the last matrix instructions of step i. */
    gm_weights<WP, NB> b0, b1;
    aregs ra0, ra1;                       /* the rows of even and of odd steps (AHEAD 1: ra0 of all) */
    frags f0, f1;
#define GW_FENCE() __builtin_amdgcn_sched_barrier(0)
#define GW_MFMA() __builtin_amdgcn_sched_group_barrier(0x008, NB * (1 + WP) / 2, 0)
#define GW_DSR1() __builtin_amdgcn_sched_group_barrier(0x100, 1, 0)
#define GW_DSW1() __builtin_amdgcn_sched_group_barrier(0x200, 1, 0)
#define GW_VMR1() __builtin_amdgcn_sched_group_barrier(0x020, 1, 0)
    auto step = [&](const gw_item &it, int i, int stage, gm_weights<WP, NB> &cur, aregs &ra) {
        const int other = (stage ^ 1) * STAGE;
        GW_FENCE();
        store_a(ra.hi, other);
        fetch_a(it, Ahi, ra.hi, i + 1 + AHEAD);
        read_frags(f1, stage, 1);
        mma(f0, cur, 0);
#pragma unroll
        for (int k = 0; k < READS; k++) { GW_MFMA(); GW_DSR1(); if (k < NP) { GW_DSW1(); GW_VMR1(); } }
        GW_FENCE();
        store_a(ra.lo, other + PLANE);
        fetch_a(it, Alo, ra.lo, i + 1 + AHEAD);
        fetch_b_slice(it, cur, i + 2, 0);
        read_frags(f0, stage, 2);
        mma(f1, cur, 1);
#pragma unroll
        for (int k = 0; k < READS; k++) { GW_MFMA(); GW_DSR1(); if (k < NP) { GW_DSW1(); GW_VMR1(); } if (k < NB * WP) GW_VMR1(); }
        GW_FENCE();
        fetch_b_slice(it, cur, i + 2, 1);
        read_frags(f1, stage, 3);
        mma(f0, cur, 2);
#pragma unroll
        for (int k = 0; k < READS; k++) { GW_MFMA(); GW_DSR1(); if (k < NB * WP) GW_VMR1(); }
        GW_FENCE();
        __syncthreads();
        GW_FENCE();
        fetch_b_slice(it, cur, i + 2, 2);
        read_frags(f0, stage ^ 1, 0);
        mma(f1, cur, 3);
#pragma unroll
        for (int k = 0; k < READS; k++) { GW_MFMA(); GW_DSR1(); if (k < NB * WP) GW_VMR1(); }
        GW_FENCE();
        fetch_b_slice(it, cur, i + 2, 3);
    };
    /* The first requests of an item: T::SCALED: the exponents of its rows and of this lane's columns; the planes and weights of steps 0
     * and 1.  (The exponents asked for where the sums are stored, four rows at a time, each behind the stores before it, took 4.6 us of a
     * 12 us launch at 84 rows, and 10 of an item's 40 us at 1696.) */
    int next_row_exp = 0, next_ec[NB] = {}, ec[NB];
    auto begin = [&](const gw_item &it) {
        if constexpr (T::SCALED) {
            const gw_part &P = list.part[it.part];
            const int rows = min(M - it.mt * TM, TM);
            next_row_exp = __builtin_amdgcn_raw_buffer_load_b32(__builtin_amdgcn_make_buffer_rsrc((void *)(P.row_exp + it.mt * TM), 0, rows * 4, 0x00020000), (int)threadIdx.x * 4, 0, 0);
            const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc((void *)(P.col_exp + it.nt * TN), 0, TN * 4, 0x00020000);
#pragma unroll
            for (int b = 0; b < NB; b++) next_ec[b] = __builtin_amdgcn_raw_buffer_load_b32(d, (32 * (NB * cw + b) + (lane & 31)) * 4, 0, 0);
        }
        fetch_a(it, Ahi, ra0.hi, 0);
        fetch_a(it, Alo, ra0.lo, 0);
#pragma unroll
        for (int j = 0; j < 4; j++) fetch_b_slice(it, b0, 0, j);
        if constexpr (AHEAD == 2) {
            fetch_a(it, Ahi, ra1.hi, 1);
            fetch_a(it, Alo, ra1.lo, 1);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) fetch_b_slice(it, b1, 1, j);
        GW_FENCE();
    };
    auto multiply = [&](const gw_item &it) {
#pragma unroll
        for (int a = 0; a < MB; a++)
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[a][b][v] = 0.f;
        if constexpr (T::SCALED) {
            if ((int)threadIdx.x < TM) tile_exp[threadIdx.x] = next_row_exp;
#pragma unroll
            for (int b = 0; b < NB; b++) ec[b] = next_ec[b];
        }
        store_a(ra0.hi, 0);
        store_a(ra0.lo, PLANE);
        fetch_a(it, Ahi, ra0.hi, AHEAD);
        fetch_a(it, Alo, ra0.lo, AHEAD);
        GW_FENCE();
        __syncthreads();
        read_frags(f0, 0, 0);
        const int n = (it.ns + KW - 1) / KW;
        aregs &odd = AHEAD == 2 ? ra1 : ra0;
        int i = 0;
        for (; i + 1 < n; i += 2) {
            step(it, i, 0, b0, odd);
            step(it, i + 1, 1, b1, ra0);
        }
        if (i < n) step(it, i, 0, b0, odd);
    };
#undef GW_MFMA
#undef GW_DSR1
#undef GW_DSW1
#undef GW_VMR1
#undef GW_FENCE

    /* accumulator element v of lane l: row 8*(v/4) + 4*(l/32) + v%4, column l%32; quads (a, vq) hold v = 4 vq .. + 3 */
    auto emit = [&](const gw_part &P, const gw_item &it, int lane, int a, int vq, const f32x4 (&q)[NB]) {
        const int quad_row = (PAIR ? 16 : 32) * a + 8 * vq, rows = min(M - it.mt * TM, TM), c = lane & 31;      /* of the tile; a lane's first one is 4 (l / 32) on */
        if constexpr (!T::SCALED) {
            if (P.h_hi) {
                /* a column block holds the gates and the ups of 16 h columns (voxtral_tts_llm.c:346-350) */
                float g[2 * NB], u[2 * NB], h[2 * NB];
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    float g2[2], u2[2];
                    vt_pair_rows(q[b], g2, u2);
                    g[2 * b] = g2[0]; g[2 * b + 1] = g2[1]; u[2 * b] = u2[0]; u[2 * b + 1] = u2[1];
                }
                vt_silu_mul<2 * NB>(h, g, u);
                const size_t tile = (size_t)it.mt * TM * P.ldh;
                const __amdgpu_buffer_rsrc_t d_hi = __builtin_amdgcn_make_buffer_rsrc(P.h_hi + tile, 0, rows * P.ldh * 2, 0x00020000);
                const __amdgpu_buffer_rsrc_t d_lo = __builtin_amdgcn_make_buffer_rsrc(P.h_lo + tile, 0, rows * P.ldh * 2, 0x00020000);
                const int at = ((4 * (lane >> 5) + 2 * (lane >> 4 & 1) + (lane & 1)) * P.ldh + it.nt * (TN / 2) + 16 * NB * cw + (lane & 14)) * 2 + quad_row * P.ldh * 2;
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    unsigned hi, lo;
                    vt_pair_words(h[2 * b], h[2 * b + 1], hi, lo);
                    __builtin_amdgcn_raw_buffer_store_b32(hi, d_hi, at + 32 * b, 0, 0);
                    __builtin_amdgcn_raw_buffer_store_b32(lo, d_lo, at + 32 * b, 0, 0);
                }
                return;
            }
        }
        const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc(P.C + (size_t)it.sp * P.plane_stride + (size_t)it.mt * TM * P.ldc, 0, rows * P.ldc * 4, 0x00020000);
        const int at = 4 * (lane >> 5) * P.ldc * 4 + (it.nt * TN + 32 * NB * cw + c) * 4 + quad_row * P.ldc * 4;
        i32x4 er = {};
        if constexpr (T::SCALED) er = *reinterpret_cast<const i32x4 *>(tile_exp + quad_row + 4 * (lane >> 5));
        gm_store_quad<T, NB>(d, at, P.ldc * 4, q, er, ec);
    };
    constexpr int QUADS = PAIR ? 2 : 4, HALF = QUADS / 2;        /* quads per a; PAIR: elements 8 + v are row v's sums over the lo plane */
    auto quads = [&](f32x4 (&q)[NB], int a, int vq) {
#pragma unroll
        for (int b = 0; b < NB; b++) {
            q[b] = f32x4{acc[a][b][4 * vq], acc[a][b][4 * vq + 1], acc[a][b][4 * vq + 2], acc[a][b][4 * vq + 3]};
            if constexpr (PAIR) {
#pragma unroll
                for (int v = 0; v < 4; v++) q[b][v] = __fadd_rn(q[b][v], acc[a][b][8 + 4 * vq + v]);
            }
        }
    };
    auto finish = [&](const gw_item &it) {
        const gw_part &P = list.part[it.part];
        const int lane = vt_lane();       /* offsets are made here, not kept through the steps (16 of them were spilled) */
        f32x4 q[NB];
        if constexpr (KW == 1) {
#pragma unroll
            for (int a = 0; a < MB; a++)
#pragma unroll
                for (int vq = 0; vq < QUADS; vq++) { quads(q, a, vq); emit(P, it, lane, a, vq, q); }
        } else {
            /* the two waves of a column block hold the sums over the even and the odd K steps: each parks the half
             * of its quads that the other one finishes */
            float *park = reinterpret_cast<float *>(lds) + (size_t)wave * (MB * NB * HALF * 256);
            const float *theirs = reinterpret_cast<const float *>(lds) + (size_t)(wave ^ CW) * (MB * NB * HALF * 256);
            __syncthreads();
#pragma unroll
            for (int a = 0; a < MB; a++)
#pragma unroll
                for (int h = 0; h < HALF; h++) {
                    if (kw == 0) quads(q, a, HALF + h); else quads(q, a, h);
#pragma unroll
                    for (int b = 0; b < NB; b++) *reinterpret_cast<f32x4 *>(park + (((a * HALF + h) * NB + b) * 64 + lane) * 4) = q[b];
                }
            __syncthreads();
#pragma unroll
            for (int a = 0; a < MB; a++)
#pragma unroll
                for (int h = 0; h < HALF; h++) {
                    if (kw == 0) quads(q, a, h); else quads(q, a, HALF + h);
#pragma unroll
                    for (int b = 0; b < NB; b++) {
                        const f32x4 o = *reinterpret_cast<const f32x4 *>(theirs + (((a * HALF + h) * NB + b) * 64 + lane) * 4), m = q[b];
                        q[b] = f32x4{__fadd_rn(m.x, o.x), __fadd_rn(m.y, o.y), __fadd_rn(m.z, o.z), __fadd_rn(m.w, o.w)};
                    }
                    emit(P, it, lane, a, kw == 0 ? h : HALF + h, q);
                }
        }
    };

    /* (one copy of the code that finishes an item: where it runs once, it comes from memory, and so do its instructions) */
    int part = 0, id = (int)blockIdx.x;
    gw_item it = gw_item_at<TN, WP>(list, 0, id, K);
    if constexpr (EARLY) begin(it);
    for (;;) {
        if constexpr (!EARLY) begin(it);
        multiply(it);
        id += (int)gridDim.x;
        while (part < list.n_parts && id >= list.part[part].items) {
            part++;
            id = (int)blockIdx.x;
        }
        const bool more = part < list.n_parts;
        gw_item nx = it;
        if (more) {
            nx = gw_item_at<TN, WP>(list, part, id, K);
            if constexpr (EARLY) begin(nx);
        }
        finish(it);
        if (!more) break;
        __syncthreads();                  /* the next item stages over what this one read */
        it = nx;
    }
}


/* ---- up to 64 rows (the codec's first stages) ---------------------------------------------------------------
 * With so few rows the product is a weight stream, and what counts is that every CU has a share of it, and an equal one.  A
 * workgroup owns 64 columns and
 * its waves share K among themselves: wave w takes the 64-wide K steps w, w + NW, ... of the workgroup's range,
 * keeps its own sums for all rows, and the waves' sums are added through LDS at the end (in wave order: the
 * result does not depend on timing).
 *
 * No two waves work on the same K step, so nobody shares anything before the end: a wave stages its own
 * activation rows through its own piece of LDS (one stage; the LDS serves a wave's accesses in order, so the
 * rows of the next step are written over those of this one behind its last reads) and there is no barrier in
 * the K loop.  The weights of a step go straight into the B operand registers, two steps ahead.  Every request
 * goes through a buffer descriptor whose size says whether there is anything to load: steps past a wave's last
 * one and rows past M ask for nothing, without a branch (behind a branch the compiler would wait for all
 * outstanding loads).
 */
struct gr_list {
    float *C;                             /* cuts.n planes of [M, ldc], plane_stride floats apart */
    const uint16_t *Wf;                   /* fragment-order weights */
    size_t plane_stride;
    int ldc, items;
    vt_divisor n_tiles;
    gm_cuts cuts;
    const int *row_exp, *col_exp;         /* T::SCALED: exponents of the rows and of the columns */
};

/* non-temporal: with this few rows the weights are read once */
__device__ __forceinline__ u32x4 gr_ld_nt(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 2);
}

/* One workgroup's piece of a product: a 64-column tile over one K cut */
struct gr_item {
    const unsigned char *w;               /* weights of the tile */
    int nt, sp, s0, n;                    /* n: this wave's K steps s0 + wave + NW i */
};

template <int NW, int WP>
__device__ __forceinline__ gr_item gr_item_at(const gr_list &P, int id, int K, int wave) {
    /* slot id lands on XCD id % 8: an XCD takes a run of items, N tile fastest, i.e. few K cuts: the slice of
     * the planes that its L2 has to fetch is that of its cuts */
    const int li = (P.items & 7) == 0 ? (id & 7) * (P.items >> 3) + (id >> 3) : id;
    gr_item it;
    it.sp = vt_div(li, P.n_tiles);
    it.nt = li - it.sp * P.n_tiles.d;
    const int ns = P.cuts.steps + (it.sp < P.cuts.longer ? 1 : 0);
    it.s0 = it.sp * P.cuts.steps + min(it.sp, P.cuts.longer);
    it.n = ns > wave ? (ns - wave + NW - 1) / NW : 0;
    it.w = (const unsigned char *)(P.Wf + (size_t)it.nt * GR_TN * K * WP);
    return it;
}

/* NP passes of 8 rows: M <= 8 NP; NW waves */
template <class T, int NP, int NW>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW / 4, NW / 4)))
vt_gemm_rows_kernel(gr_list P, const uint16_t *Ahi, const uint16_t *Alo, int M, int K) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    constexpr int WP = T::WP;
    constexpr int MB = (NP + 3) / 4;                                         /* blocks of 32 rows */
    constexpr int PLANE = 32 * MB * GM_STAGE_ROW;
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int blk_bytes = 64 * K * WP;                                       /* 32 columns x K x 2 bytes x planes */
    const int a_bytes = M * K * 2;
    unsigned char *mine = lds + wave * (2 * PLANE);
    const int lr = lane >> 3, lc = lane & 7;                                 /* staging: row lr + 8 p, 16-byte chunk lc */
    const int a_voff = (lr * K + lc * 8) * 2, a_pass = 16 * K;               /* byte distance of two passes */
    const int st_off = lr * GM_STAGE_ROW + lc * 16;
    const int fa_off = (lane & 31) * GM_STAGE_ROW + (lane >> 5) * 64;

    u32x4 ra_hi[NP], ra_lo[NP];
    auto fetch_a = [&](const gr_item &it, int i) {
        const int soff = i < it.n ? (it.s0 + wave + NW * i) * 128 : 0;
        const __amdgpu_buffer_rsrc_t h = __builtin_amdgcn_make_buffer_rsrc((void *)Ahi, 0, i < it.n ? a_bytes : 0, 0x00020000);
        const __amdgpu_buffer_rsrc_t l = __builtin_amdgcn_make_buffer_rsrc((void *)Alo, 0, i < it.n ? a_bytes : 0, 0x00020000);
#pragma unroll
        for (int p = 0; p < NP; p++) {
            ra_hi[p] = gm_ldb(h, a_voff + p * a_pass, soff);
            ra_lo[p] = gm_ldb(l, a_voff + p * a_pass, soff);
        }
    };
    auto fetch_b_slice = [&](const gr_item &it, gm_weights<WP, 2> &r, int i, int j) {
        const int soff = i < it.n ? (it.s0 + wave + NW * i) * 4096 * WP : 0;
        const __amdgpu_buffer_rsrc_t w = __builtin_amdgcn_make_buffer_rsrc((void *)it.w, 0, i < it.n ? 2 * blk_bytes : 0, 0x00020000);
#pragma unroll
        for (int p = 0; p < WP; p++) {
            r.v[p][0][j] = gr_ld_nt(w, lane * 16 + 1024 * j, soff + 4096 * p);
            r.v[p][1][j] = gr_ld_nt(w, lane * 16 + 1024 * j, soff + 4096 * p + (i < it.n ? blk_bytes : 0));
        }
    };
    auto store_a = [&]() {
#pragma unroll
        for (int p = 0; p < NP; p++) {
            *reinterpret_cast<u32x4 *>(mine + st_off + 8 * p * GM_STAGE_ROW) = ra_hi[p];
            *reinterpret_cast<u32x4 *>(mine + PLANE + st_off + 8 * p * GM_STAGE_ROW) = ra_lo[p];
        }
    };
    typedef gm_frags<MB> frags;
    auto read_frags = [&](frags &f, int ks) {
#pragma unroll
        for (int a = 0; a < MB; a++) {
            f.hi[a] = *reinterpret_cast<const u32x4 *>(mine + fa_off + 32 * a * GM_STAGE_ROW + 16 * ks);
            f.lo[a] = *reinterpret_cast<const u32x4 *>(mine + PLANE + fa_off + 32 * a * GM_STAGE_ROW + 16 * ks);
        }
    };
    f32x16 acc[MB][2];
    auto mma = [&](const frags &f, const gm_weights<WP, 2> &w, int ks) { gm_multiply<T, MB, 2>(acc, f, w, ks); };
    gm_weights<WP, 2> b0, b1;
    frags f0, f1;
    /* wave w finishes the quads w, w + NW, ...: rows 8 q + 4 (lane / 32) + 0..3, column lane % 32 of both blocks; T::SCALED: their exponents */
    constexpr int NQ = (NP + NW - 1) / NW;
    i32x4 er[NQ] = {};
    int next_ec[2] = {}, ec[2];
    if constexpr (T::SCALED) {
        const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc((void *)P.row_exp, 0, M * 4, 0x00020000);
#pragma unroll
        for (int i = 0; i < NQ; i++) er[i] = __builtin_bit_cast(i32x4, gm_ldb(d, (8 * (wave + NW * i) + 4 * (lane >> 5)) * 4, 0));
    }
    /* the first requests of an item: the exponents of its columns, the rows of step 0, the weights of steps 0 and 1 */
    auto begin = [&](const gr_item &it) {
        if constexpr (T::SCALED) {
            const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc((void *)(P.col_exp + it.nt * GR_TN), 0, GR_TN * 4, 0x00020000);
#pragma unroll
            for (int b = 0; b < 2; b++) next_ec[b] = __builtin_amdgcn_raw_buffer_load_b32(d, (32 * b + (lane & 31)) * 4, 0, 0);
        }
        fetch_a(it, 0);
#pragma unroll
        for (int j = 0; j < 4; j++) fetch_b_slice(it, b0, 0, j);
#pragma unroll
        for (int j = 0; j < 4; j++) fetch_b_slice(it, b1, 1, j);
        __builtin_amdgcn_sched_barrier(0);
    };
    /* step i: the stage holds its rows, f0 their slice 0; ra holds the rows of step i + 1.  A slice's weight
     * registers are requested again (step i + 2) as soon as the slice has been multiplied. */
    auto step = [&](const gr_item &it, int i, gm_weights<WP, 2> &cur) {
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
#pragma unroll
        for (int b = 0; b < 2; b++) ec[b] = next_ec[b];
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
        const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc(P.C + (size_t)it.sp * P.plane_stride, 0, M * P.ldc * 4, 0x00020000);
#pragma unroll
        for (int i = 0; i < NQ; i++) {
            const int qd = wave + NW * i;
            if (qd >= NP) break;
            f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int w = 0; w < NW; w++)
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    const f32x4 v = *reinterpret_cast<const f32x4 *>(lds + w * (2 * PLANE) + ((qd * 2 + b) * 64 + lane) * 16);
                    s[b].x = __fadd_rn(s[b].x, v.x); s[b].y = __fadd_rn(s[b].y, v.y);
                    s[b].z = __fadd_rn(s[b].z, v.z); s[b].w = __fadd_rn(s[b].w, v.w);
                }
            gm_store_quad<T, 2>(d, (8 * qd + 4 * (lane >> 5)) * P.ldc * 4 + (it.nt * GR_TN + (lane & 31)) * 4, P.ldc * 4, s, er[i], ec);
        }
    };

    /* items blockIdx.x, + gridDim.x, ...; the first requests of the next item go out in front of the sums of this one */
    int id = (int)blockIdx.x;
    gr_item it = gr_item_at<NW, WP>(P, id, K, wave);
    begin(it);
    for (;;) {
        multiply(it);
        id += (int)gridDim.x;
        if (id >= P.items) break;
        const gr_item nx = gr_item_at<NW, WP>(P, id, K, wave);
        begin(nx);
        finish(it);
        __syncthreads();                  /* the next item stages over the parked sums */
        it = nx;
    }
    finish(it);
}


#endif /* VT_GEMM_TILES_H */

/*
 * vt_gemm.hip - bf16 MFMA matrix product for rows of activations (seq_len > 1):
 * C[M,N] = X[M,K] * W[N,K]^T with fp32 accumulation, the sequence-level linear
 * of the CPU path (tts_linear_nobias_bf16 with seq_len > 1,
 * voxtral_tts_kernels.c:187-198, and the triple loop it falls to, :127-138).
 *
 * Weights are bf16 already.  The fp32 activations are carried as two bf16
 * planes, hi = bf16(x) and lo = bf16(x - hi), so that hi + lo represents x to
 * about 2^-17 relative; every weight tile is multiplied with both planes
 * (two MFMAs per tile pair) and the sums land in the same fp32 accumulator.
 * That keeps the result within a few fp32 ulps of the sequential CPU sum while
 * all products run on the matrix cores.
 *
 * Tiling: workgroup tile 128 x 128, K step 64, four waves in a 2 x 2 grid of
 * 64 x 64 wave tiles, v_mfma_f32_32x32x16_bf16.  Tiles are staged through LDS
 * with a row pitch of 144 bytes (128 of data + 16 of padding): the 16 lanes of
 * a 16-byte fragment read then cover all 64 banks once.  One LDS stage; the
 * next K step is fetched into registers while the current one is multiplied,
 * the fragments of the next 16-wide slice are read while the current slice is
 * multiplied, and two workgroups share a CU.  Workgroups that need the same weight tile
 * (the M tiles of one N tile) get consecutive slots on one XCD, so the tile is
 * fetched from HBM once and served from that XCD's L2 afterwards.  Long K can
 * be cut into `splits` ranges that write separate partial planes; the caller
 * adds them in a fixed order (vt_residual_norm_split_kernel).
 */
#include "vt_state.h"
#include "vt_gemm.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(1))) const u32x4 vt_gptr_u32x4;

#define GM_TILE 128
#define GM_BK   64
#define GM_ROWB 144
#define GM_MAT  (GM_TILE * GM_ROWB)

__device__ __forceinline__ u32x4 gm_ld(const uint16_t *p) { return *(vt_gptr_u32x4 *)p; }
__device__ __forceinline__ bf16x8 gm_frag(const unsigned char *p) {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(p));
}

__global__ void __launch_bounds__(256, 2)
vt_gemm_mfma_kernel(float *C, const uint16_t *Ahi, const uint16_t *Alo, const uint16_t *W,
                    int M, int N, int K, int k_split, int m_tiles, int n_tiles, int ldc, size_t plane_stride) {
    __shared__ __attribute__((aligned(16))) unsigned char lds[3 * GM_MAT];
    const int id = (int)blockIdx.x;
    int mt, nt, sp;
    if ((n_tiles & 7) == 0) {
        /* slot id lands on XCD id % 8: keep the M tiles of one N tile there */
        const int x = id & 7, q = id >> 3, r = q / m_tiles, npx = n_tiles >> 3;
        mt = q % m_tiles;
        nt = (r % npx) * 8 + x;
        sp = r / npx;
    } else {
        const int r = id / m_tiles;
        mt = id % m_tiles;
        nt = r % n_tiles;
        sp = r / n_tiles;
    }
    const int t = (int)threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int lr = t >> 3, lc = t & 7;               /* staging: row lr + 32 i, 16-byte chunk lc */
    const int k0 = sp * k_split, tiles = k_split / GM_BK;

    const uint16_t *pa[4], *pl[4], *pw[4];
    bool live[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int gm = mt * GM_TILE + lr + 32 * i;
        live[i] = gm < M;
        const size_t ao = (size_t)(live[i] ? gm : 0) * K + k0 + lc * 8;
        pa[i] = Ahi + ao;
        pl[i] = Alo + ao;
        pw[i] = W + (size_t)(nt * GM_TILE + lr + 32 * i) * K + k0 + lc * 8;
    }

    /* the next K step is fetched into registers while the current one is multiplied */
    u32x4 ra[4], rl[4], rb[4];
    const u32x4 zero = {0u, 0u, 0u, 0u};
    auto fetch = [&](int kt) {
        const int adv = kt * GM_BK;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            ra[i] = live[i] ? gm_ld(pa[i] + adv) : zero;
            rl[i] = live[i] ? gm_ld(pl[i] + adv) : zero;
            rb[i] = gm_ld(pw[i] + adv);
        }
    };
    fetch(0);

    f32x16 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[a][b][v] = 0.f;

    const int st_off = lr * GM_ROWB + lc * 16;
    const int fa_off = (64 * wm + (lane & 31)) * GM_ROWB + (lane >> 5) * 16;
    const int fb_off = (64 * wn + (lane & 31)) * GM_ROWB + (lane >> 5) * 16 + 2 * GM_MAT;

    /* fragments of one 16-wide slice: hi, lo of two row blocks and the weights of two column blocks */
    struct frags { bf16x8 fa[2], fl[2], fb[2]; };
    auto read_frags = [&](frags &f, int ks) {
#pragma unroll
        for (int b = 0; b < 2; b++) {
            f.fa[b] = gm_frag(lds + fa_off + 32 * b * GM_ROWB + ks * 32);
            f.fl[b] = gm_frag(lds + GM_MAT + fa_off + 32 * b * GM_ROWB + ks * 32);
            f.fb[b] = gm_frag(lds + fb_off + 32 * b * GM_ROWB + ks * 32);
        }
    };
    auto mma = [&](const frags &f) {
        /* four independent accumulators between two products into the same one */
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int b = 0; b < 2; b++)
                acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.fl[a], f.fb[b], acc[a][b], 0, 0, 0);
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int b = 0; b < 2; b++)
                acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.fa[a], f.fb[b], acc[a][b], 0, 0, 0);
    };

    for (int kt = 0; kt < tiles; kt++) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; i++) {
            *reinterpret_cast<u32x4 *>(lds + st_off + 32 * i * GM_ROWB) = ra[i];
            *reinterpret_cast<u32x4 *>(lds + GM_MAT + st_off + 32 * i * GM_ROWB) = rl[i];
            *reinterpret_cast<u32x4 *>(lds + 2 * GM_MAT + st_off + 32 * i * GM_ROWB) = rb[i];
        }
        __syncthreads();
        if (kt + 1 < tiles) fetch(kt + 1);
        /* the fragments of slice ks+1 are read while slice ks is multiplied */
        frags f0, f1;
        read_frags(f0, 0);
        read_frags(f1, 1);
        mma(f0);
        read_frags(f0, 2);
        mma(f1);
        read_frags(f1, 3);
        mma(f0);
        mma(f1);
    }

    /* accumulator element v of lane l: row 8*(v/4) + 4*(l/32) + v%4, column l%32 */
    float *Cs = C + (size_t)sp * plane_stride;
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const int col = nt * GM_TILE + 64 * wn + 32 * b + (lane & 31);
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int row = mt * GM_TILE + 64 * wm + 32 * a + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                if (row < M) Cs[(size_t)row * ldc + col] = acc[a][b][v];
            }
        }
}

static int gm_blocks(size_t n);

/* Row-major W[N, K] (N % 32 == 0, K % 64 == 0) -> fragment order: the 16 bytes that lane l = 32 g + n % 32
 * feeds to slice j of K step ks of column block nb = n / 32, i.e. W[n][64 ks + 32 g + 8 j .. + 8], go to
 * 16-byte slot ((nb * K/64 + ks) * 4 + j) * 64 + l.  A block of 32 rows occupies the same 32 K elements
 * in both layouts. */
/* pair: W is a gate|up matrix with (gate, up) rows interleaved; fragment column n' of every 32 takes row
 * 32 (n'/32) + 2 (n' % 16) + (n' % 32) / 16, so that a column block of the product holds 16 gates and their ups, and a wave any number of blocks. */
__global__ void vt_frag_layout_kernel(u32x4 *out, const uint16_t *W, size_t n_slots, int K, int pair) {
    const int ksteps = K / GM_BK;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_slots; i += (size_t)gridDim.x * blockDim.x) {
        const int l = (int)(i & 63), j = (int)((i >> 6) & 3);
        const size_t blk = i >> 8;
        const int ks = (int)(blk % ksteps);
        const size_t nb = blk / ksteps;
        size_t n = nb * 32 + (l & 31);
        if (pair) n = nb * 32 + 2 * (l & 15) + (l >> 4 & 1);
        out[i] = gm_ld(W + n * K + 64 * ks + 32 * (l >> 5) + 8 * j);
    }
}

void vt_launch_frag_layout(uint16_t *d_Wf, const uint16_t *d_W, int N, int K, int pair) {
    const size_t n_slots = (size_t)N * K / 8;
    hipLaunchKernelGGL(vt_frag_layout_kernel, dim3(gm_blocks(n_slots)), dim3(256), 0, g_vt.stream, (u32x4 *)d_Wf, d_W,
                       n_slots, K, pair);
}

int vt_gemm_shape_ok(int M, int N, int K, int splits) {
    return M >= 1 && splits >= 1 && N % GM_TILE == 0 && K % splits == 0 && (K / splits) % GM_BK == 0;
}

void vt_launch_gemm_ex(float *d_C, int ldc, size_t plane_stride, const uint16_t *d_Ahi, const uint16_t *d_Alo,
                       const uint16_t *d_W, int M, int N, int K, int splits) {
    const int m_tiles = (M + GM_TILE - 1) / GM_TILE, n_tiles = N / GM_TILE;
    hipLaunchKernelGGL(vt_gemm_mfma_kernel, dim3(m_tiles * n_tiles * splits), dim3(256), 0, g_vt.stream,
                       d_C, d_Ahi, d_Alo, d_W, M, N, K, K / splits, m_tiles, n_tiles, ldc, plane_stride);
}

void vt_launch_gemm(float *d_C, const uint16_t *d_Ahi, const uint16_t *d_Alo, const uint16_t *d_W,
                    int M, int N, int K, int splits) {
    vt_launch_gemm_ex(d_C, N, (size_t)M * N, d_Ahi, d_Alo, d_W, M, N, K, splits);
}

/* ---- fp32 -> (hi, lo) bf16 planes ---------------------------------------------- */

__global__ void vt_split_kernel(uint16_t *hi, uint16_t *lo, const float *x, size_t n2) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n2;
         i += (size_t)gridDim.x * blockDim.x) {
        const f32x2 v = reinterpret_cast<const f32x2 *>(x)[i];
        unsigned h, l;
        vt_split_planes2(v.x, v.y, h, l);
        reinterpret_cast<unsigned *>(hi)[i] = h;
        reinterpret_cast<unsigned *>(lo)[i] = l;
    }
}

static int gm_blocks(size_t n) { size_t b = (n + 255) / 256; return (int)(b > 8192 ? 8192 : b); }

void vt_launch_split(uint16_t *d_hi, uint16_t *d_lo, const float *d_x, size_t n) {
    hipLaunchKernelGGL(vt_split_kernel, dim3(gm_blocks(n / 2)), dim3(256), 0, g_vt.stream, d_hi, d_lo, d_x, n / 2);
}

/* CALL(P) with P = planes, 1 .. VT_MAX_CUTS */
#define GM_BY_PLANES(planes, CALL) do { switch (planes) { case 1: CALL(1); break; case 2: CALL(2); break; case 3: CALL(3); break; \
    case 4: CALL(4); break; case 5: CALL(5); break; case 6: CALL(6); break; case 7: CALL(7); break; default: CALL(8); } } while (0)
static_assert(VT_MAX_CUTS == 8, "GM_BY_PLANES");

/* One workgroup per row of 3072 floats (256 threads x 12):
 *   x[row] += part[0][row] (+ part[1][row] + ... for the columns from col0 on)   (C > 0 cuts; fixed order)
 *   (hi, lo)[row] = split(rmsnorm(x[row]) * w)                                   (w != NULL)
 * x before the sum comes from x_in: x itself or, for a prefill's input rows, host memory.
 * The residual add and the normalisation of voxtral_tts_llm.c:332-336,354 /
 * :338-341 in one pass over the row.  Up to a few hundred rows a launch is one chain of memory latencies per
 * workgroup, so everything is requested in front of the first sum;
 * with the planes in a loop that waited for each of them a launch took 8.5 us at 226 rows and takes 6.0 to 6.6 now; us per
 * prefill of 37 / 226 / 512 / 1531 rows 2632 / 4414 / 7236 / 20457 -> 2481 / 4326 / 7186 / 20181, results the same. */
template <int C>
__global__ void __launch_bounds__(256)
vt_residual_norm_split_kernel(float *x, const float *x_in, const float *part, int col0, size_t part_stride,
                              const float *w, uint16_t *hi, uint16_t *lo, float eps) {
    /* a thread owns 4 consecutive columns at 4 (t + 256 j): 16-byte loads and stores, 8-byte plane
     * stores (a quarter of the memory instructions of element-wise accesses) */
    __shared__ float red[4];
    const size_t row = blockIdx.x;
    constexpr int NJ = VT_DIM / 1024;
    const __amdgpu_buffer_rsrc_t dx = vt_buffer(x + row * VT_DIM, VT_DIM * 4);
    const int at = 16 * (int)threadIdx.x;
    f32x4 v[NJ], g[NJ], p[NJ][C > 0 ? C : 1];
#pragma unroll
    for (int j = 0; j < NJ; j++) v[j] = vt_buffer_ld4(vt_buffer(x_in + row * VT_DIM, VT_DIM * 4), at + 4096 * j);
#pragma unroll
    for (int s = 0; s < C; s++) {
        /* the planes behind the first have the columns from col0 on, and zeros for the others */
        const int from = s ? col0 : 0;
        const __amdgpu_buffer_rsrc_t d = vt_buffer(part + s * part_stride + row * VT_DIM + from, (VT_DIM - from) * 4);
#pragma unroll
        for (int j = 0; j < NJ; j++) p[j][s] = vt_buffer_ld4(d, at + 4096 * j - from * 4);
    }
    const __amdgpu_buffer_rsrc_t dw = vt_buffer(w, w ? VT_DIM * 4 : 0);
#pragma unroll
    for (int j = 0; j < NJ; j++) g[j] = vt_buffer_ld4(dw, at + 4096 * j);
    __builtin_amdgcn_sched_barrier(0);
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        f32x4 a = v[j];
        if (C > 0) {
            f32x4 q = p[j][0];
#pragma unroll
            for (int s = 1; s < C; s++) {
                q.x = __fadd_rn(q.x, p[j][s].x); q.y = __fadd_rn(q.y, p[j][s].y);
                q.z = __fadd_rn(q.z, p[j][s].z); q.w = __fadd_rn(q.w, p[j][s].w);
            }
            a.x = __fadd_rn(a.x, q.x); a.y = __fadd_rn(a.y, q.y);
            a.z = __fadd_rn(a.z, q.z); a.w = __fadd_rn(a.w, q.w);
        }
        if (C > 0 || x != x_in) vt_buffer_st4(dx, at + 4096 * j, a);
        v[j] = a;
        ss = fmaf(a.x, a.x, ss); ss = fmaf(a.y, a.y, ss);
        ss = fmaf(a.z, a.z, ss); ss = fmaf(a.w, a.w, ss);
    }
    if (!w) return;
    ss = vt_wave_sum(ss);
    if (vt_lane() == 0) red[vt_wave()] = ss;
    __syncthreads();
    const float tot = (red[0] + red[1]) + (red[2] + red[3]);
    const float inv = 1.0f / sqrtf(tot / (float)VT_DIM + eps);
    const __amdgpu_buffer_rsrc_t dh = vt_buffer(hi + row * VT_DIM, VT_DIM * 2), dl = vt_buffer(lo + row * VT_DIM, VT_DIM * 2);
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        u32x2 sph, spl;
        vt_split_planes4(__fmul_rn(__fmul_rn(v[j].x, inv), g[j].x), __fmul_rn(__fmul_rn(v[j].y, inv), g[j].y),
                         __fmul_rn(__fmul_rn(v[j].z, inv), g[j].z), __fmul_rn(__fmul_rn(v[j].w, inv), g[j].w), sph, spl);
        vt_buffer_st2(dh, at / 2 + 2048 * j, sph);
        vt_buffer_st2(dl, at / 2 + 2048 * j, spl);
    }
}

void vt_launch_residual_norm_split(float *d_x, const float *x_in, const float *d_part, int col0, int cuts, size_t part_stride,
                                   const float *d_w, uint16_t *d_hi, uint16_t *d_lo, int rows) {
#define CALL(C) hipLaunchKernelGGL(vt_residual_norm_split_kernel<C>, dim3(rows), dim3(256), 0, g_vt.stream, d_x, x_in, d_part, \
                                   col0, part_stride, d_w, d_hi, d_lo, VT_EPS)
    if (cuts <= 0) CALL(0);
    else GM_BY_PLANES(cuts, CALL);
#undef CALL
}

/* gu [rows, 2*ffn] with (gate, up) adjacent -> (hi, lo) planes of silu(gate)*up
 * (voxtral_tts_llm.c:346-350 on the row-interleaved gate/up matrix).  Columns from
 * tail_col0 on are taken as the sum of `tail_planes` split-K planes [rows, 2*ffn - tail_col0]
 * instead (tail_planes == 0: everything is in gu). */
__global__ void vt_swiglu_split_kernel(uint16_t *hi, uint16_t *lo, const float *gu, size_t n8,
                                       int tail_col0, const float *tail, int tail_planes, size_t tail_stride) {
    /* a thread owns 8 consecutive floats, i.e. 4 (gate, up) pairs: 16-byte loads, 8-byte plane
     * stores; rows and the tail boundary are multiples of 8 columns */
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n8;
         i += (size_t)gridDim.x * blockDim.x) {
        f32x4 g0 = reinterpret_cast<const f32x4 *>(gu)[2 * i];
        f32x4 g1 = reinterpret_cast<const f32x4 *>(gu)[2 * i + 1];
        if (tail_planes > 0) {
            const size_t row = (8 * i) / (2 * VT_FFN);
            const int col = (int)((8 * i) % (2 * VT_FFN));
            if (col >= tail_col0) {
                const int tw = 2 * VT_FFN - tail_col0;
                const float *tp = tail + row * tw + (col - tail_col0);
                g0 = *reinterpret_cast<const f32x4 *>(tp);
                g1 = *reinterpret_cast<const f32x4 *>(tp + 4);
                for (int p = 1; p < tail_planes; p++) {
                    const f32x4 w0 = *reinterpret_cast<const f32x4 *>(tp + p * tail_stride);
                    const f32x4 w1 = *reinterpret_cast<const f32x4 *>(tp + p * tail_stride + 4);
                    g0.x = __fadd_rn(g0.x, w0.x); g0.y = __fadd_rn(g0.y, w0.y);
                    g0.z = __fadd_rn(g0.z, w0.z); g0.w = __fadd_rn(g0.w, w0.w);
                    g1.x = __fadd_rn(g1.x, w1.x); g1.y = __fadd_rn(g1.y, w1.y);
                    g1.z = __fadd_rn(g1.z, w1.z); g1.w = __fadd_rn(g1.w, w1.w);
                }
            }
        }
        const f32x4 h = vt_silu_mul4(f32x4{g0.x, g0.z, g1.x, g1.z}, f32x4{g0.y, g0.w, g1.y, g1.w});
        u32x2 sph, spl;
        vt_split_planes4(h.x, h.y, h.z, h.w, sph, spl);
        reinterpret_cast<u32x2 *>(hi)[i] = sph;
        reinterpret_cast<u32x2 *>(lo)[i] = spl;
    }
}

void vt_launch_swiglu_split(uint16_t *d_hi, uint16_t *d_lo, const float *d_gu, size_t n_out, int tail_col0,
                            const float *d_tail, int tail_planes, size_t tail_stride) {
    hipLaunchKernelGGL(vt_swiglu_split_kernel, dim3(gm_blocks(n_out / 4)), dim3(256), 0, g_vt.stream, d_hi, d_lo,
                       d_gu, n_out / 4, tail_col0, d_tail, tail_planes, tail_stride);
}

/* The K-cut tail of the paired gate|up product: tail [planes][rows, tw] fp32 in the paired column order
 * (of every 32 columns the first 16 are gates, the other 16 the ups of the same h columns) -> the
 * (hi, lo) planes of SiLU(gate) * up at h columns h_col0 .. h_col0 + tw/2 (row pitch ldh).  A thread owns 4
 * consecutive h columns and requests all its planes at once. */
template <int P>
__global__ void __launch_bounds__(256) vt_swiglu_pair_tail_kernel(uint16_t *hi, uint16_t *lo, int ldh, int h_col0, const float *tail,
                                                                  size_t stride, int rows, int tw) {
    const int q = (int)(blockIdx.x * 256 + threadIdx.x), blk = q >> 2, c = (q & 3) * 4;
    if (q >= tw / 8) return;
    for (size_t row = blockIdx.y; row < (size_t)rows; row += gridDim.y) {
        f32x4 gs[P], us[P];
#pragma unroll
        for (int p = 0; p < P; p++) {
            const __amdgpu_buffer_rsrc_t d = vt_buffer(tail + p * stride + row * tw, tw * 4);
            gs[p] = vt_buffer_ld4(d, (32 * blk + c) * 4);
            us[p] = vt_buffer_ld4(d, (32 * blk + c) * 4 + 64);
        }
        __builtin_amdgcn_sched_barrier(0);
        f32x4 g = gs[0], u = us[0];
#pragma unroll
        for (int p = 1; p < P; p++) {
            g.x = __fadd_rn(g.x, gs[p].x); g.y = __fadd_rn(g.y, gs[p].y); g.z = __fadd_rn(g.z, gs[p].z); g.w = __fadd_rn(g.w, gs[p].w);
            u.x = __fadd_rn(u.x, us[p].x); u.y = __fadd_rn(u.y, us[p].y); u.z = __fadd_rn(u.z, us[p].z); u.w = __fadd_rn(u.w, us[p].w);
        }
        const f32x4 h = vt_silu_mul4(g, u);
        u32x2 sph, spl;
        vt_split_planes4(h.x, h.y, h.z, h.w, sph, spl);
        const size_t at = row * ldh + h_col0;
        vt_buffer_st2(vt_buffer(hi + at, tw), (16 * blk + c) * 2, sph);
        vt_buffer_st2(vt_buffer(lo + at, tw), (16 * blk + c) * 2, spl);
    }
}

void vt_launch_swiglu_pair_tail(uint16_t *d_hi, uint16_t *d_lo, int ldh, int h_col0, const float *d_tail, int planes,
                                size_t stride, int rows, int tw) {
#define CALL(P) hipLaunchKernelGGL(vt_swiglu_pair_tail_kernel<P>, dim3((tw / 8 + 255) / 256, rows < 65535 ? rows : 65535), dim3(256), 0, g_vt.stream, \
                                   d_hi, d_lo, ldh, h_col0, d_tail, stride, rows, tw)
    GM_BY_PLANES(planes, CALL);
#undef CALL
}

/* C = sum of `splits` partial planes (fixed order), for callers that want the plain product. */
__global__ void vt_sum_planes_kernel(float *out, const float *part, int splits, size_t stride, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (size_t)gridDim.x * blockDim.x) {
        float p = part[i];
        for (int s = 1; s < splits; s++) p = __fadd_rn(p, part[(size_t)s * stride + i]);
        out[i] = p;
    }
}

void vt_launch_sum_planes(float *d_out, const float *d_part, int splits, size_t stride, size_t n) {
    hipLaunchKernelGGL(vt_sum_planes_kernel, dim3(gm_blocks(n)), dim3(256), 0, g_vt.stream, d_out, d_part,
                       splits, stride, n);
}

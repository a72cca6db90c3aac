/*
 * vt_codec_gemm.hip - the codec decoder's products (fp32 weights, fp32 activations) on the fp16 matrix cores.
 *
 * Every fp32 operand is carried as two fp16 planes, hi = fp16(s x) and lo = fp16(2^6 (s x - hi)), with a power of two s
 * per row that brings the row's largest magnitude to 2^14 .. 2^15: hi + 2^-6 lo then holds s x to 2^-23 of itself down
 * to 2^-22 of the row's largest, and to 2^-46 of that below.  A product is hi hi + hi lo + lo hi, three matrix
 * instructions on the same fp32 sums; the lo lo term left out is at most 2^-22 of the product.  An operand so has up to
 * one bit less than fp32, and the sums have fewer roundings (one per instruction, not one per product): where they
 * matter more, the result is closer to 64 bits than with fp32 instructions.
 * Three fp16 instructions do 16 times the work of an fp32 one each, so the
 * same product takes 3/16 of the matrix-core time; what it then runs into is the card's power limit.
 * Measured against float64, error of a row over its l2 norm, K 1024 / 4096: 1.4e-7 / 2.1e-7, worst row 2.7e-7 / 4.0e-7
 * (rows and elements of log-normal magnitude), where fp32 sums in order have 5.7e-7 / 1.1e-6, worst 1.6e-6 / 1.9e-6.
 * The 2^6 is for rows with values far apart whose large ones meet zeros: with one channel of the activations and one of
 * the weights 2^20 / 2^24 times the others, 1.4e-7 / 4.4e-7 at K = 1024 (2.1e-7 / 4.6e-7 at 4096); without it the operands alone
 * leave 2.4e-6 / 3.7e-5 at K = 1024.  hi times 2^-6, which it takes, costs 0.7 / 1.6 / 1.5 % of a decode of 21 / 212 / 1003 frames.
 * Rates, TFLOP/s of the product itself (v_mfma_f32_32x32x2f32 in 128 x 128 tiles before: 75 .. 105): gate|up
 * 8192 x 1024 at 212 / 848 / 1696 / 8024 rows 170 / 329 / 329 / 377, down 1024 x 4096 125 / 254 / 323 / 409.
 */
#include "vt_gemm_tiles.h"

/* ---- weights: row-major fp32 [N, K] -> fragment order, two fp16 planes --------------------------------------- */

/* row n is stored times 2^col_exp[n] */
__global__ void __launch_bounds__(256) vt_codec_weight_exp_kernel(int *col_exp, const float *W, int K) {
    __shared__ float red[4];
    const size_t n = blockIdx.x;
    float m = 0.f;
    for (int k = threadIdx.x; k < K; k += 256) m = fmaxf(m, fabsf(W[n * K + k]));
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) col_exp[n] = vt_f16_exp(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])));
}

/* 16-byte slot (((n/32 * K/64 + ks) * 2 + plane) * 4 + j) * 64 + l holds elements 64 ks + 32 (l/32) + 8 j .. + 8 of row
 * 32 (n/32) + l % 32 */
__global__ void vt_codec_weight_layout_kernel(u32x4 *out, const float *W, const int *col_exp, size_t n_slots, int K) {
    const int ksteps = K / 64;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_slots; i += (size_t)gridDim.x * blockDim.x) {
        const int l = (int)(i & 63), j = (int)((i >> 6) & 3);
        const size_t blk = i >> 8, n = blk / ksteps * 32 + (l & 31);
        const int ks = (int)(blk % ksteps);
        const f32x4 *p = reinterpret_cast<const f32x4 *>(W + n * K + 64 * ks + 32 * (l >> 5) + 8 * j);
        const f32x4 a = vt_ldexp4(p[0], col_exp[n]), b = vt_ldexp4(p[1], col_exp[n]);
        u32x2 h0, l0, h1, l1;
        vt_split_f16x4(a, h0, l0);
        vt_split_f16x4(b, h1, l1);
        out[(blk * 2) * 256 + j * 64 + l] = u32x4{h0.x, h0.y, h1.x, h1.y};
        out[(blk * 2 + 1) * 256 + j * 64 + l] = u32x4{l0.x, l0.y, l1.x, l1.y};
    }
}

int vt_codec_weight_layout(uint16_t *d_Wf, int *d_col_exp, const float *d_W, int N, int K) {
    if (vt_check(hipStreamSynchronize(NULL), "codec weight copy")) return -1;      /* d_W may have been copied from device memory */
    hipLaunchKernelGGL(vt_codec_weight_exp_kernel, dim3(N), dim3(256), 0, g_vt.stream, d_col_exp, d_W, K);
    const size_t n_slots = (size_t)N * K / 8;
    hipLaunchKernelGGL(vt_codec_weight_layout_kernel, dim3((unsigned)((n_slots + 255) / 256 > 8192 ? 8192 : (n_slots + 255) / 256)), dim3(256), 0, g_vt.stream,
                       (u32x4 *)d_Wf, d_W, d_col_exp, n_slots, K);
    return vt_check(hipGetLastError(), "codec weight layout") || vt_check(hipStreamSynchronize(g_vt.stream), "codec weight layout") ? -1 : 0;
}

/* ---- launches -------------------------------------------------------------------------------------------------- */

template <int NP>
static void cg_rows(const gr_list &plan, int grid, const uint16_t *d_hi, const uint16_t *d_lo, int M, int K) {
    constexpr int NW = VT_CODEC_ROW_WAVES;
    static int attr_set = 0;
    const int lds = NW * 2 * 32 * ((NP + 3) / 4) * GM_STAGE_ROW;
    if (!attr_set) {
        if (vt_check(hipFuncSetAttribute((const void *)vt_gemm_rows_kernel<gm_f16x2, NP, NW>, hipFuncAttributeMaxDynamicSharedMemorySize, lds), "product LDS size"))
            return;
        attr_set = 1;
    }
    hipLaunchKernelGGL((vt_gemm_rows_kernel<gm_f16x2, NP, NW>), dim3(grid), dim3(64 * NW), lds, g_vt.stream, plan, d_hi, d_lo, M, K);
}

template <int MB, int CW>
static void cg_wide(const gw_list &list, const uint16_t *d_hi, const uint16_t *d_lo, int M, int K) {
    constexpr int LDS = 2 * gw_shape<MB, CW, false>::STAGE + gw_shape<MB, CW, false>::TM * (int)sizeof(int);
    static int attr_set = 0;
    if (!attr_set) {
        if (vt_check(hipFuncSetAttribute((const void *)vt_gemm_wide_kernel<gm_f16x2, MB, CW, 2>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS), "product LDS size"))
            return;
        attr_set = 1;
    }
    const int items = list.part[0].items;
    hipLaunchKernelGGL((vt_gemm_wide_kernel<gm_f16x2, MB, CW, 2>), dim3(items < g_vt.n_cu ? items : g_vt.n_cu), dim3(256), LDS, g_vt.stream, list, d_hi, d_lo, M, K);
}

void vt_launch_codec_gemm(float *d_C, const uint16_t *d_hi, const uint16_t *d_lo, const int *d_row_exp,
                          const uint16_t *d_Wf, const int *d_col_exp, int M, int N, int K, const vt_gemm_plan &pl) {
    if (pl.tm == 0) {
        const int items = N / GR_TN * pl.cuts, grid = items < g_vt.n_cu ? items : g_vt.n_cu;
        const gr_list plan = {d_C, d_Wf, (size_t)M * N, N, items, vt_divisor_of(N / GR_TN, items), gm_cuts_of(K, pl.cuts), d_row_exp, d_col_exp};
        static void (*const launch[4])(const gr_list &, int, const uint16_t *, const uint16_t *, int, int) = {cg_rows<2>, cg_rows<4>, cg_rows<6>, cg_rows<8>};
        launch[(M + 15) / 16 - 1](plan, grid, d_hi, d_lo, M, K);
        return;
    }
    gw_list list = {};
    gw_part whole = {d_C, d_Wf, 0, pl.col0, pl.col0 / pl.tn, 1, NULL, NULL, 0, d_row_exp, d_col_exp};
    gw_part cut = {d_C + (size_t)M * pl.col0, d_Wf + (size_t)pl.col0 * K * 2, (size_t)M * (N - pl.col0), N - pl.col0, (N - pl.col0) / pl.tn, pl.cuts, NULL, NULL, 0,
                   d_row_exp, d_col_exp + pl.col0};
    gw_add(list, whole, M, pl.tm, K);
    gw_add(list, cut, M, pl.tm, K);
    static void (*const launch[2][2])(const gw_list &, const uint16_t *, const uint16_t *, int, int) = {{cg_wide<3, 2>, cg_wide<3, 4>}, {cg_wide<4, 2>, cg_wide<4, 4>}};
    launch[pl.tm == 128][pl.tn == 256](list, d_hi, d_lo, M, K);
}

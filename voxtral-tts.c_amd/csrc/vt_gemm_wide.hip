/*
 * vt_gemm_wide.hip - the backbone's prefill products on the tile kernels of vt_gemm_tiles.h, more than 64 rows, and
 * the plans of all of them: which tile, and which columns in how many K cuts.
 */
#include "vt_gemm_tiles.h"

/* ---- plans and launches ---------------------------------------------------------------------------- */

/* What a product is expected to take, in us, for the choice between tiles and cuts.  A round of items takes as
 * long as the operands of its steps need to arrive (step_us: a step of the 128- and 192-column tiles is two K steps, half
 * of the waves at each) and item_us for sums and stores, but no less than the card's
 * power limit lets the matrix cores of its items run (pflops, executed, padding included: narrow tiles pay
 * for their bytes here, too); cut planes are written and read once more.  (The codec's item_us is what an item takes beside its steps and what its
 * matrix instructions take beyond them: the choice depends on their sum.)
 * The backbone's 192 columns divide 6144 and 3072 into 32 and 16 tiles, so that 1, 2, 4, .. row tiles fill the 256 CUs
 * where 256-column tiles come in multiples of 192 items: q|k|v / output / down at 700 rows 57.5 / 40.7 / 79.4 -> 51.1 / 37.2 /
 * 72.5 us, at 1000 75.0 / 53.3 / 104.9 -> 68.5 / 49.2 / 97.0, output / down at 1531 73.3 / 149.4 -> 67.1 / 140.6.
 * Measured against every tile and cut count at 47 row counts from 65 to 2048 of the backbone's products, the plan taken is 0.3 % behind the
 * fastest on average, at worst 5.5 % (q|k|v at 113 rows, 80 x 256 in 5 cuts instead of 4); for the codec's at 108 of 65 to 8024
 * rows, 0.6 % and at worst 8.1 % (output at 128 rows).  Single products exchanged inside prefills of 150 to 1531 rows were at most 2.7 %
 * of the prefill faster (gate|up at 700 rows, 96 x 384 in part cut).  Tiles x 384, which draw less power per product, are taken from 400 rows on
 * (gate|up) and from 690 (down): below, too few items are left for the CUs.  80 and 112 rows, where those of 96 and 128 have many to pad: us of
 * the four products at 200 / 226 / 290 / 400 / 800 rows 140 / 144 / 173 / 197 / 334 -> 130 / 136 / 163 / 186 / 322, a prefill of 226 rows 4274 -> 4020. */
struct gw_format {
    int products;                         /* matrix instructions per pair of operands */
    float launch_us, planes;              /* planes: passes over a cut column's planes */
    float sums_us, stream_tbps;           /* the launch that adds them (0: whoever reads the result does); the weights' rate (0: no bound) */
    float item_us[4];                     /* [128, 192, 256, 384 columns] */
    float step_us[4][4];                  /* [128, 192, 256, 384 columns][80, 96, 112, 128 rows]; 0: tile not used */
    float pflops[4];                      /* [128, 192, 256, 384 columns] */
};
static int gw_width(int tn) { return tn == 384 ? 3 : tn / 64 - 2; }
static int gw_height(int tm) { return tm / 16 - 5; }
static const gw_format gw_backbone = {2, 0.f, 2.60f, 0.f, 0.f, {1.47f, 3.96f, 0.09f, 2.37f}, {{0.f, 1.397f, 0.f, 0.f}, {1.521f, 1.652f, 0.f, 1.967f}, {0.904f, 0.976f, 1.206f, 1.202f},
    {1.302f, 1.398f, 0.f, 1.714f}}, {99.f, 1.381f, 1.496f, 99.f}};
static const gw_format gw_codec = {3, 1.03f, 2.33f, 0.f, 0.f, {4.56f, 0.f, 4.56f, 0.f}, {{0.f, 1.874f, 0.f, 2.375f}, {}, {0.f, 1.45f, 0.f, 1.944f}, {}}, {99.f, 0.f, 1.76f, 0.f}};

static float gw_rounds(int items, float item_us, float power_us) {
    const int full = items / g_vt.n_cu, rem = items % g_vt.n_cu;
    return full * fmaxf(item_us, g_vt.n_cu * power_us) + (rem ? fmaxf(item_us, rem * power_us) : 0.f);
}

static float gw_cost(const gw_format &f, int M, int N, int K, int tm, int tn, int n_main, int cuts, int swiglu) {
    const int kw = tn < 256 ? 2 : 1, mt = (M + tm - 1) / tm, w = gw_width(tn);
    const float t_step = f.step_us[w][gw_height(tm)];
    const float tile_us = 2.f * f.products * tm * tn * (float)K / (f.pflops[w] * 1e9f);
    const int rest = N / tn - n_main;
    float t = f.launch_us + gw_rounds(mt * n_main, (float)((K / 64 + kw - 1) / kw) * t_step + f.item_us[w], tile_us);
    if (rest) {
        t += gw_rounds(mt * rest * cuts, (float)((K / 64 + cuts * kw - 1) / (cuts * kw)) * t_step + f.item_us[w], tile_us / cuts);
        if (cuts > 1 || swiglu) t += f.planes * cuts * M * (float)(rest * tn) * 4.f / 4.5e6f + (swiglu ? 4.5f : cuts > 1 ? f.sums_us : 0.f);
    }
    return f.stream_tbps > 0.f ? fmaxf(t, f.launch_us + N * 2.f * K / (f.stream_tbps * 1e6f)) : t;
}

static vt_gemm_plan gw_plan(const gw_format &f, int M, int N, int K, int swiglu, int most = VT_MAX_CUTS, float *us = NULL) {
    vt_gemm_plan best = {0, 64, 0, 1};
    float best_cost = 0.f;
    for (int tm = 80; tm <= 128; tm += 16)
        for (int tn : {128, 192, 256, 384}) {
            if (N % tn || f.step_us[gw_width(tn)][gw_height(tm)] == 0.f) continue;
            const int mt = (M + tm - 1) / tm, nt = N / tn;
            /* whole tiles: as many as make full rounds over the CUs, or one round fewer, or all */
            const int full = mt * nt / g_vt.n_cu;
            for (int pick = 0; pick < 3; pick++) {
                int n_main = pick == 2 ? nt : (full - pick) * g_vt.n_cu / mt;
                if (n_main < 0 || n_main > nt) continue;
                if (n_main * tn % 128) n_main--;          /* heads of 128 columns are cut or not */
                for (int cuts = 1; cuts <= most && cuts <= K / 64; cuts++) {
                    if (n_main == nt && cuts > 1) break;
                    if (swiglu && n_main < nt && cuts == 1) continue;
                    const float c = gw_cost(f, M, N, K, tm, tn, n_main, cuts, swiglu);
                    if (best_cost == 0.f || c < best_cost) {
                        best_cost = c;
                        best = vt_gemm_plan{tm, tn, n_main * tn, n_main == nt ? 1 : cuts};
                    }
                }
            }
        }
    if (us) *us = best_cost;
    return best;
}

vt_gemm_plan vt_gemm_frag_plan(int M, int N, int K, int swiglu) {
    return vt_gemm_rows_ok(M, N, K) ? vt_gemm_few_rows_plan(N, swiglu) : gw_plan(gw_backbone, M, N, K, swiglu);
}

vt_gemm_plan vt_codec_gemm_plan(int M, int N, int K) {
    if (vt_gemm_rows_ok(M, N, K)) return vt_gemm_plan{0, 64, 0, vt_gemm_rows_cuts(VT_CODEC_ROW_WAVES, N, K, VT_MAX_CUTS)};
    return gw_plan(gw_codec, M, N, K, 0);
}

template <int MB, int CW, int NB, bool FRAG = true, bool PAIR = false>
static int gw_prepare(void) {
    static int attr_device = -1;
    if (attr_device == g_vt.device) return 0;
    if (vt_check(hipFuncSetAttribute((const void *)vt_gemm_wide_kernel<gm_bf16, MB, CW, NB, FRAG, PAIR>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     2 * gw_shape<MB, CW, PAIR>::STAGE), "product LDS size"))
        return -1;
    attr_device = g_vt.device;
    return 0;
}

/* With the context: a product on a caller's weights may be the first call inside a stream capture */
int vt_gemm_row_major_prepare(void) {
    return gw_prepare<3, 2, 2, false>() || gw_prepare<3, 2, 3, false>() || gw_prepare<3, 4, 2, false>() || gw_prepare<4, 2, 3, false>() || gw_prepare<4, 4, 2, false>() ? -1 : 0;
}

template <int MB, int CW, int NB, bool FRAG = true, bool PAIR = false>
static void gw_launch(const gw_list &list, const uint16_t *d_Ahi, const uint16_t *d_Alo, int M, int K) {
    constexpr int LDS = 2 * gw_shape<MB, CW, PAIR>::STAGE;
    if (gw_prepare<MB, CW, NB, FRAG, PAIR>()) return;
    const int items = list.part[0].items;      /* every workgroup takes an item of the first part */
    hipLaunchKernelGGL((vt_gemm_wide_kernel<gm_bf16, MB, CW, NB, FRAG, PAIR>), dim3(items < g_vt.n_cu ? items : g_vt.n_cu), dim3(256), LDS, g_vt.stream,
                       list, d_Ahi, d_Alo, M, K);
}

static void gw_run(const vt_gemm_plan &pl, gw_part whole, gw_part cut, const uint16_t *d_Ahi, const uint16_t *d_Alo, int M, int N, int K) {
    gw_list list = {};
    whole.n_tiles = pl.col0 / pl.tn;
    whole.splits = 1;
    cut.n_tiles = (N - pl.col0) / pl.tn;
    cut.splits = pl.cuts;
    gw_add(list, whole, M, pl.tm, K);
    gw_add(list, cut, M, pl.tm, K);
    typedef void (*fn)(const gw_list &, const uint16_t *, const uint16_t *, int, int);
    static const fn launch[4][4] = {{NULL, gw_launch<5, 2, 3, true, true>, gw_launch<5, 4, 2, true, true>, gw_launch<5, 4, 3, true, true>},
                                    {gw_launch<3, 2, 2>, gw_launch<3, 2, 3>, gw_launch<3, 4, 2>, gw_launch<3, 4, 3>},
                                    {NULL, NULL, gw_launch<7, 4, 2, true, true>, NULL},
                                    {NULL, gw_launch<4, 2, 3>, gw_launch<4, 4, 2>, gw_launch<4, 4, 3>}};
    static const fn row_major[2][3] = {{gw_launch<3, 2, 2, false>, gw_launch<3, 2, 3, false>, gw_launch<3, 4, 2, false>}, {NULL, gw_launch<4, 2, 3, false>, gw_launch<4, 4, 2, false>}};
    (pl.row_major ? row_major[pl.tm == 128][gw_width(pl.tn)] : launch[gw_height(pl.tm)][gw_width(pl.tn)])(list, d_Ahi, d_Alo, M, K);
}

/* Products on a caller's row-major weights: tiles (a lane's own row costs four times the lines per request, hence constants of
 * their own; a step's four requests of a line stand one in each of its regions, as with fragments: all in the last one, 42 us instead of
 * 39 for 9216 x 3072 at 150 rows), up to 64 rows strips of 96 columns, and the 128 x 128 tiles of vt_launch_gemm, two
 * workgroups per CU, which stage the weights through LDS in whole lines.  Each is taken where it is expected to be the fastest.  Fitted
 * to 1312 shapes, 28 of N and K from 512 x 8192 to 131072 x 3072 and 8 .. 1000 rows, the launch that adds planes included: the choice is
 * 0.9 % behind the fastest of all tiles, strips and cuts on average, 3.2 % where bounds on M, N and K made it, and takes 0.882 of the time
 * of 128 x 128 tiles alone, 0.902; above 1.05 of it at 5 shapes, 84 (18 rows of 4608 x 1024 1.25; at most 1.83).  No part of it came near
 * the card's power limit (pflops). */
static const gw_format gw_row_major = {2, 6.875f, 1.892f, 2.173f, 4.638f, {2.226f, 2.226f, 2.226f, 0.f}, {{0.f, 1.446f, 0.f, 0.f}, {0.f, 1.968f, 0.f, 2.054f}, {0.f, 1.138f, 0.f, 1.189f}, {}}, {99.f, 99.f, 99.f, 99.f}};

/* Strips: a workgroup goes through its K steps three at a time, which takes longer by the group of 8 rows, and so do its sums; but no
 * less than its or the card's share of the weights' rate allows */
static float gw_strip_us(int M, int N, int K, int tn, int cuts) {
    const int groups = (M + 7) / 8, rounds = ((N + tn - 1) / tn * cuts + g_vt.n_cu - 1) / g_vt.n_cu, steps = ((K / 64 + cuts - 1) / cuts + 2) / 3 * 3;
    const float work = steps * (0.2246f + 0.02967f * groups) + 3.623f + 0.3222f * groups, share = steps * 0.6939f;
    const float t = 0.3942f + fmaxf(rounds * fmaxf(work, share), N * 2.f * K / 13.36e6f);
    return cuts > 1 ? t + gw_row_major.sums_us + gw_row_major.planes * cuts * M * (float)N * 4.f / 4.5e6f : t;
}

/* 128 x 128 tiles: a step takes longer the more CUs take one, and shorter with rows to pad */
float vt_gemm_equal_us(int M, int N, int K, int cuts) {
    const int items = (M + 127) / 128 * (N / 128) * cuts, slots = 2 * g_vt.n_cu, rem = items % slots;
    const float steps = K / cuts / 64, short_rows = 0.3468f * (1.f - (M < 128 ? M : 128) / 128.f);
    float t = 4.158f + items / slots * (steps * 1.737f + 3.122f);
    if (rem) t += steps * ((rem <= g_vt.n_cu ? 0.8687f + 0.1399f * rem / g_vt.n_cu : 1.737f) - short_rows) + 3.122f;
    return cuts > 1 ? t + gw_row_major.sums_us + 0.2854f * cuts + 0.7692f * (cuts + 1) * M * (float)N * 4.f / 4.5e6f : t;
}

vt_gemm_plan vt_gemm_row_major_plan(int M, int N, int K, int most, float *us) {
    vt_gemm_plan pl = gw_plan(gw_row_major, M, N, K, 0, most, us);
    if (pl.cuts == 1) pl.col0 = N;
    if (vt_gemm_rows_ok(M, N, K)) {
        const vt_gemm_plan strips = vt_gemm_few_rows_plan(N, 0);
        for (int cuts = 1; cuts <= strips.cuts && cuts <= most && cuts <= K / 64; cuts++) {
            const float t = gw_strip_us(M, N, K, strips.tn, cuts);
            if (t < *us) { *us = t; pl = strips; pl.cuts = cuts; }
        }
    }
    pl.row_major = 1;
    return pl;
}

/* y[:, col0 ..] = the planes' sum, in order, all of them requested in front of the first addition: a chain of memory latencies */
__global__ void __launch_bounds__(256) vt_sum_cut_columns_kernel(float *y, const float *part, int cuts, int M, int N, int col0) {
    const int w = (N - col0) / 4;
    const size_t n = (size_t)M * w;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        f32x4 q[VT_MAX_CUTS];
#pragma unroll
        for (int p = 0; p < VT_MAX_CUTS; p++) q[p] = reinterpret_cast<const f32x4 *>(part)[(p < cuts ? p : 0) * n + i];
        f32x4 v = q[0];
#pragma unroll
        for (int p = 1; p < VT_MAX_CUTS; p++)
            if (p < cuts) { v.x = __fadd_rn(v.x, q[p].x); v.y = __fadd_rn(v.y, q[p].y); v.z = __fadd_rn(v.z, q[p].z); v.w = __fadd_rn(v.w, q[p].w); }
        *reinterpret_cast<f32x4 *>(y + i / w * N + col0 + i % w * 4) = v;
    }
}

void vt_launch_gemm_row_major(float *d_y, float *d_part, const uint16_t *d_Ahi, const uint16_t *d_Alo, const uint16_t *d_W, int M, int N, int K,
                              const vt_gemm_plan &pl) {
    const int cut = N - pl.col0;
    const size_t plane = (size_t)M * cut;
    if (pl.tm == 0) vt_launch_gemm_few_rows(pl.cuts > 1 ? d_part : d_y, N, plane, d_Ahi, d_Alo, d_W, M, N, K, pl);
    else gw_run(pl, gw_part{d_y, d_W, 0, N, 0, 0, NULL, NULL, 0, NULL, NULL},
                gw_part{d_part, d_W + (size_t)pl.col0 * K, plane, cut, 0, 0, NULL, NULL, 0, NULL, NULL}, d_Ahi, d_Alo, M, N, K);
    if (pl.cuts > 1) {
        const size_t n = plane / 4;
        hipLaunchKernelGGL(vt_sum_cut_columns_kernel, dim3((unsigned)((n + 255) / 256 > 4096 ? 4096 : (n + 255) / 256)), dim3(256), 0, g_vt.stream, d_y, d_part, pl.cuts, M, N, pl.col0);
    }
}

void vt_launch_gemm_frag(float *d_C, int ldc, size_t plane_stride, const uint16_t *d_Ahi, const uint16_t *d_Alo,
                         const uint16_t *d_Wf, int M, int N, int K, const vt_gemm_plan &pl) {
    if (pl.tm == 0) { vt_launch_gemm_few_rows(d_C, ldc, plane_stride, d_Ahi, d_Alo, d_Wf, M, N, K, pl); return; }
    gw_run(pl, gw_part{d_C, d_Wf, plane_stride, ldc, 0, 0, NULL, NULL, 0, NULL, NULL},
           gw_part{d_C + pl.col0, d_Wf + (size_t)pl.col0 * K, plane_stride, ldc, 0, 0, NULL, NULL, 0, NULL, NULL}, d_Ahi, d_Alo, M, N, K);
}

void vt_launch_gemm_frag_swiglu(uint16_t *d_hhi, uint16_t *d_hlo, int ldh, float *d_tail, const uint16_t *d_Ahi,
                                const uint16_t *d_Alo, const uint16_t *d_Wf, int M, int N, int K, const vt_gemm_plan &pl) {
    const int tail = N - pl.col0;
    if (pl.tm == 0)
        vt_launch_gemm_few_rows(d_tail, N, (size_t)M * N, d_Ahi, d_Alo, d_Wf, M, N, K, pl);
    else
        gw_run(pl, gw_part{NULL, d_Wf, 0, 0, 0, 0, d_hhi, d_hlo, ldh, NULL, NULL},
               gw_part{d_tail, d_Wf + (size_t)pl.col0 * K, (size_t)M * tail, tail, 0, 0, NULL, NULL, 0, NULL, NULL}, d_Ahi, d_Alo, M, N, K);
    if (tail) vt_launch_swiglu_pair_tail(d_hhi, d_hlo, ldh, pl.col0 / 2, d_tail, pl.cuts, (size_t)M * tail, M, tail);
}

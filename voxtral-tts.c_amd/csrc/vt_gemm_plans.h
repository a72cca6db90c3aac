/*
 * vt_gemm_plans.h - which tile a product takes, and which columns in how many K cuts: the choice from a shape and the number of
 * CUs.  Host code without HIP, so that a host test can walk it.
 */
#ifndef VT_GEMM_PLANS_H
#define VT_GEMM_PLANS_H

#include <initializer_list>
#include <math.h>
#include <stddef.h>

/* How a product of the backbone is done on fragment-order weights (vt_launch_frag_layout): the columns below
 * col0 as whole tiles (one plane), the others with K in `cuts` cuts (that many partial planes, to be added in
 * order by whoever reads the result).  tm, tn: rows and columns of the tile
 * (vt_gemm_wide.hip; tm 0: vt_gemm_rows.hip).  col0 is a multiple of 128. */
#define VT_MAX_CUTS 8
struct vt_gemm_plan { int tm, tn, col0, cuts, row_major; };      /* row_major: W as it is (vt_gemm_row_major_plan) */

/* ---- up to 64 rows --------------------------------------------------------------------------------- */

#define GR_TN 64                          /* columns of a tile of vt_gemm_rows_kernel */
#define GS_WIDE 288                       /* columns of a strip of vt_gemm_strip_kernel: gate|up, the others */
#define GS_NARROW 96
#define VT_CODEC_ROW_WAVES 4     /* of a workgroup of vt_gemm_rows_kernel: with two weight planes a wave's registers do not fit two waves per SIMD */

static inline int vt_gemm_rows_ok(int M, int N, int K) { return M >= 1 && M <= 64 && N % GR_TN == 0 && K % 64 == 0; }

static inline int gp_rows_cuts(int n_cu, int nw, int N, int K, int most) {
    /* of the cut counts that leave every CU at most one item, the fewest planes among those with the fewest
     * K steps on the busiest wave */
    const int tiles = N / GR_TN, steps = K / 64;
    int best = 1, best_cost = steps;
    for (int c = 1; c <= most && tiles * c <= n_cu; c++) {
        const int cost = ((steps + c - 1) / c + nw - 1) / nw;
        if (c == 1 || cost < best_cost) { best = c; best_cost = cost; }
    }
    return best;
}

static inline vt_gemm_plan gp_few_rows(int n_cu, int N, int swiglu) {
    const int tn = swiglu ? GS_WIDE : GS_NARROW, cuts = n_cu / ((N + tn - 1) / tn);
    return vt_gemm_plan{0, tn, 0, cuts < 1 ? 1 : cuts < VT_MAX_CUTS ? cuts : VT_MAX_CUTS};
}

/* ---- tiles ----------------------------------------------------------------------------------------- */

/* What a product is expected to take, in us, for the choice between tiles and cuts.  A round of items takes as
 * long as the operands of its steps need to arrive (step_us: a step of the 128- and 192-column tiles is two K steps, half
 * of the waves at each) and item_us for sums and stores, but no less than the card's
 * power limit lets the matrix cores of its items run (pflops, executed, padding included: narrow tiles pay
 * for their bytes here, too); cut planes are written and read once more.  (The codec's item_us is what an item takes beside its steps and what its
 * matrix instructions take beyond them: the choice depends on their sum.)
 * The backbone's 192 columns divide 6144 and 3072 into 32 and 16 tiles, so that 1, 2, 4, .. row tiles fill the 256 CUs
 * where 256-column tiles come in multiples of 192 items: q|k|v / output / down at 700 rows 57.5 / 40.7 / 79.4 -> 51.1 / 37.2 /
 * 72.5 us, at 1000 75.0 / 53.3 / 104.9 -> 68.5 / 49.2 / 97.0, output / down at 1531 73.3 / 149.4 -> 67.1 / 140.6.
 * Measured against every tile and cut count at 19 row counts from 65 to 1531 of the backbone's four products, the plan taken is 0.8 % behind
 * the fastest on average, at worst 5.2 % (down at 1200 rows, 128 x 384 in 3 cuts instead of 80 x 384 in 2); for the codec's at 17 row counts from
 * 84 to 8024, 0.6 % and at worst 6.9 %, which is how far two measurements of one division of the work (listed as whole and as cut columns)
 * are apart.  Single products exchanged inside prefills of 150 to 1531 rows were at most 2.7 %
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
static inline int gw_width(int tn) { return tn == 384 ? 3 : tn / 64 - 2; }
static inline int gw_height(int tm) { return tm / 16 - 5; }
static const gw_format gw_backbone = {2, 0.f, 2.60f, 0.f, 0.f, {1.47f, 3.96f, 0.09f, 2.37f}, {{0.f, 1.397f, 0.f, 0.f}, {1.521f, 1.652f, 0.f, 1.967f}, {0.904f, 0.976f, 1.206f, 1.202f},
    {1.302f, 1.398f, 0.f, 1.714f}}, {99.f, 1.381f, 1.496f, 99.f}};
static const gw_format gw_codec = {3, 1.03f, 2.33f, 0.f, 0.f, {4.56f, 0.f, 4.56f, 0.f}, {{0.f, 1.874f, 0.f, 2.375f}, {}, {0.f, 1.45f, 0.f, 1.944f}, {}}, {99.f, 0.f, 1.76f, 0.f}};

static inline float gw_rounds(int n_cu, int items, float item_us, float power_us) {
    const int full = items / n_cu, rem = items % n_cu;
    return full * fmaxf(item_us, n_cu * power_us) + (rem ? fmaxf(item_us, rem * power_us) : 0.f);
}

static inline float gw_cost(int n_cu, const gw_format &f, int M, int N, int K, int tm, int tn, int n_main, int cuts, int swiglu) {
    const int kw = tn < 256 ? 2 : 1, mt = (M + tm - 1) / tm, w = gw_width(tn);
    const float t_step = f.step_us[w][gw_height(tm)];
    const float tile_us = 2.f * f.products * tm * tn * (float)K / (f.pflops[w] * 1e9f);
    const int rest = N / tn - n_main;
    float t = f.launch_us + gw_rounds(n_cu, mt * n_main, (float)((K / 64 + kw - 1) / kw) * t_step + f.item_us[w], tile_us);
    if (rest) {
        t += gw_rounds(n_cu, mt * rest * cuts, (float)((K / 64 + cuts * kw - 1) / (cuts * kw)) * t_step + f.item_us[w], tile_us / cuts);
        if (cuts > 1 || swiglu) t += f.planes * cuts * M * (float)(rest * tn) * 4.f / 4.5e6f + (swiglu ? 4.5f : cuts > 1 ? f.sums_us : 0.f);
    }
    return f.stream_tbps > 0.f ? fmaxf(t, f.launch_us + N * 2.f * K / (f.stream_tbps * 1e6f)) : t;
}

/* Strips and these tiles store the rows that they have room for through one descriptor, whose size drops those past the last one.  Its
 * offsets have 32 bits, so all of these rows have to lie within them, not only those that exist: at 16,640,000 columns row 65 of a tile
 * would be row 0.  The same holds for what they load: rows of activations and, up to 96 of a wave, of weights, 2 K bytes each. */
static inline int gw_fits(int rows, int N, int K) { return 4ll * rows * N <= 0x7fffffff && 2ll * (rows > 96 ? rows : 96) * K <= 0x7fffffff; }

static inline vt_gemm_plan gw_plan(int n_cu, const gw_format &f, int M, int N, int K, int swiglu, int most = VT_MAX_CUTS, float *us = NULL) {
    vt_gemm_plan best = {0, 64, 0, 1};
    float best_cost = 0.f;
    for (int tm = 80; tm <= 128; tm += 16)
        for (int tn : {128, 192, 256, 384}) {
            if (N % tn || f.step_us[gw_width(tn)][gw_height(tm)] == 0.f || !gw_fits(tm, N, K)) continue;
            const int mt = (M + tm - 1) / tm, nt = N / tn;
            /* whole tiles: as many as make full rounds over the CUs, or one round fewer, or all */
            const int full = mt * nt / n_cu;
            for (int pick = 0; pick < 3; pick++) {
                int n_main = pick == 2 ? nt : (full - pick) * n_cu / mt;
                if (n_main < 0 || n_main > nt) continue;
                if (n_main * tn % 128) n_main--;          /* heads of 128 columns are cut or not */
                for (int cuts = 1; cuts <= most && cuts <= K / 64; cuts++) {
                    if (n_main == nt && cuts > 1) break;
                    if (swiglu && n_main < nt && cuts == 1) continue;
                    const float c = gw_cost(n_cu, f, M, N, K, tm, tn, n_main, cuts, swiglu);
                    if (best_cost == 0.f || c < best_cost) {
                        best_cost = c;
                        best = vt_gemm_plan{tm, tn, n_main * tn, n_main == nt ? 1 : cuts};
                    }
                }
            }
        }
    if (us) *us = best_cost > 0.f ? best_cost : INFINITY;      /* no tile fits */
    return best;
}

static inline vt_gemm_plan gp_frag(int n_cu, int M, int N, int K, int swiglu) {
    return vt_gemm_rows_ok(M, N, K) ? gp_few_rows(n_cu, N, swiglu) : gw_plan(n_cu, gw_backbone, M, N, K, swiglu);
}

static inline vt_gemm_plan gp_codec(int n_cu, int M, int N, int K) {
    if (vt_gemm_rows_ok(M, N, K)) return vt_gemm_plan{0, 64, 0, gp_rows_cuts(n_cu, VT_CODEC_ROW_WAVES, N, K, VT_MAX_CUTS)};
    return gw_plan(n_cu, gw_codec, M, N, K, 0);
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
static inline float gw_strip_us(int n_cu, int M, int N, int K, int tn, int cuts) {
    const int groups = (M + 7) / 8, rounds = ((N + tn - 1) / tn * cuts + n_cu - 1) / n_cu, steps = ((K / 64 + cuts - 1) / cuts + 2) / 3 * 3;
    const float work = steps * (0.2246f + 0.02967f * groups) + 3.623f + 0.3222f * groups, share = steps * 0.6939f;
    const float t = 0.3942f + fmaxf(rounds * fmaxf(work, share), N * 2.f * K / 13.36e6f);
    return cuts > 1 ? t + gw_row_major.sums_us + gw_row_major.planes * cuts * M * (float)N * 4.f / 4.5e6f : t;
}

/* 128 x 128 tiles: a step takes longer the more CUs take one, and shorter with rows to pad */
static inline float gp_equal_us(int n_cu, int M, int N, int K, int cuts) {
    const int items = (M + 127) / 128 * (N / 128) * cuts, slots = 2 * n_cu, rem = items % slots;
    const float steps = K / cuts / 64, short_rows = 0.3468f * (1.f - (M < 128 ? M : 128) / 128.f);
    float t = 4.158f + items / slots * (steps * 1.737f + 3.122f);
    if (rem) t += steps * ((rem <= n_cu ? 0.8687f + 0.1399f * rem / n_cu : 1.737f) - short_rows) + 3.122f;
    return cuts > 1 ? t + gw_row_major.sums_us + 0.2854f * cuts + 0.7692f * (cuts + 1) * M * (float)N * 4.f / 4.5e6f : t;
}

static inline vt_gemm_plan gp_row_major(int n_cu, int M, int N, int K, int most, float *us) {
    vt_gemm_plan pl = gw_plan(n_cu, gw_row_major, M, N, K, 0, most, us);
    if (pl.cuts == 1) pl.col0 = N;
    if (vt_gemm_rows_ok(M, N, K) && gw_fits((M + 7) / 8 * 8, N, K)) {
        const vt_gemm_plan strips = gp_few_rows(n_cu, N, 0);
        for (int cuts = 1; cuts <= strips.cuts && cuts <= most && cuts <= K / 64; cuts++) {
            const float t = gw_strip_us(n_cu, M, N, K, strips.tn, cuts);
            if (t < *us) { *us = t; pl = strips; pl.cuts = cuts; }
        }
    }
    pl.row_major = 1;
    return pl;
}

#endif /* VT_GEMM_PLANS_H */

"""Plans of the products (vt_gemm_plans.h), walked on the CPU: the header compiled with g++, 256 CUs.  And that the row counts of the tests on
the device run the tiles, whole and cut columns that they are there for."""
import plansupport as P
import test_gpu_codec_attention
import test_gpu_mixed_plans
import test_gpu_prefill_paired_tiles
import test_gpu_prefill_row_counts
import test_gpu_prefill_tiles192
import test_gpu_prefill_tiles384

ROW_MAJOR = r"""
#include <stdio.h>
#include "vt_gemm_plans.h"
/* a plan's tile and strips store the rows that they have room for, those past the last one too: how many that is */
static int padded(const vt_gemm_plan &p, int M) { return p.tm ? p.tm : (M + 7) / 8 * 8; }
int main(void) {
    long long checked = 0, bad = 0, near = 0;
    for (int M = 8; M <= 300; M += M < 66 ? 1 : 31)
        for (long long N = 128; N <= 67108864; N += 128 + N / 300 / 128 * 128)
            for (int K = 64; K <= 4096; K *= 4) {
                float us;
                const vt_gemm_plan p = gp_row_major(256, M, (int)N, K, VT_MAX_CUTS, &us);
                if (!(us < gp_equal_us(256, M, (int)N, K, 1))) continue;         /* 128 x 128 tiles, an address per row */
                checked++;
                const long long bytes = padded(p, M) * N * 4;
                near += bytes > 0x7fffffffll / 2 && bytes <= 0x7fffffffll;
                if (bytes > 0x7fffffffll && bad++ < 5) printf("%d rows, N %lld, K %d: tile %d x %d\n", M, N, K, p.tm, p.tn);
            }
    printf("%lld %lld %lld\n", checked, near, bad);
    return 0;
}
"""


def test_rows_that_a_descriptor_stores():
    """Strips and tiles on row-major weights store through one descriptor: the offset of every row that a tile has room for, those past
    the last one included (which the descriptor's size drops), is a 32-bit number that did not wrap."""
    out = P.run(ROW_MAJOR)
    checked, near, bad = map(int, out.splitlines()[-1].split())
    assert checked > 10000 and near > 100
    assert bad == 0, out


LONG_K = r"""
#include <stdio.h>
#include "vt_gemm_plans.h"
int main(void) {
    long long checked = 0, near = 0, bad = 0;
    for (int M = 8; M <= 300; M += M < 66 ? 1 : 31)
        for (int N = 128; N <= 1024; N += 128)
            for (long long K = 1 << 20; K <= 1 << 26; K += 64 + K / 200 / 64 * 64) {
                float us;
                const vt_gemm_plan p = gp_row_major(256, M, N, (int)K, VT_MAX_CUTS, &us);
                if (!(us < gp_equal_us(256, M, N, (int)K, 1))) continue;
                checked++;
                /* rows of a tile, columns of a wave: what a descriptor covers, 2 K bytes each */
                const int rows = p.tm ? p.tm : (M + 7) / 8 * 8, cols = p.tm ? p.tn / (p.tn < 256 ? 2 : 4) : 32;
                const long long bytes = (rows > cols ? rows : cols) * 2 * K;
                near += bytes > 0x7fffffffll / 2 && bytes <= 0x7fffffffll;
                if (bytes > 0x7fffffffll && bad++ < 5) printf("%d rows, N %d, K %lld: tile %d x %d\n", M, N, K, p.tm, p.tn);
            }
    printf("%lld %lld %lld\n", checked, near, bad);
    return 0;
}
"""


def test_rows_and_weights_that_a_descriptor_loads():
    """The same of what they load: a tile's rows of activations and a wave's rows of weights, K elements of 2 bytes each."""
    out = P.run(LONG_K)
    checked, near, bad = map(int, out.splitlines()[-1].split())
    assert checked > 10000 and near > 100
    assert bad == 0, out


# rows of a prompt -> a product and its plan (plansupport.plans)
BACKBONE = {
    test_gpu_prefill_tiles192: {
        100: [], 300: [], 690: [],
        511: [("q|k|v", "80x192 x 1")], 760: [("down", "96x192 x 2")], 1400: [("output", "96x192 x 1"), ("down", "96x192 x 1")],
        969: [("output", "128x192 x 2"), ("q|k|v", "128x192 all")], 2020: [("output", "128x192 all")]},
    test_gpu_prefill_tiles384: {
        450: [("gate|up", "96x384 all")], 515: [("gate|up", "128x384 all")], 697: [("down", "96x384 x 4")],
        1050: [("gate|up", "96x384 17664 + 6")], 1200: [("down", "128x384 x 3"), ("q|k|v", "128x256 x 1")],
        1450: [("q|k|v", "96x384 all")], 1600: [("gate|up", "128x384 14976 + 2"), ("q|k|v", "128x384 x 1")]},
    test_gpu_prefill_paired_tiles: {
        65: [("q|k|v", "80x256 x 6"), ("gate|up", "80x256 x 3")], 79: [("q|k|v", "80x256 x 6"), ("gate|up", "80x256 x 3")],
        97: [("down", "80x256 x 8")], 129: [("output", "80x256 x 8"), ("gate|up", "80x192 all")], 150: [("gate|up", "80x192 all")],
        160: [("gate|up", "80x192 all")], 161: [("gate|up", "80x256 all")], 225: [("gate|up", "80x256 all")], 240: [("gate|up", "80x256 all")],
        335: [("gate|up", "112x256 all")], 399: [("gate|up", "80x384 all")], 560: [("q|k|v", "80x192 x 1")], 690: [("q|k|v", "80x256 x 1")],
        780: [("down", "112x256 x 3")], 1051: [("q|k|v", "112x256 x 1"), ("down", "112x256 x 2")]},
    test_gpu_mixed_plans: {
        1281: [], 1531: [], 2100: [("q|k|v", "128x384 5760 + 6"), ("gate|up", "128x384 17280 + 4")]},
}
LONG = {2200: [("output", "112x256 x 1"), ("down", "112x256 x 1")], 2500: [("output", "80x384 all"), ("down", "80x384 all")],
        3100: [("q|k|v", "96x384 5760 + 6")], 4200: [("down", "128x384 2688 + 7"), ("k|v", "128x256 1792 + 4")],
        4600: [("output", "128x384 2688 + 5")], 6600: [("q|k|v", "128x384 5376 + 2"), ("down", "96x384 2688 + 3")]}
# frames of a decode -> rows of the stage, product and plan
CODEC = {163: [], 291: [(8, "gate|up", "96x256 7680 + 4")], 350: [(8, "q|k|v", "128x256 2816 + 4")], 512: [(8, "q|k|v", "128x128 all")],
         527: [(4, "upsampling", "128x256 3840 + 4"), (8, "gate|up", "128x256 7936 + 4"), (8, "q|k|v", "128x256 1792 + 1")],
         580: [(8, "waveform", "96x256 1280 + 2")], 1110: [(8, "down", "128x256 768 + 3"), (8, "q|k|v", "96x256 2816 + 2")]}
V_IN_PLACE = {151: "128x128 x 1", 212: "96x256 x 1", 255: "128x256 x 1"}


def test_row_counts_of_the_device_tests():
    cases = []                                # (rows, product, codec), plan
    for module, rows in list(BACKBONE.items()) + [(None, LONG)]:
        assert set(rows) == set(module.ROWS if module else test_gpu_mixed_plans.LONG)
        cases += [((m, product, False), plan) for m in rows for product, plan in rows[m]]
    assert set(CODEC) == set(test_gpu_mixed_plans.FRAMES) and set(V_IN_PLACE) == set(test_gpu_codec_attention.IN_PLACE)
    cases += [((n * f, product, True), plan) for n in CODEC for f, product, plan in CODEC[n]]
    cases += [((8 * n, "q|k|v", True), plan) for n, plan in V_IN_PLACE.items()]
    got = P.plans([c[0] for c in cases])
    assert [(c[0], plan) for c, plan in zip(cases, got)] == cases


def test_no_mixed_products_in_the_chunks():
    """What test_long_prompts_against_chunks compares with: chunks whose columns are all whole or all cut."""
    sizes = {test_gpu_mixed_plans.CHUNK} | {n % test_gpu_mixed_plans.CHUNK for n in test_gpu_mixed_plans.LONG}
    asked = [(m, product, False) for m in sizes if m > 64 for product in P.BACKBONE]
    for case, plan in zip(asked, P.plans(asked)):
        assert "+" not in plan or plan.endswith("+ 1"), (case, plan)


def test_every_tile_is_run_by_a_listed_row_count():
    """All tiles of prompts of 65 to 8192 rows, whole columns, cut ones and gate|up apart."""
    def kinds(asked):
        out = {}
        for (m, product, _), plan in zip(asked, P.plans(asked)):
            tile, _, rest = plan.partition(" ")
            for k in (("whole", "cut") if "+" in plan and not plan.endswith("+ 1") else ("whole",) if rest == "all" or plan.endswith(" 1") else ("cut",)):
                out.setdefault((tile, k, product == "gate|up"), m)
        return out
    products = [p for p in P.BACKBONE if p != "k|v"]
    listed = [m for module in BACKBONE for m in module.ROWS] + test_gpu_mixed_plans.LONG + sum(test_gpu_prefill_row_counts.WIDE, [])
    reached = kinds([(m, p, False) for m in range(65, 8193) for p in products])
    run = kinds([(m, p, False) for m in sorted(listed) for p in products])
    assert not set(reached) - set(run), {k: reached[k] for k in set(reached) - set(run)}

"""Plans of the products (vt_gemm_plans.h), walked on the CPU: the header compiled with g++, 256 CUs."""
import os
import subprocess

import pytest

import vtsupport as S

CSRC = os.path.join(S.ROOT, "voxtral-tts.c_amd", "csrc")


@pytest.fixture(scope="module")
def compiled(tmp_path_factory):
    def run(name, prog):
        d = tmp_path_factory.mktemp(name)
        src, exe = d / "p.cpp", d / "p"
        src.write_text(prog)
        subprocess.check_call(["g++", "-O2", "-Wall", "-Werror", "-Wno-unused-function", "-I", CSRC, "-o", str(exe), str(src)])
        return subprocess.check_output([str(exe)], text=True)
    return run


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


def test_rows_that_a_descriptor_stores(compiled):
    """Strips and tiles on row-major weights store through one descriptor: the offset of every row that a tile has room for, those past
    the last one included (which the descriptor's size drops), is a 32-bit number that did not wrap."""
    out = compiled("rows", ROW_MAJOR)
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


def test_rows_and_weights_that_a_descriptor_loads(compiled):
    """The same of what they load: a tile's rows of activations and a wave's rows of weights, K elements of 2 bytes each."""
    out = compiled("long_k", LONG_K)
    checked, near, bad = map(int, out.splitlines()[-1].split())
    assert checked > 10000 and near > 100
    assert bad == 0, out

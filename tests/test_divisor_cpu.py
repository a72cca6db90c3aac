"""Division by a multiplication (vt_divisor, vt_requests.h), as the product kernels find an item's tile and cut: exact for every number of
items up to the largest, also where the host falls back to a division.  The header compiled with g++."""
import os
import subprocess

import vtsupport as S

CSRC = os.path.join(S.ROOT, "voxtral-tts.c_amd", "csrc")

PROG = r"""
#include <stdio.h>
#include "vt_requests.h"
int main(void) {
    long long n_checked = 0, by_mul = 0;
    const int most[] = {1, 255, 256, 4096, 70000, 3000000, 2000000000};
    for (int d = 1; d <= 5000; d = d < 600 ? d + 1 : d + 37)
        for (unsigned i = 0; i < sizeof most / sizeof most[0]; i++) {
            const vt_divisor v = vt_divisor_of(d, most[i]);
            by_mul += v.m != 0;
            /* every n near a multiple of d, where a wrong quotient shows first, and the ends of the range */
            for (long long q = 0; q * d <= most[i]; q += 1 + (most[i] / d) / 500)
                for (long long n = q * d - 1; n <= q * d + 1; n++)
                    if (n >= 0 && n <= most[i]) { n_checked++; if (vt_div((int)n, v) != n / d) { printf("%lld / %d\n", n, d); return 1; } }
            if (vt_div(most[i], v) != most[i] / d) { printf("%d / %d\n", most[i], d); return 1; }
        }
    printf("%lld %lld\n", n_checked, by_mul);
    return 0;
}
"""


def test_quotients(tmp_path):
    src, exe = tmp_path / "d.cpp", tmp_path / "d"
    src.write_text(PROG)
    subprocess.check_call(["g++", "-O2", "-Wall", "-Werror", "-I", CSRC, "-o", str(exe), str(src)])
    checked, by_mul = map(int, subprocess.check_output([str(exe)]).split())
    assert checked > 100000 and by_mul > 2000

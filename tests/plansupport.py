"""The plans of the products (vt_gemm_plans.h), compiled with g++ and asked on the CPU for 256 CUs."""
import os
import subprocess
import tempfile

import vtsupport as S

CSRC = os.path.join(S.ROOT, "voxtral-tts.c_amd", "csrc")
BACKBONE = {"q|k|v": (6144, 3072, 0), "output": (3072, 4096, 0), "gate|up": (18432, 3072, 1), "down": (3072, 9216, 0),
            "k|v": (2048, 3072, 0)}          # k|v: the last layer of a prompt that only leaves cache rows, more than 64 of them
CODEC = {"input": (1024, 896), "q|k|v": (3072, 1024), "output": (1024, 1024), "gate|up": (8192, 1024), "down": (1024, 4096),
         "upsampling": (4096, 1024), "waveform": (1792, 1024)}

ASK = r"""
#include <stdio.h>
#include "vt_gemm_plans.h"
int main(void) {
    int codec, M, N, K, swiglu;
    while (scanf("%d %d %d %d %d", &codec, &M, &N, &K, &swiglu) == 5) {
        const vt_gemm_plan p = codec ? gp_codec(256, M, N, K) : gp_frag(256, M, N, K, swiglu);
        printf("%d %d %d %d\n", p.tm, p.tn, p.col0, p.cuts);
    }
    return 0;
}
"""
_exe = None


def run(prog, text=""):
    with tempfile.TemporaryDirectory() as d:
        src, exe = os.path.join(d, "p.cpp"), os.path.join(d, "p")
        with open(src, "w") as f:
            f.write(prog)
        subprocess.check_call(["g++", "-O2", "-Wall", "-Werror", "-Wno-unused-function", "-I", CSRC, "-o", exe, src])
        return subprocess.run([exe], input=text, text=True, capture_output=True, check=True).stdout


def plans(asked):
    """[(rows, product, codec?)] -> what each runs on: "96x128 all" (columns in whole tiles), "96x128 x 4" (all columns in 4 K cuts; 1: one
    plane), "96x128 4608 + 3" (whole tiles below column 4608, 3 cuts from there on); "x 96" instead of the tile up to 64 rows"""
    lines = []
    for rows, product, codec in asked:
        n, k, swiglu = CODEC[product] + (0,) if codec else BACKBONE[product]
        lines.append(f"{int(codec)} {rows} {n} {k} {swiglu}")
    out = []
    for (rows, product, codec), line in zip(asked, run(ASK, "\n".join(lines)).splitlines()):
        tm, tn, col0, cuts = map(int, line.split())
        tile = f"{tm}x{tn}" if tm else f"x {tn}"
        n = (CODEC if codec else BACKBONE)[product][0]
        out.append(f"{tile} all" if col0 == n else f"{tile} x {cuts}" if col0 == 0 else f"{tile} {col0} + {cuts}")
    return out

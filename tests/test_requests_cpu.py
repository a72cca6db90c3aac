"""Requests through buffer descriptors that have nothing to bring (vt_requests.h): every one the prefill attention and the linear
layers' row kernel make is either of size 0 at offset 0, or wholly inside the bytes its descriptor covers, scalar offset included,
and these inside the buffer.  The functions are the kernels' own; this test compiles the header with g++ and walks the loops."""
import os
import subprocess

import vtsupport as S

CSRC = os.path.join(S.ROOT, "voxtral-tts.c_amd", "csrc")

PROG = r"""
#include <stdio.h>
#include "vt_requests.h"
static int bad = 0, dead = 0, live = 0;
/* a request for `bytes` from vector offset voff on; room: bytes of the buffer behind the descriptor's base */
static void check(vt_request r, long long voff, long long bytes, long long room, const char *what, int a, int b) {
    if (r.bytes == 0) { dead++; if (r.soff) { bad++; printf("%s %d %d: dead at %d\n", what, a, b, r.soff); } return; }
    live++;
    if (r.bytes > room || r.soff < 0 || voff + r.soff + bytes > r.bytes) { bad++; printf("%s %d %d: %d + %lld of %d, room %lld\n", what, a, b, r.soff, voff, r.bytes, room); }
}
int main(void) {
    const int TILE = 32768;
    /* attention: two waves per residue and four residues, K and V of a tile by themselves; four and two, whole tiles */
    for (int ntiles = 1; ntiles <= 300; ntiles++)
        for (int ns = 2; ns <= 4; ns += 2)
            for (int pz = 0; pz < ns; pz++) {
                const int steps = (ntiles + ns - 1) / ns, kb = ns == 2 ? 32768 : 16384;
                for (int step = 0; step <= steps + 1; step++)
                    for (int from = 0; from < TILE; from += kb)
                        check(vt_tile_request(step * ns + pz, ntiles, TILE, from), 0, kb, (long long)ntiles * TILE, "tile", ntiles, step);
            }
    const int tl = live, td = dead;
    /* linear rows: the four kernels, K in one to three passes, any number of rows per workgroup */
    const int HP[4][2] = {{3, 2}, {2, 2}, {1, 2}, {1, 1}};
    for (int v = 0; v < 4; v++)
        for (int passes = 1; passes <= 3; passes++) {
            const int H = HP[v][0], P = HP[v][1], in_dim = passes * 8 * 64 * H * P;
            for (int rows = 1; rows <= 70; rows++) {
                const int n = (rows + 15) / 16 * passes * P;
                for (int t = 0; t < n + 2; t++)
                    for (int wave = 0; wave < 8; wave++) {
                        const vt_request r = vt_rows_request(t, n, H, P, passes, rows, in_dim, wave);
                        const int first = 16 * r.block;
                        if (first >= rows) { bad++; printf("block %d of %d rows\n", first, rows); }
                        /* the last row that the descriptor holds, all lines of the part; rows behind it lie beyond its size */
                        const int last = (rows - first < 16 ? rows - first : 16) - 1;
                        check(r, (long long)last * in_dim * 2, 128 * H, (long long)(rows - first) * in_dim * 2, "rows", rows, t);
                        if (r.bytes && r.bytes != (last + 1) * in_dim * 2) bad++;
                    }
            }
        }
    printf("%d %d %d %d %d\n", bad, tl, td, live - tl, dead - td);
    return bad != 0;
}
"""


def test_every_request_is_dead_or_in_bounds(tmp_path):
    src, exe = tmp_path / "requests.cc", tmp_path / "requests"
    src.write_text(PROG)
    subprocess.check_call(["g++", "-O1", "-Wall", "-I", CSRC, "-o", str(exe), str(src)])
    run = subprocess.run([str(exe)], text=True, capture_output=True)
    assert run.returncode == 0, run.stdout[-2000:]
    bad, *counts = map(int, run.stdout.split())
    assert bad == 0 and all(c > 0 for c in counts)

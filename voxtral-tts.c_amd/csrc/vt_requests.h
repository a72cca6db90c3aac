/*
 * vt_requests.h - which bytes the kernels' requests through a buffer descriptor ask for where some of them have nothing to
 * bring: the number of requests is fixed (the waits count them), so one for a tile past the last visible one, or for a part past
 * a workgroup's last, still goes out.  Such a request has size 0 AND scalar offset 0: whether the hardware's range check
 * takes the scalar offset into account (and how, where that is the larger one) then makes no difference.  Pure integer
 * functions, compiled for the device by hipcc and for the host by any C++ compiler; a host test walks every request.
 */
#ifndef VT_REQUESTS_H
#define VT_REQUESTS_H

#include "vt_rowsplit.h"

struct vt_request { int block, bytes, soff; };       /* which block of rows; the descriptor's size; the scalar offset */

/* Prefill attention: `from` bytes into tile `tile` of the ntiles that are visible, counted from tile 0 */
VT_HD vt_request vt_tile_request(int tile, int ntiles, int tile_bytes, int from) {
    const bool live = tile < ntiles;
    return vt_request{0, live ? ntiles * tile_bytes : 0, live ? tile * tile_bytes + from : 0};
}

/* Linear layers of a few rows: part t of a workgroup's n, i.e. part t % P of pass t / P % passes over K of a block of 16 of its
 * `rows` weight rows, H lines of 128 bytes per row; counted from the block's first row (t >= n: none) */
VT_HD vt_request vt_rows_request(int t, int n, int H, int P, int passes, int rows, int in_dim, int wave) {
    const bool live = t < n;
    const int block = t / (P * passes), at = t - block * (P * passes), left = rows - 16 * block;
    return vt_request{live ? block : 0, live ? (left < 16 ? left : 16) * in_dim * 2 : 0, live ? ((at / P * 8 + wave) * P + at % P) * 128 * H : 0};
}

/* Division by a number that the host knows: n / d = (n m) >> 32 with m = 2^32 / d + 1 rounded down, exact where n d < 2^32; where that
 * does not hold for every n up to `largest`, and for d = 1, m is 0 and the kernel divides.  (A division by a kernel's argument is a
 * chain of 20 to 30 instructions that run once, in front of a launch's first request.) */
struct vt_divisor { unsigned m; int d; };
VT_HD vt_divisor vt_divisor_of(int d, long long largest) {
    return vt_divisor{d > 1 && largest * d < (1ll << 32) ? (unsigned)((1ull << 32) / (unsigned)d + 1) : 0u, d};
}
VT_HD int vt_div(int n, const vt_divisor &by) { return by.m ? (int)((unsigned long long)(unsigned)n * by.m >> 32) : n / by.d; }

#endif /* VT_REQUESTS_H */

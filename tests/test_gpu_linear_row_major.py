"""Linear layers of more rows than one stream of the weights serves, on the caller's row-major weights: column strips up to 64
rows, tiles of 96 and 128 rows beyond, at the edges of both.  Against float64."""
import numpy as np
import pytest

import hipsupport as H
import vtsupport as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    h = H.Hip(kv_max=8)
    yield h
    h.close()


# strips (N a multiple of 96): groups of 8 rows, the first and the last of one; other widths and from 65 rows on tiles of 128, 192
# and 256 columns, the last rows of a tile; one K step, and K steps that the cuts do not share evenly
@pytest.mark.parametrize("m,n,k", [(8, 384, 704), (17, 768, 3072), (24, 384, 640), (33, 1152, 64), (57, 3072, 1088), (64, 384, 128),
                                   (8, 128, 64), (20, 1024, 3072), (64, 640, 192), (65, 128, 64), (96, 384, 192), (97, 256, 1088),
                                   (128, 768, 320), (129, 9216, 192), (150, 1152, 3072), (300, 640, 4096), (300, 3072, 1088),
                                   (700, 8320, 192), (33, 32768, 128), (110, 640, 320),
                                   # short and long K, few and many columns: strips in 1 to 8 cuts, tiles whole and cut, tiles of 128 x 128
                                   (33, 384, 448), (33, 384, 512), (64, 640, 576), (20, 32768, 448), (65, 128, 1984), (65, 128, 2048), (96, 384, 2112),
                                   (150, 256, 2048), (96, 384, 128), (110, 384, 768), (257, 640, 448), (300, 256, 3072), (300, 256, 3136),
                                   (512, 512, 2048), (512, 512, 2112), (300, 8320, 256), (16, 12288, 4096), (40, 131072, 64), (192, 5120, 1024)])
@pytest.mark.parametrize("noalloc", [False, True])
def test_rows(hip, m, n, k, noalloc):
    W = S.bf16_normal((n, k), 5000 + n + k)
    x = S.f32_normal((m, k), 5100 + m + k)
    want = x.astype(np.float64) @ S.bf16_to_f32(W).astype(np.float64).T
    size = np.abs(x).astype(np.float64) @ np.abs(S.bf16_to_f32(W)).astype(np.float64).T
    y0 = np.full((m + 1, n), 7.0, np.float32)
    dx, dW, dy = H.DevBuf.from_numpy(hip.lib, x), H.DevBuf.from_numpy(hip.lib, W), H.DevBuf.from_numpy(hip.lib, y0)
    if noalloc:
        assert hip.lib.tts_hip_linear_bf16_noalloc(dy.ptr, dx.ptr, m, k, n, dW.ptr) == 0
    else:
        hip.lib.tts_hip_linear_bf16(dy.ptr, dx.ptr, None, m, k, n, dW.ptr)
    hip.lib.tts_hip_sync()
    hip.check()
    got = dy.to_numpy(np.float32, (m + 1, n))
    assert np.all(got[m] == 7.0)
    # x as two bf16 planes: 2^-16; fp32 sums in any order: 2^-24 per addition, of which the deepest chain has K / 16 + 40
    tol = (2.0 ** -24 * (k / 16 + 40) + 2.0 ** -16) * size
    assert np.all(np.abs(got[:m] - want) <= tol), float((np.abs(got[:m] - want) / tol).max())
    for b in (dx, dW, dy):
        b.free()


# Columns of which a tile's rows are more than 32 bits of bytes apart: 2 and 4 GiB of rows that exist; fewer rows, whose tiles have room for
# rows past them at offsets beyond 2^32; the last number of columns that tiles of 96 rows can store, and the first that they cannot.
@pytest.mark.parametrize("m,reps", [(64, 99), (128, 99), (8, 196), (16, 196), (40, 196), (8, 65), (70, 65), (70, 66)])
def test_rows_of_more_than_32_bits_of_bytes(hip, m, reps):
    """The weights repeat.  Bound as above."""
    n0, k = 84736, 64
    n = n0 * reps
    W = S.bf16_normal((n0, k), 5301)
    x = S.f32_normal((m, k), 5302)
    want = x.astype(np.float64) @ S.bf16_to_f32(W).astype(np.float64).T
    size = np.abs(x).astype(np.float64) @ np.abs(S.bf16_to_f32(W)).astype(np.float64).T
    dx, dW = H.DevBuf.from_numpy(hip.lib, x), H.DevBuf.from_numpy(hip.lib, np.tile(W, (reps, 1)))
    dy = H.DevBuf.from_numpy(hip.lib, np.full((m + 1, n), 7.0, np.float32))
    print(f"{m} rows of {n} columns", flush=True)
    hip.lib.tts_hip_linear_bf16(dy.ptr, dx.ptr, None, m, k, n, dW.ptr)
    hip.lib.tts_hip_sync()
    hip.check()
    got = dy.to_numpy(np.float32, (m + 1, n))
    assert np.all(got[m] == 7.0)
    tol = (2.0 ** -24 * (k / 16 + 40) + 2.0 ** -16) * size
    for row in range(m) if m < 64 else sorted({0, 1, 31, 32, 63, m // 2, m - 2, m - 1}):
        assert np.all(np.abs(got[row].reshape(reps, n0) - want[row]) <= tol[row]), row
    for b in (dx, dW, dy):
        b.free()

"""Linear layers on caller-owned weights at the edges of their kernels: 1 row beside 2, the 16 rows of a workgroup (8 and 16
used to go to the matrix cores' bf16 planes), K in one pass and in several, weight rows that do not fill a block of 16 or a
workgroup, K of up to 64 and shapes no kernel but the general one takes.  Against float64."""
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


@pytest.mark.parametrize("n,k", [(36, 3072), (1000, 4096), (9216, 3072), (3072, 9216), (17, 256), (300, 1280), (3072, 36), (257, 64), (5, 1), (36, 100),
                                 # each instance (K / 512 a multiple of 4, even, odd) with more than 16 rows per workgroup at 49 rows, in passes over K
                                 (1111, 8192), (1300, 1024), (1200, 5120), (1100, 2560)])
@pytest.mark.parametrize("m", [1, 2, 7, 15, 16, 17, 49])
def test_rows(hip, m, n, k):
    W = S.bf16_normal((n, k), 4000 + n + k)
    x = S.f32_normal((m, k), 4100 + m + k)
    want = x.astype(np.float64) @ S.bf16_to_f32(W).astype(np.float64).T
    size = np.abs(x).astype(np.float64) @ np.abs(S.bf16_to_f32(W)).astype(np.float64).T
    dx, dW, dy = H.DevBuf.from_numpy(hip.lib, x), H.DevBuf.from_numpy(hip.lib, W), H.DevBuf(hip.lib, m * n * 4)
    hip.lib.tts_hip_linear_bf16(dy.ptr, dx.ptr, None, m, k, n, dW.ptr)
    hip.lib.tts_hip_sync()
    hip.check()
    got = dy.to_numpy(np.float32, (m, n))
    # fp32 products and sums in any order: 2^-24 per addition, of which the deepest chain has K / 32 + 40; with more
    # than 16 rows or 12 of 4096 x enters as 16 bits where N is a multiple of 128 and K of 64
    planes = (m > 16 or m * k > 12 * 4096) and n % 128 == 0 and k % 64 == 0
    tol = (2.0 ** -24 * (k / 32 + 40) + (2.0 ** -16 if planes else 0.0)) * size
    assert np.all(np.abs(got - want) <= tol), float((np.abs(got - want) / tol).max())
    for b in (dx, dW, dy):
        b.free()


def test_a_row_with_infinities_stays_alone(hip):
    m, n, k = 11, 100, 512
    W, x = S.bf16_normal((n, k), 1), S.f32_normal((m, k), 2)
    clean = x.copy()
    x[4, 5], x[4, 300] = np.inf, -np.inf
    out = []
    for a in (clean, x):
        y = np.zeros((m, n), np.float32)
        hip.lib.tts_hip_linear_bf16(y.ctypes.data, a.ctypes.data, W.ctypes.data, m, k, n, None)
        hip.check()
        out.append(y)
    others = [i for i in range(m) if i != 4]
    assert np.array_equal(out[0][others], out[1][others]) and not np.isfinite(out[1][4]).any()

"""Linear layers whose sums are fp32: no further from float64 than the order they are measured against, a wave's 64 lanes (each
every 64th group of the reduction index, in turn) and a tree over the lanes, evaluated in fp32 on the CPU."""
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


def lanes_and_tree(x, W, group):
    """group consecutive k per lane and turn; x [m, k], W [n, k] fp32 -> [m, n]"""
    (m, k), n = x.shape, W.shape[0]
    pad = -k % (64 * group)
    x, W = (np.pad(a, ((0, 0), (0, pad))).reshape(a.shape[0], -1, 64, group) for a in (x, W))
    acc = np.zeros((m, n, 64), np.float32)
    for t in range(x.shape[1]):
        for j in range(group):
            acc = (x[:, None, t, :, j].astype(np.float64) * W[None, :, t, :, j] + acc).astype(np.float32)
    while acc.shape[2] > 1:
        half = acc.shape[2] // 2
        acc = acc[:, :, :half] + acc[:, :, half:]
    return acc[:, :, 0]


def compare(hip, m, n, k, group):
    W = S.bf16_normal((n, k), 7000 + n + k)
    x = S.f32_normal((m, k), 7100 + m + k)
    Wf = S.bf16_to_f32(W)
    exact = x.astype(np.float64) @ Wf.astype(np.float64).T
    dx, dW, dy = H.DevBuf.from_numpy(hip.lib, x), H.DevBuf.from_numpy(hip.lib, W), H.DevBuf(hip.lib, m * n * 4)
    hip.lib.tts_hip_linear_bf16(dy.ptr, dx.ptr, None, m, k, n, dW.ptr)
    hip.lib.tts_hip_sync()
    hip.check()
    got = dy.to_numpy(np.float32, (m, n))
    for b in (dx, dW, dy):
        b.free()
    err, ref = (np.sqrt(np.mean((a - exact) ** 2)) for a in (got, lanes_and_tree(x, Wf, group)))
    # both are samples over m n outputs; an error's own spread is about its size, so the ratio's is sqrt(2 / (m n)): five of these
    assert err <= ref * (1.0 + 5.0 * np.sqrt(2.0 / (m * n))), (err, ref, err / ref)


@pytest.mark.parametrize("m,n,k", [(2, 3072, 36), (5, 3072, 64), (300, 300, 36), (40, 257, 63), (7, 1000, 16), (9, 999, 50), (33, 200, 5)])
def test_short_rows(hip, m, n, k):
    compare(hip, m, n, k, 1)


# the fp32 matrix instructions: each kernel (K / 512 a multiple of 6, of 4, even, odd), one pass over K and several
@pytest.mark.parametrize("m,n,k", [(16, 36, 3072), (8, 50, 9216), (12, 60, 4096), (8, 70, 2048), (9, 100, 1024), (16, 50, 5120), (20, 100, 512),
                                   (8, 60, 2560), (4, 3072, 3072)])
def test_a_few_rows(hip, m, n, k):
    compare(hip, m, n, k, 8)

"""Causal attention of a prompt at the edges of its kernels (16 queries per workgroup up to 1200 rows, 32 beyond): a block
with one query more, key tiles that begin before the first new row, and scores that grow along the keys, so that the
running maximum changes with every tile.  Against float64."""
import ctypes as C

import numpy as np
import pytest

import hipsupport as H
import vtsupport as S

pytestmark = pytest.mark.gpu

HEADS = (0, 13, 31)


def reference(Q, K, V, start, scale, head):
    q = Q[:, 128 * head:128 * head + 128].astype(np.float64)
    k, v = (a[:, 128 * (head // 4):128 * (head // 4) + 128].astype(np.float64) for a in (K, V))
    s = q @ k.T * scale
    s[np.arange(K.shape[0])[None, :] > start + np.arange(Q.shape[0])[:, None]] = -np.inf
    p = np.exp(s - s.max(axis=1, keepdims=True))
    return p @ v / p.sum(axis=1, keepdims=True), np.abs(p) @ np.abs(v) / p.sum(axis=1, keepdims=True)


@pytest.mark.parametrize("seq,start,growth", [(8, 0, 0.0), (16, 31, 0.0), (17, 15, 0.7), (209, 3, 0.02), (1200, 0, 0.3),
                                              (1201, 0, 0.0), (1217, 45, 0.3), (1231, 0, 0.02)])
def test_edges(seq, start, growth):
    print(f"attention of {seq} rows behind {start}, growth {growth}", flush=True)
    scale = 1.0 / np.sqrt(128.0)
    Q, K, V = (S.f32_normal((n, d), 900 + seq + i) for i, (n, d) in enumerate(((seq, S.Q_DIM), (start + seq, S.KV_DIM), (start + seq, S.KV_DIM))))
    Q[:, ::128] = 2.0                              # dim 0 of a head: a score that grows by `growth` per key
    K[:, ::128] = (growth / 2.0 / scale * np.arange(start + seq, dtype=np.float32))[:, None]
    hip = H.Hip(kv_max=8)
    try:
        dQ, dK, dV = (H.DevBuf.from_numpy(hip.lib, a) for a in (Q, K, V))
        dO = H.DevBuf(hip.lib, Q.nbytes)
        hip.lib.tts_hip_causal_attention_prefill(dO.ptr, dQ.ptr, dK.ptr, dV.ptr, seq, start, S.HEADS, S.KV_HEADS, S.HEAD_DIM, C.c_float(scale))
        hip.lib.tts_hip_sync()
        hip.check()
        got = dO.to_numpy(np.float32, Q.shape)
        assert np.all(np.isfinite(got))
        for head in HEADS:
            ref, size = reference(Q, K, V, start, scale, head)
            # Operands hold 16 bits, 2^-17 of themselves each, V and P with three products of which one is left out (2^-18): 2^-15
            # of the terms' sizes.  A score's error is 2^-15 of its own terms, |q| |k| scale, and exp makes it a relative one
            # of that size; the growing part of a score is up to growth * keys, of which all keys near the maximum carry the
            # same rounding of q (2, exact) and their own of k.
            terms = np.abs(Q[:, 128 * head:128 * head + 128]).astype(np.float64) @ np.abs(K[:, 128 * (head // 4):128 * (head // 4) + 128]).astype(np.float64).T * scale
            terms[np.arange(start + seq)[None, :] > start + np.arange(seq)[:, None]] = 0.0      # keys that a row does not see
            tol = (2.0 ** -15 * (1.0 + 2.0 * terms.max(axis=1)))[:, None] * size
            bad = np.abs(got[:, 128 * head:128 * head + 128] - ref) > tol
            assert not bad.any(), (head, np.argwhere(bad)[:3], (np.abs(got[:, 128 * head:128 * head + 128] - ref) / tol).max())
        for b in (dQ, dK, dV, dO):
            b.free()
    finally:
        hip.close()

"""Weights uploaded from device memory.  Such copies return before they are made, and the kernels that lay the weights out run on
another stream: with two dozen large copies queued in front, every layout has to wait for them.  Bit-equal to an upload from host memory."""
import ctypes as C

import numpy as np
import pytest

import hipsupport as H
import vtsupport as S

pytestmark = pytest.mark.gpu

BUSY_BYTES, BUSY_COPIES = 1 << 30, 24          # about 0.5 ms each


def results(hip):
    hip.pos = 0
    out = [hip.llm_forward(S.f32_normal(S.DIM, 81))]          # the row-major matrices and the final norm
    for n in (37, 200):                                       # the fragment-order copies
        hip.pos = 0
        out.append(hip.llm_prefill(S.f32_normal((n, S.DIM), 80 + n), want_x=True))
    return out


def test_backbone_from_device_memory():
    hip = H.Hip(kv_max=256)
    libhip = C.CDLL("libamdhip64.so.7")
    try:
        layers, norm = [S.Layer(13), S.Layer(14)], S.norm_weight(S.DIM, 96)
        hip.upload_decoder(layers, norm, 2)
        want = results(hip)
        for l in layers:                       # other weights in the places that the next upload gets
            for name in ("wq", "wk", "wv", "wo", "w1", "w2", "w3"):
                setattr(l, name, np.ascontiguousarray(getattr(l, name)[::-1]))
        hip.upload_decoder(layers, norm * 2, 2)
        assert not np.array_equal(results(hip)[0], want[0])
        bufs, structs = [], []
        for l in (S.Layer(13), S.Layer(14)):
            dev = [H.DevBuf.from_numpy(hip.lib, a) for a in (l.wq, l.wk, l.wv, l.wo, l.attention_norm, l.w1, l.w2, l.w3, l.ffn_norm)]
            bufs += dev
            structs.append(type(H.host_layer(l))(*(b.ptr for b in dev)))
        bufs.append(H.DevBuf.from_numpy(hip.lib, norm))
        busy = [H.DevBuf(hip.lib, BUSY_BYTES) for _ in range(2)]

        def queue():
            for _ in range(BUSY_COPIES):
                assert libhip.hipMemcpyAsync(C.c_void_p(busy[0].ptr), C.c_void_p(busy[1].ptr), C.c_size_t(BUSY_BYTES), C.c_int(3), None) == 0

        hip.close()
        hip = H.Hip(kv_max=256)                # (to free what an earlier upload left would wait for the queue)
        for i, s in enumerate(structs):
            queue()
            assert hip.lib.tts_hip_upload_llm_layer(i, C.byref(s)) == 0
        queue()
        assert hip.lib.tts_hip_upload_llm_norm(bufs[-1].ptr) == 0
        got = results(hip)
        hip.check()
        same = [np.array_equal(a.view(np.uint32), b.view(np.uint32)) for a, b in zip(want, got)]
        assert same == [True] * 3
        for b in bufs + busy:
            b.free()
    finally:
        hip.close()

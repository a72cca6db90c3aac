"""An acoustic frame takes its hidden state and noise from pageable memory or from the device, also while the work that makes
them is still on its way on the library's stream; the codec its codes likewise."""
import ctypes as C

import numpy as np
import pytest

import codecsupport as K
import hipsupport as H
import vtsupport as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    h = H.Hip(kv_max=8)
    h.upload_acoustic(S.Acoustic(50))
    yield h
    h.close()


def frame(hip, hidden, x0):
    codes, x = np.zeros(S.CODES, np.int32), np.zeros(S.ACOUSTIC_DIM, np.float32)
    hip.lib.tts_hip_acoustic_frame(codes.ctypes.data, hidden, x0, x.ctypes.data)
    hip.check()
    return codes, x


def test_hidden_state_and_noise_still_being_written(hip):
    lib = hip.lib
    big = H.DevBuf.from_numpy(lib, S.bf16_normal((32768, S.DIM), 3))
    W, Wx = H.DevBuf.from_numpy(lib, S.bf16_normal((S.DIM, S.DIM), 1)), H.DevBuf.from_numpy(lib, S.bf16_normal((S.ACOUSTIC_DIM, S.DIM), 2))
    v = H.DevBuf.from_numpy(lib, S.f32_normal(S.DIM, 4))
    out, dh, dx = H.DevBuf(lib, 32768 * 4), H.DevBuf.from_numpy(lib, np.zeros(S.DIM, np.float32)), H.DevBuf.from_numpy(lib, np.zeros(S.ACOUSTIC_DIM, np.float32))
    for _ in range(60):                                   # some milliseconds of work in front
        lib.tts_hip_linear_bf16(out.ptr, v.ptr, None, 1, S.DIM, 32768, big.ptr)
    lib.tts_hip_linear_bf16(dh.ptr, v.ptr, None, 1, S.DIM, S.DIM, W.ptr)
    lib.tts_hip_linear_bf16(dx.ptr, v.ptr, None, 1, S.DIM, S.ACOUSTIC_DIM, Wx.ptr)
    got = frame(hip, dh.ptr, dx.ptr)
    h, x = dh.to_numpy(np.float32, (S.DIM,)), dx.to_numpy(np.float32, (S.ACOUSTIC_DIM,))
    assert np.abs(h).max() > 0 and np.abs(x).max() > 0
    want = frame(hip, h.ctypes.data, x.ctypes.data)
    mixed = frame(hip, dh.ptr, x.ctypes.data)
    for g in (got, mixed):
        assert np.array_equal(g[0], want[0]) and np.array_equal(g[1], want[1])
    for b in (big, W, Wx, v, out, dh, dx):
        b.free()


def test_codes_on_the_device(hip):
    hc = K.HostCodec(8, distinct_layers=2)
    cs = hc.struct()
    assert hip.lib.tts_hip_upload_codec_weights(C.addressof(cs)) == 0, hip.lib.tts_hip_last_error()
    codes = np.ascontiguousarray(K.random_codes(5, 65), np.int32)
    dev = H.DevBuf.from_numpy(hip.lib, codes)
    res = []
    for p in (codes.ctypes.data, dev.ptr):
        out, n = C.POINTER(C.c_float)(), C.c_int(0)
        hip.lib.tts_hip_codec_decode(p, 5, C.byref(out), C.byref(n))
        hip.check()
        res.append(np.ctypeslib.as_array(out, shape=(n.value,)).copy())
        C.CDLL(None).free(C.cast(out, C.c_void_p))
    assert np.array_equal(res[0], res[1])
    dev.free()

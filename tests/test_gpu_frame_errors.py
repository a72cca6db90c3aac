"""A frame that ends in an error has left the stream when the call is back: what its kernels read in pinned memory may be
filled again.  The error is one that the calling thread's HIP runtime holds already, and other work stands in front."""
import time

import numpy as np
import pytest

import hipsupport as H
import vtsupport as S

pytestmark = pytest.mark.gpu


def test_an_error_comes_back_behind_the_work():
    hip = H.Hip(kv_max=8)
    lib = hip.lib
    try:
        hip.upload_acoustic(S.Acoustic(50))
        W, v, out = H.DevBuf(lib, 131072 * S.DIM * 2), H.DevBuf(lib, S.DIM * 4), H.DevBuf(lib, 131072 * 4)
        h, x0 = S.f32_normal(S.DIM, 4), S.f32_normal(S.ACOUSTIC_DIM, 5)
        codes = np.full(S.CODES, -7, np.int32)

        def call():
            lib.tts_hip_acoustic_frame(codes.ctypes.data, h.ctypes.data, x0.ctypes.data, None)

        call()
        hip.check()
        codes[:] = -7
        lib.tts_hip_sync()
        start = time.perf_counter()
        for _ in range(200):                              # about 20 ms
            lib.tts_hip_linear_bf16(out.ptr, v.ptr, None, 1, S.DIM, 131072, W.ptr)
        before = lib.tts_hip_error_count()
        assert lib.hipSetDevice(1 << 20) != 0             # refused; the runtime remembers it
        call()
        back = time.perf_counter()
        lib.tts_hip_sync()
        end = time.perf_counter()
        assert lib.tts_hip_error_count() > before and np.all(codes == -7)
        assert end - back < (end - start) / 4, (back - start, end - back)
        hip.err0 = lib.tts_hip_error_count()
        call()
        hip.check()
        assert np.all(codes >= 0)
        for b in (W, v, out):
            b.free()
    finally:
        hip.close()

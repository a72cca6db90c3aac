"""Input rows of a prefill in pageable memory, which cross in pieces of 64 through pinned memory from 97 rows on: the same rows in
pageable, pinned and device memory leave the same residual stream and cache rows, bit for bit, at the edges of a piece and of that rule, with a
longer prompt and a shorter one behind it, and the caller's buffer is free behind the call."""
import ctypes as C

import numpy as np
import pytest

import hipsupport as H
import vtsupport as S

pytestmark = pytest.mark.gpu

ROWS = [96, 97, 128, 129, 300, 2048, 2049, 200]


def test_rows_from_any_memory():
    hip = H.Hip(kv_max=2100)
    libhip = C.CDLL("libamdhip64.so")
    try:
        hip.upload_decoder([S.Layer(11)], S.norm_weight(S.DIM, 98), 1)
        for n in ROWS:
            print(f"prefill of {n} rows", flush=True)
            e = S.f32_normal((n, S.DIM), 60 + n)
            pinned = C.c_void_p()
            assert libhip.hipHostMalloc(C.byref(pinned), C.c_size_t(e.nbytes), C.c_uint(0)) == 0
            C.memmove(pinned, e.ctypes.data, e.nbytes)
            dev = H.DevBuf.from_numpy(hip.lib, e)
            got = []
            for ptr in (e.ctypes.data, pinned.value, dev.ptr):
                x = np.zeros_like(e)
                hip.lib.tts_hip_llm_prefill_out(ptr, n, 0, x.ctypes.data)
                if ptr == e.ctypes.data:
                    e[:] = np.nan
                hip.check()
                k, v = hip.kv()
                got.append((x, k[0, :n].copy(), v[0, :n].copy()))
            assert np.isfinite(got[0][0]).all()
            for other in got[1:]:
                for a, b in zip(got[0], other):
                    assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), n
            dev.free()
            assert libhip.hipHostFree(pinned) == 0
    finally:
        hip.close()

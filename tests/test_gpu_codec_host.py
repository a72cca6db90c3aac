"""The codec's host entry returns what the device entry computes, sample for sample: lengths at which the waveform leaves in
one part and in two, in sixteen (the most), and a short one behind a long one; the codes given in memory that is overwritten
as soon as the call is back."""
import ctypes as C

import numpy as np
import pytest

import codecsupport as K
import hipsupport as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def codec():
    hc = K.HostCodec(8, distinct_layers=2)
    cs = hc.struct()
    hip = H.Hip(kv_max=8)
    assert hip.lib.tts_hip_upload_codec_weights(C.addressof(cs)) == 0, hip.lib.tts_hip_last_error()
    yield hip
    hip.close()


@pytest.mark.parametrize("n_frames", [1, 127, 128, 129, 1031, 3])
def test_host_entry_is_the_device_entry(codec, n_frames):
    print(f"codec of {n_frames} frames", flush=True)
    lib = codec.lib
    codes = np.ascontiguousarray(K.random_codes(n_frames, 60 + n_frames), np.int32)
    d_codes, d_out = H.DevBuf.from_numpy(lib, codes), H.DevBuf(lib, n_frames * 1920 * 4)
    assert lib.tts_hip_codec_decode_device(d_codes.ptr, n_frames, d_out.ptr) == 0
    lib.tts_hip_sync()
    want = d_out.to_numpy(np.float32, (n_frames * 1920,))
    out, n = C.POINTER(C.c_float)(), C.c_int(0)
    lib.tts_hip_codec_decode(codes.ctypes.data, n_frames, C.byref(out), C.byref(n))
    codes[:] = 0
    codec.check()
    assert n.value == n_frames * 1920
    got = np.ctypeslib.as_array(out, shape=(n.value,)).copy()
    C.CDLL(None).free(C.cast(out, C.c_void_p))
    assert np.array_equal(want, got)
    d_codes.free()
    d_out.free()

"""The frame entry points without one of the buffers they need: an error is recorded in front of any work (no codes, no
latent, no row of the cache is written), and the next good call gives what it gave before."""
import numpy as np
import pytest

import hipsupport as H
import vtsupport as S
from test_gpu_frame_loop import AUDIO_ROWS, offsets

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    h = H.Hip(kv_max=8)
    h.upload_decoder([S.Layer(1)], S.norm_weight(S.DIM, 99), 1)
    h.upload_acoustic(S.Acoustic(50))
    table = S.bf16_normal((AUDIO_ROWS, S.DIM), 4242, 0.05)
    assert h.lib.tts_hip_upload_audio_embeddings(table.ctypes.data, AUDIO_ROWS, offsets().ctypes.data) == 0
    yield h
    h.close()


def refused(hip, call):
    before = hip.lib.tts_hip_error_count()
    call()
    hip.lib.tts_hip_sync()
    assert hip.lib.tts_hip_error_count() == before + 1 and b"NULL argument" in hip.lib.tts_hip_last_error()
    hip.err0 = before + 1


@pytest.mark.parametrize("missing", ["codes", "hidden", "x0"])
def test_acoustic_frame(hip, missing):
    h, x0 = S.f32_normal(S.DIM, 4), S.f32_normal(S.ACOUSTIC_DIM, 5)
    want = hip.acoustic_frame(h, x0)
    codes, x = np.full(S.CODES, -7, np.int32), np.full(S.ACOUSTIC_DIM, 7.0, np.float32)
    ptr = {"codes": codes.ctypes.data, "hidden": h.ctypes.data, "x0": x0.ctypes.data}
    ptr[missing] = None
    refused(hip, lambda: hip.lib.tts_hip_acoustic_frame(ptr["codes"], ptr["hidden"], ptr["x0"], x.ctypes.data))
    assert np.all(codes == -7) and np.all(x == 7.0)
    got = hip.acoustic_frame(h, x0)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("missing", ["codes", "embed", "x0"])
def test_generate_frame(hip, missing):
    x0, embed = S.f32_normal(S.ACOUSTIC_DIM, 5), S.f32_normal(S.DIM, 6)
    hip.set_kv(*(np.zeros((26, 8, S.KV_DIM), np.float32) for _ in range(2)))
    d_embed = H.DevBuf.from_numpy(hip.lib, embed)
    codes = np.full(S.CODES, -7, np.int32)
    ptr = {"codes": codes.ctypes.data, "embed": d_embed.ptr, "x0": x0.ctypes.data}
    ptr[missing] = None
    refused(hip, lambda: hip.lib.tts_hip_generate_frame(ptr["codes"], ptr["embed"], ptr["x0"], 0))
    assert np.all(codes == -7) and np.array_equal(d_embed.to_numpy(np.float32, (S.DIM,)), embed)
    assert not any(a.any() for a in hip.kv())
    hip.lib.tts_hip_generate_frame(codes.ctypes.data, d_embed.ptr, x0.ctypes.data, 0)
    hip.check()
    assert np.all(codes >= 0) and hip.kv()[0][0, 0].any()
    d_embed.free()

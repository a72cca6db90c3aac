"""The codec's products run on two fp16 planes per fp32 operand, each row scaled by a power of two, on tiles and K
cuts that follow the row count.  Frame counts whose four stages (1, 2, 4, 8 rows a frame) fall on the edges of the
tiles (16, 32, 48, 64 rows of the few-row kernel, then 96- and 128-row tiles), and magnitudes far outside the
range of fp16.  The bound: an operand is carried to 2^-23, a product's left-out term is at most 2^-22 of it, and the
sums are fp32 as on the CPU, whose own sequential sums differ from these by a few 1e-6 of the waveform's rms
(measured 4e-6 in l2, 2e-5 at most per sample); four times that."""
import ctypes as C

import numpy as np
import pytest

import codecsupport as K
import hipsupport as H
import vtsupport as S
from test_gpu_codec import hip_decode

pytestmark = pytest.mark.gpu


def close(ref, got):
    rms = float(np.sqrt(np.mean(ref.astype(np.float64) ** 2)))
    d = (ref.astype(np.float64) - got.astype(np.float64))
    assert np.isfinite(got).all()
    assert np.sqrt(np.mean(d ** 2)) <= 1.6e-5 * rms and np.abs(d).max() <= 1e-4 * rms, (np.sqrt(np.mean(d ** 2)) / rms, np.abs(d).max() / rms)


@pytest.fixture(scope="module")
def session():
    S.oracle().orc_set_threads(16)
    hc = K.HostCodec(8, distinct_layers=2)
    cs = hc.struct()
    hip = H.Hip(kv_max=8)
    assert hip.lib.tts_hip_upload_codec_weights(C.addressof(cs)) == 0, hip.lib.tts_hip_last_error()
    yield hip, cs
    hip.close()
    S.oracle().orc_set_threads(1)


@pytest.mark.parametrize("n_frames", [2, 4, 6, 8, 9, 12, 13, 16, 17, 24, 25, 32, 33, 48, 49, 65])
def test_row_counts_at_the_edges_of_the_tiles(session, n_frames):
    hip, cs = session
    codes = K.random_codes(n_frames, 500 + n_frames)
    print(f"codec of {n_frames} frames", flush=True)
    close(K.oracle_decode(cs, codes), hip_decode(hip, codes))


def test_magnitudes_outside_the_range_of_fp16():
    """2^40 in one upsampling convolution and 2^-40 in the next (the residual stream between them runs at 1e12), rows
    of the gate|up matrices apart by 2^20, and an all-zero row."""
    S.oracle().orc_set_threads(16)
    hc = K.HostCodec(9, distinct_layers=1)
    for conv, f in ((hc.stage_convs[0], 2.0 ** 40), (hc.stage_convs[1], 2.0 ** -40)):
        conv.weight *= np.float32(f)
        conv.bias *= np.float32(f)
    l = hc.layers[0]
    l.w1[::7] *= np.float32(2.0 ** -20)
    l.w3[3] = 0.0
    cs = hc.struct()
    hip = H.Hip(kv_max=8)
    try:
        assert hip.lib.tts_hip_upload_codec_weights(C.addressof(cs)) == 0, hip.lib.tts_hip_last_error()
        for n in (5, 20):
            codes = K.random_codes(n, 40 + n)
            close(K.oracle_decode(cs, codes), hip_decode(hip, codes))
    finally:
        hip.close()
        S.oracle().orc_set_threads(1)

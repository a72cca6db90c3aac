"""Products that have columns in whole tiles beside columns in K cuts (vt_gemm_plan with 0 < col0 < N), which the
kernels behind them sum apart.  At 256 CUs the codec's q|k|v has both from 161 frames on, the output convolution from
289, the upsampling products from 513; the backbone's q|k|v at 1281 to 1531 rows, with the boundary among the k
columns.  Against the oracle."""
import ctypes as C

import numpy as np
import pytest

import codecsupport as K
import hipsupport as H
import vtsupport as S
from test_gpu_codec import hip_decode
from test_gpu_codec_planes import close
from test_gpu_prefill_mfma import _prefill_case

pytestmark = pytest.mark.gpu

# The decoder is causal and sees 17 frames back (windows of 2, 4, 8 and 16 tokens in two layers each, the convolutions'
# taps): from its frame 18 on a slice decodes to the samples of the whole.
SEEN, SLICE = 18, 23


@pytest.fixture(scope="module")
def codec():
    S.oracle().orc_set_threads(16)
    hc = K.HostCodec(8, distinct_layers=2)
    cs = hc.struct()
    hip = H.Hip(kv_max=8)
    assert hip.lib.tts_hip_upload_codec_weights(C.addressof(cs)) == 0, hip.lib.tts_hip_last_error()
    yield hip, cs
    hip.close()
    S.oracle().orc_set_threads(1)


@pytest.mark.parametrize("n_frames", [163, 291, 527])
def test_codec(codec, n_frames):
    hip, cs = codec
    codes = K.random_codes(n_frames, 800 + n_frames)
    got = hip_decode(hip, codes).reshape(n_frames, -1)
    for at in (0, n_frames // 2, n_frames - SLICE):
        print(f"codec of {n_frames} frames, slice at {at}", flush=True)
        first = SEEN if at else 0
        ref = K.oracle_decode(cs, codes[at:at + SLICE]).reshape(SLICE, -1)[first:]
        close(ref, got[at + first:at + SLICE])


@pytest.mark.parametrize("rows", [1281, 1531])
def test_prefill(rows):
    print(f"prefill of {rows} rows", flush=True)
    _prefill_case(1, [rows], rows + 4, lambda n: range(0, n, 5))

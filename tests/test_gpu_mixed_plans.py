"""Products that have columns in whole tiles beside columns in K cuts (vt_gemm_plan with 0 < col0 < N), which the
kernels behind them sum apart: the backbone's q|k|v and gate|up from 2049 rows on, with the boundary among the v columns, its output and
down products and the last layer's k|v at some lengths above 4096; the codec's gate|up (291 frames), q|k|v (350), third upsampling product (527),
waveform (580) and down product (1110).  512 frames have all columns of the last stage's q|k|v in whole tiles, where the attention reads v.  Which plans these
are: test_plans_cpu.py.  Against the oracle, the longest prompts against the same rows in chunks of 700, whose plans have no such product."""
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


FRAMES = [163, 291, 350, 512, 527, 580, 1110]


@pytest.mark.parametrize("n_frames", FRAMES)
def test_codec(codec, n_frames):
    hip, cs = codec
    codes = K.random_codes(n_frames, 800 + n_frames)
    got = hip_decode(hip, codes).reshape(n_frames, -1)
    for at in (0, n_frames // 2, n_frames - SLICE):
        print(f"codec of {n_frames} frames, slice at {at}", flush=True)
        first = SEEN if at else 0
        ref = K.oracle_decode(cs, codes[at:at + SLICE]).reshape(SLICE, -1)[first:]
        close(ref, got[at + first:at + SLICE])


ROWS = [1281, 1531, 2100]


@pytest.mark.parametrize("rows", ROWS)
def test_prefill(rows):
    print(f"prefill of {rows} rows", flush=True)
    _prefill_case(1, [rows], rows + 4, lambda n: range(0, n, 5))


# 2200, 2500 and 6600 rows also have tiles that shorter prompts do not take: 112 x 256 and 80 x 384 whole, 96 x 384 whole beside cuts
LONG, CHUNK = [2200, 2500, 3100, 4200, 4600, 6600], 700


@pytest.mark.parametrize("rows", LONG)
def test_long_prompts_against_chunks(rows):
    """The two differ by the order of fp32 sums, and by that a value that passes between products rounds to another pair of bf16 planes:
    each side by up to 2^-17 of it, 2^-17 / sqrt(3) in l2, for the inputs of each of the eight products, sqrt(2 * 8) 2^-17 / sqrt(3) = 1.8e-5 in
    all.  A plane too few or at the wrong columns is of the size of the result."""
    print(f"prefill of {rows} rows", flush=True)
    e = S.f32_normal((rows, S.DIM), 900 + rows)
    layers, norm = [S.Layer(31), S.Layer(32)], S.norm_weight(S.DIM, 95)
    hip = H.Hip(kv_max=rows)
    try:
        hip.upload_decoder(layers, norm, 2)
        got = []
        for step in (rows, CHUNK):
            x = []
            for want_x in (False, True):           # the cache alone: the last layer's k|v product; then the rows as well
                hip.pos = 0
                for at in range(0, rows, step):
                    x.append(hip.llm_prefill(e[at:at + step], want_x=want_x))
                if not want_x:
                    kv = [c[:2].copy() for c in hip.kv(2)]
                    x = []
            got.append([np.concatenate(x)] + kv + [c[:2].copy() for c in hip.kv(2)])
    finally:
        hip.close()
    for a, b in zip(*got):
        assert np.isfinite(a).all()
        a, b = a.reshape(-1, a.shape[-1]), b.reshape(-1, b.shape[-1])
        rms = np.sqrt(np.mean(a.astype(np.float64) ** 2, axis=1))
        d = np.abs(a.astype(np.float64) - b)
        assert (np.sqrt(np.mean(d ** 2, axis=1)) <= 1.8e-5 * rms).all() and (d.max(axis=1) <= 1e-4 * rms).all(), \
            (float((np.sqrt(np.mean(d ** 2, axis=1)) / rms).max()), float((d.max(axis=1) / rms).max()))

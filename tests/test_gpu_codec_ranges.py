"""The codec's products hold an fp32 operand as two fp16 planes and an exponent per row.  What fp32 arithmetic takes in
its stride: rows whose values stand near either end of fp32, and rows of values that are far apart, whose small ones
still carry the result because the large ones meet zeros.  And the memory that a decode takes."""
import ctypes as C

import numpy as np
import pytest
import torch

import codecsupport as K
import hipsupport as H
import vtsupport as S
from test_gpu_codec import hip_decode
from test_gpu_codec_planes import close

pytestmark = pytest.mark.gpu


def decode_both(hc, frames):
    S.oracle().orc_set_threads(16)
    cs = hc.struct()
    hip = H.Hip(kv_max=8)
    try:
        assert hip.lib.tts_hip_upload_codec_weights(C.addressof(cs)) == 0, hip.lib.tts_hip_last_error()
        for n in frames:
            codes = K.random_codes(n, 60 + n)
            print(f"codec of {n} frames", flush=True)
            close(K.oracle_decode(cs, codes), hip_decode(hip, codes))
    finally:
        hip.close()
        S.oracle().orc_set_threads(1)


def test_rows_near_the_ends_of_fp32():
    """The residual stream of the second stage at 1e34 (its RMSNorms overflow and give zeros, as on the CPU) between
    convolutions of 2^113 and 2^-113 times ordinary weights."""
    hc = K.HostCodec(9, distinct_layers=1)
    for conv, f in ((hc.stage_convs[0], 2.0 ** 113), (hc.stage_convs[1], 2.0 ** -113)):
        conv.weight *= np.float32(f)
    hc.stage_convs[0].bias *= np.float32(2.0 ** 113)
    decode_both(hc, (5, 40))


@pytest.mark.parametrize("log2", [20, 24])
def test_rows_of_values_far_apart(log2):
    """One channel of the normalised rows 2^20 and 2^24 times the others, which no weight reads, and weights as far from
    the rest of their rows at a channel that is zero: the result is that of the small values, whose 24 bits count."""
    f = np.float32(2.0 ** log2)
    hc = K.HostCodec(11, distinct_layers=1)
    l = hc.layers[0]
    for norm, weights in ((l.attention_norm, (l.wq, l.wk, l.wv)), (l.ffn_norm, (l.w1, l.w3))):
        norm[5] = f
        norm[6] = 0
        for w in weights:
            w[:, 5] = 0
            w[:, 6] = f * np.abs(w).max(axis=1)
    decode_both(hc, (5, 40))


def test_work_area_follows_the_frame_count():
    """A product's partial planes hold the cut columns only.  527 frames, whose last gate|up product has 256 of 8192
    columns in 6 cuts, need the 138 MB of that product, a quarter and 17 MB more for cut planes, and the 142 MB of the
    other buffers; 20 MB are left for what the runtime takes.  A decode then finds room where a longer one did."""
    hip = H.Hip(kv_max=8)
    try:
        cs = K.HostCodec(5, distinct_layers=1).struct()
        assert hip.lib.tts_hip_upload_codec_weights(C.addressof(cs)) == 0, hip.lib.tts_hip_last_error()

        def used_by(n):
            before = torch.cuda.mem_get_info()[0]
            hip_decode(hip, K.random_codes(n, n))
            return before - torch.cuda.mem_get_info()[0]

        used_by(9)                     # the runtime takes some memory of its own with the first launches of a kernel
        used_by(65)
        assert used_by(527) <= 352e6
        used_by(612)
        for n in (527, 288, 575):
            assert used_by(n) <= 20e6, n
    finally:
        hip.close()

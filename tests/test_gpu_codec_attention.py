"""The codec's windowed attention has a kernel for few tokens (eight key groups per query, merged) and one for many
(two neighbouring queries per lane group share their keys): windows of one key, of less and more than a group, odd
ones and none, in every stage, with token counts that leave the last workgroup of 16
partly empty.  Bounds as for the
tile edges: fp32 sums in another order, four times the measured difference."""
import ctypes as C

import pytest

import codecsupport as K
import hipsupport as H
import vtsupport as S
from test_gpu_codec import hip_decode
from test_gpu_codec_planes import close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_frames,windows", [(9, (1, 8, 9, 17)), (33, (0, 1, 3, 0)), (129, (16, 0, 5, 1)), (131, (3, 2, 33, 16))])
def test_windows_and_token_counts(n_frames, windows):
    S.oracle().orc_set_threads(16)
    hc = K.HostCodec(8, distinct_layers=2)
    for i, l in enumerate(hc.layers):
        l.window = windows[i // 2]
    cs = hc.struct()
    hip = H.Hip(kv_max=8)
    try:
        assert hip.lib.tts_hip_upload_codec_weights(C.addressof(cs)) == 0, hip.lib.tts_hip_last_error()
        codes = K.random_codes(n_frames, 700 + n_frames)
        print(f"codec of {n_frames} frames, windows {windows}", flush=True)
        close(K.oracle_decode(cs, codes), hip_decode(hip, codes))
    finally:
        hip.close()
        S.oracle().orc_set_threads(1)


IN_PLACE = [151, 212, 255]


@pytest.mark.parametrize("n_frames", IN_PLACE)
def test_v_where_the_product_left_it(n_frames):
    """From 1024 rows on v is read from the q|k|v product's result where its columns are in one plane (1208, 1696 and 2040 rows
    here, all columns in one; all whole, and some: 512 and 527 frames in test_gpu_mixed_plans.py); fewer rows have it copied or summed from
    several planes."""
    S.oracle().orc_set_threads(16)
    hc = K.HostCodec(9, distinct_layers=2)
    cs = hc.struct()
    hip = H.Hip(kv_max=8)
    try:
        assert hip.lib.tts_hip_upload_codec_weights(C.addressof(cs)) == 0, hip.lib.tts_hip_last_error()
        codes = K.random_codes(n_frames, 90 + n_frames)
        print(f"codec of {n_frames} frames", flush=True)
        close(K.oracle_decode(cs, codes), hip_decode(hip, codes))
    finally:
        hip.close()
        S.oracle().orc_set_threads(1)


def test_an_odd_token_count_on_workgroups_of_16():
    """1025 rows in the first stage leave the last workgroup one token.  The decoder is causal: the samples are the
    first ones of a longer decode, up to the sums of another plan."""
    hc = K.HostCodec(8, distinct_layers=2)
    cs = hc.struct()
    hip = H.Hip(kv_max=8)
    try:
        assert hip.lib.tts_hip_upload_codec_weights(C.addressof(cs)) == 0, hip.lib.tts_hip_last_error()
        codes = K.random_codes(1040, 77)
        whole = hip_decode(hip, codes)
        part = hip_decode(hip, codes[:1025])
        close(whole[:part.size], part)
        tail = slice(1020 * 1920, 1025 * 1920)
        close(whole[tail], part[tail])
    finally:
        hip.close()


@pytest.mark.parametrize("n_frames", [513, 1030, 2049])
def test_four_tokens_to_a_lane_group(n_frames):
    """Rows that give two tokens to a lane group more workgroups than compute units: 4104, 8240 and 16392 rows in the last
    stage, 4120 in the third, and 4098 already in the second, where the last lane group has two of its four.  With windows of 2, 4,
    8 and 16 a sample depends on fewer than 40 frames in front of it, so the ends of a long decode are those of short
    ones, up to the sums of another plan."""
    hc = K.HostCodec(8, distinct_layers=2)
    cs = hc.struct()
    hip = H.Hip(kv_max=8)
    try:
        assert hip.lib.tts_hip_upload_codec_weights(C.addressof(cs)) == 0, hip.lib.tts_hip_last_error()
        codes = K.random_codes(n_frames, 78)
        print(f"codec of {n_frames} frames", flush=True)
        whole = hip_decode(hip, codes)
        head, tail = hip_decode(hip, codes[:100]), hip_decode(hip, codes[-100:])
        close(whole[:head.size], head)
        close(whole[-60 * 1920:], tail[-60 * 1920:])
        mid = n_frames // 2
        close(whole[(mid - 60) * 1920:mid * 1920], hip_decode(hip, codes[mid - 100:mid])[-60 * 1920:])
    finally:
        hip.close()

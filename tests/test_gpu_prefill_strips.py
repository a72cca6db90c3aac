"""Prefill products of up to 64 rows on column strips (vt_gemm_strip_kernel): one instance per eight rows, the planes of 16
rows in one matrix instruction.  Row counts at the edges of both, alone, as a continued prompt and for the cache alone
(whose last layer takes k and v with 64 columns of q), against the oracle."""
import numpy as np
import pytest

import hipsupport as H
import vtsupport as S
from test_gpu_prefill_mfma import _prefill_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", [[1, 15], [2, 17], [23], [24, 39], [47], [55, 56], [62]])
def test_edges(chunks):
    print(f"prefill of {chunks} rows", flush=True)
    _prefill_case(1, chunks, sum(chunks) + 4, lambda n: range(n))


def test_a_row_does_not_reach_its_neighbours():
    """The last row behind all others is another and 1e18 times as large: nothing of it is seen in them."""
    layer, norm = S.Layer(21), S.norm_weight(S.DIM, 97)
    hip = H.Hip(kv_max=64)
    try:
        hip.upload_decoder([layer], norm, 1)
        e = S.f32_normal((40, S.DIM), 77)
        ref = hip.llm_prefill(e, want_x=True)
        hip.check()
        bad = e.copy()
        bad[39] = 1e18 * S.f32_normal(S.DIM, 78)
        hip.pos = 0
        got = hip.llm_prefill(bad, want_x=True)
        hip.check()
        assert np.array_equal(ref[:39], got[:39])
    finally:
        hip.close()

"""The prefill's products take their tiles and K cuts from the row count: up to 64 rows the column strips of
vt_gemm_rows.hip (one instance per 8 rows), then the tiles of 80 to 128 rows
of vt_gemm_wide.hip.  Row counts at the edges of those, alone and as a continued prompt, against the oracle
(rows, cache rows, and the decode step that reads them)."""
import pytest

from test_gpu_prefill_mfma import _prefill_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", [[1, 7], [8, 9], [16, 17], [24, 25, 31], [32, 33], [40, 41], [48, 49], [57, 63], [64, 65]])
def test_prefill_row_counts_of_the_few_row_tiles(chunks):
    _prefill_case(2, chunks, sum(chunks) + 4, lambda n: range(n))


# the last three: 128 x 256 whole with SiLU, 96 x 256 whole, 128 x 256 in cuts (test_plans_cpu.py: every tile is run by one of the lists)
WIDE = [[96, 97], [128, 129], [192, 193], [225], [256, 257], [288, 289], [350], [850], [1130]]


@pytest.mark.parametrize("chunks", WIDE)
def test_prefill_row_counts_of_the_wide_tiles(chunks):
    _prefill_case(1, chunks, sum(chunks) + 4, lambda n: range(0, n, 3))


def test_prefill_with_gates_far_from_zero():
    """SiLU(gate) * up for gates of +-100 and more, where exp(-gate) over- and underflows: w1 scaled by 64, w2 by 2^-6."""
    import numpy as np
    import cases
    import hipsupport as H
    import vtsupport as S
    layer = S.Layer(13)
    for w, f in ((layer.w1, 64.0), (layer.w2, 2.0 ** -6)):           # powers of two: the bf16 values stay exact
        w[...] = S.f32_to_bf16_trunc(S.bf16_to_f32(w) * np.float32(f))
    norm = S.norm_weight(S.DIM, 98)
    orc = cases.OracleBackend(threads=16)
    orc.llm_open([layer], norm, 128, n_layers=1)
    hip = H.Hip(kv_max=128)
    try:
        hip.upload_decoder([layer], norm, 1)
        for s in (37, 80):                                           # both gate|up kernels
            e = S.f32_normal((s, S.DIM), 90 + s)
            rx, gx = orc.llm_prefill(e, want_x=True), hip.llm_prefill(e, want_x=True)
            hip.check()
            assert np.all(np.isfinite(gx))
            for r in range(s):
                mx, l2 = S.rel_errors(rx[r], gx[r])
                assert mx < 1e-3 and l2 < 1e-3, (s, r, mx, l2)
    finally:
        hip.close()


def test_prefill_with_gates_near_the_ends_of_fp32():
    """Gates of -1e37 leave SiLU(gate) * up = 0 and gates of 2.8e38 times an up of 0 as well: h columns of both kinds
    between ordinary ones.  Channel 0 of the normalised rows is about 37 everywhere (the first embedding column is 50, the
    attention adds nothing), so a w1 row that reads it alone gives all rows the same gate, to a few per cent."""
    import numpy as np
    import cases
    import hipsupport as H
    import vtsupport as S
    layer = S.Layer(14)
    layer.wo[...] = 0
    x0 = 50.0 / np.sqrt((50.0 ** 2 + S.DIM - 1) / S.DIM) * float(layer.ffn_norm[0])
    for cols, gate in ((slice(0, None, 3), -1e37), (slice(1, None, 97), 2.8e38)):
        w = np.zeros(S.DIM, np.float32)
        w[0] = gate / x0
        layer.w1[cols] = S.f32_to_bf16_trunc(w)
    layer.w3[1::97] = 0
    norm = S.norm_weight(S.DIM, 98)
    orc = cases.OracleBackend(threads=16)
    orc.llm_open([layer], norm, 192, n_layers=1)
    hip = H.Hip(kv_max=192)
    try:
        hip.upload_decoder([layer], norm, 1)
        for s in (37, 80):                                           # both gate|up kernels, whole tiles and cut ones
            e = S.f32_normal((s, S.DIM), 95 + s)
            e[:, 0] = 50.0
            rx, gx = orc.llm_prefill(e, want_x=True), hip.llm_prefill(e, want_x=True)
            hip.check()
            assert np.all(np.isfinite(rx)) and np.all(np.isfinite(gx))
            for r in range(s):
                mx, l2 = S.rel_errors((rx - e)[r, 1:], (gx - e)[r, 1:])
                assert mx < 1e-3 and l2 < 1e-3, (s, r, mx, l2)
    finally:
        hip.close()


@pytest.mark.parametrize("chunks", [[1, 8], [37, 64], [65, 97], [226, 41]])
def test_prefill_for_the_cache_alone(chunks):
    """Without the rows the last layer is its k|v product only: the cache is the one of the whole prefill, the last
    layer's up to the order of sums (K cuts of a 2048-column product; fp32 sums of 3072 products differ by ~3e-7)."""
    import numpy as np
    import hipsupport as H
    import vtsupport as S
    layers, got = [S.Layer(21), S.Layer(22)], []
    hip = H.Hip(kv_max=sum(chunks) + 1)
    try:
        hip.upload_decoder(layers, S.norm_weight(S.DIM, 97), 2)
        for want_x in (True, False):
            hip.pos = 0
            for i, n in enumerate(chunks):
                hip.llm_prefill(S.f32_normal((n, S.DIM), 300 + i), want_x=want_x)
            got.append([c[:2, :sum(chunks)].copy() for c in hip.kv(2)])
            if want_x:
                hip.set_kv(np.zeros((26, hip.kv_max, S.KV_DIM)), np.zeros((26, hip.kv_max, S.KV_DIM)))
    finally:
        hip.close()
    for a, b in zip(*got):
        assert np.array_equal(a[0], b[0])
        mx, l2 = S.rel_errors(a[1].ravel(), b[1].ravel())
        assert mx < 1e-5 and l2 < 3e-6, (mx, l2)

"""The prefill's products take their tiles and K cuts from the row count: up to 64 rows the 64-column tiles of
vt_gemm_rows.hip (one instance per 8 rows, 8 waves up to 40 rows and 4 beyond), then the 96- and 128-row tiles
of vt_gemm_wide.hip.  Row counts at the edges of those, alone and as a continued prompt, against the oracle
(rows, cache rows, and the decode step that reads them)."""
import pytest

from test_gpu_prefill_mfma import _prefill_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", [[1, 7], [8, 9], [16, 17], [24, 25, 31], [32, 33], [40, 41], [48, 49], [57, 63], [64, 65]])
def test_prefill_row_counts_of_the_few_row_tiles(chunks):
    _prefill_case(2, chunks, sum(chunks) + 4, lambda n: range(n))


@pytest.mark.parametrize("chunks", [[96, 97], [128, 129], [192, 193], [225], [256, 257], [288, 289]])
def test_prefill_row_counts_of_the_wide_tiles(chunks):
    _prefill_case(1, chunks, sum(chunks) + 4, lambda n: range(0, n, 3))

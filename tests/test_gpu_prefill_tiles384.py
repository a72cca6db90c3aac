"""Prefill products on tiles of 384 columns: 96 and 128 rows, whole columns (450, 515 rows), whole columns of gate|up beside K cuts of the
others (697, 1050 rows, the latter in many cuts), the down projection in cuts only (697), q|k|v whole and in part cut with the boundary among
the v columns (1450, 1600); the last rows of a tile each time.  Against the oracle."""
import pytest

from test_gpu_prefill_mfma import _prefill_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [450, 515, 697, 1050, 1450, 1600])
def test_prefill_row_counts_of_the_384_column_tiles(rows):
    print(f"prefill of {rows} rows", flush=True)
    _prefill_case(1, [rows], rows + 4, lambda n: range(0, n, 7))

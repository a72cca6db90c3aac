"""Prefill products on tiles of 192 columns, which at 256 CUs are taken at row counts whose 256-column tiles leave CUs
idle: 96 rows in K cuts (100 rows, a remainder of four behind one tile; 300) and whole (690), 128 rows in cuts (511) and
whole (969).  Against the oracle."""
import pytest

from test_gpu_prefill_mfma import _prefill_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [100, 300, 511, 690, 969])
def test_prefill_row_counts_of_the_192_column_tiles(rows):
    print(f"prefill of {rows} rows", flush=True)
    _prefill_case(1, [rows], rows + 4, lambda n: range(0, n, 7))

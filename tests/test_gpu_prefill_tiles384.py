"""Prefill products on tiles of 384 columns: 96 and 128 rows, gate|up whole (450, 515 rows) and whole beside K cuts (1050: 96 rows, 1600: 128),
down in cuts (697: 96 rows, 1200: 128), q|k|v whole (1450, 1600); the last rows of a tile each time.  Which plans these are: test_plans_cpu.py.
Against the oracle."""
import pytest

from test_gpu_prefill_mfma import _prefill_case

pytestmark = pytest.mark.gpu

ROWS = [450, 515, 697, 1050, 1200, 1450, 1600]


@pytest.mark.parametrize("rows", ROWS)
def test_prefill_row_counts_of_the_384_column_tiles(rows):
    print(f"prefill of {rows} rows", flush=True)
    _prefill_case(1, [rows], rows + 4, lambda n: range(0, n, 7))

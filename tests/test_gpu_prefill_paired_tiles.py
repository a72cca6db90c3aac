"""Prefill products on tiles of 80 and 112 rows, whose groups of 16 rows stand with both planes in one matrix instruction: 80 rows by 256
columns in K cuts (65, 79, 97, 129 rows), whole with SiLU (161, 225, 240) and without (690), by 192 columns whole (129, 150, 160 with SiLU,
560 without), by 384 with SiLU (399), 112 rows in cuts (780), whole with SiLU (335) and without (1051); full tiles, and the first and the last
row of a group of 16 as the last row.  Which plans these are: test_plans_cpu.py.  Against the oracle."""
import pytest

from test_gpu_prefill_mfma import _prefill_case

pytestmark = pytest.mark.gpu

ROWS = [65, 79, 97, 129, 150, 160, 161, 225, 240, 335, 399, 560, 690, 780, 1051]


@pytest.mark.parametrize("rows", ROWS)
def test_prefill_row_counts_of_the_paired_tiles(rows):
    print(f"prefill of {rows} rows", flush=True)
    _prefill_case(1, [rows], rows + 4, lambda n: range(0, n, 7 if n > 100 else 1))

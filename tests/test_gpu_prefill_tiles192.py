"""Prefill products on tiles of 192 columns, which at 256 CUs are taken at row counts whose 256-column tiles leave CUs idle: 80 rows whole
(511: q|k|v), 96 rows in K cuts (760: down) and whole (1400: output, down), 128 rows in cuts (969: output) and whole (969: q|k|v, 2020: output).
100, 300 and 690 rows are lengths beside them.  Which plans these are: test_plans_cpu.py.  Against the oracle."""
import pytest

from test_gpu_prefill_mfma import _prefill_case

pytestmark = pytest.mark.gpu

ROWS = [100, 300, 511, 690, 760, 969, 1400, 2020]


@pytest.mark.parametrize("rows", ROWS)
def test_prefill_row_counts_of_the_192_column_tiles(rows):
    print(f"prefill of {rows} rows", flush=True)
    _prefill_case(1, [rows], rows + 4, lambda n: range(0, n, 7))

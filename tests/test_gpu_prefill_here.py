"""Prompts of up to 64 rows in all, whose attention makes its tiles of K and V itself: chunks that begin and end at the edges of a tile of 32
keys and of a block of 16 queries, one row behind cached ones, the last row that fits, and a prompt that goes on past it (the tile
images of a launch of their own from there).  Against the oracle."""
import pytest

from test_gpu_prefill_mfma import _prefill_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", [[16, 16, 1], [31, 2, 31], [33, 30, 1], [5, 28, 15], [1, 32], [64, 1], [63, 2], [48, 16]])
def test_chunks(chunks):
    print(f"prefill of {chunks} rows", flush=True)
    _prefill_case(2, chunks, sum(chunks) + 1, lambda n: range(n))

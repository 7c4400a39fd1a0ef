"""The converters on both sides of the rule by which a window's distinct columns are listed: through a set of bits
(columns up to 2^24, not far more of them than entries) or by sorting."""
import numpy as np
import pytest

DT = {0: "fp16", 1: "tf32"}


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("cols,per_row", [(63, 9), (64, 9), (65, 9), (4097, 40), (262145, 300), (1 << 24, 40000),
                                          ((1 << 24) + 1, 40000), (1 << 24, 3), (0xFFFFFFFE, 50)])
def test_windows_of_few_and_of_very_many_columns(hs, oracle, dtype, cols, per_row):
    rng = np.random.default_rng(cols % 1000 + per_row)
    rows = 21
    lists = [np.unique(np.concatenate([rng.integers(0, cols, per_row), [cols - 1] if r % 3 == 0 else [0]])) for r in range(rows)]
    lists[5] = lists[5][:0]
    row_ptr = np.concatenate([[0], np.cumsum([len(x) for x in lists])]).astype(np.uint32)
    col_idx = np.concatenate(lists).astype(np.uint32)
    values = rng.uniform(0.5, 1.0, col_idx.size).astype(np.float32)
    values = values.astype(np.float16).view(np.uint16) if dtype == 0 else values
    got = hs.csr_to_btcf(rows, cols, row_ptr, col_idx, values, dtype)
    want = oracle.csr_to_btcf(rows, cols, row_ptr, col_idx, values, DT[dtype])
    for k in ("rowOffset", "tcA2B", "data", "rowIdx"):
        assert got[k].tobytes() == want[k].tobytes(), k
    # the bitmap converter lists the same columns; its tiles expanded are these tiles
    wide = hs.bitmap_expand(hs.csr_to_bitmap(rows, cols, row_ptr, col_idx, values, dtype))
    for k in ("rowOffset", "tcA2B", "data", "rowIdx"):
        assert wide[k].tobytes() == got[k].tobytes(), k

"""TOPK-32's kernel at the edges of its runs of four chunks (256 rows, then
1024 each): a run that ends with its last row, one of a single row, as many
earlier runs as wavefronts and one more, the most runs there are; values that
rise through the vector, so that every run changes the list, with and without
a row that equals entry 31 when a run begins.  Bit-exact against the oracle's
running list."""
import numpy as np
import pytest

from oracle import law

pytestmark = pytest.mark.gpu

RUN0, RUN = 256 + 3 * 1024, 4 * 1024   # rows of the first run and of the others


@pytest.mark.parametrize("tie", [False, True])
@pytest.mark.parametrize("n", [
    257, 256 + 1024, RUN0 - 1, RUN0, RUN0 + 1, RUN0 + 1025, RUN0 + 4 * RUN, RUN0 + 4 * RUN + 1,
    RUN0 + 16 * RUN + 1, RUN0 + 17 * RUN + 2049, 248320, 1 << 18])
def test_topk32_runs(engine, n, tie):
    rng = np.random.default_rng(n)
    # distinct values whose level rises by a third of their spread per run
    y = rng.permutation(n).astype(np.int64) * 3 + np.arange(n) * 3 // RUN * n
    last = (n - 1 - RUN0) // RUN * RUN + RUN0 if n > RUN0 else min(n - 1, 256)
    if tie:   # the first row of the last run equals entry 31 of the rows before it
        y[last] = np.sort(y[:last])[-32]
    y = y.astype(np.int32)
    vals, rows, count, ovf = law.topk32(y)
    assert ovf or not tie
    g_vals, g_rows, g_count, g_ovf = engine.topk32(y)
    assert g_count == count and g_ovf == ovf
    assert np.array_equal(g_vals, vals) and np.array_equal(g_rows, rows)

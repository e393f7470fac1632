"""Row sums over thousands of columns (zk_row_sum_wide) at the edges of their
blocks."""

import numpy as np
import pytest

from zealot_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(3, 2047), (3, 2048), (1, 8191), (2, 8192), (5, 8193), (2, 24_581), (300, 4096)])
def test_row_sum_exact_on_integers(ctx, m, n):
    """Whole numbers below 2^24 in every partial sum: any order gives the same."""
    x = np.random.default_rng(n).integers(-300, 300, (m, n)).astype(np.float32)
    out = ctx.alloc(m)
    ops.row_sum(ctx, out, ctx.to_device(x), m, n)
    assert np.array_equal(out.numpy(), x.sum(1, dtype=np.float64).astype(np.float32))


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_row_sum_not_finite(ctx, bad):
    x = np.ones((2, 9000), np.float32)
    x[1, 8999] = bad
    out = ctx.alloc(2)
    ops.row_sum(ctx, out, ctx.to_device(x), 2, 9000)
    assert np.array_equal(out.numpy(), np.array([9000, bad], np.float32), equal_nan=True)

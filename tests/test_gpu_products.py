"""Products without a lane count on both sides of every line of their rule (rows
and mean row length), against numpy in 64 bits."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(rows, mean, seed, longest):
    """rows x (rows - 7) with exactly rows * mean entries (rounded down), among
    them rows without an entry (the first and the last too) and a longest one."""
    rng = np.random.default_rng(seed)
    total = int(rows * mean)
    count = rng.integers(max(0, int(mean * 0.5)), int(np.ceil(mean * 1.5)) + 1, rows)
    count[[0, rows // 3, rows - 1]] = 0
    count[rows // 2] = longest
    free = np.setdiff1d(np.arange(1, rows - 1), [rows // 3, rows // 2])
    while (d := total - int(count.sum())) != 0:
        pick = rng.choice(free, min(abs(d), free.size), replace=False)
        count[pick] = np.maximum(0, count[pick] + np.sign(d))
    start = np.zeros(rows + 1, np.int32)
    np.cumsum(count, out=start[1:])
    row = np.repeat(np.arange(rows), count)
    column = (row + rng.integers(-900, 901, row.size)) % (rows - 7)
    return start, column.astype(np.int32), rng.standard_normal(row.size), row, count


# the lines: 16,384 (one latency long below), 32,768 (5 to 9 entries), 65,536 (11
# to 12, 12 to 24, 24 to 48), 393,216 (4 to 5, FP64) rows; a row longer than 4 x
# mean + 16 keeps the general shape
@pytest.mark.parametrize("rows,mean", [(16383, 37.5), (16385, 37.5), (16385, 30), (32767, 7), (32769, 7), (65535, 11.4), (65537, 11.4),
                                       (65535, 15), (65537, 15), (65537, 30), (393215, 4.7), (393217, 4.7),
                                       (65539, 4), (65539, 5), (65539, 9), (65539, 11), (65539, 12), (65539, 24), (65539, 48)])
@pytest.mark.parametrize("over", [0, 1])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_default_shapes(rows, mean, dtype, over):
    from nsfem_amd import cu
    start, column, values, row, count = _matrix(rows, mean, rows + int(10 * mean), int(4 * mean + 16) + over)
    assert count.max() == int(4 * mean + 16) + over
    cols = rows - 7
    values = values.astype(dtype)
    A = cu.csrF(rows, cols, start, column, values)
    rng = np.random.default_rng(1)
    x = rng.standard_normal((3, cols)).astype(dtype)
    y0 = rng.standard_normal((3, rows)).astype(dtype)
    v, x64 = values.astype(np.float64), x.astype(np.float64)
    for nch in (1, 2, 3):
        for alpha, beta in ((1.0, 0.0), (-1.5, 0.75)):
            y = cu.vec(y0[:nch].ravel() if beta else np.full(nch * rows, np.nan, dtype))  # beta 0 reads no y
            A.mul(cu.vec(x[:nch].ravel()), y, numCh=nch, alpha=alpha, beta=beta)
            got = y.download().reshape(nch, rows).astype(np.float64)
            for c in range(nch):
                term = v * x64[c][column]
                ref = alpha * np.bincount(row, term, rows) + beta * y0[c]
                size = abs(alpha) * np.bincount(row, np.abs(term), rows) + beta * np.abs(y0[c])
                # count + 2 roundings of partial sums no larger than the sum of the terms' sizes, in each of the two
                bound = (count + 2) * (np.finfo(dtype).eps + np.finfo(np.float64).eps) * size
                assert np.all(np.abs(got[c] - ref) <= bound), (nch, c, alpha)

"""The fp32 linear over 128 rows at the ends of fp32's range: the scales of a row
of x and of a row of W leave the sums one after the other, so a product of the
two that is no float (past 2^127, under 2^-149) must not show.

Whole numbers and powers of two, so float64 gives the result bit for bit where it
is a float; sums that round are held to 2e-6 of |x||w|, as fp32 sums give.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(200, 96, 64), (1100, 200, 1024), (2500, 96, 1024), (300, 1100, 400)]  # each tile form, split K


def halves(M, K, N, seed):
    """x on the first half of the columns, W on the second: every product is 0."""
    r = np.random.default_rng(seed)
    x, W = r.standard_normal((M, K), dtype=np.float32), r.standard_normal((N, K), dtype=np.float32)
    x[:, K // 2:] = 0
    W[:, :K // 2] = 0
    return x, W


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_zero_sums_of_large_rows(vla, M, K, N):
    x, W = halves(M, K, N, 1)
    got = vla.dense_linear(x * np.float32(1e37), W * np.float32(1e37), None)
    assert np.array_equal(got, np.zeros((M, N), np.float32))


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("ex,ew", [(-60, -64), (-66, -70), (-70, -66), (-100, -20), (-20, -104), (-120, 60), (100, -110), (120, -120)])
def test_whole_numbers_times_powers(vla, M, K, N, ex, ew):
    """Small whole numbers scaled by powers of two: every sum is exact."""
    r = np.random.default_rng(2)
    x = np.ldexp(r.integers(-15, 16, (M, K)), ex).astype(np.float32)
    W = np.ldexp(r.integers(-15, 16, (N, K)), ew).astype(np.float32)
    want = x.astype(np.float64) @ W.astype(np.float64).T
    assert np.array_equal(vla.dense_linear(x, W, None), want.astype(np.float32))


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_outlier_columns(vla, M, K, N):
    """A few channels 4 to 1000 times the others, outside the first 64 columns: the
    sums keep the rows' precision whichever pass finds them."""
    r = np.random.default_rng(3)
    x, W = r.standard_normal((M, K), dtype=np.float32), r.standard_normal((N, K), dtype=np.float32)
    for c, f in ((70, 4), (75, 30), (90, 1000)):
        x[:, c] *= np.float32(f)
    W[::5, 80] *= np.float32(300)
    got = vla.dense_linear(x, W, None)
    want = x.astype(np.float64) @ W.astype(np.float64).T
    size = np.linalg.norm(x.astype(np.float64), axis=1)[:, None] * np.linalg.norm(W.astype(np.float64), axis=1)[None]
    assert float((np.abs(got - want) / size).max()) < 2e-6

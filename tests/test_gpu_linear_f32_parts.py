"""The fp16-part tiles of the fp32 linear (more than 128 rows) where they can go
wrong: both sides of every tile choice, ragged rows, columns and K slabs,
unaligned rows, and rows whose scale the guess from one slab does not give.
Against float64, per output row: a row's parts keep 2^-22 of every value or
2^-28 of the row's largest, so a row's error stays what fp32 sums give
(a few 2^-24 sqrt(K) of |x||w|; 2e-6 of the row's 2-norm bound is held).
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(vla, x, W, b=None, tol=2e-6):
    got = vla.dense_linear(x, W, b)
    want = x.astype(np.float64) @ W.astype(np.float64).T + (0 if b is None else b)
    # each output against its own row norms, so that no row hides behind another
    size = np.linalg.norm(x.astype(np.float64), axis=1)[:, None] * np.linalg.norm(W.astype(np.float64), axis=1)[None]
    err = np.abs(got - want) / np.maximum(size, 1e-300)
    assert float(err.max()) < tol, float(err.max())


def data(M, K, N, seed=0):
    r = np.random.default_rng(seed)
    return (r.standard_normal((M, K), dtype=np.float32), r.standard_normal((N, K), dtype=np.float32) / np.float32(K) ** 0.5,
            r.standard_normal(N, dtype=np.float32))


@pytest.mark.parametrize("M,K,N", [
    (129, 32, 32), (129, 33, 33), (160, 64, 40), (177, 960, 96), (511, 96, 510), (512, 100, 512),     # 32 x 32
    (1024, 160, 1024), (1025, 161, 1023), (1030, 100, 1030), (1024, 32, 1000), (700, 65, 768),       # 64 x 64, two groups
    (2500, 70, 1024), (2500, 96, 830),                                                               # 64 x 64
    (4096, 70, 1024), (4100, 64, 1030),                                                              # 128 x 64
    (300, 1100, 400), (1200, 1100, 260),                                                             # few tiles, long K
])
@pytest.mark.parametrize("pad", [0, 1])
def test_shapes(vla, M, K, N, pad):
    x, W, b = data(M, K + pad, N)
    check(vla, x, W, b)


@pytest.mark.parametrize("M,N", [(200, 64), (1100, 1024)])
def test_rows_of_every_size(vla, M, N):
    """Rows of x and W over 2^-60 .. 2^60: each keeps its own precision."""
    x, W, _ = data(M, 200, N, 1)
    r = np.random.default_rng(2)
    x *= np.exp2(r.integers(-60, 61, (M, 1))).astype(np.float32)
    W *= np.exp2(r.integers(-60, 61, (N, 1))).astype(np.float32)
    check(vla, x, W)


@pytest.mark.parametrize("M,N", [(200, 64), (1100, 1024)])
@pytest.mark.parametrize("step", [1e-15, 1e-6, 1e6, 1e15])
def test_guess_slab_misleads(vla, M, N, step):
    """Values after the first slab far above or below it, or only there."""
    x, W, _ = data(M, 256, N, 3)
    x[::3, 40:] *= np.float32(step)
    W[1::3, 40:] *= np.float32(step)
    x[5::7, :64] = 0
    W[3::11, :64] = 0
    x[11] = 0
    check(vla, x, W)


def test_smallest_and_largest(vla):
    x, W, _ = data(200, 128, 64, 4)
    check(vla, (x * np.float32(1e-36)), W)
    check(vla, (x * np.float32(1e30)), (W * np.float32(1e-34)))
    big = x.copy()
    big[:, 7] = np.float32(3.0e38) * np.sign(x[:, 7])
    check(vla, big, (W * np.float32(1e-3)))


def test_not_finite(vla):
    """Infinities and NaN stay in their own rows and columns."""
    x, W, _ = data(200, 128, 64, 5)
    W = np.abs(W)
    xi = x.copy()
    xi[17, 100] = np.inf
    xi[90, 3] = np.nan
    got = vla.dense_linear(xi, W, None)
    assert np.all(got[17] == np.inf) and np.all(np.isnan(got[90]))
    rows = np.setdiff1d(np.arange(200), [17, 90])
    want = x.astype(np.float64) @ W.astype(np.float64).T
    assert float(np.abs(got - want)[rows].max()) < 1e-5

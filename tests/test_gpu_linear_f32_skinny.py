"""The fp32 linear at 1 to 128 rows, whose operands cross to the matrix order
through LDS: every count of 16-row groups, K steps short of and past each
wave's share, ragged and unaligned rows. Whole-number inputs small enough that
every sum is exact, so the results have to be the float64 ones bit for bit.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 15, 16, 17, 33, 64, 65, 81, 100, 112, 113, 128])
@pytest.mark.parametrize("K,N", [(1, 5), (16, 16), (18, 17), (132, 48), (512, 3200), (1031, 33), (2060, 16)])
def test_whole_numbers(vla, M, K, N):
    r = np.random.default_rng(M * 4096 + K)
    x = r.integers(-15, 16, (M, K)).astype(np.float32)
    W = r.integers(-15, 16, (N, K)).astype(np.float32)  # sums below 15^2 2060 < 2^24
    b = r.integers(-99, 100, N).astype(np.float32)
    want = x.astype(np.float64) @ W.astype(np.float64).T + b
    np.testing.assert_array_equal(vla.dense_linear(x, W, b), want.astype(np.float32))

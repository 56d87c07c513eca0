"""GPU parity of the running median's scrunch: exact sums, so every bit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("factor", [2, 3, 16, 38, 63, 64, 1000, 2049, 4096, 4097])
def test_scrunch_factors(gpu, port, factor):
    """Detrended series around the sizes at which the lanes of an output change
    (powers of two), one output a workgroup (past 2048) and a wave per output
    (past 4096); values past 2^24 round to float before they are summed."""
    rng = np.random.default_rng(factor)
    n = factor * 23 + factor // 2
    print(f"scrunch: factor {factor}, {n} samples", flush=True)
    x = rng.integers(0, 2 ** 32, size=(3, n), dtype=np.uint32)
    x[1] = rng.integers(0, 4000, size=n)
    window = (5 * factor) | 1
    got = gpu._preprocess_batch_gpu(x, window_samples=window, min_points=5, normalise=False)
    for i in range(3):
        want = port.detrend(x[i].astype(np.float32), window, 5)
        np.testing.assert_array_equal(got[i], want)

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


@pytest.mark.parametrize("factor,ns,outputs", [
    (2, 5, 430001),     # as many outputs a workgroup as LDS holds, the last one partly full
    (38, 9, 14001),     # the same
    (256, 7, 300),      # 2 of 16
    (256, 3, 6001),     # 16
    (257, 7, 292),      # spans (2044 outputs) ...
    (257, 7, 293),      # ... and a wave per output (2051)
    (1000, 23, 101),
    (400, 8, 10486),    # spans in a large plane (2^25 samples) ...
    (401, 8, 10460),    # ... and a wave per output
    (400, 8, 10485),    # a wave per output in the largest plane below
])
def test_scrunch_outputs(gpu, port, factor, ns, outputs):
    """Both sides of the lines between fewer and more outputs a workgroup and between
    spans and a wave per output."""
    rng = np.random.default_rng(factor + outputs)
    n = factor * outputs + factor // 3
    print(f"scrunch: factor {factor}, {ns} series x {n}", flush=True)
    x = rng.integers(0, 60000, size=(ns, n)).astype(np.uint32)
    window = (5 * factor) | 1
    got = gpu._preprocess_batch_gpu(x, window_samples=window, min_points=5, normalise=False)
    for i in range(ns):
        np.testing.assert_array_equal(got[i], port.detrend(x[i].astype(np.float32), window, 5))

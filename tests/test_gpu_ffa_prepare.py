"""GPU parity of the downsampling before the FFA, every bit."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("factors", [
    [1.0, 1.03, 1.5, 2.0, 7.9, 8.0, 9.01, 17.3, 100.25, 511.7],  # the fused pass: windows around
    [300.5, 1.2, 64.0, 3.7],                                     # the read-ahead; factors not sorted
    [4094.0, 2.5],                                               # the longest halo
    [4095.5, 1.7, 10.0, 31.9],                                   # past it: a pass per group
    [8185.0, 8190.3, 3.3],                                       # one output a block; not staged
])
def test_prepare_factors(gpu, port, factors):
    """One plan of several downsample factors: every prepared sample equals the
    CPU's weighted sum in sample order, over spans, their edges and the end of
    the series."""
    from oracle.oracle import TASK_DTYPE

    rng = np.random.default_rng(len(factors))
    n = 8192 * 9 + 4321
    x = rng.normal(size=(2, n)).astype(np.float32)
    t = np.zeros(len(factors), TASK_DTYPE)
    for i, f in enumerate(factors):
        m = port.downsampled_size(n, f) if f != 1.0 else n
        bins = 4 if m < 800 else 200
        rows = m // bins
        t[i] = (f, f * 1e-3, n, m, bins, rows, rows, bins * f * 1e-3, (bins + 1) * f * 1e-3)
    plan = gpu.FfaPlan(t, [1])
    for i, f in enumerate(factors):
        bins, rows = int(t["bins"][i]), int(t["rows"][i])
        print(f"prepare: factor {f}, {rows} x {bins}", flush=True)
        got = gpu._ffa_transform_rows_gpu(x, plan, i)
        for k in range(2):
            y = port.downsample(x[k], f) if f != 1.0 else x[k]
            np.testing.assert_array_equal(got[k],
                                          port.ffa_transform(y[: rows * bins], bins))

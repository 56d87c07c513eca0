"""GPU parity of the FFA subtree kernels at the edges of their node shapes."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bins", [7, 63, 64, 65, 100, 126, 128, 160, 180, 185, 192, 193, 246, 249,
                                  250, 255, 256, 257, 303, 304, 305])
def test_ffa_nodes_bit_exact(gpu, port, bins):
    """Trees of depth 1 whose nodes are the smallest and largest of each path:
    fewer rows than sub-nodes or bins (one level at a time), 8 rows, odd and
    even counts, as many rows as the LDS or the register path holds (160), one
    more (the kernel of larger nodes), rows beyond the bins (rolls of more than
    a row), rows of whole 64-phase chunks and one phase either side, and the
    most bins the register path takes.  Three series, so that a workgroup's
    units change series and node; every value equals the CPU tree's."""
    from oracle.oracle import TASK_DTYPE

    top = min(160, 20192 // bins)
    rng = np.random.default_rng(bins)
    for rows in sorted({2, 9, 15, 16, 17, 33, 2 * top - 3, 2 * top - 1, 2 * top, 2 * top + 1}):
        if rows < 2:
            continue
        print(f"ffa nodes: rows={rows} bins={bins}", flush=True)
        n = rows * bins + 3
        x = rng.normal(size=(3, n)).astype(np.float32)
        t = np.zeros(1, TASK_DTYPE)
        t[0] = (1.0, 1e-3, n, n, bins, rows, rows, bins * 1e-3, (bins + 1) * 1e-3)
        got = gpu._ffa_transform_rows_gpu(x, gpu.FfaPlan(t, [1]), 0)
        for k in range(3):
            want = port.ffa_transform(x[k, : rows * bins], bins)
            np.testing.assert_array_equal(got[k], want)

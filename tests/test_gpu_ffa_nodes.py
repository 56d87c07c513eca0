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


@pytest.mark.parametrize("nsamples,level_rows", [(1 << 20, 0), (1 << 21, 7), (1 << 18, 0)])
def test_level_rows_built_on_the_device(gpu, nsamples, level_rows):
    """The leaf rows the device builds for a plan's level items (whole items,
    short ones, a last workgroup that is not full, a plan with none) are the
    host's, entry for entry."""
    import ctypes

    import gaffa_amd
    from gaffa_amd.ffa import make_riptide_plan

    plan = make_riptide_plan(nsamples=nsamples, tsamp=6.4e-5, period_min=0.1, period_max=10.0,
                             duty_cycle_max=0.18, width_trial_spacing=2.0)
    d = gpu._ffa_level_layout(plan, level_rows)
    items, spans, want = (np.ascontiguousarray(d[k]) for k in ("items", "spans", "leaf_rows"))
    print(f"level rows: {len(items)} items, {len(want)} rows", flush=True)
    tasks = np.zeros((plan.task_count, 62), np.uint32)  # gaffa_hip_ffa_task: bins, rows
    tasks[:, 1], tasks[:, 2] = plan.tasks["bins"], plan.tasks["rows"]
    lib = ctypes.CDLL(gaffa_amd.HIP_LIBRARY)
    ptrs = []

    def put(arr):
        p = ctypes.c_void_p()
        assert lib.gaffa_hip_malloc(ctypes.byref(p), ctypes.c_uint64(max(arr.nbytes, 256))) == 0
        ptrs.append(p)
        assert lib.gaffa_hip_memcpy(p, arr.ctypes.data_as(ctypes.c_void_p),
                                    ctypes.c_uint64(arr.nbytes), None) == 0
        return p

    try:
        out = np.full(want.shape, 0xABABABAB, np.uint32)
        args = [put(tasks), put(items), put(spans)]
        dev = put(out)
        assert lib.gaffa_hip_ffa_build_level_rows(*args, ctypes.c_uint32(len(items)), dev,
                                                  None) == 0
        assert lib.gaffa_hip_memcpy(out.ctypes.data_as(ctypes.c_void_p), dev,
                                    ctypes.c_uint64(out.nbytes), None) == 0
    finally:
        for p in ptrs:
            lib.gaffa_hip_free(p)
    np.testing.assert_array_equal(out, want)

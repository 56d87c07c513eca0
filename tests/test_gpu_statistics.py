"""GPU parity of the FP64 statistics with sums in sample order, bit for bit."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class PreprocessArgs(ctypes.Structure):
    _fields_ = [("data", ctypes.c_void_p), ("nseries", ctypes.c_uint64),
                ("nsamples", ctypes.c_uint64), ("stride", ctypes.c_uint64),
                ("input_is_u32", ctypes.c_int32), ("detrend", ctypes.c_int32),
                ("scrunch_factor", ctypes.c_uint64), ("median_window", ctypes.c_uint64),
                ("normalise", ctypes.c_int32), ("reject_constant", ctypes.c_int32),
                ("workspace", ctypes.c_void_p), ("workspace_bytes", ctypes.c_uint64),
                ("status", ctypes.c_void_p)]


def _series(kind, n, rng):
    if kind == "integers":       # exact sums, squares that round once they are large
        return np.rint(rng.normal(0.0, 300.0, n))
    if kind == "tenths":         # multiples of 2^-10, as detrended series: half the adds tie
        return np.rint(rng.normal(0.0, 90.0, n) * 1024.0) / 1024.0
    if kind == "bursts":         # the sum of squares crosses binades inside blocks
        x = np.rint(rng.normal(0.0, 2.0, n))
        x[rng.integers(0, n, 12)] = 2.0 ** rng.integers(3, 19, 12)
        return x
    if kind == "late":           # zeros, then one sample, then noise
        x = np.rint(rng.normal(0.0, 50.0, n))
        x[: 2 * n // 3] = 0.0
        x[n // 3] = 7.0
        return x
    if kind == "tiny":           # squares below the float range
        return np.rint(rng.normal(0.0, 50.0, n)) * 2.0 ** -100
    return rng.normal(0.0, 1.0, n)  # "floats": the sum itself rounds


def _statistics(x, factor, stride):
    """(mean, 1/sigma) the library leaves in its workspace, per series."""
    import gaffa_amd

    lib = ctypes.CDLL(gaffa_amd.HIP_LIBRARY)
    f = lib.gaffa_hip_preprocess_workspace_bytes
    f.restype, f.argtypes = ctypes.c_uint64, [ctypes.c_uint64] * 3
    ns, n = x.shape
    rows = np.zeros((ns, stride), np.float32)
    rows[:, :n] = x
    need = f(ns, n, factor)
    ptrs = []

    def dev(nbytes):
        p = ctypes.c_void_p()
        assert lib.gaffa_hip_malloc(ctypes.byref(p), ctypes.c_uint64(nbytes)) == 0
        ptrs.append(p)
        return p

    def copy(dst, src, nbytes):
        assert lib.gaffa_hip_memcpy(dst, src, ctypes.c_uint64(nbytes), None) == 0

    try:
        d, st, ws = dev(rows.nbytes), dev(4 * ns), dev(need)
        copy(d, rows.ctypes.data_as(ctypes.c_void_p), rows.nbytes)
        assert lib.gaffa_hip_memset(st, 0, ctypes.c_uint64(4 * ns), None) == 0
        a = PreprocessArgs(d, ns, n, stride, 0, 0, 1, 1, 1, 1, ws, need, st)
        assert lib.gaffa_hip_detrend_normalise_batch(ctypes.byref(a), None) == 0
        assert lib.gaffa_hip_device_synchronize() == 0
        # the scratch of n floats a series, then the statistics
        at = (ns * n * 4 + 255) // 256 * 256
        out = np.empty((ns, 2), np.float64)
        copy(out.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(ws.value + at), out.nbytes)
        return out
    finally:
        for p in ptrs:
            lib.gaffa_hip_free(p)


@pytest.mark.parametrize("kind", ["integers", "tenths", "bursts", "late", "tiny", "floats"])
def test_statistics_equal_sums_in_sample_order(gpu, kind):
    """Mean and 1/sigma of every series equal the FP64 sums in sample order bit
    for bit, around the block (4096) and run sizes, over binade crossings, and
    where the plain sum rounds (the serial chain); aligned rows and rows that
    are not."""
    rng = np.random.default_rng(len(kind))
    for ns, n, stride in ((3, 2, 4), (2, 31, 31), (66, 4095, 4096), (3, 4096, 4096),
                          (5, 4097, 4099), (2, 70001, 70001), (3, 300000, 300032)):
        print(f"statistics: {kind}, {ns} series x {n} (stride {stride})", flush=True)
        x = np.stack([_series(kind, n, rng) for _ in range(ns)]).astype(np.float32)
        x[:, 0] += 1.0  # never constant
        got = _statistics(x, 1, stride)
        d = x.astype(np.float64)
        mean = np.cumsum(d, axis=1)[:, -1] / n
        var = np.cumsum(d * d, axis=1)[:, -1] / n - mean * mean
        np.testing.assert_array_equal(got[:, 0], mean)
        np.testing.assert_array_equal(got[:, 1], 1.0 / np.sqrt(var))


def _normalise(x, sentinel):
    """Normalises x in place on the device with a workspace of `sentinel` bytes;
    the workspace afterwards."""
    import gaffa_amd

    lib = ctypes.CDLL(gaffa_amd.HIP_LIBRARY)
    f = lib.gaffa_hip_preprocess_workspace_bytes
    f.restype, f.argtypes = ctypes.c_uint64, [ctypes.c_uint64] * 3
    ns, n = x.shape
    work = np.full(f(ns, n, 1), sentinel, np.uint8)
    status = np.zeros(ns, np.int32)
    ptrs = []
    try:
        for host in (x, work, status):
            p = ctypes.c_void_p()
            assert lib.gaffa_hip_malloc(ctypes.byref(p), ctypes.c_uint64(host.nbytes)) == 0
            ptrs.append(p)
            assert lib.gaffa_hip_memcpy(p, host.ctypes.data_as(ctypes.c_void_p),
                                        ctypes.c_uint64(host.nbytes), None) == 0
        a = PreprocessArgs(ptrs[0], ns, n, n, int(x.dtype == np.uint32), 0, 1, 1, 1, 1, ptrs[1],
                           work.nbytes, ptrs[2])
        assert lib.gaffa_hip_detrend_normalise_batch(ctypes.byref(a), None) == 0
        assert lib.gaffa_hip_memcpy(work.ctypes.data_as(ctypes.c_void_p), ptrs[1],
                                    ctypes.c_uint64(work.nbytes), None) == 0
        return work
    finally:
        for p in ptrs:
            lib.gaffa_hip_free(p)


def test_no_maps_where_the_serial_chain_runs(gpu):
    """One series whose plain sum rounds sends its batch to the serial chain, and no
    maps are built for it (the workspace behind the block sums stays as it was)."""
    rng = np.random.default_rng(3)
    ns, n, blocks = 66, 3 * 4096 + 5, 4
    x = np.stack([_series("integers", n, rng) for _ in range(ns)]).astype(np.float32)
    at = (ns * blocks * 24 + 15) // 16 * 16
    for rounds in (None, 0, 65):
        y = x.copy()
        if rounds is not None:
            y[rounds, 7] = 2.0 ** -60
        print(f"maps: series that rounds {rounds}", flush=True)
        maps = _normalise(y, 0xCD)[at:at + 16 * ns * blocks]
        assert (maps == 0xCD).all() == (rounds is not None)


def _block_shift(ns, n, factor):
    """Blocks of 4096 << shift samples: the first whose sums (24 bytes a block) and
    maps (16) fit the low-resolution series and the medians that they replace; None
    where none does and every series runs in the serial chain."""
    low = 4 * ns * (n // factor)
    for shift in range(5):
        blocks = ns * -(-n // (4096 << shift))
        if 24 * blocks <= low and (low + 15) // 16 * 16 + 16 * blocks <= 2 * low:
            return shift
    return None


def test_statistics_in_every_block_size(gpu, port):
    """Detrended and normalised series equal the oracle's bit for bit on both sides of
    each scrunch factor at which the blocks of the statistics double (whose sums then
    fill the scratch to the last byte), and past the last one; a last block that is
    nearly full, and one that is not; whole numbers, and floats whose sum rounds."""
    rng = np.random.default_rng(11)
    seen = set()
    for n in (96 * 4096 - 5, 300001):
        for factor in (2, 682, 683, 1365, 1366, 2730, 2731, 5461, 5462, 10922, 10923):
            whole = n != 300001 or factor % 2 == 0
            x = rng.integers(0, 4000, size=(3, n)) if whole else rng.normal(size=(3, n))
            x = x.astype(np.uint32 if whole else np.float32)
            seen.add(_block_shift(3, n, factor))
            print(f"statistics: factor {factor}, {n} samples, block shift "
                  f"{_block_shift(3, n, factor)}", flush=True)
            window = (5 * factor) | 1
            got = gpu._preprocess_batch_gpu(x, window_samples=window, min_points=5)
            for i in range(3):
                want = port.normalise(port.detrend(x[i].astype(np.float32), window, 5))
                np.testing.assert_array_equal(got[i], want)
    assert seen == {0, 1, 2, 3, 4, None}


@pytest.mark.parametrize("dtype,least", [(np.uint32, 2048), (np.float32, 4096)])
def test_short_series_run_the_serial_chain(gpu, dtype, least):
    """Series below the length at which blocks pay run in the serial chain alone: the
    workspace in front of the statistics stays as it was."""
    rng = np.random.default_rng(4)
    for ns, n in ((1, least - 1), (65, least - 1), (1, least)):
        x = rng.integers(1, 4000, size=(ns, n)).astype(dtype)
        print(f"short series: {ns} x {n} {np.dtype(dtype)}", flush=True)
        assert (_normalise(x, 0xCD)[:4 * ns * n] == 0xCD).all() == (n < least)

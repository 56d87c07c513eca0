"""GPU parity of the sample-major dedispersion over its layouts, every bit."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class MultiArgs(ctypes.Structure):
    _fields_ = [("samples", ctypes.c_void_p), ("nsamples", ctypes.c_uint64),
                ("nchans", ctypes.c_uint64), ("chan_begin", ctypes.c_uint64),
                ("chan_end", ctypes.c_uint64), ("delays", ctypes.c_void_p),
                ("ndm", ctypes.c_uint64), ("out", ctypes.c_void_p),
                ("out_nsamples", ctypes.c_uint64), ("out_stride", ctypes.c_uint64),
                ("max_block_spread", ctypes.c_int32)]


def _sums(x, delays, begin, end, n_out):
    padded = np.concatenate([x, np.zeros((int(delays.max()) + n_out, x.shape[1]), np.uint8)])
    out = np.zeros((delays.shape[0], n_out), np.uint32)
    for i, row in enumerate(delays):
        for c, d in enumerate(row):
            out[i] += padded[d:d + n_out, begin + c]
    return out


@pytest.mark.parametrize("n,nch,begin,end,ndm,spread,offset", [
    (3000, 64, 0, 64, 16, 90, 0),      # whole blocks, dword loads
    (1031, 96, 4, 75, 17, 33, 0),      # a last channel block of 7, one DM in the last block
    (1031, 96, 3, 75, 5, 33, 0),       # channels that start off a dword: byte loads
    (1031, 96, 3, 75, 5, 33, 1),       # ... and a base that puts them back on one
    (700, 37, 0, 37, 33, 0, 0),        # rows off a dword, no spread
    (259, 32, 0, 32, 1, 3, 0),         # one DM, reads past the last sample
    (6000, 40, 0, 40, 16, 4728, 0),    # the largest slab that LDS takes
])
def test_dedisperse_layouts(gpu, n, nch, begin, end, ndm, spread, offset):
    import gaffa_amd

    print(f"dedisperse: {n} x {nch}[{begin}:{end}], {ndm} DMs, spread {spread}", flush=True)
    lib = ctypes.CDLL(gaffa_amd.HIP_LIBRARY)
    rng = np.random.default_rng(n + ndm)
    x = rng.integers(0, 256, size=(n, nch), dtype=np.uint8)
    x[: n // 2] |= 0xF0  # block sums near 32 * 255
    # the delays of a block span `spread` at most and start anywhere
    delays = rng.integers(0, spread + 1, size=(ndm, end - begin)).astype(np.int32)
    delays[0, 0], delays[-1, -1] = 0, spread
    delays += rng.integers(0, 50)
    n_out, stride = n - 7, n - 7 + ndm % 3
    ptrs = []

    def dev(nbytes):
        p = ctypes.c_void_p()
        assert lib.gaffa_hip_malloc(ctypes.byref(p), ctypes.c_uint64(nbytes)) == 0
        ptrs.append(p)
        return p

    def copy(dst, src, nbytes):
        assert lib.gaffa_hip_memcpy(dst, src, ctypes.c_uint64(nbytes), None) == 0

    try:
        d_x, d_d, d_o = dev(x.nbytes + 16), dev(delays.nbytes), dev(ndm * stride * 4)
        at = ctypes.c_void_p(d_x.value + offset)
        copy(at, x.ctypes.data_as(ctypes.c_void_p), x.nbytes)
        copy(d_d, delays.ctypes.data_as(ctypes.c_void_p), delays.nbytes)
        a = MultiArgs(at, n, nch, begin, end, d_d, ndm, d_o, n_out, stride, spread)
        assert lib.gaffa_hip_dedisperse_multi_u8(ctypes.byref(a), None) == 0
        assert lib.gaffa_hip_dedisperse_check(None) == 0
        got = np.empty((ndm, stride), np.uint32)
        copy(got.ctypes.data_as(ctypes.c_void_p), d_o, got.nbytes)
        np.testing.assert_array_equal(got[:, :n_out], _sums(x, delays, begin, end, n_out))
    finally:
        for p in ptrs:
            lib.gaffa_hip_free(p)


@pytest.mark.parametrize("announced,spread,ok", [(64, 64, True), (64, 65, False),
                                                 (64, 92, False), (0, 28, False)])
def test_understated_spread_is_refused(gpu, announced, spread, ok):
    """A delay table wider than the announced spread is reported, also where the
    staging rows' padding (up to 28 samples) would hold it."""
    import gaffa_amd

    print(f"dedisperse: spread {spread} announced as {announced}", flush=True)
    lib = ctypes.CDLL(gaffa_amd.HIP_LIBRARY)
    n, nch = 1024, 32
    x = np.random.default_rng(spread).integers(0, 256, size=(n, nch), dtype=np.uint8)
    delays = np.zeros((2, nch), np.int32)
    delays[1, 3] = spread
    ptrs = []

    def dev(nbytes):
        p = ctypes.c_void_p()
        assert lib.gaffa_hip_malloc(ctypes.byref(p), ctypes.c_uint64(nbytes)) == 0
        ptrs.append(p)
        return p

    try:
        d_x, d_d, d_o = dev(x.nbytes), dev(delays.nbytes), dev(2 * n * 4)
        for p, host in ((d_x, x), (d_d, delays)):
            assert lib.gaffa_hip_memcpy(p, host.ctypes.data_as(ctypes.c_void_p),
                                        ctypes.c_uint64(host.nbytes), None) == 0
        a = MultiArgs(d_x, n, nch, 0, nch, d_d, 2, d_o, n, n, announced)
        assert lib.gaffa_hip_dedisperse_multi_u8(ctypes.byref(a), None) == 0
        assert (lib.gaffa_hip_dedisperse_check(None) == 0) == ok
        assert lib.gaffa_hip_dedisperse_check(None) == 0  # the report is cleared
    finally:
        for p in ptrs:
            lib.gaffa_hip_free(p)

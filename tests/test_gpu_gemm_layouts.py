"""GPU GEMM: every way an operand tile is read, at tile and chunk edges."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class _Gemm(ctypes.Structure):
    _fields_ = [("a", ctypes.c_void_p), ("a_row", ctypes.c_int64), ("a_col", ctypes.c_int64),
                ("b", ctypes.c_void_p), ("b_row", ctypes.c_int64), ("b_col", ctypes.c_int64),
                ("m", ctypes.c_uint32), ("n", ctypes.c_uint32), ("k", ctypes.c_uint32),
                ("bias", ctypes.c_void_p), ("relu", ctypes.c_uint32),
                ("c32", ctypes.c_void_p), ("c16", ctypes.c_void_p), ("ldc", ctypes.c_uint64),
                ("k_splits", ctypes.c_uint32), ("partial", ctypes.c_void_p)]


def _bits(x):
    u = np.asarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return (((u + 0x7FFF + ((u >> 16) & 1)) >> 16) & 0xFFFF).astype(np.uint16)


def _values(b):
    return (b.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


@pytest.mark.parametrize("a_by_k", [True, False])
@pytest.mark.parametrize("b_by_k", [True, False])
@pytest.mark.parametrize("m,n,k,splits", [(8, 8, 8, 1), (64, 192, 32, 1), (72, 200, 1000, 3),
                                          (136, 64, 4104, 31), (70, 66, 97, 2)])
def test_gemm_layouts(gpu, a_by_k, b_by_k, m, n, k, splits):
    """Operands contiguous along k or along their other index, with 16-byte
    loads (sizes a multiple of 8) and without (the last shape), one k step and
    many, whole tiles and remainders: against the FP64 product of the same
    bfloat16 values.  FP32 sums of k products err by at most about k 2^-24 of
    the sum of |a b|, and far less in practice: 1e-5 of the largest."""
    import gaffa_amd

    lib = ctypes.CDLL(gaffa_amd.HIP_LIBRARY)
    print(f"gemm m={m} n={n} k={k} splits={splits} a_by_k={a_by_k} b_by_k={b_by_k}", flush=True)
    rng = np.random.default_rng(m + n + k)
    A, B = _bits(rng.normal(size=(m, k))), _bits(rng.normal(size=(k, n)))
    ptrs = []

    def put(arr):
        arr = np.ascontiguousarray(arr)
        p = ctypes.c_void_p()
        assert lib.gaffa_hip_malloc(ctypes.byref(p), ctypes.c_uint64(max(arr.nbytes, 256))) == 0
        ptrs.append(p)
        assert lib.gaffa_hip_memcpy(p, arr.ctypes.data_as(ctypes.c_void_p),
                                    ctypes.c_uint64(arr.nbytes), None) == 0
        return p

    try:
        a = put(A if a_by_k else A.T)
        b = put(B.T if b_by_k else B)
        c = put(np.zeros((m, n), np.float32))
        part = put(np.zeros((splits, m, n), np.float32))
        g = _Gemm(a, k if a_by_k else 1, 1 if a_by_k else m, b, 1 if b_by_k else n,
                  k if b_by_k else 1, m, n, k, None, 0, c, None, n, splits, part)
        assert lib.gaffa_hip_gemm_bf16(ctypes.byref(g), None) == 0
        got = np.empty((m, n), np.float32)
        assert lib.gaffa_hip_memcpy(got.ctypes.data_as(ctypes.c_void_p), c,
                                    ctypes.c_uint64(got.nbytes), None) == 0
    finally:
        for p in ptrs:
            lib.gaffa_hip_free(p)
    want = _values(A) @ _values(B)
    np.testing.assert_allclose(got, want, rtol=0, atol=1e-5 * np.abs(want).max())

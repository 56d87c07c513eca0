"""GPU: device memory kept between calls never carries one call into another."""

import threading
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _peaks(found):
    return [(i, p.shift, p.phase, p.width, p.bins, p.snr) for i, p in found]


def test_reused_device_memory_keeps_results(gpu):
    """One-shot searches and folds of different sizes, in turn, from two threads
    at once and after the cache went back, give what the first call on fresh
    memory gave."""
    from gaffa_amd.ffa import ffa_search_batch, make_riptide_plan

    rng = np.random.default_rng(5)
    jobs = []
    for ns, n in ((3, 60000), (1, 90001), (7, 30011)):
        plan = make_riptide_plan(nsamples=n, tsamp=256e-6, period_min=0.2, period_max=2.0)
        x = rng.normal(size=(ns, n)).astype(np.float32)
        x[0] += 0.4 * ((np.arange(n) % 2789) < 120)
        gpu.release_device_cache()
        jobs.append((x, plan, _peaks(ffa_search_batch(x, plan))))
        assert jobs[-1][2]

    def work(order):
        """The jobs that gave something else; a call that fails raises in result()."""
        return [k for k in order if _peaks(ffa_search_batch(*jobs[k][:2])) != jobs[k][2]]

    assert work([0, 1, 2, 1, 0]) == []
    with ThreadPoolExecutor(2) as pool:
        both = [pool.submit(work, o) for o in ([0, 1, 2] * 4, [2, 0, 1] * 4)]
        assert [f.result() for f in both] == [[], []]
    gpu.release_device_cache()
    assert work([2, 1, 0]) == []


def test_gradient_padding_is_zero_in_used_memory(gpu):
    """The parameter vector is padded to a multiple of 8; its gradient there is
    zero, also where the scorer's buffers held another call's data before."""
    import gaffa_amd
    from gaffa_amd.ffa import FfaBatchedSearch, make_riptide_plan
    from oracle import scorer_oracle as so

    gpu.release_device_cache()
    size = gaffa_amd.CandidateScorer(capacity=8).parameters.size
    rng = np.random.default_rng(6)
    x = rng.integers(1, 4000, size=(1, size + size // 8)).astype(np.uint32)

    def leave():
        for _ in range(4):
            gpu._preprocess_batch_gpu(x, window_samples=None, normalise=True)
        return True

    gpu.release_device_cache()
    with ThreadPoolExecutor(6) as pool:
        assert all(f.result() for f in [pool.submit(leave) for _ in range(6)])
    # an allocation of the parameters' size gets one of the blocks, as it was left
    plan = make_riptide_plan(nsamples=size, tsamp=1e-3, period_min=1.0, period_max=1.1)
    row = FfaBatchedSearch([plan]).download_row()
    assert size <= row.size <= x.size and (row[:size] != 0).all()
    s = gaffa_amd.CandidateScorer(capacity=8)
    _, g = s.gradients(rng.normal(size=(8, so.SUBINTS, so.PHASE)).astype(np.float32),
                       rng.normal(size=(8, so.PATCH)).astype(np.float32),
                       np.ones(8, np.float32))
    lay = so.layout()
    used = lay["bias"][5] + 1
    assert g.size == size and used < size
    np.testing.assert_array_equal(g[used:], 0.0)


def test_release_beside_a_capture(gpu):
    """Device memory released by one thread leaves a graph that another thread
    captures (thread-local mode) whole: it ends, and every replay writes."""
    import ctypes

    import gaffa_amd

    lib = ctypes.CDLL(gaffa_amd.HIP_LIBRARY)
    stream, graph, out = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    words = 1024
    held = [gaffa_amd.CandidateScorer(capacity=8)]
    assert lib.gaffa_hip_stream_create(ctypes.byref(stream)) == 0
    assert lib.gaffa_hip_malloc(ctypes.byref(out), ctypes.c_uint64(4 * words)) == 0
    try:
        assert lib.gaffa_hip_graph_begin(stream) == 0
        queued = lib.gaffa_hip_fill_u32(out, 7, ctypes.c_uint64(words), stream)
        worker = threading.Thread(target=held.clear)  # the last reference
        worker.start()
        worker.join()
        ended = lib.gaffa_hip_graph_end(stream, ctypes.byref(graph))
        assert held == [] and (queued, ended) == (0, 0)
        got = np.empty(words, np.uint32)
        for _ in range(3):
            assert lib.gaffa_hip_memset(out, 0, ctypes.c_uint64(4 * words), None) == 0
            assert lib.gaffa_hip_graph_launch(graph, stream) == 0
            assert lib.gaffa_hip_stream_synchronize(stream) == 0
            assert lib.gaffa_hip_memcpy(got.ctypes.data_as(ctypes.c_void_p), out,
                                        ctypes.c_uint64(4 * words), None) == 0
            assert (got == 7).all()
    finally:
        if graph.value:
            lib.gaffa_hip_graph_destroy(graph)
        lib.gaffa_hip_stream_destroy(stream)
        lib.gaffa_hip_free(out)


def _free_bytes(lib):
    import ctypes

    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_kept_memory_goes_back(gpu):
    """What is kept is counted as free again after a C-ABI allocation that finds
    no memory (here more than any device has), and after the public release."""
    import ctypes

    import gaffa_amd

    lib = ctypes.CDLL(gaffa_amd.HIP_LIBRARY)
    x = np.random.default_rng(8).integers(1, 99, size=(1, 64 << 20)).astype(np.uint32)  # 256 MB
    for give_back in ("allocation", "release"):
        gaffa_amd.release_device_cache()
        gpu._preprocess_batch_gpu(x, window_samples=None, normalise=False)
        kept = _free_bytes(lib)
        if give_back == "allocation":
            p = ctypes.c_void_p()
            assert lib.gaffa_hip_malloc(ctypes.byref(p), ctypes.c_uint64(1 << 50)) != 0
        else:
            gaffa_amd.release_device_cache()
        assert _free_bytes(lib) >= kept + x.nbytes, give_back

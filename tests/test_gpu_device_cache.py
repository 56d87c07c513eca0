"""GPU: device memory kept between calls never carries one call into another."""

import threading

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
    bad = []

    def work(order):
        for k in order:
            x, plan, want = jobs[k]
            if _peaks(ffa_search_batch(x, plan)) != want:
                bad.append(k)

    work([0, 1, 2, 1, 0])
    threads = [threading.Thread(target=work, args=(o,)) for o in ([0, 1, 2] * 4, [2, 0, 1] * 4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    gpu.release_device_cache()
    work([2, 1, 0])
    assert bad == []

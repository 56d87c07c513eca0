"""Performance cases of the search path, each through a public entry point.

A case is one call (or the few calls that belong together) as a user's program
makes it, on inputs of the observation shapes that the package's workloads,
tests and benchmark use:

* one_*       ``ffa.ffa_search``: one host series, a plan in hand, peaks back.
              The shape of a script that looks at a single dedispersed series;
              the short one is the smallest call there is.
* batch       ``ffa.ffa_search_batch``: equal-length host series, one plan.
* octaves     ``ffa.FfaBatchedSearch.run``: resident series of different
              lengths, each with its own octave plan (bins 128..255).
* pipeline_*  ``pipeline.GpuSearchPipeline``: the resident filterbank through
              dedispersion, detrending, FFA search, candidate selection and the
              full fold of the best candidates.  ``small`` is the 64-channel
              brute-force search and returns its whole peak list, ``lband`` the
              1024-channel and ``large`` the 4096-channel subband search.
* subband     ``gaffa_hip_filterbank_transpose_u8`` and
              ``gaffa_hip_dedisperse_subband_u8`` through the C ABI on resident
              samples, as a program that keeps its own buffers calls them.
* brute       ``dedispersion.dedisperse_multi_dm``: host samples in, plane out.
* frontend    ``gaffa_hip_dedisperse_multi_u8`` and
              ``gaffa_hip_detrend_normalise_batch`` through the C ABI: what a
              program runs before any search of its own.
* pfold       ``pfold.fold_spectrum``: host dynamic spectrum to a folded cube.
* gradients   ``CandidateScorer.gradients``: forward and backward of a batch.

Peaks, sums and folds are the same bits in any correct implementation that
adds in the defined order, so their tolerance is "exact".
"""

from __future__ import annotations

import ctypes
import dataclasses
import math
from types import SimpleNamespace

import numpy as np
import torch

import gaffa_amd
from gaffa_amd import dedispersion, ffa, pfold
from gaffa_amd.pipeline import (DISPERSION_S, channel_frequencies, large_workload, lband_workload,
                                peak_records, search_candidates, small_workload)

FOLDED = 8  # the best candidates are folded in full


def listed() -> list:
    return [
        {"name": "one_short", "kind": "one", "nsamples": 32768, "tsamp": 256e-6,
         "period_min": 0.2, "period_max": 2.0, "duty": 0.09, "spacing": 2.0},
        {"name": "one_long", "kind": "one", "nsamples": 4193303, "tsamp": 64e-6,
         "period_min": 0.1, "period_max": 10.0, "duty": 0.20, "spacing": 1.5},
        {"name": "batch", "kind": "batch", "nseries": 24, "nsamples": 524291, "tsamp": 64e-6,
         "period_min": 0.1, "period_max": 10.0, "duty": 0.18, "spacing": 2.0},
        {"name": "octaves", "kind": "octaves", "nseries": 96, "log2_min": 18, "log2_max": 20,
         "per_tile": 16},
        {"name": "pipeline_small", "kind": "pipeline", "shape": "small", "nsamples": 131072,
         "ndm": 64},
        {"name": "pipeline_lband", "kind": "pipeline", "shape": "lband", "nsamples": 1 << 20,
         "ndm": 256},
        {"name": "pipeline_large", "kind": "pipeline", "shape": "large", "nsamples": 1 << 21,
         "ndm": 512},
        {"name": "subband", "kind": "subband", "nsamples": 262144, "nchans": 1024,
         "subband_channels": 32, "ndm": 192, "dm_step": 0.45},
        {"name": "brute", "kind": "brute", "nsamples": 100003, "nchans": 64, "ndm": 61,
         "dm_step": 1.0},
        {"name": "frontend", "kind": "frontend", "nsamples": 400003, "nchans": 96, "ndm": 128,
         "dm_step": 0.5},
        {"name": "pfold", "kind": "pfold", "nsamples": 262144, "nchans": 256, "out": 64,
         "dtype": "uint8", "nbin": 64, "period": 0.7143},
        {"name": "gradients", "kind": "gradients", "batch": 509},
    ]


def _log(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["one", "batch", "octaves", "pipeline", "pipeline", "subband", "brute",
                       "frontend", "pfold", "gradients"])
    if kind in ("one", "batch"):
        fast = rng.random() < 0.5
        c = {"kind": kind, "tsamp": 64e-6 if fast else 256e-6,
             "period_min": 0.1 if fast else 0.2, "period_max": rng.choice([1.0, 2.0, 5.0, 10.0]),
             "duty": rng.choice([0.09, 0.18, 0.20]), "spacing": rng.choice([1.5, 2.0])}
        if kind == "one":
            c["nsamples"] = _log(rng, 40000, 4200000)
        else:
            c["nsamples"] = _log(rng, 60000, 1100000)
            c["nseries"] = max(2, min(40, 12000000 // c["nsamples"] - rng.randrange(4)))
        # at least one full period of the longest trial
        c["period_max"] = min(c["period_max"], c["nsamples"] * c["tsamp"] / 4)
        return c
    if kind == "octaves":
        top = rng.choice([18, 19, 20])
        return {"kind": kind, "nseries": rng.randint(17, 96), "log2_min": top - rng.choice([1, 2]),
                "log2_max": top, "per_tile": rng.choice([8, 16, 32])}
    if kind == "pipeline":
        shape = rng.choice(["small", "lband", "large"])
        if shape == "small":
            return {"kind": kind, "shape": shape, "nsamples": _log(rng, 60000, 262144), "ndm": 64}
        n = _log(rng, 1 << 19, 1 << 20)
        return {"kind": kind, "shape": shape, "nsamples": n,
                "ndm": 128 * rng.randint(2, 4)}
    if kind == "subband":
        return {"kind": kind, "nsamples": _log(rng, 1 << 16, 1 << 18),
                "nchans": rng.choice([256, 500, 1024, 2048]),
                "subband_channels": rng.choice([16, 32, 64]), "ndm": rng.randint(40, 200),
                "dm_step": rng.uniform(0.1, 0.9)}
    if kind == "brute":
        return {"kind": kind, "nsamples": _log(rng, 20000, 200000),
                "nchans": rng.choice([16, 64, 100, 128]), "ndm": rng.randint(1, 128),
                "dm_step": rng.uniform(0.2, 1.5)}
    if kind == "frontend":
        return {"kind": kind, "nsamples": _log(rng, 100000, 1000000),
                "nchans": rng.choice([32, 64, 96, 128]), "ndm": rng.randint(8, 128),
                "dm_step": rng.uniform(0.2, 1.0)}
    if kind == "pfold":
        nchans = rng.choice([64, 128, 256])
        return {"kind": kind, "nsamples": _log(rng, 1 << 16, 1 << 18), "nchans": nchans,
                "out": rng.choice([nchans, nchans // 2, nchans // 4]),
                "dtype": rng.choice(["uint8", "uint16", "float32"]),
                "nbin": rng.choice([32, 64, 128]), "period": rng.uniform(0.2, 3.0)}
    return {"kind": kind, "batch": _log(rng, 33, 1024)}


# ----------------------------------------------------------------- inputs --

def _series(case: dict, count: int, seed: int) -> np.ndarray:
    """Unit-variance noise; every third series carries a pulse train."""
    rng = np.random.default_rng(seed)
    n = case["nsamples"]
    x = rng.standard_normal((count, n), dtype=np.float32)
    t = np.arange(n, dtype=np.float64) * case["tsamp"]
    for k in range(0, count, 3):
        lo = case["period_min"]
        period = lo * (case["period_max"] / lo) ** rng.uniform(0.1, 0.9)
        ph = (t / period + rng.uniform()) % 1.0 - 0.5
        width = 0.02
        amp = 12.0 / math.sqrt(n * width * math.sqrt(math.pi))
        x[k] += (amp * np.exp(-0.5 * (ph / width) ** 2)).astype(np.float32)
    return x


def _plan(case: dict):
    return ffa.make_riptide_plan(
        nsamples=case["nsamples"], tsamp=case["tsamp"], period_min=case["period_min"],
        period_max=case["period_max"], duty_cycle_max=case["duty"],
        width_trial_spacing=case["spacing"])


def _workload(case: dict, seed: int):
    """The package's workload of that shape.  The subband ones keep every k-th
    of their 128-trial DM segments, so that fewer trials still span the range;
    the small one's pulsar is faint (S/N about 20 of 120) and moves with the
    seed."""
    if case["shape"] == "small":
        w = small_workload(nsamples=case["nsamples"], seed=seed)
        rng = np.random.default_rng(seed)
        _, _, duty, _, _ = w.pulsars[0]
        return dataclasses.replace(w, pulsars=[(rng.uniform(0.3, 1.5), rng.uniform(5.0, 58.0),
                                                duty, 0.08, rng.uniform())])
    make = lband_workload if case["shape"] == "lband" else large_workload
    w = make(nsamples=case["nsamples"], seed=seed)
    keep, have = case["ndm"] // 128, len(w.dm_segments)
    at = [(2 * k + 1) * have // (2 * keep) for k in range(keep)]
    return dataclasses.replace(w, dm_segments=[w.dm_segments[k] for k in at])


def _samples(nsamples: int, nchans: int, seed: int) -> torch.Tensor:
    """uint8 noise of mean 128 and sigma 16, as digitised filterbanks have."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = torch.empty((nsamples, nchans), dtype=torch.float32, device="cuda")
    x.normal_(128.0, 16.0, generator=g)
    return x.round_().clamp_(0, 255).to(torch.uint8)


def _frequencies(nchans: int) -> np.ndarray:
    return channel_frequencies(nchans, 1520.0, -300.0 / nchans)


def _delays(dm, f, ref: float, tsamp: float) -> np.ndarray:
    d = DISPERSION_S * np.asarray(dm, np.float64)[..., None] * (f ** -2.0 - ref ** -2.0) / tsamp
    return np.rint(d).astype(np.int32)


def _brute_tables(case: dict, tsamp: float):
    f = _frequencies(case["nchans"])
    delays = _delays(np.arange(case["ndm"]) * case["dm_step"], f, float(f.max()), tsamp)
    return delays, case["nsamples"] - int(delays.max())


def _subband_tables(case: dict, tsamp: float = 64e-6, per_nominal: int = 32):
    """(coarse [groups][nchans], residual [ndm][nsub]) of nominal groups."""
    f = _frequencies(case["nchans"])
    ref, sbc, ndm = float(f.max()), case["subband_channels"], case["ndm"]
    dm = np.arange(ndm) * case["dm_step"]
    nominal = dm[::per_nominal]
    coarse = _delays(nominal, f, ref, tsamp)
    begin = np.arange(0, case["nchans"], sbc)
    end = np.minimum(begin + sbc, case["nchans"])
    mid = f[(begin + end - 1) // 2]
    resid = _delays(dm - nominal[np.arange(ndm) // per_nominal], mid, ref, tsamp)
    n_out = case["nsamples"] - int(coarse.max()) - int(resid.max())
    return coarse, resid, n_out


_FAN = [96, 192, 192, 192, 256, 512]   # the scorer's layers: inputs
_ROWS = [64, 64, 64, 64, 512, 1]       # and outputs, weights before biases


def _scorer_weights(seed: int) -> np.ndarray:
    rng = np.random.default_rng(seed + 1)
    parts = []
    for rows, fan in zip(_ROWS, _FAN):
        parts += [rng.normal(0.0, math.sqrt(2.0 / fan), rows * fan), np.zeros(rows)]
    p = np.concatenate(parts)
    return np.pad(p, (0, -len(p) % 8)).astype(np.float32)


def _scorer_arrays(case: dict, seed: int):
    rng = np.random.default_rng(seed)
    b = case["batch"]
    labels = (rng.random(b) < 0.3).astype(np.float32)
    cubes = rng.standard_normal((b, 32, 64), dtype=np.float32)
    patches = rng.standard_normal((b, 128), dtype=np.float32)
    phase = np.arange(64)[None, :] - rng.uniform(8, 56, b)[:, None]
    cubes += (0.8 * labels[:, None] * np.exp(-0.5 * (phase / 2.0) ** 2))[:, None, :].astype(
        np.float32)
    patches += (6.0 * labels[:, None]
                * np.exp(-0.5 * ((np.arange(128) - 64) / 3.0) ** 2)).astype(np.float32)
    return cubes, patches, labels


# ------------------------------------------------------------------ C ABI --

_U64, _I32, _I64, _PTR = ctypes.c_uint64, ctypes.c_int32, ctypes.c_int64, ctypes.c_void_p


class _Multi(ctypes.Structure):
    _fields_ = [("samples", _PTR), ("nsamples", _U64), ("nchans", _U64), ("chan_begin", _U64),
                ("chan_end", _U64), ("delays", _PTR), ("ndm", _U64), ("out", _PTR),
                ("out_nsamples", _U64), ("out_stride", _U64), ("max_block_spread", _I32)]


class _Transpose(ctypes.Structure):
    _fields_ = [("samples", _PTR), ("nsamples", _U64), ("nchans", _U64), ("chan_begin", _U64),
                ("chan_end", _U64), ("out", _PTR), ("out_stride", _U64), ("t_begin", _U64),
                ("t_count", _U64)]


class _Subband(ctypes.Structure):
    _fields_ = [("channels", _PTR), ("channel_stride", _U64), ("channel_length", _U64),
                ("nsamples", _U64), ("nsel", _U64), ("subband_channels", _U64),
                ("ndm_per_nominal", _U64), ("ndm", _U64), ("coarse_delays", _PTR),
                ("residual_delays", _PTR), ("out", _PTR), ("out_nsamples", _U64),
                ("out_stride", _U64), ("max_residual", _I32), ("max_coarse", _I32),
                ("groups", _PTR), ("ngroups", _U64), ("n_coarse_rows", _U64),
                ("max_group_ndm", _U64), ("residual_window", _I64)]


class _Preprocess(ctypes.Structure):
    _fields_ = [("data", _PTR), ("nseries", _U64), ("nsamples", _U64), ("stride", _U64),
                ("input_is_u32", _I32), ("detrend", _I32), ("scrunch_factor", _U64),
                ("median_window", _U64), ("normalise", _I32), ("reject_constant", _I32),
                ("workspace", _PTR), ("workspace_bytes", _U64), ("status", _PTR)]


def _library():
    lib = ctypes.CDLL(gaffa_amd.HIP_LIBRARY)
    lib.gaffa_hip_last_error.restype = ctypes.c_char_p
    lib.gaffa_hip_preprocess_workspace_bytes.restype = _U64
    lib.gaffa_hip_preprocess_workspace_bytes.argtypes = [_U64] * 3
    lib.gaffa_hip_subband_channel_stride.restype = _U64
    lib.gaffa_hip_subband_channel_stride.argtypes = [_U64, _I32, _I32]
    for name in ("gaffa_hip_dedisperse_multi_u8", "gaffa_hip_filterbank_transpose_u8",
                 "gaffa_hip_dedisperse_subband_u8", "gaffa_hip_detrend_normalise_batch"):
        getattr(lib, name).argtypes = [_PTR, _PTR]
    return lib


def _call(lib, name: str, args) -> None:
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    if getattr(lib, name)(ctypes.byref(args), stream) != 0:
        raise RuntimeError(f"{name}: {lib.gaffa_hip_last_error().decode()}")


MEDIAN_POINTS = 101


def _scrunch(case: dict) -> int:
    """Samples per low-resolution point of the 1 s running median at 256 us."""
    return max(2, min(3907, case["nsamples"] // 8) // MEDIAN_POINTS)


def _filterbank(data: np.ndarray, tsamp: float):
    """What the dedispersion calls take: samples and the header fields they read."""
    return SimpleNamespace(
        data=data[:, None, :],
        header=SimpleNamespace(nbits=8, tsamp=tsamp,
                               frequency_table=list(_frequencies(data.shape[1]))))


# ---------------------------------------------------------------- prepare --

def prepare(case: dict, seed: int):
    kind = case["kind"]
    s = SimpleNamespace(case=case, kind=kind)
    if kind == "one":
        s.series, s.plan = _series(case, 1, seed)[0], _plan(case)
    elif kind == "batch":
        s.series, s.plan = _series(case, case["nseries"], seed), _plan(case)
    elif kind == "octaves":
        from gaffa_amd.pipeline import batched_workload

        w = batched_workload(case["nseries"], seed, log2_min=case["log2_min"],
                             log2_max=case["log2_max"], injected=0.2)
        s.threshold = w.snr_threshold
        s.search = w.search(series_per_tile=case["per_tile"])
    elif kind == "pipeline":
        s.workload = _workload(case, seed)
        s.pipe = s.workload.pipeline()
        s.pipe.generate(s.workload.synth_spec())
    elif kind == "subband":
        coarse, resid, n_out = _subband_tables(case)
        s.lib = _library()
        s.x = _samples(case["nsamples"], case["nchans"], seed)
        stride = s.lib.gaffa_hip_subband_channel_stride(case["nsamples"], int(coarse.max()),
                                                        int(resid.max()))
        s.channels = torch.empty((case["nchans"], stride), dtype=torch.uint8, device="cuda")
        s.coarse = torch.from_numpy(coarse).cuda()
        s.resid = torch.from_numpy(resid).cuda()
        s.out = torch.empty((case["ndm"], n_out), dtype=torch.int32, device="cuda")
        s.transpose = _Transpose(s.x.data_ptr(), case["nsamples"], case["nchans"], 0,
                                 case["nchans"], s.channels.data_ptr(), stride, 0, 0)
        s.args = _Subband(s.channels.data_ptr(), stride, 0, case["nsamples"], case["nchans"],
                          case["subband_channels"], 32, case["ndm"], s.coarse.data_ptr(),
                          s.resid.data_ptr(), s.out.data_ptr(), n_out, n_out, int(resid.max()),
                          int(coarse.max()), None, 0, 0, 0, 0)
    elif kind == "brute":
        x = _samples(case["nsamples"], case["nchans"], seed).cpu().numpy()
        s.filterbank = _filterbank(x, 256e-6)
    elif kind == "frontend":
        delays, n_out = _brute_tables(case, 256e-6)
        ndm = case["ndm"]
        stride = (n_out + 63) // 64 * 64
        f = _scrunch(case)
        s.lib = _library()
        s.x = _samples(case["nsamples"], case["nchans"], seed)
        s.delays = torch.from_numpy(delays).cuda()
        s.plane = torch.zeros((ndm, stride), dtype=torch.float32, device="cuda")
        s.status = torch.zeros(ndm, dtype=torch.int32, device="cuda")
        need = s.lib.gaffa_hip_preprocess_workspace_bytes(ndm, n_out, f)
        s.workspace = torch.empty(need, dtype=torch.uint8, device="cuda")
        spread = max(int(b.max()) - int(b.min())
                     for i in range(0, ndm, 16) for c in range(0, case["nchans"], 32)
                     for b in (delays[i:i + 16, c:c + 32],))
        s.n_out = n_out
        s.multi = _Multi(s.x.data_ptr(), case["nsamples"], case["nchans"], 0, case["nchans"],
                         s.delays.data_ptr(), ndm, s.plane.data_ptr(), n_out, stride, spread)
        s.args = _Preprocess(s.plane.data_ptr(), ndm, n_out, stride, 1, 1, f, MEDIAN_POINTS, 1, 1,
                             s.workspace.data_ptr(), need, s.status.data_ptr())
    elif kind == "pfold":
        s.spectrum = SimpleNamespace(data=_spectrum(case, seed), tsamp=256e-6)
    else:
        s.cubes, s.patches, s.labels = _scorer_arrays(case, seed)
        s.net = gaffa_amd.CandidateScorer(capacity=1024)
        s.net.parameters = _scorer_weights(seed)
    return s


def _spectrum(case: dict, seed: int) -> np.ndarray:
    x = _samples(case["nsamples"], case["nchans"], seed)
    if case["dtype"] == "float32":
        return (x.float() - 128.0).cpu().numpy()
    return x.cpu().numpy().astype(case["dtype"])


# -------------------------------------------------------------------- run --

_PEAK_FIELDS = ("period", "frequency", "width", "phase", "shift", "bins", "snr")
_CANDIDATE_FIELDS = ("dm_index", "period", "width", "snr", "peak_count", "dm_index_min",
                     "dm_index_max", "frequency_min", "frequency_max")


def _table(columns: dict, room: int) -> dict:
    """A list of records as columns and its length.  The columns have `room`
    places (doubled until the list fits), zero behind the list's end."""
    n = len(next(iter(columns.values())))
    while room < n:
        room *= 2
    out = {"count": n}
    for k, v in columns.items():
        out[k] = np.zeros(room)
        out[k][:n] = v
    return out


def _peak_table(peaks, room: int, series=None) -> dict:
    c = {f: [getattr(p, f) for p in peaks] for f in _PEAK_FIELDS}
    if series is not None:
        c["series"] = series
    return _table(c, room)


def run(s):
    if s.kind == "one":
        return _peak_table(ffa.ffa_search(s.series, s.plan, backend="gpu"), 8192)
    if s.kind == "batch":
        found = ffa.ffa_search_batch(s.series, s.plan)
        return _peak_table([p for _, p in found], 65536, [i for i, _ in found])
    if s.kind == "octaves":
        found, _ = s.search.run(s.threshold)
        return _peak_table([p for _, p in found], 65536, [i for i, _ in found])
    if s.kind == "pipeline":
        s.pipe.run()
        if s.case["shape"] == "small":
            r = peak_records(s.pipe)
            return _table({"dm": r["dm"], "dm_index": r["dm_index"],
                           **{f: r["peak"][f] for f in _PEAK_FIELDS}}, 65536)
        cands = search_candidates(s.pipe, s.workload)
        out = _table({f: [getattr(c, f) for c in cands] for f in _CANDIDATE_FIELDS}, 32768)
        out["peaks"] = s.pipe.peak_count
        out["cubes"] = s.pipe.fold_candidates_full(cands[:FOLDED], keep_cubes=True)[1]
        s.pipe.wait_peaks()
        return out
    if s.kind == "subband":
        _call(s.lib, "gaffa_hip_filterbank_transpose_u8", s.transpose)
        _call(s.lib, "gaffa_hip_dedisperse_subband_u8", s.args)
        return s.out
    if s.kind == "brute":
        r = dedispersion.dedisperse_multi_dm(s.filterbank, dm_low=0.0, dm_step=s.case["dm_step"],
                                             ndm=s.case["ndm"], backend="gpu")
        return r.data.view(np.int32)
    if s.kind == "frontend":
        _call(s.lib, "gaffa_hip_dedisperse_multi_u8", s.multi)
        _call(s.lib, "gaffa_hip_detrend_normalise_batch", s.args)
        return {"plane": s.plane[:, :s.n_out], "status": s.status}
    if s.kind == "pfold":
        r = pfold.fold_spectrum(s.spectrum, period=s.case["period"], nbin=s.case["nbin"],
                                nsubband=s.case["out"])
        return {"cube": r.cube, "exposure": r.exposure, "profile": r.profile}
    loss, grads = s.net.gradients(s.cubes, s.patches, s.labels)
    return {"loss": float(loss), "gradients": grads}


# ------------------------------------------------------------------- work --

def _search_work(tasks, nsamples: int, widths: int) -> dict:
    """One series: its samples once; the adds of the tree and of the boxcars."""
    rows = tasks["rows"].astype(np.float64)
    cells = rows * tasks["bins"]
    levels = np.ceil(np.log2(np.maximum(rows, 1.0)))
    evaluated = tasks["rows_eval"].astype(np.float64) * tasks["bins"]
    return {"bytes": 4.0 * nsamples,
            "flops": float((cells * levels).sum() + 2.0 * widths * evaluated.sum())}


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("one", "batch"):
        p = _plan(case)
        w = _search_work(p.tasks, case["nsamples"], len(p.width_trials))
        k = case.get("nseries", 1)
        return {"bytes": k * w["bytes"], "flops": k * w["flops"]}
    if kind == "octaves":
        n = (2 ** case["log2_min"] + 2 ** case["log2_max"]) // 2
        p = ffa.make_octave_plan(nsamples=n, tsamp=64e-6)
        w = _search_work(p.tasks, n, len(p.width_trials))
        return {"bytes": case["nseries"] * w["bytes"], "flops": case["nseries"] * w["flops"]}
    if kind == "pipeline":
        small = case["shape"] == "small"
        nchans = {"small": 64, "lband": 1024, "large": 4096}[case["shape"]]
        sub = {"small": 1, "lband": 32, "large": 64}[case["shape"]]
        n, ndm = case["nsamples"], case["ndm"]
        p = ffa.make_riptide_plan(
            nsamples=n, tsamp=256e-6 if small else 64e-6, period_min=0.2 if small else 0.1,
            period_max=2.0 if small else 10.0, duty_cycle_max=0.09 if small else 0.18,
            width_trial_spacing=2.0)
        w = _search_work(p.tasks, n, len(p.width_trials))
        adds = n * nchans * ndm if small else n * (nchans * ndm / 32 + nchans / sub * ndm)
        return {"bytes": float(n * nchans), "flops": ndm * w["flops"] + float(adds)}
    if kind == "subband":
        _, _, n_out = _subband_tables(case)
        nsub = -(-case["nchans"] // case["subband_channels"])
        groups = -(-case["ndm"] // 32)
        return {"bytes": float(case["nsamples"] * case["nchans"] + 4 * case["ndm"] * n_out),
                "flops": float(n_out * (groups * case["nchans"] + case["ndm"] * nsub))}
    if kind in ("brute", "frontend"):
        _, n_out = _brute_tables(case, 256e-6)
        per = 6 if kind == "frontend" else 0  # conversion, baseline, statistics, scaling
        return {"bytes": float(case["nsamples"] * case["nchans"] + 4 * case["ndm"] * n_out),
                "flops": float(n_out * case["ndm"] * (case["nchans"] + per))}
    if kind == "pfold":
        cells = case["nsamples"] * case["nchans"]
        nsub = math.ceil(case["nsamples"] * 256e-6 / 10.0)
        return {"bytes": float(cells * np.dtype(case["dtype"]).itemsize
                               + 4 * nsub * case["out"] * case["nbin"]),
                "flops": float(cells + 3 * case["nsamples"] * case["out"])}
    b = case["batch"]
    macs = 64 * 64 * (96 + 3 * 192) + 256 * 512 + 512  # per candidate, forward
    return {"bytes": float(b * (32 * 64 + 128 + 1) * 4 + 2 * 4 * 175000),
            "flops": float(3 * 2 * macs * b)}


# -------------------------------------------------------------- tolerance --

def tolerance(case: dict):
    if case["kind"] == "gradients":
        # bfloat16 weights, activations and signals, float32 sums: 1.5e-2 off
        # the 64-bit gradients at 509 candidates, more for smaller batches
        return {"rel": 5e-2}
    if case["kind"] == "frontend":
        # float32 medians of the low-resolution points (sums of ~1e4, samples
        # of unit variance afterwards): 2.1e-6 off the 64-bit plane
        return {"rel": 1e-5}
    return "exact"


# ------------------------------------------------------------------ exact --

def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "subband":
        coarse, resid, n_out = _subband_tables(case)
        x = _samples(case["nsamples"], case["nchans"], seed).T.contiguous().to(torch.int16)
        sbc, nch = case["subband_channels"], case["nchans"]
        out = torch.zeros((case["ndm"], n_out), dtype=torch.int64, device="cuda")
        for g in range(len(coarse)):
            m = n_out + int(resid.max())
            for b, c0 in enumerate(range(0, nch, sbc)):
                part = torch.zeros(m, dtype=torch.int64, device="cuda")
                for c in range(c0, min(nch, c0 + sbc)):
                    d = int(coarse[g, c])
                    part += x[c, d:d + m]
                for i in range(32 * g, min(case["ndm"], 32 * g + 32)):
                    r = int(resid[i, b])
                    out[i] += part[r:r + n_out]
        return out
    if kind in ("brute", "frontend"):
        delays, n_out = _brute_tables(case, 256e-6)
        x = _samples(case["nsamples"], case["nchans"], seed).T.contiguous()
        plane = torch.zeros((case["ndm"], n_out), dtype=torch.int64, device="cuda")
        for i in range(case["ndm"]):
            for c in range(case["nchans"]):
                d = int(delays[i, c])
                plane[i] += x[c, d:d + n_out]
        if kind == "brute":
            return plane
        return {"plane": _detrended(plane.double(), _scrunch(case)),
                "status": torch.zeros(case["ndm"], dtype=torch.int64)}
    if kind == "pfold":
        return _folded(case, _spectrum(case, seed))
    if kind == "gradients":
        return _network_gradients(case, seed)
    # peaks and candidates are selections over millions of float32 statistics
    # whose order is part of the definition: no 64-bit value stands for them
    return None


def _detrended(x: torch.Tensor, f: int) -> torch.Tensor:
    n = x.shape[1]
    m, half = n // f, MEDIAN_POINTS // 2
    low = x[:, :m * f].reshape(x.shape[0], m, f).mean(2)
    pad = torch.cat([low[:, :1].expand(-1, half), low, low[:, -1:].expand(-1, half)], 1)
    med = torch.stack([row.unfold(0, MEDIAN_POINTS, 1).median(1).values for row in pad])
    p = (torch.arange(n, device=x.device, dtype=torch.float64) - 0.5 * (f - 1)) / f
    p = p.clamp(0.0, m - 1.0)
    lo = p.floor().long().clamp(max=m - 2)
    fr = p - lo
    x = x - ((1.0 - fr) * med[:, lo] + fr * med[:, lo + 1])
    return (x - x.mean(1, keepdim=True)) / x.std(1, unbiased=False, keepdim=True)


def _folded(case: dict, data: np.ndarray) -> dict:
    n, nbin, out, tsamp = case["nsamples"], case["nbin"], case["out"], 256e-6
    per = math.floor(10.0 / tsamp + 0.5)
    nsub = -(-n // per)
    x = data.reshape(n, out, -1).astype(np.float64).mean(2)
    step = tsamp / case["period"] * nbin
    i = np.arange(n, dtype=np.float64)
    low, high = i * step, i * step + step
    sums = np.zeros((nsub, nbin, out))
    expo = np.zeros((nsub, nbin))
    sub = np.arange(n) // per
    k = np.floor(low)
    while True:
        w = np.minimum(high, k + 1.0) - np.maximum(low, k)
        use = w > 0.0
        if not use.any():
            break
        at = (sub[use] * nbin + (k[use].astype(np.int64) % nbin))
        order = np.argsort(at, kind="stable")
        edges = np.flatnonzero(np.r_[True, np.diff(at[order]) != 0])
        cells = at[order][edges]
        weighted = x[use][order] * w[use][order][:, None]
        sums.reshape(-1, out)[cells] += np.add.reduceat(weighted, edges)
        expo.reshape(-1)[cells] += np.add.reduceat(w[use][order], edges)
        k = k + 1.0
    cube = np.where(expo[:, :, None] > 0, sums / np.maximum(expo, 1e-300)[:, :, None], 0.0)
    return {"cube": cube.transpose(0, 2, 1), "exposure": expo, "profile": None}


def _network_gradients(case: dict, seed: int) -> dict:
    p = torch.tensor(_scorer_weights(seed).astype(np.float64), requires_grad=True)
    cubes, patches, labels = (torch.from_numpy(a).double() for a in _scorer_arrays(case, seed))
    layers, at = [], 0
    for rows, fan in zip(_ROWS, _FAN):
        layers.append((p[at:at + rows * fan].reshape(rows, fan),
                       p[at + rows * fan:at + rows * fan + rows]))
        at += rows * fan + rows
    x = cubes
    for w, b in layers[:4]:
        x = torch.relu(torch.nn.functional.conv1d(
            torch.nn.functional.pad(x, (1, 1), mode="circular"),
            w.reshape(64, 3, -1).permute(0, 2, 1), b))
    f = torch.cat([x.mean(2), x.max(2).values, patches], 1)
    h = torch.relu(f @ layers[4][0].T + layers[4][1])
    z = h @ layers[5][0][0] + layers[5][1]
    loss = torch.nn.functional.binary_cross_entropy_with_logits(z, labels)
    loss.backward()
    return {"loss": float(loss.detach()), "gradients": p.grad}

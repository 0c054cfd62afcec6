"""Autotuner of the engine's launch shapes: measures the candidates of each
tunable option on the device for one (basis, operator) shape and batch size
and keeps the fastest.

Tunables (options of pnfam_gpu_set_option):
  proj_rows     16-row tiles per wave of the projection kernels (1..4): more
                rows reuse each loaded B column more often but hold more
                accumulators and lower the waves per SIMD;
  proj_freqs    frequencies per wave of the FP64 projection (1, 2): two share
                the psi operand loads of every k step, at twice the
                accumulators and staged fields; 4: four waves of a workgroup,
                one frequency each, share the psi operands through LDS;
  proj_stages   depth of the projection's operand pipeline (1, 2): the loads
                of that many k steps ahead are in flight during the products;
  proj_freqs_rt1  proj_freqs for the mean-field tiles of one row tile (0: the
                same as proj_freqs), tuned after the three above: their few
                products per staged chunk favour another grouping;
  fp64_density  the FP64 density kernel: one wave per 16 grid points (0), two
                waves splitting the tables and exchanging the products through
                LDS (1), or two waves splitting the rows by spin with transposed
                products and no exchange (2).
No projection option changes any result: every output element is summed in
the same order whatever the tile shape.  The density kernels differ in the
order four of the 28 densities add their same-spin and opposite-spin parts
(0 against 1: 1e-16 relative) and, for 2, in how the columns of a block are
grouped into tiles (a few units in the last place of the largest element).

These are the shapes of the kernels that contract over all grid points; the
factored stage, which FP64 solves take on a product basis (fp64_separable reads
1), has none, so there a tuning changes no solve.

The measurement is the FP64 grid stage over all points
(pnfam_gpu_calc_hamiltonian) on random amplitudes, run in `batch` replica slots
so that it takes the launch path of batches that size, timed with the engine's
HIP-event profile, best of `repeats`; the per-unit calls are left as they were
(unit_replicas, unit_general).  The density and projection kernels are
independent, so their options are tuned apart: the density option by the
density time, the projection options (every combination) by the projection
time, then proj_freqs_rt1 by the projection time with those applied.
Results are cached in a JSON file keyed by the problem shape and batch size
(PNFAM_GPU_TUNE_CACHE, default ~/.cache/pynfam_amd/tune.json).  A shape found
in neither that cache nor the table shipped with the package
(tuning_mi355x.json: choices measured on an MI355X for the benchmark shapes)
is measured.
"""
from __future__ import annotations

import itertools
import json
import os
import time

import numpy as np

SPACE = {"proj_rows": (1, 2, 3, 4), "proj_freqs": (1, 2, 4), "proj_stages": (1, 2), "fp64_density": (0, 1, 2),
         "proj_freqs_rt1": (0, 1, 2, 4)}
DENSITY_OPTIONS = ("fp64_density",)
PROJECTION_OPTIONS = ("proj_rows", "proj_freqs", "proj_stages")
RT1_OPTIONS = ("proj_freqs_rt1",)
DEFAULT_CACHE = os.path.join(os.path.expanduser("~"), ".cache", "pynfam_amd", "tune.json")
SHIPPED = os.path.join(os.path.dirname(os.path.abspath(__file__)), "tuning_mi355x.json")


def shape_key(eng, batch):
    b = eng.prob.basis
    return f"dqp{b.dqp}-nb{b.nb}-nghl{b.nghl}-nxy{eng.nxy}-K{eng.prob.K}-{eng.prob.operator}-batch{batch}"


def _cache_path():
    return os.environ.get("PNFAM_GPU_TUNE_CACHE", DEFAULT_CACHE)


def _read(path):
    try:
        with open(path) as fh:
            return json.load(fh)
    except (OSError, ValueError):
        return {}


def _load_cache():
    return _read(_cache_path())


def _store_cache(cache):
    path = _cache_path()
    try:
        os.makedirs(os.path.dirname(path), exist_ok=True)
        tmp = path + ".tmp"
        with open(tmp, "w") as fh:
            json.dump(cache, fh, indent=1, sort_keys=True)
        os.replace(tmp, path)
    except OSError:
        pass   # a read-only home: the choice still applies to this engine


def _stage_ms(eng, args, repeats, kernel):
    best = float("inf")
    for _ in range(repeats):
        eng.profile(True)
        eng.calc_hamiltonian(args)
        p = eng.profile_read()
        eng.profile(False)
        best = min(best, p[kernel]["ms"] if kernel in p else 0.0)
    return best


def tune(eng, batch=64, repeats=3, use_cache=True, seed=0):
    """Measures every combination of SPACE on eng's problem with `batch`
    replica slots, applies the fastest to eng and returns
    {"settings": {...}, "ms": {...}, "key": ..., "cached": bool, "seconds": ...}."""
    key = shape_key(eng, batch)
    cache = _load_cache() if use_cache else {}
    known = dict(_read(SHIPPED), **cache) if use_cache else {}
    if key in known:
        for k, v in known[key]["settings"].items():
            eng.set_option(k, v)
        return dict(known[key], key=key, cached=True)
    t0 = time.perf_counter()
    rng = np.random.default_rng(seed)
    # amplitudes of the calc_dHsp_interface argument order; any values serve timing
    args = rng.standard_normal((8, eng.nxy))
    old = [(n, eng.get_option(n)) for n in ("unit_replicas", "unit_general")]   # the first sets the second
    timings, settings = {}, {}
    try:
        eng.set_option("unit_replicas", batch)
        eng.calc_hamiltonian(args)   # workspace and code objects outside the timing
        eng.set_option("proj_freqs_rt1", 0)
        for names, kernel in ((DENSITY_OPTIONS, "density"), (PROJECTION_OPTIONS, "project"), (RT1_OPTIONS, "project")):
            part = {}
            for combo in itertools.product(*(SPACE[n] for n in names)):
                for n, v in zip(names, combo):
                    eng.set_option(n, v)
                part[",".join(f"{n}={v}" for n, v in zip(names, combo))] = _stage_ms(eng, args, repeats, kernel)
            best = min(part, key=part.get)
            for kv in best.split(","):
                settings[kv.split("=")[0]] = int(kv.split("=")[1])
                eng.set_option(kv.split("=")[0], int(kv.split("=")[1]))
            timings.update({f"{kernel}:{k}": v for k, v in part.items()})
    finally:
        for n, v in old:
            eng.set_option(n, v)
    rec = {"settings": settings, "ms": timings, "batch": batch, "seconds": time.perf_counter() - t0}
    if use_cache:
        cache[key] = rec
        _store_cache(cache)
    return dict(rec, key=key, cached=False)

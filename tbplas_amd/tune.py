"""Autotuner for the launch shape of the propagation kernels.

For a prepared Hamiltonian, a state count and a precision it times a few
Chebyshev steps (HIP events on the library stream, after warm-up steps) for
every candidate (persistent blocks per CU, LDS staging of the slice rows)
and keeps the fastest; for a Hamiltonian with spatial tiles it then times
the best shape with three, four and five terms per pass and with resident
passes and keeps the fastest.  A shape is (blocks per CU, staging, terms per
pass: 1, 3, 4, 5, or RESIDENT plus the terms per pass of runs whose tables do
not fit resident passes; RESIDENT alone: five).
Results are cached per (device name, library build, instances, rows, stored
elements, widest slice, value layout, row order and tile count, states,
precision) in memory and in a JSON file
(``$TBPLAS_AMD_TUNE_CACHE``, default ``~/.cache/tbplas_amd/tune.json``).
"""
import json
import os
import threading

import numpy as np

from . import _lib

__all__ = ["autotune", "apply", "CANDIDATES"]

CANDIDATES = [(bpc, stage) for bpc in (4, 8, 12, 16) for stage in (True, False)]
# untuned: blocks per CU and staging; the terms per pass are those the
# tiles of auto_tile_nm are sized for (sample.pass_terms)
DEFAULT = (16, True)
# added to the terms per pass of a shape that runs resident passes (up to a
# whole step)
RESIDENT = 32

_lock = threading.Lock()
_mem = {}


def _cache_path():
    return os.environ.get("TBPLAS_AMD_TUNE_CACHE",
                          os.path.join(os.path.expanduser("~"), ".cache", "tbplas_amd",
                                       "tune.json"))


def _load_disk():
    try:
        with open(_cache_path()) as f:
            return json.load(f)
    except (OSError, ValueError):
        return {}


def _save_disk(d):
    p = _cache_path()
    try:
        os.makedirs(os.path.dirname(p), exist_ok=True)
        tmp = p + ".tmp"
        with open(tmp, "w") as f:
            json.dump(d, f, indent=1, sort_keys=True)
        os.replace(tmp, p)
    except OSError:
        pass


def _key(hams, K):
    import torch
    infos = [H.info() for H in hams]
    H0 = hams[0]
    dev = torch.cuda.get_device_name(H0.handle.device)
    st = os.stat(_lib.LIB_PATH)          # a rebuilt library is tuned afresh
    lib = f"{st.st_size}.{int(st.st_mtime)}"
    n = sum(i["n"] for i in infos)
    pad = sum(i["padded"] for i in infos)
    w = max(i["max_width"] for i in infos)
    real = all(i["real_values"] for i in infos)
    # the row order and the tiles change which shape wins
    order = "|".join(f"{int(getattr(H, 'ordered', False))}.{getattr(H, 'ntiles', 0)}"
                     for H in hams)
    return (f"{dev}|lib={lib}|inst={len(hams)}|n={n}|pad={pad}|w={w}|real={int(real)}"
            f"|order={order}|K={K}|p={H0.precision}")


def autotune(H, K, bes, steps=6, warmup=2, candidates=None, use_cache=True):
    """Pick (blocks_per_cu, stage, terms per pass) for Hamiltonian H
    (or a list of Hamiltonians run as one batch) and K states each; returns
    (best, timings) and leaves the handle set to the best shape."""
    from .tbpm import DosRun
    hams = list(H) if isinstance(H, (list, tuple)) else [H]
    H = hams[0]
    key = _key(hams, K)
    with _lock:
        if use_cache:
            if key in _mem:
                best = tuple(_mem[key])
                _set(H.handle, best)
                return best, None
            disk = _load_disk()
            if key in disk and len(disk[key]) == 3:
                best = (int(disk[key][0]), bool(disk[key][1]), int(disk[key][2]))
                _mem[key] = best
                _set(H.handle, best)
                return best, None
        rng = np.random.default_rng(0)
        psis = []
        for Hi in hams:
            psi = np.exp(2j * np.pi * rng.random((K, Hi.n)))
            psis.append(psi / np.linalg.norm(psi, axis=1, keepdims=True))
        def timed(shape):
            _set(H.handle, shape)
            run = DosRun(hams, bes, psis, warmup + steps)
            run.advance(warmup)
            ms = run.advance(steps) / steps
            run.close()
            return ms

        timings = {}
        for cand in candidates or CANDIDATES:
            timings[cand + (1,)] = timed(cand + (1,))
        best = min(timings, key=timings.get)
        if all(getattr(Hi, "tiled", False) for Hi in hams):
            for terms in (3, 4, 5, RESIDENT):
                blocked = best[:2] + (terms,)
                timings[blocked] = timed(blocked)
            best = min(timings, key=timings.get)
        _set(H.handle, best)
        _mem[key] = best
        if use_cache:
            disk = _load_disk()
            disk[key] = [best[0], best[1], best[2]]
            _save_disk(disk)
        return best, timings


def _set(handle, shape):
    handle.set_tuning(shape[0], shape[1])
    terms = int(shape[2])
    resident = terms >= RESIDENT
    if resident:
        terms = terms - RESIDENT or 5
    handle.set_blocking(terms > 1, terms=max(terms, 3))
    handle.set_resident(resident)


def _few_steps(n, K, prec, steps):
    """Whether so few steps on a new Hamiltonian of n rows do not pay for the
    tables of resident passes.  Below some 70,000 rows these take longer to
    make than the tiles' (ms, one complex128 state: 0.8 / 0.3 at 2,100 rows,
    1.6 / 0.5 at 8,300, 2.7 / 1.5 at 33,000; 5.3 / 5.6 at 131,600, and less
    from there on), and a step gains 8 to 20 us.  Steps after which they are
    even: 65, 107, 140 there, 54 to 162 for one complex64 state, 36 to 162
    for four; 10 to 50 with more than 32 bytes a row (115 once), AC and DC
    runs 10 to 70."""
    from .sample import _row_bytes
    return n < 70_000 and steps < (100 if _row_bytes(K, prec) <= 32 else 40)


def apply(H, K, bes, enabled=True, steps=None):
    """Tune when enabled, otherwise use the default shape: resident passes
    (H: one Hamiltonian or the list of a batch).  With `steps`, the time
    steps of all runs that H was made for, tile passes where these are too
    few for the tables of resident passes.  Returns the shape."""
    from .sample import pass_terms
    hams = list(H) if isinstance(H, (list, tuple)) else [H]
    prec = "fp32" if hams[0].precision == _lib.TBG_FP32 else "fp64"
    if enabled:
        shape = autotune(H, K, bes)[0]
    else:
        shape = DEFAULT + (RESIDENT + pass_terms(K, prec),)
    if shape[2] >= RESIDENT and steps is not None and \
            _few_steps(sum(Hi.n for Hi in hams), K, prec, steps):
        shape = tuple(shape[:2]) + (shape[2] - RESIDENT or 5,)
    _set(hams[0].handle, shape)
    return shape

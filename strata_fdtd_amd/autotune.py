"""Autotuner for the fused step's launch shape (rows per wave, planes per wave,
waves per LDS-sharing j-stack).

For one grid shape it times each candidate over a few device steps (HIP events
on the solver's stream, after one warm-up launch), keeps the fastest and
stores it in the tiling cache that ``tuning.pick_tiling`` reads. Timing runs
real steps on the solver (which keep advancing it), so tune on a scratch
solver or call ``solver.reset()`` afterwards.

The launch shape is of single steps. A solver that takes several steps per pass
(one made without a launch shape) goes on doing so where that is faster still than
its fastest single step; the shape then serves the steps that passes leave.
"""

from __future__ import annotations

import itertools

from . import _native
from .tuning import ROW_CHOICES, STACK_CHOICES, normalize_tiling, store_tiling


def candidate_tilings(shape, rows=ROW_CHOICES, planes=(1, 2, 4, 8, 12, 16, 24, 32, 48, 64), stacks=STACK_CHOICES):
    nx, ny = shape[0], shape[1]
    out = []
    for r, p, w in itertools.product(rows, planes, stacks):
        if p <= nx and r <= max(2, ny) and (w == 1 or r * w <= ny):
            out.append((r, p, w))
    return out


def time_tiling(solver, tiling, steps: int = 10) -> float:
    """Milliseconds per step for one launch shape (device time)."""
    import ctypes as C
    solver.set_tiling(*normalize_tiling(tiling))
    solver._prepare(steps + 2)
    _native.call("fdtd_step_n", solver._ctx, 1)        # warm-up (code object load)
    solver._advance_host(1)
    ms = C.c_float()
    _native.call("fdtd_time_steps", solver._ctx, steps, 0, C.byref(ms))
    solver._advance_host(steps)
    return ms.value / steps


def _time_passes(solver, steps: int) -> float:
    """Milliseconds per step in passes (device time)."""
    import ctypes as C
    n = 3 * ((steps + 2) // 3)
    solver._prepare(n + 3)
    _native.call("fdtd_step_n", solver._ctx, 3)
    solver._advance_host(3)
    ms = C.c_float()
    _native.call("fdtd_time_steps", solver._ctx, n, 0, C.byref(ms))
    solver._advance_host(n)
    return ms.value / n


def autotune(solver, candidates=None, steps: int = 10, store: bool = True, verbose: bool = False):
    """Pick the fastest (rows, planes, stack) for this solver's shape; returns
    (best, table) with table rows (rows, planes, stack, ms). 192^3: 38 us a step with
    the fastest shape, 19 in passes, which it therefore keeps."""
    shape = solver.shape
    passes = solver._passes
    solver._prepare(1)               # materials too, before passes are switched off
    cands = [normalize_tiling(t) for t in (candidates or candidate_tilings(shape))]
    table = []
    for t in cands:
        ms = time_tiling(solver, t, steps)
        table.append((*t, ms))
        if verbose:
            print(f"[autotune] {shape} rows={t[0]} planes={t[1]} stack={t[2]}: {ms * 1e3:.1f} us/step", flush=True)
    best = min(table, key=lambda e: e[3])
    solver.set_tiling(*best[:3])
    if passes:
        solver._allow_passes(True)
        ms = _time_passes(solver, steps)
        if verbose:
            print(f"[autotune] {shape} passes: {ms * 1e3:.1f} us/step", flush=True)
        solver._allow_passes(ms < best[3])
    if store:
        store_tiling(shape, not solver.grid.is_uniform, bool(solver._ade_tensors), best[:3], best[3])
    return tuple(best[:3]), table

"""The kernels of a pass that small grids do not pick by themselves: each workgroup
size with several planes, k segments and j windows per workgroup, ordinary and
non-temporal stores, uniform and nonuniform grids, against the oracle or single steps;
and the design passes with non-temporal stores (grids beyond the Infinity Cache)
against the per-cell kernels. Bit for bit: the operations and their order are the
same, so the tolerance is 0."""

import ctypes as C

import numpy as np
import pytest

from helpers import make_solver, oracle_problem, seeded_scenario
from oracle import cpu

pytestmark = pytest.mark.gpu

FIELDS = ("p", "vx", "vy", "vz")
SHAPE = (22, 90, 70)
# threads, k segments, planes per workgroup (22: all, 21 and 1, 8 and a rest of 6)
TILES = [(256, 1, 22), (256, 2, 8), (512, 1, 21), (512, 3, 4), (1024, 1, 22), (1024, 2, 5), (1024, 3, 1)]


def _same(got, want, what):
    got = np.asarray(got)
    assert got.shape == want.shape, what
    assert np.array_equal(got, want), f"{what}: {int((got != want).sum())} of {want.size} differ"


def _counts(name, *handle):
    from strata_fdtd_amd import _native
    p, s = C.c_int64(), C.c_int64()
    _native.call(name, *handle, C.byref(p), C.byref(s))
    return p.value, s.value


def _tiled(s, tile, nts):
    from strata_fdtd_amd import _native
    _native.call("fdtd_ctx_set_multi_step", s._ctx, 3)
    _native.call("fdtd_ctx_set_pass_tiling", s._ctx, *tile, nts)
    return s


@pytest.mark.parametrize("nonuniform", [False, True])
@pytest.mark.parametrize("tile", TILES)
def test_pass_kernels_with_sources_of_every_kind(oracle_lib, tile, nonuniform):
    print(f"[variants] sources {tile} nonuniform={nonuniform}", flush=True)
    sc = seeded_scenario(31, shape=SHAPE, pml=4, nonuniform=nonuniform)
    for ax in (0, 1, 2):
        sc.sources.append(("plane", ax, 9 + ax, 7000.0 + 500 * ax))
    sc.probes += [(0, 0, 0), (21, 89, 69), (9, 44, 33)]
    n = 14
    st_o, tr_o = cpu.run(oracle_problem(sc, n), n)
    for nts in (0, 1):
        s = _tiled(make_solver(sc), tile, nts)
        s.step_n(n)
        assert _counts("fdtd_ctx_step_counts", s._ctx) == (4, 2)
        tr = s.get_probe_data()
        for q in range(len(sc.probes)):
            _same(tr[f"probe{q}"], tr_o[:, q], f"probe{q}")
        for k in FIELDS:
            _same(getattr(s, k), st_o[k], k)


@pytest.mark.parametrize("nonuniform", [False, True])
@pytest.mark.parametrize("tile", TILES)
def test_pass_kernels_with_poles_stations_and_initial_values(tile, nonuniform):
    print(f"[variants] poles {tile} nonuniform={nonuniform}", flush=True)
    sc = seeded_scenario(32, shape=SHAPE, pml=4, nonuniform=nonuniform)
    sc.material = np.zeros(SHAPE, np.uint8)
    sc.material[8:13, 40:52, 28:39] = 1
    sc.material[~sc.air] = 0
    sc.materials = {1: [dict(kind="debye", target="density", tau=2e-5, dchi=0.5),
                        dict(kind="lorentz", target="modulus", w0=2 * np.pi * 3000, gamma=500.0, dchi=0.4)]}
    rng = np.random.default_rng(5)
    sc.probes = [tuple(int(rng.integers(0, v)) for v in SHAPE) for _ in range(70)]
    values = {k: rng.standard_normal(SHAPE).astype(np.float32) for k in FIELDS}
    n = 14

    def solve(tile, nts):
        s = make_solver(sc, tiling=None if tile else (2, 2))
        if tile:
            _tiled(s, tile, nts)
        for q, ijk in enumerate(((10, 45, 33), (3, 10, 60))):
            s.add_microphone(tuple((v + 0.3) * s.dx for v in ijk), name=f"m{q}")
        for k in FIELDS:
            setattr(s, k, values[k])
        s.step_n(n)
        assert _counts("fdtd_ctx_step_counts", s._ctx) == ((4, 2) if tile else (0, n))
        return s

    one = solve(None, 0)
    tr_o = one.get_probe_data()
    for nts in (0, 1):
        s = solve(tile, nts)
        tr = s.get_probe_data()
        for k, v in tr_o.items():
            _same(tr[k], v, k)
        for m in ("m0", "m1"):
            _same(s.microphones[m].get_waveform(), np.asarray(one.microphones[m].get_waveform()), m)
        for k in FIELDS:
            _same(getattr(s, k), np.asarray(getattr(one, k)), k)


def test_windows_that_do_not_exist_are_refused():
    from strata_fdtd_amd import FDTDSolver, _native
    s = FDTDSolver(shape=SHAPE, resolution=1e-3)
    for bad in ((300, 1, 4), (256, 0, 4), (256, 1, 0), (256, 1, 23), (256, 19, 4), (256, 4, 4), (64, 1, 1)):
        with pytest.raises(_native.NativeError):
            _native.call("fdtd_ctx_set_pass_tiling", s._ctx, *bad, 0)
    s.step_n(4)


@pytest.mark.parametrize("count,passes", [(64 + 1024, True), (64 + 1025, False)])
def test_stations_past_their_scratch(count, passes):
    """1024 probes past the first 64 are recorded by stations of a pass; one more,
    and the solve steps one by one."""
    sc = seeded_scenario(14, shape=(30, 34, 48), pml=4, geometry=False)
    rng = np.random.default_rng(3)
    cells = rng.permutation(30 * 34 * 48)[:count]
    sc.probes = [tuple(int(v) for v in np.unravel_index(c, sc.shape)) for c in cells]
    s = make_solver(sc)
    s.step_n(7)
    assert _counts("fdtd_ctx_step_counts", s._ctx) == ((2, 1) if passes else (0, 7))
    one = make_solver(sc, tiling=(2, 2))
    one.step_n(7)
    want = one.get_probe_data()
    for k, v in s.get_probe_data().items():
        _same(v, want[k], k)


def test_poles_without_patch_scratch_step_one_by_one(oracle_lib):
    """Materials set while passes are off have no scratch: passes allowed later leave
    such a solve to single steps."""
    from strata_fdtd_amd import _native
    sc = seeded_scenario(3, shape=(26, 30, 40), pml=3, ade=True)
    n = 9
    st_o, tr_o = cpu.run(oracle_problem(sc, n), n)
    s = make_solver(sc)
    _native.call("fdtd_ctx_set_multi_step", s._ctx, 0)
    s._prepare(n)
    _native.call("fdtd_ctx_set_multi_step", s._ctx, 3)
    s.step_n(n)
    assert _counts("fdtd_ctx_step_counts", s._ctx) == (0, n)
    for k in FIELDS:
        _same(getattr(s, k), st_o[k], k)


@pytest.mark.parametrize("history", ["all", "checkpoint"])
@pytest.mark.parametrize("lo,hi", [((1, 1, 1), (7, 19, 21)), ((100, 90, 150), (131, 121, 199))])
def test_design_passes_beyond_the_cache(lo, hi, history):
    """204 x 200 x 201 cells (8.2 million): the instances with non-temporal stores."""
    import torch
    from strata_fdtd_amd import GaussianPulse, adjoint
    shape, steps = (204, 200, 201), 8
    src = tuple((a + b) // 2 for a, b in zip(lo, hi))
    probes = [src, tuple(v - 1 for v in lo), tuple(v - 1 for v in hi)]
    rng = np.random.default_rng(2)
    air = np.ones(shape, bool)
    air[tuple(rng.integers(0, n, 500) for n in shape)] = False
    for p in probes:
        air[p] = True
    pb = adjoint.DesignProblem(shape=shape, pml_depth=3, source=GaussianPulse(position=src, frequency=3e4),
                               probes=probes, steps=steps, box_lo=lo, box_hi=hi, checkpoint=5, geometry=air)
    rho, K = (torch.tensor(v * (1 + 0.05 * rng.standard_normal(pb.box_shape)), dtype=torch.float32, device="cuda")
              for v in (pb.rho, pb.K0))
    g = torch.tensor(rng.standard_normal((steps, len(probes))), dtype=torch.float32, device="cuda")
    out = {}
    for impl in ("cell", "fast"):
        tr, saved = adjoint.forward_traces(pb, rho, K, keep_checkpoints=True, impl=impl, history=history)
        out[impl] = (tr, *adjoint.adjoint_gradients(saved, g))
    # the last call: all steps, or the first segment of five
    assert _counts("fdtd_design_step_counts") == ((2, 2) if history == "all" else (1, 2))
    for name, x, y in zip(("traces", "rho", "K"), out["cell"], out["fast"]):
        assert torch.equal(x, y), name
    assert out["fast"][1].abs().max() > 0

"""Which steps go to the device in passes of three and which one by one: both give
the same bits, so the comparisons with the oracle cannot tell. Counts of passes and
single steps for the solves, batches and design calls that take passes and for those
that must not."""

import ctypes as C

import numpy as np
import pytest

from helpers import make_solver, seeded_scenario

pytestmark = pytest.mark.gpu

STEPS = 3  # a pass
POLES = [dict(kind="debye", target="density", tau=2e-5, dchi=0.5),
         dict(kind="debye", target="modulus", tau=1e-5, dchi=0.3)]


def _counts(name, *handle):
    from strata_fdtd_amd import _native
    p, s = C.c_int64(), C.c_int64()
    _native.call(name, *handle, C.byref(p), C.byref(s))
    return p.value, s.value


def ctx_counts(s):
    return _counts("fdtd_ctx_step_counts", s._ctx)


def _every_pass(s):
    from strata_fdtd_amd import _native
    _native.call("fdtd_ctx_set_multi_step", s._ctx, 3)
    return s


@pytest.mark.parametrize("scene", ["plain", "nonuniform", "z plane", "poles", "microphone", "70 probes"])
def test_solves_that_take_passes(scene):
    sc = seeded_scenario(2, shape=(30, 34, 48), pml=3, nonuniform=scene == "nonuniform")
    if scene == "z plane":
        sc.sources.append(("plane", 2, 9, 7000.0))
    if scene == "poles":
        sc.material = np.zeros(sc.shape, np.uint8)
        sc.material[10:14, 10:14, 10:14] = 1
        sc.materials = {1: POLES}
    if scene == "70 probes":
        sc.probes = [(1 + q % 28, 2 + q % 30, q % 48) for q in range(70)]
    s = _every_pass(make_solver(sc))
    if scene == "microphone":
        s.add_microphone(tuple(9.3 * s.dx for _ in range(3)), name="m")
    assert ctx_counts(s) == (0, 0)
    s.step_n(31)
    assert ctx_counts(s) == (10, 1)
    s.step()
    s.step_n(2)
    assert ctx_counts(s) == (10, 4)
    s.step_n(24, graph_chunk=8)      # three replays of two passes and two steps
    assert ctx_counts(s) == (16, 10)
    s.step_n(24, graph_chunk=8)
    assert ctx_counts(s) == (22, 16)


def test_solves_that_step_one_by_one():
    """A given launch shape; a microphone across the edge of the poles' boxes; a
    membrane among the sources; boundary planes; a plain grid too small to gain."""
    import strata_fdtd_amd as sfa
    sc = seeded_scenario(2, shape=(36, 44, 60), pml=3)
    tiled = make_solver(sc, tiling=(2, 2))
    small = make_solver(sc)
    bounded = _every_pass(make_solver(sc))
    bounded.add_boundary(sfa.ABCFirstOrder())
    sc.material = np.zeros(sc.shape, np.uint8)
    sc.material[14:18, 18:22, 28:32] = 1
    sc.materials = {1: POLES}
    edge = _every_pass(make_solver(sc))
    edge.add_microphone(tuple((v + 0.3) * edge.dx for v in (20, 20, 30)), name="m")
    for s in (tiled, small, bounded, edge):
        s.step_n(9)
        assert ctx_counts(s) == (0, 9)
    clear = _every_pass(make_solver(sc))
    clear.add_microphone(tuple((v + 0.3) * clear.dx for v in (25, 20, 30)), name="m")
    clear.step_n(9)
    assert ctx_counts(clear) == (3, 0)


def test_default_solves_take_passes_from_the_stated_sizes_on():
    from strata_fdtd_amd import FDTDSolver
    for shape, passes in (((100, 100, 100), True), ((45, 80, 99), False)):
        s = FDTDSolver(shape=shape, resolution=1e-3)
        s.step_n(7)
        assert ctx_counts(s) == ((2, 1) if passes else (0, 7)), shape


@pytest.mark.parametrize("use_graph", [False, True])
def test_batches_take_passes_and_equal_one_step_kernels(use_graph):
    """Served solves of 160^3, together beyond the cache, with a launch shape given
    to the lone solves they are compared with, so that those go step by step."""
    from strata_fdtd_amd.serving import SweepServer, build_solver, sweep_requests
    reqs = sweep_requests(n=3, rate=1e6, seed=3, steps=(50, 80), dims=(160,))
    srv = SweepServer(chunk=16, max_cells=None, policy="fifo", use_graph=use_graph)
    stats = srv.serve(reqs, realtime=False)
    chunks = stats.chunks
    assert _counts("fdtd_batch_step_counts", srv._batch) == (chunks * 5, chunks * (STEPS - 1))
    srv.close()
    for res in stats.results:
        r = next(x for x in reqs if x.rid == res.rid)
        s = build_solver(r, tiling=(4, 2))
        s.step_n(r.steps)
        assert ctx_counts(s) == (0, r.steps)
        for name, tr in s.get_probe_data().items():
            assert np.array_equal(res.traces[name], tr)


@pytest.mark.parametrize("history,steps", [("all", 31), ("checkpoint", 20)])
def test_design_calls_take_passes(history, steps):
    import torch
    from strata_fdtd_amd import GaussianPulse
    from strata_fdtd_amd.adjoint import DesignProblem, adjoint_gradients, forward_traces
    pb = DesignProblem(shape=(24, 26, 30), pml_depth=2, source=GaussianPulse(position=(12, 12, 12), frequency=3e4),
                       probes=[(13, 12, 12)], steps=steps, box_lo=(6, 6, 6), box_hi=(18, 18, 18), checkpoint=20)
    rho = torch.full(pb.box_shape, pb.rho * 1.01, device="cuda")
    tr, saved = forward_traces(pb, rho, None, keep_checkpoints=True, history=history)
    assert _counts("fdtd_design_step_counts") == (steps // STEPS, steps % STEPS)
    adjoint_gradients(saved, torch.ones_like(tr))
    assert _counts("fdtd_design_step_counts") == (steps // STEPS, steps % STEPS)


@pytest.mark.parametrize("what", ["microphone", "70 probes", "poles"])
def test_another_grid_ends_passes_until_their_tables_are_set_again(what):
    """fdtd_ctx_set_grid with other sides: the cells that passes keep of the
    microphones, probes and materials are of the old grid."""
    import torch
    from strata_fdtd_amd import _native
    sc = seeded_scenario(2, shape=(32, 40, 48), pml=0, geometry=False)
    if what == "70 probes":
        sc.probes = [(1 + q % 28, 2 + q % 28, q % 30) for q in range(70)]
    if what == "poles":
        sc.material = np.zeros(sc.shape, np.uint8)
        sc.material[4:10, 4:10, 4:10] = 1
        sc.materials = {1: POLES}
    s = _every_pass(make_solver(sc))
    if what == "microphone":
        s.add_microphone(tuple(9.3 * s.dx for _ in range(3)), name="m")
    s._prepare(64)                    # the tables cover every step below
    ones = torch.ones(48, device="cuda")
    _native.call("fdtd_ctx_set_pml", s._ctx, *[_native.ptr(ones)] * 3)

    def grid(nx, ny, nz):
        s.synchronize()
        _native.call("fdtd_ctx_set_grid", s._ctx, nx, ny, nz, 0, s._coeff_v, s._coeff_p, *[None] * 6)

    def take(n):
        before = ctx_counts(s)
        _native.call("fdtd_step_n", s._ctx, n)
        s.synchronize()
        return tuple(b - a for a, b in zip(before, ctx_counts(s)))

    assert take(9) == (3, 0)
    grid(32, 40, 48)                  # the same sides
    assert take(9) == (3, 0)
    grid(40, 32, 48)                  # as many cells, other sides
    assert take(9) == (0, 9)
    grid(32, 40, 48)
    assert take(9) == (0, 9)
    s._dirty_sources = s._dirty_ade = True
    s._prepare(64)
    assert take(9) == (3, 0)


def _pole_solver(n, boxes):
    import strata_fdtd_amd as sfa
    s = sfa.FDTDSolver(shape=(n, n, n), resolution=1e-3)
    s.register_material(sfa.SimpleMaterial(name="m", _rho=1.2, _c=343.0, _poles=[
        sfa.Pole(sfa.PoleType.DEBYE, 0.3, "density", tau=2e-5)]), material_id=1)
    for lo, hi in boxes:
        s.set_material_box(1, *[(lo, hi)] * 3)
    return s


@pytest.mark.parametrize("n,boxes,passes", [
    (128, [(54, 74)], True),                    # one absorber
    (128, [(2, 22), (106, 126)], False),        # two at opposite corners: air between them
    (128, [(30, 50), (78, 98)], True),          # the two a third of the sides apart
    (128, [(0, 128)], True),                    # all of the grid has poles
    (192, [(0, 20), (172, 192)], False),
    (264, [(40, 60), (204, 224)], True),        # beyond the cache, rows of 32-byte blocks
    (40, [(0, 8), (32, 40)], True)])            # a step's launches outweigh its cells
def test_passes_with_poles_where_the_patch_pays(n, boxes, passes):
    """Routes that the stated timings give; every one is bit-exact either way
    (a few steps of each against the other route)."""
    s, one = _pole_solver(n, boxes), _pole_solver(n, boxes)
    rng = np.random.default_rng(n)
    p = rng.standard_normal((n, n, n)).astype(np.float32)
    s.p, one.p = p, p
    s.step_n(9)
    assert ctx_counts(s) == ((3, 0) if passes else (0, 9))
    for _ in range(9):
        one.step()
    for k in ("p", "vx", "vy", "vz"):
        assert np.array_equal(getattr(s, k), getattr(one, k)), k


def test_patch_scratch_goes_back_with_the_materials():
    """The patch's scratch (here two copies of the fields, 67 MB) is given back when
    the materials are removed, and when they come to lie so that passes do not pay."""
    import torch
    n = 128
    s = _pole_solver(n, [(0, n)])

    def free():
        s.step_n(3)
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0]

    with_patch = free()
    assert ctx_counts(s) == (1, 0)
    s._material_id[:] = 0                         # two cells: their box is still all of the grid
    s._material_id[0, 0, 0] = s._material_id[-1, -1, -1] = 1
    s._dirty_ade = True
    apart = free()
    assert ctx_counts(s) == (1, 3)
    assert apart - with_patch > 60e6
    s._material_id[:] = 1
    s._dirty_ade = True
    again = free()
    assert ctx_counts(s) == (2, 3) and apart - again > 60e6
    s._material_id[:] = 0
    s._dirty_ade = True
    assert free() - again > 60e6
    assert ctx_counts(s)[0] == 3


@pytest.mark.parametrize("density", [0, 1])
def test_patch_scratch_has_a_second_J_of_density_poles_alone(density):
    """Eight modulus poles all over 128^3: two copies of the fields (67 MB), and 8.4
    MB for each density pole, registered last."""
    import torch
    import strata_fdtd_amd as sfa
    n = 128
    poles = [sfa.Pole(sfa.PoleType.DEBYE, 0.02 * (q + 1), "modulus", tau=1e-5 * (q + 1)) for q in range(8)]
    poles += [sfa.Pole(sfa.PoleType.DEBYE, 0.3, "density", tau=2e-5)] * density
    solvers = []
    for _ in range(2):
        s = sfa.FDTDSolver(shape=(n, n, n), resolution=1e-3)
        s.register_material(sfa.SimpleMaterial(name="m", _rho=1.2, _c=343.0, _poles=poles), material_id=1)
        s.set_material_box(1, *[(0, n)] * 3)
        s.p = np.random.default_rng(3).standard_normal((n, n, n)).astype(np.float32)
        solvers.append(s)
    s, one = solvers
    one.set_tiling(2, 2)
    s.step_n(9)
    for _ in range(9):
        one.step()
    assert ctx_counts(s) == (3, 0)
    for k in ("p", "vx", "vy", "vz"):
        assert np.array_equal(getattr(s, k), getattr(one, k)), k
    torch.cuda.synchronize()
    with_patch = torch.cuda.mem_get_info()[0]
    s._material_id[:] = 0
    s._dirty_ade = True
    s.step_n(3)
    torch.cuda.synchronize()
    scratch = torch.cuda.mem_get_info()[0] - with_patch
    cells = 4 * n**3
    assert (8 + density) * cells <= scratch < (9.5 + density) * cells


def test_autotune_keeps_passes_where_they_are_faster():
    """The launch shape that it sets is of single steps; a solver that took passes
    still does where the fastest shape is slower (128^3: 16 us a step against 11),
    with materials or without; one made with a launch shape does not begin to."""
    from strata_fdtd_amd import FDTDSolver
    from strata_fdtd_amd.autotune import autotune
    shapes = [(2, 2, 1), (4, 4, 1)]
    plain, poles = FDTDSolver(shape=(128, 128, 128), resolution=1e-3), _pole_solver(128, [(54, 74)])
    given = FDTDSolver(shape=(128, 128, 128), resolution=1e-3, tiling=(2, 2))
    for s, passes in ((plain, True), (poles, True), (given, False)):
        best, table = autotune(s, candidates=shapes, store=False)
        assert s.tiling == best and best in shapes and len(table) == 2
        before = ctx_counts(s)
        s.step_n(9)
        assert tuple(b - a for a, b in zip(before, ctx_counts(s))) == ((3, 0) if passes else (0, 9))
    plain.set_tiling(2, 2)
    before = ctx_counts(plain)
    plain.step_n(9)
    assert ctx_counts(plain) == (before[0], before[1] + 9)


@pytest.mark.parametrize("n,count,chunk,passes", [(40, 1, 100, False), (32, 4, 100, True), (64, 1, 16, False),
                                                  (64, 1, 99, True), (96, 1, 3, True), (96, 1, 2, False)])
@pytest.mark.parametrize("use_graph", [0, 1])
def test_batches_take_passes_where_they_pay(n, count, chunk, passes, use_graph):
    """Small solves in short chunks step one by one; two chunks of either way equal
    the lone solves' one-step kernels; a captured chunk of passes stays when a solve
    leaves."""
    import torch
    from strata_fdtd_amd import FDTDSolver, GaussianPulse, _native

    def solve():
        s = FDTDSolver(shape=(n, n, n), resolution=1e-3, tiling=(2, 2))
        s.add_source(GaussianPulse(position=(n // 2,) * 3, frequency=5e3))
        s.add_probe("p", (n // 3,) * 3)
        s.p = np.random.default_rng(1).standard_normal((n, n, n)).astype(np.float32)
        s._prepare(3 * chunk)
        return s

    batch, one = [solve() for _ in range(count)], solve()
    h = _native._vp()
    _native.call("fdtd_batch_create", 0, torch.cuda.current_stream().cuda_stream, 2, C.byref(h))
    try:
        def serve(solves, chunks):
            ctxs = (_native._vp * count)(*[s._ctx for s in solves])
            limits = np.full(count, 3 * chunk, dtype=np.int64)
            _native.call("fdtd_batch_set", h.value, ctxs, limits.ctypes.data, len(solves))
            before = _counts("fdtd_batch_step_counts", h.value)
            for _ in range(chunks):
                _native.call("fdtd_batch_step_n", h.value, chunk, use_graph)
            torch.cuda.synchronize()
            return tuple(b - a for a, b in zip(before, _counts("fdtd_batch_step_counts", h.value)))

        in_passes, singly = (chunk // STEPS, STEPS - 1), (0, chunk)
        want = in_passes if passes else singly
        assert serve(batch, 2) == (2 * want[0], 2 * want[1])
        if count > 1:
            assert serve(batch[:1], 1) == (in_passes if use_graph else singly)
        else:
            serve(batch, 1)
    finally:
        _native.load().fdtd_batch_destroy(h.value)
    one.step_n(3 * chunk)
    first = batch[0]
    first._advance_host(3 * chunk)
    for k in ("p", "vx", "vy", "vz"):
        assert np.array_equal(getattr(first, k), getattr(one, k)), k
    assert np.array_equal(first.get_probe_data()["p"], one.get_probe_data()["p"])

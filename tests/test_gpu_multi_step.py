"""Multi-step passes (three steps per sweep over the fields) against the CPU
oracle, bit for bit: grids at the edges of the windows, every source kind the
passes take, step counts with each remainder, and graph replays. The step
kernels keep the oracle's operations and their order, so the tolerance is 0."""

import numpy as np
import pytest

import helpers
from helpers import oracle_problem, seeded_scenario
from oracle import cpu

pytestmark = pytest.mark.gpu

FIELDS = ("p", "vx", "vy", "vz")

# nz of every remainder by 4; one and several k segments; rows that fill their
# windows exactly and by one more; fewer planes than a pass has steps
SHAPES = [(26, 37, 70), (13, 41, 33), (9, 25, 130), (3, 20, 31), (12, 61, 1030), (31, 19, 12), (40, 26, 64)]


def make_solver(sc, tiling=None):
    """A solver that takes passes on these small grids too."""
    from strata_fdtd_amd import _native
    s = helpers.make_solver(sc, tiling=tiling)
    if tiling is None:
        _native.call("fdtd_ctx_set_multi_step", s._ctx, 3)
    return s


def _same(got, want, what):
    got = np.asarray(got)
    assert got.shape == want.shape, what
    assert np.array_equal(got, want), f"{what}: {int((got != want).sum())} of {want.size} differ"


def _compare(sc, s, n, st_o, tr_o):
    tr = s.get_probe_data()
    for q in range(len(sc.probes)):
        _same(tr[f"probe{q}"], tr_o[:, q], f"probe{q}")
    for k in FIELDS:
        _same(getattr(s, k), st_o[k], k)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("steps", [3, 31, 32])
def test_pass_bitexact(oracle_lib, shape, steps):
    print(f"[pass] {shape} {steps}", flush=True)
    big = min(shape) >= 12
    sc = seeded_scenario(5, shape=shape, pml=3 if big else 0, geometry=big)
    st_o, tr_o = cpu.run(oracle_problem(sc, steps), steps)
    s = make_solver(sc)
    s.step_n(steps)
    _compare(sc, s, steps, st_o, tr_o)


@pytest.mark.parametrize("nonuniform", [False, True])
@pytest.mark.parametrize("axes", [(0,), (1,), (2,), (2, 0, 1)])
def test_pass_plane_sources(oracle_lib, axes, nonuniform):
    """Plane sources of each axis, z planes (which single steps add from tables) among them."""
    print(f"[pass] planes {axes} nonuniform={nonuniform}", flush=True)
    sc = seeded_scenario(6, shape=(22, 38, 52), pml=4, nonuniform=nonuniform)
    for ax in axes:
        sc.sources.append(("plane", ax, 7 + ax, 7000.0 + 500 * ax))
    sc.sources.append(("point", sc.sources[0][1], 5000.0))
    sc.probes.append((11, 8, 9))
    n = 26
    st_o, tr_o = cpu.run(oracle_problem(sc, n), n)
    s = make_solver(sc)
    s.step_n(5)
    s.step()
    s.step_n(n - 6)
    _compare(sc, s, n, st_o, tr_o)


def test_pass_many_probes_of_one_window(oracle_lib):
    """64 probes, the most a pass records, close together and on every wall of the grid."""
    sc = seeded_scenario(7, shape=(24, 30, 44), pml=4)
    rng = np.random.default_rng(1)
    sc.probes = [tuple(int(v) for v in rng.integers((8, 8, 8), (14, 14, 14))) for _ in range(56)]
    sc.probes += [(i, j, k) for i in (0, 23) for j in (0, 29) for k in (0, 43)]
    n = 21
    st_o, tr_o = cpu.run(oracle_problem(sc, n), n)
    s = make_solver(sc)
    s.step_n(n)
    _compare(sc, s, n, st_o, tr_o)


def test_pass_graph_replays(oracle_lib):
    """Captured chunks (two passes and a single step each), replayed between eager steps."""
    sc = seeded_scenario(8, shape=(25, 33, 47), pml=4)
    n = 7 * 4 + 5 + 7 * 3
    st_o, tr_o = cpu.run(oracle_problem(sc, n), n)
    s = make_solver(sc)
    s.step_n(28, graph_chunk=7)
    s.step_n(5)
    s.synchronize()
    s.step_n(21, graph_chunk=7)
    _compare(sc, s, n, st_o, tr_o)


def test_pass_keeps_initial_values(oracle_lib):
    """Fields written by the caller, last faces (which keep their velocity) and
    solid cells among them, evolve as single steps take them."""
    rng = np.random.default_rng(4)
    sc = seeded_scenario(9, shape=(19, 23, 41), pml=3)
    one, three = make_solver(sc, tiling=(2, 2)), make_solver(sc)
    for k in FIELDS:
        v = rng.standard_normal(sc.shape).astype(np.float32)
        setattr(one, k, v)
        setattr(three, k, v)
    one.step_n(18)
    three.step_n(18)
    for k in FIELDS:
        _same(getattr(three, k), getattr(one, k), k)


POLES = {
    "debye": [dict(kind="debye", target="density", tau=2e-5, dchi=0.5),
              dict(kind="debye", target="modulus", tau=1e-5, dchi=0.3)],
    "lorentz": [dict(kind="lorentz", target="modulus", w0=2 * np.pi * 3000, gamma=500.0, dchi=0.4),
                dict(kind="lorentz", target="density", w0=2 * np.pi * 2000, gamma=300.0, dchi=0.2)],
}


@pytest.mark.parametrize("nonuniform", [False, True])
@pytest.mark.parametrize("where", ["inside", "corner", "everywhere"])
def test_pass_ade_patch(oracle_lib, where, nonuniform):
    """Materials with poles in a pass: a sphere of two materials away from the
    walls, or in a corner (its grown boxes are cut by the grid), or all of the
    grid, with the source and probes in, next to and away from it, over passes
    and single steps."""
    print(f"[pass] ade {where} nonuniform={nonuniform}", flush=True)
    shape = (36, 44, 60)
    sc = seeded_scenario(10, shape=shape, pml=4, nonuniform=nonuniform)
    c = np.array((0, 43, 57) if where == "corner" else (15, 20, 30))
    g = np.indices(shape)
    d2 = sum((g[x] - c[x]) ** 2 for x in range(3))
    r2 = 10**6 if where == "everywhere" else 20
    sc.material = np.where(d2 <= r2, np.where(g[2] > c[2], 2, 1), 0).astype(np.uint8)
    sc.material[~sc.air] = 0
    sc.materials = {1: POLES["debye"], 2: POLES["lorentz"] + POLES["debye"][:1]}
    near = [tuple(int(v) for v in np.clip(c + d, 0, np.array(shape) - 1))
            for d in ((0, 0, 0), (0, 0, 1), (6, 0, 0), (0, -7, 0), (3, -3, -2), (1, -1, 8))]
    sc.probes += near + [(20, 5, 9)]
    sc.sources.append(("point", near[3], 7000.0))
    sc.sources.append(("point", near[1], 9000.0))
    n = 29
    st_o, tr_o = cpu.run(oracle_problem(sc, n), n)
    s = make_solver(sc)
    s.step_n(7)
    s.step()
    s.step_n(12, graph_chunk=6)
    s.step_n(n - 20)
    _compare(sc, s, n, st_o, tr_o)


@pytest.mark.parametrize("nonuniform", [False, True])
@pytest.mark.parametrize("poles", [("debye",), ("lorentz",), ("debye", "lorentz", "debye")])
def test_pass_ade_pole_tables(oracle_lib, poles, nonuniform):
    """Tables of up to four poles and of more, density Lorentz poles among them or
    not: a thin layer along the grid's last rows, whose last cell is the grid's,
    and single cells beside it, so that lanes hold cells with poles and without."""
    print(f"[pass] poles {poles} nonuniform={nonuniform}", flush=True)
    shape = (30, 27, 46)
    sc = seeded_scenario(13, shape=shape, pml=3, nonuniform=nonuniform, geometry=False)
    sc.material = np.zeros(shape, np.uint8)
    sc.material[22:, 24:, 37:] = 1
    sc.material[24, 21:23, 30:34] = 1
    sc.material[26, 22, 31] = 2
    sc.materials = {1: sum((POLES[q] for q in poles), [])}
    if len(poles) > 1:
        sc.materials[2] = POLES["debye"][:1]
    else:
        sc.material[sc.material == 2] = 0
    sc.probes += [(29, 26, 45), (24, 22, 32), (25, 23, 36), (23, 20, 30)]
    sc.sources.append(("point", (24, 22, 35), 9000.0))
    sc.sources.append(("plane", 2, 33, 7000.0))
    n = 17
    st_o, tr_o = cpu.run(oracle_problem(sc, n), n)
    s = make_solver(sc)
    s.step_n(n)
    _compare(sc, s, n, st_o, tr_o)


@pytest.mark.parametrize("nonuniform", [False, True])
@pytest.mark.parametrize("poles", [None, "clear", "edge"])
def test_pass_microphones(poles, nonuniform):
    """Microphones recorded from passes against single steps: at the walls, next to
    a source, and, with poles, in their material, in the boxes of the patch and
    clear of them; one more at the edge of the boxes makes the solve step singly."""
    print(f"[pass] microphones poles={poles} nonuniform={nonuniform}", flush=True)
    shape, c = (36, 44, 60), (15, 20, 30)
    sc = seeded_scenario(12, shape=shape, pml=4, nonuniform=nonuniform)
    if poles:
        g = np.indices(shape)
        d2 = sum((g[x] - c[x]) ** 2 for x in range(3))
        sc.material = np.where(d2 <= 20, 1, 0).astype(np.uint8)
        sc.material[~sc.air] = 0
        sc.materials = {1: POLES["debye"]}
    # cells (with an offset inside them); box: [11, 20) x [16, 25) x [26, 35)
    cells = [(0, 0, 0), (34, 42, 58), (5, 42, 30), (30, 9, 50), (15, 20, 30), (10, 20, 30), (15, 14, 36),
             (26, 20, 30), (15, 28, 30)]
    if poles == "edge":
        cells.append((22, 20, 30))
    solvers = []
    for _ in range(2):
        s = make_solver(sc)
        for q, ijk in enumerate(cells):
            pos = tuple((v + 0.3) * s.dx for v in ijk)
            kw = dict(pattern="cardioid", direction=(1, 2, 3)) if q % 2 else {}
            s.add_microphone(pos, name=f"m{q}", **kw)
        solvers.append(s)
    s, one = solvers
    s.step_n(7)
    s.step_n(12, graph_chunk=6)
    s.step_n(10)
    for _ in range(29):
        one.step()
    for q in range(len(cells)):
        got, want = (np.asarray(v.microphones[f"m{q}"].get_waveform()) for v in solvers)
        _same(got, want, f"microphone {cells[q]}")
    for k in FIELDS:
        _same(getattr(s, k), np.asarray(getattr(one, k)), k)


@pytest.mark.parametrize("poles", [False, True])
@pytest.mark.parametrize("count", [65, 200])
def test_pass_probes_past_the_sweeps(oracle_lib, count, poles):
    """More probes than a pass records itself: all over the grid, its corners and
    the boxes around a material with poles among them."""
    print(f"[pass] {count} probes poles={poles}", flush=True)
    shape = (36, 44, 60)
    sc = seeded_scenario(14, shape=shape, pml=4)
    rng = np.random.default_rng(14)
    if poles:
        sc.material = np.zeros(shape, np.uint8)
        sc.material[12:18, 18:24, 30:37] = 1
        sc.material[~sc.air] = 0
        sc.materials = {1: POLES["debye"]}
    near = [(i, j, k) for i in (8, 11, 20, 21) for j in (15, 20, 27) for k in (33, 40)]
    while len(sc.probes) < count - 26:
        sc.probes.append(tuple(int(rng.integers(0, n)) for n in shape))
    sc.probes += near + [(0, 0, 0), (35, 43, 59)]
    sc.probes = sc.probes[-count:]
    n = 20
    st_o, tr_o = cpu.run(oracle_problem(sc, n), n)
    s = make_solver(sc)
    s.step_n(n)
    _compare(sc, s, n, st_o, tr_o)

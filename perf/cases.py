"""The work a user of this package has it do, as measurable cases.

Every case goes through the public entry points. Sizes and scenes come from the package's own workloads
(``workloads.py``, ``serving.sweep_requests``, ``adjoint.design_problem_192``), the scenes of its tests (the recorded
organ pipes, the 40^3 sample run) and odd sizes between them.

kinds
  step       one whole solve driven by ``step()`` from a Python loop, as scripts with their own loop do
  solve      one whole solve: ``reset()`` and ``run(duration)``; probe traces and final fields come back
  advance    a solve in progress advanced by ``run(duration)``: the state goes on from pass to pass
  record     one whole solve with pressure snapshots and energy samples
  serve      a batch of enclosure requests through the continuous-batching server
  gradient   probe traces of a per-voxel design forward, and the gradients of their loss backward
"""

import math

import numpy as np
import torch

from strata_fdtd_amd import (PML, Box, Cylinder, Difference, FDTDSolver, GaussianPulse, MaterializedGeometry, Pole,
                             PoleType, SimpleMaterial, Sphere, UniformGrid, Union)
from strata_fdtd_amd import adjoint, serving, workloads

C, RHO, COURANT, DX = 343.0, 1.204, 0.95, 1e-3


def listed():
    return [
        # the 40^3 rigid sample run, stepped by a script's own loop: latency and launches
        dict(name="step_40", kind="step", scene="air", nx=40, ny=40, nz=40, pml=0, steps=63, probes=2, mics=0),
        # the 100^3 air box: the ordinary small solve
        dict(name="solve_100", kind="solve", scene="air", nx=100, ny=100, nz=100, pml=10, steps=250, probes=1, mics=0),
        # an organ pipe (boolean mask, ragged sides), an odd number of steps
        dict(name="solve_pipe", kind="solve", scene="pipe", nx=180, ny=76, nz=76, pml=10, steps=251, probes=7, mics=0),
        # odd sides, absorber with Debye and Lorentz poles, microphones beside the probes
        dict(name="solve_ragged_ade", kind="solve", scene="lined", nx=131, ny=157, nz=203, pml=9, steps=60, probes=3, mics=2),
        # the adjoint workload's grid size as a plain solve: the largest cube that stays in the Infinity Cache
        dict(name="solve_192", kind="solve", scene="room", nx=192, ny=192, nz=192, pml=12, steps=100, probes=4, mics=0),
        # just beyond the cache, odd sides
        dict(name="advance_ragged", kind="advance", scene="room", nx=261, ny=243, nz=307, pml=11, steps=41, probes=5, mics=0),
        # the 512^3 enclosure with its port and absorber sphere (the benchmark scene)
        dict(name="advance_enclosure_512", kind="advance", scene="enclosure", nx=512, ny=512, nz=512, pml=16, steps=40, probes=8, mics=0),
        # the nonuniform resonator plate with its plane source
        dict(name="advance_resonators", kind="advance", scene="resonators", nx=320, ny=320, nz=480, pml=16, steps=50, probes=16, mics=0),
        # a run whose snapshots and energies are wanted
        dict(name="record_128", kind="record", scene="room", nx=128, ny=96, nz=160, pml=10, steps=80, probes=4, mics=0, every=16),
        # a design sweep of enclosures through the server, all waiting at the start
        dict(name="serve_10", kind="serve", requests=10, low=64, high=128, steps=300),
        # the adjoint workload (192^3, 128^3 design box), shortened: history in memory
        dict(name="gradient_192", kind="gradient", nx=192, ny=192, nz=192, pml=12, box=128, steps=60, probes=4, history="all", checkpoint=20),
        # a smaller ragged design with checkpoints and recomputation
        dict(name="gradient_ragged", kind="gradient", nx=90, ny=75, nz=118, pml=8, box=41, steps=70, probes=3, history="checkpoint", checkpoint=20),
    ]


def _between(rng, lo, hi):
    """A whole number, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "solve", "solve", "solve", "advance", "advance", "record", "serve", "gradient"])
    if kind == "serve":
        return dict(kind=kind, requests=rng.randint(4, 10), low=64, high=rng.choice([96, 112, 128]), steps=_between(rng, 100, 300))
    if kind == "gradient":
        n = [_between(rng, 48, 160) for _ in range(3)]
        return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], pml=rng.randint(5, 10), box=rng.randint(12, min(n) // 2), steps=rng.randint(20, 60),
                    probes=rng.randint(1, 4), history=rng.choice(["all", "checkpoint"]), checkpoint=rng.randint(8, 25))
    lo, hi = {"step": (16, 96), "solve": (32, 192), "advance": (120, 420), "record": (32, 128)}[kind]
    n = [_between(rng, lo, hi) for _ in range(3)]
    cells = n[0] * n[1] * n[2]
    c = dict(kind=kind, scene=rng.choice(["air", "pipe", "room", "lined", "enclosure", "stretched"]), nx=n[0], ny=n[1], nz=n[2],
             pml=rng.choice([0, rng.randint(3, max(3, min(16, min(n) // 4)))]), steps=0, probes=rng.choice([1, 2, 4, 9, 70]), mics=rng.choice([0, 0, 0, 1, 3]))
    most = max(20, min(300, int(2e9 / cells)))
    c["steps"] = rng.randint(max(15, most // 3), most)
    if kind == "step":
        c["steps"] = min(c["steps"], 60)
    if kind == "record":
        c["every"] = rng.randint(8, 20)
        c["steps"] = min(c["steps"], 100)
    return c


# ---- scenes ---------------------------------------------------------------------------------------------------------------
def _shape(case):
    return case["nx"], case["ny"], case["nz"]


def _room_mask(shape):
    """A closed box room with a doorway and a pillar, as a boolean mask (True: air)."""
    nx, ny, nz = shape
    air = np.ones(shape, dtype=bool)
    a, b = [max(2, n // 5) for n in shape], [n - max(2, n // 5) for n in shape]
    w = max(1, min(shape) // 40)
    air[a[0]:b[0], a[1]:b[1], a[2]:b[2]] = False
    air[a[0] + w:b[0] - w, a[1] + w:b[1] - w, a[2] + w:b[2] - w] = True
    air[a[0]:a[0] + w, ny // 2 - 2:ny // 2 + 2, nz // 2 - 3:nz // 2 + 3] = True
    air[nx // 2:nx // 2 + w + 1, ny // 3:ny // 3 + w + 1, a[2]:b[2]] = False
    return air


def _pipe_mask(shape):
    """A pipe along x, open at one end, closed at the other."""
    nx, ny, nz = shape
    y, z = np.arange(ny)[:, None] - (ny - 1) / 2, np.arange(nz)[None, :] - (nz - 1) / 2
    r2, ro = y * y + z * z, 0.28 * min(ny, nz)
    wall = (r2 <= ro * ro) & (r2 > (0.75 * ro) ** 2)
    air = np.ones(shape, dtype=bool)
    i0, i1 = nx // 6, nx - nx // 6
    air[i0:i1, wall] = False
    air[i0:i0 + 2, r2 <= ro * ro] = False
    return air


def _poles(rng):
    return [Pole(PoleType.DEBYE, float(rng.uniform(0.1, 0.5)), "density", tau=float(rng.uniform(1e-5, 1e-4))),
            Pole(PoleType.DEBYE, float(rng.uniform(0.1, 0.5)), "modulus", tau=float(rng.uniform(1e-5, 1e-4))),
            Pole(PoleType.LORENTZ, float(rng.uniform(0.05, 0.2)), "modulus", omega_0=2e4, gamma=2e3)]


def _spots(rng, shape, air, count, near=None, reach=0):
    """Seeded air cells away from the grid's faces, within `reach` cells of `near` on each axis if that is given."""
    lo, hi = [max(1, n // 8) for n in shape], [n - max(1, n // 8) for n in shape]
    if near is not None:
        lo, hi = [max(l, c - reach) for l, c in zip(lo, near)], [min(h, c + reach + 1) for h, c in zip(hi, near)]
    got = []
    while len(got) < count:
        c = tuple(int(rng.integers(l, h)) for l, h in zip(lo, hi))
        if air is None or air[c]:
            got.append(c)
    return got


def _reach(steps):
    """Cells on each axis that a pulse's front passes well within so many steps (0.55 cells a step)."""
    return max(2, int(0.15 * steps))


def _solver(case, seed):
    """A configured solve of the case's scene, its sources, probes and material drawn from the seed; (solver, air mask or None, source, probes)."""
    rng = np.random.default_rng(seed)
    shape, scene = _shape(case), case["scene"]
    if scene == "resonators" or scene == "stretched":
        core = 200 if scene == "resonators" else max(2, min(shape) // 2)
        if scene == "resonators":
            grid, geo, _, index = workloads.resonators_nu_scene(shape)
        else:
            from strata_fdtd_amd import NonuniformGrid, explicit_core_stretch_coords
            grid, geo, index = NonuniformGrid(*[explicit_core_stretch_coords(n, core - (n - core) % 2, DX, 1.03) for n in shape]), None, shape[2] // 3
        s = FDTDSolver(grid=grid, c=C, rho=RHO, backend="mi355x")
        if geo is not None:
            s.set_geometry(geo)
        if case["pml"]:
            s.add_boundary(PML(depth=case["pml"]))
        s.add_source(GaussianPulse(position={"axis": 2, "index": index}, frequency=float(rng.uniform(1.5e3, 3e3)), source_type="plane"))
        for q, c in enumerate(_spots(rng, shape, None, case["probes"])):
            s.add_probe("probe%d" % q, c)
        for q in range(case["mics"]):
            s.add_microphone(tuple(float(e * rng.uniform(0.3, 0.7)) for e in grid.physical_extent()), name="mic%d" % q)
        return s, None, None, None
    s = FDTDSolver(grid=UniformGrid(shape, DX), c=C, rho=RHO, courant=COURANT, backend="mi355x")
    air = _room_mask(shape) if scene == "room" else _pipe_mask(shape) if scene == "pipe" else None
    if air is not None:
        s.set_geometry(air)
    elif scene == "enclosure":
        n = min(shape)
        geo, _, _ = workloads.enclosure_512_scene(n)
        s.set_geometry(geo)
    elif scene == "lined":
        ext = np.array(shape) * DX
        outer, inner = Box(center=tuple(ext / 2), size=tuple(0.7 * ext)), Box(center=tuple(ext / 2), size=tuple(0.6 * ext))
        port = Cylinder(p1=(0.1 * ext[0], ext[1] / 2, ext[2] / 2), p2=(0.3 * ext[0], ext[1] / 2, ext[2] / 2), radius=0.06 * min(ext))
        geo = MaterializedGeometry(Union(Difference(Box(center=tuple(ext / 2), size=tuple(4 * ext)), Difference(outer, inner)), port))
        m = SimpleMaterial(name="lining", _rho=RHO, _c=C, _poles=_poles(rng))
        geo.set_material(Difference(inner, Box(center=tuple(ext / 2), size=tuple(0.54 * ext))), m)
        geo.set_material(Sphere(center=tuple(ext / 2), radius=0.1 * float(min(ext))), m)
        s.set_geometry(geo)
    if case["pml"]:
        s.add_boundary(PML(depth=case["pml"]))
    src = _spots(rng, shape, s.geometry, 1)[0]
    pulse = GaussianPulse(position=src, frequency=float(rng.uniform(1e4, 4e4)), amplitude=float(rng.uniform(0.5, 2.0)))
    probes = _spots(rng, shape, s.geometry, case["probes"], src, _reach(case["steps"]))
    s.add_source(pulse)
    for q, c in enumerate(probes):
        s.add_probe("probe%d" % q, c)
    for q in range(case["mics"]):
        s.add_microphone(tuple(float(n * DX * rng.uniform(0.3, 0.7)) for n in shape), name="mic%d" % q, pattern=("omni", "cardioid", "figure8")[q % 3], direction=(1.0, 0.0, 0.0))
    return s, air, pulse, probes


def _modes(case, seed):
    """The pressure a solve in progress starts from: a few seeded standing modes (float32, on the GPU)."""
    g = np.random.default_rng(seed + 7)
    p = torch.zeros(_shape(case), device="cuda")
    for _ in range(4):
        f = [torch.cos(torch.arange(n, device="cuda") * float(g.uniform(0.02, 0.6)) + float(g.uniform(0, 6.28))) for n in _shape(case)]
        p += float(g.uniform(0.2, 1.0)) * f[0][:, None, None] * f[1][None, :, None] * f[2][None, None, :]
    return p


def _requests(case, seed):
    reqs = serving.sweep_requests(n=case["requests"], rate=1e6, seed=4321, steps=(case["steps"] // 3, case["steps"]), dims=tuple(range(case["low"], case["high"] + 1, 16)))
    rng = np.random.default_rng(seed)
    for r in reqs:  # the same shapes and lengths each time, other pulses
        r.source.frequency = float(rng.uniform(2e3, 2e4))
        r.source.bandwidth = 2.0 * r.source.frequency
        r.source.amplitude = float(rng.uniform(0.5, 2.0))
    return reqs


def _design(case, seed):
    rng = np.random.default_rng(seed)
    shape, b = _shape(case), case["box"]
    lo = tuple((n - b) // 2 for n in shape)
    hi = tuple(v + b for v in lo)
    src = GaussianPulse(position=tuple(n // 2 - (b // 4 if a == 0 else 0) for a, n in enumerate(shape)), frequency=float(rng.uniform(1e4, 3e4)))
    probes = _spots(rng, shape, None, case["probes"], src.position, _reach(case["steps"]))
    pb = adjoint.DesignProblem(shape=shape, pml_depth=case["pml"], source=src, probes=probes, steps=case["steps"], box_lo=lo, box_hi=hi, checkpoint=case["checkpoint"])
    rho = RHO * (1 + 0.05 * rng.standard_normal((b, b, b), dtype=np.float32))
    K = RHO * C * C * (1 + 0.05 * rng.standard_normal((b, b, b), dtype=np.float32))
    target = 1e-3 * rng.standard_normal((case["steps"], case["probes"])).astype(np.float32)
    return pb, rho.astype(np.float32), K.astype(np.float32), target


# ---- what a program holds, and one pass -----------------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "serve":
        return dict(case=case, server=serving.SweepServer(), requests=_requests(case, seed))
    if kind == "gradient":
        pb, rho, K, target = _design(case, seed)
        dev = torch.device("cuda")
        return dict(case=case, pb=pb, rho=torch.from_numpy(rho).to(dev).requires_grad_(True), K=torch.from_numpy(K).to(dev).requires_grad_(True), target=torch.from_numpy(target).to(dev))
    s = _solver(case, seed)[0]
    if kind == "advance":
        s.p = _modes(case, seed).cpu().numpy()
    if kind == "record":
        s.enable_snapshots(case["every"])
    return dict(case=case, solver=s, duration=(case["steps"] - 0.5) * s.dt)


def _results(s, fields=True):
    out = {"probes": s.get_probe_data()}
    out["probes"] = [out["probes"][n] for n in sorted(out["probes"])][:16]  # a separate array each
    if s.microphones:
        out["mics"] = [m.get_waveform() for m in s.microphones.values()]
    if fields:
        out["fields"] = s.device_fields()
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "serve":
        done = state["server"].serve(state["requests"], realtime=False)
        return {str(r.rid): np.stack(list(r.traces.values())) for r in done.results}
    if kind == "gradient":
        rho, K = state["rho"], state["K"]
        rho.grad = K.grad = None
        tr = adjoint.probe_traces(rho, K, state["pb"], history=case["history"])
        ((tr - state["target"]) ** 2).sum().backward()
        return {"traces": tr, "rho": rho.grad, "K": K.grad}
    s = state["solver"]
    if kind == "step":
        s.reset()
        for _ in range(case["steps"]):
            s.step()
        return _results(s)
    if kind == "solve":
        s.reset()
        s.run(state["duration"])
        return _results(s)
    if kind == "advance":
        s.run(state["duration"])
        return _results(s)
    s.reset()
    s.run(state["duration"], track_energy=True, energy_sample_interval=case["every"])
    out = _results(s)
    out["snapshots"] = [p for _, p in s.get_snapshots()]
    out["energy"] = np.array([e for _, _, e in s.get_energy_history()])
    return out


# ---- what a pass cannot do without ------------------------------------------------------------------------------------------
# One state (four float32 fields) and the cell flags read, one state written; the steps between stay on the chip as far as this count
# goes. Per cell and step 22 operations: 3 faces x (subtract, multiply, add), 5 for the divergence, 2 for the pressure, 6 of damping.
FLOPS = 22


def work(case):
    kind = case["kind"]
    if kind == "serve":
        reqs = _requests(case, 0)
        return {"bytes": float(sum(17 * r.cells + 4 * r.steps * len(r.probes) for r in reqs)), "flops": float(sum(FLOPS * r.cells * r.steps for r in reqs))}
    cells = case["nx"] * case["ny"] * case["nz"]
    if kind == "gradient":  # forward and adjoint steps, the gradient's terms, the parameters in and the gradients out
        box = case["box"] ** 3
        return {"bytes": float(16 * box + cells), "flops": float(case["steps"] * (2 * FLOPS * cells + 40 * box))}
    start = 16 if kind == "advance" else 0
    b = (start + 17) * cells + 4 * case["steps"] * case["probes"]
    if kind == "record":
        b += 4 * cells * len(range(0, case["steps"], case["every"]))
    return {"bytes": float(b), "flops": float(FLOPS * cells * case["steps"])}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------------------
def _decays(shape, pml, dt):
    """exp(-sigma dt) of a cubic profile of reflection 1e-6 in both slabs of each axis."""
    out = []
    for n in shape:
        sig = np.zeros(n)
        if pml:
            top = -4 * C * math.log(1e-6) / (2 * pml * DX)
            for q in range(pml):
                sig[q] = top * ((pml - q) / pml) ** 3
                sig[n - pml + q] = top * ((q + 1) / pml) ** 3
        out.append(torch.from_numpy(np.exp(-sig * dt)).cuda())
    return out


def _pulse(pulse, dt, steps):
    t = np.cumsum(np.concatenate([[0.0], np.full(steps - 1, dt)]))
    sg = 1.0 / (math.pi * pulse.bandwidth)
    return pulse.amplitude * np.exp(-((t - 4 * sg) ** 2) / (2 * sg * sg)) * np.sin(2 * math.pi * pulse.frequency * (t - 4 * sg))


def _diff(v, axis):
    """v(face above) - v(face below); nothing comes in below the first cell."""
    return torch.cat([v.narrow(axis, 0, 1), v.narrow(axis, 1, v.shape[axis] - 1) - v.narrow(axis, 0, v.shape[axis] - 1)], axis)


def _reference(shape, pml, air, pulse, probes, steps, p, r=None, kappa=None):
    """The staggered pressure-velocity step in float64: (p, vx, vy, vz, traces [steps, probes])."""
    dt = COURANT * DX / (C * math.sqrt(3))
    cv, cp = -dt / (RHO * DX), -RHO * C * C * dt / DX
    dec = [d.view([-1 if a == b else 1 for b in range(3)]) for a, d in enumerate(_decays(shape, pml, dt))]
    w = _pulse(pulse, dt, steps)
    at = torch.zeros(shape, dtype=torch.float64, device="cuda")
    at[pulse.position] = 1.0
    cells = None if air is None else torch.from_numpy(air).cuda().double()
    coef, openf = [], []
    for a in range(3):
        lo, hi = (lambda t: t.narrow(a, 0, shape[a] - 1)), (lambda t: t.narrow(a, 1, shape[a] - 1))
        coef.append(cv if r is None else cv / ((lo(r) + hi(r)) / 2))
        openf.append(None if cells is None else lo(cells) * hi(cells))
    v = [torch.zeros_like(at) for _ in range(3)]
    scale = cp if kappa is None else cp * kappa
    rows = []
    for n in range(steps):
        new = []
        for a in range(3):
            m = shape[a] - 1
            u = v[a].narrow(a, 0, m) + coef[a] * (p.narrow(a, 1, m) - p.narrow(a, 0, m))
            new.append(torch.cat([u if openf[a] is None else u * openf[a], v[a].narrow(a, m, 1)], a))
        p = p + scale * (_diff(new[0], 0) + _diff(new[1], 1) + _diff(new[2], 2))
        if cells is not None:
            p = p * cells
        p = p * dec[0] * dec[1] * dec[2] + float(w[n]) * at
        v = [u * d for u, d in zip(new, dec)]
        rows.append(torch.stack([p[c] for c in probes]))
    return p, v[0], v[1], v[2], torch.stack(rows)


def exact(case, seed):
    kind, shape = case["kind"], None if case["kind"] == "serve" else _shape(case)
    if kind == "gradient":
        cells = shape[0] * shape[1] * shape[2]
        if cells * case["steps"] > 2.5e8:  # the graph of every step is held
            return None
        pb, rho, K, target = _design(case, seed)
        rho, K = [torch.from_numpy(x).cuda().double().requires_grad_(True) for x in (rho, K)]
        pad = [q for a in (2, 1, 0) for q in (pb.box_lo[a], shape[a] - pb.box_hi[a])]
        r, kappa = [1 + torch.nn.functional.pad(x - 1, pad) for x in (rho / RHO, K / (RHO * C * C))]
        tr = _reference(shape, case["pml"], None, pb.source, pb.probes, case["steps"], torch.zeros(shape, dtype=torch.float64, device="cuda"), r, kappa)[4]
        ((tr - torch.from_numpy(target).cuda().double()) ** 2).sum().backward()
        return {"traces": tr.detach(), "rho": rho.grad, "K": K.grad}
    if kind not in ("step", "solve", "advance") or case["scene"] not in ("air", "room", "pipe") or case["mics"]:
        return None
    _, air, pulse, probes = _solver(case, seed)
    p = _modes(case, seed).double() if kind == "advance" else torch.zeros(shape, dtype=torch.float64, device="cuda")
    p, vx, vy, vz, rows = _reference(shape, case["pml"], air, pulse, probes, case["steps"], p)
    order = sorted(range(len(probes)), key=lambda q: "probe%d" % q)[:16]
    return {"probes": [rows[:, q].contiguous() for q in order], "fields": {"p": p, "vx": vx, "vy": vy, "vz": vz}}

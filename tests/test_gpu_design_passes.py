"""Multi-step passes of the per-voxel design solve: traces and gradients of the
float32 march kernels, which take three steps per pass, equal the per-cell
kernels' bit for bit (the same operations in the same order, so the tolerance is
0) where windows, lanes, the design box and the step count have their edges."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# shape, box: lanes of every remainder; boxes one cell from the grid's faces, one
# voxel wide, off and on lane edges; several windows along j and along k
CASES = [((16, 14, 18), (1, 1, 1), (15, 13, 17)), ((12, 30, 31), (4, 9, 10), (5, 10, 11)),
         ((19, 61, 64), (3, 20, 4), (12, 47, 32)), ((9, 40, 129), (2, 6, 31), (7, 33, 98)),
         ((30, 12, 50), (11, 2, 3), (29, 9, 46)), ((5, 9, 1100), (1, 2, 500), (4, 7, 700))]


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("steps,history", [(3, "all"), (31, "all"), (32, "checkpoint"), (33, "checkpoint")])
def test_passes_equal_cell_kernels(case, steps, history):
    import torch
    from strata_fdtd_amd import GaussianPulse
    from strata_fdtd_amd.adjoint import DesignProblem, probe_traces
    shape, lo, hi = CASES[case]
    print(f"[design pass] {shape} {lo} {hi} {steps} {history}", flush=True)
    rng = np.random.default_rng(case)
    air = np.ones(shape, bool)
    air[tuple(rng.integers(0, n, 25) for n in shape)] = False
    src = tuple((a + b) // 2 for a, b in zip(lo, hi))
    probes = [src, lo, tuple(v - 1 for v in lo), hi, tuple(v - 1 for v in hi), lo]
    for p in [src] + probes:
        air[p] = True
    pb = DesignProblem(shape=shape, pml_depth=2 if min(shape) >= 9 else 0,
                       source=GaussianPulse(position=src, frequency=3e4), probes=probes, steps=steps, box_lo=lo,
                       box_hi=hi, checkpoint=14, geometry=air)
    rho = torch.tensor(pb.rho * (1 + 0.05 * rng.standard_normal(pb.box_shape)), dtype=torch.float32, device="cuda")
    K = torch.tensor(pb.K0 * (1 + 0.05 * rng.standard_normal(pb.box_shape)), dtype=torch.float32, device="cuda")
    target = torch.tensor(1e-3 * rng.standard_normal((steps, len(probes))), dtype=torch.float32, device="cuda")
    out = {}
    for impl in ("cell", "fast"):
        r, k = rho.clone().requires_grad_(True), K.clone().requires_grad_(True)
        tr = probe_traces(r, k, pb, impl=impl, history=history)
        ((tr - target) ** 2).sum().backward()
        out[impl] = (tr.detach(), r.grad, k.grad)
    for name, x, y in zip(("traces", "rho", "K"), out["cell"], out["fast"]):
        assert torch.equal(x, y), name
    assert out["fast"][0].abs().max() > 0

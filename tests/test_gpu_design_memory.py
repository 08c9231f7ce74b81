"""Design gradients where the passes' memory is not to be had: single steps with a
history of the box's own rows, the same traces and gradients bit for bit."""

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _counts():
    from strata_fdtd_amd import _native
    p, s = C.c_int64(), C.c_int64()
    _native.call("fdtd_design_step_counts", C.byref(p), C.byref(s))
    return p.value, s.value


@pytest.mark.parametrize("history", ["all", "checkpoint", "auto"])
@pytest.mark.parametrize("refused", ["scratch", "lanes"])
def test_single_steps_where_memory_is_refused(history, refused, monkeypatch):
    import torch
    from strata_fdtd_amd import GaussianPulse, adjoint
    pb = adjoint.DesignProblem(shape=(24, 26, 39), pml_depth=2, probes=[(13, 12, 12), (12, 12, 31)], steps=20,
                               source=GaussianPulse(position=(12, 12, 12), frequency=3e4), box_lo=(6, 6, 31),
                               box_hi=(18, 18, 33), checkpoint=20)
    rng = np.random.default_rng(1)
    rho = torch.tensor(pb.rho * (1 + 0.05 * rng.standard_normal(pb.box_shape)), dtype=torch.float32, device="cuda")
    g = torch.tensor(rng.standard_normal((20, 2)), dtype=torch.float32, device="cuda")

    def gradient():
        tr, saved = adjoint.forward_traces(pb, rho, None, keep_checkpoints=True, history=history)
        return (tr, *adjoint.adjoint_gradients(saved, g)), _counts()

    want, taken = gradient()
    assert taken == (6, 2)
    if history == "auto":
        free = 2 * adjoint.history_bytes(pb, lanes=False)
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device: (free, 10 * free))
    elif refused == "scratch":
        monkeypatch.setattr(adjoint, "pass_scratch_bytes", lambda pb, adjoint=True: 1 << 50)
    else:
        rows = adjoint._Fast._history

        def no_lanes(self, steps):
            if self._scratch is not None:
                raise torch.cuda.OutOfMemoryError("refused")
            return rows(self, steps)

        monkeypatch.setattr(adjoint._Fast, "_history", no_lanes)
    got, taken = gradient()
    assert taken == (0, 20)
    for a, b in zip(want, got):
        assert torch.equal(a, b)
    assert want[0].abs().max() > 0

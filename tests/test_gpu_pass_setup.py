"""What multi-step passes read is in place before they run, and passes are taken
where they should be: set-up orders, streams, and which route a solve takes."""

import numpy as np
import pytest

from helpers import make_solver, oracle_problem, seeded_scenario
from oracle import cpu

pytestmark = pytest.mark.gpu

FIELDS = ("p", "vx", "vy", "vz")


def _same(got, want, what):
    got = np.asarray(got)
    assert got.shape == want.shape, what
    assert np.array_equal(got, want), f"{what}: {int((got != want).sum())} of {want.size} differ"


def _compare(sc, s, st_o, tr_o):
    tr = s.get_probe_data()
    for q in range(len(sc.probes)):
        _same(tr[f"probe{q}"], tr_o[:, q], f"probe{q}")
    for k in FIELDS:
        _same(getattr(s, k), st_o[k], k)


def test_pass_sources_of_a_solver_on_a_side_stream(oracle_lib):
    """A z-plane source (in the single steps' per-cell tables, in the passes' own
    list beside them) of a solver made under a side stream, run while another stream
    with work queued is current: the passes see the whole waveform."""
    import torch
    sc = seeded_scenario(21, shape=(24, 36, 52), pml=4)
    sc.sources.append(("plane", 2, 9, 7000.0))
    n = 30
    st_o, tr_o = cpu.run(oracle_problem(sc, n), n)
    with torch.cuda.stream(torch.cuda.Stream()):
        s = make_solver(sc)
    torch.cuda.synchronize()
    busy = torch.ones(1 << 27, device="cuda")
    for _ in range(200):
        busy.mul_(1.0)
    s.step_n(n)
    torch.cuda.synchronize()
    _compare(sc, s, st_o, tr_o)


@pytest.mark.parametrize("every,waits", [(1, 0), (4, 10), (None, 1)])
def test_progress_bar_waits_for_runs_of_steps_only(every, waits, monkeypatch):
    """run(progress=True): a recorded step by itself is enqueued and not waited for
    (snapshots of every step would otherwise each stop the device); between recorded
    steps one wait per run of steps."""
    import torch
    from strata_fdtd_amd import FDTDSolver
    s = FDTDSolver(shape=(24, 24, 24), resolution=1e-3)
    if every:
        s.enable_snapshots(every)
    s.step_n(40 if every is None else 4 * every)       # set up
    s.reset()
    n = []
    real = torch.cuda.Stream.synchronize
    monkeypatch.setattr(torch.cuda.Stream, "synchronize", lambda self: (n.append(1), real(self))[1])
    during = []
    from tqdm import tqdm
    close = tqdm.close
    monkeypatch.setattr(tqdm, "close", lambda self: (during.append(len(n)), close(self))[1])
    s.run(39.5 * s.dt, progress=True)
    assert during[0] == waits
    if every:
        assert len(s.get_snapshots()) == 40 // every

"""Bytes of the design solve's history and the choice made from them (host code)."""

import numpy as np
import pytest

from strata_fdtd_amd.adjoint import DesignProblem, _pick_history, history_bytes, pass_scratch_bytes


def problem(lo, hi, steps=1000):
    return DesignProblem(shape=(64, 64, 64), pml_depth=4, source=None, probes=[], steps=steps, box_lo=lo, box_hi=hi)


def lanes(lo, hi):
    return 4 * (-(-hi // 4) - lo // 4)


@pytest.mark.parametrize("lo,hi", [((8, 8, 31), (40, 40, 33)), ((8, 8, 32), (40, 40, 33)), ((5, 9, 7), (6, 50, 12)),
                                   ((16, 16, 16), (48, 48, 48)), ((1, 1, 1), (63, 63, 63))])
def test_history_bytes_count_what_is_allocated(lo, hi):
    """Rows along z of whole 4-cell lanes (p's reach one cell past the box), the
    other axes' as they are; lanes=False: the box's own."""
    pb = problem(lo, hi)
    bx, by, bz = (h - l for l, h in zip(lo, hi))
    p = (bx + 2) * (by + 2) * lanes(lo[2] - 1, hi[2] + 1)
    div = bx * by * lanes(lo[2], hi[2])
    assert history_bytes(pb) == 4 * 1000 * (p + div)
    assert history_bytes(pb, 7) == 4 * 7 * (p + div)
    own = (bx + 2) * (by + 2) * (bz + 2) + bx * by * bz
    assert history_bytes(pb, lanes=False) == 4 * 1000 * own <= history_bytes(pb)
    assert pass_scratch_bytes(pb) > pass_scratch_bytes(pb, adjoint=False) > 0


def test_auto_history_fits_half_the_free_memory(monkeypatch):
    """A panel two voxels thick off the lanes: its lanes take 2.6 times its rows, so
    there is memory for the one and not the other, and for neither."""
    import torch
    pb = problem((8, 8, 31), (40, 40, 33))
    whole, own, scratch = history_bytes(pb), history_bytes(pb, lanes=False), pass_scratch_bytes(pb)
    assert whole > 2.5 * own
    for free, want in ((2 * (whole + scratch), ("all", True)), (2 * (whole + scratch) - 2, ("all", False)),
                       (2 * own, ("all", False)), (2 * own - 2, ("checkpoint", True))):
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device, f=free: (f, 10 * f))
        assert _pick_history(pb, "auto", "cuda:0") == want
    assert _pick_history(pb, "checkpoint", "cuda:0") == ("checkpoint", True)

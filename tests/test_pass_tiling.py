"""How a multi-step pass splits a grid (fdtd_pass_tiling, host code): every cell
is stored by exactly one workgroup, far enough inside its window that three
steps of lost edge cells do not reach it, and every index the kernel forms from
the split stays inside the workgroup's threads and LDS."""

import numpy as np
import pytest

STEPS = 3
SHAPES = [(2, 2, 2), (3, 5, 9), (40, 40, 40), (100, 100, 100), (180, 76, 76), (131, 157, 203), (261, 243, 307),
          (512, 512, 512), (320, 320, 480), (12, 61, 1030), (5000, 7, 3), (7, 5000, 9), (4, 6, 4000), (9, 40, 2049)]


def _tiling(shape):
    from strata_fdtd_amd import _native
    out = np.zeros(9, np.int32)
    _native.call("fdtd_pass_tiling", *shape, out.ctypes.data)
    return dict(zip(("steps", "nt", "kt", "ko", "rows", "nseg", "njt", "units", "nwg"), (int(v) for v in out)))


def _random_shapes(n):
    rng = np.random.default_rng(3)
    return [tuple(int(np.exp(rng.uniform(np.log(2), np.log(900)))) + 1 for _ in range(3)) for _ in range(n)]


@pytest.mark.parametrize("shape", SHAPES + _random_shapes(60))
def test_windows_cover_the_grid_once(shape):
    nx, ny, nz = shape
    t = _tiling(shape)
    assert t["steps"] == STEPS
    assert t["rows"] * t["kt"] <= t["nt"] and t["kt"] <= 256
    # rows stored by window b, and how far they lie from window edges that are not the grid's
    rows = np.zeros(ny, int)
    inner = t["rows"] - 2 * STEPS
    for b in range(t["njt"]):
        w0 = b * inner
        lo = 0 if b == 0 else w0 + STEPS
        hi = ny if b == t["njt"] - 1 else w0 + t["rows"] - STEPS
        assert 0 <= w0 and lo < hi
        assert w0 == 0 or lo - w0 >= STEPS
        assert w0 + t["rows"] >= ny if b == t["njt"] - 1 else w0 + t["rows"] - hi >= STEPS
        rows[lo:hi] += 1
    assert np.all(rows == 1)
    cells = np.zeros(nz, int)
    for b in range(t["nseg"]):
        k0 = 4 * (0 if b == 0 else b * t["ko"] - 1)
        lo, hi = 4 * b * t["ko"], nz if b == t["nseg"] - 1 else 4 * (b + 1) * t["ko"]
        end = k0 + 4 * t["kt"]
        assert lo < nz and lo < hi
        assert k0 == 0 or lo - k0 >= STEPS
        assert end >= nz if b == t["nseg"] - 1 else end - hi >= STEPS
        cells[lo:hi] += 1
    assert np.all(cells == 1)
    chunks = -(-nx // t["units"])
    assert t["nwg"] == t["nseg"] * t["njt"] * chunks and (chunks - 1) * t["units"] < nx


def test_no_passes_beyond_32_bit_offsets():
    assert _tiling((1024, 1024, 1024))["steps"] == 0
    assert _tiling((1024, 1024, 1023))["steps"] == STEPS


def test_long_grids_are_split_quickly():
    """The split of 10^8 planes takes milliseconds (one look at each chunk length,
    not at each number of chunks: 82 seconds)."""
    import time
    start = time.perf_counter()
    t = _tiling((100_000_000, 2, 2))
    assert time.perf_counter() - start < 5.0
    assert (t["units"], t["nwg"], t["nseg"]) == (97657, 1024, 1)

"""The per-cell kernels on their own, with tiles in contiguous runs (no LDS family, no
non-temporal launches), for every tile width that the host picks on planes up to 200 x
90 cells, 16 to 36 columns: against the oracle bit for bit, in place and with E in
ring slots.  For most widths one plane that whole tiles cover and one whose last
column and row of tiles are cut."""
import pytest

from tests.test_gpu_tiles import test_tiles_bitwise as tiles_bitwise

# width, ix, iy
PLANES = [(16, 29, 25), (16, 16, 16), (17, 33, 22), (18, 35, 22), (18, 18, 14), (19, 37, 17),
          (20, 39, 17), (21, 41, 17), (22, 43, 17), (22, 22, 11), (23, 45, 17), (24, 47, 17),
          (25, 49, 17), (25, 25, 10), (26, 51, 17), (27, 53, 17), (28, 55, 17), (28, 28, 9),
          (29, 85, 23), (30, 88, 23), (31, 91, 23), (31, 31, 8), (32, 94, 21), (32, 32, 8),
          (33, 65, 34), (33, 33, 21), (34, 101, 19), (35, 103, 19), (36, 36, 18)]


def cell_tile(ix, iy):
    """The library's choice (cell_tile): fewest idle lanes and halo loads."""
    best, w = 0, 0
    for cw in range(16, 39):
        ch = min(256 // cw, 42 - cw)
        if (cw + 3) * (ch + 3) > 400:
            continue
        cost = -(-ix // cw) * -(-iy // ch) * (256 + cw + ch)
        if best == 0 or cost < best:
            best, w = cost, cw
    return w


def test_the_planes_cover_every_width():
    assert all(cell_tile(ix, iy) == w for w, ix, iy in PLANES)
    assert {cell_tile(ix, iy) for ix in range(8, 200) for iy in range(8, 90)} == {w for w, _, _ in PLANES}


@pytest.mark.gpu
@pytest.mark.parametrize("ring", [0, 5])
@pytest.mark.parametrize("plane", PLANES)
def test_runs_of_tiles_bitwise(plane, ring, monkeypatch):
    monkeypatch.setenv("MITTET_FDTD_NOLDS", "1")
    monkeypatch.setenv("MITTET_FDTD_NT", "0")
    _, ix, iy = plane
    tiles_bitwise((ix, iy, 11, 2 + ix % 2 if min(ix, iy) >= 10 else 2), ring)

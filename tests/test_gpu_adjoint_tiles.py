"""Adjoint tiles around a narrow LDS region: the region starts at a multiple of 8
on x, the edge tiles beside it are 16 wide, and each cell belongs to one tile only.
Where the region ends inside the first segment's last tile the gradient is that of
the per-cell passes alone up to rounding (1e-12 of the largest component: 60 steps
of some 50 operations at 1.1e-16 each), the same in every run, and the host's count
of the tiles is the library's."""
import numpy as np
import pytest

import mittet_main_amd._lib as lib
from mittet_main_amd import Grid, Model, firstderiv_gauss, serving
from mittet_main_amd.adjoint import GradientProblem, ShotSpec
from mittet_main_amd.configs import dt_for

pytestmark = pytest.mark.gpu

OM0 = 2 * np.pi
# region columns [8, 12), [8, 15), [8, 16), [8, 17), [24, 26); of rows and planes some whole tiles
GRIDS = [(20, 40, 33, 7), (23, 39, 33, 7), (24, 40, 33, 7), (25, 40, 33, 7), (50, 66, 60, 23)]


@pytest.mark.parametrize("dims", GRIDS)
def test_no_cell_is_in_two_tiles(dims, monkeypatch):
    print(f"adjoint tiles: {dims}", flush=True)
    ix, iy, iz, nc = dims
    it = 61
    dt, cmax = dt_for(50.0, 45.0, 40.0, sig_min=0.1)
    g = Grid(ix, iy, iz, nc, 50.0, 45.0, 40.0, dt, OM0, cmax)
    rng = np.random.default_rng(ix)
    sig = np.exp(rng.uniform(np.log(0.1), np.log(2.0), g.shape))
    src = (ix - nc - 3, iy // 2, iz // 2)
    rec = [(ix // 2, iy // 2 - 3, iz // 2), (ix - 3, iy // 2, iz // 2 + 1)]

    def run():
        P = GradientProblem(g, [ShotSpec(src, firstderiv_gauss(it, dt, 0.2 / dt))], rec, it, [6.0])
        P.d_obs = [np.zeros((3, 2, 1))]
        out = P.value_and_grad(np.log(sig))[1]
        P.close()
        return out

    region = [run() for _ in range(3)]
    m = Model(g)
    sh = m.shot(it, np.zeros(it), src, 0, np.array(rec, np.int32))
    assert serving.plan_bytes(g, it - 1, 2, 1) == lib.load().fwi3d_grad_plan_bytes(sh._h, 1)
    sh.close()
    m.close()
    monkeypatch.setenv("MITTET_FDTD_NOLDS", "1")
    want = run()
    assert np.abs(want).max() > 0
    for r in region:
        assert np.abs(r - want).max() <= 1e-12 * np.abs(want).max()
        np.testing.assert_array_equal(r, region[0])

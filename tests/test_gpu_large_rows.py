"""Families on large grids: rows that 8 does not divide take the LDS kernels from 12 M
cells by default if they fill their columns, others the per-cell kernels; both give
the same bits on both sides of the rule."""
import numpy as np
import pytest

from mittet_main_amd import Grid, Model, firstderiv_gauss
from mittet_main_amd.configs import dt_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(234, 230, 226), (237, 228, 226), (230, 229, 230), (240, 226, 228),
                                  (182, 270, 250)])
def test_the_default_family_equals_the_other(dims, monkeypatch):
    monkeypatch.delenv("MITTET_FDTD_LDS")
    print(f"family on {dims}", flush=True)
    ix, iy, iz = dims
    dt, cmax = dt_for(50.0, 45.0, 40.0, sig_min=0.1)
    g = Grid(ix, iy, iz, 6, 50.0, 45.0, 40.0, dt, 2 * np.pi, cmax)
    m = Model(g)
    m.media_coeff_3d(np.exp(np.random.default_rng(ix).uniform(-2.0, 0.7, g.shape)))
    it, out = 14, []
    for env in (None, "MITTET_FDTD_NOLDS", "MITTET_FDTD_LDS"):
        if env:
            monkeypatch.setenv(env, "1")
        s = m.shot(it, firstderiv_gauss(it, dt, 0.5 / dt / it), (ix // 2, iy // 2, iz // 2), 1,
                   np.array([[ix // 2, iy // 2 + 2, iz // 2]], np.int32))
        # fields at the shell's and the interior's border too
        s.set_field(0, np.random.default_rng(1).standard_normal(g.shape))
        s.run()
        out.append([s.traces()] + [s.field(q) for q in (0, 2, 4)])
        s.close()
        if env:
            monkeypatch.delenv(env)
    m.close()
    assert np.abs(out[0][1]).max() > 0
    for o in out[1:]:
        for a, b in zip(out[0], o):
            np.testing.assert_array_equal(a, b)

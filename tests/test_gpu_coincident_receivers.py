"""Receivers on one cell: each has its own residual, and the adjoint source of the
cell is their sum.  The gradient of a shot with coincident receivers is bit for bit
that of a shot with one receiver per cell that has the summed sensitivities (the
sums taken in receiver order), with the adjoint's LDS region and without it, and
agrees with central differences of the misfit."""
import ctypes as C

import numpy as np
import pytest

from mittet_main_amd import Grid, Model, _lib, firstderiv_gauss
from mittet_main_amd.adjoint import GradientProblem, ShotSpec
from mittet_main_amd.configs import dt_for

pytestmark = pytest.mark.gpu

OM0 = 2 * np.pi


def setup(seed):
    ix, iy, iz, nc = 30, 27, 25, 5
    dt, cmax = dt_for(50.0, 45.0, 40.0, sig_min=0.1)
    g = Grid(ix, iy, iz, nc, 50.0, 45.0, 40.0, dt, OM0, cmax)
    rng = np.random.default_rng(seed)
    return g, np.exp(rng.uniform(np.log(0.1), np.log(2.0), g.shape)), dt, rng


def gradient(model, rec, it, signal, src, djdt):
    L, h = _lib.load(), C.c_void_p()
    s = model.shot(it, signal, src, 0, np.asarray(rec, np.int32))
    _lib.check(L.fwi3d_grad_create(s._h, 0, C.byref(h)))
    dj, gg = np.zeros(model.grid.ncells), np.ascontiguousarray(djdt)
    try:
        _lib.check(L.fwi3d_grad_forward(h))
        _lib.check(L.fwi3d_grad_backward(h, gg.ctypes.data_as(C.c_void_p), dj.ctypes.data_as(C.c_void_p)))
    finally:
        _lib.check(L.fwi3d_grad_destroy(h))
    s.close()
    return dj


@pytest.mark.parametrize("region", [True, False])
@pytest.mark.parametrize("copies", [(0, 1, 0), (0, 0), (0, 1, 2, 3, 1, 0, 1, 3, 3)])
def test_sensitivities_of_one_cell_are_summed(copies, region, monkeypatch):
    print(f"coincident receivers {copies}, region {region}", flush=True)
    monkeypatch.setenv("MITTET_FDTD_LDS" if region else "MITTET_FDTD_NOLDS", "1")
    g, sig, dt, rng = setup(3)
    it, src = 40, (15, 13, 12)
    # inside the region, in the CPML shell, on the source cell
    cells = [(14, 12, 11), (3, 20, 4), src, (20, 9, 15)]
    # one receiver per cell, in the order of its first copy
    order = list(dict.fromkeys(copies))
    djdt = rng.standard_normal((3, len(copies), it))
    summed = np.zeros((3, len(order), it))
    for r, c in enumerate(copies):
        summed[:, order.index(c)] += djdt[:, r]
    m = Model(g)
    m.media_coeff_3d(sig)
    signal = firstderiv_gauss(it, dt, 0.2 / dt)
    got = gradient(m, [cells[c] for c in copies], it, signal, src, djdt)
    want = gradient(m, [cells[c] for c in order], it, signal, src, summed)
    m.close()
    assert np.all(np.isfinite(got)) and np.abs(want).max() > 0
    np.testing.assert_array_equal(got, want)


def test_gradient_matches_central_differences():
    """Relative error at most 1e-6, as for distinct receivers (h = 1e-6 in log sigma)."""
    print("coincident receivers: central differences", flush=True)
    g, sig, dt, rng = setup(8)
    it = 200
    rec = [(14, 12, 11), (20, 9, 15), (14, 12, 11), (14, 12, 11), (9, 17, 8), (20, 9, 15)]
    P = GradientProblem(g, [ShotSpec((15, 13, 12), firstderiv_gauss(it, dt, 6.0))], rec, it,
                        2 * np.pi * np.array([1.0, 2.5]))
    P.d_obs = P.forward_data(sig)
    logs = np.log(np.full(g.shape, float(np.exp(np.mean(np.log(sig))))))
    _, grad = P.value_and_grad(logs)
    gmax, h = np.abs(grad).max(), 1e-6
    for _ in range(8):
        k, j, i = (int(v) for v in rng.integers(0, g.shape))
        lp = logs.copy()
        lp[k, j, i] += h
        jp = P.misfit(np.exp(lp))
        lp[k, j, i] -= 2 * h
        fd = (jp - P.misfit(np.exp(lp))) / (2 * h)
        err = abs(fd - grad[k, j, i]) / max(abs(grad[k, j, i]), 1e-3 * gmax)
        assert err <= 1e-6, ((k, j, i), grad[k, j, i], fd, err)
    P.close()

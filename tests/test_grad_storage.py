"""Device memory of a gradient: the adjoint's weights take no memory of their own
beyond 3 values per cell, so that a byte budget that once held a plan still holds it."""
import ctypes as C

import numpy as np
import pytest

from mittet_main_amd import Grid, Model, _lib, firstderiv_gauss, serving
from mittet_main_amd.adjoint import grad_plan
from mittet_main_amd.configs import dt_for

OM0 = 2 * np.pi


def grid(ix, iy, iz, nc):
    dt, cmax = dt_for(50.0, 45.0, 40.0, sig_min=0.1)
    return Grid(ix, iy, iz, nc, 50.0, 45.0, 40.0, dt, OM0, cmax)


@pytest.mark.parametrize("dims", [(61, 50, 44, 8), (152, 152, 152, 12), (416, 416, 416, 16),
                                  (300, 250, 200, 2), (500, 500, 8, 2), (90, 40, 40, 6)])
@pytest.mark.parametrize("levels", [1, 2, 3, 4, 8])
def test_no_plan_needs_more_than_states_and_one_phase_of_weights(dims, levels):
    """Every stored state with its psi, the weights of one phase (3 values per cell
    and one per psi value), the gradient, the receivers, the profiles, and the 16-byte
    tiles of the list for every 32 x 8 cells and 7 more per plane."""
    g = grid(*dims)
    nt, nrec = 1000, 64
    _, _, states = grad_plan(nt, levels)
    psi = 8 * g.ncpml * (g.iy * g.iz + g.ix * g.iz + g.ix * g.iy)
    state = -(-(6 * g.ncells + psi) // 32) * 32
    other = 3 * g.ncells + psi + g.ncells + 1 + 3 * nrec * (nt + 1) + 2 * (g.ix + g.iy + g.iz)
    tiles = g.iz * (-(-g.ix // 32) * -(-g.iy // 8) + 7)
    assert serving.plan_bytes(g, nt, nrec, levels) <= 8 * (states * state + other) + 16 * tiles


@pytest.mark.gpu
@pytest.mark.parametrize("segment", [0, 7, 39])
@pytest.mark.parametrize("region", [True, False])
def test_a_second_backward_sweep_gives_the_same_gradient(segment, region, monkeypatch):
    """The sweep uses idle states for its weights; the checkpoints are whole again
    after it.  39 steps: whole segments, a short last one, one segment."""
    print(f"two backward sweeps: segment {segment}, region {region}", flush=True)
    monkeypatch.setenv("MITTET_FDTD_LDS" if region else "MITTET_FDTD_NOLDS", "1")
    g, it = grid(31, 27, 25, 5), 40
    rng = np.random.default_rng(1)
    m = Model(g)
    m.media_coeff_3d(np.exp(rng.uniform(np.log(0.1), np.log(2.0), g.shape)))
    s = m.shot(it, firstderiv_gauss(it, g.dt, 0.2 / g.dt), (15, 13, 12), 0,
               np.array([[9, 9, 9], [20, 12, 14]], np.int32))
    L, h = _lib.load(), C.c_void_p()
    _lib.check(L.fwi3d_grad_create(s._h, segment, C.byref(h)))
    _lib.check(L.fwi3d_grad_forward(h))
    djdt = [rng.standard_normal((3, 2, it)) for _ in range(2)]

    def backward(d):
        out = np.zeros(g.ncells)
        _lib.check(L.fwi3d_grad_backward(h, d.ctypes.data_as(C.c_void_p), out.ctypes.data_as(C.c_void_p)))
        return out

    first = backward(djdt[0])
    fields = [s.field(q) for q in range(6)]
    other = backward(djdt[1])
    again = backward(djdt[0])
    assert np.abs(first).max() > 0 and np.abs(other - first).max() > 0
    np.testing.assert_array_equal(first, again)
    for q in range(6):   # the shot's fields at the end of a sweep depend on the forward pass alone
        np.testing.assert_array_equal(s.field(q), fields[q])
    _lib.check(L.fwi3d_grad_destroy(h))
    s.close()
    m.close()

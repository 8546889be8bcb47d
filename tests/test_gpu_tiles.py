"""Tiles of the per-cell forward kernels: rows and columns cut by the grid's
edges, planes of less than one tile, and the thinnest CPML, against the oracle
bit for bit: all six fields and the traces, in place and with E in ring slots,
per operator and fused (with the LDS family over the interior where it has one;
the per-cell kernels alone: test_gpu_tile_shapes.py)."""
import numpy as np
import pytest

import oracle
from mittet_main_amd import Batch, Grid, Model, firstderiv_gauss
from mittet_main_amd.adjoint import GradientProblem, ShotSpec
from mittet_main_amd.configs import dt_for

pytestmark = pytest.mark.gpu

OM0 = 2 * np.pi
# ix, iy, iz, ncpml: a plane below one tile; one cell more or less than a
# tile's columns or rows
GRIDS = [(8, 8, 8, 2), (9, 31, 8, 2), (17, 13, 9, 2), (21, 12, 11, 3), (22, 37, 13, 3),
         (33, 24, 14, 5), (43, 25, 12, 4), (71, 20, 15, 5), (96, 19, 12, 4), (131, 11, 12, 3)]


@pytest.mark.parametrize("ring", [0, 5])
@pytest.mark.parametrize("dims", GRIDS)
def test_tiles_bitwise(dims, ring):
    ix, iy, iz, nc = dims
    print(f"tiles {dims} ring {ring}", flush=True)
    rng = np.random.default_rng(ix + iy)
    sig = np.exp(rng.uniform(np.log(0.05), np.log(3.0), (iz, iy, ix)))
    dl = (50.0, 45.0, 40.0)
    dt, cmax = dt_for(*dl, sig_min=0.05)
    it = 17
    signal = firstderiv_gauss(it, dt, 0.5 / dt / it)
    src = (ix // 2, iy // 2, iz // 2)
    rec = np.array([[1, 1, 1], [ix - 2, iy - 2, iz - 2], [ix // 2, iy - 3, iz // 2]], np.int32)
    m = Model(Grid(ix, iy, iz, nc, *dl, dt, OM0, cmax))
    m.media_coeff_3d(sig)
    S = oracle.OracleSim(ix, iy, iz, nc, *dl, dt, OM0, cmax)
    S.set_sigma(sig)
    S.init_cpml()
    S.media_coeff_3d()
    # fields of every magnitude at the edges too: random, the same on both sides
    shot = m.shot(it, signal, src, 1, rec, [3.0] if ring else None, ring)
    for q, nm in enumerate(oracle.FIELD_NAMES):
        v = rng.standard_normal((iz, iy, ix))
        shot.set_field(q, v)
        S.arr(nm)[...] = v
    src1 = tuple(c + 1 for c in src)
    if ring:
        shot.step_n(7)
    else:   # three steps by the single operators, which advance no step counter
        for n in range(3):
            shot.e_field_cpml42()
            shot.epml_abcs4()
            shot.read_source_3d(n)
            shot.h_field_cpml42()
            shot.hpml_abcs4()
        S.forward(1, signal, src1, 3)
    shot.run()
    tr, _ = S.forward(1, signal, src1, it - 1, rec1=rec + 1, it=it)
    np.testing.assert_array_equal(shot.traces()[:3, :, : it - 1], tr[:, :, : it - 1])
    for q, nm in enumerate(oracle.FIELD_NAMES):
        np.testing.assert_array_equal(shot.field(q), S.arr(nm), err_msg=nm)
    m.close()


@pytest.mark.parametrize("family", ["cells", "lds", "batch"])
@pytest.mark.parametrize("dims", [(8, 8, 8, 2), (17, 13, 9, 2), (43, 25, 19, 4), (131, 11, 17, 3),
                                  (70, 37, 22, 3)])
def test_tiles_in_layers_bitwise(dims, family, monkeypatch):
    """Launches that take their tiles in layers of a plane or a z-chunk (those
    with non-temporal fields; MITTET_FDTD_NT=1): planes of fewer tiles than
    XCDs and of a number that 8 does not divide, more and fewer than 8 planes
    per turn, a shell list, and two shots in one launch, against the oracle
    bit for bit."""
    ix, iy, iz, nc = dims
    monkeypatch.setenv("MITTET_FDTD_NT", "1")
    monkeypatch.setenv("MITTET_FDTD_LDS" if family == "lds" else "MITTET_FDTD_NOLDS", "1")
    print(f"layers {dims} {family}", flush=True)
    rng = np.random.default_rng(ix)
    dl = (50.0, 45.0, 40.0)
    dt, cmax = dt_for(*dl, sig_min=0.05)
    it = 12
    signal = firstderiv_gauss(it, dt, 0.5 / dt / it)
    src = (ix // 2, iy // 2, iz // 2)
    rec = np.array([[1, 1, 1], [ix - 2, iy - 2, iz - 2]], np.int32)
    runs = []
    for _ in range(2 if family == "batch" else 1):
        sig = np.exp(rng.uniform(np.log(0.05), np.log(3.0), (iz, iy, ix)))
        m = Model(Grid(ix, iy, iz, nc, *dl, dt, OM0, cmax))
        m.media_coeff_3d(sig)
        S = oracle.OracleSim(ix, iy, iz, nc, *dl, dt, OM0, cmax)
        S.set_sigma(sig)
        S.init_cpml()
        S.media_coeff_3d()
        runs.append((m, m.shot(it, signal, src, 2, rec), S))
    if family == "batch":
        b = Batch(2)
        for _, shot, _ in runs:
            b.add(shot)
        b.step(it - 1)
        b.sync()
        for _, shot, _ in runs:
            b.remove(shot)
        b.close()
    else:
        runs[0][1].run()
    for m, shot, S in runs:
        tr, _ = S.forward(2, signal, tuple(c + 1 for c in src), it - 1, rec1=rec + 1, it=it)
        np.testing.assert_array_equal(shot.traces()[:3], tr)
        for q, nm in enumerate(oracle.FIELD_NAMES):
            np.testing.assert_array_equal(shot.field(q), S.arr(nm), err_msg=nm)
        shot.close()
        m.close()


def test_replayed_states_are_complete():
    """A replay writes each state to memory no step has written before; H cells
    outside every update range are part of it.  The gradient is the same
    whatever the memory held: before and after NaN fields lived there."""
    ix, iy, iz, nc, it = 30, 27, 25, 5, 40
    dt, cmax = dt_for(50.0, 45.0, 40.0, sig_min=0.1)
    g = Grid(ix, iy, iz, nc, 50.0, 45.0, 40.0, dt, OM0, cmax)
    sig = np.exp(np.random.default_rng(5).uniform(np.log(0.1), np.log(2.0), g.shape))

    def gradient():
        P = GradientProblem(g, [ShotSpec((15, 13, 12), firstderiv_gauss(it, dt, 0.2 / dt))],
                            [[9, 9, 9], [20, 12, 14]], it, [6.0])
        P.d_obs = [np.zeros((3, 2, 1))]
        out = P.value_and_grad(np.log(sig))
        P.close()
        return out

    J0, g0 = gradient()
    m = Model(g)
    m.media_coeff_3d(sig)
    poison = [m.shot(it, None, ring=r, omega_vol=[1.0] if r else None) for r in (0, 8, 16)]
    for s in poison:
        for q in range(6):
            s.set_field(q, np.full(g.shape, np.nan))
        s.run()
        s.sync()
    m.close()
    J1, g1 = gradient()
    assert J0 == J1 and np.all(np.isfinite(g1))
    np.testing.assert_array_equal(g0, g1)


@pytest.mark.parametrize("members", [1, 3])
def test_fortran_receivers_on_the_source_cells(members):
    """H of a step is sampled before the next step's source changes it, alone
    and in a batch, over chunk borders (32 steps)."""
    from mittet_main_amd import Batch
    from tests.test_gpu_fortran import gpu_shot, oracle_run, setup

    nt = 37
    g, sig, mu, sigw, src, rec, *_ = setup(27, 23, 21, nt=nt)
    rec = np.concatenate([rec, np.array(src)])
    _, tr_o = oracle_run(g, sig, mu, sigw, src, rec, nt)
    m = Model(g, variant=1)
    m.set_mu(mu)
    m.media_coeff_3d(sig)
    shots = [gpu_shot(m, g, sigw, src, rec, nt) for _ in range(members)]
    if members > 1:
        b = Batch(members)
        for s in shots:
            b.add(s)
        b.step(nt)
        b.sync()
        for s in shots:
            b.remove(s)
    else:
        shots[0].run()
    for s in shots:
        np.testing.assert_array_equal(s.traces()[:, :, :nt], tr_o[:, :, :nt])
    m.close()

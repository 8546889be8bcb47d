"""Members of a batch that have finished their time loop cost next to nothing until
they are removed: they get no blocks from the next chunk on, and until then their
blocks end before they load a field.  They keep their results, and run again when
they are removed, cleared and added."""
import time

import numpy as np
import pytest

from mittet_main_amd import Batch, Grid, Model, firstderiv_gauss
from mittet_main_amd.configs import dt_for
from mittet_main_amd.fwi3d import SRC_HZ, fortran_grid

pytestmark = pytest.mark.gpu

OM0 = 2 * np.pi


@pytest.mark.parametrize("variant", [0, 1])
def test_finished_members_load_nothing(variant, monkeypatch):
    """A running 24^3 shot beside six of 120^3: steps after those have finished take
    less than half the time of steps before, and no more than twice the small shot's
    own plus 20 us a launch.  (Loads alone are two thirds of a step's traffic: a
    finished member that still loaded its fields would leave more than half.)"""
    monkeypatch.setenv("MITTET_FDTD_NOLDS", "1")
    print(f"finished members, variant {variant}", flush=True)
    n_run, n_done = 24, 120
    models, shots, b = [], [], Batch(7)
    for q, n in enumerate([n_run] + 6 * [n_done]):
        dt, cmax = dt_for(50.0, 50.0, 50.0, sig_min=0.1)
        args = (n, n, n, 6, 50.0, 50.0, 50.0, dt, OM0, cmax)
        m = Model(fortran_grid(*args) if variant else Grid(*args), variant=variant)
        if variant:
            m.set_mu(np.full((n, n, n), 1.2566370614e-6))
        m.media_coeff_3d(np.ones((n, n, n)))
        it = 4001 if n == n_run else 257
        s = m.shot(it, firstderiv_gauss(it, dt, 0.1 / dt), (n // 2,) * 3, SRC_HZ if variant else 0)
        models.append(m)
        shots.append(s)
        b.add(s)

    def steps(k):
        b.sync()
        t = time.perf_counter()
        b.step(k)
        b.sync()
        return (time.perf_counter() - t) / k

    steps(64)
    running = min(steps(64) for _ in range(3))     # 256 steps: all six have finished
    assert all(s.step == 256 for s in shots)
    done = min(steps(128) for _ in range(8))
    for s in shots[1:]:
        b.remove(s)
    steps(64)
    alone = min(steps(128) for _ in range(8))
    print(f"us a step: running {1e6 * running:.1f}, finished {1e6 * done:.1f}, alone {1e6 * alone:.1f}",
          flush=True)
    b.remove(shots[0])
    b.close()
    for m in models:
        m.close()
    assert done < 0.5 * running
    assert done < 2 * alone + 40e-6


@pytest.mark.parametrize("ring", [0, 8])
@pytest.mark.parametrize("lds", ["MITTET_FDTD_LDS", "MITTET_FDTD_NOLDS"])
def test_members_end_at_different_steps(ring, lds, monkeypatch):
    """Chunks of 8 steps; members end inside a chunk, at its border and one step
    beyond it; one is removed, starts again and joins the others.  Each equals the same shot
    run alone, bit for bit."""
    print(f"members end at different steps, ring {ring}, {lds}", flush=True)
    monkeypatch.setenv(lds, "1")
    its, dims = (12, 17, 18, 61, 30), ((24, 20, 21), (18, 25, 20), (33, 19, 22), (20, 20, 20), (40, 21, 24))

    def build():
        out = []
        for it, (ix, iy, iz) in zip(its, dims):
            dt, cmax = dt_for(50.0, 45.0, 40.0, sig_min=0.1)
            m = Model(Grid(ix, iy, iz, 5, 50.0, 45.0, 40.0, dt, OM0, cmax))
            m.media_coeff_3d(np.exp(np.random.default_rng(ix).uniform(-2, 1, (iz, iy, ix))))
            out.append((m, m.shot(it, firstderiv_gauss(it, dt, 0.2 / dt), (ix // 2, iy // 2, iz // 2), 1,
                                  np.array([[6, 7, 8], [ix // 2, 9, 10]], np.int32),
                                  [3.0, 5.0] if ring else None, ring)))
        return out

    def result(s):
        return [s.traces()] + [s.field(q) for q in range(6)] + ([s.volume_dft()] if ring else [])

    want = build()
    for _, s in want:
        s.run()
    got = build()
    b = Batch(len(its), chunk=8)
    for _, s in got:
        b.add(s)
    b.step(20)
    b.sync()
    again = got[1][1]
    first = result(again)
    b.remove(again)
    again.set_zero_eh()
    again.sync()
    b.add(again)
    b.step(100)
    b.sync()
    for (_, s), (_, w) in zip(got, want):
        assert s.step == s.it - 1
        b.remove(s)
        for x, y in zip(result(s), result(w)):
            np.testing.assert_array_equal(x, y)
    for x, y in zip(first, result(again)):
        np.testing.assert_array_equal(x, y)
    b.close()
    for m, _ in got + want:
        m.close()

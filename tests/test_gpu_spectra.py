"""Receiver and waveform spectra at the edges of the DFT kernels' tiles (16 rows,
1024 samples) against the sums in numpy, and two threads asking one shot."""
import threading

import numpy as np
import pytest

from mittet_main_amd import Grid, Model, firstderiv_gauss
from mittet_main_amd.configs import dt_for

pytestmark = pytest.mark.gpu

OM0 = 2 * np.pi
# Relative to the sum of |terms|: up to 2100 additions of 1.1e-16 in each of the two
# orders of summation and the weights' few units in the last place
TOL = 2 * 2100 * 1.2e-16


def make(nrec, it):
    dl = (50.0, 45.0, 40.0)
    dt, cmax = dt_for(*dl, sig_min=0.1)
    m = Model(Grid(14, 13, 12, 3, *dl, dt, OM0, cmax))
    m.media_coeff_3d(np.full((12, 13, 14), 0.4))
    rec = np.array([[3 + r % 7, 3 + r % 5, 3 + r % 4] for r in range(nrec)], np.int32)
    s = m.shot(it, firstderiv_gauss(it, dt, 0.5 / dt / it), (7, 6, 5), 0, rec)
    s.run()
    return m, s, dt


def weights(it, dt, om):
    n = np.arange(it)[None, :]
    a = np.sqrt(OM0 * om)[:, None]
    return dt * np.exp((-1.0 + 1.0j) * a * n * dt)


@pytest.mark.parametrize("nrec, it", [(1, 2), (2, 64), (3, 1023), (5, 1024), (6, 1025), (11, 2100)])
def test_spectra_at_tile_edges(nrec, it):
    print(f"spectra: {6 * nrec} rows of {it} samples", flush=True)
    m, s, dt = make(nrec, it)
    tr = s.traces().reshape(6 * nrec, it)
    om = 2 * np.pi * np.array([0.0, 0.5, 3.0])
    w = weights(it, dt, om)
    got = s.receiver_dft(om, h_factor=False).reshape(6 * nrec, om.size)
    lim = TOL * (np.abs(tr) @ np.abs(w).T)
    assert np.all(np.abs(got - tr @ w.T) <= lim + 1e-300)
    # bins of the waveforms and the traces
    nb = min(it, 5)
    strue = np.cos(np.arange(it) * 0.37) + 0.1
    ob = 2 * np.pi / it / dt * np.arange(nb)
    wb = weights(it, dt, ob)
    res = s.laplace_to_freq(nb, strue)
    e = tr[: 3 * nrec] @ wb.T
    assert np.all(np.abs(res["E"].reshape(3 * nrec, nb) - e) <= TOL * (np.abs(tr[: 3 * nrec]) @ np.abs(wb).T) + 1e-300)
    bins = np.exp(2j * np.pi * (np.outer(np.arange(nb), np.arange(it)) % it) / it)
    tru = bins @ strue
    g = res["G"]
    ok = np.isfinite(g) & np.isfinite(res["OBS"])
    t = np.broadcast_to(tru, g.shape)
    assert np.all(np.abs(res["OBS"] - g * t)[ok] <= (TOL * np.abs(strue).sum() * np.abs(g) + 1e-15 * np.abs(g * t))[ok])
    # a request of its own memory gives the same bits as the kept one
    many = 2 * np.pi * np.linspace(0.1, 5.0, 400000 // (6 * nrec))
    big = s.receiver_dft(np.concatenate([om, many]), h_factor=False).reshape(6 * nrec, -1)
    np.testing.assert_array_equal(big[:, : om.size], got)
    s.close()
    m.close()


def test_two_threads_ask_one_shot():
    print("spectra of one shot from two threads", flush=True)
    m, s, dt = make(4, 300)
    oms = [2 * np.pi * np.linspace(0.1, 4.0, 7), 2 * np.pi * np.linspace(0.2, 3.0, 50)]
    want = [s.receiver_dft(om) for om in oms]
    got = [[], []]

    def ask(q):
        for _ in range(20):
            got[q].append(s.receiver_dft(oms[q]))

    th = [threading.Thread(target=ask, args=(q,)) for q in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for q in range(2):
        for a in got[q]:
            np.testing.assert_array_equal(a, want[q])
    s.close()
    m.close()

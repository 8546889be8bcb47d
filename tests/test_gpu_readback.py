"""Volume spectra read back through pinned pieces by several host threads (32 MiB
and more into pageable memory) against the direct copy into pinned memory: the
same bytes for rows that the pieces do and do not divide, on both sides of the
limit, and for two shots of one model read at the same time."""
import ctypes as C
import threading

import numpy as np
import pytest
import torch

from mittet_main_amd import Grid, Model, _lib, firstderiv_gauss
from mittet_main_amd.configs import dt_for

pytestmark = pytest.mark.gpu

OM0 = 2 * np.pi


def shots_of(dims, nf, count):
    ix, iy, iz = dims
    dl = (50.0, 45.0, 40.0)
    dt, cmax = dt_for(*dl, sig_min=0.1)
    rng = np.random.default_rng(ix)
    m = Model(Grid(ix, iy, iz, 4, *dl, dt, OM0, cmax))
    m.media_coeff_3d(np.exp(rng.uniform(np.log(0.1), np.log(2.0), (iz, iy, ix))))
    it = 24
    shots = []
    for q in range(count):
        s = m.shot(it, firstderiv_gauss(it, dt, 1.0 + q), (ix // 2, iy // 2, iz // 2), q % 3,
                   np.array([[5, 5, 5]], np.int32), [1.0 + f for f in range(nf)], 8)
        s.enable_volume_dft_h()
        s.run()
        shots.append(s)
    return m, shots


def pinned(shot, h):
    n = 3 * shot.nf * shot.model.grid.ncells * 2
    t = torch.zeros(n, dtype=torch.float64, pin_memory=True)
    fn = _lib.load().fwi3d_get_volume_dft_h if h else _lib.load().fwi3d_get_volume_dft
    _lib.check(fn(shot._h, C.c_void_p(t.data_ptr())))
    return t.numpy().view(np.complex128).copy()


# just below and above the limit, odd rows below and above one piece
@pytest.mark.parametrize("dims, nf", [((64, 64, 85), 2), ((64, 64, 86), 2), ((61, 57, 53), 5),
                                      ((131, 127, 97), 1), ((149, 151, 73), 3)])
def test_volume_readback_equals_the_direct_copy(dims, nf):
    print(f"read-back {dims} nf {nf}: {np.prod(dims) * 48 * nf} bytes", flush=True)
    m, (shot,) = shots_of(dims, nf, 1)
    for h, get in ((False, shot.volume_dft), (True, shot.volume_dft_h)):
        want = pinned(shot, h)
        assert np.abs(want).max() > 0
        np.testing.assert_array_equal(get().reshape(-1), want)
    shot.close()
    m.close()


def test_two_shots_read_back_at_the_same_time():
    print("read-back of two shots of one model from two threads", flush=True)
    m, shots = shots_of((96, 90, 80), 2, 2)
    want = [pinned(s, False) for s in shots]
    got = [None, None]

    def read(q):
        for _ in range(3):
            got[q] = shots[q].volume_dft().reshape(-1)

    th = [threading.Thread(target=read, args=(q,)) for q in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)
    for s in shots:
        s.close()
    m.close()

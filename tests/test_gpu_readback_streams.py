"""Large volume read-backs of models on streams of the caller's: a torch stream, and
the per-thread stream, whose handle names another stream in every host thread, so
that only the caller's thread may queue the copies.  The spectra are those of a model
on the library's own stream, read right behind the run, with no wait in between."""
import numpy as np
import pytest
import torch

from mittet_main_amd import Grid, Model, firstderiv_gauss
from mittet_main_amd.configs import dt_for

pytestmark = pytest.mark.gpu

OM0 = 2 * np.pi
PER_THREAD = 2   # hipStreamPerThread


@pytest.mark.parametrize("kind", ["torch", "per-thread"])
def test_readback_waits_for_the_run_on_the_callers_stream(kind):
    ix, iy, iz = 96, 90, 80       # 63 MiB at two frequencies
    print(f"read-back on the caller's stream: {kind}", flush=True)
    dt, cmax = dt_for(50.0, 45.0, 40.0, sig_min=0.1)
    grid = Grid(ix, iy, iz, 4, 50.0, 45.0, 40.0, dt, OM0, cmax)
    it = 97
    own = torch.cuda.Stream() if kind == "torch" else None
    got = []
    for stream in (None, own.cuda_stream if own else PER_THREAD):
        m = Model(grid, stream=stream)
        m.media_coeff_3d(np.ones(grid.shape))
        s = m.shot(it, firstderiv_gauss(it, dt, 0.2 / dt), (48, 45, 40), 0, None, [1.0, 2.0], 16)
        for _ in range(2):        # the second pass runs on the captured steps
            s.set_zero_eh()
            s.run()
            got.append(s.volume_dft())
        s.close()
        m.close()
    assert np.abs(got[0]).max() > 0
    for g in got[1:]:
        np.testing.assert_array_equal(g, got[0])

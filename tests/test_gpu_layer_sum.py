"""W-stacked images at sizes without a line transform (odd, and a prime factor
above 5): the layer sum over the subgrids' boxes, after griddings of two
observations with different boxes, eager and from a recorded cycle, against
numpy in FP64 (2e-6: about eps log2(N) of an FP32 transform at these sizes)."""
import numpy as np
import pytest

import p9idg
from p9idg import observation

pytestmark = pytest.mark.gpu
TOL = 2e-6


def _swap(a):
    """FFT.Shift: the h x h blocks swap, an odd size's last row and column stay."""
    h = a.shape[0] // 2
    out = a.copy()
    out[:h, :h], out[h:2 * h, h:2 * h] = a[h:2 * h, h:2 * h], a[:h, :h]
    out[:h, h:2 * h], out[h:2 * h, :h] = a[h:2 * h, :h], a[:h, h:2 * h]
    return out


def _check(p):
    layers = p.download_grid(p9idg.GRID_WSTACK).astype(np.complex128).sum(axis=0)
    ref = _swap(np.fft.ifft2(layers, norm="forward").real / float(p.c.VisibilitiesCount))
    got = p.download_image()
    assert np.abs(got - ref).max() <= TOL * np.abs(ref).max()


@pytest.mark.parametrize("G", [161, 182])
def test_wstacked_image_of_two_observations(G):
    wide = observation.custom(G=G, S=16, K=4, L=3, n_ant=6, T=20, C=2, f1=1.02e9, noise=0.2, seed=1)
    narrow = observation.custom(G=G, S=16, K=4, L=3, n_ant=6, T=20, C=2, f1=1.02e9, core_diam=60.0, noise=0.2, seed=2)
    narrow.c = wide.c
    with p9idg.Plan(wide.c) as p:
        for ob in (wide, narrow, wide):
            p.set_observation(ob.uvw, ob.freq, p9idg.Partitioner.CreatePartition(wide.c, ob.uvw, ob.freq))
            p.upload_vis(ob.vis)
            for _ in range(2):
                p.exec_grid(p9idg.GRID_WSTACK)
                p.exec_grid_to_image(p9idg.GRID_WSTACK)
                _check(p)
        p.capture_cycle(p9idg.GRID_WSTACK)
        for _ in range(3):
            p.upload_image(np.random.default_rng(4).standard_normal((G, G)).astype(np.float32))
            p.launch_cycle()
            _check(p)

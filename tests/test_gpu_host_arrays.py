"""Host arrays of complex doubles against the device buffers they come from:
one piece of pinned memory, its edges, more pieces than slots, a rest."""
import numpy as np
import pytest

import p9idg
from p9idg import observation

pytestmark = pytest.mark.gpu


# grids of G^2 values: pieces are 2^16, four of them in flight
@pytest.mark.parametrize("G", [48, 256, 258, 512, 600, 800])
def test_downloaded_doubles_are_the_device_floats(G):
    ob = observation.custom(G=G, S=8, K=2, L=2, n_ant=5, T=6, C=2, f1=1.02e9, core_diam=300.0, noise=0.2, seed=G)
    with p9idg.Plan(ob.c, kernel="fp32") as p:
        p.set_observation(ob.uvw, ob.freq, ob.partition())
        for seed in (1, 2):  # the second pass reuses the pieces
            ob2 = ob.vis * seed
            layers = p.gridw(ob2)
            assert layers.dtype == np.complex128
            assert np.array_equal(layers, p.download_grid(p9idg.GRID_WSTACK).astype(np.complex128))
            vis = p.degridw(layers.sum(axis=0))
            assert np.array_equal(vis, p.download_model_vis().astype(np.complex128))

"""The LDS line transforms between grid and image (csrc/kernels_fft.hip)
against numpy in FP64: every radix (16, 8, 4, 2, 5, 3) and remainder of the
line length, the sizes at the edges of the LDS variants, and a size without a
line transform (library path).

An FP32 transform of N points carries about eps log2(N) of relative rounding:
2e-6 of the largest value covers 2-D sizes up to 4096^2 (24 stages)."""
import numpy as np
import pytest

import p9idg
from p9idg import observation

pytestmark = pytest.mark.gpu
TOL = 2e-6


def _swap(a):
    return np.roll(a, (a.shape[0] // 2, a.shape[1] // 2), (0, 1))


def _plan(G, L):
    ob = observation.custom(G=G, S=8, K=2, L=L, n_ant=5, T=6, C=2, f1=1.02e9, core_diam=3000.0, noise=0.2, seed=G)
    p = p9idg.Plan(ob.c, kernel="fp32")
    p.set_observation(ob.uvw, ob.freq, ob.partition())
    p.upload_vis(ob.vis)
    return p


def _rel(got, ref):
    return np.abs(got - ref).max() / np.abs(ref).max()


# 2^4 6 .. 2^12, with 3s, 5s, a lone 2 before 5s and 3s, and 2 * 5 * 13 (library)
@pytest.mark.parametrize("G", [96, 130, 160, 270, 486, 512, 514, 1000, 1024, 1250, 1458, 2048, 3000, 3072, 4096])
def test_grid_and_image_transforms(G):
    rng = np.random.default_rng(G)
    with _plan(G, 2) as p:
        image = rng.standard_normal((G, G)).astype(np.float32)
        p.upload_image(image)
        p.exec_image_to_grid()
        assert _rel(p.download_model_grid(), np.fft.fft2(_swap(image.astype(np.float64)))) <= TOL
        n = float(p.c.VisibilitiesCount)
        for mode in (p9idg.GRID_WSTACK, p9idg.GRID_WSUM, p9idg.GRID_PLAIN):
            p.exec_grid(mode)
            grid = p.download_grid(mode).astype(np.complex128)
            if mode == p9idg.GRID_WSTACK:
                grid = grid.sum(axis=0)
            ref = _swap(np.fft.ifft2(grid, norm="forward").real / n)
            p.exec_grid_to_image(mode)
            assert _rel(p.download_image(), ref) <= TOL


def test_unknown_contents_use_the_whole_grid():
    """After the buffers were handed out, the grid may hold anything: the
    transform then reads all of it (and the next gridding clears all of it)."""
    G = 160
    with _plan(G, 1) as p:
        p.exec_grid(p9idg.GRID_PLAIN)
        grid = p.download_grid(p9idg.GRID_PLAIN).astype(np.complex128)
        vp = [p9idg._lib._vp() for _ in range(5)]
        p9idg._lib.check(p9idg._lib.idg().p9idg_device_buffers(p._h, *[p9idg._lib.ctypes.byref(v) for v in vp]))
        p.exec_grid_to_image(p9idg.GRID_PLAIN)
        ref = _swap(np.fft.ifft2(grid, norm="forward").real / float(p.c.VisibilitiesCount))
        assert _rel(p.download_image(), ref) <= TOL
        p.exec_grid(p9idg.GRID_PLAIN)
        assert _rel(p.download_grid(p9idg.GRID_PLAIN), grid) <= TOL

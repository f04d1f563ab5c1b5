"""A caller that holds a plan's buffer pointers (p9idg_device_buffers) may write
through them between any two calls: what it added to the grid is imaged, and
nothing of it stays in the next gridding or prediction.

An FP32 transform of N points carries about eps log2(N) of relative rounding:
2e-6 of the largest value covers these sizes; two griddings of the same
visibilities differ by the order of their float atomics (1e-5)."""
import numpy as np
import pytest
import torch

import p9idg
from p9idg import _lib, observation

pytestmark = pytest.mark.gpu
TOL, ORDER = 2e-6, 1e-5


class _Buffer:
    def __init__(self, address, shape):
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<c8", "data": (address, False), "version": 2}


def _plan(G, L=1):
    ob = observation.custom(G=G, S=8, K=2, L=L, n_ant=5, T=6, C=2, f1=1.02e9, core_diam=500.0, noise=0.2, seed=G)
    p = p9idg.Plan(ob.c, kernel="fp32")
    p.set_observation(ob.uvw, ob.freq, ob.partition())
    p.upload_vis(ob.vis)
    return p


def _pointers(p):
    """(grid, model visibilities) as tensors on the plan's buffers."""
    v = [_lib._vp() for _ in range(5)]
    _lib.check(_lib.idg().p9idg_device_buffers(p._h, *[_lib.ctypes.byref(x) for x in v]))
    G = p.c.GridSize
    return (torch.as_tensor(_Buffer(v[1].value, (G, G)), device="cuda"),
            torch.as_tensor(_Buffer(v[3].value, p.shape), device="cuda"))


def _rel(got, ref):
    return np.abs(got - ref).max() / np.abs(ref).max()


def _swap(a):
    """FFT.Shift: the h x h blocks swap, an odd size's last row and column stay."""
    h = a.shape[0] // 2
    out = a.copy()
    out[:h, :h], out[h:2 * h, h:2 * h] = a[h:2 * h, h:2 * h], a[:h, :h]
    out[:h, h:2 * h], out[h:2 * h, :h] = a[h:2 * h, :h], a[:h, h:2 * h]
    return out


def _add(p, grid, rng):
    """The caller's own kernel: noise over the whole grid."""
    p.sync()
    noise = rng.standard_normal(grid.shape + (2,)).astype(np.float32).view(np.complex64)[..., 0]
    grid += 100.0 * torch.from_numpy(noise).cuda()
    torch.cuda.synchronize()


@pytest.mark.parametrize("G", [160, 161])  # line transforms, library
@pytest.mark.parametrize("mode", [p9idg.GRID_PLAIN, p9idg.GRID_WSUM])
def test_image_of_a_grid_that_the_caller_wrote(G, mode):
    rng = np.random.default_rng(G)
    with _plan(G) as p:
        p.exec_grid(mode)
        clean = p.download_grid(mode)
        grid, _ = _pointers(p)
        for _ in range(2):  # held from here on
            p.exec_grid(mode)
            assert _rel(p.download_grid(mode), clean) <= ORDER
            _add(p, grid, rng)
            held = p.download_grid(mode).astype(np.complex128)
            assert np.abs(held - clean).max() > np.abs(clean).max()
            p.exec_grid_to_image(mode)
            ref = _swap(np.fft.ifft2(held, norm="forward").real / float(p.c.VisibilitiesCount))
            assert _rel(p.download_image(), ref) <= TOL


def test_nothing_of_the_callers_stays_after_recorded_work():
    """Replayed cycles and batches clear the buffers themselves; the eager call
    after them clears what the caller wrote since."""
    rng = np.random.default_rng(3)
    with _plan(160) as p:
        p.exec_grid(p9idg.GRID_WSUM)
        clean = p.download_grid(p9idg.GRID_WSUM)
        p.upload_image(rng.standard_normal((160, 160)).astype(np.float32))
        p.exec_image_to_grid()
        p.exec_degrid()
        vis, model = p.download_model_vis(), p.download_model_grid()
        grid, model_vis = _pointers(p)
        p.capture_cycle(p9idg.GRID_WSUM)
        batch = p9idg.Batch([p], p9idg.GRID_WSUM, p9idg.DEGRID_WSTACK)
        for recorded in (p.launch_cycle, lambda: batch.exec(3)):
            recorded()
            _add(p, grid, rng)
            model_vis += 5.0
            torch.cuda.synchronize()
            p.exec_grid(p9idg.GRID_WSUM)
            assert _rel(p.download_grid(p9idg.GRID_WSUM), clean) <= ORDER
            p.upload_model_grid(model)
            p.exec_degrid()
            assert _rel(p.download_model_vis(), vis) <= ORDER
        batch.close()

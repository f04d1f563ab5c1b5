"""The deconvolver's three forms (gradients in LDS; in memory; one workgroup for
everything, with its tile table in LDS and in memory) on the same input: the
picks, x and gradients of the oracle bit for bit.  Which form runs is decided by
what else is on the card, so the launches are called directly."""
import ctypes

import numpy as np
import pytest
import torch

import p9idg
from p9idg import _lib

pytestmark = pytest.mark.gpu

RESIDENT, SHARED, SINGLE = 0, 1, 2


class Shape(ctypes.Structure):
    _fields_ = [("OH", ctypes.c_int), ("OW", ctypes.c_int), ("local", ctypes.c_int)]


def _launch(x, g, amap, psf2, form, lam, alpha, eps, limit):
    """p9idg::cd::launch_descent on the null stream; done, converged, updates, stalled."""
    lib = ctypes.CDLL(_lib.IDG_LIB_PATH)
    H, W = x.shape
    h, w = psf2.shape
    shape = Shape()
    assert getattr(lib, "_ZN5p9idg2cd13descent_shapeEiiiiPNS0_12DescentShapeE")(H, W, h, w, ctypes.byref(shape)) == 0
    slots_of = getattr(lib, "_ZN5p9idg2cd13descent_slotsERKNS0_12DescentShapeE")
    slots_of.restype = ctypes.c_size_t
    tiles_n = max(shape.OH * shape.OW * shape.local, ((H + 31) // 32) * ((W + 31) // 32))
    slots = torch.zeros(slots_of(ctypes.byref(shape)), dtype=torch.int64, device="cuda")
    tiles = torch.zeros(tiles_n, dtype=torch.int64, device="cuda")
    state = torch.zeros(8, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    f = getattr(lib, "_ZN5p9idg2cd14launch_descentEPfS1_PKfS3_iiiiRKNS0_12DescentShapeENS0_11DescentFormEfffiPyS8_PNS0_5StateEP12ihipStream_t")
    ptr, c = ctypes.c_void_p, ctypes.c_float
    assert f(ptr(x.data_ptr()), ptr(g.data_ptr()), ptr(amap.data_ptr()), ptr(psf2.data_ptr()), h, w, H, W, ctypes.byref(shape), form,
             c(lam), c(alpha), c(eps), limit, ptr(slots.data_ptr()), ptr(tiles.data_ptr()), ptr(state.data_ptr()), None) == 0
    torch.cuda.synchronize()
    return state[:4].tolist()


@pytest.mark.parametrize("shape,n", [((320, 320), 32), ((70, 45), 8), ((1060, 1050), 40)])  # 100, 6 and 1122 tiles
@pytest.mark.parametrize("form", [RESIDENT, SHARED, SINGLE])
def test_forms_match_the_oracle(O, shape, n, form):
    rng = np.random.default_rng(n)
    psf = np.exp(-((np.mgrid[0:n, 0:n] - n // 2) ** 2).sum(0) / (2.0 * (n / 6.0) ** 2)).astype(np.float32)
    psf += (0.05 * rng.standard_normal((n, n))).astype(np.float32)
    psf2, amap = p9idg.PSF.CalcPSFSquared(psf), p9idg.PSF.CalcAMap(psf, shape)
    x = np.where(rng.random(shape) < 0.01, rng.random(shape), 0.0).astype(np.float32)
    g = rng.normal(0.0, 1.0, shape).astype(np.float32)
    g[0, 0] = g[-1, -1] = 30.0
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (x, g, amap, psf2)]
    done, converged, updates, stalled = _launch(*dev, form, 0.05, 0.1, 1e-6, 40)
    xr, gr, conv, made = O.cd_deconvolve(amap, psf2, x, g, 0.05, 0.1, 40, 1e-6)
    assert (updates, bool(converged), stalled) == (made, bool(conv), 0) and made > 0
    assert np.array_equal(dev[0].cpu().numpy(), xr) and np.array_equal(dev[1].cpu().numpy(), gr)

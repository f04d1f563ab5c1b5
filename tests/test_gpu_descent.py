"""The deconvolver's one-launch descent (csrc/kernels_cd.hip) against the
oracle, bit for bit: one tile, fewer tiles than workgroups, several window
tiles per workgroup, edge tiles on all sides, images of one row or column, a
tile table beyond LDS, more iterations than one launch makes, and values that
have no best update."""
import numpy as np
import pytest

import p9idg

pytestmark = pytest.mark.gpu


def _psf(n, rng):
    y, x = np.mgrid[0:n, 0:n] - n // 2
    s = max(1.0, n / 6.0)
    p = (np.exp(-(x * x + y * y) / (2.0 * s * s)) + 0.05 * rng.standard_normal((n, n))).astype(np.float32)
    p[n // 2, n // 2] = 1.0
    return p


def _compare(O, shape, n, x, g, lam, alpha, iters, eps):
    rng = np.random.default_rng(n)
    psf = _psf(n, rng)
    psf2 = p9idg.PSF.CalcPSFSquared(psf)
    amap = p9idg.PSF.CalcAMap(psf, shape)
    with p9idg.FastSerialCD(shape, psf) as cd:
        assert cd.GetAbsMaxDiff(x, g, lam, alpha) == O.cd_abs_max_diff(amap, x, g, lam, alpha)
        xg, gg = x.copy(), g.copy()
        res = cd.Deconvolve(xg, gg, lam, alpha, iters, eps)
    xr, gr, conv, made = O.cd_deconvolve(amap, psf2, x, g, lam, alpha, iters, eps)
    assert (res.IterationCount, res.Converged) == (made, conv)
    assert np.array_equal(xg, xr, equal_nan=True) and np.array_equal(gg, gr, equal_nan=True)
    return made, conv


@pytest.mark.parametrize("shape,n,iters", [
    ((1, 1), 1, 3), ((32, 32), 4, 40), ((33, 31), 8, 40), ((16, 700), 10, 60), ((515, 40), 12, 60),
    ((640, 640), 300, 25),       # windows of 600 pixels: two tiles per workgroup and direction
    ((513, 545), 33, 60),        # 17 x 18 tiles on 8 x 8 workgroups
    ((256 * 32 * 39 + 5, 1), 4, 12),  # 40 tiles per workgroup: gradients not in LDS
    ((1, 5000), 3, 30), ((9000, 1), 3, 30),
])
def test_descent_matches_the_oracle(O, shape, n, iters):
    rng = np.random.default_rng(shape[0] * 7 + shape[1])
    x = np.where(rng.random(shape) < 0.01, rng.random(shape), 0.0).astype(np.float32)
    g = rng.normal(0.0, 1.0, shape).astype(np.float32)
    g[0, 0] = g[-1, -1] = 30.0  # windows over two corners
    made, _ = _compare(O, shape, n, x, g, 0.05, 0.1, iters, 1e-6)
    assert made > 0


def test_descent_with_tile_tables_in_memory(O):
    """One column of 8.5 million pixels: more tiles per workgroup than LDS holds."""
    shape = (256 * 32 * 1024 + 4097, 1)
    rng = np.random.default_rng(1)
    g = np.full(shape, -1.0, np.float32)
    g[rng.integers(0, shape[0], 40)] = rng.uniform(5.0, 9.0, (40, 1)).astype(np.float32)
    made, conv = _compare(O, shape, 2, np.zeros(shape, np.float32), g, 0.5, 0.01, 8, 1e-6)
    assert made == 8 and not conv


def test_descent_over_several_launches(O):
    """2^14 iterations per launch; a limit beyond that continues in the next."""
    shape = (130, 130)
    rng = np.random.default_rng(2)
    g = rng.normal(0.0, 5.0, shape).astype(np.float32)
    made, _ = _compare(O, shape, 9, np.zeros(shape, np.float32), g, 1e-4, 0.01, (1 << 14) + 500, 0.0)
    assert made > 1 << 14


@pytest.mark.parametrize("what", ["nothing", "ties", "nan", "inf", "no iterations"])
def test_descent_special_values(O, what):
    shape = (70, 45)
    x = np.zeros(shape, np.float32)
    g = np.full(shape, -1.0, np.float32)
    iters = 20
    if what == "ties":
        g[5:60:9, 3:40:7] = 4.0
    elif what == "nan":
        g[10, 10], g[40, 20], x[3, 3] = np.nan, 6.0, np.nan
    elif what == "inf":
        g[10, 10], g[40, 20], iters = np.inf, 6.0, 1
    elif what == "no iterations":
        g[40, 20], iters = 6.0, 0
    _compare(O, shape, 5, x, g, 0.3, 0.05, iters, 1e-6)

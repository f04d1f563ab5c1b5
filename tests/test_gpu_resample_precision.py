"""Errors of gridding and degridding on time-resampled rows against the FP64
oracle, RMS over RMS, for white visibilities and grids (of a bright source's
coherent sums the roundings are a smaller part).  A resampled row stands for some
ten timesteps, so what the kernels round per row averages out less than on the
rows themselves.

Bounds, u = 2^-24:
  split BF16 gridder: operands in three parts of 8 bits are exact to u, as FP32:
  1e-6 leaves the phasors' and the sums' roundings ten u.  In two parts, with the
  product of the low ones left out, an operand is off by 2.5e-6 (RMS; a part's
  rounding is uniform in +-2^-8 of its binade) and that product by as much, and
  so is a sum of uncorrelated rows.
  split BF16 degridder: two parts each for pixels and phasors with all four
  products, sqrt(2) 2.5e-6 = 3.5e-6; without the low ones' product 4.3e-6.
  FP32 degridder: S roundings in a row's sum and S among the rows, each of 0.6 u
  of a sum that grows with the square root of its terms: 0.6 u sqrt(2 S) = 3e-7 at
  S = 32 and 4e-7 at 64, and the hardware sines and cosines; 7e-7.  In one sum of
  S^2 terms 0.6 u S = 1.1e-6 and 2.3e-6."""
import numpy as np
import pytest

import oracle as O
import p9idg
from p9idg import observation

pytestmark = pytest.mark.gpu


def _rms(got, ref):
    return np.sqrt((np.abs(got - ref) ** 2).sum() / (np.abs(ref) ** 2).sum())


@pytest.mark.parametrize("S,C,kernel,grid_bound,degrid_bound", [
    (24, 8, "mfma_bf16", 1e-6, 3.5e-6),  # channel steps
    (32, 9, "mfma_bf16", 1e-6, 3.5e-6),  # none
    (48, 8, "mfma_bf16", 1e-6, 3.5e-6),
    (64, 8, "mfma_bf16", 1e-6, 3.5e-6),
    (32, 8, "fp32", 1e-6, 7e-7),
    (64, 8, "fp32", 1e-6, 7e-7),
])
def test_errors_on_resampled_rows(S, C, kernel, grid_bound, degrid_bound):
    ob = observation.custom(G=320, S=S, K=4, L=2, n_ant=10, T=760, C=C, f1=1.05e9, noise=0.1, seed=8)
    part = ob.partition()
    rows = part.subgrids["timeSampleCount"].sum()
    assert rows * C >= 1 << 18  # resampled on every kernel
    c = ob.c
    oc = O.make_constants(c.VisibilitiesCount, c.GridSize, c.SubgridSize, c.KernelSize, c.MaxTimestepsPerSubgrid,
                          float(c.ScaleArcSec), c.WLayerCount, c.WStep)
    rng = np.random.default_rng(S)
    white = lambda shape: (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)
    sky, model = white(ob.vis.shape), white((320, 320))
    ref_layers = O.gridw(oc, part.subgrids, sky.astype(np.complex128), ob.uvw, ob.freq)
    ref_vis = O.degridw(oc, part.subgrids, model.astype(np.complex128), ob.uvw, ob.freq)
    with p9idg.Plan(ob.c, kernel=kernel) as plan:
        plan.set_observation(ob.uvw, ob.freq, part)
        layers = plan.gridw(sky)
        plan.upload_model_grid(model)
        plan.exec_degrid()
        vis = plan.download_model_vis()
        batch = p9idg.Batch([plan])
        batch.exec(3)
        batch.sync()
        again = plan.download_grid(p9idg.GRID_WSTACK), plan.download_model_vis()
        batch.close()
    print("%s S %d: %.2e %.2e, batch %.2e %.2e" % (kernel, S, _rms(layers, ref_layers), _rms(vis, ref_vis),
                                                   _rms(again[0], ref_layers), _rms(again[1], ref_vis)))
    for got, ref, bound in ((layers, ref_layers, grid_bound), (vis, ref_vis, degrid_bound), (again[0], ref_layers, grid_bound),
                            (again[1], ref_vis, degrid_bound)):
        assert _rms(got, ref) <= bound

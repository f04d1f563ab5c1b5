"""The gather's two forms and the longest chunk, against the FP64 oracle: from
8192 (chunk, 16 columns) units each of a workgroup's waves has a unit of its own,
with a last workgroup that is not full, a partial last column tile and chunks that
keep their rows; below, four waves share a unit, at chunks of 511 and 512
timesteps and at 513, which are two.

The interpolants are exact to 1e-8 of a unit phasor and everything else rounds in
FP32, so results stay within the parity suite's 1e-5 of the oracle (maximum error
over the maximum value)."""
import numpy as np
import pytest

import oracle as O
import p9idg
from p9idg import observation

pytestmark = pytest.mark.gpu
TOL = 1e-5


def _rel(got, ref):
    return np.abs(got - ref).max() / np.abs(ref).max()


def _check(ob, part, uvw):
    c = ob.c
    oc = O.make_constants(c.VisibilitiesCount, c.GridSize, c.SubgridSize, c.KernelSize, c.MaxTimestepsPerSubgrid,
                          float(c.ScaleArcSec), c.WLayerCount, c.WStep)
    ref = O.gridw(oc, part.subgrids, ob.vis, uvw, ob.freq)
    model = ref.sum(axis=0)
    ref_vis = O.degridw(oc, part.subgrids, model, uvw, ob.freq)
    with p9idg.Plan(c, kernel="fp32") as plan:
        plan.set_observation(uvw, ob.freq, part)
        assert _rel(plan.gridw(ob.vis), ref) <= TOL
        assert not plan.get_launch()["queue"]  # resampled
        plan.upload_model_grid(model.astype(np.complex64))
        plan.exec_degrid()
        assert _rel(plan.download_model_vis(), ref_vis) <= TOL


@pytest.mark.parametrize("C", [17, 24])  # three column tiles, the last of 2 and of 16 columns
@pytest.mark.parametrize("broken", [False, True])
def test_a_unit_per_wave(C, broken):
    T = 40  # not halved: a chunk per subgrid
    ob = observation.custom(G=160, S=8, K=2, L=2, n_ant=91, T=T, C=C, f1=1.01e9, core_diam=600.0, noise=0.1, seed=7)
    part = ob.partition()
    units = 3 * int((part.subgrids["timeSampleCount"] > 0).sum())
    assert units >= 8192 and units % 4 != 0
    uvw = ob.uvw.copy()
    if broken:
        uvw[::3, 20:] += 0.5
    _check(ob, part, uvw)


@pytest.mark.parametrize("T", [511, 512, 513])
def test_the_longest_chunk(T):
    ob = observation.custom(G=640, S=32, K=4, L=2, n_ant=7, T=T, C=2, f1=1.01e9, noise=0.1, seed=6)
    part = ob.partition()
    assert part.subgrids["timeSampleCount"].max() == T and part.subgrids["timeSampleCount"].sum() * 2 >= 1 << 14
    _check(ob, part, ob.uvw)

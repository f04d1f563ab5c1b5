"""Time resampling of the visibilities (csrc/kernels_resample.hip) on the GPU
against the FP64 oracle: chunk lengths around the 16- and 256-timestep edges,
partial column tiles, tracks that must not be resampled, and mixed ones.

The interpolants are exact to 1e-8 of a unit phasor, below the FP32 rounding
of the kernels, so results stay within the parity suite's 1e-5 of the oracle
(maximum error over the maximum value)."""
import numpy as np
import pytest

import oracle as O
import p9idg
from p9idg import observation

pytestmark = pytest.mark.gpu
TOL = 1e-5


def _constants(c):
    return O.make_constants(c.VisibilitiesCount, c.GridSize, c.SubgridSize, c.KernelSize, c.MaxTimestepsPerSubgrid,
                            float(c.ScaleArcSec), c.WLayerCount, c.WStep)


def _rel(got, ref):
    return np.abs(got - ref).max() / np.abs(ref).max()


def _observe(S, T, C, n_ant=10, L=2, kernel_size=4):
    return observation.custom(G=160, S=S, K=kernel_size, L=L, n_ant=n_ant, T=T, C=C, f1=1.05e9, noise=0.1, seed=5)


def _both(ob, part, uvw, kernel):
    """Layers and device-path visibilities of a plan, the oracle's, and the
    visibilities of the call that evaluates every timestep directly."""
    oc = _constants(ob.c)
    ref_layers = O.gridw(oc, part.subgrids, ob.vis, uvw, ob.freq)
    # the model grid comes from the observation's own tracks: finite whatever `uvw` holds
    model = O.gridw(oc, part.subgrids, ob.vis, ob.uvw, ob.freq).sum(axis=0)
    ref_vis = O.degridw(oc, part.subgrids, model, uvw, ob.freq)
    with p9idg.Plan(ob.c, kernel=kernel) as plan:
        plan.set_observation(uvw, ob.freq, part)
        layers = plan.gridw(ob.vis)
        direct = plan.degridw(model)
        plan.upload_model_grid(model)
        plan.exec_degrid()
        vis = plan.download_model_vis()
    return layers, vis, ref_layers, ref_vis, direct


# rows per subgrid: one chunk below, at and above the 16-step granularity, the
# longest chunk, and two and three chunks with remainders
@pytest.mark.parametrize("S,T,C", [(32, 47, 8), (32, 256, 2), (24, 257, 3), (32, 300, 9), (8, 530, 1), (64, 100, 5)])
@pytest.mark.parametrize("kernel", ["fp32", "fp32_sep"])
def test_resampled_rows_match_oracle(S, T, C, kernel):
    ob = _observe(S, T, C, kernel_size=2 if S == 8 else 4)
    part = ob.partition()
    assert part.subgrids["timeSampleCount"].sum() * C >= 1 << 14
    layers, vis, ref_layers, ref_vis, direct = _both(ob, part, ob.uvw, kernel)
    assert _rel(layers, ref_layers) <= TOL
    assert _rel(vis, ref_vis) <= TOL
    assert _rel(direct, ref_vis) <= TOL
    assert not np.array_equal(vis, direct.astype(np.complex64))  # the rows were resampled


# the longest chunk (1024 timesteps) and one more, and a short wavelength whose
# subgrids need more nodes than a whole chunk may have
@pytest.mark.parametrize("S,T,C,f0", [(32, 1024, 2, 1e9), (32, 1050, 2, 1e9), (64, 700, 3, 3e9)])
def test_long_chunks(S, T, C, f0):
    ob = observation.custom(G=640, S=S, K=4, L=2, n_ant=6, T=T, C=C, f0=f0, f1=1.01 * f0, noise=0.1, seed=6)
    layers, vis, ref_layers, ref_vis, direct = _both(ob, ob.partition(), ob.uvw, "fp32")
    assert _rel(layers, ref_layers) <= TOL
    assert _rel(vis, ref_vis) <= TOL
    assert not np.array_equal(vis, direct.astype(np.complex64))


@pytest.mark.parametrize("kernel", ["mfma_bf16", "mfma_fp16"])
def test_resampled_rows_on_the_matrix_kernels(kernel):
    """From 2^18 visibilities the split-precision kernels work on resampled rows."""
    ob = _observe(32, 600, 11, n_ant=10)
    part = ob.partition()
    assert part.subgrids["timeSampleCount"].sum() * 11 >= 1 << 18
    layers, vis, ref_layers, ref_vis, direct = _both(ob, part, ob.uvw, kernel)
    assert _rel(layers, ref_layers) <= TOL
    assert _rel(vis, ref_vis) <= TOL
    assert not np.array_equal(vis, direct.astype(np.complex64))


@pytest.mark.parametrize("what", ["noise", "jump", "nan"])
def test_tracks_that_cannot_be_interpolated_keep_their_rows(what):
    """Noise on every track: nothing is resampled (the device path then gives
    the direct call's values bit for bit); a jump or a missing coordinate on
    some baselines: those keep their rows beside resampled ones."""
    ob = _observe(32, 120, 8)
    part = ob.partition()
    uvw = ob.uvw.copy()
    rng = np.random.default_rng(3)
    if what == "noise":
        uvw += rng.normal(0.0, 1e-2, uvw.shape)
    elif what == "jump":
        uvw[::3, 60:] += 0.5
    else:
        uvw[::3, 50] = np.nan
    layers, vis, ref_layers, ref_vis, direct = _both(ob, part, uvw, "fp32")
    if what == "nan":
        # a NaN coordinate spoils its subgrid's pixels and its own visibilities,
        # nothing else
        assert np.array_equal(np.isnan(vis), np.isnan(direct.astype(np.complex64)))
        ok = ~np.isnan(direct)
        assert np.abs(vis[ok] - direct[ok]).max() <= TOL * np.abs(direct[ok]).max()
        return
    assert _rel(layers, ref_layers) <= TOL
    assert _rel(vis, ref_vis) <= TOL
    assert np.array_equal(vis, direct.astype(np.complex64)) == (what == "noise")


def test_kernel_switch_changes_the_rows_and_the_graph():
    """set_kernel moves a plan between resampled (FP32) and direct rows (split
    precision below 2^18 visibilities); both match the oracle, with the
    ordered adder and after an observation of another size too."""
    with p9idg.Plan(_observe(32, 60, 8).c, kernel="fp32") as plan:
        plan.set_deterministic(True)
        for T in (60, 200, 20):
            ob = _observe(32, T, 8)
            part = ob.partition()
            ref = O.gridw(_constants(ob.c), part.subgrids, ob.vis, ob.uvw, ob.freq)
            plan.set_observation(ob.uvw, ob.freq, part)
            for kernel in ("fp32", "mfma_bf16", "fp32"):
                plan.set_kernel(kernel)
                assert _rel(plan.gridw(ob.vis), ref) <= TOL

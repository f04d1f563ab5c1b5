"""What a plan knows about its grid buffers after work that runs without its
calls: a replayed cycle or a batch, in one mode, between eager gridding and
images in another."""
import numpy as np
import pytest

import p9idg
from p9idg import observation

pytestmark = pytest.mark.gpu
TOL = 2e-6  # FP32 transforms and the float atomics' order, relative to the largest value


def _rel(got, ref):
    return np.abs(got - ref).max() / np.abs(ref).max()


def _image_of(grid, n):
    img = np.fft.ifft2(grid.astype(np.complex128), norm="forward").real / n
    return np.roll(img, (img.shape[0] // 2, img.shape[1] // 2), (0, 1))


@pytest.fixture(scope="module")
def ob():
    return observation.custom(G=160, S=16, K=4, L=3, n_ant=8, T=60, C=4, f1=1.05e9, core_diam=2500.0, noise=0.1, seed=4)


def _plan(ob, kernel="fp32"):
    p = p9idg.Plan(ob.c, kernel=kernel)
    p.set_observation(ob.uvw, ob.freq, ob.partition())
    p.upload_vis(ob.vis)
    return p


# 160: line transforms over the subgrids' box; the cycle's grid keeps its contents
@pytest.mark.parametrize("mode,other", [(p9idg.GRID_WSUM, p9idg.GRID_PLAIN), (p9idg.GRID_WSTACK, p9idg.GRID_PLAIN),
                                        (p9idg.GRID_PLAIN, p9idg.GRID_WSUM)])
def test_cycle_replays_between_other_modes(ob, mode, other):
    n = float(ob.c.VisibilitiesCount)
    with _plan(ob) as p:
        p.exec_grid(other)
        alone = p.download_grid(other)
        model = np.zeros((160, 160), np.float32)
        model[70, 90] = 1.0
        p.upload_image(model)
        p.capture_cycle(mode)
        for _ in range(3):
            p.upload_image(model)
            p.exec_grid(other)
            p.launch_cycle()
            grid = p.download_grid(mode)
            summed = grid.sum(axis=0) if mode == p9idg.GRID_WSTACK else grid
            assert _rel(p.download_image(), _image_of(summed, n)) <= TOL
            # the replayed grid once more, now outside the graph
            p.exec_grid_to_image(mode)
            assert _rel(p.download_image(), _image_of(summed, n)) <= TOL
            p.exec_grid(other)
            assert _rel(p.download_grid(other), alone) <= TOL


def test_batch_replays_between_other_modes(ob):
    small = observation.custom(G=96, S=8, K=2, L=3, n_ant=6, T=40, C=2, f1=1.05e9, core_diam=2500.0, noise=0.1, seed=5)
    obs = [ob, small]
    plans = [_plan(o) for o in obs]
    try:
        alone = []
        for p in plans:
            p.exec_grid(p9idg.GRID_PLAIN)
            plain = p.download_grid(p9idg.GRID_PLAIN)
            p.exec_grid(p9idg.GRID_WSUM)
            p.upload_model_grid(plain)
            p.exec_degrid(p9idg.DEGRID_WSTACK)
            alone.append((plain, p.download_grid(p9idg.GRID_WSUM), p.download_model_vis()))
        with p9idg.Batch(plans, p9idg.GRID_WSUM, p9idg.DEGRID_WSTACK) as batch:
            batch.capture(3)
            for what in ("replay", "replay", "eager"):
                for p in plans:
                    p.exec_grid(p9idg.GRID_PLAIN)
                batch.exec(3) if what == "eager" else batch.launch()
                for p, o, (plain, wsum, vis) in zip(plans, obs, alone):
                    p.exec_grid_to_image(p9idg.GRID_WSUM)
                    assert _rel(p.download_image(), _image_of(wsum, float(o.c.VisibilitiesCount))) <= 2 * TOL
                    assert _rel(p.download_grid(p9idg.GRID_WSUM), wsum) <= TOL
                    assert _rel(p.download_model_vis(), vis) <= TOL
                    p.exec_grid(p9idg.GRID_PLAIN)
                    assert _rel(p.download_grid(p9idg.GRID_PLAIN), plain) <= TOL
    finally:
        for p in plans:
            p.close()

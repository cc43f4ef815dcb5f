"""The learned relaxation's gradient at the edges of its splits: fewer
particles than a 16-row block, odd block counts, a half-filled row tile, more
blocks than partial gradients."""
import numpy as np
import pytest

from nbodysimulation_experiment_amd.scenes import SPHParams, SceneSpec, volume_positions, wall_planes
from nbodysimulation_experiment_amd.sim import ParticleSimulation
from tests.test_gpu_surrogate import DT, GRAVITY, check_frame

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cols", [(7, 4), (16, 4), (17, 5), (48, 8), (65, 9), (2048 * 16 + 5, 181)])
def test_gradient_at_block_edges(n, cols):
    rows = -(-n // cols)
    w, h = 2.0 * (cols // 2 + 6), 2.0 * (rows // 2 + 6)
    pos = volume_positions((0.0, 0.0), cols, rows, 0.5, 1.0, seed=n, limit=n)
    with ParticleSimulation.from_scene(SceneSpec(w, h, 1.0, pos, planes=wall_planes(w, h)), SPHParams(),
                                       GRAVITY) as sim:
        rng = np.random.RandomState(n)
        sim.set_state(pos, rng.normal(0.0, 1.0, pos.shape).astype(np.float32))
        sim.surrogate_init(3)
        sim.surrogate_calibrate(DT)
        check_frame(sim)


@pytest.mark.parametrize("sizes,spacing", [((1,), 0.5), ((33,), 0.5), ((64,), 0.5), ((97, 2, 64, 31), 0.5),
                                           ((700,), 0.12), ((130, 400), 0.12), ((1500,), 0.05)])
def test_inference_and_training_forward_agree(sizes, spacing):
    # the two forms of the head add the same products in the same order: bit-equal states, for partial row
    # tiles, rows of more than 32 candidates and more candidates than the tile holds
    states = []
    for lr in (0.0, 1e-3):
        specs = []
        for k, n in enumerate(sizes):
            cols = int(np.ceil(np.sqrt(n)))
            pos = volume_positions((0.1, 0.2), cols, cols, spacing, 1.0, seed=n + k, limit=n)
            specs.append(SceneSpec(30.0, 24.0, 1.0, pos, planes=wall_planes(30.0, 24.0), circles=[(3.0, 3.0, 1.5)]))
        with ParticleSimulation.from_scenes(specs, SPHParams(k=1e-4, k_near=1e-4), GRAVITY) as sim:
            sim.surrogate_init(7)
            sim.surrogate_calibrate(DT)
            sim.surrogate_set_online_training(lr)
            sim.surrogate_set_mode(True, 1, 1e30)
            sim.Update(DT, 1)
            assert sim.surrogate_report()["fallbacks"] == 0
            states.append(sim.get_state())
    for k in ("x", "v", "density"):
        assert np.array_equal(states[0][k].view(np.uint32), states[1][k].view(np.uint32)), k


@pytest.mark.parametrize("n,spacing", [(65, 0.12), (300, 0.12), (700, 0.06)])
def test_gradient_of_crowded_rows(n, spacing):
    # rows of more than 32 candidates, up to three chunks of them buffered per lane, some lanes without pairs
    cols = int(np.ceil(np.sqrt(n)))
    pos = volume_positions((0.0, 0.0), cols, cols, spacing, 1.0, seed=n, limit=n)
    pos[-5:] += np.array([[4.0, 4.0]], np.float32) * np.arange(1, 6, dtype=np.float32)[:, None] / 2
    with ParticleSimulation.from_scene(SceneSpec(32.0, 32.0, 1.0, pos, planes=wall_planes(32.0, 32.0)),
                                       SPHParams(k=1e-4, k_near=1e-4), GRAVITY) as sim:
        rng = np.random.RandomState(n)
        sim.set_state(pos, rng.normal(0.0, 0.1, pos.shape).astype(np.float32))
        sim.surrogate_init(3)
        sim.surrogate_calibrate(DT)
        check_frame(sim)

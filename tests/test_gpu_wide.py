"""The wide pair kernels (several lanes per particle) and the binning rules,
bit-exact against the oracle at the edges of their choices: groups past the
last particle, both group widths, empty and overfull lists, placement binning
from its smallest step on."""
import numpy as np
import pytest

from nbodysimulation_experiment_amd.scenes import SPHParams, SceneSpec, volume_positions, wall_planes
from tests.helpers import DT, assert_bit_exact, gpu_for, oracle_for

pytestmark = pytest.mark.gpu


def _spec(cols, rows, box, seed=41, limit=None):
    pos = volume_positions((-box / 2 + cols * 0.25, -box / 2 + rows * 0.25), cols, rows, 0.5, 1.0, seed, limit)
    return SceneSpec(box, box, 1.0, pos, planes=wall_planes(box, box), circles=[(0.3 * box, -0.3 * box, 2.0)])


def _check(spec, params, gravity, marks, caps=None):
    sim, ref = gpu_for([spec], params, gravity), oracle_for([spec], params, gravity=gravity)
    if caps is not None:
        sim.set_tuning(autotune=False, tile_cap=caps)
    done = 0
    for m in marks:
        sim.Update(DT, m - done)
        ref.step(DT, m - done)
        done = m
        assert_bit_exact(sim.get_state(), ref.state(), f"step {m}: ")
        for got, want in zip(sim.get_grid(), ref.grid()):
            np.testing.assert_array_equal(got, want)
        st, rs = sim.GetStats(), ref.stats()
        for key in ("minParticleNeighborCount", "maxParticleNeighborCount"):
            assert st[key] == rs[key]
    sim.close()
    ref.close()


@pytest.mark.parametrize("n", [1, 3, 17, 255, 1025, 32768, 32769])
def test_default_kernels_at_group_edges(n):
    cols = int(np.ceil(np.sqrt(n)))
    _check(_spec(cols, cols, 2.0 * (cols // 2 + 4), limit=n), SPHParams(sigma=0.3), (0.0, -9.8), [2, 9])


@pytest.mark.parametrize("side,box", [(70, 40.0), (190, 130.0)])
def test_crowded_lists_with_both_group_widths(side, box):
    # all particles in a tenth of the box: hundreds of pairs each, lists worked off many times
    rng = np.random.RandomState(7)
    pos = rng.uniform(-0.1 * box, 0.1 * box, (side * side, 2)).astype(np.float32)
    pos[: side // 2] = pos[side // 2]  # coincident particles
    pos[side] = (0.0, 0.0)
    spec = SceneSpec(box, box, 1.0, pos, planes=wall_planes(box, box))
    _check(spec, SPHParams(k=0.0005, k_near=0.001), (0.0, -9.8), [1, 4])


@pytest.mark.parametrize("side,box,h", [(20, 24.0, 1.0), (260, 130.0, 1.0), (260, 130.0, 2.0 ** -37)])
def test_coordinates_near_zero_and_far_outside(side, box, h):
    # |x| below 2^-23, and h below 2^-36, take the square root's form for tiny operands (260 x 260: the
    # one-lane-per-particle kernels, from the staged and the global positions);
    # particles outside the grid share its border cells
    pos = volume_positions((0.0, 0.0), side, side, 0.4, 1.0, seed=5)
    pos[:6] = [(0.0, 0.0), (1e-20, -1e-20), (1e-30, 0.2), (1e-7, 1e-9), (400.0, 3.0), (400.2, 3.1)]
    spec = SceneSpec(box, box, 1.0, pos, planes=[])
    _check(spec, SPHParams(h=h, sigma=0.2), (0.0, 0.0), [1, 5])


def test_placement_from_its_smallest_step_on():
    # 640 x 615 = 393,600 particles: placed; far movers (many cells per step) and a crowded cell
    spec = _spec(640, 615, 400.0)
    spec.positions[:3000] = (np.array([100.2, 100.2]) + np.random.RandomState(3).uniform(0, 0.6, (3000, 2))).astype(np.float32)
    _check(spec, SPHParams(k=0.0, k_near=0.0, sigma=0.0, beta=0.0), (0.0, -4000.0), [2, 6], caps=(1024, 1024, 1024))


@pytest.mark.parametrize("cap", [0, 1024])
def test_workgroups_across_scenes_and_past_the_binned_particles(cap):
    # scenes of 1 to 600 particles: 256-slot workgroups within one scene, across several, and partly filled;
    # then particles added past the binned ones
    specs = []
    for s, n in enumerate([1, 2, 600, 255, 257, 3, 512, 31, 64, 400]):
        cols = int(np.ceil(np.sqrt(n)))
        spec = _spec(cols, cols, 2.0 * (cols // 2 + 4), seed=50 + s, limit=n)
        specs.append(spec)
    sim, ref = gpu_for(specs, SPHParams(sigma=0.2), (0.0, -9.8)), oracle_for(specs, SPHParams(sigma=0.2), gravity=(0.0, -9.8))
    sim.set_tuning(autotune=False, tile_cap=(cap,) * 3, wide_max_particles=0)
    for m in (1, 4):
        sim.Update(DT, m)
        ref.step(DT, m)
        assert_bit_exact(sim.get_state(), ref.state(), f"{m}: ")
        for k in range(2):
            sim.AddParticle((0.3 * k, 0.2 * m), scene=2)
            ref.add_particles(2, np.array([[0.3 * k, 0.2 * m]], np.float32))
    sim.close()
    ref.close()


@pytest.mark.parametrize("box", [130.0, 512.0, 1480.0, 2078.0])
def test_cell_starts_of_grids_of_many_scan_workgroups(box):
    # 16,900 to 4.3 million cells: up to 4,217 scan workgroups, whose preceding totals are added eight in flight;
    # particles in the first and last cells and in between
    rng = np.random.RandomState(int(box))
    pos = rng.uniform(-0.5 * box, 0.5 * box, (700, 2)).astype(np.float32)
    pos[0], pos[1] = (-0.5 * box, -0.5 * box), (0.499 * box, 0.4995 * box)
    pos[2:300] = (np.array([0.3 * box, 0.44 * box]) + rng.uniform(0, 3.0, (298, 2))).astype(np.float32)
    _check(SceneSpec(box, box, 1.0, pos, planes=wall_planes(box, box)), SPHParams(), (0.0, -9.8), [1, 3])

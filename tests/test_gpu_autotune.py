"""The autotuner in its own range: 65,537 to 131,072 particles, where the wide
kernels are timed beside the tiles (all five candidates), with periodic
retuning and graph replay between; the choices give identical results."""
import pytest

from nbodysimulation_experiment_amd.scenes import SPHParams, batched_scenes
from tests.helpers import DT, assert_bit_exact, gpu_for, oracle_for

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [False, True])
def test_autotuned_batched_run_in_the_tuned_range(graph):
    specs = batched_scenes(seed=8, count=16, n_min=4096, n_max=8192)
    n = sum(s.n for s in specs)
    assert 65536 < n <= 131072
    sim, ref = gpu_for(specs), oracle_for(specs)
    # a step that builds lists, then two rounds of five candidates; from there every 8 steps two rounds of three
    untuned = (0, 4096, 0)
    sim.set_tuning(autotune=True, retune_interval=8, tile_cap=untuned)
    sim.set_options(hip_graph=graph)
    sim.Update(DT, 1)
    assert tuple(sim.get_tuning()["tile_cap"]) == untuned
    seen = set()  # capacities of the tuning steps, one call per step
    for _ in range(10):
        sim.Update(DT, 1)
        seen.add(tuple(sim.get_tuning()["tile_cap"]))
    assert {(c,) * 3 for c in (0, 1024, 2048, 4096, -1)} <= seen
    ref.step(DT, 11)
    assert_bit_exact(sim.get_state(), ref.state(), "first tuning: ")
    sim.Update(DT, 50)  # three retunings, with replays between when graphs are on
    ref.step(DT, 50)
    assert_bit_exact(sim.get_state(), ref.state(), "retuned: ")
    tuned = sim.get_tuning()["tile_cap"]
    print(f"{n} particles: chosen {tuned}", flush=True)
    assert all(c in (0, 1024, 2048, 4096, -1) for c in tuned)
    sim.close()
    ref.close()

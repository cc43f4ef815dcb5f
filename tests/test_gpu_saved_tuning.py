"""Kernel-shape tuning of small steps: capacities brought as an earlier tuning's
result are used and retuned, and nbs_get_tuning reports what the steps use."""
import pytest

from nbodysimulation_experiment_amd.scenes import SPHParams, SceneSpec, dam_break_4k, volume_positions
from nbodysimulation_experiment_amd.sim import ParticleSimulation
from tests.helpers import DT, GRAVITY, assert_bit_exact

pytestmark = pytest.mark.gpu


def _sim(spec=None):
    return ParticleSimulation.from_scene(spec or dam_break_4k(0), SPHParams(), GRAVITY)


def test_reported_capacities_are_those_used():
    with _sim() as sim:
        sim.set_tuning(autotune=True, tile_cap=(1024, 0, 4096))
        assert sim.get_tuning()["tile_cap"] == [1024, 0, 4096]  # no step yet
        sim.Update(DT, 3)
        t = sim.get_tuning()
        assert t["tile_cap"] == [-1, -1, -1] and t["autotune"]
        sim.set_tuning(tile_cap=t["tile_cap"], retune_interval=4, tuned=True)  # saved and restored
        sim.Update(DT, 20)
        assert sim.get_tuning()["tile_cap"] == [-1, -1, -1]
        sim.set_tuning(autotune=False, tile_cap=(1024, 0, 4096))
        sim.Update(DT, 2)
        assert sim.get_tuning()["tile_cap"] == [1024, 0, 4096]


def test_saved_capacities_are_used():
    with _sim() as sim, _sim() as ref:
        # kept when no retuning is due
        sim.set_tuning(tile_cap=(0, 4096, 1024), retune_interval=0, tuned=True)
        sim.Update(DT, 12)
        ref.Update(DT, 12)
        assert sim.get_tuning()["tile_cap"] == [0, 4096, 1024]
        assert_bit_exact(sim.get_state(), ref.get_state())
        # retuned against their neighbours: 16 workgroups of one lane per particle lose to the wide kernels
        sim.set_tuning(tile_cap=(4096, 4096, 4096), retune_interval=4, tuned=True)
        sim.Update(DT, 24)
        ref.Update(DT, 24)
        assert sim.get_tuning()["tile_cap"] != [4096, 4096, 4096]
        assert_bit_exact(sim.get_state(), ref.get_state())


def test_saved_capacities_below_their_range():
    with _sim(SceneSpec(40.0, 40.0, 1.0, volume_positions((0.0, 0.0), 31, 33, 0.5, 1.0, seed=2), planes=[])) as sim:
        assert sim.GetParticleCount() == 1023
        sim.set_tuning(tile_cap=(1024, 1024, 1024), retune_interval=0, tuned=True)
        sim.Update(DT, 3)
        assert sim.get_tuning()["tile_cap"] == [-1, -1, -1]
        sim.AddParticle((0.0, 0.0))  # from 1,024 on they are used
        sim.Update(DT, 3)
        assert sim.get_tuning()["tile_cap"] == [1024, 1024, 1024]

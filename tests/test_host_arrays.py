"""Arrays that hold a state or a frame on the host: each has memory of its own,
so that keeping one does not hold the others."""
import numpy as np
import pytest

from nbodysimulation_experiment_amd.scenes import SPHParams, dam_break_4k
from nbodysimulation_experiment_amd.sim import ParticleSimulation, _host_arrays


def _assert_own(arrays, rows):
    for k, a in arrays.items():
        assert a.flags.owndata and a.base is None, k
        assert a.flags.c_contiguous and a.flags.writeable and a.shape[0] == rows, k
    names = list(arrays)
    for i, k in enumerate(names):
        for other in names[i + 1:]:
            assert not np.shares_memory(arrays[k], arrays[other]), (k, other)


@pytest.mark.parametrize("n", [0, 1, 4097, 300001])
def test_host_arrays_own_their_memory(n):
    out = _host_arrays({"x": (n, 2, np.float32), "key": (n, 0, np.uint32), "v": (n, 2, np.float32)})
    assert list(out) == ["x", "key", "v"]
    assert out["x"].shape == (n, 2) and out["x"].dtype == np.float32
    assert out["key"].shape == (n,) and out["key"].dtype == np.uint32
    _assert_own(out, n)


@pytest.mark.gpu
def test_state_and_frame_arrays_own_their_memory():
    with ParticleSimulation.from_scene(dam_break_4k(0), SPHParams(), (0.0, -9.8)) as sim:
        sim.Update(0.005, 3)
        n = sim.GetParticleCount()
        state = sim.get_state()
        assert list(state) == ["x", "prev", "v", "density", "pressure", "key", "scene"]
        _assert_own(state, n)
        sim.surrogate_init(3)
        sim.surrogate_calibrate(0.005)
        frame = sim.surrogate_frame(0.005)
        grad, loss = frame.pop("grad"), frame.pop("loss")
        assert set(frame) == {"out", "x", "prev", "density", "target", "scene"}
        _assert_own(frame, n)
        assert isinstance(loss, float) and np.isfinite(grad).all()
        np.testing.assert_array_equal(frame["scene"], 0)

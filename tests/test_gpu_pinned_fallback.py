"""State in and out where the system refuses pinned host memory: the small
transfers then use pageable copies, as the large ones do.  The library runs in
a process of its own, under a hipHostMalloc that always fails."""
import os
import subprocess
import sys

import numpy as np
import pytest

from nbodysimulation_experiment_amd import _lib

pytestmark = pytest.mark.gpu

REFUSE = """
static int calls;
int refused_calls(void) { return calls; }
int hipHostMalloc(void **p, unsigned long bytes, unsigned flags) {
  (void)bytes, (void)flags;
  *p = 0;
  ++calls;
  return 2;  /* hipErrorOutOfMemory */
}
"""

CHILD = """
import ctypes, sys
import numpy as np
refuse = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL) if sys.argv[1] else None
from nbodysimulation_experiment_amd.scenes import SPHParams, dam_break_4k
from nbodysimulation_experiment_amd.sim import ParticleSimulation
sim = ParticleSimulation.from_scene(dam_break_4k(0), SPHParams(), (0.0, -9.8))
n = sim.GetParticleCount()
rng = np.random.RandomState(3)
sim.set_state(sim.get_state()["x"], rng.normal(0.0, 1.0, (n, 2)).astype(np.float32))
sim.Update(0.005, 20)
out = {"state_" + k: v for k, v in sim.get_state().items()}
out["colors"] = sim.get_colors()
sim.surrogate_init(3)
sim.surrogate_calibrate(0.005)
out.update({"frame_" + k: v for k, v in sim.surrogate_frame(0.005).items()})
sim.close()
np.savez(sys.argv[2], refused=refuse.refused_calls() if refuse else 0, **out)
"""


def _run(lib, out):
    env = dict(os.environ, PYTHONPATH=_lib.ROOT)
    subprocess.run([sys.executable, "-c", CHILD, lib, str(out)], check=True, timeout=100, env=env, cwd=_lib.ROOT)
    return np.load(out)


def test_transfers_without_pinned_memory(tmp_path):
    src, lib = tmp_path / "refuse.c", tmp_path / "librefuse.so"
    src.write_text(REFUSE)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src)], check=True)
    want, got = _run("", tmp_path / "want.npz"), _run(str(lib), tmp_path / "got.npz")
    assert want["refused"] == 0 and got["refused"] > 0
    for k in want.files:
        if k != "refused":
            np.testing.assert_array_equal(got[k], want[k], err_msg=k)

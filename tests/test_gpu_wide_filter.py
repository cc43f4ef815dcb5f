"""The wide viscosity kernel lists only the pairs that may approach
((v_i - v_j) . R > 0 up to rounding).  Pairs whose products (v_i - v_j) R are
subnormal, rounded so that their sum is a whole subnormal unit below its true
value, still get the impulse of the reference's own test, u = (v_i - v_j) . n >
0 (sph.h:506-507): bit-exact against the oracle."""
import numpy as np
import pytest

from nbodysimulation_experiment_amd.scenes import SPHParams, SceneSpec, volume_positions
from tests.helpers import DT, assert_bit_exact, gpu_for, oracle_for

pytestmark = pytest.mark.gpu


def _pairs(count):
    """(R, v): a particle at the origin moving at v and one at rest at R.  The
    products v R of x and y are about +-(k + 1/2) units of 2^-149, the first just
    below and the second just above, and round to k and -(k + 1); u, from the
    normalised R, rounds to a positive number.  R is so large against the step
    v dt that the second step still finds R."""
    rng, f = np.random.RandomState(1), np.float32
    n = 100000
    R = (rng.uniform(1, 2, (n, 2)) * 2.0 ** -58).astype(f)
    k = rng.randint(20, 4000, n) + 0.5
    v = (np.stack([k, -k], 1) * 2.0 ** -149 / R.astype(np.float64)).astype(f)
    v1 = (v * f(DT)) * (f(1) / f(DT))  # the velocity after the first step
    prod = v1 * R
    inv = f(1) / np.sqrt(R[:, 0] * R[:, 0] + R[:, 1] * R[:, 1])
    u = v1[:, 0] * (R[:, 0] * inv) + v1[:, 1] * (R[:, 1] * inv)
    hit = np.flatnonzero((prod.sum(1, dtype=f) <= -f(2.0 ** -149)) & (u > 0))[:count]
    assert hit.size == count
    return R[hit], v[hit]


@pytest.mark.parametrize("padding", [0, 33000])  # 16 and 4 lanes per particle
def test_subnormal_products_keep_their_pair(padding):
    R, v = _pairs(12)
    specs = [SceneSpec(8.0, 8.0, 1.0, np.stack([np.zeros(2, np.float32), r]), planes=[]) for r in R]
    vel = np.zeros((2 * len(specs) + padding, 2), np.float32)
    vel[:2 * len(specs):2] = v
    if padding:
        pos = volume_positions((0.0, 0.0), 220, 150, 0.5, 1.0, seed=3)
        specs.append(SceneSpec(140.0, 120.0, 1.0, pos, planes=[]))
    params = SPHParams(k=0.0, k_near=0.0, sigma=1.0e6, beta=0.0)
    sim, ref = gpu_for(specs, params, (0.0, 0.0)), oracle_for(specs, params, gravity=(0.0, 0.0))
    x = sim.get_state()["x"]
    sim.set_state(x, vel)
    ref.set_state(x, vel)
    sim.Update(DT, 1)
    ref.step(DT, 1)
    before = ref.state()["v"].copy()
    sim.Update(DT, 1)
    ref.step(DT, 1)
    want = ref.state()
    assert (want["v"][:2 * len(R):2] != before[:2 * len(R):2]).any(axis=1).all()  # the impulse is visible
    assert_bit_exact(sim.get_state(), want)
    sim.close()
    ref.close()

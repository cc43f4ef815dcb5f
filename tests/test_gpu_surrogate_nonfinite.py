"""The weight gradient where some of the network's values are not finite.

Half of the particles (scene 0) have infinite features, pair sums or messages.
W3 M + b3 adds infinities of both signs or takes zero times infinity: a NaN, of
which [G > 0] is false, so that no gradient flows through these particles.  A
non-finite factor times that zero makes NaN of the gradient entries that it
belongs to: one feature's column of W1, one hidden unit's column of W2 or W3.
The other columns are the gradient of the other half of the particles, which
the oracle computes alone; with n = 2 n_1 the loss scale 1/n is half its 1/n_1,
exactly."""
import numpy as np
import pytest

from nbodysimulation_experiment_amd.scenes import SPHParams, SceneSpec, volume_positions
from nbodysimulation_experiment_amd.sim import ParticleSimulation
from oracle import surrogate_oracle as so
from tests.test_gpu_surrogate import DT, REL_TOL, rel

pytestmark = pytest.mark.gpu

N = 256  # particles per scene: whole 64-particle waves of one kind
K, A = 37, 5  # a hidden unit of the pair layer, and one of the second layer


def _frame(change, velocity=0.0):
    """surrogate_frame of two scenes after change(parameter views): the crowded
    scene 0 and a lattice at 0.6 h; and the oracle's gradient of the lattice."""
    rng = np.random.RandomState(5)
    blob = rng.uniform(-0.2, 0.2, (N, 2)).astype(np.float32)
    lattice = volume_positions((0.0, 0.0), 16, 16, 0.6, 1.0, seed=6)
    with ParticleSimulation.from_scenes([SceneSpec(16.0, 16.0, 1.0, p, planes=[]) for p in (blob, lattice)],
                                        SPHParams(k=1e-3, k_near=1e-3), (0.0, 0.0)) as sim:
        v = np.zeros((2 * N, 2), np.float32)
        v[:N] = rng.uniform(0.5, 1.0, (N, 2)) * rng.choice([-velocity, velocity], (N, 2))
        x = np.concatenate([blob, lattice])
        sim.set_state(x, v)
        sim.surrogate_init(7)
        sim.surrogate_calibrate(DT)
        params = sim.surrogate_params().astype(np.float64)
        change(so.unpack(params))  # views of float64 parameters
        params = params.astype(np.float32)
        sim.surrogate_set_params(params)
        sim.set_state(x, v)
        fr = sim.surrogate_frame(DT)
    assert (fr["scene"][:N] == 0).all() and (fr["scene"][N:] == 1).all()
    _, g, _ = so.loss_and_grad(params, {k: fr[k][N:] for k in ("x", "prev", "density", "target", "scene")}, 1.0, DT)
    assert np.isfinite(fr["out"][N:]).all()
    return fr["grad"], 0.5 * g


def _check_columns(got, want, lo, hi, cols, except_):
    keep = np.setdiff1d(np.arange(cols), except_)
    g, w = got[lo:hi].reshape(-1, cols)[:, keep], want[lo:hi].reshape(-1, cols)[:, keep]
    assert np.isfinite(g).all()
    assert np.abs(w).max() > 0.0 and rel(g, w) < REL_TOL


def test_infinite_features_stay_in_their_columns():
    # velocity differences of scene 0 overflow when scaled; the lattice is at rest
    def change(w):
        w["norm"][0] = 1e37
    got, want = _frame(change, velocity=100.0)
    _check_columns(got, want, so.OFF_W1, so.OFF_W2, so.FEAT, [2, 3])


def test_infinite_pair_sums_stay_in_their_columns():
    # hidden unit K is 3e38 (q - 1/2), q = 1 - r/h: its sum overflows in the crowd and is 0 in the lattice
    def change(w):
        w["W1"][K] = 0.0
        w["W1"][K, 8:10] = -1.5e38, 3e38
    got, want = _frame(change)
    _check_columns(got, want, so.OFF_W2, so.OFF_B2, so.HID, [K])
    _check_columns(got, want, so.OFF_W1, so.OFF_W2, so.FEAT, [])


def test_infinite_messages_stay_in_their_columns():
    # message A is 1e38 H_K, infinite in the crowd and 0 in the lattice, and no output of W3 uses it (0 times infinity)
    def change(w):
        w["W1"][K] = 0.0
        w["W1"][K, 8:10] = -5.0, 10.0
        w["W2"][A] = 0.0
        w["W2"][A, K] = 1e38
        w["W3"][:, A] = 0.0
    got, want = _frame(change)
    _check_columns(got, want, so.OFF_W3, so.OFF_B3, so.HID, [A])
    _check_columns(got, want, so.OFF_W2, so.OFF_B2, so.HID, [])

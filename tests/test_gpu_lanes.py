"""The lane pipeline's last iteration: every lane reaches it at its own time
step and forms its velocities afterwards.  Point counts around the edges of the
lanes' shares, fewer iterations than lanes, both velocity modes, strands in
contact with two colliders.  The step performs the oracle's operations in the
oracle's order, so the results are compared bit for bit."""
import numpy as np
import pytest

import barbu_amd as ba
from tests.test_gpu_parity import run_compare

pytestmark = pytest.mark.gpu

SPHERES = [(0, 0, 0, 1), (0.3, 1.1, 0.0, 0.35)]


@pytest.mark.parametrize("npoints,lanes", [(8, 2), (9, 2), (16, 2), (16, 4), (17, 2), (24, 2), (25, 2), (32, 2), (32, 4),
                                           (33, 2), (47, 2), (49, 4), (63, 4), (64, 2), (64, 4)])
@pytest.mark.parametrize("iterations,dftl", [(1, 0), (2, 1), (5, 0), (8, 1)])
def test_last_iteration(ctx, npoints, lanes, iterations, dftl):
    pos, vel, _ = ba.sphere_groom(517, npoints, radius=1.0, length=0.3, seed=npoints + iterations)
    pos[:, 1:, :3] += np.float32([0.0, -0.05, 0.0])  # towards the colliders
    vel[:, 1:, :3] = np.random.default_rng(npoints).normal(scale=0.5, size=vel[:, 1:, :3].shape)
    params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=1.2, iterations=iterations, velocity_mode=dftl,
                            max_velocity=2.0)
    run_compare(ctx, pos, vel, params, SPHERES, 2, lanes=lanes, label="N=%d G=%d K=%d" % (npoints, lanes, iterations))

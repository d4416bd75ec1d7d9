"""The lane pipeline's last iteration: every lane reaches it at its own time
step and forms its velocities afterwards.  Point counts around the edges of the
lanes' shares, fewer iterations than lanes, both velocity modes, strands in
contact with two colliders.  The step performs the oracle's operations in the
oracle's order, so the results are compared bit for bit."""
import numpy as np
import pytest

import barbu_amd as ba
from oracle import ftl_oracle as orc
from tests.helpers import assert_bitexact, oracle_params_for
from tests.test_gpu_parity import DT, run_compare

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


@pytest.mark.parametrize("npoints,lanes", [(4, 1), (8, 1), (7, 1), (13, 1), (16, 1), (31, 1), (12, 2), (16, 2), (27, 2),
                                           (32, 2), (32, 4), (47, 4), (64, 4), (5, 0), (16, 0), (40, 0), (63, 0)])
def test_hits_of_some_points(ctx, npoints, lanes):
    """Waves in which some lanes' points are hit and others' are not, by four
    overlapping colliders, beside points that are not finite, far away, inside
    a collider's centre or on top of their leader: the points that are not hit
    keep their bits."""
    rng = np.random.default_rng(npoints)
    pos, vel, _ = ba.sphere_groom(203, npoints, radius=1.0, length=0.3, seed=npoints)
    pos[::3, 1:, :3] += np.float32([0.0, -0.1, 0.0])
    pos[5, npoints // 2, 0] = np.nan
    pos[70, npoints - 1, 1] = np.inf
    pos[71, 1, :3] = 1e19
    pos[72, 1, :3] = 0.0
    pos[130, 2, :3] = pos[130, 1, :3]
    vel[:, 1:, :3] = rng.normal(scale=0.5, size=vel[:, 1:, :3].shape)
    vel[130] = 0.0
    spheres = [(0, 0, 0, 1), (0.3, 1.0, 0.0, 0.35), (-0.4, 0.9, 0.1, 0.3), (0.2, 1.05, 0.0, 0.3)]
    params = ba.make_params(force_scale=0.0, damping=0.9, length_scale=1.0, iterations=3)
    g = ba.Groom(ctx, pos, vel)
    g.set_params(params)
    g.set_colliders(np.float32(spheres))
    g.set_lanes(lanes)
    P, V = pos.copy(), vel.copy()
    for k in range(2):
        g.step(DT)
        orc.step_f32(oracle_params_for(params, npoints, DT, spheres=spheres), P, V)
        gp, gv = g.download()
        assert_bitexact(gp, P, "step %d positions" % k)
        assert_bitexact(gv, V, "step %d velocities" % k)
    g.close()

"""Launches on both sides of the state sizes at which the step kernels change
how their loads and stores use the caches (144 and 384 MB of positions and
velocities): the operations and their order stay the oracle's, bit for bit,
and a second step reads back what the first one wrote."""
import numpy as np
import pytest

import barbu_amd as ba
from tests.helpers import assert_bitexact
from tests.test_gpu_parity import DT, _oracle_frame, _rigid, run_compare

pytestmark = pytest.mark.gpu

SPHERES = [(0, 0, 0, 1), (0.3, 1.1, 0.0, 0.35)]


@pytest.mark.parametrize("mb", [144, 384])
@pytest.mark.parametrize("npoints,wind", [(4, 0), (32, 1), (20, 0)])
@pytest.mark.parametrize("above", [0, 1])
def test_single(ctx, mb, npoints, wind, above):
    nstrands = (mb << 20) // (32 * npoints) + above
    pos, vel, _ = ba.sphere_groom(nstrands, npoints, radius=1.0, length=0.3, seed=npoints)
    params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=1.0, iterations=1, wind_amplitude=2.0 * wind,
                            wind_frequency=2.0, wind_seed=5)
    run_compare(ctx, pos, vel, params, SPHERES, 2, label="N=%d %d MB + %d" % (npoints, mb, above))


@pytest.mark.parametrize("mb", [100, 200, 400])
def test_batch(ctx, mb):
    """The whole batch's state decides for all of its kernels."""
    grooms, states = [], []
    params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=1.0, iterations=1)
    for i, n in enumerate((8, 20, 64)):
        pos, vel, roots = ba.sphere_groom((mb << 20) // (3 * 32 * n), n, radius=1.0, length=0.3, seed=i)
        g = ba.Groom(ctx, pos, vel, rest_roots=roots)
        g.set_params(params)
        g.set_root_mode(ba.FTL_ROOT_REST)
        g.set_colliders(np.float32(SPHERES))
        g.set_root_transform(_rigid(0, i))
        grooms.append(g)
        states.append(dict(pos=pos.copy(), vel=vel.copy(), roots=roots, params=params, spheres=np.float32(SPHERES), N=n))
    batch = ba.Batch(ctx, grooms)
    batch.launch([DT] * len(grooms))
    _oracle_frame(states, [DT] * len(grooms), [_rigid(0, i) for i in range(len(grooms))])
    for i, (g, s) in enumerate(zip(grooms, states)):
        p, v = g.download()
        assert_bitexact(p, s["pos"], "groom %d positions" % i)
        assert_bitexact(v, s["vel"], "groom %d velocities" % i)
    batch.close()
    for g in grooms:
        g.close()


@pytest.mark.parametrize("mb", [100, 390])
@pytest.mark.parametrize("npoints,lanes,wind", [(7, 1, 0), (11, 1, 1), (3, 0, 0), (20, 2, 0), (48, 1, 0), (40, 4, 0)])
def test_guarded_classes(ctx, mb, npoints, lanes, wind):
    """Strands that are no whole lines, by the launch classes."""
    nstrands = (mb << 20) // (32 * npoints) + 1
    pos, vel, _ = ba.sphere_groom(nstrands, npoints, radius=1.0, length=0.3, seed=npoints)
    params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=1.0, iterations=1, wind_amplitude=2.0 * wind,
                            wind_frequency=2.0, wind_seed=5)
    run_compare(ctx, pos, vel, params, SPHERES, 1, lanes=lanes, label="N=%d lanes %d %d MB" % (npoints, lanes, mb))

"""Batches of several launch classes and wide forms as one kernel, with every
root mode, unscaled rest lengths read back, and streaming in wind; and the
tiles of a batch by the plan its grooms get.  Bit for bit the oracle's step."""
import numpy as np
import pytest
import torch

import barbu_amd as ba
from barbu_amd import _hip as hipm
from oracle import ftl_oracle as orc
from tests.helpers import assert_bitexact, oracle_params_for
from tests.test_gpu_parity import DT, _rigid

pytestmark = pytest.mark.gpu

SPHERES = [(0, 0, 0, 1), (0.3, 1.1, 0.0, 0.35)]
POINTS = [2, 4, 5, 8, 11, 14, 16, 20, 27, 32, 40, 48, 63, 64]


@pytest.mark.parametrize("scale", [1.0, 1.45])
@pytest.mark.parametrize("wind,dftl", [(0, 0), (1, 1)])
def test_root_modes(ctx, scale, wind, dftl):
    """Model, rest and skinned roots in one batch past the last level."""
    params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=scale, iterations=2, velocity_mode=dftl,
                            max_velocity=2.0, wind_amplitude=2.0 * wind, wind_frequency=2.0, wind_seed=5)
    table = ba.wind_table(params) if wind else None
    grooms, skins, states = [], [], []
    for i, n in enumerate(POINTS * 2):
        mode = (ba.FTL_ROOT_MODEL, ba.FTL_ROOT_REST, ba.FTL_ROOT_SKINNED)[i % 3]
        s = 2500 + 37 * i
        if mode == ba.FTL_ROOT_SKINNED:
            sc = ba.skinned_scene(s, n, ntris=600, nbones=8, seed=i)
            skin = ba.Skin(ctx, sc["rest"], sc["joints"], sc["weights"], sc["tris"], sc["nbones"])
            b = ba.bones(sc, 0.3 * i)
            skin.set_bones(b)
            skin.update()
            skins.append(skin)
            g = ba.Groom(ctx, sc["pos"], sc["vel"])
            g.bind_skin(skin, sc["tri"], sc["bary"])
            verts = orc.skin_f32(b, sc["joints"], sc["weights"], sc["rest"])
            pos, vel, roots = sc["pos"], sc["vel"], orc.bary_roots_f32(sc["tris"], sc["tri"], sc["bary"], verts)
            model, omode = None, ba.FTL_ROOT_REST
        else:
            pos, vel, roots = ba.sphere_groom(s, n, radius=1.0, length=0.3, seed=i)
            g = ba.Groom(ctx, pos, vel, rest_roots=roots)
            g.set_root_mode(mode)
            model, omode = _rigid(0, 0.01 * i), mode
            g.set_root_transform(model)
        g.set_params(params)
        g.set_colliders(np.float32(SPHERES))
        grooms.append(g)
        states.append((pos.copy(), vel.copy(), roots, model, omode))
    batch = ba.Batch(ctx, grooms)
    for _ in range(2):
        batch.launch([DT] * len(grooms))
    for i, (g, (pos, vel, roots, model, omode)) in enumerate(zip(grooms, states)):
        op = oracle_params_for(params, pos.shape[1], DT, spheres=SPHERES, model=model, root_mode=omode, wind=table)
        for _ in range(2):
            orc.step_f32(op, pos, vel, roots if omode else None)
        p, v = g.download()
        assert_bitexact(p, pos, "groom %d (%d points) positions" % (i, pos.shape[1]))
        assert_bitexact(v, vel, "groom %d (%d points) velocities" % (i, pos.shape[1]))
    batch.close()
    for x in grooms + skins:
        x.close()


def test_streaming_in_wind(ctx):
    """A batch above 384 MB in wind: streaming stores, loads by class and form."""
    params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=1.0, iterations=1, wind_amplitude=2.0,
                            wind_frequency=2.0, wind_seed=5)
    table = ba.wind_table(params)
    grooms, states = [], []
    for i, n in enumerate((4, 8, 14, 20, 32, 63)):
        pos, vel, _ = ba.sphere_groom((66 << 20) // (32 * n) + i, n, radius=1.0, length=0.3, seed=i)
        g = ba.Groom(ctx, pos, vel)
        g.set_params(params)
        g.set_colliders(np.float32(SPHERES))
        grooms.append(g)
        states.append((pos, vel))
    ba.batch_step(ctx, grooms, [DT] * len(grooms))
    for i, (g, (pos, vel)) in enumerate(zip(grooms, states)):
        orc.step_f32(oracle_params_for(params, pos.shape[1], DT, spheres=SPHERES, wind=table), pos, vel)
        p, v = g.download()
        assert_bitexact(p, pos, "groom %d positions" % i)
        assert_bitexact(v, vel, "groom %d velocities" % i)
        g.close()


def _lanes_of(level, n):
    """Lanes per strand of an n-point groom in a launch of that level, as the
    library's rule states them."""
    if level == 16:
        return 16 if n > 8 else 8 if n > 4 else 4
    if level == 8:
        return 8 if n > 4 else 4
    return 8 if n > 32 else 4


@pytest.mark.parametrize("strands", [30, 700, 3000])
@pytest.mark.parametrize("points", [(16,), (4, 8, 20), (3, 33, 64, 12)])
def test_tiles_of_the_plan(ctx, strands, points):
    """The workgroups of a small batch are the tiles of its level's forms, those
    of a batch with its lanes set the tiles of their classes."""
    shapes = [(strands + 17 * i, points[i % len(points)]) for i in range(12)]
    ncu = torch.cuda.get_device_properties(0).multi_processor_count
    waves = {lv: sum(-(-s // (64 // _lanes_of(lv, n))) for s, n in shapes) for lv in (16, 8, 4)}
    level = next((lv for lv in (16, 8, 4) if waves[lv] <= (8 if lv == 16 else 16) * ncu), 0)
    assert level  # every shape here is a launch smaller than the chip
    grooms = [ba.Groom(ctx, *ba.sphere_groom(s, n, radius=1.0, length=0.3, seed=i)[:2]) for i, (s, n) in enumerate(shapes)]
    b = ba.Batch(ctx, grooms)
    ntiles, grid = b.info()
    assert grid == waves[level]
    assert ntiles == sum(-(-s // (64 // ctx.lanes_for(n))) for s, n in shapes)
    b.close()
    for g in grooms:
        g.set_lanes(1)
    b = ba.Batch(ctx, grooms)
    # (64 points have an exact class of two lanes and none of one)
    assert b.info() == (sum(-(-s // (32 if n == 64 else 64)) for s, n in shapes),) * 2
    b.close()
    hipm.device_synchronize()
    for g in grooms:
        g.close()

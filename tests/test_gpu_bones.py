"""Bones that change every frame, frames in a row: on one stream they are
uploaded behind the frame before; once a second stream or a batch has used the
skin, by copies that wait.  Bit for bit the oracle's frames in both."""
import numpy as np
import pytest

import barbu_amd as ba
from barbu_amd import _hip as hipm
from oracle import ftl_oracle as orc
from tests.helpers import assert_bitexact, oracle_params_for
from tests.test_gpu_parity import DT
from tests.test_skinning import scene_matrices, scene_normals

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["dq", "lbs"])
@pytest.mark.parametrize("uses", ["default stream", "own stream", "second stream", "batch"])
def test_frames_in_a_row(ctx, mode, uses):
    sc = ba.skinned_scene(4000, 8, ntris=2000, nbones=16, seed=5)
    skin = ba.Skin(ctx, sc["rest"], sc["joints"], sc["weights"], sc["tris"], sc["nbones"])
    if mode == "lbs":
        skin.set_mode(ba.FTL_SKIN_LBS)
    g = ba.Groom(ctx, sc["pos"], sc["vel"])
    g.bind_skin(skin, sc["tri"], sc["bary"])
    params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=1.0)
    g.set_params(params)
    g.set_colliders(np.float32([[0, 0, 0, 1.0]]))
    streams = [None if uses == "default stream" else hipm.Stream() for _ in range(2)]
    P, V = sc["pos"].copy(), sc["vel"].copy()
    for k in range(12):
        second = uses == "second stream" and k >= 5
        if second and k == 5:
            streams[0].synchronize()  # the caller's order between its streams
        st = streams[1] if second else streams[0]
        h = st.h if st else None
        b = scene_matrices(sc, (k + 1) * 0.2) if mode == "lbs" else ba.bones(sc, (k + 1) * float(DT) * 10)
        skin.set_matrices(b) if mode == "lbs" else skin.set_bones(b)
        skin.update(h)
        if uses == "batch" and k == 4:
            ba.batch_step(ctx, [g], [DT], h)
        else:
            g.step(DT, h)
        if mode == "lbs":
            normals = scene_normals(sc["rest"])
            verts, _ = orc.skin_full(ba.FTL_SKIN_LBS, b, sc["joints"], sc["weights"], sc["rest"], normals)
        else:
            verts = orc.skin_f32(b, sc["joints"], sc["weights"], sc["rest"])
        roots = orc.bary_roots_f32(sc["tris"], sc["tri"], sc["bary"], verts)
        op = oracle_params_for(params, 8, DT, spheres=[(0, 0, 0, 1.0)], root_mode=ba.FTL_ROOT_REST)
        orc.step_f32(op, P, V, roots)
    gp, gv = g.download()
    assert_bitexact(gp, P, "positions")
    assert_bitexact(gv, V, "velocities")
    g.close()
    skin.close()

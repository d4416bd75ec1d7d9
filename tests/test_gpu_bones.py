"""Bones that change every frame, frames in a row: on one stream they are
uploaded behind the frame before; once a second stream or a batch has used the
skin, by copies that wait.  Bit for bit the oracle's frames in both."""
import ctypes as C

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


def _frames(ctx):
    """A skinned groom with its skin, a function that makes the bones of frame k
    and steps the oracle `steps` times on them, and the final comparison."""
    sc = ba.skinned_scene(4000, 8, ntris=2000, nbones=16, seed=6)
    skin = ba.Skin(ctx, sc["rest"], sc["joints"], sc["weights"], sc["tris"], sc["nbones"])
    g = ba.Groom(ctx, sc["pos"], sc["vel"])
    g.bind_skin(skin, sc["tri"], sc["bary"])
    params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=1.0)
    g.set_params(params)
    g.set_colliders(np.float32([[0, 0, 0, 1.0]]))
    P, V = sc["pos"].copy(), sc["vel"].copy()

    def bones(k, steps=1):
        b = ba.bones(sc, (k + 1) * float(DT) * 10)
        roots = orc.bary_roots_f32(sc["tris"], sc["tri"], sc["bary"], orc.skin_f32(b, sc["joints"], sc["weights"], sc["rest"]))
        op = oracle_params_for(params, 8, DT, spheres=[(0, 0, 0, 1.0)], root_mode=ba.FTL_ROOT_REST)
        for _ in range(steps):
            orc.step_f32(op, P, V, roots)
        return b

    def finish():
        hipm.device_synchronize()
        gp, gv = g.download()
        assert_bitexact(gp, P, "positions")
        assert_bitexact(gv, V, "velocities")
        g.close()
        skin.close()

    return skin, g, bones, finish


def test_second_stream_only_steps(ctx):
    """Another stream than the updates' steps the grooms (the caller orders the
    two): from then on new bones wait."""
    skin, g, bones, finish = _frames(ctx)
    a, b = hipm.Stream(), hipm.Stream()
    for k in range(8):
        skin.set_bones(bones(k))
        skin.update(a.h)
        if k < 3:
            g.step(DT, a.h)
        else:
            a.synchronize()
            g.step(DT, b.h)
            b.synchronize()
    finish()


def test_captured_frame(ctx):
    """An update and a step recorded into a graph between frames with new bones:
    replays use the bones of the time, later frames the new ones."""
    skin, g, bones, finish = _frames(ctx)
    st, graph, run = hipm.Stream(), C.c_void_p(), C.c_void_p()
    hip = hipm.hip()
    for k in range(4):
        skin.set_bones(bones(k, 1 if k < 3 else 4))
        skin.update(st.h)
        g.step(DT, st.h)
    st.synchronize()
    assert hip.hipStreamBeginCapture(st.h, 1) == 0  # hipStreamCaptureModeThreadLocal
    skin.update(st.h)
    g.step(DT, st.h)
    assert hip.hipStreamEndCapture(st.h, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
    for _ in range(3):
        assert hip.hipGraphLaunch(run, st.h) == 0
    for k in range(4, 9):
        skin.set_bones(bones(k))
        skin.update(st.h)
        g.step(DT, st.h)
    finish()
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0

"""The wide forms (2 to 16 lanes per strand, at most 8 points per lane): small
launches at each level, point counts around the edges of the lanes' shares,
partial tiles, and the ragged point counts of launches that fill the chip.
They perform the oracle's operations in the oracle's order: bit for bit."""
import ctypes as C

import numpy as np
import pytest

import barbu_amd as ba
from barbu_amd import _hip as hipm
from oracle import ftl_oracle as orc
from tests.helpers import assert_bitexact, oracle_params_for
from tests.test_gpu_parity import DT, _oracle_frame, _rigid, run_compare

pytestmark = pytest.mark.gpu

SPHERES = [(0, 0, 0, 1), (0.3, 1.1, 0.0, 0.35)]


def scene(nstrands, npoints, seed):
    pos, vel, roots = ba.sphere_groom(nstrands, npoints, radius=1.0, length=0.3, seed=seed)
    pos[:, 1:, :3] += np.float32([0.0, -0.05, 0.0])  # towards the colliders
    vel[:, 1:, :3] = np.random.default_rng(seed).normal(scale=0.3, size=vel[:, 1:, :3].shape)
    return pos, vel, roots


@pytest.mark.parametrize("npoints", [2, 3, 4, 5, 7, 8, 9, 12, 15, 16, 17, 20, 31, 32, 33, 48, 49, 63, 64])
@pytest.mark.parametrize("nstrands,iterations,dftl,scale,wind", [(1, 8, 0, 1.0, 0), (37, 1, 1, 1.45, 1), (517, 2, 0, 1.45, 1),
                                                                 (2049, 8, 1, 1.0, 0)])
def test_small_launches(ctx, npoints, nstrands, iterations, dftl, scale, wind):
    pos, vel, roots = scene(nstrands, npoints, npoints)
    params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=scale, iterations=iterations, velocity_mode=dftl,
                            max_velocity=2.0, wind_amplitude=2.0 * wind, wind_frequency=2.0, wind_seed=5)
    run_compare(ctx, pos, vel, params, SPHERES, 2, roots=roots, root_mode=ba.FTL_ROOT_REST,
                models=lambda k: _rigid(0, 0.1 * k), label="N=%d S=%d" % (npoints, nstrands))


@pytest.mark.parametrize("nstrands", [8193, 32769, 70001])
@pytest.mark.parametrize("npoints", [3, 4, 5, 6, 8, 10, 12, 13, 16, 20, 24, 27, 29, 32, 40, 47, 56, 64])
def test_levels(ctx, npoints, nstrands):
    """Past the lines between the levels (8,192 and 32,768 strands for the
    longer strands) and between the wide forms and the launch classes."""
    pos, vel, _ = scene(nstrands, npoints, 100 + npoints)
    params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=-1.1 if npoints == 20 else 1.0)
    run_compare(ctx, pos, vel, params, SPHERES, 1, label="N=%d S=%d" % (npoints, nstrands))


@pytest.mark.parametrize("npoints", [12, 13, 14, 15, 17])
@pytest.mark.parametrize("nstrands", [32767, 32769, 70001])
@pytest.mark.parametrize("wind,dftl", [(0, 0), (1, 0), (1, 1)])
def test_launches_of_13_to_15_points(ctx, npoints, nstrands, wind, dftl):
    """On both sides of the last level and of the point counts whose plain step
    keeps its launch class in launches that fill the chip."""
    pos, vel, roots = scene(nstrands, npoints, npoints)
    params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=1.1, iterations=2, velocity_mode=dftl,
                            max_velocity=2.0, wind_amplitude=2.0 * wind, wind_frequency=2.0, wind_seed=5)
    run_compare(ctx, pos, vel, params, SPHERES, 2, roots=roots, root_mode=ba.FTL_ROOT_REST,
                models=lambda k: _rigid(0, 0.1 * k), label="N=%d S=%d" % (npoints, nstrands))


@pytest.mark.parametrize("npoints", [7, 20])
def test_streaming_stores(ctx, npoints):
    """A ragged groom above the state size from which stores are hinted."""
    nstrands = (384 << 20) // (32 * npoints) + 1001
    pos, vel, _ = ba.sphere_groom(nstrands, npoints, radius=1.0, length=0.3, seed=3)
    run_compare(ctx, pos, vel, ba.make_params(force_scale=1.0, damping=0.9, length_scale=1.0), SPHERES, 1,
                label="streaming N=%d" % npoints)


def test_nan_stays_in_its_strand(ctx):
    pos, vel, _ = scene(300, 20, 9)
    g = ba.Groom(ctx, pos, vel)
    g.step(DT)
    assert g.status() is False
    p, v = g.download()
    v[17, 5, 0] = np.nan
    p[40, 19, 1] = np.inf
    g.upload(p, v)
    g.step(DT)
    assert g.status() is True
    p, v = g.download()
    bad = ~np.isfinite(p).all((1, 2))
    assert bad[17] and set(np.nonzero(bad)[0]) <= {17, 40}
    g.close()


@pytest.mark.parametrize("scale", [1, 40, 400])
def test_batch_levels(ctx, scale):
    """The same scene as one launch of the common kernel (small), at the last
    level, and grouped by classes and ragged forms (large)."""
    grooms, states = [], []
    for i, (s, n) in enumerate([(1, 8), (13, 16), (77, 32), (64, 64), (24, 4), (5, 2), (90, 20), (30, 5), (20, 48),
                                (11, 9), (50, 33), (41, 63)]):
        pos, vel, roots = scene(s * scale, n, 200 + i)
        params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=1.0, iterations=4 + i % 5)
        g = ba.Groom(ctx, pos, vel, rest_roots=roots)
        g.set_params(params)
        g.set_root_mode(ba.FTL_ROOT_REST)
        spheres = np.float32(SPHERES)[: 1 + i % 2]
        g.set_colliders(spheres)
        grooms.append(g)
        states.append(dict(pos=pos.copy(), vel=vel.copy(), roots=roots, params=params, spheres=spheres, N=n))
    b = ba.Batch(ctx, grooms)
    for k in range(3):
        models = [_rigid(k, i) for i in range(len(grooms))]
        for g, m in zip(grooms, models):
            g.set_root_transform(m)
        if k < 2:
            b.launch([DT] * len(grooms))
        else:
            ba.batch_step(ctx, grooms, [DT] * len(grooms))
        _oracle_frame(states, [DT] * len(grooms), models)
        for i, (g, s) in enumerate(zip(grooms, states)):
            p, v = g.download()
            assert_bitexact(p, s["pos"], "groom %d frame %d positions" % (i, k))
            assert_bitexact(v, s["vel"], "groom %d frame %d velocities" % (i, k))
    b.close()


@pytest.mark.parametrize("wind,dftl,iterations", [(0, 0, 2), (1, 0, 1), (0, 1, 3)])
def test_mixed_batch(ctx, wind, dftl, iterations):
    """A batch past the last level whose grooms need every class and form: one
    kernel, whichever of them a groom's point count names, partial tiles in
    all.  Stepped as a batch object, at once, and by class."""
    grooms, states = [], []
    params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=1.0, iterations=iterations, velocity_mode=dftl,
                            max_velocity=2.0, wind_amplitude=2.0 * wind, wind_frequency=2.0, wind_seed=5)
    for i, n in enumerate([2, 3, 4, 5, 6, 8, 9, 11, 13, 15, 16, 17, 20, 24, 25, 32, 33, 40, 41, 48, 49, 56, 57, 63, 64]):
        pos, vel, roots = scene(3000 + 37 * i, n, 300 + i)
        g = ba.Groom(ctx, pos, vel, rest_roots=roots)
        g.set_params(params)
        g.set_root_mode(ba.FTL_ROOT_REST)
        g.set_colliders(np.float32(SPHERES))
        g.set_root_transform(_rigid(0, i))
        grooms.append(g)
        states.append((pos.copy(), vel.copy(), roots))
    table = ba.wind_table(params) if wind else None
    b = ba.Batch(ctx, grooms)
    for k in range(3):
        if k == 0:
            b.launch([DT] * len(grooms))
        elif k == 1:
            ba.batch_step(ctx, grooms, [DT] * len(grooms))
        else:  # by class again: some grooms' lanes are set
            for g in grooms[::5]:
                g.set_lanes(1)
            ba.batch_step(ctx, grooms, [DT] * len(grooms))
        for i, (g, (pos, vel, roots)) in enumerate(zip(grooms, states)):
            op = oracle_params_for(params, pos.shape[1], DT, spheres=SPHERES, model=_rigid(0, i),
                                   root_mode=ba.FTL_ROOT_REST, wind=table)
            orc.step_f32(op, pos, vel, roots)
            p, v = g.download()
            assert_bitexact(p, pos, "groom %d step %d positions" % (i, k))
            assert_bitexact(v, vel, "groom %d step %d velocities" % (i, k))
    b.close()
    for g in grooms:
        g.close()


@pytest.mark.parametrize("ngrooms", [63, 64, 65, 129, 4097])
@pytest.mark.parametrize("mixed", [0, 1])
def test_many_spans(ctx, ngrooms, mixed):
    """The search for a tile's groom over one round of 64 spans, two, and three:
    every groom is stepped exactly once."""
    grooms, states = [], []
    params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=1.0, iterations=1)
    big = 70000 if mixed else 3  # past the last level: by class, or the kernel of several
    for i in range(ngrooms):
        s, n = (big, 32) if i == ngrooms // 2 else (1 + (7 * i) % 11, (4, 8, 20)[i % 3])
        pos, vel, roots = scene(s, n, i % 50)
        g = ba.Groom(ctx, pos, vel, rest_roots=roots)
        g.set_params(params)
        g.set_root_mode(ba.FTL_ROOT_REST)
        g.set_colliders(np.float32(SPHERES))
        grooms.append(g)
        states.append(dict(pos=pos.copy(), vel=vel.copy(), roots=roots, params=params, spheres=np.float32(SPHERES), N=n))
    ba.batch_step(ctx, grooms, [DT] * ngrooms)
    _oracle_frame(states, [DT] * ngrooms, [None] * ngrooms)
    for i, (g, s) in enumerate(zip(grooms, states)):
        p, v = g.download()
        assert_bitexact(p, s["pos"], "groom %d positions" % i)
        assert_bitexact(v, s["vel"], "groom %d velocities" % i)
        g.close()


@pytest.mark.parametrize("lanes", [0, 1])
def test_batch_launch_while_capturing(ctx, lanes):
    """A frame launched on a stream that is being captured runs at once and
    leaves nothing in the caller's graph, with one kernel (lanes 0) as with
    several."""
    grooms, states = [], []
    for i, n in enumerate((8, 16)):
        pos, vel, roots = scene(100 + i, n, i)
        params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=1.0)
        g = ba.Groom(ctx, pos, vel, rest_roots=roots)
        g.set_params(params)
        g.set_root_mode(ba.FTL_ROOT_REST)
        g.set_colliders(np.float32(SPHERES))
        g.set_lanes(lanes)
        grooms.append(g)
        states.append(dict(pos=pos.copy(), vel=vel.copy(), roots=roots, params=params, spheres=np.float32(SPHERES), N=n))
    b = ba.Batch(ctx, grooms)
    b.launch([DT] * 2)
    stream, graph, nodes = hipm.Stream(), C.c_void_p(), C.c_size_t(99)
    hipm.device_synchronize()
    assert hipm.hip().hipStreamBeginCapture(stream.h, 1) == 0  # hipStreamCaptureModeThreadLocal
    b.launch([DT] * 2, stream.h)
    assert hipm.hip().hipStreamEndCapture(stream.h, C.byref(graph)) == 0
    assert hipm.hip().hipGraphGetNodes(graph, None, C.byref(nodes)) == 0 and nodes.value == 0
    assert hipm.hip().hipGraphDestroy(graph) == 0
    hipm.device_synchronize()
    b.launch([DT] * 2)
    for _ in range(3):
        _oracle_frame(states, [DT] * 2, [None] * 2)
    for g, s in zip(grooms, states):
        p, v = g.download()
        assert_bitexact(p, s["pos"], "positions")
        assert_bitexact(v, s["vel"], "velocities")
    b.close()
    for g in grooms:
        g.close()


def _queued_batch(ctx, lanes, points, nstrands=6000):
    """Grooms with enough work that frames queue up behind each other; their
    batch, states for the oracle, and a function that launches one frame with
    new root transforms."""
    grooms, states, frames = [], [], []
    for i, n in enumerate(points):
        pos, vel, roots = scene(nstrands + i, n, i)
        params = ba.make_params(force_scale=1.0, damping=0.9, length_scale=1.0, iterations=32)
        g = ba.Groom(ctx, pos, vel, rest_roots=roots)
        g.set_params(params)
        g.set_root_mode(ba.FTL_ROOT_REST)
        g.set_colliders(np.float32(SPHERES))
        g.set_lanes(lanes)
        grooms.append(g)
        states.append(dict(pos=pos.copy(), vel=vel.copy(), roots=roots, params=params, spheres=np.float32(SPHERES), N=n))
    b = ba.Batch(ctx, grooms)

    def frame(stream):
        models = [_rigid(len(frames), i) for i in range(len(grooms))]
        frames.append(models)
        for g, m in zip(grooms, models):
            g.set_root_transform(m)
        b.launch([DT] * len(grooms), stream)

    def finish():
        hipm.device_synchronize()
        for models in frames:
            _oracle_frame(states, [DT] * len(grooms), models)
        for i, (g, s) in enumerate(zip(grooms, states)):
            p, v = g.download()
            assert_bitexact(p, s["pos"], "groom %d positions" % i)
            assert_bitexact(v, s["vel"], "groom %d velocities" % i)
        b.close()
        for g in grooms:
            g.close()

    return frame, finish


@pytest.mark.parametrize("lanes,points", [(0, (16, 32)), (1, (16, 32)), (1, (4, 8, 16, 32))])
@pytest.mark.parametrize("null_stream", [0, 1])
def test_batch_frames_follow_each_other(ctx, lanes, points, null_stream):
    """Frames launched one behind the other without a wait between them: each
    kernel of a frame follows all of the frame before (lanes 1: a kernel per
    class)."""
    frame, finish = _queued_batch(ctx, lanes, points)
    stream = None if null_stream else hipm.Stream().h
    for _ in range(7):
        frame(stream)
    finish()


@pytest.mark.parametrize("lanes", [0, 1])
def test_batch_frames_around_a_capture(ctx, lanes):
    """Frames inside and after a capture, none of them waited for: each one's
    descriptors stay as they are until it has read them.  (The frames in the
    capture come back to a buffer that one of them used.)"""
    frame, finish = _queued_batch(ctx, lanes, (16, 32))
    stream, graph, nodes = hipm.Stream(), C.c_void_p(), C.c_size_t(99)
    frame(None)
    hipm.device_synchronize()
    assert hipm.hip().hipStreamBeginCapture(stream.h, 1) == 0  # hipStreamCaptureModeThreadLocal
    for _ in range(4):
        frame(stream.h)
    assert hipm.hip().hipStreamEndCapture(stream.h, C.byref(graph)) == 0
    assert hipm.hip().hipGraphGetNodes(graph, None, C.byref(nodes)) == 0 and nodes.value == 0
    assert hipm.hip().hipGraphDestroy(graph) == 0
    for _ in range(4):
        frame(stream.h)
    finish()

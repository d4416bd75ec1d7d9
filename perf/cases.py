"""The work a program has this library do, as cases that can be timed and compared.

Four kinds of pass, each through the public entry points:

* "step": one frame of one groom (`Groom.step`), the emitter and the colliders moving;
* "skinned": one frame of a groom whose roots ride a dual-quaternion skinned mesh (`Skin.update` + `Groom.step`);
* "batch": one frame of many uneven grooms (`Batch.launch`);
* "expand": the render-side strand expansion of a groom (`Expand.run`);
* "luts": the two Marschner lookup tables (`ftl_marschner_luts`).

The state of a step lives on the device and is updated in place; a pass returns views of it (the zero-copy buffers a
renderer reads).  Inputs are made on the GPU from the seed with torch; `exact` restates every pass in float64.
"""
import ctypes
import math
import os

import numpy as np
import torch

import barbu_amd as ba

DT = np.float32(1.0 / 60.0)
PERIOD = 240  # frames of the cyclic motion of emitters, colliders and bones (4 s)
GRID = 8      # side of the wind lattice


# --- cases ------------------------------------------------------------------------------------------------------------

def _step(name, strands, points, **kw):
    c = dict(name=name, kind="step", strands=strands, points=points, iterations=8, colliders=1, wind=False, dftl=False,
             root="rest", length_scale=1.0, force_scale=1.0, damping=0.9)
    c.update(kw)
    return c


def listed():
    return [
        # The reference's own demo: one 448-strand groom of 4 control points with the shipped constants, one sphere.
        _step("demo_448x4", 448, 4, root="model", length_scale=1.45, force_scale=20.0, damping=0.8),
        # The small groom of the CPU configuration: one character, one head sphere.
        _step("head_4096x16", 4096, 16, root="model"),
        # Ragged strands (no power of two anywhere), DFTL velocities, wind: an authored groom.
        _step("ragged_60013x20", 60013, 20, wind=True, dftl=True, colliders=2),
        # The most strands of the reference's own length (4 points), in wind: fur.
        _step("fur_1048576x4", 1048576, 4, wind=True, colliders=2),
        # The single large groom of the benchmark: rotating emitter, wind, a head and an orbiting sphere.
        _step("single_262144x32", 262144, 32, wind=True, colliders=2),
        # Long hair at the longest strand, an odd strand count, twice the iterations.
        _step("long_50021x64", 50021, 64, iterations=16, colliders=3),
        # The skinned emitter: 100k triangles, 64 bones, four colliders (half the benchmark's strands).
        dict(name="skinned_2097152x32", kind="skinned", strands=2097152, points=32, tris=100000, bones=64, colliders=4,
             iterations=8),
        # A scene of small creatures standing in the wind: launches and latency count.
        dict(name="crowd_24_small", kind="batch", grooms=24, least=300, most=5000, points="4,8,16,20", wind=True,
             moving=False, iterations=8),
        # The uneven frame of the benchmark (half its grooms): every groom moves, 1 to 3 colliders each.
        dict(name="frame_32_uneven", kind="batch", grooms=32, least=1024, most=262144, points="8,16,32,64", wind=False,
             moving=True, iterations=8),
        # The render-side expansion at the reference's tessellation on the benchmark's scalp.
        dict(name="expand_100k_3x2x16", kind="expand", tris=100000, points=4, instances=3, lines=2, subsegments=16),
        # The same at another setting of the reference's sliders, on longer guides.
        dict(name="expand_20011_4x3x7", kind="expand", tris=20011, points=16, instances=4, lines=3, subsegments=7),
        # The shading tables at the reference's resolution, regenerated when a slider moves.
        dict(name="luts_128", kind="luts", res=128),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("step", "step", "step", "step", "skinned", "batch", "expand", "expand", "luts"))
    if kind == "step":
        points = rng.choice((4, 8, 16, 32, 64, rng.randint(2, 64), rng.randint(2, 64)))
        strands = _log(rng, 200, min(1 << 20, (1 << 24) // points))
        c = _step("", strands, points, iterations=rng.choice((4, 8, 8, 8, 16)), colliders=rng.randint(0, 4),
                  wind=rng.random() < 0.5, dftl=rng.random() < 0.25, root=rng.choice(("model", "rest")),
                  length_scale=rng.choice((1.0, 1.0, 1.45)))
        del c["name"]
        return c
    if kind == "skinned":
        points = rng.choice((4, 8, 16, 32, 64, rng.randint(5, 63)))
        return dict(kind=kind, strands=_log(rng, 2000, (1 << 25) // points), points=points, tris=_log(rng, 2000, 200000),
                    bones=rng.randint(4, 128), colliders=rng.randint(1, 4), iterations=8)
    if kind == "batch":
        return dict(kind=kind, grooms=rng.randint(2, 32), least=rng.randint(200, 2000), most=_log(rng, 4000, 150000),
                    points=rng.choice(("8,16,32,64", "4,8,16,20", "16,32", "12,24,48,64")), wind=rng.random() < 0.5,
                    moving=rng.random() < 0.5, iterations=8)
    if kind == "expand":
        points = rng.choice((4, 4, 8, 16))
        inst, lines, sub = rng.randint(1, 8), rng.randint(1, 4), rng.randint(2, 16)
        most = 50_000_000 // (2 * inst * lines * sub * (points - 1))
        return dict(kind=kind, tris=_log(rng, 500, min(100000, most)), points=points, instances=inst, lines=lines,
                    subsegments=sub)
    return dict(kind=kind, res=rng.randint(40, 512))


# --- inputs -----------------------------------------------------------------------------------------------------------

def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _gen(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(int(seed) % (1 << 62))
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=_dev())


def _sphere_dirs(g, n):
    """n directions on the sphere in patches (neighbours in the array are neighbours on the scalp)."""
    z = 2.0 * _rand(g, n) - 1.0
    a = 2.0 * math.pi * _rand(g, n)
    bands = max(1, int(math.sqrt(n) / 8))
    band = torch.clamp(((z + 1.0) * 0.5 * bands).long(), max=bands - 1)
    order = torch.argsort(band.double() * 8.0 + a.double())
    z, a = z[order], a[order]
    s = torch.sqrt(torch.clamp(1.0 - z * z, min=0.0))
    return torch.stack([s * torch.cos(a), z, s * torch.sin(a)], 1)


def _strands(g, roots, dirs, points, length):
    """Strands from roots, hanging from the scalp's normals `dirs` as combed hair does (those at the crown lie against
    the head): float32 [S, N, 4] positions (w: rest length) and velocities."""
    n = roots.shape[0]
    d = dirs + 0.05 * torch.randn(n, 3, generator=g, device=_dev()) - torch.tensor([0.0, 1.3, 0.0], device=_dev())
    d = d / d.norm(dim=1, keepdim=True)
    seg = (length / (points - 1)) * (1.0 + 0.1 * (1.0 - 2.0 * _rand(g, n)))
    step = d[:, None, :] + 0.1 * torch.randn(n, points, 3, generator=g, device=_dev())
    step = step / step.norm(dim=2, keepdim=True) * seg[:, None, None]
    step[:, 0] = 0.0
    pos = torch.empty(n, points, 4, device=_dev())
    pos[..., :3] = roots[:, None, :] + torch.cumsum(step, 1)
    pos[..., 3] = seg[:, None]
    pos[:, 0, 3] = 0.0
    vel = torch.zeros(n, points, 4, device=_dev())
    vel[..., :3] = 0.01 * torch.randn(n, points, 3, generator=g, device=_dev())
    return pos, vel


def _yaw(angle, shift=(0.0, 0.0, 0.0)):
    c, s = math.cos(angle), math.sin(angle)
    m = np.eye(4)
    m[0, 0], m[0, 2], m[2, 0], m[2, 2] = c, s, -s, c
    m[:3, 3] = shift
    return m.astype(np.float32)


def _spheres(k, count, centre=(0.0, 0.0, 0.0)):
    """The head (r = 1) and up to three spheres orbiting it, at frame k."""
    t = 2.0 * math.pi * k / PERIOD
    s = np.array([[0, 0, 0, 1.0], [1.2 * math.cos(t), 0.0, 1.2 * math.sin(t), 0.3],
                  [-1.2, -0.5 + 0.2 * math.sin(2 * t), 0.3, 0.4], [0.3 * math.sin(t), 1.25, -1.1 * math.cos(t), 0.3]],
                 np.float64)[:count]
    s[:, :3] += np.asarray(centre)
    return np.ascontiguousarray(s, np.float32)


def _params(case, seed):
    kw = dict(force_scale=case.get("force_scale", 1.0), damping=case.get("damping", 0.9),
              length_scale=case.get("length_scale", 1.0), iterations=case["iterations"],
              velocity_mode=1 if case.get("dftl") else 0, max_velocity=100.0)
    if case.get("wind"):
        kw.update(wind_amplitude=2.0, wind_frequency=2.0, wind_scroll=(0.5, 0.0, 0.25), wind_seed=2 + seed % 1000)
    return kw


def _groom_inputs(case, seed):
    g = _gen(seed)
    dirs = _sphere_dirs(g, case["strands"])
    pos, vel = _strands(g, dirs, dirs, case["points"], 0.2)
    roots = torch.cat([dirs, torch.zeros_like(dirs[:, :1])], 1)
    return pos, vel, roots


def _batch_sizes(case):
    pts = [int(p) for p in case["points"].split(",")]
    out = []
    for i in range(case["grooms"]):
        f = (0.5 + i * 0.6180339887498949) % 1.0
        out.append((int(round(case["least"] * (case["most"] / case["least"]) ** f)), pts[(i * 7 + i // 4) % len(pts)]))
    return out


def _batch_groom(case, seed, i, strands, points):
    """Groom i: its state at its place in the scene, its rest roots, its place and its turn per cycle."""
    g = _gen(seed * 1000 + i)
    dirs = _sphere_dirs(g, strands)
    pos, vel = _strands(g, dirs, dirs, points, 0.05 + 0.35 * ((i * 0.37) % 1.0))
    roots = torch.cat([dirs, torch.zeros_like(dirs[:, :1])], 1)
    place = (3.0 * (i % 8), 0.0, 3.0 * (i // 8))
    pos[..., :3] += torch.tensor(place, device=_dev())
    return pos, vel, roots, place, 1 + i % 3


def _mesh(tris):
    """A latitude/longitude sphere of about `tris` triangles: float32 vertices [V, 3] and int32 [T, 3]."""
    m = max(4, int(math.sqrt(tris / 2.0)))
    lat = (np.arange(m + 1) / m * 0.98 + 0.01) * math.pi
    lon = np.arange(m + 1) / m * 2.0 * math.pi
    la, lo = np.meshgrid(lat, lon, indexing="ij")
    v = np.stack([np.sin(la) * np.cos(lo), np.cos(la), np.sin(la) * np.sin(lo)], -1).reshape(-1, 3).astype(np.float32)
    i, j = np.meshgrid(np.arange(m), np.arange(m), indexing="ij")
    a = (i * (m + 1) + j).reshape(-1)
    t = np.concatenate([np.stack([a, a + 1, a + m + 1], 1), np.stack([a + 1, a + m + 2, a + m + 1], 1)], 1)
    return v, np.ascontiguousarray(t.reshape(-1, 3), np.int32)


def _skin_inputs(case, seed):
    rng = np.random.default_rng(seed)
    v, t = _mesh(case["tris"])
    nb = case["bones"]
    centres = rng.normal(size=(nb, 3))
    centres /= np.linalg.norm(centres, axis=1, keepdims=True)
    d = ((v[:, None, :].astype(np.float64) - centres[None]) ** 2).sum(-1)
    joints = np.argpartition(d, 3, axis=1)[:, :4].astype(np.int32)
    w = np.exp(-4.0 * np.take_along_axis(d, joints.astype(np.int64), 1))
    w = (w / w.sum(1, keepdims=True)).astype(np.float32)
    axes = rng.normal(size=(nb, 3))
    axes /= np.linalg.norm(axes, axis=1, keepdims=True)
    phase = rng.uniform(0, 2 * math.pi, nb)
    g = _gen(seed)
    s = case["strands"]
    tri = torch.sort((_rand(g, s) * t.shape[0]).long().clamp(max=t.shape[0] - 1)).values
    b = _rand(g, s, 2)
    b = torch.where(b.sum(1, keepdim=True) > 1.0, 1.0 - b, b).contiguous()
    vt, tt = torch.from_numpy(v).to(_dev()), torch.from_numpy(t).to(_dev()).long()
    corner = vt[tt[tri]]
    roots = corner[:, 0] * (1.0 - b.sum(1, keepdim=True)) + corner[:, 1] * b[:, :1] + corner[:, 2] * b[:, 1:]
    pos, vel = _strands(g, roots, roots / roots.norm(dim=1, keepdim=True), case["points"], 0.2)
    return dict(verts=v, tris=t, joints=joints, weights=w, axes=axes, phase=phase, tri=tri, bary=b, pos=pos, vel=vel)


def _bones(sk, k):
    """Dual quaternions of frame k: rotations of up to 30 degrees and a small shift: float32 [nb, 8]."""
    a = math.radians(30.0) * np.sin(2.0 * math.pi * k / PERIOD + sk["phase"])
    q = np.concatenate([sk["axes"] * np.sin(a / 2)[:, None], np.cos(a / 2)[:, None]], 1)
    t = 0.02 * math.sin(2.0 * math.pi * k / PERIOD) * sk["axes"][:, [1, 2, 0]]
    dv = 0.5 * (t * q[:, 3:] + np.cross(t, q[:, :3]))
    dw = -0.5 * (t * q[:, :3]).sum(1, keepdims=True)
    return np.ascontiguousarray(np.concatenate([q, dv, dw], 1), np.float32)


def _expand_inputs(case, seed):
    v, t = _mesh(case["tris"])
    g = _gen(seed)
    n = torch.from_numpy(v).to(_dev())
    n = n / n.norm(dim=1, keepdim=True)
    pos, _ = _strands(g, n, n, case["points"], 0.2)
    tan = torch.zeros_like(pos)
    x = pos[..., :3]
    tan[:, 1:-1, :3] = 0.5 * (x[:, 2:] - x[:, :-2])
    tan[:, 0, :3], tan[:, -1, :3] = x[:, 1] - x[:, 0], x[:, -1] - x[:, -2]
    rnd = torch.cat([_rand(g, 4096, 2), torch.zeros(4096, 2, device=_dev())], 1)
    return t, pos, tan, rnd


def _lut_params(seed):
    rng = np.random.default_rng(seed)
    return dict(eta=float(np.float32(rng.uniform(1.45, 1.65))), absorption=float(np.float32(rng.uniform(0.1, 0.4))),
                ar=float(np.float32(-rng.uniform(4, 8))), br=float(np.float32(rng.uniform(4, 8))))


# --- what a program keeps ---------------------------------------------------------------------------------------------

_CTX = None


def _ctx():
    """The process's context, with the launch-shape tables the package ships."""
    global _CTX
    if _CTX is None:
        _CTX = ba.Context(0)
        _CTX.autotune(os.path.join(os.path.dirname(os.path.abspath(ba.__file__)), "tuned_gfx950.json"))
    return _CTX


class _View:
    """Zero-copy view of one of a groom's device buffers, which it keeps alive."""

    def __init__(self, groom, ptr, shape):
        self.groom = groom
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<f4", data=(int(ptr), False), version=2,
                                             strides=None)


def _views(g):
    views = []
    for a in g.device_buffers():
        t = torch.as_tensor(_View(g, a, (g.nstrands, g.npoints, 4)), device="cuda")
        t.groom = g  # a view that outlives the state it came from still has its memory
        views.append(t)
    return views


def _groom(pos, vel, roots, params):
    g = ba.Groom(_ctx(), pos.cpu().numpy(), vel.cpu().numpy(), rest_roots=None if roots is None else roots.cpu().numpy())
    g.set_params(params)
    return g


def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind, k=0)
    if kind == "step":
        pos, vel, roots = _groom_inputs(case, seed)
        rest = case["root"] == "rest"
        g = _groom(pos, vel, roots if rest else None, ba.make_params(**_params(case, seed)))
        if rest:
            g.set_root_mode(ba.FTL_ROOT_REST)
        s.update(g=g, out=_views(g), rest=rest, wind=case["wind"])
        s["spheres"] = [_spheres(k, case["colliders"]) for k in range(PERIOD)]
        s["model"] = [_yaw(2.0 * math.pi * (k + 1) / PERIOD) for k in range(PERIOD)]
    elif kind == "skinned":
        sk = _skin_inputs(case, seed)
        one = np.ones((sk["verts"].shape[0], 1), np.float32)
        skin = ba.Skin(_ctx(), np.concatenate([sk["verts"], one], 1), sk["joints"], sk["weights"], sk["tris"],
                       case["bones"])
        g = _groom(sk["pos"], sk["vel"], None, ba.make_params(**_params(case, seed)))
        g.bind_skin(skin, sk["tri"].int().cpu().numpy(), sk["bary"].cpu().numpy())
        s.update(g=g, skin=skin, out=_views(g), bones=[_bones(sk, k + 1) for k in range(PERIOD)])
        s["spheres"] = [_spheres(k, case["colliders"]) for k in range(PERIOD)]
    elif kind == "batch":
        grooms, out, models, spheres = [], [], [], []
        for i, (strands, points) in enumerate(_batch_sizes(case)):
            pos, vel, roots, place, turns = _batch_groom(case, seed, i, strands, points)
            g = _groom(pos, vel, roots, ba.make_params(**_params(case, seed + i)))
            g.set_root_mode(ba.FTL_ROOT_REST)
            m = [np.ascontiguousarray(_yaw(2.0 * math.pi * turns * k / PERIOD, place).T) for k in range(PERIOD)]
            sp = [_spheres(k, 1 + i % 3, place) for k in range(PERIOD)]
            g.set_root_transform(m[0].T)
            g.set_colliders(sp[0])
            grooms.append(g)
            out += _views(g)
            models.append(m)
            spheres.append(sp)
        s.update(grooms=grooms, out=out, batch=ba.Batch(_ctx(), grooms), moving=case["moving"],
                 dt=np.full(len(grooms), DT, np.float32))
        if case["moving"]:  # the addresses of the frames' inputs, ready for the C calls
            s["keep"] = (models, spheres)
            s["frames"] = [[(g.handle, m[k].ctypes.data, sp[k].ctypes.data, sp[k].shape[0])
                            for g, m, sp in zip(grooms, models, spheres)] for k in range(PERIOD)]
    elif kind == "expand":
        tris, pos, tan, rnd = _expand_inputs(case, seed)
        g = ba.Groom(_ctx(), pos.cpu().numpy())
        e = ba.Expand(_ctx(), pos.shape[0], case["points"], tris, tan.cpu().numpy(), rnd.cpu().numpy())
        p = ba.expand_params(case["instances"], case["lines"], case["subsegments"])
        n = e.vertex_count(p)
        s.update(g=g, e=e, p=p, n=n, out=torch.empty(n, 4, device="cuda"), pos=g.device_buffers()[0])
    else:
        res = case["res"]
        p = ba.marschner_params(**_lut_params(seed))
        s.update(ctx=_ctx(), p=p, res=res, out=[torch.empty(res, res, 4, device="cuda") for _ in range(2)])
    return s


# --- one pass ---------------------------------------------------------------------------------------------------------

def run(s):
    kind, k = s["kind"], s["k"] % PERIOD
    s["k"] += 1
    if kind == "step":
        g = s["g"]
        if s["rest"]:
            g.set_root_transform(s["model"][k])
        g.set_colliders(s["spheres"][k])
        if s["wind"]:
            g.set_time(s["k"] * float(DT))
        g.step(DT)
    elif kind == "skinned":
        s["skin"].set_bones(s["bones"][k])
        s["skin"].update()
        s["g"].set_colliders(s["spheres"][k])
        s["g"].step(DT)
    elif kind == "batch":
        if s["moving"]:
            lib = ba.lib()
            for h, m, sp, n in s["frames"][k]:
                lib.ftl_groom_set_root_transform(h, m)
                lib.ftl_groom_set_colliders(h, sp, n)
        s["batch"].launch(s["dt"])
    elif kind == "expand":
        s["e"].run(s["pos"], s["out"].data_ptr(), s["n"], s["p"])
    else:
        ba.check(ba.lib().ftl_marschner_luts(s["ctx"].handle, ctypes.byref(s["p"]), s["res"], s["out"][0].data_ptr(),
                                             s["out"][1].data_ptr(), None), "ftl_marschner_luts")
    return s["out"]


def work(case):
    kind = case["kind"]

    def step(strands, points, ncol, wind):
        cps = strands * points
        return 64.0 * cps + 16.0 * strands, cps * (case["iterations"] * (24.0 + 7.0 * ncol) + 12.0 + (90.0 if wind else 0.0))

    if kind == "step":
        b, f = step(case["strands"], case["points"], case["colliders"], case["wind"])
    elif kind == "skinned":
        b, f = step(case["strands"], case["points"], case["colliders"], False)
        b += 32.0 * case["tris"]
    elif kind == "batch":
        both = [step(n, p, 1 + i % 3, case["wind"]) for i, (n, p) in enumerate(_batch_sizes(case))]
        b, f = sum(x[0] for x in both), sum(x[1] for x in both)
    elif kind == "expand":
        m = max(4, int(math.sqrt(case["tris"] / 2.0)))
        n = 2.0 * case["instances"] * case["lines"] * case["subsegments"] * 2 * m * m * (case["points"] - 1)
        b, f = 16.0 * n + 32.0 * (m + 1) * (m + 1) * case["points"] + 32.0 * m * m, 15.0 * n
    else:
        b, f = 32.0 * case["res"] ** 2, 1500.0 * case["res"] ** 2
    return {"bytes": b, "flops": f}


# --- the same in 64 bits ----------------------------------------------------------------------------------------------

def _wind_lattice(amplitude, seed):
    """The seeded value-noise lattice: [z, y, x, 3] of amplitude * U[-1, 1) from SplitMix64."""
    mask = (1 << 64) - 1
    out = np.zeros(GRID ** 3 * 3)
    for i in range(GRID ** 3):
        for c in range(3):
            z = (seed * 0x632be59bd9b4e019 + 4 * i + c + 0x9e3779b97f4a7c15) & mask
            z = ((z ^ (z >> 30)) * 0xbf58476d1ce4e5b9) & mask
            z = ((z ^ (z >> 27)) * 0x94d049bb133111eb) & mask
            z ^= z >> 31
            out[3 * i + c] = amplitude * (2.0 * ((z >> 40) * 2.0 ** -24) - 1.0)
    return torch.from_numpy(out.reshape(GRID, GRID, GRID, 3)).to(_dev())


def _wind64(x, lattice, freq, offset):
    u = x * freq + torch.tensor(offset, dtype=torch.float64, device=x.device)
    fl = torch.floor(u)
    f = u - fl
    s = f * f * (3.0 - 2.0 * f)
    i = fl.long()
    out = 0.0
    for dz in (0, 1):
        for dy in (0, 1):
            for dx in (0, 1):
                w = (s[..., 0] if dx else 1 - s[..., 0]) * (s[..., 1] if dy else 1 - s[..., 1]) * \
                    (s[..., 2] if dz else 1 - s[..., 2])
                v = lattice[(i[..., 2] + dz) % GRID, (i[..., 1] + dy) % GRID, (i[..., 0] + dx) % GRID]
                out = out + w[..., None] * v
    return out


def _step64(pos, vel, roots0, kw, spheres, time):
    """One step in float64: pos, vel float32 [S, N, 4], roots0 float64 [S, 3] the strands' new roots."""
    f64 = torch.float64
    dt = float(DT)
    x = pos[..., :3].to(f64).transpose(0, 1).contiguous()
    rest = pos[..., 3].to(f64).t().contiguous() * float(np.float32(kw["length_scale"]))
    points = x.shape[0]
    force = torch.tensor([0.0, -float(np.float32(9.81)) * float(np.float32(kw["force_scale"])), 0.0], dtype=f64,
                         device=x.device)
    p = x + dt * vel[..., :3].to(f64).transpose(0, 1)
    if "wind_amplitude" in kw:
        lat = _wind_lattice(kw["wind_amplitude"], kw["wind_seed"])
        off = [float(np.float32(c * time)) for c in kw["wind_scroll"]]
        for i in range(points):
            p[i] += dt * dt * (force + _wind64(x[i], lat, kw["wind_frequency"], off))
    else:
        p += dt * dt * force
    p[0] = roots0
    sph = [[float(c) for c in s] for s in spheres]
    u = torch.zeros_like(p)
    for it in range(kw["iterations"]):
        last = it == kw["iterations"] - 1
        corr = torch.zeros_like(p) if last else None
        for j in range(1, points):
            d = p[j] - p[j - 1]
            new = p[j - 1] + d * (rest[j] / d.norm(dim=1))[:, None]
            if last:
                corr[j] = new - p[j]
            p[j] = new
        if last:
            u[1:-1] = float(np.float32(kw["damping"])) * corr[2:]
            u[-1] = corr[-1]
        for cx, cy, cz, r in sph:
            c = torch.tensor([cx, cy, cz], dtype=f64, device=x.device)
            w = p[1:] - c
            dist = w.norm(dim=2, keepdim=True)
            n = w / dist
            hit = dist < r
            p[1:] = torch.where(hit, c + r * n, p[1:])
            if last:
                u[1:] = torch.where(hit, u[1:] - 2.0 * (n * u[1:]).sum(2, keepdim=True) * n, u[1:])
    u[0] = p[0] - x[0]
    if kw["velocity_mode"] == 1:
        v = (p - x - u) / dt
        size = v.norm(dim=2, keepdim=True)
        u = torch.where(size > kw["max_velocity"], v * (kw["max_velocity"] / size), v)
    p, u = p.transpose(0, 1), u.transpose(0, 1)
    return [torch.cat([p, pos[..., 3:].to(f64)], 2), torch.cat([u, torch.zeros_like(u[..., :1])], 2)]


def _transform64(m, x):
    m = torch.from_numpy(m.astype(np.float64)).to(x.device)
    return x.to(torch.float64) @ m[:3, :3].t() + m[:3, 3]


def _skin64(sk, k):
    """Dual-quaternion blending of the mesh's vertices at frame k."""
    dq = _bones(sk, k).astype(np.float64)[sk["joints"]]
    w = sk["weights"].astype(np.float64)
    w[:, 3] = 1.0 - w[:, :3].sum(1)
    side = np.sign((dq[:, :, :4] * dq[:, 3:, :4]).sum(2))
    side[:, 3] = 1.0
    b = (dq * (w * side)[:, :, None]).sum(1)
    b /= np.linalg.norm(b[:, :4], axis=1, keepdims=True)
    a, aw, d, dw = b[:, :3], b[:, 3:4], b[:, 4:7], b[:, 7:8]
    v = sk["verts"].astype(np.float64)
    out = v + 2.0 * np.cross(a, np.cross(a, v) + aw * v) + 2.0 * (aw * d - dw * a + np.cross(a, d))
    return np.where(sk["weights"][:, :1] <= np.float32(1e-6), v, out)


def _expand64(case, seed):
    tris, pos, tan, rnd = _expand_inputs(case, seed)
    f64 = torch.float64
    tri = torch.from_numpy(tris).to(_dev()).long()
    n, ns = case["subsegments"], case["points"] - 1
    e = torch.arange(2 * n, device=_dev())
    u = ((e // 2 + e % 2).to(f64) / n)[None, None, :, None]
    P, T = pos[..., :3].to(f64), tan[..., :3].to(f64)
    guides = []
    for c in range(3):
        p, t = P[tri[:, c]], T[tri[:, c]]
        p0, p1, t0, t1 = (y[:, :, None, :] for y in (p[:, :-1], p[:, 1:], t[:, :-1], t[:, 1:]))
        guides.append((2 * u ** 3 - 3 * u ** 2 + 1) * p0 + (3 * u ** 2 - 2 * u ** 3) * p1 +
                      (u ** 3 - 2 * u ** 2 + u) * t0 + (u ** 3 - u ** 2) * t1)
    x = torch.arange(ns, device=_dev()).to(f64)[None, :, None] / case["points"] + u[..., 0] / case["points"]
    x = x.clamp(0, 1)
    rel = (x ** 3 * (10.0 + x * (6.0 * x - 15.0))).expand(tri.shape[0], ns, 2 * n)
    out = torch.empty(case["instances"], tri.shape[0], ns, case["lines"], 2 * n, 4, dtype=f64, device=_dev())
    table = rnd.double().cpu().numpy()
    for i in range(case["instances"]):
        for line in range(case["lines"]):
            at = int(np.float32(np.float32(line) / np.float32(case["lines"])) * np.float32(40.0) + np.float32(i)) % 4096
            sx, sy = table[at, 0], table[at, 1]
            if np.float32(sx) + np.float32(sy) > 1.0:
                sx = 1.0 - max(sx, sy)
            out[i, :, :, line, :, :3] = sx * guides[0] + sy * guides[1] + (1.0 - (sx + sy)) * guides[2]
            out[i, :, :, line, :, 3] = rel
    return out.reshape(-1, 4)


def _longitudinal64(case, seed):
    """The M table: three gaussians of the half angle in degrees and the cosine of the difference angle."""
    p, res = _lut_params(seed), case["res"]
    s = np.clip(2.0 * np.arange(res) / res - 1.0, -1.0, 1.0)
    ti, tr = np.arcsin(s)[None, :], np.arcsin(s)[:, None]
    h = np.degrees((ti + tr) / 2.0)
    out = np.empty((res, res, 4))
    for c, (width, shift) in enumerate(((1.0, 1.0), (0.5, -0.5), (2.0, -1.5))):
        w = width * p["br"]
        out[..., c] = np.exp(-(h - shift * p["ar"]) ** 2 / (2.0 * w * w)) / (2.5066282 * abs(w))
    out[..., 3] = np.cos((ti - tr) / 2.0)
    return out


def exact(case, seed):
    """What run() returns for a new state, in float64.  The shipped velocity is the last iteration's correction: unless
    two colliders pull a strand between them, the chain has settled by then and the correction is the rounding of the
    type it is computed in, so it has no value in 64 bits."""
    kind = case["kind"]

    def moved(out, colliders):
        return out if colliders > 1 or case.get("dftl") else [out[0], None]

    if kind == "step":
        pos, vel, roots = _groom_inputs(case, seed)
        root = _transform64(_yaw(2.0 * math.pi / PERIOD), roots[:, :3]) if case["root"] == "rest" else \
            pos[:, 0, :3].to(torch.float64)
        return moved(_step64(pos, vel, root, _params(case, seed), _spheres(0, case["colliders"]), float(DT)),
                     case["colliders"])
    if kind == "skinned":
        sk = _skin_inputs(case, seed)
        v = torch.from_numpy(_skin64(sk, 1)).to(_dev())
        corner = v[torch.from_numpy(sk["tris"]).to(_dev()).long()[sk["tri"]]]
        b = sk["bary"].to(torch.float64)
        root = corner[:, 0] * (1.0 - b.sum(1, keepdim=True)) + corner[:, 1] * b[:, :1] + corner[:, 2] * b[:, 1:]
        del corner
        return moved(_step64(sk["pos"], sk["vel"], root, _params(case, seed), _spheres(0, case["colliders"]), 0.0),
                     case["colliders"])
    if kind == "batch":
        out = []
        for i, (strands, points) in enumerate(_batch_sizes(case)):
            pos, vel, roots, place, turns = _batch_groom(case, seed, i, strands, points)
            out += moved(_step64(pos, vel, _transform64(_yaw(0.0, place), roots[:, :3]), _params(case, seed + i),
                                 _spheres(0, 1 + i % 3, place), 0.0), 1 + i % 3)
        return out
    if kind == "expand":
        return _expand64(case, seed)
    # The azimuthal table branches on discriminants and saturates: it has no value in 64 bits to compare with.
    return [_longitudinal64(case, seed), None]

"""The work that programs give this framework, as cases that can be timed and compared.

  listed()            the cases
  draw(rng)           one more case of the same ranges
  prepare(case, seed) what a program holds before the call (scene, camera, buffers), from the seed
  run(state)          one pass through the public entry points, and its outputs
  work(case)          the bytes and operations that a pass cannot do without
  exact(case, seed)   the outputs in 64 bits, where they have such a value

Scenes are the sphere scenes of the "one weekend" recipe (a ground sphere, a
grid of small diffuse, metal and glass spheres, three big ones) at the
tessellation levels that the reference's batch program, the tests and the
benchmark use, from another recipe seed and another point of view for each
seed.  The closest-hit queries of the "rays" kind over a few spheres made here
have outputs that plain FP64 arithmetic can check.
"""
import ctypes
import math
import random

import numpy as np
import torch

import rtxplay_amd as rtx
from rtxplay_amd.diff import DiffRender, material_params
from rtxplay_amd.scene import RTOWScene, sphere_things

DEV = "cuda"


def listed():
    return [
        # a click in the viewer: which thing is under the cursor (one ray, the smallest call)
        dict(name="pick", kind="pick", level=6, two_level=False, w=1280, h=720),
        # visibility queries of a program that keeps its rays on the host: a few
        # thousand rays through Scene.trace, over a scene of 40 meshes
        dict(name="rays_host_4k", kind="rays", things=40, sub=3, two_level=False, n=4096),
        # a preview of the scene at the size of the reference's CPU tracer
        dict(name="preview_400x225", kind="frame", level=4, two_level=False, w=400, h=225, spp=10, depth=16,
             iterative=False, srgb=True),
        # the viewer's frame: one sample per pixel and the sRGB image, per camera move
        dict(name="viewer_720p_1spp", kind="frame", level=6, two_level=False, w=1280, h=720, spp=1, depth=16,
             iterative=False, srgb=True),
        # an edit in the viewer: some things moved, the structure brought up to date
        # (the reference's two-level layout, its own tessellation levels), a frame
        dict(name="edit_mixed_720p", kind="edit", level="mixed", two_level=True, w=1280, h=720, spp=1, depth=16,
             moved=48),
        # closest hits of a ray buffer that stays on the GPU: camera rays and the
        # incoherent rays that leave the surfaces, 2 M in all, over 8 M triangles
        dict(name="trace_2m", kind="trace", level=6, two_level=False, n=2073600),
        # the acceleration structure of the full scene, and a first query of it
        dict(name="build_level6", kind="build", level=6, two_level=False, n=65536),
        # one step of the material optimisation: render, image loss, gradients of
        # every albedo and fuzz
        dict(name="train_640x360", kind="train", level=4, two_level=False, w=640, h=360, spp=64, depth=8),
        # an ordinary frame: half a million triangles, 720p, 50 samples
        dict(name="frame_720p_50spp", kind="frame", level=4, two_level=False, w=1280, h=720, spp=50, depth=16,
             iterative=False, srgb=False),
        # the reference's own scene and layout (mixed levels, instanced meshes) under
        # its default program set
        dict(name="frame_mixed_1080p", kind="frame", level="mixed", two_level=True, w=1920, h=1080, spp=64, depth=16,
             iterative=True, srgb=False),
        # a queue of uneven frames, each with its own scene, in one launch
        dict(name="batch_16", kind="batch", frames=16, mix=1, spp_hi=64, two_level=False),
        # the headline frame: 8 M triangles, 1080p, 500 samples
        dict(name="frame_1080p_500spp", kind="frame", level=6, two_level=False, w=1920, h=1080, spp=500, depth=16,
             iterative=False, srgb=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "frame", "trace", "trace", "rays", "train", "build", "edit", "batch",
                       "pick"])
    two = rng.random() < 0.35
    level = rng.choice([2, 3, 4, 5, 6, "mixed"])
    w = _log(rng, 65, 1920)
    h = max(33, min(1080, int(round(w * rng.uniform(0.45, 1.0)))))
    if kind == "frame":
        spp = max(1, min(_log(rng, 1, 300), int(2.5e8 / (w * h))))
        return dict(kind=kind, level=level, two_level=two, w=w, h=h, spp=spp, depth=rng.randint(2, 50),
                    iterative=rng.random() < 0.5, srgb=rng.random() < 0.5)
    if kind == "trace":
        return dict(kind=kind, level=level, two_level=two, n=_log(rng, 1000, 4000000))
    if kind == "rays":
        return dict(kind=kind, things=_log(rng, 1, 60), sub=rng.randint(1, 3), two_level=two, n=_log(rng, 1, 6000))
    if kind == "train":
        w, h = max(64, w // 3), max(33, h // 3)
        return dict(kind=kind, level=rng.choice([2, 3, 4, 5]), two_level=two, w=w, h=h, spp=_log(rng, 4, 64),
                    depth=rng.randint(2, 16))
    if kind == "build":
        return dict(kind=kind, level=level, two_level=two, n=_log(rng, 100, 65536))
    if kind == "edit":
        return dict(kind=kind, level=rng.choice([2, 3, 4, 5, "mixed"]), two_level=rng.random() < 0.7, w=w, h=h,
                    spp=rng.randint(1, 4), depth=rng.randint(4, 16), moved=_log(rng, 1, 200))
    if kind == "batch":
        return dict(kind=kind, frames=rng.randint(2, 12), mix=rng.randrange(1000), spp_hi=_log(rng, 8, 64), two_level=two)
    return dict(kind="pick", level=level, two_level=two, w=w, h=h)


# ---------------------------------------------------------------------------
# what a program holds
# ---------------------------------------------------------------------------
def _ok(status):
    if status:
        raise RuntimeError(rtx.lib().rtx_last_error().decode())


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _camera(rng, aspect):
    """A point of view on the recipe's radius-13 ring, looking at the centre."""
    a = rng.uniform(0.0, 2.0 * math.pi)
    eye = (13.0 * math.cos(a), rng.uniform(1.0, 4.0), 13.0 * math.sin(a))
    return rtx.Camera().set(eye, (0., 0., 0.), (0., 1., 0.), 20.0, aspect, 0.1, 10.0)


def _scene(rng, level, two_level, half=11, build=True):
    spec = sphere_things(rng.randrange(1 << 30), half)
    # the recipe leaves out the few small spheres that meet a big one, other
    # ones for each seed: keep a number that every seed has
    spec = spec[:1 + (2 * half) ** 2 - 12] + spec[-3:]
    s = RTOWScene(level=level, spec=spec, two_level=two_level)
    s.load()
    if build:
        s.build()
    return s


def _frame(rng, scene, w, h, spp, depth, guides=True):
    """Launch parameters and the buffers they point at."""
    lp = rtx.LpGeneral()
    lp.image_w, lp.image_h, lp.spp, lp.depth, lp.is_handle = w, h, spp, depth, scene.handle
    lp.camera = _camera(rng, w / h).c
    out = {"rawRGB": torch.zeros((h, w, 3), dtype=torch.float32, device=DEV),
           "rpp": torch.zeros((h, w), dtype=torch.int32, device=DEV)}
    if guides:
        out["normals"] = torch.zeros((h, w, 3), dtype=torch.float32, device=DEV)
        out["albedos"] = torch.zeros((h, w, 3), dtype=torch.float32, device=DEV)
    for k, t in out.items():
        setattr(lp, k, t.data_ptr())
    return lp, out


def _launch(scene, lp, once=0):
    _ok(rtx.lib().rtx_launch(scene.ctx, ctypes.byref(lp), once, _stream()))


def _hits_of(t):
    """The fields of an rtx_hit buffer (8 words each)."""
    f = t.view(torch.float32)
    return {"t": f[:, 0], "uv": f[:, 1:3], "ids": t[:, 3:6]}


def _view_rays(rng, n):
    """n rays float32[n, 8]: half of them camera rays of one point of view in
    image order, half of them rays that leave the ground and the spheres'
    heights in all directions, as scattered light does."""
    g = np.random.RandomState(rng.randrange(1 << 30))
    c = _camera(rng, 16 / 9).c
    nc = (n + 1) // 2
    wd = max(1, int(math.sqrt(nc * 16 / 9)))
    i = np.arange(nc)
    ht = max(1, (nc + wd - 1) // wd)
    s = 2.0 * ((i % wd) + g.rand(nc)) / wd - 1.0
    t = 2.0 * ((i // wd) + g.rand(nc)) / ht - 1.0
    rays = np.zeros((n, 8), np.float32)
    rays[:nc, 0:3] = tuple(c.eye)
    rays[:nc, 4:7] = s[:, None] * np.array(tuple(c.wvec)) + t[:, None] * np.array(tuple(c.hvec)) - np.array(tuple(c.dvec))
    ns = n - nc
    o = np.stack([g.uniform(-11, 11, ns), g.uniform(0.0, 0.45, ns) ** 2 * 2, g.uniform(-11, 11, ns)], 1)
    d = g.standard_normal((ns, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    d[:, 1] = np.abs(d[:, 1]) + g.uniform(0, 0.3, ns)
    rays[nc:, 0:3] = o
    rays[nc:, 4:7] = d
    rays[:, 3] = 1e-3
    rays[:, 7] = 1e16
    return rays


def _ball(sub):
    """A unit sphere: an octahedron subdivided `sub` times (float32 vertices, indices)."""
    v = np.array([[1, 0, 0], [-1, 0, 0], [0, 1, 0], [0, -1, 0], [0, 0, 1], [0, 0, -1]], np.float64)
    tri = [v[[a, b, c]] for a in (0, 1) for b in (2, 3) for c in (4, 5)]
    t = np.stack(tri)
    for _ in range(sub):
        a, b, c = t[:, 0], t[:, 1], t[:, 2]
        n = lambda x: x / np.linalg.norm(x, axis=1, keepdims=True)  # noqa: E731
        ab, bc, ca = n(a + b), n(b + c), n(c + a)
        t = np.concatenate([np.stack(q, 1) for q in ((a, ab, ca), (ab, b, bc), (ca, bc, c), (ab, bc, ca))])
    p = t.reshape(-1, 3).astype(np.float32)
    return p, np.arange(len(p), dtype=np.uint32).reshape(-1, 3)


def _balls(case, seed):
    """The spheres and rays of a "rays" case: mesh, per-thing 3x4 transforms, rays."""
    g = np.random.RandomState((seed * 7919 + case["n"] * 31 + case["things"]) % (1 << 31))
    mesh = _ball(case["sub"])
    xf = np.zeros((case["things"], 3, 4), np.float32)
    r = g.uniform(0.2, 1.0, case["things"])
    for k in range(3):
        xf[:, k, k] = r
    xf[:, :, 3] = g.uniform(-5, 5, (case["things"], 3))
    n = case["n"]
    o = g.standard_normal((n, 3))
    o = 9.0 * o / np.linalg.norm(o, axis=1, keepdims=True)
    at = xf[g.randint(0, case["things"], n), :, 3] + g.uniform(-1, 1, (n, 3))
    rays = np.zeros((n, 8), np.float32)
    rays[:, 0:3] = o
    rays[:, 4:7] = at - o
    rays[:, 3] = 1e-3
    rays[:, 7] = 1e16
    return mesh, xf, rays


def prepare(case, seed):
    rng = random.Random((seed << 8) ^ 0x5EED)
    kind = case["kind"]
    st = {"case": case}
    if kind == "rays":
        mesh, xf, rays = _balls(case, seed)
        s = rtx.Scene()
        if case["two_level"]:
            s.build_mode(rtx.Scene.TWO_LEVEL)
        m = s.add(mesh)
        for x in xf:
            s.set(s.add(rtx.Thing.diffuse((.5, .5, .5)), m), x)
        s.build()
        st.update(scene=s, rays=rays)
        return st
    if kind == "batch":
        jobs, lps, outs = [], [], []
        mix = random.Random(case["mix"])       # the frames' sizes, the same for every seed
        for _ in range(case["frames"]):
            k = 6.0 ** mix.random()
            w, h = min(2 * round(160 * k), 1920), min(2 * round(90 * k), 1080)
            spp = round(4.0 * (case["spp_hi"] / 4.0) ** mix.random())
            s = _scene(rng, mix.randint(2, 6), case["two_level"], mix.randint(3, 11))
            lp, out = _frame(rng, s, w, h, spp, 16, guides=False)
            jobs.append(s)
            lps.append(lp)
            outs.append(out)
        st.update(scene=jobs[0], scenes=jobs, lps=lps, out=outs, stream=torch.cuda.Stream())
        st["batch"] = rtx.Batch(jobs[0], lps, use_graph=True)
        torch.cuda.synchronize()
        return st
    s = _scene(rng, case["level"], case["two_level"], build=kind != "build")
    st["scene"] = s
    if kind == "pick":
        lp, _ = _frame(rng, s, case["w"], case["h"], 1, 16, guides=False)
        lp.picker, lp.pick_x, lp.pick_y = True, rng.randrange(case["w"]), rng.randrange(case["h"] // 2 + 1)
        st["id"] = torch.zeros(1, dtype=torch.int32, device=DEV)
        lp.pick_id = st["id"].data_ptr()
        st["lp"] = lp
    elif kind in ("trace", "build"):
        st["rays"] = torch.from_numpy(_view_rays(rng, case["n"])).to(DEV)
        st["hits"] = torch.zeros((case["n"], 8), dtype=torch.int32, device=DEV)
    elif kind == "frame":
        s.semantics(rtx.Scene.ITERATIVE if case["iterative"] else rtx.Scene.RECURSIVE)
        st["lp"], st["out"] = _frame(rng, s, case["w"], case["h"], case["spp"], case["depth"])
        if case["srgb"]:
            st["out"]["srgb"] = torch.zeros((case["h"], case["w"], 4), dtype=torch.uint8, device=DEV)
    elif kind == "edit":
        st["lp"], st["out"] = _frame(rng, s, case["w"], case["h"], case["spp"], case["depth"])
        st["out"]["srgb"] = torch.zeros((case["h"], case["w"], 4), dtype=torch.uint8, device=DEV)
        # the moved things and their new places
        st["moves"] = []
        for i in rng.sample(range(1, len(s)), min(case["moved"], len(s) - 1)):
            x = s.get(i).reshape(3, 4).copy()
            x[0, 3] += np.float32(rng.uniform(-0.1, 0.1))
            x[2, 3] += np.float32(rng.uniform(-0.1, 0.1))
            st["moves"].append((i, x))
    elif kind == "train":
        st["lp"], _ = _frame(rng, s, case["w"], case["h"], case["spp"], case["depth"], guides=False)
        st["render"] = DiffRender(s, st["lp"])
        st["params"] = material_params(s.things_spec).to(DEV)
        g = torch.Generator(device="cpu").manual_seed(seed % (1 << 31))
        # a target that some blur of brightness separates from the scene's image
        y = torch.linspace(0.3, 0.9, case["h"])[:, None, None].expand(case["h"], case["w"], 3)
        st["target"] = (y + 0.1 * torch.rand((case["h"], case["w"], 3), generator=g)).to(DEV)
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    s = st["scene"]
    if kind == "frame":
        _launch(s, st["lp"])
        if case["srgb"]:
            rtx.pp_sRGB(st["out"]["rawRGB"].data_ptr(), st["out"]["srgb"].data_ptr(), case["w"], case["h"], _stream())
        return st["out"]
    if kind == "trace":
        _ok(rtx.lib().rtx_trace(s.ctx, s.handle, st["rays"].data_ptr(), case["n"], st["hits"].data_ptr(), _stream()))
        return _hits_of(st["hits"])
    if kind == "rays":
        h = s.trace(st["rays"])
        return {"t": h["t"], "uv": np.stack([h["u"], h["v"]], 1),
                "ids": np.stack([h["instance_id"], h["primitive_index"], h["prim"]], 1).astype(np.int64)}
    if kind == "build":
        s.build(_stream())
        _ok(rtx.lib().rtx_trace(s.ctx, s.handle, st["rays"].data_ptr(), case["n"], st["hits"].data_ptr(), _stream()))
        out = _hits_of(st["hits"])
        tree = s.stats()
        out["tree"] = [int(tree[k]) for k in ("num_prims", "num_nodes", "num_leaves", "max_depth", "max_leaf",
                                              "wide_nodes", "wide_depth", "unique_prims", "tlas_nodes")]
        out["sah_cost"] = float(tree["sah_cost"])
        return out
    if kind == "pick":
        _launch(s, st["lp"], 1)
        return {"id": st["id"]}
    if kind == "edit":
        for i, x in st["moves"]:
            s.set(i, x)
        s.update(s.handle, _stream())
        _launch(s, st["lp"])
        rtx.pp_sRGB(st["out"]["rawRGB"].data_ptr(), st["out"]["srgb"].data_ptr(), case["w"], case["h"], _stream())
        return st["out"]
    if kind == "train":
        p = st["params"].clone().requires_grad_()
        img = st["render"](p)
        loss = ((img - st["target"]) ** 2).sum()
        loss.backward()
        return {"image": img.detach(), "loss": loss.detach(), "grad": p.grad}
    st["batch"].launch(st["stream"].cuda_stream, sync=False)
    return st["out"]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _triangles(level, half=11):
    if level == "mixed":
        return 8.8e6, 1.33e6              # instanced, stored
    n = (2 * half) ** 2 - 8
    return n * 4.0 ** (level + 1), 4.0 ** (level + 1)


def _ray_flops(tris):
    # one box test of 4 children (18 operations each) per level of a 4-wide
    # tree, one triangle test
    return 72.0 * max(1.0, math.log(max(tris, 4.0), 4.0)) + 60.0


def _scene_bytes(case, half=11):
    # 48 B per stored triangle and half a 128 B node for each 2 triangles
    n, stored = _triangles(case["level"], half)
    return 80.0 * (stored if case["two_level"] else n)


def work(case):
    kind = case["kind"]
    if kind == "rays":
        tris = case["things"] * 8 * 4 ** case["sub"]
        return {"bytes": 64.0 * case["n"] + 80.0 * tris, "flops": case["n"] * _ray_flops(tris)}
    if kind == "batch":
        px, spp, rays = 6.2e5, (4.0 * case["spp_hi"]) ** 0.5 * 1.3, 2.4
        return {"bytes": case["frames"] * (16.0 * px + 80.0 * 1.1e6),
                "flops": case["frames"] * px * spp * rays * (_ray_flops(1.1e6) + 120.0)}
    tris = _triangles(case["level"])[0]
    scene = _scene_bytes(case)
    if kind == "pick":
        return {"bytes": 4.0 + 20 * 128.0, "flops": _ray_flops(tris)}
    if kind == "trace":
        return {"bytes": 64.0 * case["n"] + min(scene, 700.0 * case["n"]), "flops": case["n"] * _ray_flops(tris)}
    if kind == "build":
        n, stored = _triangles(case["level"])
        # read the meshes, write triangles and nodes; a cost for each of 3 axes
        # and each level of the tree per triangle
        made = stored if case["two_level"] else n
        return {"bytes": 30.0 * stored + 96.0 * made, "flops": made * 3.0 * 10.0 * math.log2(max(made, 2.0))}
    px = case["w"] * case["h"]
    rays = px * case["spp"] * 2.5
    if kind == "train":
        return {"bytes": 24.0 * px + 2 * scene, "flops": 2 * rays * (_ray_flops(tris) + 120.0)}
    out = 40.0 + (4.0 if kind == "edit" or case.get("srgb") else 0.0)
    return {"bytes": out * px + min(scene, 700.0 * rays), "flops": rays * (_ray_flops(tris) + 120.0)}


# ---------------------------------------------------------------------------
# in 64 bits
# ---------------------------------------------------------------------------
def exact(case, seed):
    """Distances and barycentrics of the "rays" cases by testing every triangle in FP64.

    A rendered frame has no such value (a path's later rays depend on the
    rounding of its earlier ones), nor have identifiers; the other closest-hit
    queries are over too many triangles."""
    if case["kind"] != "rays":
        return None
    (v, i), xf, rays = _balls(case, seed)
    dev = DEV if torch.cuda.is_available() else "cpu"
    p = v.astype(np.float64)[i]                                             # [m, 3, 3]
    x = xf.astype(np.float64)
    tri = np.einsum("ark,mvk->amvr", x[:, :, :3], p) + x[:, None, None, :, 3]
    tri = torch.from_numpy(tri.reshape(-1, 3, 3)).to(dev)
    r = torch.from_numpy(rays.astype(np.float64)).to(dev)
    a, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    ts, uvs = [], []
    for c in range(0, len(r), 256):
        o, d = r[c:c + 256, None, 0:3], r[c:c + 256, None, 4:7]
        q = torch.linalg.cross(d.expand(-1, len(a), -1), e2[None].expand(len(o), -1, -1))
        det = (e1 * q).sum(-1)
        w = o - a
        u = (w * q).sum(-1) / det
        k = torch.linalg.cross(w, e1[None].expand(len(o), -1, -1))
        vv = (d * k).sum(-1) / det
        t = (e2 * k).sum(-1) / det
        hit = (det != 0) & (u >= 0) & (vv >= 0) & (u + vv <= 1) & (t > r[c:c + 256, None, 3])
        t = torch.where(hit, t, torch.full_like(t, math.inf))
        best, at = t.min(1)
        row = torch.arange(len(t), device=dev)
        miss = torch.isinf(best)
        ts.append(best)
        uv = torch.stack([u[row, at], vv[row, at]], 1)
        uvs.append(torch.where(miss[:, None], torch.zeros_like(uv), uv))
    return {"t": torch.cat(ts).cpu().numpy(), "uv": torch.cat(uvs).cpu().numpy(), "ids": None}

"""The work a program has this library do, as measurable cases.

Eight kinds of pass, each through the public entry points of `ptamd`, at the
library's default settings, on one stream:

  trace        a batch of closest-hit queries against one scene
  rebuild      a dynamic scene's frame: the LBVH rebuilt, then a batch of
               camera rays traced in it
  batch        the same for a batch of scenes of different sizes
  render       a progressive render from an empty accumulator: frames of one
               pass, as a viewer asks for them, or of several passes
  cache_frame  radiance-cache frames (queries, training paths, Adam steps)
  infer        radiance-cache predictions for a batch of samples
  gradient     the cache's loss gradient for a batch of samples

Scenes come from the library's own seeded generators, rays and samples from
torch's, all from the seed alone.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("cuda-path-tracer_amd"))
import ptamd  # noqa: E402

HAIR_STEPS = 144  # ribbon segments of one strand of the hair ball
FLT_MAX = float(np.finfo(np.float32).max)


def listed():
    return [
        # A picking or visibility query against a small object: the smallest
        # call, where the launches count.
        {"name": "trace_pick", "kind": "trace", "scene": "soup", "tris": 4096, "rays": 2000, "view": "camera", "uv": True},
        # The headline batch: rays from all around a large mesh.
        {"name": "trace_mesh_16m", "kind": "trace", "scene": "mesh", "tris": 871200, "rays": 16777216, "view": "shell",
         "uv": False},
        # Primary visibility of a 1920 x 1080 image of a hair ball.
        {"name": "trace_hair_1080p", "kind": "trace", "scene": "hair", "tris": 2880000, "rays": 2073600, "view": "camera",
         "uv": True},
        # A small animated object: rebuilt and traced every frame.
        {"name": "rebuild_mesh_10k", "kind": "rebuild", "scene": "mesh", "tris": 9800, "rays": 4096},
        # A large dynamic scene in no order: the build's own benchmark size.
        {"name": "rebuild_soup_1m", "kind": "rebuild", "scene": "soup", "tris": 1048576, "rays": 131072},
        # Many scenes of 1,024 to 262,144 triangles built by one call.
        {"name": "batch_64", "kind": "batch", "scenes": 64, "most": 262144, "rays": 262144},
        # Interactive preview of a soup: short frames of one pass.
        {"name": "render_soup_256", "kind": "render", "scene": "soup", "tris": 65536, "w": 256, "h": 256, "bounces": 4,
         "rr": -1, "frames": 8, "per_frame": 1, "lights": 0, "detail": False},
        # A viewer on a closed room with a large mesh, Russian roulette.
        {"name": "render_room_1024", "kind": "render", "scene": "room", "tris": 871200, "w": 1024, "h": 1024, "bounces": 8,
         "rr": 3, "frames": 2, "per_frame": 1, "lights": 0, "detail": False},
        # An offline render of a textured object under two directional
        # lights, sixteen passes to a frame, at an odd size.
        {"name": "render_lit_textured", "kind": "render", "scene": "mesh", "tris": 180000, "w": 637, "h": 359, "bounces": 4,
         "rr": 2, "frames": 1, "per_frame": 16, "lights": 2, "detail": True},
        # The radiance cache in use: 1920 x 1080 frames that also train.
        {"name": "cache_frame_1080p", "kind": "cache_frame", "tris": 871200, "w": 1920, "h": 1080, "samples": 65536,
         "steps": 4, "frames": 2},
        # The cache asked for a whole image's vertices.
        {"name": "infer_2m", "kind": "infer", "samples": 2073600},
        # One training batch's gradient.
        {"name": "gradient_16k", "kind": "gradient", "samples": 16384},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["trace", "trace", "rebuild", "batch", "render", "render", "cache_frame", "infer", "gradient"])
    if kind == "trace":
        return {"kind": kind, "scene": rng.choice(["soup", "mesh", "hair", "room"]), "tris": _log(rng, 2000, 2000000),
                "rays": _log(rng, 1000, 8000000), "view": rng.choice(["shell", "camera"]), "uv": rng.random() < 0.5}
    if kind == "rebuild":
        return {"kind": kind, "scene": rng.choice(["soup", "mesh", "hair", "room"]), "tris": _log(rng, 2000, 2000000),
                "rays": _log(rng, 1000, 200000)}
    if kind == "batch":
        return {"kind": kind, "scenes": _log(rng, 2, 96), "most": _log(rng, 4000, 262144), "rays": _log(rng, 10000, 500000)}
    if kind == "render":
        w, h = _log(rng, 100, 800), _log(rng, 100, 600)
        scene = rng.choice(["soup", "mesh", "hair", "room"])
        tris = _log(rng, 5000, 400000)
        return {"kind": kind, "scene": scene, "tris": tris, "w": w, "h": h, "bounces": rng.randint(1, 8),
                "rr": rng.choice([-1, 2, 3]), "frames": rng.randint(1, 2), "per_frame": rng.choice([1, 1, 1, 4]),
                "lights": rng.choice([0, 0, 1, 2]), "detail": rng.random() < 0.25}
    if kind == "cache_frame":
        w, h = _log(rng, 200, 1920), _log(rng, 150, 1080)
        return {"kind": kind, "tris": _log(rng, 5000, 871200), "w": w, "h": h,
                "samples": min(w * h // 16, _log(rng, 1000, 65536)), "steps": rng.randint(1, 4), "frames": 2}
    if kind == "infer":
        return {"kind": kind, "samples": _log(rng, 1000, 2000000)}
    return {"kind": kind, "samples": _log(rng, 1000, 65536)}


# ---- scenes, rays and samples ---------------------------------------------------


def _bands(tris):
    return max(3, round(math.sqrt(tris / 2.0)))


def _strands(tris):
    return max(1, round(tris / (2.0 * HAIR_STEPS)))


def _ntris(case):
    """Triangles of the scene a case names (its size as the generator rounds it)."""
    s, n = case.get("scene", "room"), case["tris"]
    if s == "soup":
        return n + 2
    if s == "hair":
        return 2 * _strands(n) * HAIR_STEPS + 2
    return 2 * _bands(n) ** 2 + (14 if s == "room" else 0)


def _scene(case, seed):
    s, n = case.get("scene", "room"), case["tris"]
    if s == "soup":
        return ptamd.gen_soup(n, seed)
    if s == "hair":
        return ptamd.gen_hairball(_strands(n), HAIR_STEPS, seed)
    return ptamd.gen_sphere(_bands(n), seed, room=s == "room")


_VIEW = {"soup": ((0.5, 0.5, -1.5), (0.5, 0.5, 0.5)), "mesh": ((0.0, 0.4, -3.0), (0.0, 0.0, 0.0)),
         "hair": ((0.0, 0.6, -3.2), (0.0, 0.0, 0.0)), "room": ((0.0, 0.0, -1.9), (0.0, 0.0, 0.0))}


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _shell_rays(n, seed, bmin, bmax, enlarge=1.5):
    """Origins uniform on the box enlarged about its centre, directions uniform on the sphere."""
    g = _generator(seed)
    c = torch.tensor((np.asarray(bmin) + np.asarray(bmax)) * 0.5, device="cuda", dtype=torch.float32)
    e = torch.tensor((np.asarray(bmax) - np.asarray(bmin)) * 0.5 * enlarge, device="cuda", dtype=torch.float32)
    area = torch.stack([e[1] * e[2], e[0] * e[2], e[0] * e[1]])
    axis = torch.bucketize(torch.rand(n, generator=g, device="cuda"), torch.cumsum(area / area.sum(), 0)[:2])
    p = torch.rand(n, 3, generator=g, device="cuda") * 2 - 1
    side = torch.where(torch.rand(n, 1, generator=g, device="cuda") < 0.5, -1.0, 1.0)
    p = p.scatter(1, axis[:, None], side) * e + c
    d = torch.randn(n, 3, generator=g, device="cuda")
    d = d / d.norm(dim=1, keepdim=True)
    return torch.cat([p, d], 1).contiguous()


def _camera_rays(n, seed, scene):
    """One ray through each of n pixels of a 16:9 image, in pixel order, jittered."""
    eye, target = _VIEW[scene]
    w = max(1, round(math.sqrt(n * 16 / 9)))
    k = torch.arange(n, device="cuda")
    j = torch.rand(n, 2, generator=_generator(seed), device="cuda")
    x = ((k % w).float() + j[:, 0]) / w
    y = ((k // w).float() + j[:, 1]) / max(1.0, n / w)
    dirs = torch.tensor(ptamd.camera_corners(eye, target, aspect=16 / 9).reshape(4, 3), device="cuda")
    a = dirs[0] + x[:, None] * (dirs[1] - dirs[0])
    b = dirs[3] + x[:, None] * (dirs[2] - dirs[3])
    d = a + y[:, None] * (b - a)
    return torch.cat([torch.tensor(eye, device="cuda").expand(n, 3), d], 1).contiguous()


def _detail(n, seed):
    """Surface detail of n triangles and three textures: vertex colours, uvs,
    tangent frames; most triangles textured, half of them normal-mapped."""
    rng = np.random.default_rng(seed)
    det = np.zeros(n, ptamd.DETAIL_DTYPE)
    det["color"] = rng.uniform(0.05, 1.0, (n, 3, 3))
    det["uv"] = rng.uniform(0.0, 1.0, (n, 3, 2))
    det["tangent"] = rng.normal(size=(n, 3, 3))
    det["bitangent"] = rng.normal(size=(n, 3, 3))
    det["albedo_tex"] = np.where(rng.random(n) < 0.7, rng.integers(0, 2, n), ptamd.NO_TEXTURE)
    det["normal_tex"] = np.where(rng.random(n) < 0.5, 2, ptamd.NO_TEXTURE)
    texs = [rng.integers(60, 256, (s, s, 4), dtype=np.uint8) for s in (512, 256, 256)]
    texs[2][..., 2] = 255
    return det, texs


def _params(seed):
    """Network parameters of a cache in training: He-uniform weights, small biases."""
    rng = np.random.default_rng(seed)
    out = []
    for ni, no in ((96, 64), (64, 64), (64, 64), (64, 64), (64, 3)):
        out.append(rng.uniform(-1, 1, ni * no) * math.sqrt(6.0 / ni) * (0.3 if no == 3 else 1.0))
        out.append(rng.uniform(-0.1, 0.1, no))
    return np.concatenate(out).astype(np.float32)


_BOX = ((-2.0, -2.0, -2.0), (2.0, 2.0, 2.0))  # the room


def _samples(n, seed):
    """Path vertices in the room: positions on its walls, unit normals and directions, albedos."""
    g = _generator(seed)
    r = _shell_rays(n, seed + 1, *_BOX, enlarge=1.0)
    nrm = torch.randn(n, 3, generator=g, device="cuda")
    nrm = nrm / nrm.norm(dim=1, keepdim=True)
    alb = torch.rand(n, 3, generator=g, device="cuda") * 0.6 + 0.3
    return torch.cat([r[:, :3], nrm, r[:, 3:], alb], 1).contiguous()


def _targets(n, seed):
    """Radiance targets, one in twenty masked (a path that never reached its vertex)."""
    g = _generator(seed)
    t = torch.rand(n, 3, generator=g, device="cuda") ** 3 * 4
    return torch.where(torch.rand(n, 1, generator=g, device="cuda") < 0.05, float("nan"), t).contiguous()


_stream = None


def _context():
    """A context on the program's one stream."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    ctx = ptamd.Context(0)
    ctx.set_stream(_stream.cuda_stream)
    return ctx


def _hits(n, uv):
    return {"id": torch.zeros(n, dtype=torch.int32, device="cuda"), "t": torch.zeros(n, device="cuda"),
            "uv": torch.zeros(n, 2, device="cuda") if uv else None}


def _batch_counts(case):
    return ptamd.batch_counts(case["scenes"], 3, 1024, case["most"])


def _batch(case, seed):
    return ptamd.gen_batch(case["scenes"], seed % 4093, counts=_batch_counts(case))


def _batch_rays(case, seed):
    n = case["rays"]
    rays = _shell_rays(n, seed, (0, 0, 0), (1, 1, 1))
    ids = torch.randint(0, case["scenes"], (n,), generator=_generator(seed + 1), device="cuda", dtype=torch.int32)
    return rays, ids


# ---- the passes -----------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "ctx": _context()}
    ctx = s["ctx"]
    if kind in ("trace", "rebuild"):
        tris, infos = _scene(case, seed)
        ctx.upload_scene(tris, infos)
        if case.get("view") == "shell":
            s["rays"] = _shell_rays(case["rays"], seed + 7, *ptamd.scene_bounds(tris))
        else:
            s["rays"] = _camera_rays(case["rays"], seed + 7, case["scene"])
        s["out"] = _hits(case["rays"], case.get("uv", True))
    elif kind == "batch":
        tris, infos, offsets = _batch(case, seed)
        ctx.upload_scenes(tris, offsets, infos)
        s["rays"], s["ids"] = _batch_rays(case, seed + 7)
        s["out"] = _hits(case["rays"], True)
    elif kind == "render":
        tris, infos = _scene(case, seed)
        rr = ptamd.INVALID if case["rr"] < 0 else case["rr"]
        lights = np.array([[1.0, 0.9, 0.8, 0.28, -0.94, 0.19, 1.5], [0.2, 0.3, 1.0, -0.42, -0.34, 0.84, 0.7]], np.float32)
        infos["specularity"] = np.where(infos["emission"].sum(1) > 0, 0, (np.arange(len(infos)) % 3) * 8.0)
        ctx.upload_scene(tris, infos, settings=ptamd.Settings(case["bounces"], rr, 1.0, 1), lights=lights[:case["lights"]])
        if case["detail"]:
            ctx.upload_detail(*_detail(len(infos), seed))
        _view(s, case, case["scene"], seed, case["frames"] * case["per_frame"])
    elif kind == "cache_frame":
        tris, infos = _scene(case, seed)
        ctx.upload_scene(tris, infos, settings=ptamd.Settings(9, 3, 1.0, 1))
        ctx.cache_init(seed, *ptamd.scene_bounds(tris))
        s["settings"] = ptamd.CacheSettings(case["samples"], case["steps"], 8, train=True)
        _view(s, case, "room", seed, case["frames"])
    else:
        n = case["samples"]
        ctx.cache_init(seed, *_BOX)
        ctx.cache_set_params(_params(seed))
        s["raw"] = _samples(n, seed)
        if kind == "infer":
            s["out"] = torch.zeros(n, 3, device="cuda")
        else:
            s["target"] = _targets(n, seed + 2)
            s["out"] = torch.zeros(ptamd.CACHE_PARAMS, device="cuda")
    torch.cuda.synchronize()
    return s


def _view(s, case, scene, seed, passes):
    """Corner rays and seeds of every pass, and the image."""
    w, h = case["w"], case["h"]
    eye, target = _VIEW[scene]
    s["eye"] = eye
    s["dirs"] = np.stack([ptamd.camera_corners(eye, target, (0, 1, 0), 60.0, w / h, *ptamd.pass_jitter(seed, p, w, h))
                          for p in range(passes)])
    s["seeds"] = np.arange(seed, seed + passes, dtype=np.uint64)
    s["out"] = torch.zeros(h, w, 4, device="cuda")


def run(s):
    case, ctx, out = s["case"], s["ctx"], s["out"]
    kind = case["kind"]
    if kind in ("trace", "rebuild"):
        if kind == "rebuild":
            ctx.build_bvh(timed=False)
        uv = out["uv"]
        ctx.trace_closest_device(s["rays"].data_ptr(), case["rays"], out["id"].data_ptr(), out["t"].data_ptr(),
                                 0 if uv is None else uv.data_ptr())
    elif kind == "batch":
        ctx.build_bvh(timed=False)
        ctx.trace_closest_scenes_device(s["rays"].data_ptr(), s["ids"].data_ptr(), case["rays"], out["id"].data_ptr(),
                                        out["t"].data_ptr(), out["uv"].data_ptr())
    elif kind in ("render", "cache_frame"):
        w, h = case["w"], case["h"]
        per = case.get("per_frame", 1)
        ctx.reset_frames()
        for f in range(case["frames"]):
            ctx.set_primary_rays(s["dirs"][f * per], s["eye"])
            if kind == "cache_frame":
                ctx.render_cache_frame(w, h, int(s["seeds"][f]), s["settings"])
            elif per == 1:
                ctx.render_pass(w, h, int(s["seeds"][f]))
            else:
                ctx.render_passes(w, h, s["seeds"][f * per:(f + 1) * per], s["dirs"][f * per:(f + 1) * per])
        ctx.read_image_device(out.data_ptr(), w, h)
    elif kind == "infer":
        ctx.cache_infer_device(s["raw"].data_ptr(), case["samples"], out.data_ptr())
    else:
        ctx.cache_gradient_device(s["raw"].data_ptr(), s["target"].data_ptr(), case["samples"], out.data_ptr())
    return out


# ---- what a pass cannot do without ------------------------------------------------

MLP_MACS = 18624          # weights of the network: multiplications of one forward pass
BOX_FLOPS, TRI_FLOPS = 24, 50


def _ray_flops(ntris):
    """One walk from the root to a leaf: both child boxes of each node, one triangle."""
    return 2 * BOX_FLOPS * math.ceil(math.log2(max(2, ntris))) + TRI_FLOPS


def work(case):
    kind = case["kind"]
    if kind in ("trace", "rebuild", "batch"):
        hit = 8 + (8 if case.get("uv", True) else 0)
        n = int(_batch_counts(case).sum()) if kind == "batch" else _ntris(case)
        bytes_ = case["rays"] * (24 + hit + (4 if kind == "batch" else 0))
        flops = case["rays"] * _ray_flops(n / case["scenes"] if kind == "batch" else n)
        if kind != "trace":
            # A build reads 40 bytes a triangle and writes its node (64) and its sorted triangle (48).
            bytes_ += n * 152
            flops += n * 40
        return {"bytes": bytes_, "flops": flops}
    if kind in ("render", "cache_frame"):
        npix = case["w"] * case["h"]
        frames, per = case["frames"], case.get("per_frame", 1)
        # The image once, the FP64 accumulator read and written by every frame.
        bytes_ = npix * (16 + 48 * frames)
        flops = npix * frames * per * _ray_flops(_ntris(case))
        if kind == "cache_frame":
            flops += frames * (2 * MLP_MACS * npix + 6 * MLP_MACS * case["samples"])
        return {"bytes": bytes_, "flops": flops}
    n = case["samples"]
    if kind == "infer":
        return {"bytes": 60 * n + 4 * ptamd.CACHE_PARAMS, "flops": 2 * MLP_MACS * n}
    return {"bytes": 60 * n + 8 * ptamd.CACHE_PARAMS, "flops": 6 * MLP_MACS * n}


# ---- the same in 64 bits ------------------------------------------------------------

MOST_PAIRS = 4e9  # ray-triangle pairs that brute force takes


def _brute(rays, tris):
    """Nearest hit of each ray over all triangles, in 64 bits: t (FLT_MAX on a miss), uv."""
    r = rays.double()
    v = [torch.tensor(np.ascontiguousarray(tris[k]), device="cuda").double() for k in ("v0", "v1", "v2")]
    n = len(r)
    best = torch.full((n,), FLT_MAX, dtype=torch.float64, device="cuda")
    uv = torch.zeros(n, 2, dtype=torch.float64, device="cuda")
    rc, tc = 4096, 16384
    for a in range(0, n, rc):
        o, d = r[a:a + rc, None, :3], r[a:a + rc, None, 3:]
        for b in range(0, len(v[0]), tc):
            p = v[0][None, b:b + tc]
            e1, e2 = v[1][None, b:b + tc] - p, v[2][None, b:b + tc] - p
            q = torch.cross(d.expand(-1, e2.shape[1], -1), e2.expand(d.shape[0], -1, -1), dim=2)
            det = (e1 * q).sum(2)
            ok = det.abs() >= 1.192092896e-07
            inv = 1.0 / torch.where(ok, det, 1.0)
            t0 = o - p
            u = (t0 * q).sum(2) * inv
            del q
            rr = torch.cross(t0, e1.expand_as(t0), dim=2)
            w = (d * rr).sum(2) * inv
            t = (e2 * rr).sum(2) * inv
            del rr, t0
            ok &= (u >= 0) & (w >= 0) & (u + w <= 1) & (t >= 0)
            t = torch.where(ok, t, FLT_MAX)
            m, k = t.min(1)
            near = m < best[a:a + rc]
            best[a:a + rc] = torch.where(near, m, best[a:a + rc])
            pick = torch.stack([u.gather(1, k[:, None])[:, 0], w.gather(1, k[:, None])[:, 0]], 1)
            uv[a:a + rc] = torch.where(near[:, None], pick, uv[a:a + rc])
    return best, uv


def _encode(raw, bmin, bmax):
    """The network's 96 inputs: 12 frequencies of sin, cos of the position in the box, the rest as it is."""
    r = raw.double()
    lo = torch.tensor(bmin, dtype=torch.float64, device=r.device)
    hi = torch.tensor(bmax, dtype=torch.float64, device=r.device)
    p = (r[:, :3] - lo) / (hi - lo)
    a = math.pi * p[:, :, None] * (2.0 ** torch.arange(12, dtype=torch.float64, device=r.device))
    enc = torch.stack([a.sin(), a.cos()], 3).reshape(len(r), 72)
    return torch.cat([enc, r[:, 3:], torch.zeros(len(r), 15, dtype=torch.float64, device=r.device)], 1)


def _network(params, x):
    k = 0
    for i, (ni, no) in enumerate(((96, 64), (64, 64), (64, 64), (64, 64), (64, 3))):
        w = params[k:k + ni * no].reshape(ni, no)
        x = x @ w + params[k + ni * no:k + ni * no + no]
        k += ni * no + no
        x = x.relu() if i < 4 else x.exp()
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind in ("trace", "rebuild"):
        if case["rays"] * _ntris(case) > MOST_PAIRS:
            return None
        tris, _ = _scene(case, seed)
        if case.get("view") == "shell":
            rays = _shell_rays(case["rays"], seed + 7, *ptamd.scene_bounds(tris))
        else:
            rays = _camera_rays(case["rays"], seed + 7, case["scene"])
        t, uv = _brute(rays, tris)
        return {"id": None, "t": t, "uv": uv if case.get("uv", True) else None}
    if kind == "batch":
        counts = _batch_counts(case)
        if case["rays"] * float(counts.mean()) > MOST_PAIRS:
            return None
        tris, _, offsets = _batch(case, seed)
        rays, ids = _batch_rays(case, seed + 7)
        t = torch.zeros(case["rays"], dtype=torch.float64, device="cuda")
        uv = torch.zeros(case["rays"], 2, dtype=torch.float64, device="cuda")
        for k in range(case["scenes"]):
            at = (ids == k).nonzero()[:, 0]
            if len(at):
                t[at], uv[at] = _brute(rays[at], tris[offsets[k]:offsets[k + 1]])
        return {"id": None, "t": t, "uv": uv}
    if kind in ("render", "cache_frame"):
        return None  # a path's later vertices depend on every rounding before them
    params = torch.tensor(_params(seed), device="cuda").double()
    raw = _samples(case["samples"], seed)
    if kind == "infer":
        return torch.cat([_network(params, _encode(part, *_BOX)) for part in raw.split(1 << 17)])
    target = _targets(case["samples"], seed + 2).double()
    params.requires_grad_(True)
    y = _network(params, _encode(raw, *_BOX))
    kept = ~target[:, 0].isnan()
    den = y.detach() ** 2 + 0.01
    loss = ((y[kept] - target[kept]) ** 2 / den[kept]).sum() / case["samples"]
    return torch.autograd.grad(loss, params)[0]

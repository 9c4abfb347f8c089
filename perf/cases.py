"""What a user of the renderer has it do, as cases that can be timed.

Four kinds of work, each through the public entry points of ``adop_amd.render`` and ``adop_amd.preprocess``:

* ``view``     a frame for display or evaluation: ``BlendPointCloud`` without gradients, with or without the environment
               map composed into it
* ``step``     the render stage of a training step: ``BlendPointCloud`` and its backward pass with every gradient
* ``prepare``  the processing of a new scene: ``PreprocessPointCloud``
* ``filter``   the point filters of a new scene: ``FilterPointCloud``

``listed()`` holds cases of the repository's own configurations and of the shapes around them, ``draw()`` one more of the
same ranges: clouds of 20 thousand to 100 million points, images of 96 to 2200 pixels a side, 1 to 16 views, 1 to 5
levels, 3, 4 or 8 channels, fp32 and fp16 descriptors, pinhole cameras with and without distortion and fisheye cameras,
the LOD radius test on (as the reference ships it) and off, near and far cameras.

Everything is made on the GPU from the seed.  Clouds go through ``PreprocessPointCloud`` before they are rendered, as
every scene does; ``ordered = False`` leaves a cloud in the order it was generated in.
"""
import gc
import math

import numpy as np
import torch

from adop_amd import _capi, preprocess, render, scenes

_MODELS = {"pinhole": _capi.CAMERA_PINHOLE_DISTORTION, "distorted": _capi.CAMERA_PINHOLE_DISTORTION,
           "fisheye": _capi.CAMERA_OCAM}
_ENV_SIZE = (512, 1024)
_WHOLE_PREPARATION = 1 << 25  # points


def _case(kind, cloud, points, **kw):
    c = {"kind": kind, "cloud": cloud, "points": int(points), "ordered": True, "normals": True}
    if kind in ("view", "step"):
        c.update({"w": 512, "h": 512, "views": 1, "levels": 4, "channels": 4, "half": False, "camera": "pinhole",
                  "crops": False, "lod": True, "dropout": kind == "step", "env": False, "distance": 1.0})
    if kind == "filter":
        c.update({"frames": 100})
    for k, v in kw.items():
        assert k in c, k
        c[k] = v
    return c


def listed():
    return [
        # The smallest frame: a thumbnail or a smoke test of a raw cloud, nothing but latency and launches.
        {"name": "view_small", **_case("view", "box", 100_000, w=256, h=256, lod=False, ordered=False)},
        # The viewer on a large scene: 100 M points, Full HD, descriptors stored as halves.
        {"name": "view_100m", **_case("view", "volume", 100_000_000, w=1920, h=1080, levels=5, half=True, lod=False,
                                      normals=False)},
        # A frame of a photographed scene at the size of its photo: odd sides, lens distortion, environment map.
        {"name": "view_photo", **_case("view", "patches", 12_000_000, w=1365, h=911, camera="distorted", env=True)},
        # The viewer's camera moved away: the whole cloud falls on a small part of the image.
        {"name": "view_far", **_case("view", "surface", 8_000_000, w=1920, h=1080, distance=6.0)},
        # A training step on one full frame.
        {"name": "step_frame", **_case("step", "surface", 10_000_000, w=1920, h=1080, channels=8, lod=False)},
        # The training batch as the reference forms it: 4 random crops of 512 x 512 from each of 4 frames.
        {"name": "step_crops", **_case("step", "surface", 10_000_000, views=16, crops=True, camera="distorted")},
        # The reference's setting for small cards: crops of 256 x 256.
        {"name": "step_crops_256", **_case("step", "surface", 2_000_000, w=256, h=256, views=16, crops=True)},
        # A small batch of whole images.
        {"name": "step_batch", **_case("step", "ball", 1_000_000, views=4, lod=False)},
        # An object of a few thousand points on a small odd image: the smallest training step.
        {"name": "step_small", **_case("step", "ball", 50_000, w=161, h=121, levels=3, channels=3)},
        # Fisheye images with the spherical environment map and its texture gradient.
        {"name": "step_fisheye", **_case("step", "patches", 20_000_000, w=2200, h=1500, views=8, camera="fisheye",
                                         dropout=False, env=True, lod=False)},
        # A new scene: Morton order, block shuffle, radii from the nearest neighbours, blocks sorted by radius.
        {"name": "prepare_10m", **_case("prepare", "patches", 10_000_000)},
        # The filters of a new scene against its 100 frames.
        {"name": "filter_3m", **_case("filter", "surface", 3_000_000, frames=100)},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["view", "view", "view", "step", "step", "step", "step", "prepare", "filter"])
    cloud = rng.choice(["surface", "surface", "patches", "volume", "ball"])
    if kind == "prepare":
        return _case(kind, cloud, _log(rng, 50_000, 10_000_000), normals=rng.random() < 0.8)
    if kind == "filter":
        return _case(kind, rng.choice(["surface", "patches"]), _log(rng, 50_000, 3_000_000),
                     frames=_log(rng, 8, 100))
    kw = {"levels": rng.choice([1, 3, 4, 4, 4, 5]), "channels": rng.choice([3, 4, 4, 4, 8, 8]),
          "half": rng.random() < 0.2, "lod": rng.random() < 0.6, "ordered": rng.random() < 0.9,
          "camera": rng.choice(["pinhole", "distorted", "distorted", "fisheye"]), "env": rng.random() < 0.25}
    kw["normals"] = cloud != "volume"
    kw["lod"] = kw["lod"] and kw["ordered"]  # the radii of the LOD test come with the preparation
    if kind == "view":
        return _case(kind, cloud, _log(rng, 30_000, 30_000_000), w=_log(rng, 128, 2200), h=_log(rng, 96, 1500),
                     distance=math.exp(rng.uniform(0.0, math.log(6.0))), **kw)
    kw["dropout"] = rng.random() < 0.8
    if rng.random() < 0.4:
        side = rng.choice([256, 384, 512])
        kw["camera"] = rng.choice(["pinhole", "distorted"])
        return _case(kind, cloud, _log(rng, 100_000, 10_000_000), w=side, h=side, views=rng.choice([4, 8, 16]),
                     crops=True, **kw)
    return _case(kind, cloud, _log(rng, 20_000, 10_000_000), w=_log(rng, 96, 2000), h=_log(rng, 96, 1200),
                 views=rng.choice([1, 1, 1, 2, 3, 4]), **kw)


# ---- inputs -----------------------------------------------------------------------------------------------------

def _unit(v):
    return v / v.norm(dim=1, keepdim=True)


def _pack_normals(n):
    """3 x 10 bits, x lowest (as ``scenes.pack_normals``, on the device)."""
    q = torch.round((n * 0.5 + 0.5) * 1023.0).clamp_(0, 1023).to(torch.int32)
    return q[:, 0] | (q[:, 1] << 10) | (q[:, 2] << 20)


def _cloud(kind, n, gen):
    """(positions [n,3], unit normals [n,3] or None, distance of a camera that fills its image with the cloud)"""
    def uniform(lo, hi, *shape):
        return torch.rand(*shape, generator=gen, device="cuda") * (hi - lo) + lo

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device="cuda")

    if kind == "surface":  # a sphere above a plane
        ns = int(round(n * 0.6))
        s = _unit(normal(ns, 3))
        p = uniform(-2.0, 2.0, n - ns, 3)
        p[:, 1] = -1.0
        up = torch.zeros_like(p)
        up[:, 1] = 1.0
        return torch.cat([s, p]), torch.cat([s, up]), 3.0
    if kind == "ball":  # a Gaussian cloud, normals outward
        p = normal(n, 3) * 0.5
        return p, _unit(p + 1e-12), 3.0
    if kind == "box":  # a cube full of points with normals in every direction
        return uniform(-1.0, 1.0, n, 3), _unit(normal(n, 3)), 3.0
    if kind == "volume":  # a cube full of points without normals
        return uniform(-5.0, 5.0, n, 3), None, 12.0
    if kind == "patches":  # planar patches of all orientations
        k = 1000
        centre = uniform(-3.0, 3.0, k, 3)
        nrm = _unit(normal(k, 3))
        a = _unit(torch.cross(nrm, normal(k, 3), dim=1))
        b = torch.cross(nrm, a, dim=1)
        pid = torch.randint(0, k, (n,), generator=gen, device="cuda")
        u, v = uniform(-0.25, 0.25, n, 1), uniform(-0.25, 0.25, n, 1)
        return centre[pid] + u * a[pid] + v * b[pid], nrm[pid], 5.0
    raise ValueError(kind)


def _points(case, seed, gen):
    xyz, nrm, near = _cloud(case["cloud"], case["points"], gen)
    position = torch.zeros(case["points"], 4, device="cuda")
    position[:, :3] = xyz
    del xyz
    packed = _pack_normals(nrm) if (nrm is not None and case["normals"]) else None
    return position, packed, near


def _order(position, normal, seed):
    n = int(position.shape[0])
    if n <= _WHOLE_PREPARATION:
        position, normal, _, _ = preprocess.PreprocessPointCloud(position, normal, seed=seed)
        return position, normal
    order = preprocess.ReorderMorton64(position)
    order = order[preprocess.RandomBlockShuffle(n, 256, torch.Generator().manual_seed(seed))]
    parts = order.split(1 << 24)  # (one gather of this many rows comes back wrong)
    return (torch.cat([position[o] for o in parts]),
            None if normal is None else torch.cat([normal[o] for o in parts]))


def _poses(count, radius, host):
    rows = []
    for _ in range(count):
        az, el = host.uniform(0.0, 2.0 * math.pi), host.uniform(math.radians(10.0), math.radians(35.0))
        rows.append(scenes.look_at_view((radius * math.cos(el) * math.sin(az), radius * math.sin(el),
                                         -radius * math.cos(el) * math.cos(az))))
    return np.stack(rows)


def _intrinsics(camera, w, h, seed):
    if camera == "fisheye":
        return scenes.ocam_row(w, h, seed)
    f = w * 1400.0 / 1920.0 if w > h else float(w)
    dist = [-0.06, 0.02, -0.003, 0.0, 0.0, 0.0, 4e-4, -3e-4] if camera == "distorted" else None
    return scenes.pinhole_row(f, f, w / 2, h / 2, dist=dist)


def _frame(case):
    """Size of the images the views are taken from."""
    return (1920, 1080) if case["crops"] else (case["w"], case["h"])


def prepare(case, seed):
    gc.collect()  # a render info and its cache refer to each other: the last scene's buffers go with this
    gen = torch.Generator(device="cuda").manual_seed(seed)
    host = np.random.default_rng(seed)
    position, normal, near = _points(case, seed, gen)
    if case["kind"] == "prepare":
        return {"case": case, "position": position, "normal": normal, "seed": seed}
    if case["kind"] == "filter":
        poses = torch.from_numpy(_poses(case["frames"], near, host)).cuda()
        intrinsics = torch.from_numpy(_intrinsics("distorted", 1920, 1080, seed)[None]).cuda()
        frames = [scenes.make_view(1920, 1080, image_index=f) for f in range(case["frames"])]
        return {"case": case, "position": position, "poses": poses, "intrinsics": intrinsics, "frames": frames}

    n, c, w, h = case["points"], case["channels"], case["w"], case["h"]
    if case["ordered"]:
        position, normal = _order(position, normal, seed)
    texture = torch.rand(c, n, generator=gen, device="cuda")
    if case["half"]:
        texture = texture.half()
    fw, fh = _frame(case)
    model = _MODELS[case["camera"]]
    views = []
    if case["crops"]:  # as many frames as crops per frame; a crop is a window of 1/zoom of its size in the frame
        per_frame = int(math.isqrt(case["views"]))
        for i in range(case["views"]):
            zoom = float(host.uniform(0.75, 1.5))
            x0, y0 = float(host.uniform(0, fw - w / zoom)), float(host.uniform(0, fh - h / zoom))
            views.append(scenes.make_view(w, h, image_index=i // per_frame, model=model,
                                          crop=(zoom, zoom, -x0 * zoom, -y0 * zoom, 0.0)))
        frames = (case["views"] + per_frame - 1) // per_frame
    else:
        frames = case["views"]
        views = [scenes.make_view(w, h, image_index=i, model=model) for i in range(frames)]
    scene = render.NeuralScene(
        render.NeuralPointCloud(position, normal, torch.arange(n, dtype=torch.int32, device="cuda")), texture,
        torch.rand(c, generator=gen, device="cuda"), torch.from_numpy(_poses(frames, near * case.get("distance", 1.0), host)),
        torch.from_numpy(_intrinsics(case["camera"], fw, fh, seed)[None]),
        environment_map=torch.rand(c, *_ENV_SIZE, generator=gen, device="cuda") if case["env"] else None)
    step = case["kind"] == "step"
    params = scenes.default_params(
        check_normal=1 if normal is not None else 0, ghost_gradients=1 if case["dropout"] else 0,
        drop_out_points_by_radius=1 if case["lod"] else 0, output_background_mask=1 if case["env"] else 0,
        dist_cutoff=math.radians(5.0) if case["camera"] == "fisheye" else 1.0e4)
    dropout = None
    if case["dropout"]:
        dropout = torch.empty(case["views"], n, device="cuda").bernoulli_(0.25, generator=gen)
    info = render.NeuralRenderInfo(scene=scene, images=views, params=params, num_layers=case["levels"],
                                   cache=render.PointRendererCache(), dropout_points=dropout, train=step)
    state = {"case": case, "info": info}
    if step:
        state["leaves"] = [scene.texture, scene.background_color, scene.point_cloud_cuda.t_position, scene.tangent_poses,
                           scene.intrinsics]
        for t in state["leaves"]:
            t.requires_grad_(True)
        state["grads"] = [torch.randn(case["views"], c, h >> l, w >> l, generator=gen, device="cuda")
                          for l in range(case["levels"])]
    return state


# ---- one pass ---------------------------------------------------------------------------------------------------

def run(state):
    case = state["case"]
    if case["kind"] == "prepare":
        position, normal, data, order = preprocess.PreprocessPointCloud(state["position"], state["normal"],
                                                                        seed=state["seed"])
        return [position, data, order] + ([] if normal is None else [normal])
    if case["kind"] == "filter":
        ids = preprocess.FilterPointCloud(state["position"], state["poses"], state["intrinsics"], state["frames"])
        keep = torch.zeros(case["points"], dtype=torch.bool, device="cuda")
        keep[ids] = True
        return keep
    info, levels = state["info"], case["levels"]
    if case["kind"] == "view":
        with torch.no_grad():
            out = render.BlendPointCloud(info)
            if case["env"]:
                render.EnvironmentMapSample(info, add_to_out=True)
        return out
    out = render.BlendPointCloud(info)
    for mask in out[levels:]:
        mask.detach_()  # what was left uncovered carries no gradient
    result = [t.detach() for t in out]
    if case["env"]:
        with torch.no_grad():
            uv, composed = render.EnvironmentMapSample(info, add_to_out=2, want_uv=True)
            result[:levels] = composed
            result.append(render.EnvironmentMapSampleBackward(info, state["grads"], uv=uv))
    result += torch.autograd.grad(out[:levels], state["leaves"], state["grads"])
    info.cache.output_forward = []  # the images hold the graph, the graph holds info and with it this cache
    return result


def work(case):
    """Bytes and operations a pass cannot do without: every input read once, every output written once.

    A point is a position, and a packed normal where the back-face test reads it.  Descriptors are read for at most one
    point per pixel of the finest level and view; the dropout flags of a batch of crops, which see a small part of the
    cloud, are left out.  Operations: the projection of every point into every view."""
    n = case["points"]
    point = 16 + (4 if case["normals"] else 0)
    if case["kind"] == "prepare":
        return {"bytes": n * (2 * point + 16 + 8), "flops": n * 60 * 8}
    if case["kind"] == "filter":
        return {"bytes": n * (16 + 8), "flops": n * (case["frames"] * 45 + 2 * 60 * 8)}
    b, c = case["views"], case["channels"]
    pixels = b * sum((case["w"] >> l) * (case["h"] >> l) for l in range(case["levels"]))
    seen = min(n, b * case["w"] * case["h"])
    frames = int(math.isqrt(b)) if case["crops"] else b
    total = n * point + seen * c * (2 if case["half"] else 4) + pixels * c * 4
    flops = n * frames * (120 if case["camera"] == "fisheye" else 60)
    if case["env"]:
        total += pixels * 4 + c * _ENV_SIZE[0] * _ENV_SIZE[1] * 4
        flops += pixels * 60
    if case["kind"] == "step":
        total += pixels * c * 4  # upstream gradients
        total += n * c * (2 if case["half"] else 4) + n * 16  # descriptor and point gradients
        if case["dropout"] and not case["crops"]:
            total += n * b * 4
        if case["env"]:
            total += c * _ENV_SIZE[0] * _ENV_SIZE[1] * 4
        flops *= 2
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """About four times what the sums in another order show (the two forward paths of the library against each other and
    against themselves): images 4e-8 to 8e-8, gradients 3e-7 to 5e-7."""
    if case["kind"] in ("prepare", "filter"):
        return "exact"  # orders, ids, and distances of given pairs of points
    if case["kind"] == "view":
        return {"rel": 3e-7}
    # (gradients of half descriptors are rounded to halves: a sum next to the middle of two may go to either)
    return {"rel": 3e-5 if case["half"] else 2e-6}

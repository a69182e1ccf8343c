"""The work that users of this package have it do, as cases to time and to compare.

Each case is one pass through the public ops as a program calls them: a whole fitting step
(render, loss, gradients), a frame of a viewer, or a single op forward and backward on inputs
rendered beforehand. ``draw`` gives more cases of the same kinds over the sizes they are used at.
``exact`` computes a case in float64 with plain torch.
"""

import functools
import math

import torch
import torch.nn.functional as F

import diffrast_amd as dr
from diffrast_amd import workloads as wl

DEVICE = torch.device("cuda", 0)


def listed():
    return [
        # Fitting the colours and shape of a small object at thumbnail size, the first thing a
        # program using a differentiable renderer does (the "sphere" workload): latency-bound.
        dict(name="fit small", kind="fit", mesh="sphere", detail=32, noise=0.0, batch=1,
             height=256, width=256, channels=3, tex=0),
        # Fitting a texture and the vertices from a few views per step (the "textured" workload).
        dict(name="fit textured", kind="fit", mesh="icosphere", detail=5, noise=0.0, batch=4,
             height=512, width=512, channels=0, tex=512, tex_channels=3),
        # The same for a dense scan with vertex colours (the "large" workload's mesh and images).
        dict(name="fit large", kind="fit", mesh="icosphere", detail=8, noise=0.02, batch=8,
             height=1024, width=1024, channels=4, tex=1024, tex_channels=4),
        # A viewer's frame: full HD, mip levels built once, no gradients (the benchmark grid).
        dict(name="frame", kind="frame", mesh="grid", detail=100_000, noise=0.0, batch=1,
             height=1080, width=1920, tex=1024, tex_channels=3),
        # Rasterizing a mid-sized mesh from several cameras at an odd size, both outputs'
        # gradients back to the vertices (normals or footprints in the loss).
        dict(name="rasterize odd", kind="rasterize", mesh="icosphere", detail=7, noise=0.02,
             batch=5, height=601, width=803, grad=True),
        # A few large triangles on a 4K image: proxies, skies, user-interface planes.
        dict(name="rasterize coarse", kind="rasterize", mesh="sphere", detail=8, noise=0.0,
             batch=1, height=2160, width=3840, grad=True),
        # Depth layers of many small items, one range of triangles each (transparency; the
        # "instances" workload at a quarter of its items and half its image size).
        dict(name="peel items", kind="peel", mesh="icosphere", detail=4, noise=0.0, items=64,
             height=256, width=256, layers=4),
        # Deferred shading of learned per-vertex features.
        dict(name="features", kind="interpolate", mesh="icosphere", detail=6, noise=0.0, batch=4,
             height=512, width=512, channels=16, diff=False, shared=True),
        # A learned multi-channel texture, trilinear with its mip chain built in the call.
        dict(name="neural texture", kind="texture", mesh="grid", detail=20_000, noise=0.0,
             batch=2, height=720, width=1280, tex_height=1024, tex_width=1024, tex_channels=16,
             filter="linear-mipmap-linear", boundary="wrap"),
        # A photograph sampled bilinearly with clamped borders (no mip chain), RGB.
        dict(name="photo texture", kind="texture", mesh="grid", detail=10_000, noise=0.0,
             batch=1, height=1080, width=1920, tex_height=1365, tex_width=2047, tex_channels=3,
             filter="linear", boundary="clamp"),
        # Environment lighting from a cube map, mipmapped (the "cubemap" workload's sizes).
        dict(name="environment", kind="texture", mesh="knot", detail=32, noise=0.0, batch=4,
             height=1024, width=1024, tex_height=512, tex_width=512, tex_channels=3,
             filter="linear-mipmap-linear", boundary="cube"),
        # Antialiasing alone, RGB images of a thin, self-occluding shape at an odd size.
        dict(name="antialias", kind="antialias", mesh="knot", detail=32, noise=0.0, batch=4,
             height=1001, width=999, channels=3),
    ]


# ---- drawn cases --------------------------------------------------------------------------------


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _mesh(rng):
    mesh = rng.choice(["sphere", "icosphere", "grid", "knot"])
    if mesh == "icosphere":
        return dict(mesh=mesh, detail=rng.randint(3, 8), noise=rng.choice([0.0, 0.02]))
    detail = {"sphere": _log(rng, 8, 128), "grid": _log(rng, 100, 1_000_000),
              "knot": _log(rng, 4, 96)}[mesh]
    return dict(mesh=mesh, detail=detail, noise=0.0)


def _images(rng, most=8 << 20):
    """A batch of images of 64 to 2048 pixels a side, no more than ``most`` pixels in all."""
    while True:
        batch, height = _log(rng, 1, 8), _log(rng, 64, 2048)
        width = height if rng.random() < 0.5 else max(64, min(3840, _log(rng, height / 2,
                                                                         2 * height)))
        if batch * height * width <= most:
            return dict(batch=batch, height=height, width=width)


def draw(rng):
    kind = rng.choice(["fit", "fit", "frame", "rasterize", "peel", "interpolate", "interpolate",
                       "texture", "texture", "antialias", "antialias"])
    if kind == "peel":
        side = _log(rng, 64, 512)
        return dict(kind=kind, mesh="icosphere", detail=rng.randint(1, 4), noise=0.0,
                    items=max(1, min(_log(rng, 4, 256), (4 << 20) // side ** 2)), height=side,
                    width=side, layers=rng.randint(1, 4))
    case = dict(kind=kind, **_mesh(rng))
    if kind == "fit":
        case.update(_images(rng, 4 << 20))
        tex = rng.choice([0, _log(rng, 64, 1024), 1024])
        channels = rng.choice([1, 3, 4])
        case.update(channels=channels if tex == 0 or rng.random() < 0.5 else 0, tex=tex)
        if tex:
            case.update(tex_channels=channels)
        return case
    case.update(_images(rng))
    if kind == "frame":
        case.update(tex=_log(rng, 64, 2048), tex_channels=rng.choice([3, 4]))
    elif kind == "rasterize":
        case.update(grad=rng.random() < 0.7)
    elif kind == "interpolate":
        channels = _log(rng, 1, 32)
        while case["batch"] * case["height"] * case["width"] * channels > 64 << 20:
            channels = max(1, channels // 2)
        case.update(channels=channels, diff=channels <= 4 and rng.random() < 0.5,
                    shared=rng.random() < 0.7)
    elif kind == "texture":
        boundary = rng.choice(["wrap", "wrap", "clamp", "zero", "cube"])
        side = _log(rng, 32, 512 if boundary == "cube" else 2048)
        channels = _log(rng, 1, 16)
        while case["batch"] * case["height"] * case["width"] * channels > 32 << 20:
            channels = max(1, channels // 2)
        case.update(tex_height=side,
                    tex_width=side if boundary == "cube" or rng.random() < 0.6
                    else _log(rng, 32, 2048), tex_channels=channels,
                    filter=rng.choice(["linear-mipmap-linear", "linear-mipmap-linear", "linear",
                                       "linear-mipmap-nearest", "nearest"]), boundary=boundary)
    else:
        case.update(channels=rng.choice([1, 3, 3, 4, 8]))
    return case


# ---- inputs -------------------------------------------------------------------------------------


@functools.lru_cache(maxsize=32)
def _base_mesh(mesh, detail):
    """Vertices, triangles and texture coordinates on the CPU."""
    if mesh == "grid":
        verts, tri, n = wl.displaced_grid(detail)
        return verts, tri, wl.grid_uv(n)
    if mesh == "sphere":
        verts, tri = wl.uv_sphere(detail, 2 * detail)
    elif mesh == "icosphere":
        verts, tri = wl.icosphere(detail)
    else:
        verts, tri = wl.torus_knot(2, 3, 16 * detail, detail)
    return verts, tri, wl.spherical_uv(verts)


def _scene(case, seed):
    """Clip-space positions of a batch of views, indices and texture coordinates on the GPU."""
    verts, tri, uv = _base_mesh(case["mesh"], case["detail"])
    cpu = torch.Generator().manual_seed(seed)
    if case["mesh"] == "grid":
        # The benchmark's cameras, each seed's grid turned by an angle of its own.
        turn = 2 * math.pi * float(torch.rand((), generator=cpu))
        c, s = math.cos(turn), math.sin(turn)
        verts = torch.stack([c * verts[:, 0] + s * verts[:, 2], verts[:, 1],
                             c * verts[:, 2] - s * verts[:, 0]], -1)
        eyes, pos = None, wl.grid_views(verts, case["batch"])
    else:
        if case["noise"]:
            verts = verts * (1 + case["noise"] * torch.randn(verts.shape[0], 1, generator=cpu))
        eyes = wl.random_eyes(case["batch"], 3.0, cpu)
        pos = wl.clip_positions(verts, eyes, case["width"] / case["height"])
    gen = torch.Generator(DEVICE).manual_seed(seed)
    return dict(case=case, gen=gen, eyes=eyes, verts=verts, pos=pos.to(DEVICE),
                tri=tri.to(DEVICE), uv=uv.to(DEVICE), size=(case["height"], case["width"]),
                ctx=dr.RasterizeContext(DEVICE))


def _rand(s, *shape):
    return torch.rand(*shape, generator=s["gen"], device=DEVICE)


def _randn(s, *shape):
    return torch.randn(*shape, generator=s["gen"], device=DEVICE)


def _items(case, seed):
    """Small objects scattered in front of one camera; item i draws objects i to i + 3."""
    cpu = torch.Generator().manual_seed(seed)
    verts, faces, _ = _base_mesh(case["mesh"], case["detail"])
    count = case["items"]
    offset = torch.rand(count, 1, 3, generator=cpu) * 2 - 1
    scale = torch.rand(count, 1, 1, generator=cpu) * 0.3 + 0.2
    world = (verts[None] * scale + offset).reshape(-1, 3)
    tri = (faces[None] + torch.arange(count)[:, None, None] * verts.shape[0]).reshape(-1, 3)
    per = faces.shape[0]
    ranges = torch.tensor([[per * i, per * min(4, count - i)] for i in range(count)],
                          dtype=torch.int32)
    pos = wl.clip_positions(world, wl.random_eyes(1, 4.0, cpu), 1.0)[0]
    return dict(case=case, pos=pos.to(DEVICE), tri=tri.to(torch.int32).to(DEVICE), ranges=ranges,
                size=(case["height"], case["width"]), ctx=dr.RasterizeContext(DEVICE))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "peel":
        return _items(case, seed)
    s = _scene(case, seed)
    b, (h, w), v = case["batch"], s["size"], s["uv"].shape[0]
    if kind in ("fit", "frame"):
        channels = case.get("channels") or case["tex_channels"]
        if case["tex"]:
            s["tex"] = _rand(s, 1, case["tex"], case["tex"], channels)
        if kind == "frame":
            s["mip"] = dr.texture_construct_mip(s["tex"])
            return s
        s["pos"].requires_grad_()
        s["leaves"] = [s["pos"]]
        if case["channels"]:
            s["attr"] = _rand(s, 1, v, channels).requires_grad_()
            s["leaves"].append(s["attr"])
        if case["tex"]:
            s["leaves"].append(s["tex"].requires_grad_())
        s["target"] = _rand(s, b, h, w, channels)
        return s
    if kind == "rasterize":
        if case["grad"]:
            s["pos"].requires_grad_()
            s["grads"] = [_randn(s, b, h, w, 4), _randn(s, b, h, w, 4)]
        return s
    rast, rast_db = dr.rasterize(s["ctx"], s["pos"], s["tri"], s["size"])
    if kind == "interpolate":
        c = case["channels"]
        shape = (1, v, c) if case["shared"] else (b, v, c)
        s.update(attr=_randn(s, *shape).requires_grad_(), rast=rast.requires_grad_(),
                 rast_db=rast_db.requires_grad_() if case["diff"] else None,
                 grads=[_randn(s, b, h, w, c)])
        if case["diff"]:
            s["grads"].append(_randn(s, b, h, w, 2 * c))
    elif kind == "texture":
        th, tw, c = case["tex_height"], case["tex_width"], case["tex_channels"]
        mip = "mipmap" in case["filter"]
        if case["boundary"] == "cube":
            normals = wl.vertex_normals(s["verts"], s["tri"].cpu()).to(DEVICE)
            uv, uv_da = dr.interpolate(normals, rast, s["tri"], rast_db, "all")
            if s["eyes"] is not None and h * w <= 1 << 20:  # mirror reflections
                view, view_da = (t.to(DEVICE) for t in _rays(case, seed))
                uv, uv_da = wl.reflect(view, view_da, uv, uv_da)
        else:
            uv, uv_da = dr.interpolate(s["uv"], rast, s["tri"], rast_db, "all")
        shape = (1, 6, th, tw, c) if case["boundary"] == "cube" else (1, th, tw, c)
        s.update(tex=_rand(s, *shape).requires_grad_(),
                 sample_uv=uv.contiguous().requires_grad_(),
                 uv_da=uv_da.contiguous().requires_grad_() if mip else None,
                 grads=[_randn(s, b, h, w, c)])
    else:
        colours = _rand(s, 1, v, case["channels"])
        s.update(rast=rast, color=dr.interpolate(colours, rast, s["tri"])[0].requires_grad_(),
                 grads=[_randn(s, b, h, w, case["channels"])])
        s["pos"].requires_grad_()
    return s


@functools.lru_cache(maxsize=4)
def _rays_of(batch, height, width, eyes):
    return wl.view_rays(torch.tensor(eyes).view(batch, 3), height, width)


def _rays(case, seed):
    eyes = wl.random_eyes(case["batch"], 3.0, torch.Generator().manual_seed(seed + 1))
    return _rays_of(case["batch"], case["height"], case["width"], tuple(eyes.flatten().tolist()))


# ---- one pass -----------------------------------------------------------------------------------


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "fit":
        color = None
        rast, rast_db = dr.rasterize(s["ctx"], s["pos"], s["tri"], s["size"])
        if case["channels"]:
            color, _ = dr.interpolate(s["attr"], rast, s["tri"])
        if case["tex"]:
            uv, uv_da = dr.interpolate(s["uv"], rast, s["tri"], rast_db, "all")
            texel = dr.texture(s["tex"], uv, uv_da, filter_mode="linear-mipmap-linear")
            color = texel if color is None else color + texel
        image = dr.antialias(color, rast, s["pos"], s["tri"])
        loss = F.mse_loss(image, s["target"])
        return [image.detach(), *torch.autograd.grad(loss, s["leaves"])]
    if kind == "frame":
        with torch.no_grad():
            rast, rast_db = dr.rasterize(s["ctx"], s["pos"], s["tri"], s["size"])
            uv, uv_da = dr.interpolate(s["uv"], rast, s["tri"], rast_db, "all")
            color = dr.texture(s["tex"], uv, uv_da, mip=s["mip"],
                               filter_mode="linear-mipmap-linear")
            return [dr.antialias(color, rast, s["pos"], s["tri"])]
    if kind == "rasterize":
        rast, rast_db = dr.rasterize(s["ctx"], s["pos"], s["tri"], s["size"])
        outs = [rast, rast_db]
        grads = torch.autograd.grad(outs, [s["pos"]], s["grads"]) if case["grad"] else ()
    elif kind == "peel":
        outs, grads = [], ()
        with dr.DepthPeeler(s["ctx"], s["pos"], s["tri"], s["size"], s["ranges"]) as peeler:
            for _ in range(case["layers"]):
                outs.append(peeler.rasterize_next_layer()[0])
    elif kind == "interpolate":
        out, out_da = dr.interpolate(s["attr"], s["rast"], s["tri"], s["rast_db"],
                                     "all" if case["diff"] else None)
        outs, leaves = [out], [s["attr"], s["rast"]]
        if case["diff"]:
            outs.append(out_da)
            leaves.append(s["rast_db"])
        grads = torch.autograd.grad(outs, leaves, s["grads"])
    elif kind == "texture":
        outs = [dr.texture(s["tex"], s["sample_uv"], s["uv_da"], filter_mode=case["filter"],
                           boundary_mode=case["boundary"])]
        grads = torch.autograd.grad(outs, _texture_leaves(s), s["grads"])
    else:
        outs = [dr.antialias(s["color"], s["rast"], s["pos"], s["tri"])]
        grads = torch.autograd.grad(outs, [s["color"], s["pos"]], s["grads"])
    return [t.detach() for t in outs] + list(grads)


def _texture_leaves(s):
    leaves = [s["tex"]]
    if s["case"]["filter"] != "nearest":
        leaves.append(s["sample_uv"])
    # The footprint moves the result only where two levels are blended.
    if s["case"]["filter"] == "linear-mipmap-linear":
        leaves.append(s["uv_da"])
    return leaves


# ---- what a pass cannot do without --------------------------------------------------------------


def _counts(case):
    verts, tri, _ = _base_mesh(case["mesh"], case["detail"])
    return verts.shape[0], tri.shape[0]


def work(case):
    """Bytes of each op's inputs read once and outputs written once (the ops hand each other
    whole images, so those count where they leave one op and where they enter the next), and a
    count of the arithmetic per pixel and triangle."""
    v, t = _counts(case)
    kind = case["kind"]
    if kind == "peel":
        n, layers = case["items"], case["layers"]
        pixels = n * case["height"] * case["width"]
        return dict(bytes=layers * (n * (v * 16 + t * 12) + pixels * 32),
                    flops=layers * (4 * n * t * 100 + pixels * 100))
    b = case["batch"]
    pixels = b * case["height"] * case["width"]
    geometry = b * v * 16 + t * 12
    bytes_, flops = 0, 0
    if kind in ("fit", "frame", "rasterize"):
        bytes_ += geometry + 32 * pixels  # rast and rast_db
        flops += b * t * 100 + pixels * 100
        if kind == "fit" or case.get("grad"):
            bytes_ += geometry + b * v * 16 + (32 if kind == "rasterize" or case["tex"] else 16) * pixels
            flops += pixels * 200
    if kind == "interpolate":
        c, d = case["channels"], case["channels"] if case["diff"] else 0
        table = (1 if case["shared"] else b) * v * c * 4 + t * 12
        image = pixels * (16 + (16 if d else 0))
        bytes_ += 2 * (table + image + pixels * 4 * (c + 2 * d)) + table + image
        flops += pixels * (16 * c + 20 * d)
    tex = case.get("tex") or 0
    if kind in ("fit", "frame"):
        passes = 2 if kind == "fit" else 1
        c = case.get("channels") or 0
        if c:
            bytes_ += (passes + 1) * (v * c * 4 + pixels * 16) + 2 * t * 12 + 2 * pixels * c * 4
        if tex:
            c = case["tex_channels"]
            # uv with derivatives forward, their gradients' way back, and the lookup both ways
            bytes_ += passes * (pixels * (32 + 24) + v * 8 + t * 12) + (passes - 1) * pixels * 32
            bytes_ += passes * (pixels * (24 + 4 * c) + tex * tex * c * 4 * 4 // 3)
            bytes_ += (passes - 1) * (pixels * 24 + tex * tex * c * 4)
            flops += passes * pixels * (100 + 20 * c)
        c = case.get("channels") or case["tex_channels"]
        bytes_ += passes * (2 * pixels * c * 4 + pixels * 16 + geometry)
        bytes_ += (passes - 1) * (2 * pixels * c * 4 + b * v * 16)
        flops += passes * pixels * (50 + 10 * c)
    if kind == "texture":
        c = case["tex_channels"]
        cube = case["boundary"] == "cube"
        texels = case["tex_height"] * case["tex_width"] * (6 if cube else 1)
        coords = (12 if cube else 8)
        if "mipmap" in case["filter"]:
            coords += 24 if cube else 16
        bytes_ += 3 * pixels * coords + 2 * pixels * c * 4 + 3 * texels * c * 4
        flops += pixels * (200 + 40 * c)
    if kind == "antialias":
        c = case["channels"]
        bytes_ += pixels * (4 * c * 4 + 2 * 16) + 3 * b * v * 16 + 2 * t * 12
        flops += pixels * (100 + 20 * c)
    return dict(bytes=bytes_, flops=flops)


def tolerance(case):
    """About four times the distance from ``exact`` that float32 shows: the sums alone round to
    1e-7 or better; what is larger comes from thin triangles (barycentrics, their derivatives and
    crossings divide by small areas) and from texel coordinates, whose rounding moves a few
    pixels to another texel cell, where the gradient of a noise texture is another one."""
    kind = case["kind"]
    if kind in ("peel", "interpolate"):
        return dict(rel=1e-5, max=1e-3)
    if kind in ("texture", "antialias"):
        return dict(rel=1e-3, max=0.5)
    if kind == "frame" or (kind == "fit" and not case["tex"]):
        return dict(rel=4e-3, max=0.9)
    return dict(rel=3e-2, max=0.9)


# ---- float64 ------------------------------------------------------------------------------------
#
# Which triangle a pixel shows, which edge a pair of pixels crosses and which texel cell a
# coordinate falls in are whole numbers that the float32 operations of the definition decide:
# they are taken in float32. Everything computed from them is float64, its gradients by autograd.

_PAIRS = 1 << 25  # (triangle, pixel) pairs tested at once
EPS = 2.0 ** -23


def _centres(n, dtype):
    return (torch.arange(n, dtype=dtype, device=DEVICE) * 2 + 1) / n - 1


def _edges(x, y, w, px, py):
    """a, c and the edge functions e of triangles [n, 3] at centres [n]."""
    a, c = x - px[:, None] * w, y - py[:, None] * w
    i, j = [1, 2, 0], [2, 0, 1]
    return a, c, a[:, i] * c[:, j] - a[:, j] * c[:, i]


def _covered(corners, px, py):
    """Whether triangles [n, 3, 4] cover centres [n], and their depth there, in float32."""
    x, y, z, w = corners.unbind(-1)
    a, c, e = _edges(x, y, w, px, py)
    area = e[:, 0] + e[:, 1] + e[:, 2]
    ew = e[:, 0] * w[:, 0] + e[:, 1] * w[:, 1] + e[:, 2] * w[:, 2]
    depth = (e[:, 0] * z[:, 0] + e[:, 1] * z[:, 1] + e[:, 2] * z[:, 2]) / ew
    front = area > 0
    ok = torch.where(front, ew > 0, ew < 0) & (depth >= -1) & (depth <= 1)
    for k in range(3):
        i, j = (k + 1) % 3, (k + 2) % 3
        gx, gy = c[:, i] * w[:, j] - c[:, j] * w[:, i], a[:, j] * w[:, i] - a[:, i] * w[:, j]
        side = torch.where(e[:, k] == 0, torch.where(gx == 0, gy, gx), e[:, k])
        ok &= torch.where(front, side > 0, side < 0)
    reach_x, reach_y = (x.abs() + w.abs()).amax(1), (y.abs() + w.abs()).amax(1)
    a, c = a.abs(), c.abs()
    span_x, span_y = a[:, 0] + a[:, 1] + a[:, 2], c[:, 0] + c[:, 1] + c[:, 2]
    ok &= area.abs() > (reach_x * span_y + span_x * (reach_y + span_y)) * (2 * EPS)
    return ok, depth


def _visible(pos, tri, image, rows, batch, size, previous=None):
    """Keys [batch * h * w] (depth above triangle row, as ordered int64) of the nearest triangle
    among the instances (image, row of tri), behind ``previous``."""
    h, w = size
    none = torch.iinfo(torch.int64).max
    best = torch.full((batch * h * w,), none, device=DEVICE)
    px, py = _centres(w, torch.float32), _centres(h, torch.float32)
    corners = pos[image[:, None] if pos.shape[0] > 1 else 0, tri[rows]]
    ndc = corners[..., :2].double() / corners[..., 3:].double()
    limit = torch.tensor([w, h], device=DEVICE)
    at = (ndc + 1) * limit / 2 - 0.5
    low = (at.amin(1) - 0.1).ceil().clamp(min=0).minimum(limit + 0.0).long()
    high = (at.amax(1) + 0.1).floor().clamp(min=-1).minimum(limit - 1.0).long()
    extent = (high - low + 1).clamp(min=0)
    ends = extent.prod(1).cumsum(0)
    start, n = 0, rows.shape[0]
    while start < n:
        before = int(ends[start - 1]) if start else 0
        stop = int(torch.searchsorted(ends, before + _PAIRS, right=True))
        stop = min(n, max(stop, start + 1))
        count = extent[start:stop].prod(1)
        who = torch.repeat_interleave(torch.arange(start, stop, device=DEVICE), count)
        cell = torch.arange(who.shape[0], device=DEVICE) - (ends[who] - extent[who].prod(1) - before)
        col = low[who, 0] + cell % extent[who, 0]
        row = low[who, 1] + cell // extent[who, 0]
        ok, depth = _covered(corners[who], px[col], py[row])
        bits = (depth + 0.0).view(torch.int32).long()
        key = (torch.where(bits < 0, -1 - bits - (1 << 31), bits) << 32) | rows[who]
        pixel = (image[who] * h + row) * w + col
        if previous is not None:
            ok &= key > previous[pixel]
        best.scatter_reduce_(0, pixel[ok], key[ok], "amin")
        start = stop
    return best


def _shown(keys, shape):
    """Triangle rows [batch, h, w], -1 for background."""
    return torch.where(keys == torch.iinfo(torch.int64).max, -1, keys & 0xffffffff).view(shape)


def _instanced_ids(s):
    pos, tri = s["pos"].detach(), s["tri"].long()
    b, t = pos.shape[0], tri.shape[0]
    image = torch.arange(b, device=DEVICE).repeat_interleave(t)
    rows = torch.arange(t, device=DEVICE).repeat(b)
    return _shown(_visible(pos, tri, image, rows, b, s["size"]), (b, *s["size"]))


def _resolve64(pos, tri, ids):
    b, h, w = ids.shape
    at = (ids >= 0).nonzero(as_tuple=True)
    image = at[0] if pos.shape[0] > 1 else torch.zeros_like(at[0])
    x, y, z, ww = pos[image[:, None], tri[ids[at]]].unbind(-1)
    a, c, e = _edges(x, y, ww, _centres(w, torch.float64)[at[2]], _centres(h, torch.float64)[at[1]])
    area = e.sum(1, keepdim=True)
    bary = e / area
    depth = (bary * z).sum(1) / (bary * ww).sum(1)
    dx, dy = torch.linalg.cross(c, ww, dim=1), torch.linalg.cross(ww, a, dim=1)
    dx = (dx - bary * dx.sum(1, keepdim=True)) / area * (2 / w)
    dy = (dy - bary * dy.sum(1, keepdim=True)) / area * (2 / h)
    rast = torch.stack([bary[:, 0], bary[:, 1], depth, (ids[at] + 1).double()], -1)
    db = torch.stack([dx[:, 0], dy[:, 0], dx[:, 1], dy[:, 1]], -1)
    empty = pos.new_zeros(b, h, w, 4)
    return empty.index_put(at, rast), empty.index_put(at, db)


def _interpolate64(attr, rast, tri, rast_db, diff):
    ids = rast[..., 3].detach().round().long() - 1
    at = (ids >= 0).nonzero(as_tuple=True)
    image = at[0] if attr.shape[0] > 1 else torch.zeros_like(at[0])
    a0, a1, a2 = attr[image[:, None], tri[ids[at]]].unbind(1)
    u, v = rast[at][:, :1], rast[at][:, 1:2]
    empty = rast.new_zeros(*ids.shape, attr.shape[-1])
    out = empty.index_put(at, u * a0 + v * a1 + (1 - u - v) * a2)
    if not diff:
        return out, None
    db = rast_db[at][:, :, None]
    du, dv = a0 - a2, a1 - a2
    da = torch.stack([db[:, 0] * du + db[:, 2] * dv, db[:, 1] * du + db[:, 3] * dv], -1)
    return out, torch.cat([empty, empty], -1).index_put(at, da.flatten(1))


def _halve(image, dim):
    """n texels along ``dim`` into ceil(n / 2) equal bins by area."""
    n = image.shape[dim]
    m = (n + 1) // 2
    if n == 1:
        return image
    edge = torch.arange(m + 1, dtype=torch.float64, device=DEVICE) * n / m
    texel = torch.arange(n, dtype=torch.float64, device=DEVICE)
    share = torch.minimum(edge[1:, None], texel + 1) - torch.maximum(edge[:-1, None], texel)
    share = share.clamp(min=0) * m / n
    return torch.tensordot(image, share, dims=([dim], [1])).movedim(-1, dim)


_MAJOR = [[1, 0, 0], [-1, 0, 0], [0, 1, 0], [0, -1, 0], [0, 0, 1], [0, 0, -1]]
_S = [[0, 0, -1], [0, 0, 1], [1, 0, 0], [1, 0, 0], [1, 0, 0], [-1, 0, 0]]
_T = [[0, -1, 0], [0, -1, 0], [0, 0, 1], [0, 0, -1], [0, -1, 0], [0, -1, 0]]


def _axes(dtype):
    return (torch.tensor(t, dtype=dtype, device=DEVICE) for t in (_MAJOR, _S, _T))


def _project(d, d_da):
    """OpenGL cube face, face coordinates in [0, 1] and their derivatives of directions [n, 3]."""
    size = d.detach().abs()
    axis = torch.where((size[:, 0] >= size[:, 1]) & (size[:, 0] >= size[:, 2]), 0,
                       torch.where(size[:, 1] >= size[:, 2], 1, 2))
    face = 2 * axis + (d.detach().gather(1, axis[:, None])[:, 0] < 0)
    length = size.amax(1, keepdim=True)
    d = d / length
    major, s_axis, t_axis = (table[face] for table in _axes(d.dtype))
    ma = (d * major).sum(1, keepdim=True)
    ratio = torch.stack([(d * s_axis).sum(1), (d * t_axis).sum(1)], 1) / ma
    if d_da is None:
        return face, 0.5 * (ratio + 1), None
    da = (d_da / length).unflatten(1, (3, 2))
    dm, ds, dt = ((da * axis_[:, :, None]).sum(1) for axis_ in (major, s_axis, t_axis))
    return face, 0.5 * (ratio + 1), torch.cat([0.5 * (ds - ratio[:, :1] * dm) / ma,
                                               0.5 * (dt - ratio[:, 1:] * dm) / ma], 1)


def _fold(face, row, col, size):
    """A texel up to one step outside a cube face on the face it lies on, and whether there is
    one (there is none beyond a corner)."""
    major, s_axis, t_axis = _axes(torch.long)
    over_c, over_r = (col < 0) | (col >= size), (row < 0) | (row >= size)
    n = size[..., None]
    point = n * major[face] + (2 * col + 1 - size)[..., None] * s_axis[face] + \
        (2 * row + 1 - size)[..., None] * t_axis[face]
    point = torch.minimum(torch.maximum(point, -n), n) - (over_c | over_r)[..., None] * major[face]
    axis = point.abs().argmax(-1)
    face = 2 * axis + (point.gather(-1, axis[..., None])[..., 0] < 0)
    col = (((point * s_axis[face]).sum(-1) + size - 1) // 2).clamp(min=0)
    row = (((point * t_axis[face]).sum(-1) + size - 1) // 2).clamp(min=0)
    return face, row, col, ~(over_c & over_r)


def _level64(texels, h, w, offset, face, st, st32, boundary, linear):
    """A lookup [n, channels] in the levels of size (h, w) at texel ``offset``, per sample."""
    def axis(coord, coord32, n, shift):
        if boundary == "wrap":
            coord, coord32 = coord - coord32.floor().double(), coord32 - coord32.floor()
        x, x32 = coord * n - shift, coord32 * n - shift
        if boundary in ("clamp", "zero"):
            x = torch.minimum(x.clamp(min=-1), n.double())
            x32 = torch.minimum(x32.clamp(min=-1), n.float())
        return x, x32.floor().long()

    shift = 0.5 if linear else 0.0
    x, col = axis(st[:, 0], st32[:, 0], w, shift)
    y, row = axis(st[:, 1], st32[:, 1], h, shift)
    flat = texels.reshape(-1, texels.shape[-1])
    taps, corner = [], []
    for k in range(4 if linear else 1):
        r, c, f = row + k // 2, col + k % 2, face
        valid = torch.ones_like(r, dtype=torch.bool)
        corner.append(((r < 0) | (r >= h)) & ((c < 0) | (c >= w)))
        if boundary == "cube" and linear:
            f, r, c, valid = _fold(face, r, c, w)
        elif boundary == "wrap":
            r, c = r % h, c % w
        elif boundary == "zero":
            valid = (r >= 0) & (r < h) & (c >= 0) & (c < w)
        r, c = torch.minimum(r.clamp(min=0), h - 1), torch.minimum(c.clamp(min=0), w - 1)
        if f is not None:
            r = r + f * h
        taps.append(flat[offset + r * w + c] * valid[:, None])
    if not linear:
        return taps[0]
    fx, fy = (x - col)[:, None], (y - row)[:, None]
    weights = [(1 - fy) * (1 - fx), (1 - fy) * fx, fy * (1 - fx), fy * fx]
    out = sum(wt * tap for wt, tap in zip(weights, taps))
    if boundary == "cube":
        out = out + sum(wt * m[:, None] for wt, m in zip(weights, corner)) * sum(taps) / 3
    return out


def _texture64(tex, uv, uv_da, filter_mode, boundary):
    cube = boundary == "cube"
    mip = "mipmap" in filter_mode
    levels = [tex[0] if cube else tex]  # [faces, h, w, channels]
    while mip and max(levels[-1].shape[1:3]) > 1:
        levels.append(_halve(_halve(levels[-1], 1), 2))
    texels = torch.cat([level.reshape(-1, tex.shape[-1]) for level in levels])
    sizes = torch.tensor([[level.shape[1], level.shape[2], level.shape[:3].numel()]
                          for level in levels], device=DEVICE)
    offsets = sizes[:, 2].cumsum(0) - sizes[:, 2]
    shape = uv.shape[:3]
    coords = uv.reshape(-1, uv.shape[-1])
    da = None if uv_da is None else uv_da.reshape(-1, uv_da.shape[-1])
    live = torch.ones(coords.shape[0], dtype=torch.bool, device=DEVICE)
    if cube:  # a zero direction (background) selects nothing
        live = coords.detach().float().abs().amax(1) >= torch.finfo(torch.float32).tiny
    coords, da = coords[live], None if da is None else da[live]

    def place(c, d):
        if cube:
            face, c, d = _project(c, d)
        else:
            face = None
        if not mip:
            return face, c, torch.zeros_like(c[:, 0])
        n = sizes[0, [1, 1, 0, 0]].to(c.dtype)
        foot = d * n
        long = torch.maximum(foot[:, 0] ** 2 + foot[:, 2] ** 2, foot[:, 1] ** 2 + foot[:, 3] ** 2)
        return face, c, 0.5 * torch.log2(long.clamp(min=1e-30))

    face, st, lod = place(coords, da)
    with torch.no_grad():
        face, st32, lod32 = place(coords.float(), None if da is None else da.float())
        top = sizes.shape[0] - 1
        linear = filter_mode != "nearest"
        blend = filter_mode == "linear-mipmap-linear"
        lower = (lod32.clamp(0, top) + (0.0 if blend else 0.5)).floor().long()

    def level(k):
        return _level64(texels, sizes[k, 0], sizes[k, 1], offsets[k], face, st, st32, boundary,
                        linear)

    out = level(lower)
    if blend:
        part = (lod.clamp(0, top) - lower)[:, None]
        out = out * (1 - part) + level((lower + 1).clamp(max=top)) * part
    full = tex.new_zeros(live.shape[0], tex.shape[-1]).index_put((live,), out)
    return full.view(*shape, -1)


def _silhouettes(pos, tri):
    """Whether each edge [batch, triangles, 3] (opposite vertex k) bounds the shape as seen:
    shared by no second triangle, or with both of its triangles on one side of it."""
    start, end = tri[:, [1, 2, 0]].flatten(), tri[:, [2, 0, 1]].flatten()
    key = torch.minimum(start, end) << 32 | torch.maximum(start, end)
    _, group, count = torch.unique(key, return_inverse=True, return_counts=True)
    order = torch.argsort(group, stable=True)
    first = (count.cumsum(0) - count)[count == 2]
    partner = torch.full_like(key, -1)
    partner[order[first]], partner[order[first + 1]] = order[first + 1], order[first]
    out = []
    for p in pos[..., [0, 1, 3]]:
        line = torch.linalg.cross(p[start], p[end], dim=-1)

        def side(vertex):
            q = p[vertex]
            return torch.sign((line * q).sum(-1) * q[:, 2])

        opposite = tri.flatten()
        fold = side(opposite) * side(opposite[partner.clamp(min=0)]) > 0
        out.append(((partner < 0) | fold).view(-1, 3))
    return torch.stack(out)


def _exit(pos, tri, silhouette, image, rows, src, dst, horizontal, size):
    """Where (share of the way) the triangle shown at ``src`` ends towards ``dst``; found only
    at a silhouette edge that pairs along this axis handle."""
    has = (rows >= 0).nonzero()[:, 0]
    image, rows = image[has], rows[has]
    (sx, sy), (dx, dy) = ((px[has], py[has]) for px, py in (src, dst))
    with torch.no_grad():
        x, y, _, w = pos.float()[image[:, None], tri[rows]].unbind(-1)
        e0 = _edges(x, y, w, sx.float(), sy.float())[2]
        a, c, e1 = _edges(x, y, w, dx.float(), dy.float())
        i, j = [1, 2, 0], [2, 0, 1]
        rx, ry, a, c = x.abs() + w.abs(), y.abs() + w.abs(), a.abs(), c.abs()
        slack = ((rx[:, i] + a[:, i]) * c[:, j] + (rx[:, j] + a[:, j]) * c[:, i]
                 + ry[:, j] * a[:, i] + ry[:, i] * a[:, j]) * (4 * EPS)
        sign = torch.where(e0.sum(1, keepdim=True) < 0, -1.0, 1.0)
        crossed = (e1 * sign <= slack) & ((e0 - e1) * sign > 2 * slack)
        edge = torch.where(crossed, e0 / torch.where(crossed, e0 - e1, 1.0), math.inf).argmin(1)
        steep = (w[:, j] * y[:, i] - w[:, i] * y[:, j]).abs() * size[0] * torch.tensor(
            1 + 1e-4, device=DEVICE)
        flat = (x[:, j] * w[:, i] - x[:, i] * w[:, j]).abs() * size[1]
        along = (steep >= flat) if horizontal else (flat > steep)
        pick = edge[:, None]
        good = crossed.any(1) & silhouette[image, rows, edge] & along.gather(1, pick)[:, 0]
    has, image, rows, pick = has[good], image[good], rows[good], pick[good]
    x, y, _, w = pos[image[:, None], tri[rows]].unbind(-1)
    e0 = _edges(x, y, w, sx[good], sy[good])[2].gather(1, pick)[:, 0]
    e1 = _edges(x, y, w, dx[good], dy[good])[2].gather(1, pick)[:, 0]
    found = torch.zeros(src[0].shape[0], dtype=torch.bool, device=DEVICE)
    found[has] = True
    return found, pos.new_zeros(src[0].shape[0]).index_put((has,), e0 / (e0 - e1))


def _antialias64(color, rast, pos, tri):
    ids, depth = rast[..., 3].detach().round().long() - 1, rast[..., 2].detach().float()
    b, h, w = ids.shape
    silhouette = _silhouettes(pos.detach(), tri)
    px, py = _centres(w, torch.float32).double(), _centres(h, torch.float32).double()
    out = color
    for down, right in ((0, 1), (1, 0)):
        id_p, id_q = ids[:, :h - down, :w - right], ids[:, down:, right:]
        i, r, c = (id_p != id_q).nonzero(as_tuple=True)
        p, q = (i, r, c), (i, r + down, c + right)
        at_p, at_q = (px[c], py[r]), (px[c + right], py[r + down])
        common = (right == 1, (h, w))
        from_p, t_p = _exit(pos, tri, silhouette, i, ids[p], at_p, at_q, *common)
        from_q, t_q = _exit(pos, tri, silhouette, i, ids[q], at_q, at_p, *common)
        use_p = from_p & (~from_q | (depth[p] <= depth[q]))
        t = torch.where(use_p, t_p, 1 - t_q)[:, None]
        active = (from_p | from_q)[:, None]
        lend = color[q] - color[p]
        out = out.index_put(p, torch.where(active & (t < 0.5), (0.5 - t) * lend, 0.0), True)
        out = out.index_put(q, torch.where(active & (t >= 0.5), (0.5 - t) * lend, 0.0), True)
    return out


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    tri = s["tri"].long()

    def leaf(name):
        t = s.get(name)
        return None if t is None else t.detach().double().requires_grad_(t.requires_grad)

    if kind == "peel":
        pos, h, w = s["pos"], *s["size"]
        image = torch.cat([torch.full((n,), k) for k, (_, n) in enumerate(s["ranges"].tolist())])
        rows = torch.cat([torch.arange(f, f + n) for f, n in s["ranges"].tolist()])
        keys, outs = None, []
        for _ in range(case["layers"]):
            keys = _visible(pos[None], tri, image.to(DEVICE), rows.to(DEVICE), case["items"],
                            (h, w), keys)
            ids = _shown(keys, (case["items"], h, w))
            outs.append(_resolve64(pos.double()[None], tri, ids)[0])
        return outs
    pos = leaf("pos")
    if kind in ("fit", "frame", "rasterize"):
        rast, rast_db = _resolve64(pos, tri, _instanced_ids(s))
        if kind == "rasterize":
            outs, leaves = [rast, rast_db], [pos] if case["grad"] else []
    if kind in ("fit", "frame"):
        color, attr, tex = None, leaf("attr"), leaf("tex")
        if attr is not None:
            color, _ = _interpolate64(attr, rast, tri, None, False)
        if tex is not None:
            uv, uv_da = _interpolate64(s["uv"].double()[None], rast, tri, rast_db, True)
            texel = _texture64(tex, uv, uv_da, "linear-mipmap-linear", "wrap")
            color = texel if color is None else color + texel
        outs = [_antialias64(color, rast, pos, tri)]
        if kind == "frame":
            return outs
        loss = F.mse_loss(outs[0], s["target"].double())
        leaves = [t for t in (pos, attr, tex) if t is not None]
        return [outs[0].detach(), *torch.autograd.grad(loss, leaves)]
    if kind == "interpolate":
        attr, rast, rast_db = leaf("attr"), leaf("rast"), leaf("rast_db")
        outs = [t for t in _interpolate64(attr, rast, tri, rast_db, case["diff"])
                if t is not None]
        leaves = [t for t in (attr, rast, rast_db) if t is not None]
    elif kind == "texture":
        tex, uv, uv_da = leaf("tex"), leaf("sample_uv"), leaf("uv_da")
        outs = [_texture64(tex, uv, uv_da, case["filter"], case["boundary"])]
        s.update(tex=tex, sample_uv=uv, uv_da=uv_da)
        leaves = _texture_leaves(s)
    elif kind == "antialias":
        color = leaf("color")
        outs, leaves = [_antialias64(color, s["rast"].double(), pos, tri)], [color, pos]
    grads = []
    if leaves:
        grads = torch.autograd.grad(outs, leaves, [g.double() for g in s["grads"]])
    return [t.detach() for t in outs] + list(grads)

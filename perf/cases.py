"""Performance cases of the renderer: what its users run, through the public
entry points, from the smallest calls to the largest.

Five kinds of use, each over a range of sizes:

- frame: one view drawn call by call, as the reference's main loop does
  (clear, cull and draw, resolve), optionally with occlusion culling against
  the previous frame's depth map;
- gbuffer, overdraw: the deferred pipeline read back to the host, and the
  overdraw heat map;
- batch: many views as one launch (eager or one captured graph), with or
  without their resolves;
- fit: the differentiable resolve in texture fitting, forward and backward.

Scenes are grid patches laid out as in ``glimpsw_amd.scene.frame_1080p``
(triangle areas over three decades, half of them outside the view, one in
twenty patches straddling the camera plane), sized so that the depth
complexity stays about three, or in depth-stacked layers as in
``stress_views``. Every input is made from the seed.
"""
import math

import numpy as np
import torch

import glimpsw_amd as g
from glimpsw_amd import diff as D
from glimpsw_amd import scene as S
from glimpsw_amd import textures as TX

_CTX = None


def _context():
    """One context for the process, as a program on one GPU keeps it."""
    global _CTX
    if _CTX is None:
        torch.cuda.init()
        _CTX = g.Context(0)
    return _CTX


# ---------------------------------------------------------------- cases

def _frame(name, width, height, meshlets, **more):
    c = {"name": name, "kind": "frame", "width": width, "height": height, "meshlets": meshlets, "layout": "spread",
         "mode": "lit", "textures": 8, "tex_size": 512, "cutouts": False, "normal_maps": False, "sky": False,
         "occlusion": False}
    c.update(more)
    return c


def _batch(name, views, meshlets, scenes, width, height, **more):
    c = {"name": name, "kind": "batch", "views": views, "scenes": scenes, "meshlets": meshlets, "width": width,
         "height": height, "same_size": False, "layout": "spread", "mode": "none", "graph": True, "textures": 4,
         "tex_size": 256, "bin_size": 32, "bin_capacity": 4096, "raster_threads": 128}
    c.update(more)
    return c


def _fit(name, views, width, height, meshlets, textures, tex_size):
    return {"name": name, "kind": "fit", "views": views, "width": width, "height": height, "meshlets": meshlets,
            "textures": textures, "tex_size": tex_size, "cell_texels": 12.0}


def listed():
    return [
        # an icon or asset-browser preview: a handful of meshlets, all launch latency
        _frame("preview_96x64", 96, 64, 8, mode="albedo", textures=1, tex_size=64),
        # the interactive viewer at the size the tests render: 512 meshlets, lit
        _frame("viewer_640x480", 640, 480, 512, textures=1, tex_size=256),
        # the benchmark's frame: a million triangles at 1080p as one eager batch launch with its lit resolve
        _batch("frame_1080p", 1, 10240, 1, 1920, 1080, same_size=True, mode="lit", graph=False, textures=8,
               tex_size=1024, bin_capacity=2048, raster_threads=256),
        # the same frame call by call with the near-plane crossers inside the view: guard-band clipping, much overdraw
        _frame("crossers_1080p", 1920, 1080, 10240, layout="crossers"),
        # foliage and normal-mapped materials under a sky, at a ragged size (no multiple of the bins)
        _frame("cutouts_2044x1412", 2044, 1412, 6000, cutouts=True, normal_maps=True, sky=True),
        # a frame culled against the previous frame's depth pyramid, which it rebuilds
        _frame("occlusion_1280x720", 1280, 720, 16000, layout="layers", mode="albedo", occlusion=True),
        # the deferred pipeline feeding host code: draw, then the three G-buffer layers read back
        {"name": "gbuffer_960x540", "kind": "gbuffer", "width": 960, "height": 540, "meshlets": 2500,
         "layout": "spread", "textures": 4, "tex_size": 512, "cutouts": True, "normal_maps": True},
        # the overdraw heat map of a layered scene
        {"name": "overdraw_1600x900", "kind": "overdraw", "width": 1600, "height": 900, "meshlets": 8000,
         "layout": "layers", "textures": 1, "tex_size": 64},
        # dataset rendering: views of mixed sizes over several scenes, vis-buffers only, one graph
        _batch("views_24", 24, 8000, 3, 1600, 900),
        # close to the largest framebuffer, depth complexity about eight, lit, four cameras in one graph
        _batch("stress_4x2880x1620", 4, 24000, 1, 2880, 1620, same_size=True, layout="layers", mode="lit",
               textures=8, tex_size=512),
        # a small texture fit: one training step at thumbnail size
        _fit("fit_256x256", 1, 256, 256, 400, 2, 256),
        # the large fit: several cameras of one scene against a set of full-size textures
        _fit("fit_3x1280x720", 3, 1280, 720, 6000, 12, 1024),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    return max(4, 4 * (_log_int(rng, lo, hi) // 4))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "gbuffer", "overdraw", "batch", "batch", "fit", "fit"])
    if kind == "frame":
        occ = rng.random() < 0.25
        c = _frame("", _size(rng, 64, 2200), _size(rng, 64, 1450), _log_int(rng, 5, 12000),
                   layout="layers" if occ else rng.choice(["spread", "spread", "layers", "crossers"]),
                   mode=rng.choice(["lit", "lit", "albedo", "normals"]), textures=rng.randint(1, 8),
                   tex_size=rng.choice([64, 128, 256, 512]), cutouts=rng.random() < 0.4,
                   normal_maps=rng.random() < 0.4, sky=rng.random() < 0.4, occlusion=occ)
    elif kind in ("gbuffer", "overdraw"):
        c = {"kind": kind, "width": _size(rng, 64, 1600), "height": _size(rng, 64, 900),
             "meshlets": _log_int(rng, 5, 8000), "layout": rng.choice(["spread", "layers"]),
             "textures": rng.randint(1, 4), "tex_size": rng.choice([64, 128, 256, 512])}
        if kind == "gbuffer":
            c.update(cutouts=rng.random() < 0.5, normal_maps=rng.random() < 0.5)
    elif kind == "batch":
        width, height, meshlets = _size(rng, 128, 1920), _size(rng, 128, 1080), _log_int(rng, 20, 8000)
        # no more pixels and meshlets than the largest listed case
        views = max(1, min(_log_int(rng, 1, 24), int(15e6 / (width * height)), 80000 // meshlets))
        c = _batch("", views, meshlets, min(views, rng.randint(1, 3)), width, height,
                   same_size=rng.random() < 0.3, layout=rng.choice(["spread", "layers"]),
                   mode=rng.choice(["none", "lit", "albedo"]), graph=rng.random() < 0.6,
                   bin_size=rng.choice([16, 32]), bin_capacity=rng.choice([1024, 2048, 4096]),
                   raster_threads=rng.choice([128, 256]))
    else:
        c = _fit("", rng.randint(1, 3), _size(rng, 64, 1280), _size(rng, 64, 720), _log_int(rng, 20, 6000),
                 rng.randint(1, 12), rng.choice([64, 128, 256, 512, 1024]))
        c["cell_texels"] = round(math.exp(rng.uniform(math.log(2.0), math.log(64.0))), 2)
    c.pop("name", None)
    return c


# ---------------------------------------------------------------- inputs

def _rotations(rng, n):
    q = rng.normal(size=(n, 4))
    w, x, y, z = (q / np.linalg.norm(q, axis=1, keepdims=True)).T
    R = np.empty((n, 3, 3))
    R[:, 0] = np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y)], axis=1)
    R[:, 1] = np.stack([2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x)], axis=1)
    R[:, 2] = np.stack([2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], axis=1)
    return R


def _textures(rng, case):
    seed = int(rng.integers(1 << 30))
    size, out = case["tex_size"], []
    for i in range(case["textures"]):
        if case.get("normal_maps") and i % 2 == 0:
            out.append(TX.nmr_texture(size, seed + i))
        elif case.get("cutouts"):
            out.append(TX.cutout_texture(size, seed + i))
        else:
            out.append(TX.noise_texture(size, seed + i))
    return out


def _scene(rng, case, width, height):
    """Grid patches in front of a camera at the origin looking down -z."""
    n = case["meshlets"]
    aspect = width / height
    f = 1.0 / math.tan(math.radians(30.0))
    R = _rotations(rng, n)
    if case["layout"] == "layers":
        # depth-stacked layers, each covering the view about once; three
        # patches in ten with sub-pixel triangles
        layers = 8
        layer = np.sort(rng.integers(layers, size=n))
        depth = 2.0 * 1.35 ** layer.astype(np.float64)
        xy = rng.uniform(-1.05, 1.05, size=(2, n))
        depth_j = depth * (1.0 + rng.uniform(-0.05, 0.05, size=n))
        centers = np.stack([xy[0] * depth * aspect / f, xy[1] * depth / f, -depth_j], axis=1)
        scales = depth * 0.049 * math.sqrt(40960 / max(n, 1)) * rng.uniform(0.8, 1.25, size=n)
        scales[rng.random(n) < 0.3] /= 12.0
    else:
        # triangle areas log-uniform over three decades, scaled with the
        # pixels per patch of the 1080p frame with 10,240 of them
        area = np.exp(rng.uniform(math.log(0.5), math.log(500.0), size=n))
        area *= (width * height / (1920.0 * 1080.0)) * (10240.0 / max(n, 1))
        depth = np.exp(rng.uniform(0.0, math.log(60.0), size=n))
        ndc = rng.uniform(-2.0, 2.0, size=(2, n))
        scales = 7.0 * np.sqrt(2.0 * area) / ((height / 2.0) * f / depth)
        centers = np.stack([ndc[0] * depth * aspect / f, ndc[1] * depth / f, -depth], axis=1)
        near = rng.random(n) < 0.05
        k = int(near.sum())
        s = rng.uniform(0.5, 2.0, size=k)
        off = (0.5, 0.7) if case["layout"] == "crossers" else (0.85, 1.05)
        centers[near] = np.stack([np.where(rng.random(k) < 0.5, -1.0, 1.0) * rng.uniform(*off, size=k) * s,
                                  rng.uniform(-0.4, 0.4, size=k) * s,
                                  rng.uniform(-0.3, 0.3, size=k) * s - S.NEAR_Z], axis=1)
        scales[near] = s
    texs = _textures(rng, case)
    cut = bool(case.get("cutouts"))
    mats = [(i, cut and i % 4 == 3, 128 if cut and not (case.get("normal_maps") and i % 2 == 0) else 255)
            for i in range(len(texs))]
    return S.build_patches(centers, R, scales, (np.arange(n) % len(mats)).astype(np.uint32), mats, texs)


def _near_camera(rng, width, height, count):
    """A camera within three degrees of the layout's own."""
    yaw, pitch = (float(v) for v in rng.uniform(-0.05, 0.05, size=2))
    return S.make_view(width, height, 60.0, S.view_matrix((0.0, 0.0, 0.0), yaw, pitch), 0, count)


class _Handles:
    """The library's objects of one state. What refers to their device memory
    refers to this: they are closed when the state and its outputs are gone."""

    def __init__(self):
        self.batch, self.fbs, self.scenes, self.other = None, [], [], []

    def __del__(self):
        try:
            torch.cuda.synchronize()
            for h in [self.batch, *self.fbs, *self.scenes, *self.other]:
                if h is not None:
                    h.close()
        except Exception:
            pass


class _State:
    """What a program holds between frames."""

    def __init__(self, case):
        self.case, self.handles, self.outs = case, _Handles(), None


class _Device:
    """A device buffer of the library, as torch sees it."""

    def __init__(self, handles, ptr, shape, typestr):
        self.handles = handles
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 2}


class _Outputs(dict):
    """Tensors over the state's own buffers, which they keep."""

    handles = None


def _keys(handles, fb):
    ptr, size = fb.keys_ptr()
    return torch.as_tensor(_Device(handles, ptr, (size // 8,), "<i8"), device="cuda")


def _color(handles, fb):
    return torch.as_tensor(_Device(handles, fb.color_ptr(), (fb.height, fb.width), "<i4"), device="cuda")


def _outputs(st, color):
    """The vis-buffer keys of every framebuffer, and its resolved image."""
    if st.outs is None:
        st.outs = _Outputs(keys=[_keys(st.handles, fb) for fb in st.handles.fbs])
        if color:
            st.outs["color"] = [_color(st.handles, fb) for fb in st.handles.fbs]
        st.outs.handles = st.handles
    return st.outs


_MODES = {"albedo": g.GLIMP_RESOLVE_ALBEDO, "lit": g.GLIMP_RESOLVE_LIT, "normals": g.GLIMP_RESOLVE_NORMALS}


def _prepare_draws(case, rng):
    """A scene, a framebuffer and a camera for the call-by-call kinds."""
    st = _State(case)
    ctx = _context()
    W, H = case["width"], case["height"]
    sc = _scene(rng, case, W, H)
    st.handles.scenes = [g.Scene(ctx, sc)]
    st.handles.fbs = [g.Framebuffer(ctx, W, H)]
    st.view = S.make_view(W, H, count=sc.count)
    st.planes = st.view.frustum_planes()
    st.lighting = S.default_lighting(st.view)
    st.sky = None
    if case.get("sky"):
        st.sky = g.Texture(ctx, TX.sky_texture(128))
        st.handles.other.append(st.sky)
    st.occ = None
    if case.get("occlusion"):
        # the depth map of the frame before this one
        st.hiz = g.DepthMap(ctx, W, H)
        st.handles.other.append(st.hiz)
        g.render_frame(ctx, st.handles.scenes[0], st.view, st.handles.fbs[0])
        st.hiz.build(st.handles.fbs[0])
        st.occ = g.Occlusion(st.hiz, *S.occlusion_terms(st.view.proj, st.view.view))
    return st


def _prepare_batch(case, rng):
    st = _State(case)
    ctx = _context()
    W, H = case["width"], case["height"]
    host = []
    for i in range(case["scenes"]):
        host.append(_scene(rng, dict(case, meshlets=max(4, case["meshlets"] // (1 << i))), W, H))
        st.handles.scenes.append(g.Scene(ctx, host[i]))
    views, resolves = [], []
    for v in range(case["views"]):
        si = v % len(host)
        w, h = W, H
        if not case["same_size"]:
            # sides log-uniform over a factor of four, the same for every seed
            w = max(4, 4 * int(W * 0.25 ** (v * 0.6180339887 % 1.0) / 4))
            h = max(4, 4 * int(H * 0.25 ** (v * 0.7548776662 % 1.0) / 4))
        view = S.make_view(w, h, count=host[si].count) if v == 0 else _near_camera(rng, w, h, host[si].count)
        st.handles.fbs.append(g.Framebuffer(ctx, w, h))
        views.append((st.handles.scenes[si], st.handles.fbs[v], view))
        if case["mode"] != "none":
            resolves.append((view.object_to_clip, _MODES[case["mode"]], S.default_lighting(view)))
    st.handles.batch = g.Batch(ctx, views, shape={k: case[k] for k in ("bin_size", "bin_capacity", "raster_threads")})
    if resolves:
        st.handles.batch.set_resolve(resolves)
    return st


def _prepare_fit(case, rng):
    """Texture fitting: fixed vis-buffers of a few cameras, fp32 texel chains,
    per-vertex UVs (a patch of every texture per meshlet) and colours, and the
    gradient of the loss with respect to the image."""
    st = _State(case)
    ctx = _context()
    W, H, size, count = case["width"], case["height"], case["tex_size"], case["textures"]
    small = dict(case, layout="spread", tex_size=8)
    st.host = sc = _scene(rng, small, W, H)
    st.handles.scenes = [g.Scene(ctx, sc)]
    st.views = []
    for v in range(case["views"]):
        view = S.make_view(W, H, count=sc.count) if v == 0 else _near_camera(rng, W, H, sc.count)
        st.handles.fbs.append(g.render_frame(ctx, st.handles.scenes[0], view))
        st.views.append((st.handles.fbs[v], view.object_to_clip))
    gen = torch.Generator("cuda")
    gen.manual_seed(int(rng.integers(1 << 40)))
    # textures of soft blobs with some grain, every level the 2x2 mean of the last
    levels, parts, sizes, offsets, total = int(math.log2(size)) - 1, [], [], [], 0
    for _ in range(count):
        coarse = torch.rand((1, 4, max(2, size // 16), max(2, size // 16)), generator=gen, device="cuda")
        level = torch.nn.functional.interpolate(coarse, size=(size, size), mode="bilinear")
        level = level + 0.02 * torch.rand((1, 4, size, size), generator=gen, device="cuda")
        offs = []
        for m in range(levels):
            offs.append(total)
            parts.append(level[0].permute(1, 2, 0).reshape(-1, 4))
            total += parts[-1].shape[0]
            level = torch.nn.functional.avg_pool2d(level, 2)
        sizes.append((size, size, levels))
        offsets.append(offs)
    st.chains = D.TexelChains(np.broadcast_to(np.zeros((1, 4), np.float32), (total, 4)), sizes, offsets)
    texels = torch.cat(parts).contiguous()
    uv = D.vertex_uv(sc).reshape(sc.count, 64, 2) * np.float32(case["cell_texels"] / size)
    uv = (uv + rng.random((sc.count, 1, 2))).astype(np.float32).reshape(-1, 2)
    color = rng.uniform(0.5, 1.5, size=(sc.count * 64, 4)).astype(np.float32)
    st.params = [texels.requires_grad_(), torch.from_numpy(uv).cuda().requires_grad_(),
                 torch.from_numpy(color).cuda().requires_grad_()]
    st.op = D.DiffResolveViews(ctx, st.handles.scenes[0], st.views, st.chains)
    st.grad = torch.randn((st.op.binding.total_pixels, 4), generator=gen, device="cuda")
    return st


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] == "batch":
        return _prepare_batch(case, rng)
    if case["kind"] == "fit":
        return _prepare_fit(case, rng)
    return _prepare_draws(case, rng)


# ---------------------------------------------------------------- one pass

def run(st):
    case = st.case
    kind = case["kind"]
    stream = torch.cuda.current_stream()
    if kind == "fit":
        out = st.op(*st.params)
        grads = torch.autograd.grad(out, st.params, grad_outputs=st.grad)
        return {"image": out.detach(), "texels": grads[0], "uv": grads[1], "color": grads[2]}
    if kind == "batch":
        st.handles.batch.launch(case["graph"], stream)
        return _outputs(st, case["mode"] != "none")
    fb, sc, view = st.handles.fbs[0], st.handles.scenes[0], st.view
    fb.clear(0, 0.0, stream)
    if kind == "gbuffer":
        fb.draw(sc, view.object_to_clip, view.meshlet_count, 0, st.planes, 0, stream,
                pipeline=g.GLIMP_PIPELINE_DEFERRED)
        return [fb.read_layer(k, stream=stream) for k in range(3)]
    if kind == "overdraw":
        fb.draw(sc, view.object_to_clip, view.meshlet_count, 0, st.planes, 0, stream,
                pipeline=g.GLIMP_PIPELINE_OVERDRAW)
        fb.resolve(sc, view.object_to_clip, g.GLIMP_RESOLVE_OVERDRAW_QUAD, stream=stream)
    else:
        fb.draw(sc, view.object_to_clip, view.meshlet_count, 0, st.planes, 0, stream, occlusion=st.occ)
        if st.occ is not None:
            st.hiz.build(fb, stream)
        lit = case["mode"] != "albedo"
        fb.resolve(sc, view.object_to_clip, _MODES[case["mode"]], st.lighting if lit else None, stream,
                   st.sky if case["mode"] == "lit" else None)
    return _outputs(st, True)


# ---------------------------------------------------------------- work

def work(case):
    """Bytes: bounds of all meshlets, the data of those in view (a third of a
    spread layout, nearly all of a layered one), every pixel's key and colour
    written once, a texel per pixel. Operations: transform and setup of the
    triangles in view, and per pixel the coverage of about three triangles
    (eight in layers) and the shading."""
    kind = case["kind"]
    layers = case.get("layout") == "layers"
    views = case.get("views", 1)
    px = case["width"] * case["height"] * views
    if kind == "batch" and not case["same_size"]:
        px *= 0.29                       # mean of 0.25^u, squared
    M = case["meshlets"]
    seen = (0.9 if layers else 0.32) * M * views
    if kind == "batch":
        seen /= sum(1.0 / case["scenes"] / (1 << i) for i in range(case["scenes"])) ** -1
    shade = {"albedo": 200, "lit": 500, "normals": 300}.get(case.get("mode"), 0)
    if kind == "fit":
        texels = case["textures"] * case["tex_size"] ** 2 * 4 / 3
        grads = 16 * texels + 24 * 64 * M
        # key, image and gradient per pixel twice, four texels, then the gradients written once
        return {"bytes": px * (8 + 16 + 8 + 16 + 64) + seen * 64 * 40 + grads, "flops": px * 700.0}
    out = {"gbuffer": 8 + 12, "overdraw": 8 + 4 + 4}.get(kind, 8 + (4 + 4 if shade else 0))
    return {"bytes": 16.0 * M * views + seen * 1157 + px * out,
            "flops": seen * 98 * 120 + px * ((8 if layers else 3) * 14 + (shade or 100))}


# ---------------------------------------------------------------- 64 bits

def exact(case, seed):
    """The image and gradients of a fit in float64 with plain torch: the
    vis-buffer (which triangle each pixel shows) is an input of the path, the
    rest is evaluated from the meshlets and the parameters. The other kinds
    give whole numbers only."""
    if case["kind"] != "fit":
        return None
    st = prepare(case, seed)
    dev = torch.device("cuda")
    sc = st.host
    texels, uv, color = (p.detach().double() for p in st.params)
    g_tex, g_uv, g_col = torch.zeros_like(texels), torch.zeros_like(uv), torch.zeros_like(color)
    pos = torch.from_numpy(sc.positions).to(dev).double()
    idx = torch.from_numpy(sc.indices.astype(np.int64)).to(dev)
    tex_of = torch.tensor([m[0] for m in sc.materials], device=dev)[
        torch.from_numpy(sc.material_id.astype(np.int64)).to(dev)]
    offs = torch.tensor(st.chains.offsets, device=dev)
    size, levels = st.chains.sizes[0][0], st.chains.sizes[0][2]
    images, base = [], 0
    for fb, clip in st.views:
        W, H = fb.width, fb.height
        ids, depth = fb.read()
        ids = torch.from_numpy(ids.astype(np.int64)).to(dev)
        cover = torch.from_numpy(depth > 0).to(dev)
        py, px = torch.nonzero(cover, as_tuple=True)
        ids = ids[py, px]
        mi, tri = ids >> 7, ids & 127
        vi = idx[mi, :, tri]                                     # (n, 3)
        p = pos[mi[:, None], :, vi]                              # (n, 3, xyz)
        M = torch.from_numpy(np.asarray(clip)).to(dev).double().reshape(4, 4)
        c = p @ M[:3] + M[3]                                     # column-major: rows of M are columns
        iw = 1.0 / c[..., 3]
        q = c[..., :2] * iw[..., None]
        x0, y0, x1, y1, x2, y2 = q[:, 0, 0], q[:, 0, 1], q[:, 1, 0], q[:, 1, 1], q[:, 2, 0], q[:, 2, 1]
        det = (x2 - x1) * (y0 - y1) + (y1 - y2) * (x0 - x1)
        a = iw / det[:, None]
        dx = a * torch.stack([y1 - y2, y2 - y0, y0 - y1], 1)
        dy = a * torch.stack([x2 - x1, x0 - x2, x1 - x0], 1)
        rx = px.double() * (2.0 / W) + (1.0 / W - 1.0) - x0
        ry = py.double() * (2.0 / H) + (1.0 / H - 1.0) - y0
        kx, ky = 2.0 / W, -2.0 / H
        iiw = iw[:, 0] + dx.sum(1) * rx + dy.sum(1) * ry
        b12 = (dx[:, 1:] * rx[:, None] + dy[:, 1:] * ry[:, None]) / iiw[:, None]
        b = torch.cat([1.0 - b12.sum(1, keepdim=True), b12], 1)
        ddx = (b * iiw[:, None] + kx * dx) / (iiw + kx * dx.sum(1))[:, None] - b
        ddy = (b * iiw[:, None] + ky * dy) / (iiw + ky * dy.sum(1))[:, None] - b
        vert = mi[:, None] * 64 + vi
        t = uv[vert]                                             # (n, 3, 2)
        t10, t20 = t[:, 1] - t[:, 0], t[:, 2] - t[:, 0]
        UV = t[:, 0] + b[:, 1:2] * t10 + b[:, 2:3] * t20
        gx = ((t20 * ddx[:, 2:3] + t10 * ddx[:, 1:2]) * size).square().sum(1)
        gy = ((t20 * ddy[:, 2:3] + t10 * ddy[:, 1:2]) * size).square().sum(1)
        step = torch.maximum(gx, gy).clamp_min(1e-30)
        mip = torch.floor(torch.floor(torch.log2(step)) / 2).long()
        # one filter per 4x4 tile: nearest when a pixel of it is minified
        small = torch.zeros((H // 4, W // 4), dtype=torch.bool, device=dev)
        small[py[mip > 0] // 4, px[mip > 0] // 4] = True
        near = small[py // 4, px // 4]
        level = torch.where(near, mip.clamp(0, levels - 1), torch.zeros_like(mip))
        wide = size >> level
        frac = UV - torch.floor(UV)
        nx = torch.minimum((frac * wide[:, None]).long(), wide[:, None] - 1)
        xf = (frac * size - 0.5)
        inner = xf > 0
        xf = xf.clamp_min(0.0)
        cell = torch.minimum(xf.long(), torch.full_like(nx, size - 1))
        edge = cell < size - 1
        fr = torch.where(edge, xf - cell, torch.zeros_like(xf))
        fr = torch.where(near[:, None], torch.zeros_like(fr), fr)
        cell = torch.where(near[:, None], nx, cell)
        nxt = torch.where(edge & ~near[:, None], cell + 1, cell)
        row0 = offs[tex_of[mi], level] + cell[:, 1] * wide
        row1 = offs[tex_of[mi], level] + nxt[:, 1] * wide
        at = torch.stack([row0 + cell[:, 0], row0 + nxt[:, 0], row1 + cell[:, 0], row1 + nxt[:, 0]], 1)
        fx, fy = fr[:, 0], fr[:, 1]
        w = torch.stack([(1 - fx) * (1 - fy), fx * (1 - fy), (1 - fx) * fy, fx * fy], 1)
        q4 = texels[at]                                          # (n, 4, rgba)
        val = (w[..., None] * q4).sum(1)
        slope = torch.where(inner & edge & ~near[:, None], float(size), 0.0).double()
        du = slope[:, 0:1] * ((1 - fy)[:, None] * (q4[:, 1] - q4[:, 0]) + fy[:, None] * (q4[:, 3] - q4[:, 2]))
        dv = slope[:, 1:2] * ((1 - fx)[:, None] * (q4[:, 2] - q4[:, 0]) + fx[:, None] * (q4[:, 3] - q4[:, 1]))
        col = (b[..., None] * color[vert]).sum(1)
        image = torch.zeros((H, W, 4), dtype=torch.float64, device=dev)
        image[py, px] = val * col
        images.append(image.reshape(-1, 4))
        go = st.grad[base:base + W * H].double().reshape(H, W, 4)[py, px]
        base += W * H
        gv, gc = go * col, go * val
        g_tex.index_add_(0, at.reshape(-1), (w[..., None] * gv[:, None]).reshape(-1, 4))
        g_at = torch.stack([(gv * du).sum(1), (gv * dv).sum(1)], 1)
        g_uv.index_add_(0, vert.reshape(-1), (b[..., None] * g_at[:, None]).reshape(-1, 2))
        g_col.index_add_(0, vert.reshape(-1), (b[..., None] * gc[:, None]).reshape(-1, 4))
    return {"image": torch.cat(images), "texels": g_tex, "uv": g_uv, "color": g_col}

"""The work a user of lucid_amd has it do, as timed cases.

Every case goes through the package's own entry points: ``LucidRenderer.render`` (one frame,
waited for, re-rendered after an internal buffer grew), ``LucidRenderer.render_async`` (a
viewer's loop), ``LucidBatch.render`` (many frames at once) and ``autograd.render_image`` (the
differentiable frame and its backward). Scenes come from the package's generators at the sizes
of its benchmark and tests, with the default tuning.

Kinds:
  frame   a soup of triangles ("uniform": centroids all over the image, "blobs": clustered),
          RGBA8 samples, image + fragment counts
  mesh    icospheres paired into quads; "lit" adds RGBA8 vertex colours, packed vertex normals,
          instance colours and a sun
  planes  overlapping quads with depth slopes; "textured" samples albedo atlases, otherwise the
          planes intersect each other, so their order changes from pixel to pixel
  fp32    a frame of fp32 samples (the differentiable renderer's forward)
  train   the differentiable frame and its backward for a given dL/d(image)
  batch   independent scenes of mixed sizes and resolutions in one launch
"""

from __future__ import annotations

import math

import numpy as np
import torch

from lucid_amd import _lib, autograd, scenes
from lucid_amd.batch import LucidBatch
from lucid_amd.renderer import GpuScene, LucidRenderer
from lucid_amd.scene_io import encode_normals

# Vertex offsets (NDC) of the uniform soup: a mean of about 7.9e-4 fragments per pixel and
# triangle at every resolution. A blob triangle covers about 68 pixels (median edge 6 px).
SIGMA = 0.0615
FRAGS_PER_PIXEL_TRI = 7.9e-4
FRAGS_PER_BLOB_TRI = 68.0
# Floating-point operations of one fragment: depth plane, colour, sample, blend; and of its
# adjoint (two walks over the fragments).
FLOPS_FORWARD, FLOPS_BACKWARD = 40, 120


def listed():
    return [
        # a thumbnail: launches and host work, next to no fragments
        dict(name="thumb", kind="frame", style="uniform", tris=2_000, w=128, h=128,
             colors="f32", blend="over", loop=False),
        # the small scene of the parity tests: a preview frame
        dict(name="preview", kind="frame", style="uniform", tris=10_000, w=512, h=512,
             colors="f32", blend="over", loop=False),
        # RGBA8 vertex colours (the reference's format), additive particles, a ragged size
        dict(name="particles", kind="frame", style="blobs", tris=60_000, w=767, h=431,
             colors="rgba8", blend="additive", loop=False),
        # the headline frame: 1 M triangles at 1080p in a viewer's loop (frames queued)
        dict(name="headline", kind="frame", style="blobs", tris=1_000_000, w=1920, h=1080,
             colors="f32", blend="over", loop=True),
        # 4096 spheres, about 2.7 M quads, at 1440p
        dict(name="mesh", kind="mesh", gx=16, gy=16, gz=16, level=3, w=2560, h=1440, lit=False),
        # a loaded model: vertex normals, sun, instance colours, RGBA8 vertex colours
        dict(name="lit", kind="mesh", gx=10, gy=8, gz=6, level=3, w=1280, h=720, lit=True),
        # textured glass
        dict(name="textured", kind="planes", textured=True, n=96, w=1024, h=768),
        # intersecting panes: the order differs from pixel to pixel (exact per-pixel sorts)
        dict(name="panes", kind="planes", textured=False, n=32, w=640, h=360),
        # the differentiable scene's forward, as an evaluation renders it
        dict(name="fp32", kind="fp32", tris=200_000, w=512, h=512),
        # one optimisation step of that scene
        dict(name="train", kind="train", tris=200_000, w=512, h=512),
        # a step at the start of a coarse-to-fine fit
        dict(name="train_small", kind="train", tris=10_000, w=200, h=136),
        # a serving batch: scenes of 5 k to 500 k triangles at four resolutions
        dict(name="batch", kind="batch", n=32, lo=5_000, hi=500_000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("frame", "frame", "frame", "mesh", "planes", "fp32", "train", "batch"))
    if kind == "frame":
        w, h = _log_int(rng, 96, 1920), _log_int(rng, 96, 1080)
        style = rng.choice(("uniform", "blobs"))
        top = 1_000_000
        if style == "uniform":  # at most as many fragments as the headline frame
            top = min(top, int(68e6 / (FRAGS_PER_PIXEL_TRI * w * h)))
        return dict(kind=kind, style=style, tris=_log_int(rng, 1_000, max(top, 2_000)), w=w, h=h,
                    colors=rng.choice(("f32", "f32", "rgba8")),
                    blend=rng.choice(("over", "over", "over", "additive", "threshold")),
                    loop=rng.choice((True, False)))
    if kind == "mesh":
        return dict(kind=kind, gx=rng.randint(2, 14), gy=rng.randint(2, 14),
                    gz=rng.randint(1, 12), level=rng.choice((2, 3)), w=_log_int(rng, 160, 2000),
                    h=_log_int(rng, 120, 1200), lit=rng.choice((True, False)))
    if kind == "planes":
        return dict(kind=kind, textured=rng.choice((True, False)), n=rng.randint(4, 32),
                    w=_log_int(rng, 120, 640), h=_log_int(rng, 90, 360))
    if kind == "batch":
        return dict(kind=kind, n=rng.randint(4, 24), lo=rng.randint(2_000, 8_000),
                    hi=_log_int(rng, 10_000, 200_000))
    w, h = _log_int(rng, 96, 512), _log_int(rng, 96, 512)
    return dict(kind=kind, tris=_log_int(rng, 2_000, 200_000), w=w, h=h)


# ------------------------------------------------------------------ scenes


def _lit(sc, case, rng):
    """The mesh as a model file gives it: byte colours, normals, one colour per instance."""
    n = case["gx"] * case["gy"] * case["gz"]
    sphere, _ = scenes.icosphere(case["level"])
    sc.normals = np.tile(encode_normals(sphere), n)
    rgb = rng.uniform(0.3, 1.0, (sc.num_verts, 3)).astype(np.float32)
    sc.colors_rgba8 = scenes.pack_rgba8(rgb, np.full(sc.num_verts, 0.5, np.float32))
    sc.colors_rgb = sc.tri_alpha = None
    sc.instances["flags"] |= scenes.INST_HAS_VERTEX_NORMALS | scenes.INST_HAS_COLOR
    k = len(sc.instances)
    sc.instance_colors = scenes.pack_rgba8(rng.uniform(0.5, 1.0, (k, 3)).astype(np.float32),
                                           rng.uniform(0.6, 1.0, k).astype(np.float32))
    sc.config = scenes.make_config(scenes.scene_camera(sc), k, ambient=(0.4, 0.45, 0.5),
                                   sun_color=(1.0, 0.95, 0.9), sun_dir=(0.36, -0.48, -0.8),
                                   sun_power=0.8)
    return sc


def _pixel_corners(sc):
    """Pixel coordinates (T, 3, 2) and view depths (T, 3) of a soup's corners, in 64 bits, from
    the float32 positions and the frustum in the frame's LucidConfig (pixel (x, y) is sampled
    at its centre)."""
    cfg = np.frombuffer(sc.config, np.float32).astype(np.float64)
    p = torch.from_numpy(sc.positions.reshape(-1, 3, 3)).cuda().double()
    z = -p[..., 2]
    x = (p[..., 0] / z - cfg[36]) / cfg[40] - 0.5
    y = (p[..., 1] / z - cfg[37]) / cfg[45] - 0.5
    return torch.stack([x, y], -1), z


def _samples(sc, chunk=1 << 24):
    """Yields (triangle, x, y, lam, dist) of every pixel of every triangle's bounding box:
    screen-space barycentrics and the signed pixel distances to the three edges."""
    xy, _ = _pixel_corners(sc)
    lo = xy.amin(1).floor().long() - 1
    hi = xy.amax(1).ceil().long() + 1
    size = torch.tensor([sc.width, sc.height], device=xy.device)
    lo = torch.minimum(lo.clamp(min=0), size)
    hi = torch.minimum(hi.clamp(min=-1), size - 1)
    ext = (hi - lo + 1).clamp(min=0)
    area = ext[:, 0] * ext[:, 1]
    ends = area.cumsum(0)
    first = 0
    while first < len(area):
        base = int(ends[first] - area[first])
        last = int(torch.searchsorted(ends, base + chunk, right=True))
        last = max(last, first + 1)
        n = int(ends[last - 1]) - base
        tri = torch.repeat_interleave(torch.arange(first, last, device=xy.device),
                                      area[first:last], output_size=n)
        k = torch.arange(n, device=xy.device) + base - (ends[tri] - area[tri])
        px = lo[tri, 0] + k % ext[tri, 0]
        py = lo[tri, 1] + k // ext[tri, 0]
        c = xy[tri]
        pt = torch.stack([px, py], -1).double()
        lam, dist = [], []
        d1, d2 = c[:, 1] - c[:, 0], c[:, 2] - c[:, 0]
        det = d1[:, 0] * d2[:, 1] - d1[:, 1] * d2[:, 0]
        for i in range(3):
            a, b = c[:, (i + 1) % 3], c[:, (i + 2) % 3]
            e, r = b - a, pt - a
            l = (e[:, 0] * r[:, 1] - e[:, 1] * r[:, 0]) / det
            lam.append(l)
            dist.append(l * det.abs() / e.norm(dim=1))
        yield tri, px, py, torch.stack(lam, -1), torch.stack(dist, -1)
        first = last


def _soup(case, seed):
    """The differentiable scenes: the uniform soup with depths on a shuffled even grid (so that
    the order in 32 bits is the order in 64) and without the triangles that have an edge within
    1/4000 of a pixel of some pixel's centre (so that their coverage is the same, too)."""
    rng = np.random.default_rng(seed)
    n = case["tris"] + case["tris"] // 4 + 64  # a few per cent are left out
    c = rng.uniform(-1.0, 1.0, (n, 1, 2))
    e = rng.normal(0.0, SIGMA, (n, 3, 2))
    depth = 1.0 + 99.0 * (rng.permutation(n) + rng.uniform(0.3, 0.7, n)) / n
    rgb = rng.uniform(0.01, 0.99, (n, 3, 3))
    alpha = rng.uniform(0.2, 0.8, n)
    ndc = c + e
    sc = scenes.soup_scene(case["w"], case["h"], ndc, depth, rgb, alpha)
    close = torch.zeros(n, dtype=torch.bool, device="cuda")
    for tri, _, _, _, dist in _samples(sc):
        near = (dist.abs() < 2.5e-4).any(1) & (dist > -2.5e-4).all(1)
        close[tri[near]] = True
    keep = np.flatnonzero(~close.cpu().numpy())[:case["tris"]]
    assert len(keep) == case["tris"]
    return scenes.soup_scene(case["w"], case["h"], ndc[keep], depth[keep], rgb[keep], alpha[keep])


def _scene(case, seed):
    kind, w, h = case["kind"], case["w"], case["h"]
    if kind == "frame":
        make = scenes.config0 if case["style"] == "uniform" else scenes.config1
        return make(seed=seed, num_tris=case["tris"], width=w, height=h,
                    color_format=case["colors"])
    if kind == "mesh":
        sc = scenes.config2(seed=seed, grid=(case["gx"], case["gy"], case["gz"]), width=w,
                            height=h, level=case["level"])
        return _lit(sc, case, np.random.default_rng(seed + 1)) if case["lit"] else sc
    if kind == "planes":
        make = scenes.textured_planes if case["textured"] else scenes.tilted_planes
        return make(w, h, case["n"], seed=seed)
    return _soup(case, seed)


def _batch_sizes(case):
    """(triangles, (w, h)) of each scene: log-normal triangle counts around 50 k, clipped to the
    case's range, and the four resolutions in turn (sizes are the case's, contents the seed's)."""
    rng = np.random.default_rng(case["n"])
    counts = np.clip(np.exp(rng.normal(np.log(50_000), 1.0, case["n"])), case["lo"], case["hi"])
    res = scenes.BATCH_RESOLUTIONS
    return [(int(t), res[i % len(res)]) for i, t in enumerate(counts)]


def _batch_scenes(case, seed):
    return [scenes.config0(seed=seed * 1000 + i, num_tris=t, width=w, height=h)
            for i, (t, (w, h)) in enumerate(_batch_sizes(case))]


_BLEND = {"over": 0, "additive": _lib.OPT_ADDITIVE_BLENDING, "threshold": _lib.OPT_ALPHA_THRESHOLD}


def _grad_image(case, seed):
    """dL/d(image) as a mean-squared-error loss hands it over: small, of both signs."""
    g = torch.Generator().manual_seed(seed)
    return torch.randn((case["h"], case["w"], 4), generator=g) * 1e-3


# ------------------------------------------------------------------ the cases


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        scs = _batch_scenes(case, seed)
        rs = [LucidRenderer((s.width, s.height), max_quads=s.num_quads) for s in scs]
        return {"kind": kind, "batch": LucidBatch(rs), "scenes": [GpuScene(s) for s in scs],
                "out": [r.alloc_outputs() for r in rs]}
    sc = _scene(case, seed)
    fp32 = kind in ("fp32", "train")
    opts = _lib.OPT_FP32_SAMPLES if fp32 else _BLEND[case.get("blend", "over")]
    st = {"kind": kind, "renderer": LucidRenderer((sc.width, sc.height), opts=opts,
                                                  max_quads=sc.num_quads),
          "scene": GpuScene(sc), "loop": case.get("loop", False)}
    if kind == "train":
        shape = (-1, 3)
        st["colors"] = st["scene"].colors_rgb.reshape(shape).clone().requires_grad_()
        st["alpha"] = st["scene"].tri_alpha.clone().requires_grad_()
        st["grad"] = _grad_image(case, seed).cuda()
    else:
        st["out"] = st["renderer"].alloc_outputs(rgba8=not fp32, rgba32f=fp32)
        if st["loop"]:  # a viewer's first frame, which sizes the internal buffers
            st["renderer"].render(st["scene"], st["out"])
    return st


def run(state):
    if state["kind"] == "batch":
        return state["batch"].render(state["scenes"], state["out"])
    if state["kind"] == "train":
        img = autograd.render_image(state["renderer"], state["scene"], state["colors"],
                                    state["alpha"])
        grads = torch.autograd.grad(img, (state["colors"], state["alpha"]), state["grad"])
        return (img.detach(), *grads)
    if state["loop"]:
        state["renderer"].render_async(state["scene"], state["out"])
        return state["out"]
    return state["renderer"].render(state["scene"], state["out"])


def _fragments(case):
    kind = case["kind"]
    px = case["w"] * case["h"]
    if kind == "mesh":  # a front and a back layer of spheres per grid layer
        return 0.86 * px * case["gz"]
    if kind == "planes":
        return (0.35 if case["textured"] else 1.0) * px * case["n"]
    if kind == "frame" and case["style"] == "blobs":
        return FRAGS_PER_BLOB_TRI * case["tris"]
    return FRAGS_PER_PIXEL_TRI * px * case["tris"]


def work(case):
    """Bytes: the scene's arrays read once, the outputs (and gradients) written once. Flops:
    the fragments' shading and blending."""
    if case["kind"] == "batch":
        sizes = _batch_sizes(case)
        return {"bytes": sum(t * 96 + w * h * 8 for t, (w, h) in sizes),
                "flops": FLOPS_FORWARD * FRAGS_PER_PIXEL_TRI * sum(t * w * h
                                                                   for t, (w, h) in sizes)}
    px = case["w"] * case["h"]
    frags = _fragments(case)
    if case["kind"] == "mesh":
        n = case["gx"] * case["gy"] * case["gz"]
        verts, quads = 10 * 4 ** case["level"] + 2, 10 * 4 ** case["level"]
        per_vert = 12 + (8 if case["lit"] else 12)
        nbytes = n * (verts * per_vert + quads * (16 + (0 if case["lit"] else 8))) + 8 * px
    elif case["kind"] == "planes":
        nbytes = case["n"] * 200 + 8 * px
    else:
        rgba8 = case.get("colors") == "rgba8"
        nbytes = case["tris"] * (16 + 36 + (12 if rgba8 else 44))
        # image and counts; fp32: a float4 image; train: image, dL/dimage, the gradients
        nbytes += px * {"frame": 8, "fp32": 20, "train": 32}[case["kind"]]
        if case["kind"] == "train":
            nbytes += case["tris"] * 44
    flops = FLOPS_FORWARD + (FLOPS_BACKWARD if case["kind"] == "train" else 0)
    return {"bytes": nbytes, "flops": flops * frags}


def exact(case, seed):
    """Image (and gradients) of the fp32-sample cases in 64 bits: every triangle's pixels by
    their centres, perspective-correct colours, the fragments of a pixel sorted by depth and
    composited front to back, out = sum_i s_i a_i T_i with T_i = prod_{j<i} (1 - a_j), and for
    g = dL/d(out): dL/ds_i = g a_i T_i, dL/da_i = T_i g.s_i - sum_{j>i} g.s_j a_j T_j / (1 - a_i).
    RGBA8 images and fragment counts are whole numbers: nothing to compare in 64 bits."""
    if case["kind"] not in ("fp32", "train"):
        return None
    sc = _soup(case, seed)
    w, h = sc.width, sc.height
    _, z = _pixel_corners(sc)
    parts = []
    for tri, px, py, lam, dist in _samples(sc):
        inside = (dist >= 0.0).all(1)
        tri, lam = tri[inside], lam[inside]
        inv = lam / z[tri]
        depth = inv.sum(1)
        parts.append((tri, (py * w + px)[inside], depth, inv / depth[:, None]))
    tri, pix, depth, bary = (torch.cat(p) for p in zip(*parts))
    del parts
    order = torch.argsort(depth, descending=True, stable=True)
    order = order[torch.argsort(pix[order], stable=True)]
    tri, pix, bary = tri[order], pix[order], bary[order]
    counts = torch.bincount(pix, minlength=w * h)
    rank = torch.arange(len(pix), device=pix.device) - (counts.cumsum(0) - counts)[pix]

    colors = torch.from_numpy(sc.colors_rgb).cuda().double().reshape(-1, 3, 3)
    alpha = torch.from_numpy(sc.tri_alpha).cuda().double()[0::2]
    s = torch.einsum("fk,fkc->fc", bary, colors[tri])
    a = alpha[tri]
    dense = torch.zeros((w * h, int(counts.max()) + 1), dtype=torch.float64, device=pix.device)
    dense[pix, rank + 1] = a
    t = (1.0 - dense).cumprod(1)[pix, rank]
    img = torch.zeros((w * h, 4), dtype=torch.float64, device=pix.device)
    img[:, :3].index_add_(0, pix, s * (a * t)[:, None])
    img[:, 3] = 1.0
    img = img.clamp(0.0, 1.0).reshape(h, w, 4)
    if case["kind"] == "fp32":
        return {"image": None, "image_f": img, "frag_counts": None}

    g = _grad_image(case, seed).cuda().double().reshape(-1, 4)[:, :3]
    gs = (g[pix] * s).sum(1)
    dense.zero_()
    dense[pix, rank] = gs * a * t
    behind = dense.flip(1).cumsum(1).flip(1)[pix, rank + 1]
    g_alpha = torch.zeros(2 * len(alpha), dtype=torch.float64, device=pix.device)
    g_alpha.index_add_(0, 2 * tri, t * gs - behind / (1.0 - a))
    g_col = torch.zeros((colors.numel() // 3, 3), dtype=torch.float64, device=pix.device)
    at_g = g[pix] * (a * t)[:, None]
    for k in range(3):
        g_col.index_add_(0, 3 * tri + k, at_g * bary[:, k:k + 1])
    return img, g_col, g_alpha

"""Performance cases of the framework: what its users run, over the sizes they run it at.

Five kinds of work, each through public entry points:

  silhouette  one iteration of a silhouette fit (SilhouetteFit.step), HardSoftRas or
              screen-space AA: forward, backward and Adam on the vertex positions
  texture     one iteration of a texture fit (TextureFit.step)
  pbr         one iteration of a material + environment fit (PbrFit.step)
  surface     a loop body written against opendressi_amd.torch: forward, L2 loss against a
              target and autograd back to what is fitted
  ibl         the split-sum environment maps through opendressi_amd.ops: pooling, irradiance
              and prefilter convolutions, lookups per pixel, and the way back to the environment

The fits run at the sizes of the package's own workloads (WORKLOADS, TEX_WORKLOADS,
PBR_WORKLOADS); the others at the sizes of its tests and benchmark and ordinary larger ones.
"""
import math

import numpy as np
import torch

import opendressi_amd as od
import opendressi_amd.torch as dr
from opendressi_amd import _lib as L
from opendressi_amd import ops as K


def listed():
    return [
        # the smallest fit: one view of a 1280-face mesh, where launches and latency count
        {"name": "hsr_256x1", "kind": "silhouette", "technique": "hsr", "level": 3, "size": 256,
         "views": 1},
        # an ordinary silhouette fit
        {"name": "hsr_512x4", "kind": "silhouette", "technique": "hsr", "level": 4, "size": 512,
         "views": 4},
        # the largest silhouette fits, one for each technique
        {"name": "hsr_2048x4", "kind": "silhouette", "technique": "hsr", "level": 6, "size": 2048,
         "views": 4},
        {"name": "aa_2048x4", "kind": "silhouette", "technique": "aa", "level": 6, "size": 2048,
         "views": 4},
        # a texture fit from eight cameras a step
        {"name": "texture_1024x8", "kind": "texture", "stacks": 128, "slices": 64, "size": 1024,
         "tex": 1024, "views": 8, "sets": 16},
        # materials and environment fitted together
        {"name": "pbr_1024x6", "kind": "pbr", "level": 5, "size": 1024, "views": 6, "tex": 512,
         "env": 512, "levels": 6},
        # the torch loop of a silhouette fit: rasterize + antialias, geometry gradients from
        # eight samples a face
        {"name": "surface_aa_256x8", "kind": "surface", "mode": "aa", "level": 3, "height": 256,
         "width": 256, "views": 8, "samples": 8},
        # the same at the smallest and raggedest, with the exact geometry gradient
        {"name": "surface_aa_61x97", "kind": "surface", "mode": "aa", "level": 2, "height": 61,
         "width": 97, "views": 1, "samples": 0},
        # vertex colours: rasterize + interpolate, gradients to the colours
        {"name": "surface_color_720x1280", "kind": "surface", "mode": "color", "level": 5,
         "height": 720, "width": 1280, "views": 4, "channels": 3},
        # a texture through interpolated uv: rasterize + interpolate + texture
        {"name": "surface_texture_512x4", "kind": "surface", "mode": "texture", "stacks": 64,
         "slices": 32, "height": 512, "width": 512, "views": 4, "tex": 512},
        # soft rasterization with two depth peels, gradients to the positions
        {"name": "surface_soft_512x2", "kind": "surface", "mode": "soft", "level": 4,
         "height": 512, "width": 512, "views": 2, "peels": 2},
        # a 512 x 256 environment's maps and lookups, forward and backward
        {"name": "ibl_512", "kind": "ibl", "env": 512, "levels": 6, "size": 512},
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over the logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["silhouette", "silhouette", "texture", "pbr", "surface", "surface",
                       "surface", "surface", "ibl", "ibl"])
    if kind == "silhouette":
        size = _log(rng, 96, 2048)
        return {"kind": kind, "technique": rng.choice(["hsr", "aa"]),
                "level": rng.randint(2, 6 if size > 400 else 4), "size": size,
                "views": rng.randint(1, 4)}
    if kind == "texture":
        return {"kind": kind, "stacks": _log(rng, 16, 128), "slices": _log(rng, 12, 64),
                "size": _log(rng, 96, 1024), "tex": _log(rng, 64, 1024),
                "views": rng.randint(1, 8), "sets": rng.randint(1, 16)}
    if kind == "pbr":
        return {"kind": kind, "level": rng.randint(2, 5), "size": _log(rng, 96, 768),
                "views": rng.randint(1, 6), "tex": _log(rng, 64, 512),
                "env": rng.choice([128, 256, 512]), "levels": rng.randint(3, 6)}
    if kind == "ibl":
        return {"kind": kind, "env": 2 * _log(rng, 48, 256), "levels": rng.randint(2, 6),
                "size": _log(rng, 64, 512)}
    mode = rng.choice(["aa", "color", "texture", "soft"])
    case = {"kind": kind, "mode": mode}
    if mode == "aa":
        case.update(level=rng.randint(2, 4), height=_log(rng, 48, 256), width=_log(rng, 48, 256),
                    views=rng.randint(1, 8))
        # the exact gradient is for small images
        small = case["height"] * case["width"] <= 16384
        case["samples"] = rng.choice([0, 4, 8, 8] if small else [4, 8])
    elif mode == "color":
        case.update(level=rng.randint(2, 5), height=_log(rng, 48, 720),
                    width=_log(rng, 48, 1280), views=rng.randint(1, 4),
                    channels=rng.randint(1, 4))
    elif mode == "texture":
        case.update(stacks=_log(rng, 12, 64), slices=_log(rng, 8, 32), height=_log(rng, 48, 512),
                    width=_log(rng, 48, 512), views=rng.randint(1, 4), tex=_log(rng, 32, 512))
    else:
        case.update(level=rng.randint(2, 4), height=_log(rng, 48, 512), width=_log(rng, 48, 512),
                    views=rng.randint(1, 2), peels=rng.randint(1, 2))
    return case


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------

_CTX = []


def _context():
    """The program's one device context: fits and per-op calls share it."""
    if not _CTX:
        _CTX.append(od.Context(0))
    return _CTX[0]


class _Memory:
    """A plan's device buffer, for torch to look at in place."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape,
                                         "typestr": typestr, "version": 2}


def _view(buffer_fn, fit, which, shape, typestr="<f4"):
    ptr, nbytes = L.C.c_void_p(), L.C.c_size_t()
    L.check(buffer_fn(fit.handle, which, L.C.byref(ptr), L.C.byref(nbytes)))
    assert nbytes.value >= 4 * math.prod(shape)
    view = torch.as_tensor(_Memory(ptr.value, tuple(shape), typestr), device="cuda:0")
    view.owner = fit  # the buffer is the plan's: it lives as long as the view does
    return view


def _gen(seed, *more):
    return np.random.default_rng([seed, *more])


def _smooth(seed, h, w, c):
    """(h, w, c) float32 in [0, 1]: a coarse random field, upsampled."""
    coarse = torch.from_numpy(_gen(seed, 1).random((1, c, 16, 16), dtype=np.float32))
    up = torch.nn.functional.interpolate(coarse.cuda(), size=(h, w), mode="bilinear")
    return up[0].permute(1, 2, 0).contiguous()


def _silhouette(case, seed):
    # the scene of the package's workloads: a sphere fitted to a bumpy one. The learning rate is
    # that of a late refinement, so that the mesh stays near its start while it is measured
    n, s = case["views"], case["size"]
    w = od.Workload("case", case["level"], s, n, 0.02 if case["level"] > 4 else 0.05,
                    0.1 if case["level"] > 4 else 0.0, 1e-5, 0, seed, case["technique"])
    pos, faces, tgt, mvps = od.make_scene(w)
    fit = od.SilhouetteFit(_context(), pos, faces, mvps, s, target_mesh=(tgt, faces), lr=w.lr,
                           keep_grad=True, technique=w.technique)
    buf = L.lib.dressi_hsr_buffer
    v = len(pos)
    return {"fit": fit, "out": {"loss": _view(buf, fit, L.BUF_LOSS, (s, s)),
                                "face_id": _view(buf, fit, L.BUF_FACE_ID, (n, s, s), "<i4"),
                                "grad": _view(buf, fit, L.BUF_GRAD, (v, 3)),
                                "pos": _view(buf, fit, L.BUF_POS, (v, 3))}}


def _texture(case, seed):
    # a fit that is under way: Adam's moments are those of some steps before
    s, t = case["size"], case["tex"]
    pos, uv, faces = od.uv_sphere(case["stacks"], case["slices"])
    mvps = od.orbit_cameras(case["sets"], case["views"], seed)
    gt = np.ones((t, t, 4), np.float32)
    gt[..., :3] = _smooth(seed, t, t, 3).cpu().numpy()
    tex = np.full((t, t, 4), 0.5, np.float32)
    fit = od.TextureFit(_context(), pos, uv, faces, mvps, s, gt, tex, lr=1e-2)
    r = _gen(seed, 2)
    m = 1e-5 * r.standard_normal((t, t, 4), dtype=np.float32)
    fit.set_state(tex, m, m * m + np.float32(1e-10), 20.0)
    buf = L.lib.dressi_tex_buffer
    return {"fit": fit, "out": {"loss": _view(buf, fit, L.TEX_LOSS, (s, s, 4)),
                                "tex": _view(buf, fit, L.TEX_TEX, (t, t, 4))}}


def _pbr(case, seed):
    t, e = case["tex"], case["env"]
    scene = od.make_pbr_scene(case["level"], case["size"], case["views"], t, e, e // 2,
                              case["levels"], seed=seed)
    fit = od.PbrFit(_context(), scene, keep_grad=True)
    buf = L.lib.dressi_pbr_buffer
    return {"fit": fit, "out": {"loss": _view(buf, fit, L.PBR_LOSS, (1,)),
                                "g_albedo": _view(buf, fit, L.PBR_G_ALBEDO, (t, t, 4)),
                                "g_mr": _view(buf, fit, L.PBR_G_MR, (t, t, 4)),
                                "g_env": _view(buf, fit, L.PBR_G_ENV, (e // 2, e, 4))}}


def _mesh(case, seed):
    """A slightly uneven sphere of the case and its uv: pos, uv, faces."""
    if "stacks" in case:
        pos, uv, faces = od.uv_sphere(case["stacks"], case["slices"])
    else:
        pos, faces = od.icosphere(case["level"])
        uv = None
    wave = _gen(seed, 3).standard_normal((3, 3))
    bump = 1.0 + 0.05 * np.sin(3.0 * pos.astype(np.float64) @ wave).sum(1) / 3.0
    return pos * bump[:, None], uv, faces


def _clips(pos, case):
    """Clip positions {N, V, 4} float64, z in [-w, w], on the case's ring of cameras."""
    m = od.camera_mvps(case["views"]).reshape(-1, 4, 4).astype(np.float64)
    clip = np.concatenate([pos, np.ones_like(pos[:, :1])], 1)[None] @ m
    clip[..., 2] = 2.0 * clip[..., 2] - clip[..., 3]
    return clip


def _surface(case, seed):
    pos, uv, faces = _mesh(case, seed)
    n, h, w = case["views"], case["height"], case["width"]
    clip = torch.from_numpy(_clips(pos, case).astype(np.float32)).cuda()
    s = {"mode": case["mode"], "case": case, "clip": clip, "ctx": dr.RasterizeHipContext(0),
         "tri": torch.from_numpy(faces.astype(np.int32)).cuda()}
    c = {"aa": 1, "color": case.get("channels"), "texture": 3, "soft": 1}[case["mode"]]
    s["target"] = _smooth(seed, h, w, c).expand(n, -1, -1, -1).contiguous()
    r = _gen(seed, 4)
    if case["mode"] == "color":
        s["color"] = torch.from_numpy(r.random((len(pos), c), dtype=np.float32)).cuda()
    elif case["mode"] == "texture":
        s["uv"] = torch.from_numpy(uv).cuda()
        s["tex"] = torch.from_numpy(r.random((case["tex"], case["tex"], 3),
                                             dtype=np.float32)).cuda()
    return s


def _sizes(w, h, to_w, to_h):
    """The pooling chain from (w, h) until it fits (to_w, to_h), (w, h) first."""
    out = [(w, h)]
    while out[-1][0] > to_w or out[-1][1] > to_h:
        out.append(((out[-1][0] + 1) // 2, (out[-1][1] + 1) // 2))
    return out


def _ibl_shape(case):
    """(pooling chain, index of the prefilter's source in it, levels' sizes)"""
    chain = _sizes(case["env"], case["env"] // 2, 64, 32)
    src = len(_sizes(case["env"], case["env"] // 2, 128, 64)) - 1
    w, h = min(128, chain[src][0]), min(64, chain[src][1])
    levels = []
    for _ in range(case["levels"]):
        levels.append((w, h))
        w, h = max(w // 2, 1), max(h // 2, 1)
    return chain, src, levels


def _ibl_inputs(case, seed):
    s = case["size"]
    env = od.synthetic_env(case["env"], case["env"] // 2, seed)
    r = _gen(seed, 5)
    # normals and reflections of a sphere that fills the image, background looking out
    y, x = np.meshgrid((np.arange(s) + 0.5) / s * 2 - 1, (np.arange(s) + 0.5) / s * 2 - 1,
                       indexing="ij")
    z = np.sqrt(np.maximum(1.0 - x * x - y * y, 0.0))
    nrm = np.stack([x, -y, z], -1)
    out = np.stack([x, -y, np.full_like(x, -2.0)], -1)
    hit = (z > 0)[..., None]
    refl = 2.0 * nrm * nrm[..., 2:3] - np.array([0.0, 0.0, 1.0])
    turn = np.linalg.qr(r.standard_normal((3, 3)))[0]
    dirs = [(np.where(hit, d, out) @ turn).astype(np.float32) for d in (nrm, refl)]
    gys = r.standard_normal((case["levels"] + 1, s, s, 3), dtype=np.float32) / np.float32(s * s)
    return np.ascontiguousarray(env), dirs[0], dirs[1], gys


def _ibl(case, seed):
    env, nrm, refl, gys = (torch.from_numpy(a).cuda() for a in _ibl_inputs(case, seed))
    chain, src, levels = _ibl_shape(case)
    rough = [i / max(1, len(levels) - 1) for i in range(len(levels))]
    # the normalisers depend on the sizes alone: a program keeps them
    norms = [K.prefilter_conv_norm(_context(), w, h, *chain[src], r)
             for (w, h), r in zip(levels, rough)]
    return {"env": env, "nrm": nrm, "refl": refl, "gys": gys, "chain": chain, "src": src,
            "levels": levels, "rough": rough, "norms": norms}


def prepare(case, seed):
    state = {"silhouette": _silhouette, "texture": _texture, "pbr": _pbr, "surface": _surface,
             "ibl": _ibl}[case["kind"]](case, seed)
    state["kind"] = case["kind"]
    return state


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------

def _run_surface(s):
    case, ctx, tri = s["case"], s["ctx"], s["tri"]
    res = [case["height"], case["width"]]
    if s["mode"] == "soft":
        clip = s["clip"].detach().requires_grad_(True)
        soft = dr.rasterize_soft(ctx, clip, tri, res, radius_px=3.0, peels=case["peels"])
        clear = torch.ones_like(s["target"][..., 0])
        for k in range(case["peels"]):
            clear = clear * (1.0 - soft[:, k, ..., 3] * torch.sigmoid(soft[:, k, ..., 0]))
        image = 1.0 - clear
        loss = torch.mean((image - s["target"][..., 0]) ** 2)
        return {"soft": soft, "loss": loss, "grad": torch.autograd.grad(loss, clip)[0]}
    if s["mode"] == "aa":
        clip = s["clip"].detach().requires_grad_(True)
        rast, _ = dr.rasterize(ctx, clip, tri, resolution=res)
        mask = (rast[..., 3:4] > 0).float()
        image = dr.antialias(mask, rast, clip, tri, n_samples=case["samples"])
        leaf = clip
    elif s["mode"] == "color":
        leaf = s["color"].detach().requires_grad_(True)
        rast, _ = dr.rasterize(ctx, s["clip"], tri, resolution=res)
        image, _ = dr.interpolate(leaf, rast, tri)
    else:
        leaf = s["tex"].detach().requires_grad_(True)
        rast, _ = dr.rasterize(ctx, s["clip"], tri, resolution=res)
        uv, _ = dr.interpolate(s["uv"], rast, tri)
        image = dr.texture(leaf, uv) * (rast[..., 3:4] > 0)
    loss = torch.mean((image - s["target"]) ** 2)
    return {"rast": rast, "image": image, "loss": loss,
            "grad": torch.autograd.grad(loss, leaf)[0]}


def _run_ibl(s):
    ctx, chain, src = _context(), s["chain"], s["src"]
    pooled = [s["env"]]
    for _ in chain[1:]:
        pooled.append(K.avg_pool2x2(ctx, pooled[-1]))
    irr = K.irradiance_conv(ctx, pooled[-1], 32, 16)
    maps = [K.prefilter_conv(ctx, pooled[src], w, h, r, nrm)
            for (w, h), r, nrm in zip(s["levels"], s["rough"], s["norms"])]
    diffuse = K.equirect_sample(ctx, irr, s["nrm"])
    glossy = [K.equirect_sample(ctx, m, s["refl"]) for m in maps]
    # back from the lookups' gradients
    g_irr = K.equirect_sample_bwd(ctx, s["gys"][0], s["nrm"], 32, 16)
    g_maps = [K.equirect_sample_bwd(ctx, g, s["refl"], w, h)
              for g, (w, h) in zip(s["gys"][1:], s["levels"])]
    g_src = None
    for g, r, nrm in zip(g_maps, s["rough"], s["norms"]):
        part = K.prefilter_conv_bwd(ctx, g, *chain[src], r, nrm)
        g_src = part if g_src is None else g_src + part
    g = K.irradiance_conv_bwd(ctx, g_irr, *chain[-1])
    for k in range(len(chain) - 1, -1, -1):
        if k == src:
            g = g + g_src
        if k:
            g = K.avg_pool2x2_bwd(ctx, g, *chain[k - 1])
    return {"irr": irr, "maps": maps, "diffuse": diffuse, "glossy": glossy, "g_maps": g_maps,
            "g_env": g}


def run(state):
    if state["kind"] == "surface":
        return _run_surface(state)
    if state["kind"] == "ibl":
        return _run_ibl(state)
    state["fit"].step(1)
    return state["out"]


# --------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------

def _counts(case):
    """(vertices, faces) of the case's mesh"""
    if "stacks" in case:
        return ((case["stacks"] + 1) * (case["slices"] + 1),
                2 * (case["stacks"] - 1) * case["slices"])
    return 10 * 4 ** case["level"] + 2, 20 * 4 ** case["level"]


def work(case):
    kind = case["kind"]
    if kind == "ibl":
        chain, src, levels = _ibl_shape(case)
        px = case["size"] ** 2
        texels = sum(w * h for w, h in levels) + 512
        pairs = (texels - 512) * chain[src][0] * chain[src][1] + 512 * chain[-1][0] * chain[-1][1]
        # env, maps and normalisers, directions once, a lookup and a gradient per level and pixel
        n = case["levels"] + 1
        return {"bytes": 24 * chain[0][0] * chain[0][1] + 28 * texels + px * (24 + 24 * n),
                "flops": 2 * 30 * pairs + px * 60 * n}
    v, f = _counts(case)
    n = case["views"]
    if kind == "silhouette":
        px = case["size"] ** 2
        return {"bytes": px * (8 * n + 4) + 12 * f + 84 * v,
                "flops": n * (px * 40 + f * 300 + v * 60)}
    if kind == "texture":
        px, t = case["size"] ** 2, case["tex"] ** 2
        return {"bytes": 16 * px + 112 * t + 12 * f + 20 * v,
                "flops": n * (px * 120 + f * 150) + t * 40}
    if kind == "pbr":
        px, t, e = case["size"] ** 2, case["tex"] ** 2, case["env"] ** 2 // 2
        chain, src, levels = _ibl_shape(case)
        pairs = (sum(w * h for w, h in levels) * chain[src][0] * chain[src][1]
                 + 512 * chain[-1][0] * chain[-1][1])
        # mapped target in; parameters and moments in and out, gradients out
        return {"bytes": 12 * n * px + 2 * 84 * t + 84 * e + 12 * f + 32 * v,
                "flops": 600 * n * px + 60 * pairs + 60 * (2 * t + e)}
    px = n * case["height"] * case["width"]
    c = {"aa": 1, "color": case.get("channels"), "texture": 3, "soft": 1}[case["mode"]]
    mesh = 12 * f + 16 * n * v
    if case["mode"] == "soft":
        return {"bytes": mesh + 16 * n * v + px * (16 * case["peels"] + 4),
                "flops": px * case["peels"] * 150 + n * f * 400}
    leaf = {"aa": 16 * n * v, "color": 4 * c * v,
            "texture": 12 * case.get("tex", 0) ** 2}[case["mode"]]
    return {"bytes": mesh + 2 * leaf + px * (16 + 8 * c), "flops": px * (60 + 20 * c) + n * f * 150}


def tolerance(case):
    # ibl: the prefilter at roughness 0 is so narrow that the float32 rounding of its texel
    # directions shows: 1.6e-4 off the 64-bit maps and environment gradient
    if case["kind"] == "ibl":
        return {"rel": 5e-4, "max": 2e-2}
    # 32-bit interpolation and sums: vertex colours are 4e-6 off the 64-bit ones, their
    # gradient 4e-6. A face id, a covered pixel and a nearest texel are float32 decisions, that
    # may differ at the odd pixel
    return {"rel": 2e-5, "max": 1e-3, "differ": 1e-5}


# --------------------------------------------------------------------------
# The same in 64 bits
# --------------------------------------------------------------------------

def _raster64(clip, faces, h, w):
    """Per pixel the nearest face (-1: none) and its perspective-correct weights, z in [-w, w]."""
    with np.errstate(divide="ignore", invalid="ignore"):
        sx = (clip[:, 0] / clip[:, 3] * 0.5 + 0.5) * w
        sy = (clip[:, 1] / clip[:, 3] * 0.5 + 0.5) * h
        sz = clip[:, 2] / clip[:, 3]
    best = np.full((h, w), np.inf)
    face = np.full((h, w), -1)
    bary = np.zeros((h, w, 3))
    for f, (a, b, c) in enumerate(faces):
        x, y = sx[[a, b, c]], sy[[a, b, c]]
        area = (x[1] - x[0]) * (y[2] - y[0]) - (y[1] - y[0]) * (x[2] - x[0])
        x0, x1 = max(0, int(x.min() - 0.5)), min(w, int(x.max() + 1.5))
        y0, y1 = max(0, int(y.min() - 0.5)), min(h, int(y.max() + 1.5))
        if abs(area) < 1e-12 or x0 >= x1 or y0 >= y1:
            continue
        px, py = np.arange(x0, x1)[None, :] + 0.5, np.arange(y0, y1)[:, None] + 0.5
        l = [((x[(k + 1) % 3] - px) * (y[(k + 2) % 3] - py)
              - (y[(k + 1) % 3] - py) * (x[(k + 2) % 3] - px)) / area for k in range(3)]
        z = l[0] * sz[a] + l[1] * sz[b] + l[2] * sz[c]
        win = ((l[0] >= 0) & (l[1] >= 0) & (l[2] >= 0) & (abs(z) <= 1)
               & (z <= best[y0:y1, x0:x1]))
        q = np.stack([l[0] / clip[a, 3], l[1] / clip[b, 3], l[2] / clip[c, 3]], -1)
        q /= q.sum(-1, keepdims=True)
        best[y0:y1, x0:x1][win] = z[win]
        face[y0:y1, x0:x1][win] = f
        bary[y0:y1, x0:x1][win] = q[win]
    return face, bary


def _exact_surface(case, seed):
    """rasterize + interpolate (+ nearest texture), in 64 bits. The gather that carries the
    gradient back to a texture is a rule of its own and no adjoint: it has no such value; nor
    have face ids, where two faces hold a pixel on their common edge."""
    if case["mode"] not in ("color", "texture"):
        return None
    state = prepare(case, seed)
    clips = state["clip"].cpu().numpy().astype(np.float64)
    faces = state["tri"].cpu().numpy()
    target = state["target"].cpu().numpy().astype(np.float64)
    images, grad = [], None
    leaf = state["color" if case["mode"] == "color" else "tex"].cpu().numpy().astype(np.float64)
    uv = state["uv"].cpu().numpy().astype(np.float64) if "uv" in state else None
    for i, clip in enumerate(clips):
        face, q = _raster64(clip, faces, case["height"], case["width"])
        on = face >= 0
        corner = faces[np.maximum(face, 0)]
        if uv is None:
            image = (q[..., None] * leaf[corner]).sum(2) * on[..., None]
            if grad is None:
                grad = np.zeros_like(leaf)
            g = 2.0 * (image - target[i]) / target.size * on[..., None]
            for k in range(3):
                np.add.at(grad, corner[..., k][on], (q[..., k:k + 1] * g)[on])
        else:
            at = (q[..., None] * uv[corner]).sum(2) * on[..., None]
            t = np.clip(np.floor(at * case["tex"]).astype(int), 0, case["tex"] - 1)
            image = leaf[t[..., 1], t[..., 0]] * on[..., None]
        images.append(image)
    image = np.stack(images)
    return {"rast": None, "image": image, "loss": float(((image - target) ** 2).mean()),
            "grad": grad}


def _equirect64(w, h, device):
    v, u = torch.meshgrid((torch.arange(h, dtype=torch.float64, device=device) + 0.5) / h,
                          (torch.arange(w, dtype=torch.float64, device=device) + 0.5) / w,
                          indexing="ij")
    th, ph = v.reshape(-1) * math.pi, (u.reshape(-1) - 0.5) * 2 * math.pi
    return torch.stack([th.sin() * ph.cos(), th.cos(), th.sin() * ph.sin()], -1), th.sin()


def _lookup64(w, h, dirs):
    """Bilinear texel indices {P, 4} and weights {P, 4} of the directions."""
    d = dirs / dirs.norm(dim=-1, keepdim=True)
    x = (torch.atan2(d[:, 2], d[:, 0]) / (2 * math.pi) + 0.5) * w - 0.5
    y = torch.acos(d[:, 1].clamp(-1, 1)) / math.pi * h - 0.5
    ix, iy = x.floor(), y.floor()
    fx, fy = x - ix, y - iy
    at, wt = [], []
    for dy in (0, 1):
        for dx in (0, 1):
            at.append((iy.long() + dy).clamp(0, h - 1) * w + (ix.long() + dx) % w)
            wt.append((fx if dx else 1 - fx) * (fy if dy else 1 - fy))
    return torch.stack(at, -1), torch.stack(wt, -1)


def _pool64(x):
    h, w = x.shape[:2]
    x = torch.nn.functional.pad(x, (0, 0, 0, w % 2, 0, h % 2))
    return (x[0::2, 0::2] + x[1::2, 0::2] + x[0::2, 1::2] + x[1::2, 1::2]) * 0.25


def _exact_ibl(case, seed):
    env, nrm, refl, gys = (torch.from_numpy(a).cuda().double() for a in _ibl_inputs(case, seed))
    chain, src, levels = _ibl_shape(case)
    s = case["size"]
    nrm, refl, gys = nrm.reshape(-1, 3), refl.reshape(-1, 3), gys.reshape(-1, s * s, 3)
    pooled = [env]
    for _ in chain[1:]:
        pooled.append(_pool64(pooled[-1]))

    def back(gy, w, h, at, wt):
        out = torch.zeros(w * h, 3, dtype=torch.float64, device=gy.device)
        for k in range(4):
            out.index_add_(0, at[:, k], gy * wt[:, k:k + 1])
        return out

    res = {"maps": [], "glossy": [], "g_maps": []}
    sd, sa = _equirect64(*chain[-1], env.device)
    td, _ = _equirect64(32, 16, env.device)
    wts = (td @ sd.T).clamp(min=0) * sa * (2 * math.pi / (chain[-1][0] * chain[-1][1]))
    irr = wts @ pooled[-1].reshape(-1, 3)
    at, wt = _lookup64(32, 16, nrm)
    res["irr"] = irr.reshape(16, 32, 3)
    res["diffuse"] = (irr[at] * wt[..., None]).sum(1).reshape(s, s, 3)
    g = (wts.T @ back(gys[0], 32, 16, at, wt)).reshape(*chain[-1][::-1], 3)
    g_src = 0
    sd, sa = _equirect64(*chain[src], env.device)
    for i, (w, h) in enumerate(levels):
        alpha2 = max(i / max(1, len(levels) - 1), 0.045) ** 4
        td, _ = _equirect64(w, h, env.device)
        c = td @ sd.T
        d = (1 + c) * 0.5 * (alpha2 - 1) + 1
        wts = torch.where(c > 0, alpha2 / (math.pi * d * d) * c, torch.zeros_like(c)) * sa
        wts = wts / wts.sum(1, keepdim=True).clamp(min=1e-12)
        out = wts @ pooled[src].reshape(-1, 3)
        at, wt = _lookup64(w, h, refl)
        g_map = back(gys[i + 1], w, h, at, wt)
        g_src = g_src + wts.T @ g_map
        res["maps"].append(out.reshape(h, w, 3))
        res["glossy"].append((out[at] * wt[..., None]).sum(1).reshape(s, s, 3))
        res["g_maps"].append(g_map.reshape(h, w, 3))
    for k in range(len(chain) - 1, -1, -1):
        if k == src:
            g = g + g_src.reshape(*chain[src][::-1], 3)
        if k:
            w, h = chain[k - 1]
            g = (g * 0.25).repeat_interleave(2, 0)[:h].repeat_interleave(2, 1)[:, :w]
    res["g_env"] = g
    return res


def exact(case, seed):
    """A fit's step and a silhouette's gradient follow float32 decisions (the covering face, the
    hashed sample pixels), so that a 64-bit evaluation is one of other pixels: None."""
    if case["kind"] == "ibl":
        return _exact_ibl(case, seed)
    if case["kind"] == "surface":
        return _exact_surface(case, seed)
    return None

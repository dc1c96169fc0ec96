"""nvdiffrast-compatible differentiable ops over the library's HIP kernels
(python/dressi/torch/ops.py:95-698).

Each op runs the same per-op kernels the C ABI exports (rasterize,
LookupFaces/FaceFetch, Texture, AntiAlias, SoftClip/RasterizeSoft and their
backward kernels), stream-ordered on torch's current stream of the context's
device, with no host round trip. The backward of every op composes the
reference's backward kernels exactly as the reference's backward builder does
(src/core/build_backward.cpp:62-149): the same kernels, the same operand
order, gradient contributions summed in descending creation order of the
nodes that produced them. Every op runs the whole batch at once; per-signature
state lives in the context's `_engines`.
"""
from __future__ import annotations

import torch

from .. import ops as K
from .context import RasterizeHipContext
from .convert import (
    channels,
    clip_batch,
    image_batch,
    resolution_hw,
    to_dev,
)
from .provenance import InterpOrigin, RasterOrigin, origin, stamp


def _needs_grad(*tensors) -> bool:
    return torch.is_grad_enabled() and any(
        isinstance(t, torch.Tensor) and t.requires_grad for t in tensors)


class _Engine:
    """Per-signature state (the antialias backward's iteration counter), built
    once per key."""

    def __init__(self, **kw):
        self.__dict__.update(kw)


# ------------------------------- rasterize ---------------------------------


def rasterize(ctx: RasterizeHipContext, pos: torch.Tensor, tri: torch.Tensor, resolution,
              ranges=None, grad_db: bool = False):
    """Drop-in nvdiffrast rasterize (python/dressi/torch/ops.py:118-166):
    returns (rast, rast_db) with rast[..., :] = (u, v, z/w, triangle_id + 1),
    0 = background, rast_db zeros.

    The raster carries the corner barycentric constants (1,0), (0,1), (0,0)
    and (z, w) as perspective-correct attributes; z/w is 0 on background. Not
    differentiable w.r.t. `pos` (geometry gradients come from antialias /
    rasterize_soft)."""
    if ranges is not None:
        raise NotImplementedError("opendressi_amd.torch: range mode is not supported")
    del grad_db
    h, w = resolution_hw(resolution)
    pos_b = clip_batch(pos, ctx.device)
    md = ctx.mesh(tri)
    if md.n_verts > pos_b.shape[1]:
        raise IndexError(f"tri names vertex {md.n_verts - 1}, pos has {pos_b.shape[1]}")
    with ctx.lock:
        # every item in one pass
        rast, clip_vk = K.surface_rasterize(ctx._ctx, pos_b, md.faces_i, w, h)
    rast = rast.to(pos.device)
    stamp(rast, RasterOrigin(clip_vk=clip_vk, tri=tri, resolution=(h, w), ctx=ctx))
    return rast, torch.zeros_like(rast)


# ------------------------------ interpolate --------------------------------


class _InterpolateFn(torch.autograd.Function):
    @staticmethod
    def forward(fctx, attr, rast, vctx, md, rinfo):
        dev = vctx.device
        attr_d = to_dev(attr, dev, "attr")
        rast_d = to_dev(rast, dev, "rast")
        shared = attr_d.dim() == 2
        channels(attr_d.shape[-1], "attr")
        n = rast_d.shape[0]
        if attr_d.dim() not in (2, 3) or (not shared and attr_d.shape[0] < n):
            raise ValueError(f"attr must be [V, C] or [{n}, V, C], got {tuple(attr.shape)}")
        if not shared:
            attr_d = attr_d[:n]  # items past the raster's are not looked at
        with vctx.lock:
            # the whole batch in one launch
            out = K.surface_interpolate(vctx._ctx, attr_d, rast_d, md.faces_f)
        fctx.dressi = (vctx, md, rinfo, shared)
        fctx.save_for_backward(attr, rast)
        return out.to(attr.device)

    @staticmethod
    def backward(fctx, grad_out):
        vctx, md, rinfo, shared = fctx.dressi
        attr, rast = fctx.saved_tensors
        dev = vctx.device
        rast_d = to_dev(rast, dev, "rast")
        g = to_dev(grad_out, dev, "grad_out")
        with vctx.lock:
            g_attr = K.surface_interpolate_bwd(vctx._ctx, g, rast_d, rinfo.clip_vk, md.faces_f,
                                               md.vft, shared)
        return g_attr.to(attr.device), None, None, None, None


def interpolate(attr, rast, tri, rast_db=None, diff_attrs=None):
    """Drop-in nvdiffrast interpolate (python/dressi/torch/ops.py:279-301):
    returns (pixel_attr, None). attr is [V, C] (shared by the batch) or
    [N, V, C], C in 1..4; differentiable w.r.t. `attr` through the exact
    FaceFetch / LookupFaces backward. `rast` must come from rasterize()."""
    if rast_db is not None or diff_attrs is not None:
        raise NotImplementedError(
            "opendressi_amd.torch.interpolate: rast_db/diff_attrs are not supported")
    rinfo = origin(rast, RasterOrigin, "rasterize")
    vctx = rinfo.ctx
    md = vctx.mesh(tri)
    out = _InterpolateFn.apply(attr, rast, vctx, md, rinfo)
    stamp(out, InterpOrigin(attr=attr, raster=rinfo))
    return out, None


# -------------------------------- texture ----------------------------------


class _TextureFn(torch.autograd.Function):
    @staticmethod
    def forward(fctx, tex, uv, vctx, iinfo):
        dev = vctx.device
        tex_d = to_dev(tex, dev, "tex")
        if tex_d.dim() == 4:
            if tex_d.shape[0] != 1:
                raise NotImplementedError(
                    "opendressi_amd.torch.texture: per-item texture batches are not supported "
                    "(pass [H, W, C] or [1, H, W, C])")
            tex_d = tex_d[0]
        if tex_d.dim() != 3:
            raise ValueError(f"tex must be [H, W, C] or [1, H, W, C], got {tuple(tex.shape)}")
        channels(tex_d.shape[2], "tex")
        uv_d = to_dev(uv, dev, "uv")
        n, h, w, c = uv_d.shape
        if c != 2:
            raise ValueError(f"uv must have 2 components, got {c}")
        with vctx.lock:
            # the items' rows are one image's
            out = K.texture_nearest(vctx._ctx, tex_d, uv_d.view(n * h, w, 2))
        fctx.dressi = (vctx, iinfo)
        fctx.save_for_backward(tex, uv)
        return out.view(n, h, w, tex_d.shape[2]).to(tex.device)

    @staticmethod
    def backward(fctx, grad_out):
        vctx, iinfo = fctx.dressi
        tex, uv = fctx.saved_tensors
        dev = vctx.device
        th, tw = (tex.shape[1], tex.shape[2]) if tex.dim() == 4 else (tex.shape[0], tex.shape[1])
        uv_d = to_dev(uv, dev, "uv")
        g = to_dev(grad_out, dev, "grad_out")
        rinfo = iinfo.raster
        md = vctx.mesh(rinfo.tri)
        vtx_uv = to_dev(iinfo.attr, dev, "uv attr")
        n = uv_d.shape[0]
        if vtx_uv.shape[-1] != 2:
            raise ValueError("texture backward: the interpolated uv attribute must be [V, 2]")
        if vtx_uv.dim() == 3 and vtx_uv.shape[0] == 1:
            vtx_uv = vtx_uv[0]
        nv = min(vtx_uv.shape[-2], rinfo.clip_vk.shape[1])
        if md.n_verts > nv:
            raise IndexError(f"tri names vertex {md.n_verts - 1}, uv or pos has {nv}")
        clip = rinfo.clip_vk
        if vtx_uv.shape[-2] != clip.shape[1]:
            # vertices that no face names
            vtx_uv, clip = vtx_uv[..., :nv, :].contiguous(), clip[:, :nv].contiguous()
        with vctx.lock:
            g_tex = K.surface_texture_bwd(vctx._ctx, g, uv_d, vtx_uv, clip, md.faces_f, tw, th)
        if tex.dim() == 4:
            g_tex = g_tex.unsqueeze(0)
        return g_tex.to(tex.device), None, None, None


def texture(tex, uv, uv_da=None, mip_level_bias=None, mip=None, filter_mode="auto",
            boundary_mode="wrap", max_mip_level=None):
    """Drop-in nvdiffrast texture, nearest filtering with clamp-to-edge
    texel lookup (python/dressi/torch/ops.py:417-444). Differentiable w.r.t.
    `tex` through the inverse-UV gather, whose table is the mesh rasterized
    in UV space carrying its screen positions; `uv` must come from
    interpolate() (its provenance names the mesh and context)."""
    if uv_da is not None or mip_level_bias is not None or mip is not None:
        raise NotImplementedError("opendressi_amd.torch.texture: mipmaps unsupported")
    if filter_mode not in ("auto", "nearest"):
        raise NotImplementedError(
            f"opendressi_amd.torch.texture: filter_mode='{filter_mode}' unsupported "
            "(nearest only)")
    del boundary_mode, max_mip_level
    iinfo = origin(uv, InterpOrigin, "interpolate")
    vctx = iinfo.raster.ctx
    if uv.dim() == 3:
        uv = uv.unsqueeze(0)
    return _TextureFn.apply(tex, uv, vctx, iinfo)


# ------------------------------- antialias ---------------------------------


def _batch_pos(pos: torch.Tensor, device) -> torch.Tensor:
    """Per-item clip positions (N, V, 4), or the one (V, 4) every item shares."""
    pos_b = clip_batch(pos, device)
    return pos_b if pos_b.shape[0] > 1 else pos_b[0]


class _AntiAliasFn(torch.autograd.Function):
    @staticmethod
    def forward(fctx, color, rast, pos, vctx, md, rinfo, n_samples, boost):
        dev = vctx.device
        col_d = image_batch(to_dev(color, dev, "color"), "color")
        rast_d = to_dev(rast, dev, "rast")
        channels(col_d.shape[3], "color")
        if col_d.shape[1:3] != rast_d.shape[1:3] or col_d.shape[0] > rast_d.shape[0]:
            raise ValueError(f"color {tuple(color.shape)} does not match rast {tuple(rast.shape)}")
        pos_d = _batch_pos(pos, dev)
        with vctx.lock:
            # the whole batch in one launch
            out = K.surface_antialias(vctx._ctx, col_d, rast_d, pos_d, md.faces_f)
        fctx.dressi = (vctx, md, n_samples, boost)
        fctx.save_for_backward(color, rast, pos)
        return out.to(color.device)

    @staticmethod
    def backward(fctx, grad_out):
        vctx, md, n_samples, boost = fctx.dressi
        color, rast, pos = fctx.saved_tensors
        need_color, _, need_pos = fctx.needs_input_grad[:3]
        dev = vctx.device
        col_d = image_batch(to_dev(color, dev, "color"), "color")
        rast_d = to_dev(rast, dev, "rast")
        pos_d = _batch_pos(pos, dev)
        g = image_batch(to_dev(grad_out, dev, "grad_out"), "grad_out")
        n, h, w, c = col_d.shape
        key = ("antialias", h, w, md.n_faces, md.n_verts, c, n, n_samples)
        eng = vctx.engine(key, lambda: _Engine(iter_seed=0))
        with vctx.lock:
            # each backward pass advances the stochastic sampler's jitter;
            # items get distinct seeds so their sample patterns decorrelate
            eng.iter_seed += 1
            if need_color:
                g_col = K.surface_antialias_bwd_img(vctx._ctx, g, rast_d, pos_d, md.faces_f)
            if need_pos:
                gp = K.surface_antialias_bwd_pos(vctx._ctx, g, col_d, rast_d, pos_d, md.faces_f,
                                                 md.vft, eng.iter_seed * n, n_samples, boost)
        out_gc = out_gp = None
        if need_color:
            out_gc = (g_col[0] if color.dim() == 3 else g_col).to(color.device)
        if need_pos:
            out_gp = (gp.sum(dim=0) if pos.dim() == 2 else gp).to(pos.device)
        return out_gc, None, out_gp, None, None, None, None, None


def antialias(color, rast, pos, tri, topology_hash=None, pos_gradient_boost=1.0, n_samples=8):
    """Drop-in nvdiffrast antialias, screen-space edge AA
    (python/dressi/torch/ops.py:562-581). Differentiable w.r.t. `color` and
    `pos`; `n_samples` selects the vertex backward: 0 = exact scan, > 0 =
    n jittered edge samples per face per backward (wide partials + column
    sum). `topology_hash` is accepted and ignored."""
    del topology_hash
    rinfo = origin(rast, RasterOrigin, "rasterize")
    vctx = rinfo.ctx
    md = vctx.mesh(tri)
    return _AntiAliasFn.apply(color, rast, pos, vctx, md, rinfo, max(int(n_samples), 0),
                              float(pos_gradient_boost))


# ------------------------------ rasterize_soft -----------------------------


class _RasterizeSoftFn(torch.autograd.Function):
    @staticmethod
    def forward(fctx, pos, vctx, md, resolution, radius_px, peels):
        h, w = resolution
        pos_b = clip_batch(pos, vctx.device)
        if md.n_verts > pos_b.shape[1]:
            raise IndexError(f"tri names vertex {md.n_verts - 1}, pos has {pos_b.shape[1]}")
        with vctx.lock:
            # every item and peel from one setup
            out = K.surface_rasterize_soft(vctx._ctx, pos_b, md.faces_f, w, h, radius_px, peels)
        fctx.dressi = (vctx, md, radius_px)
        fctx.save_for_backward(pos, out)
        return out.to(pos.device)

    @staticmethod
    def backward(fctx, grad_out):
        vctx, md, radius_px = fctx.dressi
        pos, out = fctx.saved_tensors
        dev = vctx.device
        pos_b = clip_batch(pos, dev)
        g = to_dev(grad_out, dev, "grad_out")
        with vctx.lock:
            g_pos = K.surface_soft_bwd(vctx._ctx, g, to_dev(out, dev, "out"), pos_b, md.faces_f,
                                       md.vft, radius_px)
        if pos.dim() == 2:
            g_pos = g_pos.sum(dim=0)
        return g_pos.to(pos.device), None, None, None, None, None


def rasterize_soft(ctx, pos, tri, resolution, radius_px=3.0, peels=1):
    """HardSoftRas soft rasterization (python/dressi/torch/ops.py:682-698).

    Returns [N, K, H, W, 4] with channels (signed_dist_px, face_id,
    hard_depth, coverage) per depth-peel layer K. Differentiable w.r.t. `pos`
    through the signed-distance channel (the exact adjacency-bounded gather
    backward); compose silhouettes in torch, e.g.
    `cov * torch.sigmoid(dist / sigma)`."""
    h, w = resolution_hw(resolution)
    if peels < 1:
        raise ValueError("peels must be >= 1")
    md = ctx.mesh(tri)
    return _RasterizeSoftFn.apply(pos, ctx, md, (h, w), float(radius_px), int(peels))

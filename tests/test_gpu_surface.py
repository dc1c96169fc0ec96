"""The torch surface's fused ops (dressi_surface_*) against the per-op entry points they stand
for, composed as the reference's surface composes them: the same bits at the edges of the fused
kernels' steps (boxes of several steps, screens that end inside a workgroup, sample counts that
are no multiple of eight, batches whose contributions take several summation levels)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import opendressi_amd as od
    c = od.Context(0)
    yield c
    c.close()


def _same(a, b, what):
    """The same values, NaN in the same places."""
    torch.cuda.synchronize()
    assert a.shape == b.shape, (what, a.shape, b.shape)
    differ = ~((a == b) | (a.isnan() & b.isnan()))
    assert not bool(differ.any()), \
        f"{what}: {int(differ.sum())} values differ, max {float((a - b).abs().max()):.3g}"


def _scene(level, n, seed, spread=0.1):
    """n random orbit views of an icosphere: clip positions (n, V, 4) with z in [-w, w], faces
    as int32 and float ids, the adjacency."""
    import opendressi_amd as od
    pos, faces = od.icosphere(level)
    rng = np.random.default_rng(seed)
    pos = pos * (1.0 + spread * rng.standard_normal((len(pos), 1)))
    mvp = od.orbit_cameras(1, n, seed)[0].reshape(n, 4, 4).astype(np.float64)
    clip = np.concatenate([pos, np.ones((len(pos), 1))], 1)[None] @ mvp
    clip[..., 2] = 2.0 * clip[..., 2] - clip[..., 3]
    vf = od.vertex_faces_tex(faces, len(pos))
    dev = lambda a, t: torch.from_numpy(np.ascontiguousarray(a, t)).cuda()
    return (dev(clip, np.float32), dev(faces, np.int32), dev(faces, np.float32),
            dev(vf, np.float32))


def _to_vk(clip):
    out = clip.clone()
    out[..., 2] = 0.5 * (clip[..., 2] + clip[..., 3])
    return out


SCENES = [(0, 1, 40, 64), (2, 3, 61, 97), (4, 7, 33, 18), (3, 2, 1, 200), (1, 5, 130, 131)]


@pytest.mark.parametrize("level,n,h,w", SCENES)
def test_surface_rasterize(ctx, level, n, h, w):
    """Against Rasterize of the unwelded mesh with the corner constants and (z, w)."""
    from opendressi_amd import ops as K
    print(f"[surface rasterize] level {level} {n}x{h}x{w}", flush=True)
    clip, fi, ff, _ = _scene(level, n, level + n)
    nf = len(fi)
    rast, vk = K.surface_rasterize(ctx, clip, fi, w, h)
    _same(vk, _to_vk(clip), "clip")
    idx = fi.reshape(-1).long()
    corner = torch.tensor([[1.0, 0.0], [0.0, 1.0], [0.0, 0.0]]).repeat(nf, 1).cuda()
    attr = torch.cat([corner.expand(n, -1, -1), clip[:, idx][:, :, 2:4]], 2).contiguous()
    seq = torch.arange(nf * 3, dtype=torch.float32).reshape(-1, 3).cuda()
    g, tid = K.rasterize_batch(ctx, _to_vk(clip)[:, idx].contiguous(), attr, seq, w, h,
                               with_face_id=True)
    zw = g[..., 2] / (g[..., 3] + (1.0 - (tid > 0.5).float()))
    _same(rast, torch.stack([g[..., 0], g[..., 1], zw, tid], -1), "rast")
    assert (tid > 0).any()
    ctx.synchronize()


@pytest.mark.parametrize("level,n,h,w", SCENES)
@pytest.mark.parametrize("nc,shared", [(1, True), (2, False), (3, True), (4, False), (4, True)])
def test_surface_interpolate(ctx, level, n, h, w, nc, shared):
    from opendressi_amd import ops as K
    from opendressi_amd.torch.convert import sum_contribs
    print(f"[surface interpolate] level {level} {n}x{h}x{w}x{nc} shared {shared}", flush=True)
    clip, fi, ff, vf = _scene(level, n, level + n)
    rast, vk = K.surface_rasterize(ctx, clip, fi, w, h)
    gen = torch.Generator(device="cuda").manual_seed(nc)
    nv = clip.shape[1]
    attr = torch.randn((nv, nc) if shared else (n, nv, nc), device="cuda", generator=gen)
    u, v, tid = rast[..., 0:1], rast[..., 1:2], rast[..., 3].contiguous()

    def per_face(a, k):
        return (K.lookup_faces(ctx, a, ff, k) if a.dim() == 2
                else K.lookup_faces_batch(ctx, a, ff, k, n))

    pix = [K.face_fetch_batch(ctx, per_face(attr, k), tid) for k in range(3)]
    _same(K.surface_interpolate(ctx, attr, rast, ff),
          u * pix[0] + v * pix[1] + ((1.0 - u) - v) * pix[2], "forward")
    g = torch.randn((n, h, w, nc), device="cuda", generator=gen)
    gp = [g * u, g * v, g * ((1.0 - u) - v)]
    prj = [per_face(vk, k) for k in range(3)]
    seeds = torch.zeros(n, device="cuda")
    parts = [K.lookup_faces_bwd_batch(ctx, K.face_fetch_bwd_batch(
        ctx, gp[k].contiguous(), tid, prj[0], prj[1], prj[2], seeds, 1.0, 0), ff, vf, k)
        for k in (2, 1, 0)]
    per_item = [[p[i] for p in parts] for i in range(n)]
    ref = (sum_contribs([p for parts_i in reversed(per_item) for p in parts_i]) if shared
           else torch.stack([sum_contribs(p) for p in per_item], 0))
    _same(K.surface_interpolate_bwd(ctx, g, rast, vk, ff, vf, shared), ref, "backward")
    ctx.synchronize()


@pytest.mark.parametrize("level,n,h,w", SCENES)
@pytest.mark.parametrize("nc,samples,shared", [(1, 8, False), (3, 0, False), (2, 5, True),
                                               (4, 17, False)])
def test_surface_antialias(ctx, level, n, h, w, nc, samples, shared):
    """Forward and colour gradient against the per-op batch, the position gradient against the
    wide partials, ColSum, the z remap's transpose and the boost."""
    from opendressi_amd import ops as K
    print(f"[surface antialias] level {level} {n}x{h}x{w}x{nc} n={samples} {shared}", flush=True)
    clip, fi, ff, vf = _scene(level, 1 if shared else n, level + n)
    rast, vk = K.surface_rasterize(ctx, clip.expand(n, -1, -1).contiguous(), fi, w, h)
    pos, vk = (clip[0], vk[0].contiguous()) if shared else (clip, vk)
    tid = rast[..., 3].contiguous()
    gen = torch.Generator(device="cuda").manual_seed(nc)
    img = torch.rand((n, h, w, nc), device="cuda", generator=gen)
    g = torch.randn((n, h, w, nc), device="cuda", generator=gen)
    _same(K.surface_antialias(ctx, img, rast, pos, ff), K.antialias_batch(ctx, img, tid, vk, ff),
          "forward")
    _same(K.surface_antialias_bwd_img(ctx, g, rast, pos, ff),
          K.antialias_bwd_img_batch(ctx, g, tid, vk, ff), "colour gradient")
    got = K.surface_antialias_bwd_pos(ctx, g, img, rast, pos, ff, vf, 3 * n, samples, 1.5)
    seeds = torch.tensor([float(3 * n + i) for i in range(n)], device="cuda")
    ref = K.antialias_bwd_vtx_batch(ctx, g, img, tid, vk, ff, vf, seeds, samples, samples > 0)
    if samples:
        ref = K.col_sum_batch(ctx, ref)
    ref[..., 3] += 0.5 * ref[..., 2]
    ref[..., 2] *= 0.5
    assert float(ref.abs().max()) > 0 or h == 1
    _same(got, ref * 1.5, "position gradient")
    ctx.synchronize()


@pytest.mark.parametrize("samples", [1, 2, 3, 4, 5, 9])
@pytest.mark.parametrize("drop", [0, 1, 2, 3])
def test_surface_antialias_faces_of_a_wave(ctx, samples, drop):
    """Four, two or one face to a wave by the sample count, face counts that leave a wave's last
    groups empty, fewer samples than a group takes at once and more; against the wide partials
    and ColSum."""
    import opendressi_amd as od
    from opendressi_amd import ops as K
    print(f"[surface antialias] {samples} samples, {drop} faces dropped", flush=True)
    n, h, w = 2, 61, 97
    clip, fi, ff, _ = _scene(2, n, 11)
    fi, ff = fi[:len(fi) - drop].contiguous(), ff[:len(ff) - drop].contiguous()
    vf = torch.from_numpy(od.vertex_faces_tex(ff.cpu().numpy(), clip.shape[1])).cuda()
    rast, vk = K.surface_rasterize(ctx, clip, fi, w, h)
    gen = torch.Generator(device="cuda").manual_seed(samples)
    img = torch.rand((n, h, w, 3), device="cuda", generator=gen)
    g = torch.randn((n, h, w, 3), device="cuda", generator=gen)
    got = K.surface_antialias_bwd_pos(ctx, g, img, rast, clip, ff, vf, 5 * n, samples, 1.0)
    seeds = torch.tensor([float(5 * n + i) for i in range(n)], device="cuda")
    ref = K.col_sum_batch(ctx, K.antialias_bwd_vtx_batch(ctx, g, img, rast[..., 3].contiguous(),
                                                         vk, ff, vf, seeds, samples, True))
    assert float(ref.abs().max()) > 0
    _same(got, ref, "position gradient")
    ctx.synchronize()


def _peel_threshold(rs, radius_px):
    dist, z, cov = rs[..., 0], rs[..., 2], rs[..., 3]
    ge = (dist >= 0.0).to(torch.float32)
    near = torch.clamp(z, 0.0, 1.0) * 0.5
    far = torch.clamp(dist * (-1.0 / radius_px), 0.0, 1.0) * 0.5 + 0.5
    return (cov * (ge * near + (1.0 - ge) * far)).contiguous()


@pytest.mark.parametrize("level,n,h,w,peels,radius", [
    (0, 1, 40, 64, 1, 3.0), (2, 3, 61, 97, 6, 2.7), (3, 2, 33, 130, 2, 3.0), (1, 4, 1, 200, 3, 0.4),
    # 65 screens' bins: a second group of items
    (0, 65, 512, 512, 2, 3.0)])
def test_surface_rasterize_soft(ctx, monkeypatch, level, n, h, w, peels, radius):
    """Every item and peel against SoftClip / RasterizeSoft with the peel thresholds, and the
    position gradient against GatherDistGrad, ColSum, the peels' sum and the remap's transpose,
    with the items' gradients all at once and in groups."""
    from opendressi_amd import ops as K
    from opendressi_amd.torch.convert import clip_grad_vk_to_gl, sum_contribs
    print(f"[surface soft] level {level} {n}x{h}x{w} peels {peels} r {radius}", flush=True)
    clip, fi, ff, vf = _scene(level, n, level + n, 0.0)
    nf = len(fi)
    fid = torch.arange(nf, dtype=torch.float32).repeat_interleave(3).cuda()
    seq = torch.arange(nf * 3, dtype=torch.float32).reshape(-1, 3).cuda()
    got = K.surface_rasterize_soft(ctx, clip, ff, w, h, radius, peels)
    gen = torch.Generator(device="cuda").manual_seed(n)
    gy = torch.randn(got.shape, device="cuda", generator=gen)
    g_pos = K.surface_soft_bwd(ctx, gy, got, clip, ff, vf, radius)
    for i in (range(n) if n < 10 else (0, n - 2, n - 1)):
        vk = _to_vk(clip[i])
        sc = K.soft_clip(ctx, vk, ff, w, h, radius)
        prev, parts = None, []
        for k in range(peels):
            rs = K.rasterize_soft(ctx, sc, fid, seq, vk, ff, w, h, radius, prev)
            _same(got[i, k], rs, f"item {i} peel {k}")
            prev = _peel_threshold(rs, radius)
            parts.insert(0, K.col_sum(ctx, K.gather_dist_grad(ctx, gy[i, k].contiguous(), rs, vk,
                                                              ff, vf, radius, True)))
        _same(g_pos[i], clip_grad_vk_to_gl(sum_contribs(parts)), f"item {i} gradient")
    assert float(g_pos.abs().max()) > 0
    for group in (1, 3):
        monkeypatch.setattr(K, "_SCRATCH_BYTES", group * 36 * peels * nf + 1)
        _same(K.surface_soft_bwd(ctx, gy, got, clip, ff, vf, radius), g_pos, f"groups of {group}")
    ctx.synchronize()


def test_surface_soft_bwd_scratch(ctx):
    """The gradient's scratch stays within 256 MB where the batch's corner sums would take 755."""
    from opendressi_amd import ops as K
    print("[surface soft] scratch", flush=True)
    n, peels = 64, 4
    clip, fi, ff, vf = _scene(6, n, 3, 0.0)
    rs = torch.zeros((n, peels, 8, 8, 4), device="cuda")
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = K.surface_soft_bwd(ctx, rs, rs, clip, ff, vf, 3.0)
    torch.cuda.synchronize()
    took = torch.cuda.max_memory_allocated() - before
    assert 36 * n * peels * len(fi) > 750e6
    assert took <= out.numel() * 4 + (256 << 20) + (16 << 20), took
    ctx.synchronize()


@pytest.mark.parametrize("n,h,w,tw,th,nc,shared", [
    (1, 40, 64, 33, 17, 3, True), (5, 61, 97, 64, 64, 4, True), (3, 130, 33, 1, 7, 1, False),
    (2, 1, 200, 129, 50, 2, True), (17, 20, 20, 40, 40, 3, False)])
def test_surface_texture_bwd(ctx, monkeypatch, n, h, w, tw, th, nc, shared):
    """The nearest texture's gradient against UvAsClip / ScreenAttr / Rasterize /
    GatherByInverseUV per item and the contributions' sum, shared and per-item uv, uv that leave
    part of the texture to the dilation; with the items all at once and in groups."""
    import opendressi_amd as od
    from opendressi_amd import ops as K
    from opendressi_amd.torch.convert import sum_contribs
    print(f"[surface texture] {n}x{h}x{w} tex {tw}x{th}x{nc} shared {shared}", flush=True)
    pos, uv, faces = od.uv_sphere(12, 9)
    mvp = od.orbit_cameras(1, n, n)[0].reshape(n, 4, 4).astype(np.float64)
    clip = np.concatenate([pos, np.ones((len(pos), 1))], 1)[None] @ mvp
    clip[..., 2] = 2.0 * clip[..., 2] - clip[..., 3]
    dev = lambda a, t=np.float32: torch.from_numpy(np.ascontiguousarray(a, t)).cuda()
    ff, fi = dev(faces), dev(faces, np.int32)
    rast, vk = K.surface_rasterize(ctx, dev(clip), fi, w, h)
    vtx_uv = dev(0.05 + 0.8 * uv)
    if not shared:
        vtx_uv = torch.stack([vtx_uv * (0.5 + 0.5 / (i + 1)) for i in range(n)])
    pix_uv = K.surface_interpolate(ctx, vtx_uv, rast, ff)
    gen = torch.Generator(device="cuda").manual_seed(nc)
    g = torch.randn((n, h, w, nc), device="cuda", generator=gen)
    parts = []
    for i in reversed(range(n)):
        vuv = vtx_uv if shared else vtx_uv[i]
        one = torch.ones_like(vuv[:, :1])
        uv_clip = torch.cat([vuv * 2.0 - 1.0, one * 0.5, one], 1).contiguous()
        inv = K.rasterize(ctx, uv_clip, K.screen_attr(ctx, vk[i].contiguous(), w, h), ff, tw, th)
        parts.append(K.texture_nearest_bwd(ctx, g[i].contiguous(), inv, pix_uv[i].contiguous()))
    got = K.surface_texture_bwd(ctx, g, pix_uv, vtx_uv, vk, ff, tw, th)
    _same(got, sum_contribs(parts), "texture gradient")
    assert float(got.abs().max()) > 0 or h == 1
    item_bytes = 16 * (th * tw + 2 * len(pos))
    for group in (1, 2, 3):
        monkeypatch.setattr(K, "_SCRATCH_BYTES", group * item_bytes + 1)
        _same(K.surface_texture_bwd(ctx, g, pix_uv, vtx_uv, vk, ff, tw, th), got,
              f"groups of {group}")
    ctx.synchronize()


def test_surface_texture_bwd_scratch(ctx):
    """The scratch of a batch stays within its bound: beside the items' contributions (half a
    gigabyte here) 256 MB of the inverse uv images' two gigabytes."""
    import opendressi_amd as od
    from opendressi_amd import ops as K
    print("[surface texture] scratch", flush=True)
    n, t = 128, 1024
    pos, uv, faces = od.uv_sphere(12, 9)
    dev = lambda a, t=np.float32: torch.from_numpy(np.ascontiguousarray(a, t)).cuda()
    clip = dev(np.concatenate([pos, np.ones((len(pos), 1))], 1)).expand(n, -1, -1).contiguous()
    g = torch.ones((n, 8, 8, 1), device="cuda")
    pix_uv = torch.full((n, 8, 8, 2), 0.5, device="cuda")
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    K.surface_texture_bwd(ctx, g, pix_uv, dev(uv), clip, dev(faces), t, t)
    torch.cuda.synchronize()
    took = torch.cuda.max_memory_allocated() - before
    assert took <= 4 * n * t * t + (256 << 20) + (16 << 20), took
    ctx.synchronize()


@pytest.mark.parametrize("sw,sh", [(0, 4), (4, 0), (0, 0), (1, 1)])
def test_texture_bwd_of_an_empty_screen(ctx, sw, sh):
    """GatherByInverseUV of a screen without columns or rows, through the C entry point (a torch
    tensor without elements has no address): anchors everywhere, yet zeros and no read; one pixel
    finds its texel."""
    from opendressi_amd import _lib as L
    print(f"[texture bwd] empty screen {sw}x{sh}", flush=True)
    tw, th, nc = 5, 3, 3
    gy = torch.full((4, 4, nc), 7.0, device="cuda")
    uv = torch.full((4, 4, 2), 0.5, device="cuda")
    inv = torch.tensor([0.5, 1.5, 1.0, 0.0], device="cuda").repeat(th, tw, 1)
    out = torch.full((th, tw, nc), 3.0, device="cuda")
    ctx.use_torch_stream()
    p = lambda t: L.C.c_void_p(t.data_ptr())
    L.check(L.lib.dressi_texture_nearest_bwd(ctx.handle, p(gy), nc, sw, sh, p(inv), tw, th, p(uv),
                                             p(out)))
    ref = torch.zeros_like(out)
    if sw and sh:
        ref[1, 2] = 7.0  # uv (0.5, 0.5)
    _same(out, ref, "out")
    ctx.synchronize()


@pytest.mark.parametrize("w,h,ok", [(46341, 46341, True), (65535, 65534, True),
                                    (65536, 65536, False)])
def test_screen_limits(ctx, w, h, ok):
    """Screens of 2^31 pixels and more, which the per-op entry points take, are no reason to
    refuse a call; 2^32 are (a pixel's index would not fit). Batches and meshes of nothing, which
    return after the checks."""
    from opendressi_amd import _lib as L
    print(f"[surface limits] {w}x{h}", flush=True)
    some = torch.zeros(64, device="cuda")
    p, lib = L.C.c_void_p(some.data_ptr()), L.lib
    ctx.use_torch_stream()
    calls = [
        lambda: lib.dressi_surface_interpolate(ctx.handle, p, 1, 3, 0, p, w, h, 0, p, 1, p),
        lambda: lib.dressi_surface_interpolate_bwd(ctx.handle, p, 3, p, w, h, 0, p, 1, 0, p, 1, p, 1,
                                                   1, 1, p, p),
        lambda: lib.dressi_surface_soft_bwd(ctx.handle, p, p, 1, p, 1, 0, p, 1, p, 1, 1, 3.0, w, h,
                                            p, p),
        lambda: lib.dressi_gather_dist_grad(ctx.handle, p, p, p, 0, p, 1, p, 1, 3.0, 1, w, h, p)]
    for call in calls:
        assert (call() == 0) == ok, lib.dressi_last_error()
    ctx.synchronize()

"""GPU parity of the texture path (C3) against the oracle and the reference
fixtures, through the C ABI (per-op entry points and the fused dressi_tex_*
plan): bit-exact images, gradients and Adam state."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _exact(a, b, what):
    assert a.shape == b.shape, (what, a.shape, b.shape)
    if not np.array_equal(a, b):
        d = np.abs(a.astype(np.float64) - b)
        idx = np.unravel_index(d.argmax(), d.shape)
        raise AssertionError(f"{what}: {int((d > 0).sum())} values differ, max {d.max():.3g} at "
                             f"{idx}: got {a[idx]} want {b[idx]}")


@pytest.fixture(scope="module")
def ctx():
    import opendressi_amd as od
    c = od.Context(0)
    yield c
    c.close()


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda()


def host(t):
    import torch
    torch.cuda.synchronize()
    return t.cpu().numpy()


def test_texture_ops_match_reference_fixtures(ctx, golden):
    from opendressi_amd import ops
    g = golden("tex_unit.npz")
    print("[tex ops] fixtures", flush=True)
    for nc in (1, 3, 4):
        _exact(host(ops.texture_bilinear(ctx, dev(g[f"in_bl{nc}_tex"]), dev(g[f"in_bl{nc}_uv"]))),
               g[f"out_bl{nc}"], f"bilinear n={nc}")
    for name in ("g_small", "g_sparse"):
        got = host(ops.texture_bilinear_bwd(ctx, dev(g[f"in_{name}_gy"]), dev(g[f"in_{name}_iv"]),
                                            dev(g[f"in_{name}_uv"])))
        _exact(got, g[f"out_{name}"], name)
    import opendressi_amd as od
    pos, uv, faces = od.uv_sphere(16, 8)
    _exact(pos, g["out_uvs16_pos"], "uv sphere pos")
    _exact(uv, g["out_uvs16_uv"], "uv sphere uv")
    _exact(faces, g["out_uvs16_faces"], "uv sphere faces")


@pytest.mark.parametrize("seed", [0, 1])
def test_texture_ops_match_oracle(ctx, oracle, seed):
    from opendressi_amd import ops
    print(f"[tex ops] random seed={seed}", flush=True)
    rng = np.random.default_rng(seed)
    tex = rng.random((37, 53, 4)).astype(np.float32)
    uv = (rng.random((61, 47, 2)) * 1.2 - 0.1).astype(np.float32)
    _exact(host(ops.texture_bilinear(ctx, dev(tex), dev(uv))), oracle.texture_bilinear(tex, uv),
           "bilinear")
    gy = rng.standard_normal((61, 47, 4)).astype(np.float32)
    iv = np.zeros((37, 53, 4), np.float32)
    iv[..., 0] = rng.random((37, 53)) * 51 - 2
    iv[..., 1] = rng.random((37, 53)) * 65 - 2
    iv[..., 2] = (rng.random((37, 53)) < 0.5).astype(np.float32)
    uv2 = rng.random((61, 47, 2)).astype(np.float32)
    _exact(host(ops.texture_bilinear_bwd(ctx, dev(gy), dev(iv), dev(uv2))),
           oracle.gather_inv_uv_bilinear(gy, iv, uv2), "gather")
    clip = np.concatenate([rng.standard_normal((100, 3)), rng.random((100, 1)) + 0.5],
                          1).astype(np.float32)
    _exact(host(ops.screen_attr(ctx, dev(clip), 97, 61)), oracle.screen_attr(clip, 97, 61),
           "screen attr")


@pytest.mark.parametrize("seed", [0, 1])
def test_texture_nearest_ops_match_oracle(ctx, oracle, seed):
    """F::Texture (nearest, clamp to edge) and GatherByInverseUV, bit-exact,
    on random uv (some outside [0, 1]) and a half-empty inverse-UV table."""
    from opendressi_amd import ops
    print(f"[tex nearest ops] random seed={seed}", flush=True)
    rng = np.random.default_rng(100 + seed)
    for nc in (1, 3, 4):
        tex = rng.random((37, 53, nc)).astype(np.float32)
        uv = (rng.random((61, 47, 2)) * 1.2 - 0.1).astype(np.float32)
        _exact(host(ops.texture_nearest(ctx, dev(tex), dev(uv))),
               oracle.texture_nearest(tex, uv), f"nearest nc={nc}")
        gy = rng.standard_normal((61, 47, nc)).astype(np.float32)
        iv = np.zeros((37, 53, 4), np.float32)
        iv[..., 0] = rng.random((37, 53)) * 51 - 2
        iv[..., 1] = rng.random((37, 53)) * 65 - 2
        iv[..., 2] = (rng.random((37, 53)) < 0.5).astype(np.float32)
        uv2 = rng.random((61, 47, 2)).astype(np.float32)
        _exact(host(ops.texture_nearest_bwd(ctx, dev(gy), dev(iv), dev(uv2))),
               oracle.gather_inv_uv(gy, iv, uv2), f"gather nearest nc={nc}")


FAR = (3.4e38, 1e20, 3e9, 2147483648.0, 2147483520.0, 2147483008.0, 2147482880.0, 1e6)


@pytest.mark.parametrize("op", ["nearest", "bilinear"])
def test_far_anchors(ctx, oracle, op):
    """Inverse-UV anchors at infinity, at the largest integers and just off the screen beside
    ordinary ones, on one axis or both: their windows hold no pixel, as one at (-100, -100)."""
    from opendressi_amd import ops
    print(f"[tex far anchors] {op}", flush=True)
    rng = np.random.default_rng(3)
    h, w, th, tw = 61, 47, 37, 53
    gy = rng.standard_normal((h, w, 3)).astype(np.float32)
    uv = rng.random((h, w, 2)).astype(np.float32)
    iv = np.zeros((th, tw, 4), np.float32)
    iv[..., 0] = rng.random((th, tw)) * 61 - 7
    iv[..., 1] = rng.random((th, tw)) * 75 - 7
    iv[..., 2] = (rng.random((th, tw)) < 0.7).astype(np.float32)
    near = iv.copy()
    far = np.array([np.inf, *FAR], np.float32)
    far = np.concatenate([far, -far])
    for axes in ((0,), (1,), (0, 1)):
        at = rng.random((th, tw)) < 0.15
        near[at, :2] = -100.0
        for a in axes:
            iv[at, a] = rng.choice(far, int(at.sum()))
    gpu, ref = {"nearest": (ops.texture_nearest_bwd, oracle.gather_inv_uv),
                "bilinear": (ops.texture_bilinear_bwd, oracle.gather_inv_uv_bilinear)}[op]
    want = ref(gy, near, uv)
    assert np.abs(want).max() > 0
    _exact(host(gpu(ctx, dev(gy), dev(iv), dev(uv))), want, op)
    ctx.synchronize()


def test_far_bilinear_lookups(ctx, oracle):
    """uv at infinity and at the largest integers beside ordinary ones: the pixels of the others
    are the oracle's, those of the far ones read the texture's edge (whatever their weights)."""
    from opendressi_amd import ops
    print("[tex far uv] bilinear", flush=True)
    rng = np.random.default_rng(4)
    tex = rng.random((37, 53, 4)).astype(np.float32)
    uv = (rng.random((61, 47, 2)) * 1.4 - 0.2).astype(np.float32)
    uv[:3] = rng.choice(np.array([1e3, -1e3, 1e5, -1e5], np.float32), (3, 47, 2))
    far = np.array([np.inf, *FAR[:-1]], np.float32)
    at = rng.random((61, 47)) < 0.2
    odd = uv.copy()
    odd[at] = rng.choice(np.concatenate([far, -far]), (int(at.sum()), 2))
    want = oracle.texture_bilinear(tex, uv)
    got = host(ops.texture_bilinear(ctx, dev(tex), dev(odd)))
    _exact(got[~at], want[~at], "bilinear")
    ctx.synchronize()


@pytest.mark.parametrize("value,ok", [(np.inf, False), (-1e20, False), (np.nan, True), (1e6, True)])
def test_fit_refuses_uv_without_a_texel(ctx, value, ok):
    """A texture fit's lookups take any finite texel index of ordinary size: a uv at infinity, or
    whose index would pass 2^30, is refused where the mesh is set."""
    import opendressi_amd as od
    pos, uv, faces = od.uv_sphere(8, 6)
    uv = uv.copy()
    uv[7, 1] = value
    tex = np.full((16, 16, 4), 0.5, np.float32)
    print(f"[tex fit] uv {value}", flush=True)
    make = lambda: od.TextureFit(ctx, pos, uv, faces, od.orbit_cameras(1, 2, 3), 32, tex, tex)
    if ok:
        fit = make()
        fit.step(1)
        ctx.synchronize()
        fit.close()
    else:
        with pytest.raises(od.DressiError, match="uv"):
            make()


def _fit(ctx, g, images=True):
    import opendressi_amd as od
    return od.TextureFit(ctx, g["in_pos"], g["in_uv"], g["in_faces"], g["in_mvps"],
                         int(g["in_cfg"][0]), g["in_gt"], g["in_tex0"], lr=float(g["in_cfg"][2]),
                         keep_images=images, keep_grad=True)


def test_tex_first_iteration_matches_reference(ctx, golden):
    from opendressi_amd import _lib as L
    g = golden("tex_uvs16_64px_3view_3it.npz")
    print("[tex fixture] first iteration", flush=True)
    fit = _fit(ctx, g)
    fit.step(1)
    ctx.synchronize()
    _exact(fit.read(L.TEX_UV), g["out_uv0"], "g_uv")
    _exact(fit.read(L.TEX_PRED), g["out_pred0"], "pred")
    _exact(fit.read(L.TEX_TARGET), g["out_target0"], "target")
    _exact(fit.read(L.TEX_LOSS), g["out_lossimg0"], "loss image")
    _exact(fit.read(L.TEX_GRAD), g["out_grad0"], "texture gradient")
    fit.close()


@pytest.mark.parametrize("name", ["tex_uvs16_64px_3view_3it.npz", "tex_uvs32_8view_128px_3it.npz",
                                  "tex_uvs16_64px_20it.npz"])
def test_tex_trajectory_matches_reference(ctx, golden, name):
    g = golden(name)
    iters = int(g["in_cfg"][1])
    print(f"[tex trajectory] {name} iters={iters}", flush=True)
    fit = _fit(ctx, g, images=False)
    losses = []
    for _ in range(iters):
        fit.step(1)
        losses.append(fit.loss())
    tex, m, v, t = fit.state()
    fit.close()
    assert t == float(iters)
    _exact(tex, g["out_tex"], "tex")
    _exact(m, g["out_m"], "m")
    _exact(v, g["out_v"], "v")
    np.testing.assert_allclose(losses, g["out_loss"], rtol=1e-5)


def test_tex_graph_replay_equals_eager(ctx, golden):
    from opendressi_amd import _lib as L
    g = golden("tex_uvs32_8view_128px_3it.npz")
    a, b = _fit(ctx, g, images=False), _fit(ctx, g, images=False)
    for i in range(3):
        a.step(1, graph=True)
        b.step(1, graph=False)
        ctx.synchronize()
        ta, _, va, sa = a.state()
        tb, _, vb, sb = b.state()
        assert np.array_equal(ta, tb) and np.array_equal(va, vb) and sa == sb, i
        assert np.array_equal(a.read(L.TEX_GRAD), b.read(L.TEX_GRAD))
    a.close()
    b.close()


def test_tex_c3_full_size_matches_oracle(ctx, oracle):
    """1024^2 x 8 views, UV sphere 128 x 64, 1024^2 RGBA texture (the C3
    workload): images, loss image and texture gradient of one iteration,
    then the Adam state after a second."""
    import opendressi_amd as od
    from opendressi_amd import _lib as L
    w = od.TEX_WORKLOADS["c3"]
    pos, uv, faces, mvps, gt, tex0 = od.make_tex_scene(w)
    mvps = mvps[:2]
    print("[tex full-size] c3 2 iterations", flush=True)
    fit = od.TextureFit(ctx, pos, uv, faces, mvps, w.screen, gt, tex0, lr=w.lr, keep_images=True,
                        keep_grad=True)
    fit.step(1)
    ctx.synchronize()
    got = {k: fit.read(b) for k, b in (("uv0", L.TEX_UV), ("pred0", L.TEX_PRED),
                                       ("target0", L.TEX_TARGET), ("lossimg0", L.TEX_LOSS),
                                       ("grad0", L.TEX_GRAD))}
    fit.step(1)
    tex, m, v, t = fit.state()
    fit.close()
    ref = oracle.tex_fit(pos, uv, faces, mvps, w.screen, gt, tex0, lr=w.lr, iters=2)
    for k in got:
        _exact(got[k], ref[k], k)
    _exact(tex, ref["tex"], "tex")
    _exact(m, ref["m"], "m")
    _exact(v, ref["v"], "v")


def test_texture_nearest_of_many_pixels(ctx):
    """A batch of 2^32 pixels and more (65 views of 8192 x 8192, looked up as one image), more
    than a launch has threads: every pixel is written."""
    import torch

    from opendressi_amd import ops
    n, s = 65, 8192
    print(f"[texture] {n}x{s}x{s} pixels", flush=True)
    tex = torch.tensor([[1.0, 2.0], [3.0, 4.0]], device="cuda").view(2, 2, 1)
    uv = torch.full((n * s, s, 2), 0.25, device="cuda")
    uv[-1, -1] = 0.75
    uv[1 << 18, 0] = torch.tensor([0.75, 0.25])  # the second launch's first pixel
    out = ops.texture_nearest(ctx, tex, uv)
    assert float(out[-1, -1, 0]) == 4.0 and float(out[1 << 18, 0, 0]) == 2.0
    del uv
    for i in range(0, n * s, 1 << 16):
        part = out[i:i + (1 << 16)]
        ones = int((part == 1.0).sum())
        assert ones == part.numel() - (i == 1 << 18) - (i + len(part) == n * s), i

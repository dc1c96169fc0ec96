"""GPU parity of the split-sum IBL ops (C5) against the reference fixtures and
the oracle, through the C ABI per-op entry points.

Bit-exact: AvgPool2x2 and its VJP, IrradianceConv / PrefilterConvNorm /
PrefilterConv and their transposes (one thread per output texel, the
reference's loop order, the reference's texel-centre direction tables),
EquirectSample, PrefilterEnv and the BRDF LUT (per-direction uv from device
atan2f / acosf and the Schlick power from a device powf(x, 5) that return
what the host C library returns). Within 1e-5 (written per test): the per-op
EquirectSample VJP, an exact fixed-point sum where the reference adds floats
in band order (the fused PBR plan adds them in the reference's order).
The fused PBR plan is bit-exact against the oracle and, for the images and
the loss, against the reference's outputs.
"""
import math

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


def _close(a, b, tol, what):
    """|a - b| <= tol * max|b|."""
    assert a.shape == b.shape, (what, a.shape, b.shape)
    d = np.abs(a.astype(np.float64) - b).max()
    m = float(np.abs(b).max())
    assert d <= tol * max(m, 1e-30), f"{what}: max diff {d:.3g} vs max {m:.3g} (tol {tol})"


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


def smooth_map(h, w, nc, seed):
    """A smooth positive equirect map (low-frequency sinusoids, periodic in u)."""
    rng = np.random.default_rng(seed)
    yy, xx = np.meshgrid((np.arange(h) + 0.5) / h, (np.arange(w) + 0.5) / w, indexing="ij")
    out = np.zeros((h, w, nc))
    for c in range(nc):
        a, b, p = rng.integers(1, 3), rng.integers(1, 3), rng.random() * 6.28
        out[..., c] = 1.0 + 0.5 * np.sin(2 * math.pi * a * xx + p) * np.sin(math.pi * b * yy)
    return out.astype(np.float32)


def test_ibl_ops_match_reference_fixtures(ctx, golden):
    from opendressi_amd import ops
    g = golden("ibl_unit.npz")
    print("[ibl ops] fixtures: pool / irradiance / prefilter", flush=True)
    for name in ("pool_odd", "pool_even"):
        x, gy = g[f"in_{name}_x"], g[f"in_{name}_gy"]
        _exact(host(ops.avg_pool2x2(ctx, dev(x))), g[f"out_{name}"], name)
        _exact(host(ops.avg_pool2x2_bwd(ctx, dev(gy), x.shape[1], x.shape[0])),
               g[f"out_{name}_bwd"], name + " bwd")
    env, g84, g168 = dev(g["in_env"]), dev(g["in_g84"]), dev(g["in_g168"])
    _exact(host(ops.irradiance_conv(ctx, env, 8, 4)), g["out_irr"], "irradiance")
    _exact(host(ops.irradiance_conv_bwd(ctx, g84, 16, 8)), g["out_irr_bwd"], "irradiance bwd")
    for i, rough in enumerate((0.0, 0.5, 1.0)):
        _exact(host(ops.prefilter_conv(ctx, env, 16, 8, rough)), g[f"out_pref{i}_16"],
               f"pref {rough}")
        _exact(host(ops.prefilter_conv(ctx, env, 8, 4, rough)), g[f"out_pref{i}_8"],
               f"pref {rough}")
        _exact(host(ops.prefilter_conv_bwd(ctx, g168, 16, 8, rough)), g[f"out_pref{i}_16_bwd"],
               f"pref bwd {rough}")
        _exact(host(ops.prefilter_conv_bwd(ctx, g84, 16, 8, rough)), g[f"out_pref{i}_8_bwd"],
               f"pref bwd {rough}")
    print("[ibl ops] fixtures: equirect / prefilter env / lut", flush=True)
    for nc in (1, 3, 4):
        m, d, gy = g[f"in_eq{nc}_map"], g[f"in_eq{nc}_dir"], g[f"in_eq{nc}_gy"]
        _exact(host(ops.equirect_sample(ctx, dev(m), dev(d))), g[f"out_eq{nc}"],
               f"equirect n={nc}")
        _close(host(ops.equirect_sample_bwd(ctx, dev(gy), dev(d), m.shape[1], m.shape[0])),
               g[f"out_eq{nc}_bwd"], 1e-5, f"equirect bwd n={nc}")
    _exact(host(ops.prefilter_env(ctx, env, 8, 4, 0.5, 64)), g["out_prefenv"], "prefilter env")
    _exact(host(ops.brdf_lut(ctx, 16, 16, 64)), g["out_lut16"], "lut 16")
    _exact(host(ops.brdf_lut(ctx, 64, 64, 512)), g["out_lut64"], "lut 64")


@pytest.mark.parametrize("shape", [(64, 128, 128, 64), (32, 64, 32, 16)])
def test_ibl_convs_match_oracle_at_map_sizes(ctx, oracle, shape):
    """The C5 map sizes: prefilter levels from a 128 x 64 source, the
    irradiance map 32 x 16 from 64 x 32 (bit-exact)."""
    from opendressi_amd import ops
    sh, sw, oh, ow = shape
    print(f"[ibl convs] src {sw}x{sh} -> {ow}x{oh}", flush=True)
    env = smooth_map(sh, sw, 3, 5)
    rng = np.random.default_rng(6)
    gy = rng.standard_normal((oh, ow, 3)).astype(np.float32)
    for rough in (0.0, 0.6):
        _exact(host(ops.prefilter_conv(ctx, dev(env), ow, oh, rough)),
               oracle.prefilter_conv(env, ow, oh, rough), f"pref {rough}")
        _exact(host(ops.prefilter_conv_bwd(ctx, dev(gy), sw, sh, rough)),
               oracle.prefilter_conv(env, ow, oh, rough, gy), f"pref bwd {rough}")
    _exact(host(ops.irradiance_conv(ctx, dev(env), ow // 2, oh // 2)),
           oracle.irradiance_conv(env, ow // 2, oh // 2), "irradiance")


def _same_floats(a, b, what):
    """The same bits, NaN (of any kind) in the same places."""
    assert np.array_equal(np.isnan(a), np.isnan(b)), f"{what}: NaN in other places"
    _exact(np.where(np.isnan(a), 0.0, a), np.where(np.isnan(b), 0.0, b), what)


@pytest.mark.parametrize("shape", [
    # (source w, h, output w, h, channels). More than 2048 outputs: workgroups of 8 and chunks of
    # 128 sources, whole, one past and one short of them, single texels, every channel count,
    # forward ...
    (43, 3, 2051, 1, 4), (127, 1, 2050, 1, 1), (1, 1, 2049, 1, 2), (128, 2, 683, 3, 3),
    # ... and back (the source's texels are the outputs)
    (2049, 1, 1, 1, 4), (683, 3, 127, 1, 1), (2050, 1, 129, 1, 2), (2056, 1, 257, 1, 3),
    # both; at most 2048 outputs, which take the other form
    (2049, 1, 2049, 1, 1), (16, 8, 4, 2, 3), (43, 3, 1, 1, 4), (129, 1, 3, 3, 1),
    (128, 2, 9, 1, 2), (127, 3, 17, 5, 3), (1, 1, 16, 8, 3)])
def test_ibl_conv_chunks_match_oracle(ctx, oracle, shape):
    """Bit for bit, forward and back; an infinite and a NaN source value reach the sums that the
    reference's order brings them to."""
    from opendressi_amd import ops
    sw, sh, ow, oh, nc = shape
    print(f"[ibl conv chunks] {shape}", flush=True)
    rng = np.random.default_rng(sw)
    env = rng.random((sh, sw, nc), dtype=np.float32)
    gy = rng.standard_normal((oh, ow, nc)).astype(np.float32)

    def check(env, gy):
        for rough in (0.0, 0.7):
            _same_floats(host(ops.prefilter_conv(ctx, dev(env), ow, oh, rough)),
                         oracle.prefilter_conv(env, ow, oh, rough), f"pref {rough}")
            _same_floats(host(ops.prefilter_conv_bwd(ctx, dev(gy), sw, sh, rough)),
                         oracle.prefilter_conv(env, ow, oh, rough, gy), f"bwd {rough}")
        _same_floats(host(ops.irradiance_conv(ctx, dev(env), ow, oh)),
                     oracle.irradiance_conv(env, ow, oh), "irradiance")
        _same_floats(host(ops.irradiance_conv_bwd(ctx, dev(gy), sw, sh)),
                     oracle.irradiance_conv(env, ow, oh, gy), "irradiance bwd")

    check(env, gy)
    env.flat[0], gy.flat[-1] = np.inf, np.nan
    check(env, gy)


@pytest.mark.parametrize("shape", [
    # (source w, h, output w, h, channels): the form for few outputs, its chunks of 256 sources
    # (one, up to the four that are loaded ahead and past them) and workgroups of 4 outputs, on
    # both sides of 2048 outputs
    (255, 1, 5, 1, 3), (256, 1, 4, 1, 4), (257, 2, 3, 1, 2), (256, 4, 1, 1, 3), (205, 5, 7, 1, 1),
    (128, 9, 2047, 1, 3), (33, 8, 2048, 1, 4), (33, 8, 2049, 1, 3)])
def test_ibl_conv_few_outputs_match_oracle(ctx, oracle, shape):
    """Bit for bit, forward and back (where the source's texels are the outputs)."""
    from opendressi_amd import ops
    sw, sh, ow, oh, nc = shape
    print(f"[ibl conv few] {shape}", flush=True)
    rng = np.random.default_rng(ow)
    env = rng.random((sh, sw, nc), dtype=np.float32)
    gy = rng.standard_normal((oh, ow, nc)).astype(np.float32)
    _exact(host(ops.prefilter_conv(ctx, dev(env), ow, oh, 0.4)),
           oracle.prefilter_conv(env, ow, oh, 0.4), "pref")
    _exact(host(ops.prefilter_conv_bwd(ctx, dev(gy), sw, sh, 0.4)),
           oracle.prefilter_conv(env, ow, oh, 0.4, gy), "bwd")
    _exact(host(ops.irradiance_conv(ctx, dev(env), ow, oh)),
           oracle.irradiance_conv(env, ow, oh), "irradiance")
    _exact(host(ops.irradiance_conv_bwd(ctx, dev(gy), sw, sh)),
           oracle.irradiance_conv(env, ow, oh, gy), "irradiance bwd")


def test_ibl_tables_beyond_the_kept_ones(oracle):
    """More map sizes than a context keeps tables for (64), the first ones again after they had to
    give place, and the tables of one context after another's end: the oracle's bits each time."""
    import opendressi_amd as od
    from opendressi_amd import ops
    print("[ibl tables] 70 sizes", flush=True)
    env = smooth_map(4, 8, 3, 9)
    for _ in range(2):
        c = od.Context(0)
        for w in list(range(1, 71)) + [1, 2, 70]:
            _exact(host(ops.irradiance_conv(c, dev(env), w, 1)), oracle.irradiance_conv(env, w, 1),
                   f"irradiance {w}x1")
        _exact(host(ops.prefilter_env(c, dev(env), 8, 4, 0.5, 64)),
               oracle.prefilter_env(env, 8, 4, 0.5, 64), "prefilter env")
        c.close()


def test_equirect_sample_smooth_map_and_vjp(ctx, oracle):
    """A 512 x 256 smooth map sampled at 96 x 80 random directions (bit for
    bit), and the map VJP of 1024 x 8 directions (gradients 1e-5)."""
    from opendressi_amd import ops
    print("[equirect] 512x256 smooth map", flush=True)
    m = smooth_map(256, 512, 3, 7)
    rng = np.random.default_rng(8)
    d = rng.standard_normal((80, 96, 3)).astype(np.float32)
    _exact(host(ops.equirect_sample(ctx, dev(m), dev(d))), oracle.equirect_sample(m, d),
           "equirect")
    d2 = rng.standard_normal((8, 1024, 3)).astype(np.float32)
    gy = rng.standard_normal((8, 1024, 3)).astype(np.float32)
    got = host(ops.equirect_sample_bwd(ctx, dev(gy), dev(d2), 64, 32))
    _close(got, oracle.equirect_sample(np.zeros((32, 64, 3), np.float32), d2, gy), 1e-5,
           "equirect vjp")
    # determinism: the fixed-point sum does not depend on the atomics' order
    again = host(ops.equirect_sample_bwd(ctx, dev(gy), dev(d2), 64, 32))
    _exact(again, got, "equirect vjp rerun")


@pytest.mark.parametrize("shape", [
    # (map w, h, channels, dir rows, dir columns): the whole map in a workgroup's LDS, at its
    # largest (6144 entries) and smallest; one entry past it (hash table) and with four channels;
    # a list of directions; images smaller than a tile and one past its edges
    (64, 32, 3, 33, 65), (1, 1, 1, 5, 7), (4, 2, 3, 70, 31), (2049, 1, 3, 40, 40),
    (97, 49, 4, 64, 33), (3073, 2, 1, 1, 1500), (128, 64, 3, 1, 1), (128, 64, 2, 1025, 1),
    # 16 pixels per texel and more: the smaller hash table with four sums per texel, of 512 and
    # (four channels) 256 texels; one pixel row short of it
    (128, 64, 3, 512, 512), (97, 49, 4, 300, 260), (97, 49, 4, 292, 260)])
@pytest.mark.parametrize("coherent", [True, False])
def test_equirect_vjp_tiles(ctx, oracle, shape, coherent):
    """The map VJP over the forms of its tile sums: the bits of the same 64-bit sums on the host,
    and the oracle's ordered float sums within their rounding, 2^-24 of the sum of magnitudes for
    each of a texel's (at most 4 pixels each) terms. Incoherent directions overflow the hash
    table."""
    from opendressi_amd import ops
    mw, mh, nc, h, w = shape
    print(f"[equirect vjp] map {mw}x{mh}x{nc} dirs {h}x{w} coherent {coherent}", flush=True)
    rng = np.random.default_rng(mw + h)
    if coherent:
        y, x = np.meshgrid(np.arange(h) / 40.0, np.arange(w) / 50.0, indexing="ij")
        d = np.stack([np.cos(x), 0.3 + y, np.sin(x) + 0.1], -1).astype(np.float32)
    else:
        d = rng.standard_normal((h, w, 3)).astype(np.float32)
    d[0, 0] = 0.0  # no direction: no contribution
    gy = (rng.standard_normal((h, w, nc)) * 10.0 ** rng.uniform(-3, 3, (h, w, 1))).astype(np.float32)
    zero = np.zeros((mh, mw, nc), np.float32)
    got = host(ops.equirect_sample_bwd(ctx, dev(gy), dev(d), mw, mh))
    ref = oracle.equirect_sample(zero, d, gy)
    size = oracle.equirect_sample(zero, d, np.abs(gy)).astype(np.float64)
    # the fixed point itself rounds each term to 2^-62 of max|gy| times the pixels
    bar = 4.0 * h * w * (2.0 ** -24 * size + 2.0 ** -61 * h * w * float(np.abs(gy).max()))
    err = np.abs(got.astype(np.float64) - ref)
    assert (err <= bar).all(), (float(err.max()), float((err - bar).max()))
    _exact(got, oracle.equirect_vjp_fixed(d, gy, mw, mh), "64-bit sums")


def test_equirect_vjp_of_a_long_list(ctx):
    """2^27 + 33 directions in one column and in one row: the same sums, so the same bits. A thread
    per pixel of a square tile would pass a launch's 2^32 threads here."""
    import torch

    from opendressi_amd import ops
    n = (1 << 27) + 33
    print(f"[equirect vjp] list of {n}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(1)
    d = torch.randn((n, 3), device="cuda", generator=gen)
    gy = torch.randn((n, 1), device="cuda", generator=gen)
    column = ops.equirect_sample_bwd(ctx, gy.view(n, 1, 1), d.view(n, 1, 3), 8, 4)
    row = ops.equirect_sample_bwd(ctx, gy.view(1, n, 1), d.view(1, n, 3), 8, 4)
    _exact(host(column), host(row), "column and row")
    assert float(row.abs().min()) > 0


def test_ibl_conv_of_many_outputs(ctx):
    """108 M outputs, more than a launch has threads for five waves of eight: the irradiance of
    one texel, the cosine to its direction."""
    from opendressi_amd import ops
    ow, oh = 16384, 6600
    print(f"[ibl conv] {ow}x{oh} outputs", flush=True)
    got = ops.irradiance_conv(ctx, dev(np.full((1, 1, 1), 0.5, np.float32)), ow, oh)
    phi = ((np.arange(ow) + 0.5) / ow - 0.5) * 2.0 * np.pi
    for y in (0, 1, 3275, 3276, 3277, oh // 2, oh - 1):
        want = np.pi * np.maximum(np.sin((y + 0.5) / oh * np.pi) * np.cos(phi), 0.0)
        # float32 directions: a few ulp of 1, scaled
        assert np.abs(host(got[y, :, 0]) - want).max() < 3e-6, y


# ---- the fused C5 plan -------------------------------------------------------

def _scene(g):
    keys = ("pos", "normal", "uv", "faces", "mvps", "frames", "light", "gt_albedo", "gt_mr",
            "gt_env", "albedo0", "mr0", "env0")
    sc = {k: g["in_" + k] for k in keys}
    sc.update(screen=int(g["in_screen"]), levels=int(g["in_levels"]), lr=float(g["in_lr"]))
    return sc


@pytest.mark.parametrize("name", ["pbr_ico2_48px_2view_3it.npz", "pbr_ico3_96px_3view_2it.npz"])
def test_pbr_plan_matches_reference_fixtures(ctx, golden, name):
    """Against the reference's own outputs: target, prediction and loss bit
    for bit (the shading forward, the C library's transcendentals and F::Mean's
    reduction order restated); first-iteration texture / env gradients within
    1e-4 of the largest entry and the parameters after the fixture's
    iterations within 1e-5: the plan's per-pixel shading backward adds its
    terms in the oracle's hand-derived order, not the reference autodiff's
    (the oracle itself sits within those bars of the reference)."""
    from opendressi_amd.pbr import PbrFit
    g = golden(name)
    iters = len(g["out_loss"])
    print(f"[pbr plan] {name}: set-up", flush=True)
    fit = PbrFit(ctx, _scene(g), keep_pred=True, keep_grad=True)
    import opendressi_amd._lib as L
    if "out_target0" in g:
        _exact(fit.read(L.PBR_TARGET)[..., :3], g["out_target0"], "target")
    print(f"[pbr plan] {name}: step 1", flush=True)
    fit.step(1, graph=False)
    fit.synchronize()
    if "out_pred0" in g:
        _exact(fit.read(L.PBR_PRED)[..., :3], g["out_pred0"], "pred")
    _exact(np.array([fit.loss()], np.float32), g["out_loss"][:1], "loss")
    _close(fit.read(L.PBR_G_ALBEDO)[..., :3], g["out_g_albedo0"], 1e-4, "g albedo")
    _close(fit.read(L.PBR_G_MR)[..., :3], g["out_g_mr0"], 1e-4, "g mr")
    _close(fit.read(L.PBR_G_ENV)[..., :3], g["out_g_env0"], 1e-4, "g env")
    print(f"[pbr plan] {name}: steps 2..{iters}", flush=True)
    fit.step(iters - 1, graph=False)
    alb, mr, env, t = fit.state()
    assert t == float(iters)
    for x, y, what in ((alb, g["out_albedo"], "albedo"), (mr, g["out_mr"], "mr"),
                       (env, g["out_env"], "env")):
        d = float(np.abs(x.astype(np.float64) - y).max())
        assert d <= 1e-5, f"{what}: max diff {d:.3g} (tol 1e-5)"
    fit.close()


@pytest.mark.parametrize("name,chunks", [("pbr_ico2_48px_2view_3it.npz", None),
                                         ("pbr_ico3_96px_3view_2it.npz", None),
                                         ("pbr_ico3_96px_3view_2it.npz", "1")])
def test_pbr_plan_matches_oracle_bit_for_bit(ctx, oracle, golden, monkeypatch, name, chunks):
    """The fused plan against the oracle's C5 fit (or_pbr_fit: the reference's
    per-pixel order, band partials + TileSum, view order, sequential
    convolutions, the C library's atan2f / acosf / powf) on the fixture
    scenes: target, prediction, the loss, first-iteration gradients and the
    parameters after the fixture's iterations identical bit for bit. With
    `chunks` = 1 the map gather takes per-tile position lists for every band
    of more than 1024 positions (at 96 px: prefilter level 0 and the env),
    as it does for the large bands at full size."""
    from opendressi_amd.pbr import PbrFit
    import opendressi_amd._lib as L
    if chunks is not None:
        monkeypatch.setenv("DRESSI_PBR_GATHER_CHUNKS", chunks)
    g = golden(name)
    iters = len(g["out_loss"])
    sc = _scene(g)
    print(f"[pbr plan vs oracle] {name}: {iters} iterations", flush=True)
    want = oracle.pbr_fit(sc, iters=iters, want_images=True)
    fit = PbrFit(ctx, sc, keep_pred=True, keep_grad=True)
    _exact(fit.read(L.PBR_TARGET)[..., :3], want["target0"], "target")
    fit.step(1, graph=False)
    fit.synchronize()
    _exact(fit.read(L.PBR_PRED)[..., :3], want["pred0"], "pred")
    _exact(np.array([fit.loss()], np.float32), want["loss"][:1], "loss")
    _exact(fit.read(L.PBR_G_ALBEDO)[..., :3], want["g_albedo0"], "g albedo")
    _exact(fit.read(L.PBR_G_MR)[..., :3], want["g_mr0"], "g mr")
    _exact(fit.read(L.PBR_G_ENV)[..., :3], want["g_env0"], "g env")
    fit.step(iters - 1, graph=True)
    alb, mr, env, t = fit.state()
    fit.close()
    assert t == float(iters)
    _exact(alb, want["albedo"], "albedo")
    _exact(mr, want["mr"], "mr")
    _exact(env, want["env"], "env")


def test_pbr_plan_graph_replay_is_deterministic(ctx, golden):
    """Three graph replays and three eager iterations from the same state give
    bit-identical parameters (every sum in a fixed order)."""
    from opendressi_amd.pbr import PbrFit
    g = golden("pbr_ico2_48px_2view_3it.npz")
    sc = _scene(g)
    print("[pbr plan] graph vs eager", flush=True)
    fit = PbrFit(ctx, sc)
    fit.step(3, graph=True)
    a = fit.state()
    fit.set_state(sc["albedo0"], sc["mr0"], sc["env0"])
    for _ in range(3):
        fit.step(1, graph=False)
    b = fit.state()
    for x, y, what in zip(a[:3], b[:3], ("albedo", "mr", "env")):
        _exact(x, y, what)
    fit.close()

"""GPU parity of GatherDistGrad (dressi_gather_dist_grad) against the
reference fixture and the oracle, through the C ABI: bit-exact wide partials
and {V,1} sums."""
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


def test_gather_dist_grad_matches_reference_fixture(ctx, golden, oracle):
    from opendressi_amd import ops
    g = golden("ds_unit.npz")
    r = float(g["in_cfg"][1])
    for i in range(3):
        print(f"[dist grad] fixture scene {i}", flush=True)
        args = (dev(g[f"in_gy{i}"]), dev(g[f"in_rs{i}"]), dev(g[f"in_clip{i}"]), dev(g["in_faces"]),
                dev(g["in_vf"]), r)
        _exact(host(ops.gather_dist_grad(ctx, *args, wide=True)), g[f"out_wide{i}"], f"wide {i}")
        flat = oracle.gather_dist_grad(g[f"in_gy{i}"], g[f"in_rs{i}"], g[f"in_clip{i}"],
                                       g["in_faces"], g["in_vf"], wide=False)
        _exact(host(ops.gather_dist_grad(ctx, *args, wide=False)), flat, f"flat {i}")
    ctx.synchronize()


@pytest.mark.parametrize("level,s,seed", [(2, 64, 0), (3, 97, 1)])
def test_gather_dist_grad_matches_oracle(ctx, oracle, level, s, seed):
    from opendressi_amd import ops
    print(f"[dist grad] random level={level} s={s} seed={seed}", flush=True)
    rng = np.random.default_rng(seed)
    pos, faces = oracle.icosphere(level)
    proj = oracle.perspective_vk(45.0 * 3.14159265 / 180.0, 1.0, 0.1, 10.0)
    eye = [rng.standard_normal() * 0.6, rng.standard_normal() * 0.6, 2.5]
    clip = oracle.transform_to_clip(pos, oracle.mat4_mul(proj, oracle.look_at(eye)))
    nf = len(faces)
    fid = np.repeat(np.arange(nf, dtype=np.float32), 3)[:, None]
    fs = np.arange(3 * nf, dtype=np.float32).reshape(nf, 3)
    vf = oracle.vertex_faces_tex(faces, len(pos))
    soft = oracle.soft_clip(clip, faces, s, s, 3.0)
    rs = oracle.rasterize_soft(soft, fid, fs, clip, faces, s, s, 3.0)
    gy = rng.standard_normal((s, s, 4)).astype(np.float32)
    gy[rng.random((s, s)) < 0.3, 0] = 0.0
    for wide in (True, False):
        got = host(ops.gather_dist_grad(ctx, dev(gy), dev(rs), dev(clip), dev(faces), dev(vf),
                                        3.0, wide=wide))
        _exact(got, oracle.gather_dist_grad(gy, rs, clip, faces, vf, wide=wide),
               f"wide={wide}")
    ctx.synchronize()


@pytest.mark.parametrize("h,w", [(8, 8), (37, 129), (80, 50)])
def test_gather_dist_grad_boxes_and_rows(ctx, oracle, h, w):
    """Faces whose boxes are the whole screen (many steps of 512 pixels, more than 64 hits a
    step) or a few pixels, a vertex of more than 64 faces, faces that repeat a vertex, rows that
    hold a face twice or one that is not theirs: bit for bit against the oracle."""
    from opendressi_amd import ops
    print(f"[dist grad] boxes {h}x{w}", flush=True)
    rng = np.random.default_rng(h)
    n_fan = 70
    ang = np.linspace(0.0, 2.0 * np.pi, n_fan, endpoint=False)
    pos = np.concatenate([[[0.0, 0.0, 0.5]],
                          np.stack([0.9 * np.cos(ang), 0.9 * np.sin(ang), 0 * ang + 0.4], 1),
                          rng.uniform(-1, 1, (12, 3)) * [1.2, 1.2, 0.4] + [0, 0, 0.5]])
    clip = np.concatenate([pos, np.ones((len(pos), 1))], 1).astype(np.float32)
    clip *= rng.uniform(0.5, 2.0, (len(pos), 1)).astype(np.float32)
    fan = [(0, 1 + i, 1 + (i + 1) % n_fan) for i in range(n_fan)]
    k = 1 + n_fan
    faces = np.array(fan + [(k, k + 1, k + 2), (k + 3, k + 4, k + 5), (k + 6, k + 6, k + 7),
                            (k + 8, k + 9, k + 8), (0, k + 10, 0)], np.float32)
    nf = len(faces)
    fid = np.repeat(np.arange(nf, dtype=np.float32), 3)[:, None]
    fs = np.arange(3 * nf, dtype=np.float32).reshape(nf, 3)
    vf = oracle.vertex_faces_tex(faces, len(pos))
    vf = np.concatenate([vf, vf[:1], np.full_like(vf[:1], nf - 1)]).astype(np.float32)
    assert vf.shape[0] > 64
    rs = oracle.rasterize_soft(oracle.soft_clip(clip, faces, w, h, 3.0), fid, fs, clip, faces, w, h,
                               3.0)
    gy = rng.standard_normal((h, w, 4)).astype(np.float32)
    got = host(ops.gather_dist_grad(ctx, dev(gy), dev(rs), dev(clip), dev(faces), dev(vf), 3.0))
    ref = oracle.gather_dist_grad(gy, rs, clip, faces, vf, wide=True)
    assert np.abs(ref).max() > 0
    _exact(got, ref, "wide")
    ctx.synchronize()


def _lanes_mesh(oracle, seed, level=5):
    """A dense icosphere on a small part of the screen, a fan and single faces whose boxes are a
    good part of it, faces that repeat a vertex: clip positions and faces."""
    rng = np.random.default_rng(seed)
    pos, sphere = oracle.icosphere(level)
    n_fan = 40
    ang = np.linspace(0.0, 2.0 * np.pi, n_fan, endpoint=False)
    k = len(pos)
    pos = np.concatenate([pos * [0.5, 0.5, 0.2] + [-0.2, 0.1, 0.5], [[0.0, 0.0, 0.2]],
                          np.stack([0.9 * np.cos(ang), 0.9 * np.sin(ang), 0 * ang + 0.1], 1),
                          rng.uniform(-1, 1, (9, 3)) * [1.2, 1.2, 0.4] + [0, 0, 0.5]])
    clip = np.concatenate([pos, np.ones((len(pos), 1))], 1).astype(np.float32)
    clip *= rng.uniform(0.5, 2.0, (len(pos), 1)).astype(np.float32)
    a = k + 1 + n_fan
    more = [(k, k + 1 + i, k + 1 + (i + 1) % n_fan) for i in range(0, n_fan, 3)] + [
        (a, a + 1, a + 2), (a + 3, a + 3, a + 4), (a + 5, a + 6, a + 5), (k, a + 7, a + 8)]
    return clip, np.concatenate([sphere, np.array(more)]).astype(np.float32)


@pytest.mark.parametrize("h,w,radius", [(61, 97, 3.0), (50, 33, 8.0), (90, 90, 0.5)])
def test_gather_dist_grad_many_faces(ctx, oracle, h, w, radius):
    """More faces than pixels: a lane per face, more hits than a lane keeps, boxes too large for a
    lane, a last wave that is not full: bit for bit against the oracle."""
    from opendressi_amd import ops
    print(f"[dist grad] many faces {h}x{w} r {radius}", flush=True)
    clip, faces = _lanes_mesh(oracle, h)
    nf = len(faces)
    assert nf > max(16384, h * w) and nf % 64
    vf = oracle.vertex_faces_tex(faces, len(clip))
    vf = np.concatenate([vf, np.full_like(vf[:1], nf - 1)]).astype(np.float32)
    fid = np.repeat(np.arange(nf, dtype=np.float32), 3)[:, None]
    fs = np.arange(3 * nf, dtype=np.float32).reshape(nf, 3)
    rs = oracle.rasterize_soft(oracle.soft_clip(clip, faces, w, h, radius), fid, fs, clip, faces, w,
                               h, radius)
    # faces of hundreds of pixels and of a few
    ids, px = np.unique(rs[..., 1][rs[..., 3] > 0.5], return_counts=True)
    assert px.max() > 100 and (px <= 2).any() and len(ids) > 100
    gy = np.random.default_rng(w).standard_normal((h, w, 4)).astype(np.float32)
    got = host(ops.gather_dist_grad(ctx, dev(gy), dev(rs), dev(clip), dev(faces), dev(vf), radius))
    ref = oracle.gather_dist_grad(gy, rs, clip, faces, vf, wide=True)
    assert np.abs(ref).max() > 0
    _exact(got, ref, "wide")
    ctx.synchronize()


@pytest.mark.parametrize("peels,items", [(1, 7), (3, 3), (17, 1)])
def test_surface_soft_gradient_many_faces(ctx, oracle, peels, items):
    """The torch surface's gradient by lanes over items and peels (more than the launch's 16),
    each layer with its own winners, against the wide form's rows, their column sums and the
    contributions' sum."""
    import torch

    from opendressi_amd import ops
    from opendressi_amd.torch.convert import sum_contribs
    h, w = 61, 97
    print(f"[dist grad] many faces, {items} items, {peels} peels", flush=True)
    clip, faces = _lanes_mesh(oracle, 1)
    faces = faces[np.array([len(set(f)) == 3 for f in faces])]
    nf = len(faces)
    assert nf * peels * items > 131072
    clips = dev(np.stack([clip * np.float32(1.0 + 0.05 * i) for i in range(items)]))
    vf = dev(oracle.vertex_faces_tex(faces, len(clip)))
    gen = torch.Generator(device="cuda").manual_seed(peels)
    shape = (items, peels, h, w)
    rs = torch.zeros((*shape, 4), device="cuda")
    rs[..., 1] = torch.randint(0, nf, shape, device="cuda", generator=gen).float()
    rs[..., 3] = (torch.rand(shape, device="cuda", generator=gen) < 0.9).float()
    # half of the pixels: the large faces
    big = torch.randint(nf - 10, nf, shape, device="cuda", generator=gen).float()
    rs[..., 1] = torch.where(torch.rand(shape, device="cuda", generator=gen) < 0.5, big, rs[..., 1])
    gy = torch.randn((*shape, 4), device="cuda", generator=gen)
    got = ops.surface_soft_bwd(ctx, gy, rs, clips, dev(faces), vf, 3.0)
    for i in range(items):
        parts = [ops.col_sum(ctx, ops.gather_dist_grad(ctx, gy[i, k], rs[i, k], clips[i],
                                                       dev(faces), vf, 3.0, True))
                 for k in reversed(range(peels))]
        ref = sum_contribs(parts)
        assert float(ref.abs().max()) > 0
        _exact(host(got[i]), host(ref), f"item {i}")
    ctx.synchronize()

"""Host-side logic of opendressi_amd.torch (no GPU): clip-space conventions,
the gradient-sum order, provenance lifetime, argument checks."""
import gc
import threading
import weakref

import numpy as np
import pytest
import torch

from opendressi_amd.torch import convert, provenance


def test_clip_grad_is_the_transpose_of_the_remap():
    """<remap(x), g> == <x, remap^T(g)> for random x, g (the remap is
    linear), and z_vk = 0.5 (z + w) on a known vertex."""
    rng = np.random.default_rng(0)
    x = torch.from_numpy(rng.standard_normal((5, 7, 4))).double()
    g = torch.from_numpy(rng.standard_normal((5, 7, 4))).double()
    lhs = (convert.clip_gl_to_vk(x) * g).sum()
    rhs = (x * convert.clip_grad_vk_to_gl(g)).sum()
    assert abs(lhs.item() - rhs.item()) < 1e-12
    v = convert.clip_gl_to_vk(torch.tensor([[0.3, -0.2, -0.5, 2.0]]))
    assert torch.equal(v, torch.tensor([[0.3, -0.2, 0.75, 2.0]]))


def test_sum_contribs_groups_of_four_left_to_right():
    """Six contributions sum as (a+b+c+d) + (e+f): in float32, 1e8 + (3+3)
    rounds to 1e8 + 8, while a flat left fold would drop each 3 on its own."""
    vals = [torch.tensor([x], dtype=torch.float32) for x in (1e8, 0.0, 0.0, 0.0, 3.0, 3.0)]
    assert convert.sum_contribs(vals).item() == 100000008.0
    flat = vals[0]
    for v in vals[1:]:
        flat = flat + v
    assert flat.item() == 1e8
    one = torch.tensor([3.0])
    assert convert.sum_contribs([one]) is one
    nine = [torch.tensor([float(i)]) for i in range(9)]
    assert convert.sum_contribs(nine).item() == 36.0


def test_provenance_lives_with_the_tensor():
    t = torch.zeros(3)
    rec = provenance.RasterOrigin(clip_vk=None, tri=None, resolution=(1, 1), ctx=None)
    provenance.stamp(t, rec)
    assert provenance.origin(t, provenance.RasterOrigin, "rasterize") is rec
    for other in (t.clone(), t.detach(), t[:2], t + 0):
        with pytest.raises(RuntimeError):
            provenance.origin(other, provenance.RasterOrigin, "rasterize")
    with pytest.raises(RuntimeError):
        provenance.origin(t, provenance.InterpOrigin, "interpolate")
    ref = weakref.ref(rec)
    del t, rec
    gc.collect()
    assert ref() is None  # the stamp dies with its tensor


def test_argument_checks():
    assert convert.resolution_hw([4, 6]) == (4, 6)
    assert convert.resolution_hw((np.int64(2), 3)) == (2, 3)
    for bad in ([0, 6], [4], [4, 6, 1], None, ["a", 2]):
        with pytest.raises(ValueError):
            convert.resolution_hw(bad)
    assert convert.vertex_batch(torch.zeros(3, 4)).shape == (1, 3, 4)
    assert convert.vertex_batch(torch.zeros(2, 3, 4)).shape == (2, 3, 4)
    with pytest.raises(ValueError):
        convert.vertex_batch(torch.zeros(3))
    assert convert.image_batch(torch.zeros(2, 3, 1), "c").shape == (1, 2, 3, 1)
    with pytest.raises(ValueError):
        convert.channels(5, "attr")
    from opendressi_amd.torch.context import tri_int32
    with pytest.raises(TypeError):
        tri_int32(torch.zeros(2, 3))
    with pytest.raises(ValueError):
        tri_int32(torch.zeros(2, 4, dtype=torch.int32))
    assert tri_int32(torch.tensor([[0, 1, 2]])).dtype == torch.int32


def test_vertex_adjacency_of_the_mesh_cache():
    """The {max_deg, V} adjacency the surface caches per topology lists each
    vertex's incident faces in ascending order, -1 padded."""
    from opendressi_amd.runtime import vertex_faces_tex
    faces = np.array([[0, 1, 2], [1, 3, 2], [2, 3, 4]], np.float32)
    vft = vertex_faces_tex(faces, 5)
    assert vft.shape == (3, 5)
    assert vft[:, 2].tolist() == [0, 1, 2]
    assert vft[:, 0].tolist() == [0, -1, -1]
    assert vft[:, 3].tolist() == [1, 2, -1]


class _Reached(Exception):
    """Stands for a kernel launch."""


def _host_context(monkeypatch):
    """A context on the CPU whose launches raise _Reached."""
    from types import SimpleNamespace

    from opendressi_amd import ops as K
    for name in [n for n in dir(K) if n.startswith(("surface_", "antialias"))]:
        def launch(*args, **kw):
            raise _Reached
        monkeypatch.setattr(K, name, launch)
    md = SimpleNamespace(n_verts=3, n_faces=1, faces_f=None, faces_i=None, vft=None)
    return SimpleNamespace(device=torch.device("cpu"), _ctx=None, lock=threading.RLock(),
                           mesh=lambda tri: md, engine=lambda key, build: build())


@pytest.mark.parametrize("comps", [1, 2, 3, 5])
@pytest.mark.parametrize("batched", [False, True])
def test_positions_of_another_width_are_refused(monkeypatch, comps, batched):
    """The kernels read a vertex as four floats: positions of any other width are refused before
    one runs, by every op that takes them; four pass."""
    import opendressi_amd.torch as dr
    ctx = _host_context(monkeypatch)
    tri = torch.tensor([[0, 1, 2]])
    rast = torch.zeros(1, 4, 6, 4)
    provenance.stamp(rast, provenance.RasterOrigin(clip_vk=None, tri=tri, resolution=(4, 6),
                                                   ctx=ctx))
    color = torch.zeros(1, 4, 6, 3)
    calls = [lambda p: dr.rasterize(ctx, p, tri, [4, 6]),
             lambda p: dr.rasterize_soft(ctx, p, tri, [4, 6]),
             lambda p: dr.antialias(color, rast, p, tri)]
    shape = (1, 3) if batched else (3,)
    for call in calls:
        with pytest.raises(ValueError, match="4 components"):
            call(torch.zeros(*shape, comps))
        with pytest.raises(_Reached):
            call(torch.zeros(*shape, 4))


@pytest.mark.parametrize("comps", [3, 5])
def test_op_positions_of_another_width_are_refused(comps):
    """The same for the entry points below, before they touch the context."""
    from opendressi_amd import ops as K
    p, img, rast = torch.zeros(2, 3, comps), torch.zeros(2, 4, 6, 3), torch.zeros(2, 4, 6, 4)
    f, vf, uv = torch.zeros(1, 3), torch.zeros(1, 3), torch.zeros(2, 4, 6, 2)
    rs = torch.zeros(2, 1, 4, 6, 4)
    for call in (lambda: K.surface_rasterize(None, p, f.int(), 6, 4),
                 lambda: K.surface_rasterize_soft(None, p, f, 6, 4, 3.0, 1),
                 lambda: K.surface_soft_bwd(None, rs, rs, p, f, vf, 3.0),
                 lambda: K.surface_interpolate_bwd(None, img, rast, p, f, vf, True),
                 lambda: K.surface_texture_bwd(None, img, uv, torch.zeros(3, 2), p, f, 8, 8),
                 lambda: K.surface_antialias(None, img, rast, p, f),
                 lambda: K.surface_antialias_bwd_img(None, img, rast, p, f),
                 lambda: K.surface_antialias_bwd_pos(None, img, img, rast, p, f, vf, 1, 8, 1.0),
                 lambda: K.antialias_batch(None, img, rast[..., 3], p, f),
                 lambda: K.antialias_bwd_img_batch(None, img, rast[..., 3], p, f),
                 lambda: K.antialias_bwd_vtx_batch(None, img, img, rast[..., 3], p, f, vf, None, 8,
                                                   True)):
        with pytest.raises(ValueError, match="4 components"):
            call()


@pytest.mark.parametrize("faces", [torch.zeros(2, 3), torch.zeros(2, 3, dtype=torch.int64),
                                   torch.zeros(3, 2, dtype=torch.int32).t(),
                                   torch.zeros(2, 3, dtype=torch.int32)])
def test_rasterize_faces_are_checked(faces):
    """Float or 64-bit ids, strided ones and a host tensor are refused before the context is
    touched: the kernel would read other memory."""
    from opendressi_amd import ops as K
    with pytest.raises(ValueError, match="faces: expected a contiguous int32 device tensor"):
        K.surface_rasterize(None, torch.zeros(1, 3, 4), faces, 6, 4)


@pytest.mark.parametrize("items", [1, 2, 4])
def test_interpolate_items_are_checked(items):
    """Per-item attributes of another batch than the raster's are refused before the context is
    touched: item i's would be read past their end, or another item's."""
    from opendressi_amd import ops as K
    with pytest.raises(ValueError, match=f"{items} items for a batch of 3"):
        K.surface_interpolate(None, torch.zeros(items, 5, 2), torch.zeros(3, 4, 6, 4),
                              torch.zeros(1, 3))

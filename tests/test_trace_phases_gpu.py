"""Edges of the traversal kernel's box test, stack and leaf dealing.

Workload: a 1,000-triangle sphere over a quad, and an icosphere field of 8 spheres; ray counts around
whole wavefronts and around the counts where a wavefront takes more rays; accels whose child boxes hold their bounds the wrong way round or a NaN bound.
Bar: every hit and per-ray counter bit-identical with the oracle, or with the scene whose boxes are in
order: MINPS/MAXPS of the two slab values do not depend on which bound is which.
"""
import numpy as np
import pytest

import oracle
import vermeer_amd as va
from vermeer_amd import scenes

pytestmark = pytest.mark.gpu


def _meshes(name):
    if name == "sphere":
        return [scenes.uv_sphere(1.0, 25, 21), scenes.ground_quad()]
    return [scenes.icosphere_field(8, extent=2.0, rmin=0.3, rmax=0.6)[:2]]


def _bits(h):
    return h.view(np.uint32).reshape(len(h), -1)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000, 4097, 8193, 32769, 131071, 300001])
@pytest.mark.parametrize("name", ["sphere", "field"])
def test_ray_counts_around_wavefronts(name, n):
    g, o = va.Scene(0), oracle.OracleScene()
    for v, f in _meshes(name):
        g.add_geom(va.PolyMesh(v, f))
        o.add_mesh(v, f)
    g.pre_render()
    o.commit()
    rays = scenes.uniform_rays(n, lo=(-2, -1, -2), hi=(2, 2, 2), seed=n)
    for shadow in (False, True):
        hits, geoms, cnt = g.trace(rays, shadow=shadow, want_counters=True)
        ref, rc = o.trace(rays, shadow=shadow, counters=True)
        for k in ("prim", "t", "u", "v"):
            assert hits[k].tobytes() == ref[k].tobytes(), k
        assert np.array_equal(geoms, ref["geom"])
        assert np.array_equal(cnt, rc)
        plain, _, _ = g.trace(rays, shadow=shadow)
        assert np.array_equal(_bits(plain), _bits(hits))


def _prebuilt(mesh, edit):
    """A scene over mesh's own accel with its node boxes edited."""
    src = va.Scene(0)
    src.add_geom(va.PolyMesh(*mesh))
    src.pre_render()
    nodes, idxp, _ = src.mesh_accel(0)
    lo = mesh[0].min(0)
    hi = mesh[0].max(0)
    boxes = nodes["boxes"].copy().reshape(len(nodes), 2, 3, 4)   # bound, axis, child
    edit(boxes, nodes["children"])
    nodes["boxes"] = boxes.reshape(len(nodes), 24)
    g = va.Scene(0)
    g.add_prebuilt(mesh[0], idxp, nodes, np.concatenate([lo, hi]))
    g.pre_render()
    return g


@pytest.mark.parametrize("exact", [False, True])
def test_bounds_the_wrong_way_round(exact):
    """Random (child, axis) bounds swapped; `exact`: one ray in 16 has a zero direction component, so that
    its wavefront takes the box test in the reference's own form."""
    mesh = _meshes("field")[0]
    pick = np.random.default_rng(3)

    def swap(boxes, children):
        m = pick.random(boxes[:, 0].shape) < 0.5
        a, b = boxes[:, 0].copy(), boxes[:, 1].copy()
        boxes[:, 0], boxes[:, 1] = np.where(m, b, a), np.where(m, a, b)

    g = _prebuilt(mesh, lambda boxes, children: None)
    s = _prebuilt(mesh, swap)
    rays = scenes.uniform_rays(20011, lo=(-1, -1, -1), hi=(3, 3, 3), seed=4)
    if exact:
        rays["D"][::16, 1] = 0.0
    for shadow in (False, True):
        a = g.trace(rays, shadow=shadow, want_counters=True)
        b = s.trace(rays, shadow=shadow, want_counters=True)
        assert np.array_equal(_bits(a[0]), _bits(b[0]))
        assert np.array_equal(a[2], b[2])


def test_a_nan_bound_takes_the_exact_box_test():
    """An empty child's box set to NaN: never hit, so the hits are those of the unedited accel."""
    mesh = _meshes("field")[0]
    hit = []

    def nan(boxes, children):
        empty = np.argwhere(children == -1)
        assert len(empty)
        for node, c in empty:
            boxes[node, :, :, c] = np.nan
        hit.append(len(empty))

    g = _prebuilt(mesh, lambda boxes, children: None)
    s = _prebuilt(mesh, nan)
    rays = scenes.uniform_rays(5000, lo=(-1, -1, -1), hi=(3, 3, 3), seed=5)
    a, _, _ = g.trace(rays)
    b, _, _ = s.trace(rays)
    assert np.array_equal(_bits(a), _bits(b)) and (a["prim"] >= 0).any()


@pytest.mark.parametrize("n", [1, 65, 4097])
@pytest.mark.parametrize("count", [1, 7, 31])
def test_transform_scenes_at_odd_sizes(count, n):
    """Instances (still and moving), a proc and a moving
    mesh; the allocation-free entry point gives the same hits."""
    import torch
    from vermeer_amd import render
    desc = scenes.instance_scene(seed=count, count=count)
    c = desc["camera"]
    M, ttf = oracle.camera_lookat(c["from"], c["to"], c["up"], c["fov"], c["focal"])
    R = render.Renderer(desc, 16, 16, render.lookat_camera(c["from"], c["to"], c["up"], c["fov"], c["focal"], 16, 16))
    o = oracle.OracleRenderer(desc, 16, 16, M, ttf, c["focal"])
    g = np.random.default_rng(n)
    rays = np.zeros(n, va.RAY_DTYPE)
    rays["P"] = g.uniform((-0.9, 0.1, -0.9), (0.9, 1.9, 0.9), (n, 3))
    d = g.normal(size=(n, 3))
    rays["D"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays["D"][::9, 2] = 0.0
    rays["tmax"] = np.where(g.random(n) < 0.2, 0.7, np.inf)
    rays["time"] = g.uniform(0, 1, n)
    dr = torch.from_numpy(rays.view(np.uint8).copy()).cuda()
    dh = torch.empty(n, 4, dtype=torch.int32, device="cuda")
    dg = torch.empty(n, dtype=torch.int32, device="cuda")
    lib = va._lib.load()
    for shadow in (False, True):
        hits, geoms, _ = R.scene.trace(rays, shadow=shadow)
        ref, _ = o.scene.trace(rays, shadow=shadow)
        for k in ("prim", "t", "u", "v"):
            assert hits[k].tobytes() == ref[k].tobytes(), k
        assert np.array_equal(geoms, ref["geom"])
        va._lib.check(lib.vgpu_trace_noalloc(R.scene._h, va._lib.VGPU_TRACE_SHADOW if shadow else 0, dr.data_ptr(), n,
                                             dh.data_ptr(), dg.data_ptr(), None, None, None))
        torch.cuda.synchronize()
        assert np.array_equal(dh.cpu().numpy().view(np.uint32), _bits(hits))
        assert np.array_equal(dg.cpu().numpy(), geoms)
    R.close()


@pytest.mark.parametrize("sort", [0, 3])
@pytest.mark.parametrize("size", [(37, 29), (64, 33)])
def test_shadow_rays_listed_per_pass(size, sort):
    """Film, sample and shadow-ray count of the feature scene (mirrors, two lights) at pixel counts off whole
    workgroups do not depend on the scene's ray sort, and the device counts the rays listed."""
    from vermeer_amd import render
    w, h = size
    desc = scenes.feature_scene()
    c = desc["camera"]
    M, ttf = oracle.camera_lookat(c["from"], c["to"], c["up"], c["fov"], c["focal"])
    cam = np.zeros((), va._lib.CAMERA_DTYPE)
    cam["M"], cam["tan_theta_focal"], cam["aspect"], cam["focal"] = M, ttf, w / h, c["focal"]
    R = render.Renderer(desc, w, h, cam)
    R.scene.set_trace_config(64, 12, 20, sort=sort)
    plain = render.Renderer(desc, w, h, cam)
    scr = scenes.pixel_scrambles(w, h)
    total = 0
    for it in (1, 2):
        n, samp = R.render_pass(scr, it, want_sample=True)
        m, ref = plain.render_pass(scr, it, want_sample=True)
        assert n == m > 0
        total += n
        assert samp.tobytes() == ref.tobytes()
    assert R.film.tobytes() == plain.film.tobytes()
    closest, shadow = R.stats()
    assert shadow == total and closest >= 2 * w * h
    R.close()
    plain.close()

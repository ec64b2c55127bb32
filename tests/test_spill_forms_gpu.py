"""The traversal's stack spill in short launches (a wavefront takes fewer than 64 rays), in the kernel forms beside the
static one in the caller's order: motion, transforms, the shading passes' 32-byte records, device-side ray counts and
slot lists.

Workloads: dense moving spheres, two instances of a dense icosphere field (one of them moving), the occluded-light room
in path mode and the box of spheres with such a field in it, each with rays whose stacks, counted by the oracle, go
beyond the entries that the form holds in LDS.  Ray counts lie around the shifts, in ascending and descending order, so
that the spill area is grown and is reused by smaller launches.  Bar: bit-identical with the oracle.
"""
import numpy as np
import pytest

import oracle
import vermeer_amd as va
from vermeer_amd import pathtrace, render, scenes

pytestmark = pytest.mark.gpu

COUNTS = [1, 63, 65, 3001, 4096, 4097, 16385, 40000]


def _deep(o, rays, entries, want):
    """The oracle's hits, and that `want` of the first 3001 rays go deeper than `entries`."""
    hits, cnt = o.trace(rays, counters=True)
    deep = int((cnt[:3001, 3] > entries).sum())
    print(f"[case] {deep} of 3001 rays deeper than {entries} entries", flush=True)
    assert deep >= want
    return hits


def _check(g, rays, refs, order):
    for n in order:
        for shadow, ref in refs:
            hits, geoms, _ = g.trace(rays[:n], shadow=shadow)
            for k in ("prim", "t", "u", "v"):
                assert hits[k].tobytes() == ref[k][:n].tobytes(), (n, shadow, k)
            assert np.array_equal(geoms, ref["geom"][:n]), (n, shadow)


@pytest.mark.parametrize("shape", [(64, 8, 20), (128, 12, 20), (256, 16, 16)])
def test_motion(shape):
    v, f = scenes.moving_spheres(count=200, nseg=25, nring=12, extent=1.0, rmin=0.3, rmax=0.8, max_move=0.5)
    o = oracle.OracleScene()
    o.add_mesh(v, f, motion_reference_indexing=False)
    o.commit()
    r = scenes.rng(4)
    n = max(COUNTS)
    rays = scenes.make_rays(r.uniform(-2, 2, (n, 3)), scenes.uniform_sphere_dirs(r, n), time=r.random(n))
    _deep(o, rays, shape[1], 10)
    refs = [(s, o.trace(rays, shadow=s)[0]) for s in (False, True)]
    for order in (COUNTS, COUNTS[::-1]):
        g = va.Scene(0)
        g.add_geom(va.PolyMesh(v, f))
        g.pre_render()
        g.set_trace_config(*shape)
        _check(g, rays, refs, order)
        g.close()


def _scale(t, s):
    m = np.zeros(16, np.float32)
    m[[0, 5, 10]] = s
    m[12:15] = t
    m[15] = 1
    return m


def test_transforms():
    v, f = scenes.icosphere_field(64, extent=1.0, rmin=0.2, rmax=0.6)[:2]
    inst = [(_scale((0, 0, 0), 1.0)[None], (-2, -2, -2), (2, 2, 2)),
            (np.stack([_scale((1, 0, 0), 0.7), _scale((1.2, 0.2, 0), 0.8)]), (-1, -2, -2), (4, 2, 2))]
    o = oracle.OracleScene()
    o.add_mesh(v, f)
    o.set_hidden(0, True)
    for m, lo, hi in inst:
        o.add_instance(0, m, lo, hi)
    o.commit()
    n = max(COUNTS)
    rays = scenes.uniform_rays(n, lo=(-1, -1, -1), hi=(2, 1, 1), seed=3)
    rays["time"] = np.random.default_rng(1).random(n)
    _deep(o, rays, 12, 20)   # the kernel's LDS stack
    refs = [(s, o.trace(rays, shadow=s)[0]) for s in (False, True)]
    assert {0, 1} <= set(refs[0][1]["geom"].tolist())
    for order in (COUNTS, COUNTS[::-1]):
        g = va.Scene(0)
        g.add_geom(va.PolyMesh(v, f))
        g.set_hidden(0)
        for m, lo, hi in inst:
            g.add_instance(0, m, lo, hi)
        g.pre_render()
        _check(g, rays, refs, order)
        g.close()


def test_path_mode():
    """32-byte records (12 entries in LDS) and shadow rays (8), both over queues counted on the device."""
    d = scenes.guided_room_scene(res=10, nboxes=6000)
    o = oracle.OracleScene()
    for m in d["meshes"]:
        o.add_mesh(m["verts"], m["idx"])
    o.commit()
    _deep(o, scenes.uniform_rays(3001, lo=(-4, 0, -4), hi=(4, 1.5, 4), seed=6), 12, 20)
    for W, depth in ((9, 4), (48, 6)):
        print(f"[case] path {W}x{W}", flush=True)
        g = pathtrace.PathTracer(d, W, W, max_depth=depth, seed=5)
        g.scene.set_trace_config(64, 8, 20)
        p = oracle.OraclePathTracer(d, W, W, g.cam, max_depth=depth, seed=5)
        for k in range(2):
            g.render_pass(k)
            p.render_pass(k)
        assert np.all((g.accum == p.accum) | (np.isnan(g.accum) & np.isnan(p.accum)))
        assert g.accum.max() > 0
        g.close()


@pytest.mark.parametrize("size", [(23, 17), (90, 70)])
def test_listed_shadow_rays(size):
    """Closest hits in 32-byte records and shadow rays from the list of slots, 8 entries in LDS."""
    w, h = size
    desc = scenes.box_spheres_scene(nseg=16, nring=8)
    v, f = scenes.icosphere_field(64, extent=0.5, rmin=0.1, rmax=0.3)[:2]
    desc["meshes"].append({"verts": (v + np.float32([0, 1, 0])).astype(np.float32), "idx": f, "shaderidx": None,
                           "shaders": np.array([1], np.int32), "normals": None})
    o = oracle.OracleScene()
    for m in desc["meshes"]:
        o.add_mesh(m["verts"], m["idx"])
    o.commit()
    _deep(o, scenes.uniform_rays(3001, lo=(-0.6, 0.4, -0.6), hi=(0.6, 1.6, 0.6), seed=6), 12, 20)
    c = desc["camera"]
    M, ttf = oracle.camera_lookat(c["from"], c["to"], c["up"], c["fov"], c["focal"])
    cam = np.zeros((), va._lib.CAMERA_DTYPE)
    cam["M"], cam["tan_theta_focal"], cam["aspect"], cam["focal"] = M, ttf, w / h, c["focal"]
    oracle.set_normalize_ieee(True)
    try:
        R = render.Renderer(desc, w, h, cam)
        R.scene.set_trace_config(64, 8, 20)
        ref = oracle.OracleRenderer(desc, w, h, M, ttf, c["focal"])
        scr = scenes.pixel_scrambles(w, h)
        for it in (1, 2):
            n, samp = R.render_pass(scr, it, want_sample=True)
            m, want = ref.render_pass(scr, it, want_sample=True)
            want = np.ascontiguousarray(want, np.float32)
            assert n == m > 0
            assert np.all((samp.view(np.uint32) == want.view(np.uint32)) | (np.isnan(samp) & np.isnan(want)))
        R.close()
    finally:
        oracle.set_normalize_ieee(False)

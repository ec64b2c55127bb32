"""Motion nodes whose boxes are not finite with lo <= hi take the reference's own box test.

Workload: a prebuilt accel over moving spheres with its boxes edited below the root (the root's children give the mesh's
bounds): random bounds swapped in every key, which the slab test does not see; and a child whose z bounds are infinite.
Interpolated inside the shutter that child's z slab is infinite and changes no hit; at a key 0 * inf makes it NaN, and
MINPS/MAXPS of a NaN last slab never report a hit, so the child is as if it were empty.  Bar: hits (and counters where
the traversal is the same) bit-identical with the unedited accel, and with one that has that child removed.
"""
import numpy as np
import pytest

import oracle
import vermeer_amd as va
from vermeer_amd import scenes

pytestmark = pytest.mark.gpu

N = 20011


@pytest.fixture(scope="module")
def accel():
    v, f = scenes.moving_spheres(count=60, nseg=16, nring=8, extent=2.0, rmin=0.3, rmax=0.8, max_move=0.5)
    o = oracle.OracleScene()
    o.add_mesh(v, f, motion_reference_indexing=False)
    o.commit()
    topo, boxes, perm = o.mesh_motion_accel(0)
    return v, f, np.ascontiguousarray(topo, np.int32), np.ascontiguousarray(boxes, np.float32), perm


def _scene(accel, topo, boxes):
    v, f, _, _, perm = accel
    g = va.Scene(0)
    g.add_motion_prebuilt(v, f, perm, topo, boxes)
    g.pre_render()
    return g


def _rays(time):
    r = scenes.rng(9)
    rays = scenes.make_rays(r.uniform(-3, 3, (N, 3)), scenes.uniform_sphere_dirs(r, N))
    rays["time"] = time if time is not None else r.uniform(0.01, 0.99, N)
    return rays


def _hits(g, rays, shadow, shape):
    g.set_trace_config(*shape)
    h, geoms, cnt = g.trace(rays, shadow=shadow, want_counters=True)
    plain = g.trace(rays, shadow=shadow)[0]
    assert plain.tobytes() == h.tobytes()
    return h.tobytes(), geoms.tobytes(), cnt


@pytest.mark.parametrize("shape", [(64, 8, 20), (128, 16, 16)])
def test_swapped_bounds(accel, shape):
    topo, boxes = accel[2:4]
    b = boxes.reshape(len(boxes), len(topo), 2, 3, 4).copy()
    m = np.random.default_rng(3).random(b.shape[1:2] + (3, 4)) < 0.5
    m[0] = False
    b[:, :, 0], b[:, :, 1] = np.where(m, b[:, :, 1], b[:, :, 0]), np.where(m, b[:, :, 0], b[:, :, 1])
    s, g = _scene(accel, topo, b.reshape(boxes.shape)), _scene(accel, topo, boxes)
    for time in (None, 0.0, 1.0):
        for shadow in (False, True):
            x, y = (_hits(k, _rays(time), shadow, shape) for k in (s, g))
            assert x[:2] == y[:2] and np.array_equal(x[2], y[2])


@pytest.mark.parametrize("shape", [(64, 8, 20), (128, 16, 16)])
def test_infinite_bounds(accel, shape):
    topo, boxes = accel[2:4]
    node = int(topo[0, 3:7].max())                       # a child node of the root
    child = int(np.flatnonzero(topo[node, 3:7] != -1)[0])
    b = boxes.reshape(len(boxes), len(topo), 2, 3, 4).copy()
    b[:, node, 0, 2, child], b[:, node, 1, 2, child] = -np.inf, np.inf
    cut = topo.copy()
    cut[node, 3 + child] = -1
    s, g, without = _scene(accel, topo, b.reshape(boxes.shape)), _scene(accel, topo, boxes), _scene(accel, cut, boxes)
    for shadow in (False, True):
        inside, key = _rays(None), _rays(0.0)
        assert _hits(s, inside, shadow, shape)[0] == _hits(g, inside, shadow, shape)[0]
        at_key = _hits(s, key, shadow, shape)[0]
        assert at_key == _hits(without, key, shadow, shape)[0]
        assert at_key != _hits(g, key, shadow, shape)[0]   # the child holds some ray's hit

"""The GPU builder with more subtrees than the y axis of a grid holds (65,535).

Workload: 41 million random boxes, whose ranges above 2048 elements all split evenly down to about 2500 and then into
four subtrees each: 65,536 and more of them (counted from the tree).  Bar: nodes, permutation and bounds equal the host
builder's byte for byte.
"""
import ctypes as C

import numpy as np
import pytest

from vermeer_amd import _lib

pytestmark = pytest.mark.gpu

N = 41_000_000
SUBTREE_MAX = 2048   # kSubtreeMax of bvh_build.hip


def _subtrees(children):
    """Topmost nodes of at most SUBTREE_MAX elements."""
    levels, at = [], np.array([0])
    while len(at):
        levels.append(at)
        c = children[at].reshape(-1)
        at = c[c >= 0]
    size = np.zeros(len(children), np.int64)
    for at in levels[::-1]:
        c = children[at]
        leaf = np.where(c < -1, (c & 15) + 1, 0)
        size[at] = np.where(c >= 0, size[np.maximum(c, 0)], leaf).sum(axis=1)
    c = children[size > SUBTREE_MAX].reshape(-1)
    c = c[c >= 0]
    return int((size[c] <= SUBTREE_MAX).sum())


def test_more_subtrees_than_a_grid_axis():
    lib = _lib.load()
    g = np.random.default_rng(1)
    cent = g.random((N, 3), dtype=np.float32)
    half = g.random((N, 3), dtype=np.float32) * np.float32(1e-3)
    boxes = np.concatenate([cent - half, cent + half], axis=1)
    out = []
    for gpu in (True, False):
        b, c, i = boxes.copy(), cent.copy(), np.arange(N, dtype=np.int32)
        nodes, bounds, count = np.empty((N // 8, 32), np.int32), np.zeros(6, np.float32), C.c_int32(0)
        args = [_lib.ptr(b), _lib.ptr(c), _lib.ptr(i), N, 16, _lib.ptr(nodes), len(nodes), C.byref(count), _lib.ptr(bounds)]
        print(f"[case] {'GPU' if gpu else 'host'} build of {N}", flush=True)
        _lib.check(lib.vgpu_qbvh_build_gpu(*args, None) if gpu else lib.vgpu_qbvh_build(*args, 0))
        out.append((nodes[:count.value], i, bounds, b, c))
    a, ref = out
    n = _subtrees(a[0][:, 27:31])
    print(f"[case] {len(a[0])} nodes, {n} subtrees", flush=True)
    assert n > 65_535
    for x, y in zip(a, ref):
        assert x.shape == y.shape and np.array_equal(x.view(np.int32), y.view(np.int32))

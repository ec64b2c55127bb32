"""The GPU builder at the edges of its chunks and its subtree queue: byte-identical with the host builder.

Workload: random boxes at counts around whole chunks (1024 elements, 4096 from 2^20 on); a chain of
centroids at powers of two, whose splits peel off a few elements each (a deep, narrow tree); zeros of both
signs; a box with infinite bounds.
Bar: nodes, permutation and bounds equal byte for byte.
"""
import numpy as np
import pytest

import vermeer_amd as va

pytestmark = pytest.mark.gpu


def _same(boxes, cent, leaf_max):
    idx = np.arange(len(cent), dtype=np.int32)
    a = [np.ascontiguousarray(x).copy() for x in (boxes, cent, idx)]
    b = [x.copy() for x in a]
    n1, bd1 = va.build_accel(*a, leaf_max)
    n2, bd2 = va.build_accel_gpu(*b, leaf_max)
    assert n1.tobytes() == n2.tobytes() and bd1.tobytes() == bd2.tobytes()
    for x, y in zip(a, b):
        assert x.tobytes() == y.tobytes()


def _random(n, seed):
    g = np.random.default_rng(seed)
    c = g.uniform(-10, 10, (n, 3)).astype(np.float32)
    e = g.uniform(0, 0.5, (n, 3)).astype(np.float32)
    return np.concatenate([c - e, c + e], axis=1), c


@pytest.mark.parametrize("n", [3071, 3072, 3073, 5121, (1 << 20) - 1, (1 << 20) + 1])
def test_counts_around_whole_chunks(n):
    _same(*_random(n, n), 16)


@pytest.mark.parametrize("leaf_max", [1, 3])
@pytest.mark.parametrize("copies", [1, 40])
def test_a_deep_chain(copies, leaf_max):
    """`copies` nearby elements at each power of two."""
    x = np.repeat(2.0 ** -np.arange(0, 100, dtype=np.float64), copies)
    x = x * (1.0 + np.tile(np.arange(copies), 100) * 1e-3)
    c = np.zeros((len(x), 3), np.float32)
    c[:, 0] = x
    _same(np.concatenate([c - 0.25 * np.abs(c), c + 0.25 * np.abs(c)], axis=1), c, leaf_max)


@pytest.mark.parametrize("n", [700, 6000])
def test_zeros_of_both_signs(n):
    boxes, c = _random(n, 3)
    g = np.random.default_rng(5)
    z = g.random((n, 3)) < 0.3
    boxes[:, :3][z] = np.where(g.random(z.sum()) < 0.5, 0.0, -0.0)
    boxes[:, 3:][z] = np.where(g.random(z.sum()) < 0.5, 0.0, -0.0)
    c[g.random((n, 3)) < 0.2] = -0.0
    c[g.random((n, 3)) < 0.1] = 0.0
    _same(boxes, c, 4)


@pytest.mark.parametrize("n", [40, 700, 6000])
def test_an_infinite_box_is_refused_by_both_builders(n):
    """Every split of a range holding it costs inf, so none is below the first: the recursion never ends."""
    boxes, c = _random(n, 3)
    boxes[n // 2, 3:] = np.inf
    for build in (va.build_accel, va.build_accel_gpu):
        with pytest.raises(va.VgpuError):
            build(boxes.copy(), c.copy(), np.arange(n, dtype=np.int32), 4)

"""The traversal's stack spill in launches that give a wavefront fewer than 64 rays.

Workload: an icosphere field under the smallest LDS stack (8 entries), ray counts around the shifts (one ray a
wavefront, a few, all 64) and around whole wavefronts, in ascending and descending order, so that the spill area is
grown and is reused by smaller launches.  Many rays go deeper than the LDS stack (asserted on the oracle's stack
depths).  Bar: hits and counters bit-identical with the oracle, for each block size.
"""
import numpy as np
import pytest

import oracle
import vermeer_amd as va
from vermeer_amd import scenes

pytestmark = pytest.mark.gpu

COUNTS = [1, 63, 64, 65, 3001, 4096, 4097, 8193, 20000, 65536 + 1, 150001]


@pytest.mark.parametrize("block", [64, 128, 256])
def test_short_launches_spill_right(block):
    v, f = scenes.icosphere_field(64, extent=2.0, rmin=0.2, rmax=0.5)[:2]
    o = oracle.OracleScene()
    o.add_mesh(v, f)
    o.commit()
    rays = scenes.uniform_rays(max(COUNTS), lo=(-2, -2, -2), hi=(2, 2, 2), seed=3)
    ref, rc = o.trace(rays, counters=True)
    deep = rc[:, 3] > 8
    print(f"[case] block {block}: {deep.mean():.3f} of the rays deeper than 8 entries", flush=True)
    assert deep[:3001].sum() > 50
    for order in (COUNTS, COUNTS[::-1]):
        g = va.Scene(0)
        g.add_geom(va.PolyMesh(v, f))
        g.pre_render()
        g.set_trace_config(block=block, lds_stack=8, waves_per_cu=20)
        for n in order:
            hits, geoms, cnt = g.trace(rays[:n], want_counters=True)
            plain, _, _ = g.trace(rays[:n])
            for k in ("prim", "t", "u", "v"):
                assert hits[k].tobytes() == ref[k][:n].tobytes(), (n, k)
                assert plain[k].tobytes() == ref[k][:n].tobytes(), (n, k)
            assert np.array_equal(geoms, ref["geom"][:n]) and np.array_equal(cnt, rc[:n]), n

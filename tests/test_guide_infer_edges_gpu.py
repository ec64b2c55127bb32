"""Guide inference at the edges of its tiles and of the lobe decode.

- A query's result is its own: any count (one query, 16-query tiles, 32 per wave, 128 per workgroup, more than
  one turn of the grid) gives the bits that the full batch gives, and the full batch is within the network's bars
  of the bf16-emulating oracle.
- The decode against 64 bits from the kernel's own raw outputs, u = 2^-24: a direction component takes 3 products
  and 2 sums under a square root (3 u / 2), a reciprocal root (2 u) and a product (u); kappa the hardware exp2 (1
  ulp, 2 u) of an argument below 1/2 with 2 u of its own; a weight two such exponentials, the rounding of its
  logit's difference from the largest (|x| u, its own and the sum's), 8 sums and a quotient.
"""
import numpy as np
import pytest

import oracle
from vermeer_amd import guide

pytestmark = pytest.mark.gpu

BOUNDS = np.array([-4, 0, -4, 4, 4, 4], np.float32)
U = 2.0 ** -24
FULL = 4097


def _queries(n, seed):
    rng = np.random.default_rng(seed)
    nrm = rng.normal(size=(n, 3))
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    return rng.uniform(BOUNDS[:3], BOUNDS[3:], (n, 3)).astype(np.float32), nrm.astype(np.float32)


def _check_decode(raw, lob):
    r = raw.reshape(-1, 8, 5).astype(np.float64)
    len_ = np.linalg.norm(r[..., :3], axis=-1, keepdims=True)
    assert np.abs(lob[..., :3] - r[..., :3] / len_).max() <= 6 * U
    kappa = np.exp(np.clip(r[..., 3], -5.0, 7.0))
    assert np.abs(lob[..., 3] / kappa - 1).max() <= 6 * U
    x = r[..., 4] - r[..., 4].max(axis=1, keepdims=True)
    w = np.exp(x) / np.exp(x).sum(axis=1, keepdims=True)
    bound = (20 + np.abs(x) + np.abs(x).max(axis=1, keepdims=True)) * U * w + 1e-37
    assert (np.abs(lob[..., 4] - w) <= bound).all()


@pytest.fixture(scope="module")
def full():
    print("\n[case] guide create", flush=True)
    g = guide.Guide(BOUNDS, seed=5, max_batch=1024)
    p = g.params
    p[21760:24320] *= 8.0
    p[24320:24360] = np.random.default_rng(1).uniform(-1, 1, 40)
    g.params = p
    pos, nrm = _queries(FULL, 7)
    raw, lob = g.infer(pos, nrm, raw=True), g.infer(pos, nrm)
    want, _ = oracle.guide_forward(g.params, pos, nrm, BOUNDS, emulate=True)
    e = np.abs(raw - want) / np.abs(want).max(axis=0, keepdims=True)
    assert e.max() < 2e-2 and np.median(e) < 2e-3
    _check_decode(raw, lob)
    return g, pos, nrm, raw, lob


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 32, 33, 127, 128, 129, 98304 + 33])
def test_a_query_does_not_depend_on_the_count(full, n):
    g, pos, nrm, raw, lob = full
    print(f"[case] infer {n}", flush=True)
    k = np.arange(n) % FULL
    assert np.array_equal(g.infer(pos[k], nrm[k], raw=True).view(np.int32), raw[k].view(np.int32))
    assert np.array_equal(g.infer(pos[k], nrm[k]).view(np.int32), lob[k].view(np.int32))


def test_lobes_at_the_ends_of_the_range(full):
    """No output weights: every query has the output biases, exactly.  Lobe by lobe: directions from nought to
    1e18, concentrations beyond both clamps, logits down to where a weight underflows."""
    g = guide.Guide(BOUNDS, seed=5, max_batch=1024)
    p = g.params
    p[21760:24320] = 0.0
    b = np.array([[0, 0, 0, -9, 0], [1e-25, 0, 0, 12, -1], [3e-18, -4e-18, 0, -5, -79], [1e18, 2e18, -2e18, 7, -81],
                  [1e-14, 0, 1e-14, 6.999, -100], [0, 1e-15, 0, 0, -104], [1e14, 1e14, 1e14, 1e-3, -300],
                  [-1, 2, -2, -4.999, 3]], np.float32)
    p[24320:24360] = b.reshape(-1)
    g.params = p
    pos, nrm = _queries(33, 8)
    raw, lob = g.infer(pos, nrm, raw=True), g.infer(pos, nrm)
    assert np.array_equal(raw.reshape(-1, 8, 5), np.broadcast_to(b, (33, 8, 5)))
    # squares that vanish in 32 bits have no direction: the pole
    assert np.array_equal(lob[:, :2, :3], np.broadcast_to(np.float32([0, 0, 1]), (33, 2, 3)))
    given = b.copy()
    given[:2, :3] = [0, 0, 1]
    _check_decode(np.broadcast_to(given.reshape(1, 40), (33, 40)), lob)


def test_a_nan_query_stays_in_its_row(full):
    g, pos, nrm, raw, lob = full
    bad = pos[:48].copy()
    bad[20, 1] = np.nan
    keep = np.arange(48) != 20
    got = g.infer(bad, nrm[:48])
    assert np.array_equal(got[keep].view(np.int32), lob[:48][keep].view(np.int32))

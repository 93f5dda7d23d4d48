"""recent() over a frozen CSR with a ring beside it, against the oracle, where the
gather's rank takes each of its branches: rings in write order with equal times
(inside the order and across the wrap), rings out of order, CSR windows before the
ring, reaching into it and longer than K, more valid slots than K, and queries
packed several per wavefront."""
import numpy as np
import pytest
import torch

from oracle import spec as O
from tgengine_amd import TemporalGraph
from test_gpu_recent import _tied_graph, cu

pytestmark = pytest.mark.gpu


# (K, B, row width, queries): above 8,192 queries rows of 16 to 64 bytes are packed
# two (B = 32, 20) or four (B = 16) queries per wavefront
@pytest.mark.parametrize("K,B,d,Q", [
    (20, 32, 8, 9_001), (20, 20, 16, 8_193), (12, 16, 8, 9_001), (5, 16, 4, 700), (64, 64, 172, 300),
    (33, 48, 3, 700), (65, 64, 8, 300), (1, 8, 8, 64)])
def test_csr_and_ring_branches(K, B, d, Q):
    rng, g, csr, ring, tmax = _tied_graph(60 + K, 40, B, d, 3, 400, 4, 120)
    nodes = rng.integers(-1, 40, Q)
    qt = np.floor(rng.uniform(5000.0, tmax + 5.0, Q))
    qt[::2] = tmax + 1.0  # after every entry: the usual streaming query
    r = g.recent(cu(nodes), cu(qt), K)
    o = O.recent(nodes, qt, K, csr, ring, d)
    assert np.array_equal(r.neighbor_ids.cpu().numpy(), o.ids)
    assert np.array_equal(r.timestamps.cpu().numpy().view(np.int64), o.times.view(np.int64))
    assert np.array_equal(r.mask.cpu().numpy(), o.mask)
    assert np.array_equal(r.edge_feats.cpu().numpy(), o.feats)


@pytest.mark.parametrize("wrap", range(6))
def test_ring_ties_across_the_wrap(wrap):
    """A node's ring whose equal times sit at every offset from the wrap of the write
    order: slot order decides between them, not write order."""
    B = 5
    g = TemporalGraph(30, edge_feat_dim=4, device="cuda", buffer_size=B)
    g.freeze_csr()
    ring = O.Ring.empty(30, B, 4)
    rng = np.random.default_rng(wrap)
    n = B + wrap
    times = np.array([100.0 + (i // 3) for i in range(n)])
    for i in range(n):  # one event a call: the write order is the event order
        s, d, t = np.array([0]), np.array([i + 1]), times[i:i + 1]
        f = rng.standard_normal((1, 4)).astype(np.float32)
        g.advance(cu(s), cu(d), cu(t), cu(f))
        O.ring_advance(ring, s, d, t, f)
    nodes = np.zeros(4, np.int64)
    qt = np.array([100.5, 101.5, 102.5, 1e9])
    for K in (2, B, 9):
        r = g.recent(cu(nodes), cu(qt), K)
        o = O.recent(nodes, qt, K, None, ring, 4)
        assert np.array_equal(r.neighbor_ids.cpu().numpy(), o.ids)
        assert torch.equal(r.timestamps.cpu(), torch.from_numpy(o.times))
        assert np.array_equal(r.edge_feats.cpu().numpy(), o.feats)


def _directed_graph(K, N, B, d, times, ring_times):
    """A frozen CSR of 1,500 events with ``times(rng, n)`` and a ring of 400 later ones
    whose stored times are then set to ``ring_times(rng, shape)`` (None: as appended),
    both with edge ids."""
    rng = np.random.default_rng(K)
    g = TemporalGraph(N, edge_feat_dim=d, device="cuda", buffer_size=B, track_edge_ids=True)
    ring = O.Ring.empty(N, B, d, np.float32, with_eids=True)
    events, t0 = [], 0
    for b, frozen in ((900, True), (600, True), (250, False), (150, False)):
        src, dst = np.minimum(rng.zipf(1.4, b) - 1, N - 1).astype(np.int64), rng.integers(0, N, b)
        tm = times(rng, b) if frozen else 1000.0 + np.floor(np.arange(b) / 3)
        f = rng.standard_normal((b, d)).astype(np.float32)
        g.advance(cu(src), cu(dst), cu(tm), cu(f))
        if frozen:
            events.append((src, dst, tm, f, t0))
        else:
            O.ring_advance_brute(ring, src, dst, tm, f, t0)
        t0 += b
        if b == 600:
            g.freeze_csr()
    ring.times[:] = ring_times(rng, ring.times.shape)
    g._ov_times.copy_(cu(ring.times))
    return rng, g, O.csr_freeze(N, d, events), ring


def _special(rng, shape):
    x = rng.choice(np.array([-0.0, 0.0, -np.inf, np.inf, np.nan, -2.5, 1.0, 3.0, 7.5]), shape)
    return np.where(rng.random(shape) < 0.5, np.floor(rng.uniform(-10, 10, shape)), x)


def _grid(rng, shape):
    return np.floor(rng.uniform(5.0, 40.0, shape))


# one, two and four queries per wavefront, and a query split over several
@pytest.mark.parametrize("kind", ["special", "grid"])
@pytest.mark.parametrize("K,B,d,Q", [(20, 32, 8, 8_300), (12, 16, 8, 8_300), (33, 48, 3, 700), (64, 64, 4, 90),
                                     (70, 20, 4, 90), (7, 5, 4, 2_500)])
def test_csr_and_ring_any_times_and_edge_ids(K, B, d, Q, kind):
    """NaN, infinite, signed-zero and tied times in the CSR, in the ring (in any order)
    and as query times; the edge ids of both sides, merged and appended."""
    times = _special if kind == "special" else _grid
    rng, g, csr, ring = _directed_graph(K, 40, B, d, times, times)
    nodes = rng.integers(-1, 40, Q)
    qt = times(rng, Q) + (0.0 if kind == "special" else 5.0)
    if kind == "special":
        qt[::7] = 100.0
    r = g.recent(cu(nodes), cu(qt), K)
    o = O.recent_brute(nodes, qt, K, csr, ring, d)
    assert o.mask.any() and not o.mask.all()
    assert np.array_equal(r.neighbor_ids.cpu().numpy(), o.ids)
    assert np.array_equal(r.timestamps.cpu().numpy().view(np.int64), o.times.view(np.int64))
    assert np.array_equal(r.mask.cpu().numpy(), o.mask)
    assert np.array_equal(r.edge_feats.cpu().numpy(), o.feats)
    assert np.array_equal(r.edge_ids.cpu().numpy(), o.eids)

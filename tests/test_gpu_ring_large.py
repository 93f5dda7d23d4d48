"""The ring update of batches above 16,384 events (four launches) against the oracle:
group sizes around the commit's limits (64 entries per wavefront, 512 counted in LDS,
longer lists over bitmap windows), a source-only hub (none of its entries in the upper
half of the batch), long lists spread thinly, and entry counts around the 1,024-entry
workgroups."""
import numpy as np
import pytest
import torch

from oracle import spec as O
from tgengine_amd import TemporalGraph

pytestmark = pytest.mark.gpu


def _sources(kind, b, N, rng):
    src = rng.integers(N // 2, N, b)  # mostly singletons and small groups
    at = rng.permutation(b)
    if kind == "sizes":
        pos = 0
        for u, c in enumerate((2, 63, 64, 65, 66, 255, 511, 512, 513, 514, 1500)):
            src[at[pos:pos + c]] = u
            pos += c
    elif kind == "hub":
        src[rng.random(b) < 0.6] = 0
    elif kind == "thin":  # 600 entries spread over the whole batch
        src[np.linspace(0, b - 1, 600).astype(np.int64)] = 0
        src[np.linspace(0, b - 1, 70).astype(np.int64)] = 1
    elif kind == "one":
        src[:] = 3
    return src


@pytest.mark.parametrize("B,d", [(1, 4), (20, 3), (64, 8)])
@pytest.mark.parametrize("kind,b", [("sizes", 16_385), ("hub", 20_000), ("thin", 33_000), ("one", 16_896)])
def test_large_batches(kind, b, B, d):
    N = 60_000
    rng = np.random.default_rng(b + B)
    g = TemporalGraph(N, edge_feat_dim=d, device="cuda", buffer_size=B, track_edge_ids=True)
    g.freeze_csr()
    ring = O.Ring.empty(N, B, d, np.float32, with_eids=True)
    t0 = 2.0 * b
    for step in range(2):  # the second batch meets rings that have wrapped
        src = _sources(kind, b, N, rng)
        dst = np.full(b, 5) if kind == "one" and step else rng.integers(N // 2, N, b)
        time = t0 + np.arange(b, dtype=np.float64)
        t0 = time[-1] + 1.0
        feat = rng.standard_normal((b, d)).astype(np.float32)
        g.advance(*(torch.from_numpy(x).cuda() for x in (src, dst, time, feat)))
        O.ring_advance(ring, src, dst, time, feat, eid_base=step * b)
    assert np.array_equal(g._ov_write_pos.cpu().numpy(), ring.wp)
    assert np.array_equal(g._ov_ids.cpu().numpy(), ring.ids)
    assert np.array_equal(g._ov_times.cpu().numpy(), ring.times)
    assert np.array_equal(g._ov_feats.cpu().numpy(), ring.feats)
    assert np.array_equal(g._ov_eids.cpu().numpy(), ring.eids)

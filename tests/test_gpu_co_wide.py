"""Co-occurrence of wide launches (K above 32) through DataPipeline.prepare against the
oracle: over a frozen CSR alone (K above 64 counts in a launch of its own) and with a
ring beside it (counted in the gather), both modes, with hubs, padding and pad nodes."""
import numpy as np
import pytest

from oracle import spec as O
from tgengine_amd import DataPipeline, GatherSpec, NeighborSpec, RawBatch
from test_gpu_recent import _tied_graph, cu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["freq", "dygformer"])
@pytest.mark.parametrize("with_ring", [False, True])
@pytest.mark.parametrize("K,n_neg", [(33, 1), (64, 3), (65, 1), (130, 7), (511, 1), (512, 2)])
def test_wide_co_occurrence(K, n_neg, with_ring, mode):
    N = 30
    rng, g, csr, ring, tmax = _tied_graph(70 + K, N, 32, 2, 4, 700, 3 if with_ring else 0, 90)
    b = 25
    src, dst = rng.integers(0, N, b), rng.integers(0, N, b)
    src[0] = dst[0]
    src[1] = -1  # a pad node: no CSR entries
    neg = rng.integers(0, N, (b, n_neg))
    t = np.floor(rng.uniform(5000.0, tmax + 3.0, b))
    t[2] = 4000.0  # before every entry: padding only
    spec = GatherSpec(neighbors=NeighborSpec(k=K), time_encoding=8, co_occurrence=True, co_occurrence_mode=mode)
    pb = DataPipeline(spec, g).prepare(RawBatch(src=cu(src), dst=cu(dst), time=cu(t),
                                                neg=cu(neg if n_neg > 1 else neg[:, 0])))
    r = ring if with_ring else None
    a = O.recent(src, t, K, csr, r, 2)
    c = O.recent(dst, t, K, csr, r, 2)
    n = O.recent(neg.reshape(-1), np.repeat(t, n_neg), K, csr, r, 2)
    for got, want in ((pb.src_neighbors, a), (pb.dst_neighbors, c), (pb.neg_neighbors, n)):
        assert np.array_equal(got.neighbor_ids.cpu().numpy(), want.ids)
        assert np.array_equal(got.edge_feats.cpu().numpy(), want.feats)
        assert np.array_equal(got.mask.cpu().numpy(), want.mask)
    if mode == "freq":
        ea, ec = O.co_occurrence_freq(a.ids, c.ids)
    else:
        ea, ec = O.co_dygformer(np.concatenate([src[:, None], a.ids], 1).astype(np.int32),
                                np.concatenate([dst[:, None], c.ids], 1).astype(np.int32))
    fa, fc = pb.co_occurrence_freq
    assert np.array_equal(fa.cpu().numpy(), ea) and np.array_equal(fc.cpu().numpy(), ec)
    assert np.array_equal(pb.co_occurrence.cpu().numpy(), O.co_pair_count(a.ids, a.mask, c.ids, c.mask))

"""Co-occurrence of wide launches (K above 32) through DataPipeline.prepare against the
oracle: over a frozen CSR alone (K above 128, and above 64 for few queries, counts in a
launch of its own) and with a ring beside it (counted in the gather), both modes, with
hubs, padding and pad nodes."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import spec as O
from tgengine_amd import DataPipeline, GatherSpec, NeighborSpec, RawBatch, TemporalGraph
from tgengine_amd.core import _lib
from test_gpu_recent import _tied_graph, cu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["freq", "dygformer"])
@pytest.mark.parametrize("with_ring", [False, True])
@pytest.mark.parametrize("K,n_neg", [(33, 1), (64, 3), (65, 1), (100, 9), (128, 11), (130, 7), (511, 1), (512, 2)])
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


@pytest.mark.parametrize("K", [20, 200])
def test_timed_launch_spans_the_count(K):
    """timing_start / timing_stop of a call that counts in a launch of its own: the same
    outputs, and a time that covers both launches but not what surrounds them."""
    N, b, n = 400, 2_000, 40_000
    rng = np.random.default_rng(K)
    g = TemporalGraph(N, edge_feat_dim=4, device="cuda")
    g.advance(cu(rng.integers(0, N, n)), cu(rng.integers(0, N, n)), cu(np.arange(n, dtype=np.float64)),
              torch.randn(n, 4, device="cuda"))
    g.freeze_csr()
    nodes = [cu(rng.integers(0, N, b)) for _ in range(2)]
    t = torch.full((b,), n + 1.0, dtype=torch.float64, device="cuda")
    csr, outs = g._csr(), []
    stream = torch.cuda.current_stream()
    for timed in (False, True):
        out = {"ids": torch.full((2 * b, K), -7, dtype=torch.int32, device="cuda"),
               "times": torch.empty(2 * b, K, dtype=torch.float64, device="cuda"),
               "mask": torch.empty(2 * b, K, dtype=torch.uint8, device="cuda")}
        co = {k: torch.full((b, K, 2), -7, dtype=torch.int32, device="cuda") for k in ("co_a", "co_c")}
        a = _lib.TgxRecentArgs(k=K, group=2, num_queries=2 * b, num_groups=b, num_query_groups=2,
                               plan_mode=_lib.TGX_PLAN_EVENTS, co_mode=_lib.TGX_CO_FREQ,
                               **{f"out_{k}": v.data_ptr() for k, v in out.items()},
                               **{k: v.data_ptr() for k, v in co.items()})
        for i in range(2):
            a.query_groups[i].nodes, a.query_groups[i].times = nodes[i].data_ptr(), t.data_ptr()
            a.query_groups[i].count, a.query_groups[i].times_per = b, 1
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(4)]
        for e in ev:
            e.record()  # creates it
        torch.cuda.synchronize()
        if timed:
            a.timing_start, a.timing_stop = ev[1].cuda_event, ev[2].cuda_event
        ev[0].record()
        _lib.check(_lib.lib().tgx_recent(None, ctypes.byref(csr), ctypes.byref(a), stream.cuda_stream), "tgx_recent")
        ev[3].record()
        torch.cuda.synchronize()
        if timed:
            assert 0.002 < ev[1].elapsed_time(ev[2]) <= ev[0].elapsed_time(ev[3]) + 0.002
        outs.append({**out, **co})
    for k in outs[0]:
        assert torch.equal(outs[0][k], outs[1][k]), k
    assert not any((v == -7).any() for k, v in outs[1].items() if k in ("co_a", "co_c"))

"""Feature rows of every alignment through the CSR build, both ring updates and the
gathers, bit for bit against the oracle: rows just below, at and above 16 bytes, rows
that are not a multiple of 16 (their last 16-byte chunk overlaps the one before) at
4- and 2-byte alignments, and rows of one to many chunks per lane."""
import numpy as np
import pytest
import torch

from oracle import spec as O
from tgengine_amd import DataPipeline, GatherSpec, NeighborSpec, RawBatch, TemporalGraph
from tgengine_amd.synthetic import f32_to_bf16_bits

pytestmark = pytest.mark.gpu


def _np(t):
    return t.view(torch.int16).cpu().numpy().view(np.uint16) if t.dtype == torch.bfloat16 else t.cpu().numpy()


@pytest.mark.parametrize("d,bf16", [(3, False), (4, False), (5, False), (7, False), (17, False), (43, False),
                                    (171, False), (7, True), (8, True), (9, True), (10, True), (33, True),
                                    (173, True), (511, True)])
def test_row_widths(d, bf16):
    N, B = 400, 12
    rng = np.random.default_rng(d)
    fdt = np.uint16 if bf16 else np.float32
    g = TemporalGraph(N, edge_feat_dim=d, device="cuda", buffer_size=B,
                      feat_dtype=torch.bfloat16 if bf16 else torch.float32)
    t0 = 50_000.0

    def batch(b):
        nonlocal t0
        src, dst = np.minimum((N * rng.random(b) ** 3).astype(np.int64), N - 1), rng.integers(0, N, b)
        time = t0 + np.arange(b, dtype=np.float64)
        t0 = time[-1] + 1.0
        f = rng.standard_normal((b, d)).astype(np.float32)
        f = f32_to_bf16_bits(f) if bf16 else f
        x = torch.from_numpy(f)
        g.advance(torch.from_numpy(src).cuda(), torch.from_numpy(dst).cuda(), torch.from_numpy(time).cuda(),
                  (x.view(torch.bfloat16) if bf16 else x).cuda())
        return src, dst, time, f

    def same(r, o):
        assert np.array_equal(r.neighbor_ids.cpu().numpy(), o.ids)
        assert np.array_equal(_np(r.edge_feats).view(np.uint8), o.feats.view(np.uint8))

    ev = batch(6000)
    g.freeze_csr()
    csr = O.csr_freeze(N, d, [(*ev, 0)], fdt)
    assert np.array_equal(_np(g._nbr_feats).view(np.uint8), csr.feats.view(np.uint8))
    Q = 2500  # one wavefront per query; fewer are split over several
    nodes, qt = rng.integers(-1, N, Q), rng.uniform(50_000.0, t0 + 10.0, Q)
    for K, n in ((20, Q), (20, 90), (64, 90), (70, 90)):
        same(g.recent(torch.from_numpy(nodes[:n]).cuda(), torch.from_numpy(qt[:n]).cuda(), K),
             O.recent(nodes[:n], qt[:n], K, csr, None, d, fdt))
    ring = O.Ring.empty(N, B, d, fdt)
    for b in (300, 17_000, 40):  # the two-launch and the four-launch update
        O.ring_advance(ring, *batch(b))
        assert np.array_equal(_np(g._ov_feats).view(np.uint8), ring.feats.view(np.uint8))
    nodes = rng.integers(0, N, Q)
    qt = np.full(Q, t0 + 1.0)
    for K, n in ((20, Q), (20, 90), (70, 90)):
        same(g.recent(torch.from_numpy(nodes[:n]).cuda(), torch.from_numpy(qt[:n]).cuda(), K),
             O.recent(nodes[:n], qt[:n], K, csr, ring, d, fdt))
    # event-major groups
    pipe = DataPipeline(GatherSpec(neighbors=NeighborSpec(k=10), co_occurrence=True, time_encoding=4), g)
    src, dst, neg = (rng.integers(0, N, 50) for _ in range(3))
    t = torch.full((50,), t0 + 2.0, dtype=torch.float64, device="cuda")
    pb = pipe.prepare(RawBatch(*(torch.from_numpy(x).cuda() for x in (src, dst)), time=t,
                               neg=torch.from_numpy(neg).cuda()))
    for nd, u in ((pb.src_neighbors, src), (pb.dst_neighbors, dst), (pb.neg_neighbors, neg)):
        same(nd, O.recent(u, np.full(50, t0 + 2.0), 10, csr, ring, d, fdt))

"""from_dataset against the same events replayed call by call: the CSR is the same
for every layout of its arrays, and later changes to them do not reach the graph."""
import pytest
import torch

from tgengine_amd import TemporalGraph
from tgengine_amd.core import temporal_graph

pytestmark = pytest.mark.gpu


def _arrays(E, kind):
    gen = torch.Generator().manual_seed(E)
    src = torch.randint(0, 50, (E,), generator=gen)
    dst = torch.randint(0, 50, (E,), generator=gen)
    time = torch.floor(torch.arange(E, dtype=torch.float64) / 3) + 7.0
    feat = torch.randn(E, 12, generator=gen)
    if kind == "host":
        return src, dst, time, feat
    if kind == "int32":
        return src.int().cuda(), dst.int().cuda(), time.float().cuda(), feat.cuda()
    src, dst, time, feat = src.cuda(), dst.cuda(), time.cuda(), feat.cuda()
    if kind == "strided":
        return torch.stack([src, src], 1)[:, 0], torch.stack([dst, dst], 1)[:, 1], time, feat.t().contiguous().t()
    if kind == "offset":  # rows that start 4 bytes after a 16-byte boundary
        flat = torch.empty(E * 12 + 1, device="cuda")
        flat[1:].copy_(feat.reshape(-1))
        return src, dst, time, flat[1:].view(E, 12)
    if kind == "longer":  # arrays beyond the events: the calls read their first E
        return src, torch.cat([dst, dst]), torch.cat([time, time]), torch.cat([feat, feat])
    if kind == "none":
        return src, dst, time, None
    return src, dst, time, feat


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind", ["plain", "host", "int32", "strided", "offset", "longer", "none"])
@pytest.mark.parametrize("E", [1, 25_000])
@pytest.mark.parametrize("copy", [0, 1 << 40])
def test_from_dataset_equals_replay(E, kind, dtype, copy, monkeypatch):
    src, dst, time, feat = _arrays(E, kind)
    monkeypatch.setattr(temporal_graph, "_ADOPT_COPY_BYTES", copy)
    g = TemporalGraph.from_dataset(src, dst, time, feat, 50, feat_dtype=dtype, track_edge_ids=True)
    r = TemporalGraph(50, edge_feat_dim=12 if feat is not None else 172, feat_dtype=dtype, track_edge_ids=True)
    for s in range(0, E, 10_000):
        e = min(s + 10_000, E)
        r.advance(src[s:e], dst[s:e], time[s:e], None if feat is None else feat[s:e])
    r.freeze_csr()
    for x in (src, dst, time, feat):  # the graph keeps its own values
        if x is not None:
            x.zero_()
    for name in ("_offsets", "_nbr_ids", "_nbr_times", "_nbr_feats", "_nbr_eids"):
        assert torch.equal(getattr(g, name), getattr(r, name)), name
    assert g.num_edges == r.num_edges == E and g._csr_build_mode == r._csr_build_mode


def test_from_dataset_refusals():
    src, dst, time, feat = _arrays(30, "plain")
    with pytest.raises(ValueError):
        TemporalGraph.from_dataset(src, dst[:20], time, feat, 50)
    with pytest.raises(ValueError):
        TemporalGraph.from_dataset(src, dst, time, feat[:20], 50)
    with pytest.raises(IndexError):
        TemporalGraph.from_dataset(src, dst, time, feat, 5)


@pytest.mark.parametrize("copy", [False, True])
@pytest.mark.parametrize("order", ["strict", "ties", "shuffled"])
def test_from_dataset_leaves_its_arrays_to_other_streams(order, copy, monkeypatch):
    """When from_dataset returns, nothing reads its arrays any more, copied or read in
    place: a second stream that never waits for the caller's refills them at once, and
    arrays allocated on a loader's stream go back to that stream's pool and are handed
    out again."""
    monkeypatch.setattr(temporal_graph, "_ADOPT_COPY_BYTES", 1 << 40 if copy else 0)
    E, N, d = 400_000, 5_000, 64
    gen = torch.Generator(device="cuda").manual_seed(3)
    src = torch.randint(0, N, (E,), generator=gen, device="cuda")
    dst = torch.randint(0, N, (E,), generator=gen, device="cuda")
    time = torch.arange(E, dtype=torch.float64, device="cuda") + 7.0
    if order == "ties":
        time = torch.floor(time / 3)
    elif order == "shuffled":
        time = time.view(-1, 100).flip(1).reshape(-1).contiguous()
    feat = torch.randn(E, d, generator=gen, device="cuda")
    want = TemporalGraph.from_dataset(src.cpu(), dst.cpu(), time.cpu(), feat.cpu(), N, track_edge_ids=True)
    other = torch.cuda.Stream()
    for release in (False, True):
        with torch.cuda.stream(other):
            arrays = [x.clone() for x in (src, dst, time, feat)]
        torch.cuda.current_stream().wait_stream(other)
        g = TemporalGraph.from_dataset(*arrays, N, track_edge_ids=True)
        if not copy:
            assert torch.cuda.current_stream().query()  # the build is over
        with torch.cuda.stream(other):
            if release:
                del arrays
                arrays = [torch.empty_like(x) for x in (src, dst, time, feat)]
            for x in arrays:
                x.zero_()
        torch.cuda.synchronize()
        for name in ("_offsets", "_nbr_ids", "_nbr_times", "_nbr_feats", "_nbr_eids"):
            assert torch.equal(getattr(g, name), getattr(want, name)), name

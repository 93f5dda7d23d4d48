"""The CSR build's sort, segments and row gather at the sizes where their shape
changes, bit for bit against the oracle: runs of equal times and calls that start,
end and lie inside and across the 2,048-event tiles of the segment search; sorts of
one and several tiles per workgroup (2M keys, 2,048- and 4,096-key tiles); one to
three digit passes; entry counts on both sides of the event-ordered gather (2^20)."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import spec as O
from tgengine_amd import TemporalGraph
from tgengine_amd.core import _lib
from tgengine_amd.synthetic import f32_to_bf16_bits

pytestmark = pytest.mark.gpu


def _check(N, d, cuts, src, dst, time, seed=0, bf16=False):
    E = len(src)
    feat = np.random.default_rng(seed).standard_normal((E, d)).astype(np.float32)
    g = TemporalGraph(N, edge_feat_dim=d, device="cuda", track_edge_ids=True,
                      feat_dtype=torch.bfloat16 if bf16 else torch.float32)
    events = []
    dev = [torch.from_numpy(x).cuda() for x in (src, dst, time, feat)]
    if bf16:
        feat = f32_to_bf16_bits(feat)
    for lo, hi in zip(cuts[:-1], cuts[1:]):
        g.advance(*(x[lo:hi] for x in dev))
        events.append((src[lo:hi], dst[lo:hi], time[lo:hi], feat[lo:hi], lo))
    g.freeze_csr()
    ref = O.csr_freeze(N, d, events, feat.dtype)
    assert np.array_equal(g._offsets.cpu().numpy(), ref.offsets)
    assert np.array_equal(g._nbr_ids.cpu().numpy(), ref.ids)
    assert np.array_equal(g._nbr_times.cpu().numpy().view(np.int64), ref.times.view(np.int64))
    feats = g._nbr_feats.view(torch.int16).cpu().numpy().view(np.uint16) if bf16 else g._nbr_feats.cpu().numpy()
    assert np.array_equal(feats, ref.feats)
    assert np.array_equal(g._nbr_eids.cpu().numpy(), ref.eids)
    assert g.status()["bad_event_nodes"] == 0
    return g


@pytest.mark.parametrize("E", [2047, 2048, 2049, 4097, 9000])
@pytest.mark.parametrize("run", [1, 3, 2048, 5000, 100_000])
def test_segments_across_tiles(E, run):
    rng = np.random.default_rng(E + run)
    src, dst = rng.integers(0, 50, E), rng.integers(0, 50, E)
    time = 10.0 + np.floor((np.arange(E) + 7) / run)
    cuts = sorted({0, 1, 31, 32, 2047, 2048, 2049, 4096, 6000, E} & set(range(E + 1)))
    g = _check(50, 3, cuts, src, dst, time)
    if run > 1:
        assert g._csr_build_mode == "runs"
    # the same calls with a step back inside them: the time sort over whole calls
    time[E // 2] -= 5.0
    assert _check(50, 3, cuts, src, dst, time)._csr_build_mode == "sort"


@pytest.mark.parametrize("E,N,d,order", [
    (524_287, 700, 8, "strict"), (524_288, 1 << 20, 4, "ties"), (530_000, 1023, 65, "ties"),
    (1_048_577, 1024, 4, "ties"), (1_100_000, 3, 1, "shuffled"), (2_200_000, 300_000, 2, "strict")])
def test_sort_and_gather_sizes(E, N, d, order):
    rng = np.random.default_rng(E)
    skew = rng.random(E)
    src = np.minimum((N * skew ** 6).astype(np.int64), N - 1)  # a few nodes hold most entries
    dst = rng.integers(0, N, E)
    time = 5.0 + np.arange(E, dtype=np.float64)
    if order == "ties":
        time = np.floor(time / 3.0)
    elif order == "shuffled":
        time = time.reshape(-1, 100)[:, ::-1].reshape(-1).copy()
    g = _check(N, d, [0, E // 3, E], src, dst, time)
    assert g._csr_build_mode == {"strict": "pairs", "ties": "runs", "shuffled": "sort"}[order]


# 256, 170, 93 and 64 entries per workgroup, the last one short, in rows of aligned and
# of overlapping 16-byte chunks
@pytest.mark.parametrize("d,bf16", [(5, False), (17, True), (22, False), (43, False), (64, False), (86, True)])
def test_event_ordered_gather_widths(d, bf16):
    E, N = 524_299, 3_000
    rng = np.random.default_rng(d)
    src = np.minimum((N * rng.random(E) ** 4).astype(np.int64), N - 1)
    _check(N, d, [0, 200_001, E], src, rng.integers(0, N, E), 5.0 + np.arange(E, dtype=np.float64), bf16=bf16)


def _by_call(N, src, dst, time, call, flags=0):
    """tgx_csr_build of the events of advance() calls of ``call`` events: (build, outputs)."""
    L, E = _lib.lib(), src.numel()
    empty = lambda n, dt: torch.empty(n, dtype=dt, device="cuda")  # noqa: E731
    starts = torch.arange(0, E, call, device="cuda")
    out = {"offsets": empty(N + 1, torch.int64), "ids": empty(2 * E, torch.int32),
           "times": empty(2 * E, torch.float64), "eids": empty(2 * E, torch.int64)}
    ws = empty(int(L.tgx_csr_build_workspace_size(2 * E)), torch.uint8)
    a = _lib.TgxCsrBuildArgs(num_nodes=N, num_entries=2 * E, from_=src.data_ptr(), to=dst.data_ptr(),
                             time=time.data_ptr(), call_starts=starts.data_ptr(), num_calls=starts.numel(),
                             feat_dim=0, feat_dtype=_lib.TGX_F32, workspace=ws.data_ptr(), workspace_bytes=ws.numel(),
                             flags=_lib.TGX_CSR_EVENTS_BY_CALL | flags,
                             **{f"out_{k}": v.data_ptr() for k, v in out.items()})

    def build(keep=(src, dst, time, starts, ws)):
        _lib.check(L.tgx_csr_build(ctypes.byref(a), torch.cuda.current_stream().cuda_stream), "tgx_csr_build")

    return build, out


def test_build_order_is_a_permutation_while_times_change():
    """The build order of runs of equal times takes every event twice even where another
    stream writes the times while the build reads them: no position of the permutation
    is left unwritten for the row gather to follow."""
    E, N = 300_000, 1_000
    src, dst = (torch.randint(0, N, (E,), device="cuda") for _ in range(2))
    pair = [torch.full((E,), 3.0, dtype=torch.float64, device="cuda"),
            torch.arange(E, dtype=torch.float64, device="cuda")]
    time = pair[0].clone()
    build, out = _by_call(N, src, dst, time, 10_000, _lib.TGX_CSR_NONDECREASING)
    want = torch.arange(E, device="cuda").repeat_interleave(2)
    other = torch.cuda.Stream()
    torch.cuda.synchronize()
    for _ in range(20):
        with torch.cuda.stream(other):
            for i in range(8):
                time.copy_(pair[i & 1])
        build()
        torch.cuda.synchronize()
        assert torch.equal(out["eids"].sort().values, want)


def test_segments_across_steps_of_tiles():
    """Runs of equal times within, across and longer than the 4,096 tiles (8.4M events)
    that one step of the search for a tile's neighbouring starts takes."""
    E = 8_500_000
    rng = np.random.default_rng(5)
    src, dst = rng.integers(0, 900, E), rng.integers(0, 900, E)
    edges = [1, 2_047, 2_048, 2_500, 40_960, 3_000_001, 3_000_002, 8_388_600, 8_388_650, 8_499_999]
    time = 4.0 + np.searchsorted(edges, np.arange(E), side="right").astype(np.float64)
    assert _check(900, 1, [0, 6_000_000, E], src, dst, time)._csr_build_mode == "runs"


def test_long_calls_cost_no_more_than_short_ones():
    """The build order of 64M events given by one call takes the time of the same events
    in calls of 10,000: the search for a tile's neighbouring starts is linear in the
    tiles (one that walks them from every tile costs 1.5 ms more here)."""
    E, N = 64_000_000, 1_000_000
    src, dst = (torch.randint(0, N, (E,), device="cuda") for _ in range(2))
    time = torch.arange(E, dtype=torch.float64, device="cuda")
    time[1::2] -= 3.0
    took = {}
    for call in (E, 10_000):
        build, out = _by_call(N, src, dst, time, call)
        build()
        best = []
        for _ in range(5):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            build()
            b.record()
            b.synchronize()
            best.append(a.elapsed_time(b))
        took[call] = min(best)
        del build, out
    assert took[E] - took[10_000] < 0.7, took


def test_more_wide_rows_than_one_launch_gathers():
    """16.8M entries with rows above 8 KB (one entry per workgroup) are more workgroups
    than one launch may hold: every entry is written."""
    E, N = 8_388_700, 50_000
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 170e9:
        pytest.skip("the rows take 138 GB")
    rng = np.random.default_rng(8)
    src, dst = (torch.from_numpy(rng.integers(0, N, E)).cuda() for _ in range(2))
    time = torch.arange(E, dtype=torch.float64, device="cuda")
    got = TemporalGraph(N, edge_feat_dim=2052, device="cuda", track_edge_ids=True)
    want = TemporalGraph(N, edge_feat_dim=1, device="cuda", track_edge_ids=True)
    for g in (want, got):
        g.advance(src, dst, time)
        g.freeze_csr()
    for name in ("_offsets", "_nbr_ids", "_nbr_times", "_nbr_eids"):
        assert torch.equal(getattr(got, name), getattr(want, name)), name
    for s in range(0, 2 * E, 1 << 20):
        assert not got._nbr_feats[s:s + (1 << 20)].any()
    del got, g
    torch.cuda.empty_cache()

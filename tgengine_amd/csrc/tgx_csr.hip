// Frozen-CSR build (reference TemporalGraph.freeze_csr, temporal_graph.py:133-181).
//
// The n directed entries of the pre-freeze advance() calls, in build order j
// (per call: [src->dst for every event, dst->src for every event]), are sorted
// stably by time and then stably by node, so a node's entries end up
// time-ascending with ties in build order (the reference's two stable
// argsorts, :156-158).  The same permutation comes out of a stable LSD radix
// sort: seven passes over an order-preserving 64-bit image of the time, then
// ceil(log2 N / 10) passes over the node id.
//
// The passes are tgx_radix.h's.  Then offsets[u] = lower_bound(sorted nodes, u), and
// one gather writes the ids, times, edge ids and feature rows (16-byte vectors
// where aligned).
//
// Event pairs (TGX_CSR_EVENT_PAIRS): the caller hands the events themselves in
// an order whose entries 2k, 2k+1 are already the stable time order of the
// build order (a time-ordered stream); the time passes are skipped and the
// kernels read an entry's node, neighbour, time and event from its event.
#include "tgx_radix.h"
#include "tgx_rows.h"

namespace tgx {
namespace {

// order-preserving image of a float64: -0.0 maps to +0.0 and every NaN to one
// NaN above +inf, so ties are exactly the ties of a float comparison
__device__ __forceinline__ uint64_t time_key(double t) {
  uint64_t u;
  if (t != t)
    u = 0x7ff8000000000000ull;
  else if (t == 0.0)
    u = 0;
  else
    u = static_cast<uint64_t>(__double_as_longlong(t));
  return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}

__global__ __launch_bounds__(kThreads) void csr_init(const double* __restrict__ time, int64_t n,
                                                     uint64_t* __restrict__ tkey,
                                                     uint32_t* __restrict__ idx) {
  const int64_t j = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (j >= n) return;
  tkey[j] = time_key(time[j]);
  idx[j] = static_cast<uint32_t>(j);
}

// offsets[u] = #sorted node keys < u, u in [0, N]
__global__ __launch_bounds__(kThreads) void csr_offsets(const uint32_t* __restrict__ nkey, int64_t n,
                                                        int64_t N, int64_t* __restrict__ offsets) {
  const int64_t u = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (u > N) return;
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (static_cast<int64_t>(nkey[mid]) < u)
      lo = mid + 1;
    else
      hi = mid;
  }
  offsets[u] = lo;
}

// Pre-freeze scan (tgx_csr_scan): node range, time order and largest time of the
// events in one pass.  Each workgroup reduces a grid-stride share into one
// ScanPart; csr_scan_final folds the parts.
constexpr int kScanParts = 1024;

struct ScanPart {
  int64_t lo, hi, bad, nd;
  double tmax;
};

// block-wide fold of (lo, hi, bad, tmax); the result is valid in thread 0
__device__ __forceinline__ ScanPart fold_block(ScanPart v, ScanPart* sm) {
  for (int o = kWave / 2; o > 0; o >>= 1) {
    v.lo = min(v.lo, static_cast<int64_t>(__shfl_xor(static_cast<long long>(v.lo), o)));
    v.hi = max(v.hi, static_cast<int64_t>(__shfl_xor(static_cast<long long>(v.hi), o)));
    v.bad += static_cast<int64_t>(__shfl_xor(static_cast<long long>(v.bad), o));
    v.nd += static_cast<int64_t>(__shfl_xor(static_cast<long long>(v.nd), o));
    v.tmax = fmax(v.tmax, __shfl_xor(v.tmax, o));
  }
  const int w = threadIdx.x / kWave;
  if ((threadIdx.x & (kWave - 1)) == 0) sm[w] = v;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int i = 1; i < kThreads / kWave; ++i) {
      v.lo = min(v.lo, sm[i].lo);
      v.hi = max(v.hi, sm[i].hi);
      v.bad += sm[i].bad;
      v.nd += sm[i].nd;
      v.tmax = fmax(v.tmax, sm[i].tmax);
    }
  return v;
}

// Event k >= 1 keeps the time order when t[k] - t[k-1] > 0, or == 0 with k the
// first event of an advance() call (the same float64 difference and
// comparisons as the check it replaces, so NaN and inf steps break the order).
// Every step not > 0 counts against the order, and each call start whose step
// is exactly 0 takes its count back (a second pass over the few call starts, in
// place of a search of them at every tie).  Apart, every step whose time goes
// down (or is NaN) counts against a non-decreasing stream.
__global__ __launch_bounds__(kThreads) void csr_scan_part(const int64_t* __restrict__ src,
                                                          const int64_t* __restrict__ dst,
                                                          const double* __restrict__ t, int64_t E,
                                                          const int64_t* __restrict__ starts, int64_t m,
                                                          ScanPart* __restrict__ parts) {
  __shared__ ScanPart sm[kThreads / kWave];
  ScanPart v{INT64_MAX, INT64_MIN, 0, 0, -__builtin_huge_val()};
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kThreads;
#pragma unroll 4
  for (int64_t k = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; k < E; k += stride) {
    const int64_t s = src[k], d = dst[k];
    const double x = t[k];
    v.lo = min(v.lo, min(s, d));
    v.hi = max(v.hi, max(s, d));
    if (x == x) v.tmax = fmax(v.tmax, x);
    if (k > 0) {
      const double p = t[k - 1];
      if (!(x - p > 0.0)) ++v.bad;
      if (!(x >= p)) ++v.nd;
    }
  }
  for (int64_t c = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; c < m; c += stride) {
    const int64_t k = starts[c];
    if (k >= 1 && k < E && (c == 0 || starts[c - 1] != k) && t[k] - t[k - 1] == 0.0) --v.bad;
  }
  v = fold_block(v, sm);
  if (threadIdx.x == 0) parts[blockIdx.x] = v;
}

// out = {min node, max node, 2 time-ordered / 1 non-decreasing / 0, bits of the largest non-NaN time}
__global__ __launch_bounds__(kThreads) void csr_scan_final(const ScanPart* __restrict__ parts, int np,
                                                           int64_t* __restrict__ out) {
  __shared__ ScanPart sm[kThreads / kWave];
  ScanPart v{INT64_MAX, INT64_MIN, 0, 0, -__builtin_huge_val()};
  for (int i = threadIdx.x; i < np; i += kThreads) {
    const ScanPart p = parts[i];
    v.lo = min(v.lo, p.lo);
    v.hi = max(v.hi, p.hi);
    v.bad += p.bad;
    v.nd += p.nd;
    v.tmax = fmax(v.tmax, p.tmax);
  }
  v = fold_block(v, sm);
  if (threadIdx.x == 0) {
    out[0] = v.lo;
    out[1] = v.hi;
    out[2] = v.bad == 0 ? 2 : (v.nd == 0 ? 1 : 0);
    out[3] = __double_as_longlong(v.tmax);
  }
}

// Build order from the events (TGX_CSR_EVENTS_BY_CALL).  The events fall into
// segments: the advance() calls, or with TGX_CSR_NONDECREASING the runs of equal
// times within a call.  The entries of segment [s, e) take build-order positions
// [2s, 2e) -- from->to of event k at s + k, then to->from at e + k -- which for
// runs of a non-decreasing stream is already its stable time order.
//
// Three launches over tiles of kSegTile events.  csr_seg_tiles marks the tile's
// segment starts in a bitmap and writes that and the tile's first and last start;
// csr_seg_edges finds the starts nearest to each tile from those; csr_seg_order each
// event's own segment from the bitmap, and writes the entries at their positions.  Times
// and call starts are read for the marks once: the segments partition the events,
// and the positions are a permutation, whatever the arrays hold, also where
// another stream writes them meanwhile.  8M events in runs of three take 13 + 4 + 82 us, the keys
// and records of the next steps included (448 MB; before, marks, a device-wide scan
// of them, segment starts, the order and the node keys took eight launches and 230 us).
constexpr int kSegItems = 8;
constexpr int kSegTile = kThreads * kSegItems;
constexpr int kSegWords = kSegTile / 32;
static_assert(kSegWords == kWave, "one bitmap word per lane");
constexpr uint32_t kNoStart = 0xffffffffu;

// bitmap[tile][.] = the tile's segment starts; first[tile], last[tile]: its first and
// last one (kNoStart: none)
__global__ __launch_bounds__(kThreads) void csr_seg_tiles(const double* __restrict__ time, int64_t E, int runs,
                                                          const int64_t* __restrict__ starts, int64_t m,
                                                          uint32_t* __restrict__ bitmap, uint32_t* __restrict__ first,
                                                          uint32_t* __restrict__ last) {
  __shared__ uint32_t bits[kSegWords];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kSegTile;
  if (threadIdx.x < kSegWords) bits[threadIdx.x] = 0u;
  // first call start at or after base, by 64-ary rounds of every wave
  const int lane = threadIdx.x & (kWave - 1);
  int64_t lo = 0, hi = m;
  while (hi > lo) {  // wave-uniform
    const int64_t step = (hi - lo + kWave - 1) / kWave;
    const int64_t pos = lo + static_cast<int64_t>(lane + 1) * step - 1;
    const int c = __popcll(__ballot(pos < hi && starts[pos] < base));
    const int64_t nl = lo + c * step;
    const int64_t nh = lo + (c + 1) * step - 1;
    lo = nl < hi ? nl : hi;
    hi = nh < hi ? nh : hi;
  }
  __syncthreads();
  const int64_t end = base + kSegTile < E ? base + kSegTile : E;
  for (int64_t c = lo + threadIdx.x; c < m; c += kThreads) {
    const int64_t k = starts[c];
    if (k >= end) break;
    if (k >= 1 && k >= base) atomicOr(&bits[(k - base) >> 5], 1u << ((k - base) & 31));
  }
#pragma unroll
  for (int r = 0; r < kSegItems; ++r) {
    const int i = r * kThreads + static_cast<int>(threadIdx.x);
    const int64_t k = base + i;
    const bool f = k < E && (k == 0 || (runs && !(time[k] == time[k - 1])));
    const uint64_t b = __ballot(f);
    if ((lane & 31) == 0) {
      const uint32_t w = lane == 0 ? static_cast<uint32_t>(b) : static_cast<uint32_t>(b >> 32);
      if (w != 0) atomicOr(&bits[i >> 5], w);
    }
  }
  __syncthreads();
  if (threadIdx.x < kWave) {
    const uint32_t w = bits[threadIdx.x];
    bitmap[static_cast<int64_t>(blockIdx.x) * kSegWords + threadIdx.x] = w;
    const uint64_t any = __ballot(w != 0);
    if (any == 0) {
      if (threadIdx.x == 0) first[blockIdx.x] = last[blockIdx.x] = kNoStart;
    } else {
      const uint32_t at = static_cast<uint32_t>(base) + threadIdx.x * 32;
      if (static_cast<int>(threadIdx.x) == __builtin_ctzll(any)) first[blockIdx.x] = at + __builtin_ctz(w);
      if (static_cast<int>(threadIdx.x) == 63 - __builtin_clzll(any)) last[blockIdx.x] = at + 31 - __builtin_clz(w);
    }
  }
}

// prev[t]: the last segment start before tile t (0: event 0 starts one), next[t]: the
// first one after it (E), from the tiles' first and last starts.  Workgroup 0 walks the
// tiles forwards, workgroup 1 backwards, kEdgeItems consecutive ones per thread and step:
// linear in the tiles, however long a segment is: 20 us for 64M events, 4 for 8M.  (When
// every tile of csr_seg_order walked its neighbours for itself, 64 at a time, 64M events
// in one call took it 1,924 us, 356 now; 8M in one run of equal times 106, 74 now.)
constexpr int kEdgeThreads = 1024;
constexpr int kEdgeItems = 4;
__global__ __launch_bounds__(kEdgeThreads) void csr_seg_edges(const uint32_t* __restrict__ first,
                                                              const uint32_t* __restrict__ last, int64_t nt, int64_t E,
                                                              uint32_t* __restrict__ prev, uint32_t* __restrict__ next) {
  __shared__ uint32_t wlast[kEdgeThreads / kWave];
  const bool back = blockIdx.x != 0;
  const uint32_t* v = back ? first : last;
  uint32_t* out = back ? next : prev;
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = threadIdx.x / kWave;
  uint32_t carry = back ? static_cast<uint32_t>(E) : 0u;  // the latest start of the steps before
  for (int64_t t0 = 0; t0 < nt; t0 += kEdgeThreads * kEdgeItems) {  // workgroup-uniform
    const int64_t t = t0 + static_cast<int64_t>(threadIdx.x) * kEdgeItems;
    uint32_t x[kEdgeItems];
    uint32_t mine = kNoStart;  // the thread's latest start
#pragma unroll
    for (int r = 0; r < kEdgeItems; ++r) {
      x[r] = t + r < nt ? v[back ? nt - 1 - (t + r) : t + r] : kNoStart;
      mine = x[r] != kNoStart ? x[r] : mine;
    }
    const uint64_t any = __ballot(mine != kNoStart);
    const uint64_t lower = any & ((uint64_t(1) << lane) - 1);
    const uint32_t before = __shfl(mine, lower != 0 ? 63 - __builtin_clzll(lower) : 0);
    const uint32_t top = __shfl(mine, any != 0 ? 63 - __builtin_clzll(any) : 0);
    if (lane == 0) wlast[wv] = any != 0 ? top : kNoStart;
    __syncthreads();
    uint32_t run = carry;
    for (int w = 0; w < kEdgeThreads / kWave; ++w) {
      const uint32_t y = wlast[w];
      if (w < wv && y != kNoStart) run = y;
      if (y != kNoStart) carry = y;
    }
    if (lower != 0) run = before;
#pragma unroll
    for (int r = 0; r < kEdgeItems; ++r) {
      if (t + r < nt) out[back ? nt - 1 - (t + r) : t + r] = run;
      if (x[r] != kNoStart) run = x[r];
    }
    __syncthreads();  // wlast has been read
  }
}

// event record of the row gather: time and both ends
struct alignas(16) EventRec {
  double time;
  int32_t from, to;
};

// key of node u, out-of-range ones last
__device__ __forceinline__ uint32_t node_key(int64_t u, int64_t N) {
  return u < 0 || u >= N ? 0xffffffffu : static_cast<uint32_t>(u);
}

// idx[position] = entry (2k + direction); with RUNS also its node key and the
// event's record, without its time key (the time passes follow)
template <bool RUNS>
__global__ __launch_bounds__(kThreads) void csr_seg_order(
    const double* __restrict__ time, const int64_t* __restrict__ from, const int64_t* __restrict__ to, int64_t E,
    int64_t N, const uint32_t* __restrict__ bitmap, const uint32_t* __restrict__ tile_prev,
    const uint32_t* __restrict__ tile_next, uint32_t* __restrict__ idx, uint64_t* __restrict__ tkey,
    uint32_t* __restrict__ nkey, EventRec* __restrict__ rec, int32_t* __restrict__ status) {
  __shared__ uint32_t bits[kSegWords], prev[kSegWords], next[kSegWords];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * kSegTile;
  if (threadIdx.x < kWave) {
    // the last start before word `lane` and the first one after it
    const int lane = threadIdx.x;
    const uint32_t w = bitmap[static_cast<int64_t>(blockIdx.x) * kSegWords + lane];
    bits[lane] = w;
    const uint32_t at = static_cast<uint32_t>(base) + lane * 32;
    const uint64_t any = __ballot(w != 0);
    const uint32_t wl = w != 0 ? at + 31 - __builtin_clz(w) : 0u;
    const uint32_t wf = w != 0 ? at + __builtin_ctz(w) : 0u;
    const uint64_t lower = any & ((uint64_t(1) << lane) - 1);
    const uint64_t upper = lane == 63 ? 0 : any >> (lane + 1);
    const uint32_t pl = __shfl(wl, lower != 0 ? 63 - __builtin_clzll(lower) : 0);
    const uint32_t nf = __shfl(wf, upper != 0 ? lane + 1 + __builtin_ctzll(upper) : 0);
    prev[lane] = lower != 0 ? pl : tile_prev[blockIdx.x];
    next[lane] = upper != 0 ? nf : tile_next[blockIdx.x];
  }
  __syncthreads();
  int bad = 0;
#pragma unroll
  for (int r = 0; r < kSegItems; ++r) {
    const int i = r * kThreads + static_cast<int>(threadIdx.x);
    const int64_t k = base + i;
    if (k < E) {
      const uint32_t w = bits[i >> 5];
      const uint32_t upto = (2u << (i & 31)) - 1u;  // bits of the word up to event k
      const uint32_t at = static_cast<uint32_t>(base) + (i & ~31);
      const uint32_t s = (w & upto) != 0 ? at + 31 - __builtin_clz(w & upto) : prev[i >> 5];
      const uint32_t e = (w & ~upto) != 0 ? at + __builtin_ctz(w & ~upto) : next[i >> 5];
      const int64_t pf = static_cast<int64_t>(s) + k;
      const int64_t pr = static_cast<int64_t>(e) + k;
      idx[pf] = static_cast<uint32_t>(2 * k);
      idx[pr] = static_cast<uint32_t>(2 * k + 1);
      if constexpr (RUNS) {
        const int64_t u = from[k], v = to[k];
        nkey[pf] = node_key(u, N);
        nkey[pr] = node_key(v, N);
        bad += (u < 0 || u >= N) + (v < 0 || v >= N);
        rec[k] = EventRec{time[k], static_cast<int32_t>(u), static_cast<int32_t>(v)};
      } else {
        const uint64_t key = time_key(time[k]);
        tkey[pf] = key;
        tkey[pr] = key;
      }
    }
  }
  if (RUNS && bad != 0 && status != nullptr) atomicAdd(&status[TGX_ST_BAD_EVENT_NODE], bad);
}

// Node keys of the event-pair build (entry 2k = from[k] -> to[k], 2k + 1 = to[k] ->
// from[k], already in stable time order) and the events' records.
__global__ __launch_bounds__(kThreads) void csr_pair_keys(const double* __restrict__ time,
                                                          const int64_t* __restrict__ from,
                                                          const int64_t* __restrict__ to, int64_t E, int64_t N,
                                                          uint32_t* __restrict__ nkey, EventRec* __restrict__ rec,
                                                          int32_t* __restrict__ status) {
  const int64_t k = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  int bad = 0;
  if (k < E) {
    const int64_t u = from[k], v = to[k];
    reinterpret_cast<uint2*>(nkey)[k] = make_uint2(node_key(u, N), node_key(v, N));
    bad = (u < 0 || u >= N) + (v < 0 || v >= N);
    rec[k] = EventRec{time[k], static_cast<int32_t>(u), static_cast<int32_t>(v)};
  }
  if (bad != 0 && status != nullptr) atomicAdd(&status[TGX_ST_BAD_EVENT_NODE], bad);
}

// records of events (or, where entries are given one by one, of entries)
__global__ __launch_bounds__(kThreads) void csr_records(const double* __restrict__ time,
                                                        const int64_t* __restrict__ from,
                                                        const int64_t* __restrict__ to, int64_t E,
                                                        EventRec* __restrict__ rec) {
  const int64_t k = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (k < E) rec[k] = EventRec{time[k], static_cast<int32_t>(from[k]), static_cast<int32_t>(to[k])};
}

// nkey[p] = node of entry idx[p] (pairs: entry 2k is from[k]'s, 2k + 1 to[k]'s)
__global__ __launch_bounds__(kThreads) void csr_node_keys(const int64_t* __restrict__ from,
                                                          const int64_t* __restrict__ to, int pairs,
                                                          const uint32_t* __restrict__ idx, int64_t n, int64_t N,
                                                          uint32_t* __restrict__ nkey, int32_t* __restrict__ status) {
  const int64_t p = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  bool bad = false;
  if (p < n) {
    const uint32_t j = idx[p];
    const int64_t u = pairs ? ((j & 1) ? to[j >> 1] : from[j >> 1]) : from[j];
    bad = u < 0 || u >= N;
    nkey[p] = node_key(u, N);
  }
  const uint64_t bm = __ballot(bad);
  if ((threadIdx.x & (kWave - 1)) == 0 && bm != 0 && status != nullptr)
    atomicAdd(&status[TGX_ST_BAD_EVENT_NODE], __popcll(bm));
}

// out[p] = entry perm[p]: id, time, edge id, feature row.  The entries of a node
// come from all over the stream, and every read of a 16-byte record (neighbour and
// time: before, two 8-byte reads from two arrays) or a short row fetches a 128-byte
// line: node by node, 16M entries with 32-byte rows fetched 2.9 GB for 0.8 GB used,
// in 548 us (674 with the two arrays).  So tiles of `per` consecutive entries run
// in the order of their first events: the busy nodes, which hold most of a skewed
// stream's entries, then walk the stream together and share its lines, and runs of
// kGatherSlice such tiles go to one XCD, for its L2: 345 us, and 23 us for the order
// (tiles of 512 or 128 entries: 352 and 359).
// A workgroup takes one tile, its permutation in LDS, and copies the rows as one
// run of chunks, kGatherDepth per thread loaded before the first is stored,
// whatever the row's width (314,948 entries with 688-byte rows: 118 -> 75 us
// against a row per wavefront).  Output leaves as nontemporal stores, which leaves
// the caches to the events (5 of 80 us on those).
constexpr int kGatherDepth = 4;
constexpr int kGatherChunks = kThreads * kGatherDepth;  // chunks a workgroup holds in flight
constexpr int kGatherMost = 256;                        // entries per workgroup at most
constexpr int kXcds = 8;
constexpr int kGatherSlice = 64;  // tiles of neighbouring events given to one XCD
// tiles per launch: a launch holds fewer than 2^32 threads, which 16.8M entries of rows
// above 8 KB (one per workgroup) would reach in one
constexpr int64_t kGatherTiles = int64_t(1) << 20;
static_assert(kGatherTiles % (kXcds * kGatherSlice) == 0, "whole slices per launch");

// key of tile i (`per` entries) of the gather: its first entry's event
__global__ __launch_bounds__(kThreads) void csr_tile_keys(const uint32_t* __restrict__ perm, int64_t ntiles, int per,
                                                          int pairs, uint32_t* __restrict__ key) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (i < ntiles) key[i] = perm[i * per] >> (pairs ? 1 : 0);
}

template <int VEC>
__global__ __launch_bounds__(kThreads) void csr_gather(
    const uint32_t* __restrict__ perm, int64_t n, const EventRec* __restrict__ rec, int pairs,
    const int64_t* __restrict__ event, int64_t num_events, const uint8_t* __restrict__ feats, int64_t row_bytes, int nch,
    uint32_t nch_magic, int per, const uint32_t* __restrict__ order, int64_t tile0, int64_t ntiles,
    int32_t* __restrict__ out_ids, double* __restrict__ out_times, int64_t* __restrict__ out_eids,
    uint8_t* __restrict__ out_feats, int32_t* __restrict__ status) {
  using V = typename RowChunk<VEC>::T;
  __shared__ int64_t row[kGatherMost];  // an entry's feature row, -1: zeros
  int64_t tile = tile0 + blockIdx.x;
  if (order != nullptr) {  // launch-uniform
    const int64_t g = tile / (kXcds * kGatherSlice);
    const int r = static_cast<int>(tile - g * (kXcds * kGatherSlice));
    const int64_t at = (g * kXcds + r % kXcds) * kGatherSlice + r / kXcds;
    if (at >= ntiles) return;  // workgroup-uniform
    tile = order[at];
  }
  const int64_t p0 = tile * per;
  const int cnt = static_cast<int>(n - p0 < per ? n - p0 : per);
  for (int i = threadIdx.x; i < cnt; i += kThreads) {
    const uint32_t j = perm[p0 + i];
    const int64_t k = pairs ? j >> 1 : j;
    const EventRec r = rec[k];
    const int64_t ev = event != nullptr ? event[k] : (pairs ? k : -1);
    const bool have = feats != nullptr && ev >= 0 && ev < num_events;
    row[i] = have ? ev : -1;
    __builtin_nontemporal_store(pairs && (j & 1) ? r.from : r.to, out_ids + p0 + i);
    __builtin_nontemporal_store(r.time, out_times + p0 + i);
    if (out_eids != nullptr) out_eids[p0 + i] = ev;
    if (out_feats != nullptr && feats != nullptr && !have && status != nullptr)
      atomicAdd(&status[TGX_ST_BAD_EVENT_NODE], 1);
  }
  if (out_feats == nullptr) return;  // launch-uniform
  __syncthreads();
  uint8_t* dst = out_feats + p0 * row_bytes;
  const int64_t total = static_cast<int64_t>(cnt) * nch;
  for (int64_t c0 = threadIdx.x; c0 < total; c0 += kGatherChunks) {
    V v[kGatherDepth];
    int64_t at[kGatherDepth];
#pragma unroll
    for (int u = 0; u < kGatherDepth; ++u) {
      const int64_t c = c0 + u * kThreads;
      v[u] = V{};
      at[u] = 0;
      if (c < total) {
        // one entry per workgroup, or a dividend below 2^32 / nch
        const int e = per == 1 ? 0 : nch == 1 ? static_cast<int>(c) : static_cast<int>(__umulhi(static_cast<uint32_t>(c), nch_magic));
        const int64_t off = chunk_at<VEC>(c - static_cast<int64_t>(e) * nch, row_bytes);
        const int64_t ev = row[e];
        at[u] = e * row_bytes + off;
        if (ev >= 0) v[u] = load_chunk<VEC>(feats + ev * row_bytes + off);
      }
    }
#pragma unroll
    for (int u = 0; u < kGatherDepth; ++u)
      if (c0 + u * kThreads < total) store_chunk<VEC, true>(dst + at[u], v[u]);
  }
}

struct Layout {
  RadixScratch r;
  size_t tkey = 0, idx = 0, nkey = 0, count = 0, sums = 0, total = 0;
};

Layout layout(int64_t n) {
  Layout w;
  w.r = radix_scratch(n);
  const size_t un = static_cast<size_t>(std::max<int64_t>(n, 1));
  w.tkey = 0;
  w.idx = w.tkey + 2 * align256(un * 8);
  w.nkey = w.idx + 2 * align256(un * 4);
  w.count = w.nkey + 2 * align256(un * 4);
  w.sums = w.count + w.r.count_bytes;
  w.total = w.sums + w.r.sums_bytes + 16;  // the sections start at a multiple of 16
  return w;
}

}  // namespace
}  // namespace tgx

using namespace tgx;

extern "C" size_t tgx_csr_build_workspace_size(int64_t n) {
  if (n < 0) return 0;
  return layout(n).total;
}

extern "C" int tgx_csr_build(const tgx_csr_build_args* a, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  if (a == nullptr) return fail(TGX_ERR_ARG, "tgx_csr_build: args is NULL");
  const int64_t n = a->num_entries, N = a->num_nodes;
  if (N <= 0 || N >= (int64_t(1) << 31))
    return fail(TGX_ERR_LIMIT, "tgx_csr_build: num_nodes %lld outside [1, 2^31)", (long long)N);
  if (n < 0 || n >= (int64_t(1) << 31))
    return fail(TGX_ERR_LIMIT, "tgx_csr_build: %lld entries outside [0, 2^31)", (long long)n);
  if (a->feat_dim < 0) return fail(TGX_ERR_ARG, "tgx_csr_build: negative feat_dim");
  const int esz = feat_elem_bytes(a->feat_dtype);
  if (esz == 0) return fail(TGX_ERR_DTYPE, "tgx_csr_build: unsupported feat dtype %d", a->feat_dtype);
  if (a->out_offsets == nullptr) return fail(TGX_ERR_ARG, "tgx_csr_build: out_offsets is NULL");
  const int64_t row_bytes = static_cast<int64_t>(a->feat_dim) * esz;
  if ((a->flags & ~(TGX_CSR_EVENT_PAIRS | TGX_CSR_EVENTS_BY_CALL | TGX_CSR_NONDECREASING)) != 0)
    return fail(TGX_ERR_ARG, "tgx_csr_build: unknown flags 0x%x", a->flags);
  const int by_call = (a->flags & TGX_CSR_EVENTS_BY_CALL) != 0;
  const int runs = (a->flags & TGX_CSR_NONDECREASING) != 0;
  if ((a->flags & TGX_CSR_EVENT_PAIRS) && by_call)
    return fail(TGX_ERR_ARG, "tgx_csr_build: TGX_CSR_EVENT_PAIRS and TGX_CSR_EVENTS_BY_CALL exclude each other");
  if (runs && !by_call)
    return fail(TGX_ERR_ARG, "tgx_csr_build: TGX_CSR_NONDECREASING needs TGX_CSR_EVENTS_BY_CALL");
  if (by_call && (a->num_calls < 0 || (a->num_calls > 0 && a->call_starts == nullptr)))
    return fail(TGX_ERR_ARG, "tgx_csr_build: events by call need call_starts [num_calls >= 0]");
  // entries addressed through their events: 2k = from->to, 2k + 1 = to->from of event k
  const int pairs = (a->flags & TGX_CSR_EVENT_PAIRS) != 0 || by_call;
  if (pairs && n % 2 != 0)
    return fail(TGX_ERR_ARG, "tgx_csr_build: events need an even entry count, got %lld", (long long)n);
  if (n > 0) {
    if (a->from == nullptr || a->to == nullptr || a->time == nullptr || a->out_ids == nullptr ||
        a->out_times == nullptr)
      return fail(TGX_ERR_ARG, "tgx_csr_build: from/to/time/out_ids/out_times must not be NULL");
    if (row_bytes > 0 && a->out_feats == nullptr)
      return fail(TGX_ERR_ARG, "tgx_csr_build: out_feats is NULL with feat_dim > 0");
    if ((a->feats != nullptr || a->out_eids != nullptr) && a->event == nullptr && !pairs)
      return fail(TGX_ERR_ARG, "tgx_csr_build: feats / out_eids need the event index array");
    if (a->feats != nullptr && a->num_events < 0)
      return fail(TGX_ERR_ARG, "tgx_csr_build: negative num_events");
  }
  const Layout w = layout(n);
  if (a->workspace == nullptr || a->workspace_bytes < w.total)
    return fail(TGX_ERR_ARG, "tgx_csr_build: workspace of %zu bytes needed, got %zu", w.total,
                a->workspace_bytes);
  uint8_t* ws = reinterpret_cast<uint8_t*>((reinterpret_cast<uintptr_t>(a->workspace) + 15) & ~uintptr_t(15));
  const unsigned g1 = static_cast<unsigned>(std::max<int64_t>(cdiv(n, kThreads), 1));
  int rc;
  if (n == 0) {
    hipLaunchKernelGGL(csr_offsets, dim3(static_cast<unsigned>(cdiv(N + 1, kThreads))), dim3(kThreads),
                       0, stream, static_cast<const uint32_t*>(nullptr), n, N, a->out_offsets);
    return check_launch("csr_offsets");
  }
  const size_t un = static_cast<size_t>(n);
  uint64_t* tk[2] = {reinterpret_cast<uint64_t*>(ws + w.tkey),
                     reinterpret_cast<uint64_t*>(ws + w.tkey + align256(un * 8))};
  uint32_t* ix[2] = {reinterpret_cast<uint32_t*>(ws + w.idx),
                     reinterpret_cast<uint32_t*>(ws + w.idx + align256(un * 4))};
  uint32_t* nk[2] = {reinterpret_cast<uint32_t*>(ws + w.nkey),
                     reinterpret_cast<uint32_t*>(ws + w.nkey + align256(un * 4))};
  uint32_t* count = reinterpret_cast<uint32_t*>(ws + w.count);
  uint32_t* sums = reinterpret_cast<uint32_t*>(ws + w.sums);
  // the row gather's records take the time keys' place, once those are sorted
  EventRec* rec = reinterpret_cast<EventRec*>(ws + w.tkey);
  const int64_t ne = pairs ? n / 2 : n;  // events, or entries given one by one
  const unsigned ge = static_cast<unsigned>(cdiv(ne, kThreads));
  int cur = 0;
  const bool ident = pairs && !by_call;  // already in stable time order
  bool keyed = false;                    // node keys and records are done
  if (by_call) {
    // the build order from the segments; the tiles' bitmaps in nk[1] (kSegWords per kSegTile
    // events: its n words hold them), their first and last starts and the nearest ones around
    // them in tk[1] (both free until the first pass)
    const unsigned gt = static_cast<unsigned>(cdiv(ne, kSegTile));
    uint32_t* bitmap = nk[1];
    uint32_t* first = reinterpret_cast<uint32_t*>(tk[1]);
    uint32_t* last = first + gt;
    uint32_t* prev = last + gt;
    uint32_t* next = prev + gt;
    hipLaunchKernelGGL(csr_seg_tiles, dim3(gt), dim3(kThreads), 0, stream, a->time, ne, runs, a->call_starts,
                       a->num_calls, bitmap, first, last);
    if ((rc = check_launch("csr_seg_tiles"))) return rc;
    hipLaunchKernelGGL(csr_seg_edges, dim3(2), dim3(kEdgeThreads), 0, stream, static_cast<const uint32_t*>(first),
                       static_cast<const uint32_t*>(last), static_cast<int64_t>(gt), ne, prev, next);
    if ((rc = check_launch("csr_seg_edges"))) return rc;
    auto order = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(gt), dim3(kThreads), 0, stream, a->time, a->from, a->to, ne, N,
                         static_cast<const uint32_t*>(bitmap), static_cast<const uint32_t*>(prev),
                         static_cast<const uint32_t*>(next), ix[0], tk[0], nk[0], rec, a->status);
    };
    if (runs)
      order(csr_seg_order<true>);
    else
      order(csr_seg_order<false>);
    if ((rc = check_launch("csr_seg_order"))) return rc;
    keyed = runs != 0;
    // stable by time unless the runs already are
    if (!runs && (rc = radix_sort<uint64_t>(tk, ix, cur, n, 64, w.r, count, sums, stream))) return rc;
  } else if (ident) {
    hipLaunchKernelGGL(csr_pair_keys, dim3(ge), dim3(kThreads), 0, stream, a->time, a->from, a->to, ne, N, nk[0], rec,
                       a->status);
    if ((rc = check_launch("csr_pair_keys"))) return rc;
    keyed = true;
  } else {
    hipLaunchKernelGGL(csr_init, dim3(g1), dim3(kThreads), 0, stream, a->time, n, tk[0], ix[0]);
    if ((rc = check_launch("csr_init"))) return rc;
    if ((rc = radix_sort<uint64_t>(tk, ix, cur, n, 64, w.r, count, sums, stream))) return rc;
  }
  // then stable by node over ceil(log2 N) bits (out-of-range ids sort last)
  if (!keyed) {
    hipLaunchKernelGGL(csr_records, dim3(ge), dim3(kThreads), 0, stream, a->time, a->from, a->to, ne, rec);
    if ((rc = check_launch("csr_records"))) return rc;
    hipLaunchKernelGGL(csr_node_keys, dim3(g1), dim3(kThreads), 0, stream, a->from, a->to, pairs,
                       static_cast<const uint32_t*>(ix[cur]), n, N, nk[0], a->status);
    if ((rc = check_launch("csr_node_keys"))) return rc;
  }
  int bits = 1;
  while ((int64_t(1) << bits) < N + 1) ++bits;  // + 1: the out-of-range key 0xffffffff
  // the node keys ride in nk[], the permutation in ix[] (starting where the time
  // passes left it)
  uint32_t* pv[2] = {ix[cur], ix[1 - cur]};
  int ncur = 0;
  if ((rc = radix_sort<uint32_t>(nk, pv, ncur, n, bits, w.r, count, sums, stream, ident))) return rc;
  uint32_t* perm_in = pv[ncur];
  hipLaunchKernelGGL(csr_offsets, dim3(static_cast<unsigned>(cdiv(N + 1, kThreads))), dim3(kThreads), 0,
                     stream, static_cast<const uint32_t*>(nk[ncur]), n, N, a->out_offsets);
  if ((rc = check_launch("csr_offsets"))) return rc;
  const bool fe = row_bytes > 0;
  const int vec = fe ? row_vec(row_bytes, reinterpret_cast<uintptr_t>(a->feats) | reinterpret_cast<uintptr_t>(a->out_feats)) : 16;
  const int64_t nch = fe ? row_chunks(row_bytes, vec) : 1;
  const int per = static_cast<int>(std::min<int64_t>(std::max<int64_t>(kGatherChunks / nch, 1), kGatherMost));
  const uint32_t magic = nch > 1 ? 0xffffffffu / static_cast<uint32_t>(nch) + 1u : 0u;
  const int64_t ntiles = cdiv(n, per);
  int64_t gblocks = ntiles;
  const uint32_t* order = nullptr;
  // Rows of at most 256 bytes and at least 1M entries: below that the events fit
  // the caches in any order, and a wider row fills its lines by itself
  if (per >= 64 && n >= (int64_t(1) << 20)) {
    // the node keys are done with (the offsets are out): tile keys, sorted keys and order take their place
    uint32_t* key = nk[0];
    uint32_t* val = nk[0] + 2 * ntiles;
    hipLaunchKernelGGL(csr_tile_keys, dim3(static_cast<unsigned>(cdiv(ntiles, kThreads))), dim3(kThreads), 0, stream,
                       static_cast<const uint32_t*>(perm_in), ntiles, per, pairs, key);
    if ((rc = check_launch("csr_tile_keys"))) return rc;
    int ebits = 1;
    while ((int64_t(1) << ebits) < ne) ++ebits;
    const int dbits = std::min(ebits, kMaxDigitBits);
    if ((rc = radix_pass<uint32_t>(key, nullptr, key + ntiles, val, ntiles, ebits - dbits, dbits, radix_scratch(ntiles),
                                   count, sums, stream)))
      return rc;
    order = val;
    gblocks = cdiv(ntiles, kXcds * kGatherSlice) * (kXcds * kGatherSlice);
  }
  auto gather = [&](auto kernel) {
    for (int64_t t0 = 0; t0 < gblocks; t0 += kGatherTiles)
      hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(std::min(gblocks - t0, kGatherTiles))), dim3(kThreads), 0,
                         stream, static_cast<const uint32_t*>(perm_in), n, static_cast<const EventRec*>(rec), pairs,
                         a->event, a->num_events, static_cast<const uint8_t*>(a->feats), row_bytes,
                         static_cast<int>(nch), magic, per, order, t0, ntiles, a->out_ids, a->out_times, a->out_eids,
                         static_cast<uint8_t*>(fe ? a->out_feats : nullptr), a->status);
  };
  if (vec == 16)
    gather(csr_gather<16>);
  else if (vec == kAnyRow)
    gather(csr_gather<kAnyRow>);
  else if (vec == 4)
    gather(csr_gather<4>);
  else
    gather(csr_gather<2>);
  return check_launch("csr_gather");
}

extern "C" size_t tgx_csr_scan_workspace_size(void) { return kScanParts * sizeof(ScanPart); }

extern "C" int tgx_csr_scan(const int64_t* src, const int64_t* dst, const double* time, int64_t num_events,
                            const int64_t* call_starts, int64_t num_calls, int64_t* out, void* workspace,
                            size_t workspace_bytes, void* stream_) {
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  if (num_events <= 0) return fail(TGX_ERR_ARG, "tgx_csr_scan: num_events %lld must be positive", (long long)num_events);
  if (num_calls < 0) return fail(TGX_ERR_ARG, "tgx_csr_scan: negative num_calls");
  if (src == nullptr || dst == nullptr || time == nullptr || out == nullptr ||
      (num_calls > 0 && call_starts == nullptr))
    return fail(TGX_ERR_ARG, "tgx_csr_scan: src/dst/time/out (and call_starts when num_calls > 0) must not be NULL");
  if (workspace == nullptr || workspace_bytes < tgx_csr_scan_workspace_size())
    return fail(TGX_ERR_ARG, "tgx_csr_scan: workspace of %zu bytes needed, got %zu", tgx_csr_scan_workspace_size(),
                workspace_bytes);
  // about four events per thread before the grid reaches kScanParts workgroups
  const int np = static_cast<int>(std::min<int64_t>(cdiv(num_events, 4 * kThreads), kScanParts));
  ScanPart* parts = static_cast<ScanPart*>(workspace);
  hipLaunchKernelGGL(csr_scan_part, dim3(np), dim3(kThreads), 0, stream, src, dst, time, num_events, call_starts,
                     num_calls, parts);
  int rc;
  if ((rc = check_launch("csr_scan_part"))) return rc;
  hipLaunchKernelGGL(csr_scan_final, dim3(1), dim3(kThreads), 0, stream, static_cast<const ScanPart*>(parts), np,
                     out);
  return check_launch("csr_scan_final");
}

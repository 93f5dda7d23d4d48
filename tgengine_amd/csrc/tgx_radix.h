// Stable LSD radix sort of (key, uint32 value) pairs, shared by the CSR build
// (tgx_csr.hip) and the negative pool (tgx_negpool.hip).  The key bits are split
// evenly over as few passes of at most 10 bits as cover them (20 bits: two
// passes).
//
// A pass is three launches.  The keys are cut into at most kMaxBlocks
// contiguous ranges of whole tiles, one per workgroup:
//   hist    : each range's digit counts, count[digit][range].  Eight LDS counters
//             per digit (lane % 8, in neighbouring banks): the lanes of a wave
//             that hold one digit, as in the high digits of skewed node ids,
//             queue at eight counters instead of one;
//   rows    : one workgroup per digit scans its row of counts, so count[d][b] is
//             range b's place among digit d's keys, and total[d] their number;
//   scatter : a workgroup scans the totals and then takes its range tile by
//             tile.  Each wavefront ranks its consecutive part of the tile on its
//             own, 64 keys at a time: lanes with equal digits find each other
//             by ballots, and the wave's counter of the digit gives the rank
//             (no workgroup barrier between the rounds).  One prefix over digits
//             and waves gives every key its place in the tile sorted by digit;
//             keys, then values go through one LDS buffer in that order, so a
//             digit's keys leave as a run.
// A pass of 16M keys moves 320 MB.  Two passes over 16M 20-bit keys take 215 us
// with skewed digits and 332 us with uniform ones, whose runs of 4 keys leave
// partial lines (8-bit passes of 2,048-key tiles with a device-wide scan of the
// counts and four barriers per 256 keys took 480 us for three); 8,192-key tiles
// need more registers than two workgroups per CU have: 243 and 302 us.
// Everything lives in an anonymous namespace: each including file gets its own
// copy of the kernels.
#pragma once

#include "tgx_internal.h"

#include <algorithm>
#include <type_traits>
#include <vector>

namespace tgx {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;

constexpr int kSortThreads = 512;
constexpr int kSortWaves = kSortThreads / kWave;
constexpr int kMaxDigitBits = 10;
constexpr int kMaxBins = 1 << kMaxDigitBits;
constexpr int kHistCopies = 8;
constexpr int kMaxBlocks = 1024;  // ranges of a pass
static_assert(kMaxBins <= 2 * kSortThreads, "two digits per thread in the prefix steps");

template <typename K>
__device__ __forceinline__ int digit_of(K k, int shift, int bins) {
  return static_cast<int>(k >> shift) & (bins - 1);
}

__device__ __forceinline__ void sort_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// exclusive prefix of one value per thread over the workgroup (THREADS threads,
// wsum: one word per wave); `total` gets the sum
template <int THREADS>
__device__ __forceinline__ uint32_t block_exclusive(uint32_t x, uint32_t* wsum, uint32_t& total) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = threadIdx.x / kWave;
  uint32_t incl = x;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint32_t y = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += y;
  }
  if (lane == kWave - 1) wsum[wv] = incl;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < THREADS / kWave; ++w) {
    if (w < wv) before += wsum[w];
    total += wsum[w];
  }
  return before + incl - x;
}

// count[d * gridDim.x + block] = keys of digit d in the block's range
template <typename K>
__global__ __launch_bounds__(kSortThreads) void radix_hist(const K* __restrict__ keys, int64_t n, int64_t range,
                                                           int shift, int bins, uint32_t* __restrict__ count) {
  extern __shared__ uint32_t h[];  // [bins][kHistCopies]
  for (int i = threadIdx.x; i < bins * kHistCopies; i += kSortThreads) h[i] = 0;
  __syncthreads();
  constexpr int VEC = 16 / sizeof(K);
  struct alignas(16) Pack {
    K k[VEC];
  };
  const int64_t lo = static_cast<int64_t>(blockIdx.x) * range;  // a multiple of VEC, as is the full part's end
  const int64_t hi = lo + range < n ? lo + range : n;
  const int64_t full = lo + (hi - lo) / VEC * VEC;
  uint32_t* mine = h + (threadIdx.x & (kHistCopies - 1));
#pragma unroll 4
  for (int64_t j = lo + static_cast<int64_t>(threadIdx.x) * VEC; j < full; j += kSortThreads * VEC) {
    const Pack p = *reinterpret_cast<const Pack*>(keys + j);
#pragma unroll
    for (int u = 0; u < VEC; ++u) atomicAdd(&mine[digit_of(p.k[u], shift, bins) * kHistCopies], 1u);
  }
  if (full + threadIdx.x < hi) atomicAdd(&mine[digit_of(keys[full + threadIdx.x], shift, bins) * kHistCopies], 1u);
  __syncthreads();
  for (int d = threadIdx.x; d < bins; d += kSortThreads) {
    uint32_t c = 0;
#pragma unroll
    for (int u = 0; u < kHistCopies; ++u) c += h[d * kHistCopies + u];
    count[static_cast<int64_t>(d) * gridDim.x + blockIdx.x] = c;
  }
}

// exclusive scan of digit blockIdx.x's row of nblocks (<= kMaxBlocks) counts in
// place; its sum goes to total[blockIdx.x]
__global__ __launch_bounds__(kThreads) void radix_rows(uint32_t* __restrict__ count, int nblocks,
                                                       uint32_t* __restrict__ total) {
  __shared__ uint32_t wsum[kWaves];
  constexpr int PER = kMaxBlocks / kThreads;
  uint32_t* row = count + static_cast<int64_t>(blockIdx.x) * nblocks;
  uint32_t v[PER], s = 0;
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const int i = static_cast<int>(threadIdx.x) * PER + r;
    v[r] = i < nblocks ? row[i] : 0u;
    s += v[r];
  }
  uint32_t all;
  uint32_t run = block_exclusive<kThreads>(s, wsum, all);
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const int i = static_cast<int>(threadIdx.x) * PER + r;
    if (i < nblocks) row[i] = run;
    run += v[r];
  }
  if (threadIdx.x == 0) total[blockIdx.x] = all;
}

constexpr size_t scatter_lds(size_t key_bytes, int items, int bins) {
  return static_cast<size_t>(kSortThreads) * items * key_bytes + static_cast<size_t>(bins) * (2 * kSortWaves + 8);
}

template <typename K, int ITEMS>
__global__ __launch_bounds__(kSortThreads) __attribute__((amdgpu_waves_per_eu(4))) void radix_scatter(const K* __restrict__ kin,
                                                              const uint32_t* __restrict__ vin, K* __restrict__ kout,
                                                              uint32_t* __restrict__ vout, int64_t n, int64_t range,
                                                              int shift, int dbits,
                                                              const uint32_t* __restrict__ count,
                                                              const uint32_t* __restrict__ total) {
  constexpr int TILE = kSortThreads * ITEMS;
  extern __shared__ __align__(16) uint8_t smem[];
  __shared__ uint32_t wsum[kSortWaves];
  const int bins = 1 << dbits;
  K* skey = reinterpret_cast<K*>(smem);                // [TILE] the tile in digit order: its keys,
  uint32_t* sval = reinterpret_cast<uint32_t*>(smem);  // [TILE] then its values
  uint32_t* gpos = reinterpret_cast<uint32_t*>(smem + sizeof(K) * TILE);  // [bins] next output position of the digit
  uint32_t* gofs = gpos + bins;  // [bins] output position - local position of the tile's digit
  uint16_t* wcnt = reinterpret_cast<uint16_t*>(gofs + bins);  // [waves][bins] counts, then local positions
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = threadIdx.x / kWave;
  const uint64_t lt = (uint64_t(1) << lane) - 1;
  const int d0 = static_cast<int>(threadIdx.x) * 2;  // this thread's digits in the prefix steps: d0, d0 + 1
  {
    uint32_t t0 = 0, t1 = 0, all;
    if (d0 < bins) {
      t0 = total[d0];
      t1 = total[d0 + 1];
    }
    const uint32_t at = block_exclusive<kSortThreads>(t0 + t1, wsum, all);
    if (d0 < bins) {
      gpos[d0] = at + count[static_cast<int64_t>(d0) * gridDim.x + blockIdx.x];
      gpos[d0 + 1] = at + t0 + count[static_cast<int64_t>(d0 + 1) * gridDim.x + blockIdx.x];
    }
  }
  uint16_t* mycnt = wcnt + wv * bins;
  const uint32_t per = static_cast<uint32_t>(range) / TILE;  // range < 2^31, whole tiles
  for (uint32_t tile = blockIdx.x * per; tile < (blockIdx.x + 1) * per; ++tile) {  // workgroup-uniform
    const int64_t base = static_cast<int64_t>(tile) * TILE;
    if (base >= n) break;
    // the wave's consecutive part of the tile, 64 keys per item
    const uint32_t tn = static_cast<uint32_t>(n - base < TILE ? n - base : TILE);
    const uint32_t i0 = wv * (kWave * ITEMS) + lane;
    const K* kt = kin + base;
    const uint32_t* vt = vin + base;
    K k[ITEMS];
    uint32_t rank[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      const uint32_t i = i0 + r * kWave;
      k[r] = kt[i < tn ? i : tn - 1];
    }
    for (int i = lane; i < bins / 2; i += kWave) reinterpret_cast<uint32_t*>(mycnt)[i] = 0u;
    sort_wave_sync();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      const bool valid = i0 + r * kWave < tn;
      const int d = digit_of(k[r], shift, bins);
      // lanes with the same digit: AND of the digit bits' ballots
      uint64_t peers = __ballot(valid);
      uint32_t plo = static_cast<uint32_t>(peers), phi = static_cast<uint32_t>(peers >> 32);
      for (int bit = 0; bit < dbits; ++bit) {
        const int32_t on = (d << (31 - bit)) >> 31;  // all ones where the bit is set
        const uint64_t m = __ballot(on != 0);
        plo &= ~(static_cast<uint32_t>(m) ^ static_cast<uint32_t>(on));
        phi &= ~(static_cast<uint32_t>(m >> 32) ^ static_cast<uint32_t>(on));
      }
      peers = static_cast<uint64_t>(phi) << 32 | plo;
      const uint32_t before = valid ? mycnt[d] : 0u;
      sort_wave_sync();  // every lane has read its counter
      const uint32_t below = static_cast<uint32_t>(__popcll(peers & lt));
      if (valid && below == 0) mycnt[d] = static_cast<uint16_t>(before + __popcll(peers));
      sort_wave_sync();
      rank[r] = before + below;
    }
    __syncthreads();
    {  // local positions: digits in order, within a digit the waves in order
      uint32_t c[kSortWaves], s0 = 0, s1 = 0, all;
      if (d0 < bins) {
#pragma unroll
        for (int w = 0; w < kSortWaves; ++w) {
          c[w] = *reinterpret_cast<const uint32_t*>(wcnt + w * bins + d0);
          s0 += c[w] & 0xffffu;
          s1 += c[w] >> 16;
        }
      }
      uint32_t p0 = block_exclusive<kSortThreads>(s0 + s1, wsum, all);
      uint32_t p1 = p0 + s0;
      if (d0 < bins) {
        gofs[d0] = gpos[d0] - p0;
        gofs[d0 + 1] = gpos[d0 + 1] - p1;
        gpos[d0] += s0;
        gpos[d0 + 1] += s1;
#pragma unroll
        for (int w = 0; w < kSortWaves; ++w) {
          *reinterpret_cast<uint32_t*>(wcnt + w * bins + d0) = p0 | (p1 << 16);
          p0 += c[w] & 0xffffu;
          p1 += c[w] >> 16;
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      if (i0 + r * kWave < tn) {
        rank[r] += mycnt[digit_of(k[r], shift, bins)];
        skey[rank[r]] = k[r];
      }
    }
    __syncthreads();
    // the values, loaded while the keys go out
    uint32_t v[ITEMS];
    if (vin != nullptr) {
#pragma unroll
      for (int r = 0; r < ITEMS; ++r) v[r] = vt[i0 + r * kWave < tn ? i0 + r * kWave : tn - 1];
    } else {  // the identity
#pragma unroll
      for (int r = 0; r < ITEMS; ++r) v[r] = static_cast<uint32_t>(base) + static_cast<uint32_t>(i0 + r * kWave);
    }
    uint32_t at[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      const uint32_t i = r * kSortThreads + threadIdx.x;
      if (i < tn) {
        const K x = skey[i];
        at[r] = gofs[digit_of(x, shift, bins)] + i;
        kout[at[r]] = x;
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
      if (i0 + r * kWave < tn) sval[rank[r]] = v[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
      const uint32_t i = r * kSortThreads + threadIdx.x;
      if (i < tn) vout[at[r]] = sval[i];
    }
    // the next tile's first write to the buffer comes two barriers later
  }
}

size_t align256(size_t x) { return (x + 255) & ~static_cast<size_t>(255); }
int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Shape of a sort of n keys: keys per thread and tile, ranges, and the scratch for
// counts and totals.  2,048-key tiles while they are at most kMaxBlocks (up to 2M
// keys), so that small sorts still spread over the device; 4,096 above.
struct RadixScratch {
  int items = 4;
  int64_t nblocks = 1, range = 0;
  size_t count_bytes = 0, sums_bytes = 0;
};

RadixScratch radix_scratch(int64_t n) {
  RadixScratch r;
  r.items = n <= int64_t(4) * kSortThreads * kMaxBlocks ? 4 : 8;
  const int64_t tile = int64_t(kSortThreads) * r.items;
  const int64_t ntiles = std::max<int64_t>(cdiv(n, tile), 1);
  r.range = cdiv(ntiles, kMaxBlocks) * tile;
  r.nblocks = std::max<int64_t>(cdiv(n, r.range), 1);
  r.count_bytes = align256(static_cast<size_t>(r.nblocks) * kMaxBins * 4);
  r.sums_bytes = align256(kMaxBins * 4);
  return r;
}

template <typename K, int ITEMS>
int radix_scatter_launch(const K* kin, const uint32_t* vin, K* kout, uint32_t* vout, int64_t n, int shift, int dbits,
                         const RadixScratch& w, const uint32_t* count, const uint32_t* total, hipStream_t stream) {
  hipLaunchKernelGGL((radix_scatter<K, ITEMS>), dim3(static_cast<unsigned>(w.nblocks)), dim3(kSortThreads),
                     scatter_lds(sizeof(K), ITEMS, 1 << dbits), stream, kin, vin, kout, vout, n, w.range, shift, dbits,
                     count, total);
  return check_launch("radix_scatter");
}

template <typename K>
int radix_pass(const K* kin, const uint32_t* vin, K* kout, uint32_t* vout, int64_t n, int shift, int dbits,
               const RadixScratch& w, uint32_t* count, uint32_t* total, hipStream_t stream) {
  const int bins = 1 << dbits;
  hipLaunchKernelGGL(radix_hist<K>, dim3(static_cast<unsigned>(w.nblocks)), dim3(kSortThreads),
                     static_cast<size_t>(bins) * kHistCopies * 4, stream, kin, n, w.range, shift, bins, count);
  int rc = check_launch("radix_hist");
  if (rc) return rc;
  hipLaunchKernelGGL(radix_rows, dim3(static_cast<unsigned>(bins)), dim3(kThreads), 0, stream, count,
                     static_cast<int>(w.nblocks), total);
  if ((rc = check_launch("radix_rows"))) return rc;
  if (w.items == 4) return radix_scatter_launch<K, 4>(kin, vin, kout, vout, n, shift, dbits, w, count, total, stream);
  return radix_scatter_launch<K, 8>(kin, vin, kout, vout, n, shift, dbits, w, count, total, stream);
}

// passes over bits [0, bits) of the keys, ping-ponging between k[0]/v[0] and
// k[1]/v[1]; `cur` is the buffer holding the input, and then the output.  With
// ident_values the first pass takes the values 0, 1, ..., n-1 without reading them
template <typename K>
int radix_sort(K* k[2], uint32_t* v[2], int& cur, int64_t n, int bits, const RadixScratch& r,
               uint32_t* count, uint32_t* sums, hipStream_t stream, bool ident_values = false) {
  int passes = static_cast<int>(cdiv(bits, kMaxDigitBits));
  for (int shift = 0; shift < bits; --passes) {
    const int dbits = std::max(static_cast<int>(cdiv(bits - shift, passes)), 1);
    const uint32_t* vin = shift == 0 && ident_values ? nullptr : v[cur];
    const int rc = radix_pass<K>(k[cur], vin, k[1 - cur], v[1 - cur], n, shift, dbits, r, count, sums, stream);
    if (rc) return rc;
    cur = 1 - cur;
    shift += dbits;
  }
  return TGX_OK;
}

}  // namespace
}  // namespace tgx

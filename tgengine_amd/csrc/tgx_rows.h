// Feature rows as chunks of one vector access, shared by the gather, the CSR build
// and the ring update.
//
// VEC is the chunk's bytes: 16 where every row starts at a multiple of 16, else
// kAnyRow, 16-byte accesses at the row's own alignment (2 bytes or more), for rows
// of at least 16 bytes; the last chunk ends with the row, so it overlaps the one
// before it and both write the same bytes there.  Shorter rows take 4- or 2-byte
// chunks.  A 171-d fp32 row was 171 4-byte accesses before, where a 172-d one is 43:
// the gather of 200 training events at K = 64 took 28.4 us with it, 16.7 now (172-d:
// 16.0).  511-d bf16 rows went in 2-byte chunks: 14,000 queries at K = 64 took
// 554 us, 313 now (512-d: 260).
#pragma once

#include "tgx_internal.h"

namespace tgx {

constexpr int kAnyRow = 1;

typedef unsigned int row_u32x4 __attribute__((ext_vector_type(4)));
typedef row_u32x4 row_u32x4_any __attribute__((aligned(2)));

template <int VEC>
struct RowChunk {  // T: the value; M: the memory it is read from and written to
  using T = row_u32x4;
  using M = row_u32x4;
};
template <>
struct RowChunk<kAnyRow> {
  using T = row_u32x4;
  using M = row_u32x4_any;
};
template <>
struct RowChunk<4> {
  using T = uint32_t;
  using M = uint32_t;
};
template <>
struct RowChunk<2> {
  using T = uint16_t;
  using M = uint16_t;
};

// byte offset of chunk c of a row
template <int VEC, typename I>
__device__ __forceinline__ I chunk_at(I c, I row_bytes) {
  if constexpr (VEC == kAnyRow)
    return c * 16 + 16 <= row_bytes ? c * 16 : row_bytes - 16;
  else
    return c * VEC;
}

template <int VEC>
__device__ __forceinline__ typename RowChunk<VEC>::T load_chunk(const uint8_t* p) {
  return *reinterpret_cast<const typename RowChunk<VEC>::M*>(p);
}

template <int VEC, bool NT>
__device__ __forceinline__ void store_chunk(uint8_t* p, typename RowChunk<VEC>::T v) {
  using M = typename RowChunk<VEC>::M;
  if constexpr (NT)
    __builtin_nontemporal_store(static_cast<M>(v), reinterpret_cast<M*>(p));
  else
    *reinterpret_cast<M*>(p) = v;
}

// VEC of rows of row_bytes (even) whose arrays' addresses OR to `addr` (0 without rows)
inline int row_vec(int64_t row_bytes, uintptr_t addr) {
  if (row_bytes % 16 == 0 && (addr & 15) == 0) return 16;
  if (row_bytes >= 16) return kAnyRow;
  return row_bytes % 4 == 0 && (addr & 3) == 0 ? 4 : 2;
}

inline int64_t row_chunks(int64_t row_bytes, int vec) {
  return vec == kAnyRow ? (row_bytes + 15) / 16 : row_bytes / vec;
}

}  // namespace tgx

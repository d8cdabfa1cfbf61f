// Elementwise passes over packs: how many a thread takes, and how it reads and writes one.
#pragma once

#include <algorithm>
#include <initializer_list>

#include "omx_common.h"

namespace {

constexpr int BK_THREADS = 256;
constexpr int BK_PACKS = 4;  // packs per thread of a large pass

// A pack is V consecutive elements: one 16-byte (f32) or 8-byte (bf16) access
// when V == 4, one element when V == 1.
template <typename T, int V>
__device__ __forceinline__ void load_pack(const T* __restrict__ p, size_t pack, float (&v)[V]) {
  if constexpr (V == 1) {
    v[0] = dev_load<T>(p, pack);
  } else if constexpr (sizeof(T) == 4) {
    float4 q = reinterpret_cast<const float4*>(p)[pack];
    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
  } else {
    uint2 q = reinterpret_cast<const uint2*>(p)[pack];
    v[0] = __uint_as_float(q.x << 16); v[1] = __uint_as_float(q.x & 0xffff0000u);
    v[2] = __uint_as_float(q.y << 16); v[3] = __uint_as_float(q.y & 0xffff0000u);
  }
}
template <typename T, int V>
__device__ __forceinline__ void store_pack(T* __restrict__ p, size_t pack, const float (&v)[V]) {
  if constexpr (V == 1) {
    dev_store<T>(p, pack, v[0]);
  } else if constexpr (sizeof(T) == 4) {
    reinterpret_cast<float4*>(p)[pack] = make_float4(v[0], v[1], v[2], v[3]);
  } else {
    uint2 q;
    q.x = dev_pack_bf16_pair(v[0], v[1]);
    q.y = dev_pack_bf16_pair(v[2], v[3]);
    reinterpret_cast<uint2*>(p)[pack] = q;
  }
}

// Packs per thread: one up to four blocks per compute unit, two up to eight, four beyond (and twice that as often as it takes to keep a
// launch under the 2^32 threads it may have). A few thousand rows were 16 to 176
// blocks whose threads took their packs one latency after the other (rope over 1024 x 4 x 64 6.3 us on 32 blocks, 3.2 on 128).
// `blocks`: the most there may be, or (in a kernel) how many there are, which gives the same answer.
__host__ __device__ inline uint64_t packs_per_thread(uint64_t packs, uint64_t blocks) {
  if (packs <= blocks * BK_THREADS) return 1;
  uint64_t each = 2;
  while (packs > blocks * (each * BK_THREADS)) each *= 2;
  return each;
}
inline dim3 pack_grid(uint64_t packs) {
  constexpr uint64_t FEW = 1024, MOST = (1ull << 32) / BK_THREADS - 1;
  const uint64_t each = packs <= FEW * (2 * BK_THREADS) ? packs_per_thread(packs, FEW) : std::max<uint64_t>(BK_PACKS, packs_per_thread(packs, MOST));
  const uint64_t per_block = each * BK_THREADS, blocks = (packs + per_block - 1) / per_block;
  return dim3(static_cast<unsigned>(blocks > 0 ? blocks : 1));
}
#define PACK_LOOP(p, packs)                                                                                             \
  for (size_t span_ = packs_per_thread(packs, gridDim.x) * BK_THREADS, p = blockIdx.x * span_ + threadIdx.x,            \
              end_ = min(static_cast<size_t>(packs), (blockIdx.x + 1) * span_);                                          \
       p < end_; p += BK_THREADS)
// n / d in 32 bits where they allow it (a 64-bit division is some 100 instructions).
__device__ __forceinline__ size_t quotient(size_t n, size_t d) {
  return ((n | d) >> 32) == 0 ? static_cast<unsigned>(n) / static_cast<unsigned>(d) : n / d;
}

// Whether every pointer allows 4-element packs of `esz`-byte elements.
inline bool packs_of_four(uint64_t n, size_t esz, std::initializer_list<const void*> ptrs) {
  if (n % 4 != 0) return false;
  uintptr_t mask = esz * 4 - 1, bits = 0;
  for (const void* p : ptrs) bits |= reinterpret_cast<uintptr_t>(p);
  return (bits & mask) == 0;
}

}  // namespace

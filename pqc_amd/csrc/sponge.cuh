// Short-message sponge helpers for one state per lane.
#pragma once
#include "keccak.cuh"

namespace pqc {

// Absorb W full little-endian words plus one extra word `tail` (the message
// tail bytes with the domain byte already placed), pad the last rate byte, and
// permute once.  Requires W + 1 <= RATE.
// TWO: keccakf1600_two.
template <int RATE, int W, bool TWO = false>
__device__ __forceinline__ void absorb_fixed(uint64_t (&A)[25], const uint64_t (&m)[W], uint64_t tail) {
  static_assert(W + 1 <= RATE, "message must fit one block");
#pragma unroll
  for (int i = 0; i < 25; ++i) A[i] = (i < W) ? m[i] : 0;
  A[W] ^= tail;
  A[RATE - 1] ^= 0x8000000000000000ull;
  if constexpr (TWO)
    keccakf1600_two(A);
  else
    keccakf1600(A);
}

__device__ __forceinline__ uint64_t load_u64(const uint8_t* p) {
  return *reinterpret_cast<const uint64_t*>(p);
}

// The same load from global memory, as a global (not flat) load: it counts in
// vmcnt only, so waits for LDS results do not also wait for it.
__device__ __forceinline__ uint64_t load_u64_global(const uint8_t* p) {
  return *(const __attribute__((address_space(1))) uint64_t*)p;
}

// Absorb NWORDS 64-bit words from global memory, one state per lane, the next block's
// words loaded during a block's permutation (keccakf1600_two).  The whole blocks run in a
// loop without a condition on the words; the last, partial one follows.
template <int RATE, int NWORDS>
__device__ __forceinline__ void sponge_absorb_two(uint64_t (&A)[25], const uint8_t* __restrict__ msg,
                                                  uint8_t domain) {
  constexpr int FULL = NWORDS / RATE, REST = NWORDS % RATE;
  static_assert(FULL >= 1, "at least one whole block");
  const __attribute__((address_space(1))) uint64_t* p = (const __attribute__((address_space(1))) uint64_t*)msg;
  uint64_t cur[RATE];
#pragma unroll
  for (int i = 0; i < 25; ++i) A[i] = 0;
#pragma unroll
  for (int w = 0; w < RATE; ++w) cur[w] = p[w];
#pragma unroll 1
  for (int b = 0; b < FULL; ++b) {
#pragma unroll
    for (int w = 0; w < RATE; ++w) A[w] ^= cur[w];
    // after the last whole block: the message's last RATE words, REST of them new
    p = b + 1 < FULL ? p + RATE : p + REST;
#pragma unroll
    for (int w = 0; w < RATE; ++w) cur[w] = p[w];
    keccakf1600_two(A);
  }
#pragma unroll
  for (int w = 0; w < REST; ++w) A[w] ^= cur[RATE - REST + w];
  A[REST] ^= (uint64_t)domain;
  A[RATE - 1] ^= 0x8000000000000000ull;
  keccakf1600_two(A);
}

__device__ __forceinline__ void store_u64(uint8_t* p, uint64_t v) {
  *reinterpret_cast<uint64_t*>(p) = v;
}

}  // namespace pqc

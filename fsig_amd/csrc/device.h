// Device helpers for gfx950 (wave64): block ids remapped per XCD, wave
// reductions, block scans, sorted-list search and MurmurHash2.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "internal.h"

#define FSIG_BLOCK 256

// Workgroups are dispatched round-robin over the 8 XCDs of an MI355X, each
// with its own L2.  Remapping makes XCD x own the contiguous logical range
// [x*n/8, (x+1)*n/8), so neighbouring rows (which share parents, hence
// candidate lists) meet in one L2.
__device__ __forceinline__ uint32_t xcd_block() {
  const uint32_t b = blockIdx.x, n = gridDim.x;
  if ((n & 7u) != 0) return b;
  return (b & 7u) * (n >> 3) + (b >> 3);
}

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Flag of a host mailbox (pinned coherent memory): the words written before
// it, by this thread or by a block that has met at a barrier after its own
// system fences, are visible to a host that reads `seq` from it.
__device__ __forceinline__ void mail_flag(unsigned long long* flag, unsigned long long seq) {
  __threadfence_system();
  __hip_atomic_store(flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Sums into striped counters (kStripes).  Additions of 64-bit words to one
// address take 12..13 ns each, one after another, however many compute units
// send them: with one address and an addition per wavefront and counter, the
// 16,384 wavefronts of a full launch spent 410 us on two statistics.
//
// dst[i], in the block's copy, += the sum of v[i] over the block (dst[i] may
// be null).  Every thread of the block must call it.
template <int N>
__device__ __forceinline__ void block_add(const unsigned long long (&v)[N], unsigned long long* const (&dst)[N]) {
  __shared__ unsigned long long part[FSIG_BLOCK / 64][N];
#pragma unroll
  for (int i = 0; i < N; i++) {
    const unsigned long long s = wave_sum_u64(v[i]);
    if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6][i] = s;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < N; i++)
    if (threadIdx.x == (uint32_t)i && dst[i]) {
      unsigned long long s = 0;
#pragma unroll
      for (int w = 0; w < FSIG_BLOCK / 64; w++) s += part[w][i];
      if (s) atomicAdd(dst[i] + (blockIdx.x & (kStripes - 1)) * kStripeWords, s);
    }
}

__device__ __forceinline__ uint32_t lane_id() { return threadIdx.x & 63u; }

// Exclusive scan of one u64 per thread over a 256-thread block; `total`
// receives the block sum.  lds must hold 4 words.  All threads must call it.
__device__ __forceinline__ uint64_t block_exclusive_scan(uint64_t v, uint64_t* lds, uint64_t& total) {
  const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
  uint64_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    uint64_t y = __shfl_up(x, o, 64);
    if (lane >= (uint32_t)o) x += y;
  }
  if (lane == 63) lds[wid] = x;
  __syncthreads();
  uint64_t pre = 0, tot = 0;
#pragma unroll
  for (uint32_t w = 0; w < FSIG_BLOCK / 64; w++) {
    uint64_t s = lds[w];
    if (w < wid) pre += s;
    tot += s;
  }
  __syncthreads();
  total = tot;
  return pre + x - v;
}

__device__ __forceinline__ uint64_t block_sum(uint64_t v, uint64_t* lds) {
  uint64_t t;
  (void)block_exclusive_scan(v, lds, t);
  return t;
}

// Membership of x in the ascending list a[0..n).
__device__ __forceinline__ bool sorted_contains(const uint32_t* __restrict__ a, uint32_t n, uint32_t x) {
  uint32_t lo = 0, hi = n;
  while (lo < hi) {
    uint32_t mid = (lo + hi) >> 1;
    if (a[mid] < x) lo = mid + 1; else hi = mid;
  }
  return lo < n && a[lo] == x;
}

// Index of x in the ascending list a[0..n) (x must be present).
__device__ __forceinline__ uint32_t sorted_index(const uint32_t* __restrict__ a, uint32_t n, uint32_t x) {
  uint32_t lo = 0, hi = n;
  while (lo < hi) {
    uint32_t mid = (lo + hi) >> 1;
    if (a[mid] < x) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// MurmurHash2 of one 4-byte key (the published algorithm for len == 4; the
// reference's device copy is match/GSI_kernels.cuh:61-93).
__device__ __forceinline__ uint32_t murmur2_u32(uint32_t key, uint32_t seed) {
  const uint32_t mul = 0x5bd1e995u;
  uint32_t h = seed ^ 4u;
  uint32_t w = key * mul;
  w ^= w >> 24;
  w *= mul;
  h = (h * mul) ^ w;
  h ^= h >> 13;
  h *= mul;
  h ^= h >> 15;
  return h;
}

// Order-independent digest of an embedding set.  A row (data vertex ids in
// query-vertex order) hashes to x by chaining the splitmix64 finaliser
// (Steele, Lea and Flood; public domain) over its words; the set's digest is
// the pair (sum of x, sum of mix64(x ^ kDigestSalt)) modulo 2^64, which does
// not depend on the order rows are produced in.
constexpr uint64_t kDigestSalt = 0xd6e8feb86659fd93ull;

__host__ __device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

__host__ __device__ __forceinline__ uint64_t row_hash_start(uint32_t k) {
  return 0x9e3779b97f4a7c15ull * (uint64_t)(k + 1);
}

__host__ __device__ __forceinline__ uint64_t row_hash_step(uint64_t x, uint32_t i, uint32_t v) {
  return mix64(x + (uint64_t)v + ((uint64_t)i << 32));
}

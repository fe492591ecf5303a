// block_sort.hpp - stable radix ranking by waves, and sorts and scans of one 1024-thread workgroup
// over items held in registers (shared by the device-wide sorts and the one-workgroup stages).
//
// Layout: a thread holds IT items; item r of lane l of wave w is at position
// w * 64 * IT + 64 * r + l (block_pos), so a wave's items are consecutive.
#pragma once

#include "common.hpp"

namespace hgp {

// Ranking.  A wave owns consecutive keys, 64 per round; lanes with equal digits find each other
// with one ballot per digit bit, the lowest of them adds the group to the wave's own counter of
// that digit, and a key's rank is the counter before its group plus its place in it.  The
// counters belong to the wave (LDS operations of a wave are in order), so rounds need no barrier.
// Returns the rank among the wave's keys of the same digit so far.
__device__ __forceinline__ uint32_t wave_digit_rank(bool valid, uint32_t d, int nb, uint32_t* cnt) {
  uint64_t peers = __ballot(valid);
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    if (b < nb) {  // uniform
      const bool bit = (d >> b) & 1u;
      const uint64_t bb = __ballot(bit);
      peers &= bit ? bb : ~bb;
    }
  }
  const uint32_t below = lanes_below(peers);
  uint32_t before = 0;
  if (valid) before = cnt[d];
  __builtin_amdgcn_wave_barrier();
  if (valid && below == 0) cnt[d] = before + (uint32_t)__popcll(peers);
  __builtin_amdgcn_wave_barrier();
  return before + below;
}

constexpr uint32_t BLOCK_SORT_THREADS = 1024;
constexpr uint32_t BLOCK_SORT_WAVES = BLOCK_SORT_THREADS / 64;

template <typename K, uint32_t IT>
struct BlockSortMem {
  K key[BLOCK_SORT_THREADS * IT];  // after block_sort: the sorted keys (without values)
  uint32_t cnt[BLOCK_SORT_WAVES][256];
  uint32_t w[BLOCK_SORT_WAVES];
};

template <uint32_t IT>
__device__ __forceinline__ uint32_t block_pos(uint32_t r) {
  return (threadIdx.x / 64) * 64 * IT + 64 * r + lane_id();
}

// Sorts the n items by bits [lo, bits) of key - kmin, in digits of nb bits (at most 8): items stay
// in registers, every pass ranks them and exchanges them through LDS.  Every thread calls it.
template <typename K, bool HAS_VALS, uint32_t IT>
__device__ __forceinline__ void block_sort(K (&key)[IT], uint32_t (&val)[IT], uint32_t n, int lo, int bits, int nb, K kmin,
                                           BlockSortMem<K, IT>& s) {
  constexpr uint32_t W = BLOCK_SORT_WAVES;
  const uint32_t t = threadIdx.x, w = t / 64, l = lane_id();
  const uint32_t first = block_pos<IT>(0);
  for (int shift = lo; shift < bits; shift += nb) {
    const int nbp = min(nb, bits - shift);
    const uint32_t mask = (1u << nbp) - 1u;
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) (&s.cnt[0][0])[q * BLOCK_SORT_THREADS + t] = 0;
    __syncthreads();
    uint32_t pos[IT];
#pragma unroll
    for (uint32_t r = 0; r < IT; ++r) {
      const uint32_t d = (uint32_t)((key[r] - kmin) >> shift) & mask;
      pos[r] = wave_digit_rank(first + 64 * r < n, d, nbp, s.cnt[w]);
    }
    __syncthreads();
    // exclusive sums in (digit, wave) order: thread t takes four waves of digit t / 4
    uint32_t c[4], sum = 0;
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
      c[q] = s.cnt[(t & 3) * 4 + q][t >> 2];
      sum += c[q];
    }
    const uint32_t inc = wave_scan_incl(sum);
    if (l == 63) s.w[w] = inc;
    __syncthreads();
    uint32_t run = inc - sum;
#pragma unroll
    for (uint32_t q = 0; q < W; ++q) run += q < w ? s.w[q] : 0u;
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
      s.cnt[(t & 3) * 4 + q][t >> 2] = run;
      run += c[q];
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < IT; ++r) {
      const uint32_t d = (uint32_t)((key[r] - kmin) >> shift) & mask;
      pos[r] += s.cnt[w][d];
      if (first + 64 * r < n) s.key[pos[r]] = key[r];
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < IT; ++r)
      if (first + 64 * r < n) key[r] = s.key[first + 64 * r];
    if (HAS_VALS) {  // the values take the keys' place in LDS
      uint32_t* s_val = reinterpret_cast<uint32_t*>(s.key);
      __syncthreads();
#pragma unroll
      for (uint32_t r = 0; r < IT; ++r)
        if (first + 64 * r < n) s_val[pos[r]] = val[r];
      __syncthreads();
#pragma unroll
      for (uint32_t r = 0; r < IT; ++r)
        if (first + 64 * r < n) val[r] = s_val[first + 64 * r];
    }
    __syncthreads();
  }
}

// Digits of a sort's bits shared evenly over its passes.
__device__ __forceinline__ int digit_bits(int bits) {
  const int passes = (bits + 7) / 8;
  return passes ? (bits + passes - 1) / passes : 8;
}

// Inclusive prefix sums over the positions, in place.  Every thread calls it; s: one entry a wave.
template <typename T, uint32_t IT>
__device__ __forceinline__ void block_scan(T (&x)[IT], T* s) {
  const uint32_t w = threadIdx.x / 64;
  T carry = 0;
#pragma unroll
  for (uint32_t r = 0; r < IT; ++r) {
    const T inc = wave_scan_incl(x[r]);
    x[r] = inc + carry;
    carry += lane_value(inc, 63);
  }
  if (lane_id() == 0) s[w] = carry;
  __syncthreads();
  T base = 0;
#pragma unroll
  for (uint32_t q = 0; q < BLOCK_SORT_WAVES; ++q) base += q < w ? s[q] : (T)0;
#pragma unroll
  for (uint32_t r = 0; r < IT; ++r) x[r] += base;
  __syncthreads();
}

// head[r] = the last position at or before item r's whose flag is set (position 0 must be).  s: one
// entry a wave.  Every thread calls it.
template <uint32_t IT>
__device__ __forceinline__ void block_last_head(const bool (&flag)[IT], uint32_t (&head)[IT], uint32_t* s) {
  const uint32_t w = threadIdx.x / 64, l = lane_id();
  uint32_t last = 0xFFFFFFFFu;  // of the wave so far
#pragma unroll
  for (uint32_t r = 0; r < IT; ++r) {
    const uint64_t m = __ballot(flag[r]);
    const uint64_t upto = m & (l == 63 ? ~0ull : (2ull << l) - 1ull);
    const uint32_t row = w * 64 * IT + 64 * r;
    head[r] = upto ? row + 63u - (uint32_t)__clzll((long long)upto) : last;
    if (m) last = row + 63u - (uint32_t)__clzll((long long)m);
  }
  if (l == 0) s[w] = last;
  __syncthreads();
  uint32_t before = 0;
#pragma unroll
  for (uint32_t q = 0; q < BLOCK_SORT_WAVES; ++q) before = q < w && s[q] != 0xFFFFFFFFu ? s[q] : before;
#pragma unroll
  for (uint32_t r = 0; r < IT; ++r) head[r] = head[r] == 0xFFFFFFFFu ? before : head[r];
  __syncthreads();
}

}  // namespace hgp

// pin_tile.hpp - the hedge of every pin, by tiles of pins (a workgroup of 1024 threads each).
#pragma once

#include "block_sort.hpp"

namespace hgp {

// Hedges of pins.  A workgroup owns a tile of consecutive pins, finds the hedges that meet it by a
// search of the offsets in 64 steps at once, marks the pins where hedges start, and gives every pin
// the last mark at or before it: pins are read and keys written in full lines, and a long hedge is
// shared by as many workgroups as it has tiles.  (A thread per hedge writes with the stride of the
// hedges' lengths, and the longest hedge is one thread's serial work.)  The kernel is bound by its
// reads and writes: at 3.2M pins of 800k nodes' hedges 169 -> 18 us (k_touch_keys) and 290 -> 33 us
// (k_chedge_keys, which reads a group per pin).  Up to 256k pins a thread takes one pin, so that
// small levels spread over the chip; above, four.
template <uint32_t IT>
struct PinTile {
  uint32_t mark[BLOCK_SORT_THREADS * IT];
  uint32_t w[BLOCK_SORT_WAVES];
  uint32_t first, end;
};

// number of the m ascending entries that are <= key; every lane of the wave calls it
__device__ __forceinline__ uint32_t wave_upper_bound(const uint64_t* __restrict__ x, uint32_t m, uint64_t key) {
  uint32_t lo = 0, hi = m;  // entries below lo are <= key, those from hi on are not
  while (hi - lo > 64) {
    const uint32_t step = (hi - lo) / 64;
    const uint32_t c = (uint32_t)__popcll(__ballot(x[lo + lane_id() * step] <= key));
    if (c == 0) return lo;
    if (c < 64) hi = lo + c * step;
    lo += (c - 1) * step + 1;
  }
  return lo + (uint32_t)__popcll(__ballot(lo + lane_id() < hi && x[lo + lane_id()] <= key));
}

// hedge[r], in_hedge[r]: the hedge of pin block_pos<IT>(r) of the tile at `base`, and the pin's place
// in it.  Pins from p on get none.  Every thread calls it.
template <uint32_t IT>
__device__ __forceinline__ void pin_hedges(const uint64_t* __restrict__ hoff, uint32_t E, uint64_t p, uint64_t base,
                                           uint32_t (&hedge)[IT], uint64_t (&in_hedge)[IT], PinTile<IT>& s) {
  constexpr uint32_t T = BLOCK_SORT_THREADS * IT;
  const uint32_t len = (uint32_t)min((uint64_t)T, p - base);
  if (threadIdx.x < 64) {
    const uint32_t c = wave_upper_bound(hoff, E, base);
    if (lane_id() == 0) s.first = c ? c - 1 : 0;
  } else if (threadIdx.x < 128) {
    const uint32_t c = wave_upper_bound(hoff, E, base + len - 1);
    if (lane_id() == 0) s.end = c;
  }
#pragma unroll
  for (uint32_t r = 0; r < IT; ++r) s.mark[threadIdx.x + BLOCK_SORT_THREADS * r] = NONE;
  __syncthreads();
  const uint32_t h0 = s.first, h1 = s.end;
  for (uint32_t h = h0 + threadIdx.x; h < h1; h += BLOCK_SORT_THREADS) {
    const uint64_t a = hoff[h], b = hoff[h + 1];
    if (b > a && b > base) s.mark[a > base ? a - base : 0] = h;  // hedges without pins start nowhere
  }
  __syncthreads();
  bool flag[IT];
  uint32_t head[IT];
#pragma unroll
  for (uint32_t r = 0; r < IT; ++r) flag[r] = s.mark[block_pos<IT>(r)] != NONE;
  block_last_head(flag, head, s.w);
  const uint64_t before = base - hoff[h0];  // pins of the first hedge in earlier tiles
#pragma unroll
  for (uint32_t r = 0; r < IT; ++r) {
    const uint32_t i = block_pos<IT>(r);
    hedge[r] = i < len && head[r] != NONE ? s.mark[head[r]] : NONE;
    in_hedge[r] = i - head[r] + (head[r] == 0 ? before : 0);
  }
}

// f(items, tiles): pins per thread (a compile-time constant) and the number of tiles of p pins
template <typename F>
void with_pin_tiles(uint64_t p, F f) {
  if (p <= 256ull * BLOCK_SORT_THREADS)
    f(std::integral_constant<uint32_t, 1>{}, ceil_div(p, BLOCK_SORT_THREADS));
  else
    f(std::integral_constant<uint32_t, 4>{}, ceil_div(p, 4ull * BLOCK_SORT_THREADS));
}

}  // namespace hgp

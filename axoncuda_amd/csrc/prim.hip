// prim.hip - scans, stable radix sort and small helpers for gfx950 (wave64).
//
// Scans: one pass with decoupled look-back over 4096-element tiles.
// Radix sort: LSD with digits of up to 8 bits; up to 8,192 keys in one workgroup's registers and
// LDS, larger ones in tiles (counts, offsets, scatter) per pass.
#include <algorithm>
#include <type_traits>

#include "block_sort.hpp"
#include "prim.hpp"

namespace hgp {

namespace {

// Single-pass scan with decoupled look-back.  A workgroup takes the next tile number from a
// ticket counter (so every tile it waits for belongs to a workgroup that is already running),
// scans its 4096 elements, publishes its aggregate, then walks back over the predecessors'
// published aggregates / inclusive prefixes until it meets an inclusive one.  Flags carry a
// per-scan generation, so the status arrays are reused without clearing.
constexpr int SCAN_BLOCK = 256;
constexpr int SCAN_ITEMS = 16;
constexpr int SCAN_TILE = SCAN_BLOCK * SCAN_ITEMS;

template <typename TI, typename TO, bool EXCL>
__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_lookback(const TI* in, TO* out, uint64_t n, uint32_t tiles,
                                                              uint32_t* flags, TO* agg, TO* incl,
                                                              unsigned long long* ticket, uint64_t base,
                                                              uint32_t gen) {
  __shared__ uint32_t s_tile;
  __shared__ TO s_wave[SCAN_BLOCK / 64];
  __shared__ TO s_prefix;
  if (threadIdx.x == 0) s_tile = (uint32_t)(atomicAdd(ticket, 1ull) - base);
  __syncthreads();
  const uint32_t tile = s_tile;
  const uint32_t w = threadIdx.x / 64, l = lane_id();
  const uint64_t start = (uint64_t)tile * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
  TO v[SCAN_ITEMS];
  TO sum = 0;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    const uint64_t i = start + k;
    v[k] = i < n ? (TO)in[i] : (TO)0;
    sum += v[k];
  }
  const TO winc = wave_scan_incl(sum);
  if (l == 63) s_wave[w] = winc;
  __syncthreads();
  TO wbase = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < SCAN_BLOCK / 64; ++i) {
    const TO x = s_wave[i];
    if (i < (int)w) wbase += x;
    tot += x;
  }
  const TO texcl = wbase + winc - sum;
  // look-back by wave 0: each round examines the 64 preceding tiles at once
  if (w == 0) {
    const uint32_t g = gen << 2;
    TO prefix = 0;
    if (tile == 0) {
      if (l == 0) {
        incl[0] = tot;
        __hip_atomic_store(&flags[0], g | 2u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
      }
    } else {
      if (l == 0) {
        agg[tile] = tot;
        __hip_atomic_store(&flags[tile], g | 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
      }
      int64_t hi = (int64_t)tile - 1;  // window [hi - 63, hi]; lane l looks at tile hi - l
      for (;;) {
        const int64_t j = hi - (int64_t)l;
        uint32_t st = 2u;  // tiles before 0 act as an inclusive zero
        if (j >= 0) {
          const uint32_t f = __hip_atomic_load(&flags[j], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
          st = (f & ~3u) == g ? (f & 3u) : 0u;
        }
        const uint64_t incl_mask = __ballot(st == 2u);
        const uint64_t zero_mask = __ballot(st == 0u);
        // nearest inclusive tile (lowest lane with st == 2); every lane before it must be published
        const uint32_t first_incl = incl_mask ? (uint32_t)__ffsll((unsigned long long)incl_mask) - 1u : 64u;
        const uint64_t before = first_incl >= 64 ? ~0ull : ((1ull << first_incl) - 1ull);
        if (zero_mask & before) {
          __builtin_amdgcn_s_sleep(1);
          continue;
        }
        TO part = 0;
        if (l < first_incl && j >= 0) part = agg[j];
        if (l == first_incl && j >= 0) part = incl[j];
        prefix += wave_sum(part);
        if (first_incl < 64) break;
        hi -= 64;
      }
      if (l == 0) {
        incl[tile] = prefix + tot;
        __hip_atomic_store(&flags[tile], g | 2u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    if (l == 0) {
      s_prefix = prefix;
      if (EXCL && tile == tiles - 1) out[n] = prefix + tot;
    }
  }
  __syncthreads();
  TO run = s_prefix + texcl;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    const uint64_t i = start + k;
    if (EXCL) {
      if (i < n) out[i] = run;
      run += v[k];
    } else {
      run += v[k];
      if (i < n) out[i] = run;
    }
  }
}

// Three-pass scan for large inputs (tile reduce, scan of tile sums, tile scan): at thousands
// of tiles the decoupled look-back's chain of publications is slower than two extra passes.
constexpr int RS3_ITEMS = 8;
constexpr int RS3_TILE = SCAN_BLOCK * RS3_ITEMS;

template <typename T>
__device__ __forceinline__ T block_excl_scan(T v, T* lds_waves, T* total) {
  // lds_waves: SCAN_BLOCK/64 entries
  const uint32_t w = threadIdx.x / 64, l = lane_id();
  T incl = wave_scan_incl(v);
  if (l == 63) lds_waves[w] = incl;
  __syncthreads();
  T base = 0, tot = 0;
  for (uint32_t i = 0; i < blockDim.x / 64; ++i) {
    T x = lds_waves[i];
    if (i < w) base += x;
    tot += x;
  }
  *total = tot;
  __syncthreads();
  return base + incl - v;
}

template <typename TI, typename TO>
__global__ void k_tile_reduce(const TI* __restrict__ in, uint64_t n, TO* __restrict__ partial) {
  __shared__ TO sw[SCAN_BLOCK / 64];
  uint64_t base = (uint64_t)blockIdx.x * RS3_TILE;
  TO s = 0;
  for (int k = 0; k < RS3_ITEMS; ++k) {
    uint64_t i = base + (uint64_t)k * SCAN_BLOCK + threadIdx.x;
    if (i < n) s += (TO)in[i];
  }
  s = wave_sum(s);
  if (lane_id() == 0) sw[threadIdx.x / 64] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    TO t = 0;
    for (int i = 0; i < SCAN_BLOCK / 64; ++i) t += sw[i];
    partial[blockIdx.x] = t;
  }
}

// exclusive scan of partial[0..m) in place by one workgroup; partial[m] = total
template <typename TO>
__global__ void k_scan_partials(TO* partial, uint32_t m) {
  __shared__ TO sw[1024 / 64];
  __shared__ TO carry_s;
  if (threadIdx.x == 0) carry_s = 0;
  __syncthreads();
  for (uint32_t base = 0; base < m; base += blockDim.x) {
    uint32_t i = base + threadIdx.x;
    TO v = i < m ? partial[i] : 0;
    TO tot;
    TO ex = block_excl_scan(v, sw, &tot);
    TO carry = carry_s;
    if (i < m) partial[i] = carry + ex;
    __syncthreads();
    if (threadIdx.x == 0) carry_s = carry + tot;
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[m] = carry_s;
}

// Also stores the total at out[n] (block 0): the partials' scan left it at partial[gridDim.x].
template <typename TI, typename TO>
__global__ void k_tile_scan_excl(const TI* in, TO* out, uint64_t n, const TO* __restrict__ partial) {
  __shared__ TO sw[SCAN_BLOCK / 64];
  if (blockIdx.x == 0 && threadIdx.x == 0) out[n] = partial[gridDim.x];
  uint64_t base = (uint64_t)blockIdx.x * RS3_TILE + (uint64_t)threadIdx.x * RS3_ITEMS;
  TO v[RS3_ITEMS];
  TO s = 0;
#pragma unroll
  for (int k = 0; k < RS3_ITEMS; ++k) {
    uint64_t i = base + k;
    v[k] = i < n ? (TO)in[i] : (TO)0;
    s += v[k];
  }
  TO tot;
  TO ex = block_excl_scan(s, sw, &tot) + partial[blockIdx.x];
#pragma unroll
  for (int k = 0; k < RS3_ITEMS; ++k) {
    uint64_t i = base + k;
    if (i < n) out[i] = ex;
    ex += v[k];
  }
}

template <typename TI, typename TO>
__global__ void k_tile_scan_incl(const TI* in, TO* out, uint64_t n, const TO* __restrict__ partial) {
  __shared__ TO sw[SCAN_BLOCK / 64];
  uint64_t base = (uint64_t)blockIdx.x * RS3_TILE + (uint64_t)threadIdx.x * RS3_ITEMS;
  TO v[RS3_ITEMS];
  TO s = 0;
#pragma unroll
  for (int k = 0; k < RS3_ITEMS; ++k) {
    uint64_t i = base + k;
    v[k] = i < n ? (TO)in[i] : (TO)0;
    s += v[k];
  }
  TO tot;
  TO ex = block_excl_scan(s, sw, &tot) + partial[blockIdx.x];
#pragma unroll
  for (int k = 0; k < RS3_ITEMS; ++k) {
    uint64_t i = base + k;
    ex += v[k];
    if (i < n) out[i] = ex;
  }
}


// Status arrays of the context's scans (one stream: scans never overlap).
void scan_status(Ctx& c, uint32_t tiles) {
  if (tiles <= c.scan_cap_tiles && c.scan_ticket) return;
  uint32_t cap = 1024;
  while (cap < tiles) cap <<= 1;
  if (c.scan_flags) {
    dfree(c, c.scan_flags);
    dfree(c, c.scan_agg);
    dfree(c, c.scan_incl);
  }
  c.scan_flags = (uint32_t*)dmalloc(c, (uint64_t)cap * 4);
  c.scan_agg = dmalloc(c, (uint64_t)cap * 8);
  c.scan_incl = dmalloc(c, (uint64_t)cap * 8);
  memset_async(c, c.scan_flags, 0, (uint64_t)cap * 4);  // generation 0 is never used
  if (!c.scan_ticket) {
    c.scan_ticket = (unsigned long long*)dmalloc(c, 8);
    memset_async(c, c.scan_ticket, 0, 8);
    c.scan_tickets_issued = 0;
  }
  c.scan_cap_tiles = cap;
}

// in == out is safe: each workgroup reads only its own tile before writing it.
template <typename TI, typename TO>
void scan_impl(Ctx& c, const TI* in, TO* out, uint64_t n, bool exclusive) {
  if (n == 0) {
    if (exclusive) memset_async(c, out, 0, sizeof(TO));
    return;
  }
  const uint32_t tiles = ceil_div(n, SCAN_TILE);
  if (tiles > c.tune.scan_lookback_tiles) {  // default 64 (the autotuner may move it)
    const uint32_t t3 = ceil_div(n, RS3_TILE);
    DBuf<TO> partial(c, (uint64_t)t3 + 1);
    HGP_LAUNCH((k_tile_reduce<TI, TO>), t3, SCAN_BLOCK, 0, c, in, n, partial.get());
    HGP_LAUNCH((k_scan_partials<TO>), 1, 1024, 0, c, partial.get(), t3);
    if (exclusive) {
      HGP_LAUNCH((k_tile_scan_excl<TI, TO>), t3, SCAN_BLOCK, 0, c, in, out, n, partial.get());
    } else {
      HGP_LAUNCH((k_tile_scan_incl<TI, TO>), t3, SCAN_BLOCK, 0, c, in, out, n, partial.get());
    }
    return;
  }
  scan_status(c, tiles);
  c.scan_gen = (c.scan_gen + 1) & 0x3FFFFFFFu;
  if (c.scan_gen == 0) c.scan_gen = 1;
  const uint64_t base = c.scan_tickets_issued;
  c.scan_tickets_issued += tiles;
  if (exclusive)
    HGP_LAUNCH((k_scan_lookback<TI, TO, true>), tiles, SCAN_BLOCK, 0, c, in, out, n, tiles, c.scan_flags,
               (TO*)c.scan_agg, (TO*)c.scan_incl, c.scan_ticket, base, c.scan_gen);
  else
    HGP_LAUNCH((k_scan_lookback<TI, TO, false>), tiles, SCAN_BLOCK, 0, c, in, out, n, tiles, c.scan_flags,
               (TO*)c.scan_agg, (TO*)c.scan_incl, c.scan_ticket, base, c.scan_gen);
}

// ---------------------------------------------------------------------------------------
// radix sort (stable, least significant digit first; digits of at most 8 bits, the passes of a
// sort sharing its bits evenly)
constexpr int RS_BLOCK = 256;

// Whole sort of at most 1024 * IT keys by one workgroup: keys and values stay in registers, every
// pass ranks them and exchanges them through LDS, and memory is read and written once.  The
// exchange through global memory this replaces cost 64 cycles per scattered 64-lane store: two
// passes over 8,191 64-bit keys with values took 37 us and take 20 us this way, 4,096 keys 25 and
// 13 us, 64 keys 14 and 7.5 us.  Past 8,192 keys one CU's ranking is the bound (16,384 keys: 38 us)
// and the tiles below are faster (16,385 keys: 18 us).
constexpr uint32_t RS1_BLOCK = BLOCK_SORT_THREADS;
constexpr uint32_t RS1_MAX_IT = 8;
constexpr uint64_t RS1_MAX_N = (uint64_t)RS1_BLOCK * RS1_MAX_IT;

template <typename K, bool HAS_VALS, uint32_t IT>
__global__ void __launch_bounds__(RS1_BLOCK) k_rs_block(K* keys, uint32_t* vals, uint32_t n, int lo, int bits, int nb,
                                                        K kmin) {
  __shared__ BlockSortMem<K, IT> s;
  K key[IT];
  uint32_t val[IT];
#pragma unroll
  for (uint32_t r = 0; r < IT; ++r) {
    const uint32_t i = block_pos<IT>(r);
    key[r] = i < n ? keys[i] : (K)0;
    val[r] = HAS_VALS && i < n ? vals[i] : 0u;
  }
  block_sort<K, HAS_VALS, IT>(key, val, n, lo, bits, nb, kmin, s);
#pragma unroll
  for (uint32_t r = 0; r < IT; ++r) {
    const uint32_t i = block_pos<IT>(r);
    if (i < n) {
      keys[i] = key[r];
      if (HAS_VALS) vals[i] = val[r];
    }
  }
}

// Larger sorts, per pass: every tile of 512 * IT keys counts its digits; the tiles' counts become
// the number of equal digits in the tiles before (and the digits' totals); every tile ranks its
// keys again, exchanges them through LDS into digit order and writes runs.  Up to RS_DIRECT_TILES
// tiles the last step adds up the earlier tiles' counts itself, and a pass is two launches.  Two
// passes over 64-bit keys with values, against a scan of all counts and a scatter in rounds of 256
// keys: 65,536 keys 72 -> 21 us, 1,000,000 68 -> 44 us, 15.4 M 630 -> 302 us.  No workgroup waits
// for another: a single-pass look-back over the tiles, numbered by a ticket so that its waits end,
// was measured too, and the tickets (one address, about 40 ns each) bounded it above 100 tiles
// (15.4 M keys: 370 us; 1,000,000: 62 us).
constexpr uint32_t OS_BLOCK = 512;
constexpr uint32_t RS_DIRECT_TILES = 64;

// LDS add to a digit counter; when the whole wave has one digit (the high digits of small values)
// one lane adds for all instead of 64 adds to one address
__device__ __forceinline__ void count_digit(uint32_t* h, bool valid, uint32_t d) {
  const uint64_t act = __ballot(valid);
  if (!act) return;
  const int lead = __ffsll((unsigned long long)act) - 1;
  const uint32_t d0 = (uint32_t)__builtin_amdgcn_readlane((int)d, lead);
  if (__ballot(valid && d == d0) == act) {
    if ((int)lane_id() == lead) atomicAdd(&h[d0], (uint32_t)__popcll(act));
  } else if (valid) {
    atomicAdd(&h[d], 1u);
  }
}
// counts[tile][digit]
template <typename K, uint32_t IT>
__global__ void __launch_bounds__(OS_BLOCK) k_rs_count(const K* __restrict__ keys, uint64_t n, int shift, int nb, K kmin,
                                                       uint32_t* __restrict__ counts) {
  __shared__ uint32_t h[256];
  const uint32_t t = threadIdx.x, mask = (1u << nb) - 1u;
  if (t < 256) h[t] = 0;
  const uint64_t beg = (uint64_t)blockIdx.x * (OS_BLOCK * IT);
  K key[IT];
#pragma unroll
  for (uint32_t r = 0; r < IT; ++r) {
    const uint64_t i = beg + r * OS_BLOCK + t;
    key[r] = i < n ? keys[i] - kmin : (K)0;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < IT; ++r) count_digit(h, beg + r * OS_BLOCK + t < n, (uint32_t)(key[r] >> shift) & mask);
  __syncthreads();
  if (t < 256) counts[(uint64_t)blockIdx.x * 256 + t] = h[t];
}

// before[tile][digit] = the counts of the digit in the tiles before; totals[digit].  One workgroup
// per 16 digits: 64 segments of consecutive tiles, summed, scanned and walked again.
__global__ void __launch_bounds__(1024) k_rs_columns(const uint32_t* __restrict__ counts, uint32_t tiles,
                                                     uint64_t* __restrict__ before, uint64_t* __restrict__ totals) {
  __shared__ uint64_t s_seg[64][16];
  const uint32_t x = threadIdx.x & 15, seg = threadIdx.x >> 4, d = blockIdx.x * 16 + x;
  const uint32_t per = (tiles + 63) / 64;
  const uint32_t b = min(tiles, seg * per), e = min(tiles, b + per);
  uint64_t sum = 0;
#pragma unroll 8
  for (uint32_t i = b; i < e; ++i) sum += counts[(uint64_t)i * 256 + d];
  s_seg[seg][x] = sum;
  __syncthreads();
  // a wave holds 4 segments of 16 digits: each of the first 16 threads scans one digit's segments
  if (threadIdx.x < 16) {
    uint64_t run = 0;
    for (uint32_t q = 0; q < 64; ++q) {
      const uint64_t v = s_seg[q][threadIdx.x];
      s_seg[q][threadIdx.x] = run;
      run += v;
    }
    totals[d] = run;
  }
  __syncthreads();
  uint64_t run = s_seg[seg][x];
#pragma unroll 8
  for (uint32_t i = b; i < e; ++i) {
    const uint32_t v = counts[(uint64_t)i * 256 + d];
    before[(uint64_t)i * 256 + d] = run;
    run += v;
  }
}

// before == nullptr: at most RS_DIRECT_TILES tiles, whose counts are added up here
template <typename K, bool HAS_VALS, uint32_t IT>
__global__ void __launch_bounds__(OS_BLOCK) k_rs_pass(const K* __restrict__ keys, const uint32_t* __restrict__ vals,
                                                      K* __restrict__ okeys, uint32_t* __restrict__ ovals, uint64_t n,
                                                      int shift, int nb, K kmin, const uint32_t* __restrict__ counts,
                                                      const uint64_t* __restrict__ before,
                                                      const uint64_t* __restrict__ totals) {
  constexpr uint32_t W = OS_BLOCK / 64, TILE = OS_BLOCK * IT, WD = 256 / 64, HALVES = OS_BLOCK / 256;
  __shared__ K s_key[TILE];
  __shared__ uint32_t s_val[HAS_VALS ? TILE : 1];
  __shared__ uint32_t s_cnt[W][256];
  __shared__ uint32_t s_loc[256];
  __shared__ uint64_t s_base[256];
  __shared__ uint32_t s_w[WD];
  __shared__ uint64_t s_g[WD];
  __shared__ uint32_t s_sum[HALVES][2][256];
  const uint32_t t = threadIdx.x, w = t / 64, l = lane_id();
  const uint32_t mask = (1u << nb) - 1u;
  const uint32_t tile = blockIdx.x;
  const uint64_t beg = (uint64_t)tile * TILE;
  const uint32_t len = (uint32_t)min((uint64_t)TILE, n - beg);
  const uint32_t first = w * 64 * IT + l;
  K key[IT];
  uint32_t val[IT], pos[IT];
#pragma unroll
  for (uint32_t r = 0; r < IT; ++r) {
    const uint32_t i = first + 64 * r;
    key[r] = i < len ? keys[beg + i] : (K)0;
    val[r] = HAS_VALS && i < len ? vals[beg + i] : 0u;
  }
#pragma unroll
  for (uint32_t q = 0; q < W * 256 / OS_BLOCK; ++q) (&s_cnt[0][0])[q * OS_BLOCK + t] = 0;
  // per digit: keys of it in the tiles before, and in all
  uint64_t g = 0, bef = 0;
  if (before) {
    if (t < 256) {
      g = totals[t];
      bef = before[(uint64_t)tile * 256 + t];
    }
  } else {
    const uint32_t d = t & 255, half = t >> 8;
    uint32_t a = 0, b = 0;
#pragma unroll 8
    for (uint32_t i = half; i < gridDim.x; i += HALVES) {
      const uint32_t v = counts[i * 256 + d];
      a += v;
      b += i < tile ? v : 0u;
    }
    s_sum[half][0][d] = a;
    s_sum[half][1][d] = b;
  }
  __syncthreads();
  if (!before && t < 256) {
#pragma unroll
    for (uint32_t h = 0; h < HALVES; ++h) {
      g += s_sum[h][0][t];
      bef += s_sum[h][1][t];
    }
  }
  uint64_t ginc = 0;
  if (t < 256) {
    ginc = wave_scan_incl(g);
    if (l == 63) s_g[w] = ginc;
  }
#pragma unroll
  for (uint32_t r = 0; r < IT; ++r)
    pos[r] = wave_digit_rank(first + 64 * r < len, (uint32_t)((key[r] - kmin) >> shift) & mask, nb, s_cnt[w]);
  __syncthreads();
  // digit t: its start in the tile, and each wave's start in it
  uint32_t tot = 0, inc = 0;
  if (t < 256) {
#pragma unroll
    for (uint32_t q = 0; q < W; ++q) {
      const uint32_t c = s_cnt[q][t];
      s_cnt[q][t] = tot;
      tot += c;
    }
    inc = wave_scan_incl(tot);
    if (l == 63) s_w[w] = inc;
  }
  __syncthreads();
  if (t < 256) {
    uint32_t loc = inc - tot;
    uint64_t below = ginc - g;
#pragma unroll
    for (uint32_t q = 0; q < WD; ++q) {
      loc += q < w ? s_w[q] : 0u;
      below += q < w ? s_g[q] : 0ull;
    }
    s_loc[t] = loc;
    s_base[t] = below + bef - loc;  // (wraps below zero and back with the tile position)
  }
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < IT; ++r) {
    if (first + 64 * r < len) {
      const uint32_t d = (uint32_t)((key[r] - kmin) >> shift) & mask;
      const uint32_t o = s_loc[d] + s_cnt[w][d] + pos[r];
      s_key[o] = key[r];
      if (HAS_VALS) s_val[o] = val[r];
    }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < IT; ++r) {
    const uint32_t i = r * OS_BLOCK + t;
    if (i < len) {
      const K k = s_key[i];
      const uint64_t o = s_base[(uint32_t)((k - kmin) >> shift) & mask] + i;
      okeys[o] = k;
      if (HAS_VALS) ovals[o] = s_val[i];
    }
  }
}

// Size of a pass's tiles in units of 256 keys (2, 4, 8 or 16): small tiles rank sooner, few tiles
// cost less to add up.  Measured (two passes, 32-bit keys with values, at 2 / 4 / 8 / 16): 50,000
// keys 23 / 20 / 24 / 29 us; 300,000 40 / 31 / 30 / 34; 1,000,000 71 / 47 / 42 / 41; 3.2 M 181 / 117 /
// 84 / 67.  The autotuner may set it per size class (floor(log2 n)); the result is the same.
inline uint32_t rs_items(const Ctx& c, uint64_t n) {
  const int cls = bit_width(n) - 1;
  uint32_t want = 0;
  if (cls >= 0 && cls < 40) want = c.tune.sort_rounds[cls];
  if (!want) want = n <= 65536 ? 4 : n <= 1u << 20 ? 8 : 16;
  uint32_t it = 2;
  while (it < want && it < 16) it <<= 1;
  return it;
}

// LSD passes over bits [lo, bits) of key - kmin (the keys themselves are moved unchanged).  With
// `kbuf` (and `vbuf`) the result ends up in those buffers by exchanging them with the scratch ones
// after an odd pass count; otherwise it is copied back into keys / vals.
template <typename K>
void radix_impl(Ctx& c, K* keys, uint32_t* vals, uint64_t n, int bits, int lo = 0, DBuf<K>* kbuf = nullptr,
                DBuf<uint32_t>* vbuf = nullptr, K kmin = 0) {
  if (n <= 1 || bits <= lo) return;
  const int passes = (bits - lo + 7) / 8;
  const int nb = (bits - lo + passes - 1) / passes;
  if (n <= RS1_MAX_N) {
    const uint64_t sb = n * (2 * sizeof(K) + (vals ? 8 : 0));  // keys (and values) read once and written once
    auto launch = [&](auto items) {
      constexpr uint32_t IT = decltype(items)::value;
      if (vals)
        HGP_LAUNCH_B(sb, (k_rs_block<K, true, IT>), 1, RS1_BLOCK, 0, c, keys, vals, (uint32_t)n, lo, bits, nb, kmin);
      else
        HGP_LAUNCH_B(sb, (k_rs_block<K, false, IT>), 1, RS1_BLOCK, 0, c, keys, vals, (uint32_t)n, lo, bits, nb, kmin);
    };
    if (n <= 1 * RS1_BLOCK) launch(std::integral_constant<uint32_t, 1>{});
    else if (n <= 2 * RS1_BLOCK) launch(std::integral_constant<uint32_t, 2>{});
    else if (n <= 4 * RS1_BLOCK) launch(std::integral_constant<uint32_t, 4>{});
    else launch(std::integral_constant<uint32_t, RS1_MAX_IT>{});
    return;
  }
  const uint32_t it = rs_items(c, n);
  const uint64_t tiles64 = (n + (uint64_t)RS_BLOCK * it - 1) / ((uint64_t)RS_BLOCK * it);
  HGP_REQUIRE(tiles64 < (1ull << 31), HGP_E_CAPACITY, "radix sort: too many tiles");
  const uint32_t tiles = (uint32_t)tiles64;
  const bool direct = tiles <= RS_DIRECT_TILES;
  DBuf<K> k2(c, n);
  DBuf<uint32_t> v2(c, vals ? n : 0);
  DBuf<uint32_t> counts(c, (uint64_t)tiles * 256);
  DBuf<uint64_t> before(c, direct ? 0 : ((uint64_t)tiles + 1) * 256);  // and the totals
  uint64_t* totals = direct ? nullptr : before.get() + (uint64_t)tiles * 256;
  K* ka = keys;
  K* kb = k2.get();
  uint32_t* va = vals;
  uint32_t* vb = v2.get();
  // bytes: keys (and values) read once and written once, one offset per (tile, digit) read
  const uint64_t sb = n * (2 * sizeof(K) + (vals ? 8 : 0)) + 2048ull * tiles;
  for (int shift = lo; shift < bits; shift += nb) {
    const int nbp = std::min(nb, bits - shift);
    auto launch = [&](auto items) {
      constexpr uint32_t IT = decltype(items)::value;
      // bytes: keys read once, one count per (tile, digit) written
      HGP_LAUNCH_B(n * sizeof(K) + 1024ull * tiles, (k_rs_count<K, IT>), tiles, OS_BLOCK, 0, c, ka, n, shift, nbp, kmin,
                   counts.get());
      if (!direct) HGP_LAUNCH(k_rs_columns, 16, 1024, 0, c, counts.get(), tiles, before.get(), totals);
      if (vals)
        HGP_LAUNCH_B(sb, (k_rs_pass<K, true, IT>), tiles, OS_BLOCK, 0, c, ka, va, kb, vb, n, shift, nbp, kmin,
                     counts.get(), before.get(), totals);
      else
        HGP_LAUNCH_B(sb, (k_rs_pass<K, false, IT>), tiles, OS_BLOCK, 0, c, ka, va, kb, vb, n, shift, nbp, kmin,
                     counts.get(), before.get(), totals);
    };
    if (it == 2) launch(std::integral_constant<uint32_t, 1>{});
    else if (it == 4) launch(std::integral_constant<uint32_t, 2>{});
    else if (it == 8) launch(std::integral_constant<uint32_t, 4>{});
    else launch(std::integral_constant<uint32_t, 8>{});
    std::swap(ka, kb);
    std::swap(va, vb);
  }
  if (ka != keys) {
    if (kbuf && (!vals || vbuf)) {  // hand the scratch buffers over instead of copying
      std::swap(*kbuf, k2);
      if (vals) std::swap(*vbuf, v2);
      return;
    }
    copy_d2d(c, keys, ka, n * sizeof(K));
    if (vals) copy_d2d(c, vals, va, n * sizeof(uint32_t));
  }
}

__global__ void k_minmax_u64(const uint64_t* __restrict__ p, uint64_t n, unsigned long long* out) {
  uint64_t mn = ~0ull, mx = 0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t v = p[i];
    mn = v < mn ? v : mn;
    mx = v > mx ? v : mx;
  }
  __shared__ uint64_t s_mn[4], s_mx[4];
  mn = wave_min(mn);
  mx = wave_max(mx);
  if (lane_id() == 0) {
    s_mn[threadIdx.x / 64] = mn;
    s_mx[threadIdx.x / 64] = mx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < 4; ++i) {
      mn = s_mn[i] < mn ? s_mn[i] : mn;
      mx = s_mx[i] > mx ? s_mx[i] : mx;
    }
    atomicMin(&out[0], (unsigned long long)mn);
    atomicMax(&out[1], (unsigned long long)mx);
  }
}
__global__ void k_init_minmax(unsigned long long* mm) {
  mm[0] = ~0ull;
  mm[1] = 0ull;
}

template <typename K>
__global__ void k_segment_offsets(const K* __restrict__ keys, int shift, uint64_t n, uint32_t nseg,
                                  uint64_t* __restrict__ off) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i > n) return;
  int64_t a = i == 0 ? -1 : (int64_t)(uint32_t)(keys[i - 1] >> shift);
  int64_t b = i == n ? (int64_t)nseg : (int64_t)(uint32_t)(keys[i] >> shift);
  if (b > (int64_t)nseg) b = nseg;
  for (int64_t s = a + 1; s <= b; ++s) off[s] = i;
}

__global__ void k_fill_u32(uint32_t* p, uint32_t v, uint64_t n) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
__global__ void k_iota_u32(uint32_t* p, uint64_t n) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = (uint32_t)i;
}
// One atomic per workgroup (8,192 of them, one per wave, on one address took 90 us for 500,000 values):
// 256 workgroups up to 16 M values, above that one for every 65,536, since 256 keep too few loads in
// flight for memory (connectivity of 150 M pins 4.4 ms with 2,048 workgroups, 5.1 with 256).
inline uint32_t max_grid(uint64_t n) {
  return (uint32_t)std::min<uint64_t>((n + 2047) / 2048, std::min<uint64_t>(std::max<uint64_t>(256, n >> 16), 2048));
}
template <typename T, typename A>
__global__ void __launch_bounds__(256) k_max(const T* __restrict__ p, uint64_t n, A* out) {
  __shared__ T s_m[4];
  constexpr uint32_t U = 8;  // loads in flight
  T m = 0;
  for (uint64_t b = (uint64_t)blockIdx.x * (256 * U) + threadIdx.x; b < n; b += (uint64_t)gridDim.x * (256 * U)) {
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      const T v = b + 256 * u < n ? p[b + 256 * u] : (T)0;
      m = v > m ? v : m;
    }
  }
  m = wave_max(m);
  if (lane_id() == 0) s_m[threadIdx.x / 64] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < 4; ++i) m = s_m[i] > m ? s_m[i] : m;
    atomicMax(out, (A)m);
  }
}

}  // namespace

void exclusive_scan(Ctx& c, const uint32_t* in, uint64_t* out, uint64_t n) { scan_impl<uint32_t, uint64_t>(c, in, out, n, true); }
void exclusive_scan(Ctx& c, const uint64_t* in, uint64_t* out, uint64_t n) { scan_impl<uint64_t, uint64_t>(c, in, out, n, true); }
void inclusive_scan(Ctx& c, const int64_t* in, int64_t* out, uint64_t n) { scan_impl<int64_t, int64_t>(c, in, out, n, false); }
void inclusive_scan(Ctx& c, const uint64_t* in, uint64_t* out, uint64_t n) { scan_impl<uint64_t, uint64_t>(c, in, out, n, false); }
void inclusive_scan(Ctx& c, const int32_t* in, int32_t* out, uint64_t n) { scan_impl<int32_t, int32_t>(c, in, out, n, false); }

void radix_sort(Ctx& c, uint32_t* keys, uint32_t* vals, uint64_t n, int bits) { radix_impl<uint32_t>(c, keys, vals, n, bits); }
void radix_sort(Ctx& c, uint64_t* keys, uint32_t* vals, uint64_t n, int bits) { radix_impl<uint64_t>(c, keys, vals, n, bits); }
void radix_sort_buf(Ctx& c, DBuf<uint32_t>& keys, DBuf<uint32_t>& vals, uint64_t n, int lo, int hi) {
  radix_impl<uint32_t>(c, keys.get(), vals.get(), n, hi, lo, &keys, &vals);
}
void radix_sort_buf(Ctx& c, DBuf<uint64_t>& keys, DBuf<uint32_t>& vals, uint64_t n, int lo, int hi) {
  radix_impl<uint64_t>(c, keys.get(), vals.get(), n, hi, lo, &keys, &vals);
}

void segment_offsets(Ctx& c, const uint32_t* keys, int shift, uint64_t n, uint32_t nseg, uint64_t* off) {
  HGP_LAUNCH((k_segment_offsets<uint32_t>), ceil_div(n + 1, 256), 256, 0, c, keys, shift, n, nseg, off);
}
void segment_offsets(Ctx& c, const uint64_t* keys, int shift, uint64_t n, uint32_t nseg, uint64_t* off) {
  HGP_LAUNCH((k_segment_offsets<uint64_t>), ceil_div(n + 1, 256), 256, 0, c, keys, shift, n, nseg, off);
}

void radix_sort_range(Ctx& c, uint64_t* keys, uint32_t* vals, uint64_t n) {
  if (n <= 1) return;
  DBuf<unsigned long long> mm(c, 2);
  HGP_LAUNCH(k_init_minmax, 1, 1, 0, c, mm.get());  // on the stream: no host-to-device copy
  HGP_LAUNCH(k_minmax_u64, std::min<uint32_t>(ceil_div(n, 256), 512), 256, 0, c, keys, n, mm.get());
  unsigned long long h[2];
  copy_d2h(c, h, mm.get(), sizeof h);
  if (h[1] == h[0]) return;  // all keys equal: a stable sort is the identity
  // digits of key - min: the passes cover only the keys' range
  radix_impl<uint64_t>(c, keys, vals, n, bit_width(h[1] - h[0]), 0, nullptr, nullptr, (uint64_t)h[0]);
}

Fork::Fork(Ctx& c, bool enabled) : c_(c), enabled_(enabled) {
  if (!enabled_) return;
  if (!c_.fork_ev) HGP_HIP(hipEventCreateWithFlags(&c_.fork_ev, hipEventDisableTiming));
  HGP_HIP(hipEventRecord(c_.fork_ev, c_.stream));
}
void Fork::start(int i) {
  HGP_REQUIRE(i >= 0 && i < Ctx::SIDES, HGP_E_INVALID, "Fork: no such side stream");
  if (used_ & (1u << i)) return;
  if (!c_.side[i]) {
    HGP_HIP(hipStreamCreateWithFlags(&c_.side[i], hipStreamNonBlocking));
    HGP_HIP(hipEventCreateWithFlags(&c_.side_ev[i], hipEventDisableTiming));
  }
  HGP_HIP(hipStreamWaitEvent(c_.side[i], c_.fork_ev, 0));
  used_ |= 1u << i;
}
Fork::~Fork() {
  // errors here have no caller to reach: a failed join leaves the stream unsynchronised,
  // which the context's next synchronisation reports
  for (int i = 0; i < Ctx::SIDES; ++i)
    if (used_ & (1u << i)) {
      (void)hipEventRecord(c_.side_ev[i], c_.side[i]);
      (void)hipStreamWaitEvent(c_.stream, c_.side_ev[i], 0);
    }
}
void destroy_sides(Ctx& c) {
  for (int i = 0; i < Ctx::SIDES; ++i) {
    if (c.side[i]) {
      (void)hipStreamSynchronize(c.side[i]);
      (void)hipStreamDestroy(c.side[i]);
      (void)hipEventDestroy(c.side_ev[i]);
      c.side[i] = nullptr;
      c.side_ev[i] = nullptr;
    }
  }
  if (c.fork_ev) (void)hipEventDestroy(c.fork_ev);
  c.fork_ev = nullptr;
}

void fill_u32(Ctx& c, uint32_t* p, uint32_t v, uint64_t n) { HGP_LAUNCH(k_fill_u32, ceil_div(n, 256), 256, 0, c, p, v, n); }
void iota_u32(Ctx& c, uint32_t* p, uint64_t n) { HGP_LAUNCH(k_iota_u32, ceil_div(n, 256), 256, 0, c, p, n); }
uint32_t reduce_max_u32(Ctx& c, const uint32_t* p, uint64_t n) {
  DBuf<uint32_t> out(c, 1);
  memset_async(c, out.get(), 0, sizeof(uint32_t));
  if (n) HGP_LAUNCH((k_max<uint32_t, uint32_t>), max_grid(n), 256, 0, c, p, n, out.get());
  return read_scalar(c, out.get());
}

uint64_t reduce_max_u64(Ctx& c, const uint64_t* p, uint64_t n) {
  DBuf<unsigned long long> out(c, 1);
  memset_async(c, out.get(), 0, sizeof(unsigned long long));
  if (n) HGP_LAUNCH((k_max<uint64_t, unsigned long long>), max_grid(n), 256, 0, c, p, n, out.get());
  return (uint64_t)read_scalar(c, out.get());
}

}  // namespace hgp

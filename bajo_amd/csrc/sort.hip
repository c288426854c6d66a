// Onesweep LSD radix sort for gfx950 (wave64).
//
// Replaces bajo/sort/gpu/onesweep.mojo (global_histogram :31-99, scan_global
// :102-118, digit_binning :121-327) and the reduce-then-scan sort of
// bajo/sort/gpu/radix_sort.mojo:510-609 with one engine:
//   1. one histogram pass computes the 256-bin digit histogram of every
//      pass at once (LDS histograms, one global atomic per bin and block; 4M
//      64-bit keys 32.4 -> 17.3 us with one block per CU instead of four);
//   2. one binning launch per 8-bit digit: a tile of 1,024 to 4,096 keys is
//      taken by ticket, counted and published to a decoupled look-back table,
//      ranked stably with wave64 ballot match masks, staged in LDS as
//      full-width keys (64-bit keys stay 64-bit; bajo's onesweep.mojo:244,311
//      staged u32) and written out in digit-contiguous runs.
// The global exclusive digit offsets are recomputed by every tile from the
// 256-bin histogram, so no separate scan launch is needed.
//
// What bounds a pass is a tile's serial chain, not its bytes: at 4M 64-bit
// keys all 1,024 tiles are resident at once.  Hence a tile publishes its
// counts before it ranks; looks back over the tiles of its group (8 or 16) and
// then over whole groups, each round's loads in flight together (tile by tile
// four at a time the chain grew to 22 rounds); and draws its ticket from one
// of eight counters (same-address atomics serialize).  With eight counters a
// predecessor may not have started (another stream's kernel can hold its XCD),
// so a tile waits for a bounded time and then counts the missing tiles itself:
// a sort ends whatever else runs on the chip.  A pass over 4M pairs
// (100 MB moved) took 50.9 us tile by tile and takes 32.4 (3.1 TB/s), over 4M
// keys 48.2 and 30.3.  Lists of at most 8,192 keys are sorted by one block in LDS, all
// passes in one launch (8,192 64-bit pairs: 109 -> 54 us).
#include <mutex>

#include "sort_internal.h"

namespace bj {

namespace {

template <typename K>
BJ_D uint32_t digit_of(K key, uint32_t shift) {
  return (uint32_t)(key >> shift) & 0xFFu;
}

// Exclusive scan of one value per thread over a 256-thread block.
BJ_D uint32_t block_exclusive_scan_256(uint32_t v, uint32_t* s_tmp, uint32_t* total) {
  const uint32_t lane = lane_id();
  const uint32_t wave = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    uint32_t y = __shfl_up(x, off, 64);
    if (lane >= (uint32_t)off) x += y;
  }
  if (lane == 63) s_tmp[wave] = x;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) {
    uint32_t t = s_tmp[w];
    before += (w < (int)wave) ? t : 0u;
    all += t;
  }
  __syncthreads();
  if (total) *total = all;
  return before + x - v;
}

__global__ void __launch_bounds__(256) sort_init_kernel(uint32_t* hist, uint32_t hist_words, uint32_t* tickets,
                                                        uint32_t ticket_words) {
  for (uint32_t i = threadIdx.x; i < hist_words; i += blockDim.x) hist[i] = 0;
  for (uint32_t i = threadIdx.x; i < ticket_words; i += blockDim.x) tickets[i] = 0;
}

// One block per CU: a block ends with one atomic per bin, so their number is
// kept small; four histograms per block keep the waves' LDS atomics apart.
constexpr int kHistBlock = 1024, kHistCopies = 4;
template <typename K>
__global__ void __launch_bounds__(kHistBlock) sort_hist_kernel(const K* __restrict__ keys, uint64_t n,
                                                               uint32_t begin_bit, uint32_t passes,
                                                               uint32_t* __restrict__ hist,
                                                               uint32_t* __restrict__ lookback,
                                                               uint64_t lookback_words) {
  __shared__ uint32_t s_hist[kHistCopies][8 * 256];
  uint32_t* mine = s_hist[(threadIdx.x >> 6) % kHistCopies];
  for (uint32_t i = threadIdx.x; i < kHistCopies * 8 * 256; i += blockDim.x) (&s_hist[0][0])[i] = 0;
  // The look-back table of every pass starts NOT_READY.
  const uint64_t gtid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t gstride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = gtid; i < lookback_words; i += gstride) lookback[i] = 0;
  __syncthreads();
  for (uint64_t i = gtid; i < n; i += gstride) {
    K k = keys[i];
    for (uint32_t p = 0; p < passes; ++p) atomicAdd(&mine[p * 256 + digit_of(k, begin_bit + 8 * p)], 1u);
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < passes * 256; i += blockDim.x) {
    uint32_t c = 0;
#pragma unroll
    for (int w = 0; w < kHistCopies; ++w) c += s_hist[w][i];
    if (c) atomicAdd(&hist[i], c);
  }
}

// Stable rank of every key of a wave within its digit (kpt keys per lane, in
// order of k, then lane): on return s_hist holds the wave's digit counts.
// `valid` is a prefix of the wave's keys.
template <typename K, int kKpt>
BJ_D void rank_keys(const K (&key)[kKpt], uint32_t shift, uint32_t valid, uint32_t lane, uint32_t* __restrict__ s_hist,
                    uint32_t (&rank)[kKpt]) {
#pragma unroll
  for (int k = 0; k < kKpt; ++k) {
    const bool on = (uint32_t)k * 64u + lane < valid;
    const uint32_t d = digit_of(key[k], shift);
    uint64_t match = ballot(on);
    uint32_t lo = (uint32_t)match, hi = (uint32_t)(match >> 32);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      // lanes whose bit b equals this lane's
      const uint64_t m = ballot((d >> b) & 1u);
      const uint32_t off = ((d >> b) & 1u) - 1u;  // 0 if set, else all ones
      lo &= (uint32_t)m ^ off;
      hi &= (uint32_t)(m >> 32) ^ off;
    }
    const uint32_t below = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
    const uint32_t total = (uint32_t)(__builtin_popcount(lo) + __builtin_popcount(hi));
    const uint32_t base = on ? s_hist[d] : 0u;
    rank[k] = base + below;
    __builtin_amdgcn_wave_barrier();
    if (on && below + 1u == total) s_hist[d] = base + total;
    __builtin_amdgcn_wave_barrier();
  }
}

// Sums of the look-back words at p[-256 j], j = 1..count (count <= kMost), once
// all are published; their loads are in flight together.  False if one stayed
// unpublished for more than `patience` polls.
template <uint32_t kMost>
BJ_D bool sum_published(const uint32_t* p, uint32_t count, uint32_t patience, uint32_t& sum) {
  for (uint32_t spins = 0;; ++spins) {
    uint32_t v[kMost];
#pragma unroll
    for (uint32_t j = 0; j < kMost; ++j)
      v[j] = j < count ? __hip_atomic_load(p - 256 * (int64_t)(j + 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                       : kLookbackAgg;
    uint32_t total = 0;
    bool ready = true;
#pragma unroll
    for (uint32_t j = 0; j < kMost; ++j) {
      total += v[j] & kLookbackMask;
      ready = ready && (v[j] & ~kLookbackMask) != 0;
    }
    if (ready) {
      sum += total;
      return true;
    }
    if (spins >= patience) return false;
    __builtin_amdgcn_s_sleep(1);
  }
}

// The number of keys with this thread's digit in all tiles before `tile`
// (`before`), from the counts published per tile and per group of kGroup tiles.
// False if a count stayed unpublished for `patience` polls: then
// count_back finds the number.
template <uint32_t kGroup>
BJ_D bool look_back(uint32_t* __restrict__ lookback, uint32_t tiles, uint32_t tile, uint32_t count, uint32_t t,
                    uint32_t patience, uint32_t& before) {
  uint32_t* mine = lookback + (uint64_t)tile * 256 + t;
  const uint32_t g = tile / kGroup, q = tile % kGroup;
  const bool last = q == kGroup - 1;  // publishes its group's counts
  uint32_t* group = lookback + ((uint64_t)tiles + g) * 256 + t;
  before = 0;
  if (q != 0 && !sum_published<kGroup - 1>(mine, q, patience, before)) return false;
  if (last)
    __hip_atomic_store(group, (g == 0 ? kLookbackInc : kLookbackAgg) | ((before + count) & kLookbackMask),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // whole groups, two loads in flight: aggregates are added up to an
  // inclusive prefix, or to the first group not yet published, polled again.
  // (The words come from memory, past the L2s, and the prefix is mostly near:
  // 47.5M 64-bit pairs 3.60 ms, 3.65 with three and 3.69 with four in flight.)
  constexpr int kAhead = 2;
  int64_t j = (int64_t)g - 1;
  uint32_t spins = 0;
  while (j >= 0) {
    uint32_t v[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k)
      v[k] = j - k >= 0 ? __hip_atomic_load(lookback + ((uint64_t)tiles + (uint64_t)(j - k)) * 256 + t,
                                            __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                        : 0u;
    int k = 0;
    bool waiting = false, done = false;
#pragma unroll
    for (int q2 = 0; q2 < kAhead; ++q2) {
      if (waiting || done || j - q2 < 0) continue;
      const uint32_t flag = v[q2] & ~kLookbackMask;
      if (flag == 0) {
        waiting = true;
      } else {
        before += v[q2] & kLookbackMask;
        done = flag == kLookbackInc;
        ++k;
      }
    }
    if (done) break;
    j -= k;
    if (waiting) {
      if (++spins > patience) return false;
      __builtin_amdgcn_s_sleep(1);
    }
  }
  if (last && g > 0)
    __hip_atomic_store(group, kLookbackInc | ((before + count) & kLookbackMask), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// look_back's number without waiting, by the whole block: a predecessor whose
// counts are not published (its block may not have started, and need not start
// before this one ends) is counted from its keys, which no tile of the pass
// writes, and published in its place -- the same words that it would write.
// s_count: 256 words of LDS that nothing else uses now.
template <typename K, uint32_t kGroup>
BJ_D uint32_t count_back(const K* __restrict__ keys, uint32_t tile_keys, uint32_t shift,
                         uint32_t* __restrict__ lookback, uint32_t tiles, uint32_t tile, uint32_t count, uint32_t t,
                         uint32_t* __restrict__ s_count) {
  const uint32_t g = tile / kGroup;
  auto tile_count = [&](uint32_t p) {
    uint32_t* at = lookback + (uint64_t)p * 256 + t;
    uint32_t v = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!__syncthreads_and(v != 0u)) {
      s_count[t] = 0;
      __syncthreads();
      const K* first = keys + (uint64_t)p * tile_keys;  // a predecessor's tile is full
      for (uint32_t i = t; i < tile_keys; i += kSortBlock) atomicAdd(&s_count[digit_of(first[i], shift)], 1u);
      __syncthreads();
      v = kLookbackAgg | s_count[t];
      __hip_atomic_store(at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return v & kLookbackMask;
  };
  uint32_t before = 0;
  for (uint32_t p = tile; p > g * kGroup;) before += tile_count(--p);
  // a group's word only ever grows: unpublished, aggregate, inclusive prefix
  auto publish = [&](uint32_t group, uint32_t word) {
    __hip_atomic_fetch_max(lookback + ((uint64_t)tiles + group) * 256 + t, word, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
  };
  const bool last = tile % kGroup == kGroup - 1;
  if (last) publish(g, (g == 0 ? kLookbackInc : kLookbackAgg) | ((before + count) & kLookbackMask));
  bool done = false;
  for (uint32_t j = g; j-- > 0;) {
    uint32_t v = __hip_atomic_load(lookback + ((uint64_t)tiles + j) * 256 + t, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    if (!__syncthreads_and(done || v != 0u)) {
      uint32_t sum = 0;
      for (uint32_t p = j * kGroup; p < (j + 1) * kGroup; ++p) sum += tile_count(p);
      if (v == 0u) {
        v = (j == 0 ? kLookbackInc : kLookbackAgg) | sum;
        publish(j, v);
      }
    }
    if (!done) {
      before += v & kLookbackMask;
      done = (v & kLookbackInc) != 0u;
    }
    if (__syncthreads_and(done)) break;
  }
  if (last && g > 0) publish(g, kLookbackInc | ((before + count) & kLookbackMask));
  return before;
}

template <typename K, bool kValues, int kKpt>
__global__ void __launch_bounds__(kSortBlock) __attribute__((amdgpu_waves_per_eu(4))) sort_bin_kernel(const K* __restrict__ in_keys, K* __restrict__ out_keys,
                                                              const uint32_t* __restrict__ in_vals,
                                                              uint32_t* __restrict__ out_vals, uint64_t n,
                                                              uint32_t shift, const uint32_t* __restrict__ pass_hist,
                                                              uint32_t* __restrict__ lookback,
                                                              uint32_t* __restrict__ tickets, uint32_t patience) {
  constexpr uint32_t kTile = kSortBlock * kKpt, kGroup = sort_group(kKpt);
  // keys are staged first, then the values in the same words: four blocks of
  // 4,096 pairs fit a CU instead of two
  __shared__ K s_keys[kTile];
  __shared__ uint32_t s_wave_hist[kSortWaves][256];
  __shared__ uint32_t s_adjust[256];  // the tile's digit counts, then the offset from tile to global position
  __shared__ uint32_t s_tmp[kSortWaves];
  __shared__ uint32_t s_tile, s_late;

  const uint32_t t = threadIdx.x;
  const uint32_t lane = lane_id();
  const uint32_t wave = t >> 6;

  // Tiles are drawn in order within a class.  Of another class a predecessor
  // may not have started yet: where it stays out, count_back does without it.
  if (t == 0) {
    const uint32_t c = blockIdx.x % kTicketClasses;
    s_tile = kTicketClasses * atomicAdd(tickets + c * kTicketStride, 1u) + c;
    s_late = 0;
  }
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) s_wave_hist[w][t] = 0;
  s_adjust[t] = 0;
  __syncthreads();
  const uint32_t tile = s_tile;
  const uint64_t tile_base = (uint64_t)tile * kTile;
  const uint32_t tile_count = n - tile_base < kTile ? (uint32_t)(n - tile_base) : kTile;

  // ---- load (wave-striped: each load instruction covers 64 consecutive keys)
  K key[kKpt];
  const uint32_t wave_base = wave * 64 * kKpt;
  const uint32_t valid = tile_count > wave_base ? (tile_count - wave_base < 64u * kKpt ? tile_count - wave_base : 64u * kKpt) : 0u;
#pragma unroll
  for (int k = 0; k < kKpt; ++k) {
    const uint32_t o = (uint32_t)k * 64 + lane;
    key[k] = o < valid ? in_keys[tile_base + wave_base + o] : (K)0;
  }

  // ---- the tile's digit counts, published before the ranking
#pragma unroll
  for (int k = 0; k < kKpt; ++k)
    if ((uint32_t)k * 64 + lane < valid) atomicAdd(&s_adjust[digit_of(key[k], shift)], 1u);
  __syncthreads();
  const uint32_t count = s_adjust[t];
  __hip_atomic_store(lookback + (uint64_t)tile * 256 + t, kLookbackAgg | count, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);

  // ---- stable wave-level ranking
  uint32_t rank[kKpt];
  rank_keys<K, kKpt>(key, shift, valid, lane, s_wave_hist[wave], rank);
  const uint32_t digit_start = block_exclusive_scan_256(count, s_tmp, nullptr);
  const uint32_t global_excl = block_exclusive_scan_256(pass_hist[t], s_tmp, nullptr);
  // (the scans' barriers close the ranking) per-wave positions of digit t
  uint32_t run = digit_start;
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) {
    const uint32_t c = s_wave_hist[w][t];
    s_wave_hist[w][t] = run;
    run += c;
  }
  // the values' loads overlap the look-back's
  uint32_t val[kValues ? kKpt : 1];
  if constexpr (kValues) {
#pragma unroll
    for (int k = 0; k < kKpt; ++k) {
      const uint32_t o = (uint32_t)k * 64 + lane;
      val[k] = o < valid ? in_vals[tile_base + wave_base + o] : 0u;
    }
  }
  uint32_t exclusive = 0;
  if (!look_back<kGroup>(lookback, gridDim.x, tile, count, t, patience, exclusive)) s_late = 1;
  s_adjust[t] = global_excl + exclusive - digit_start;
  __syncthreads();
  if (s_late) {
    exclusive = count_back<K, kGroup>(in_keys, kTile, shift, lookback, gridDim.x, tile, count, t,
                                      reinterpret_cast<uint32_t*>(s_keys));
    s_adjust[t] = global_excl + exclusive - digit_start;
    __syncthreads();
  }

  // ---- keys into LDS in sorted order, then out in digit-contiguous runs
#pragma unroll
  for (int k = 0; k < kKpt; ++k) {
    if ((uint32_t)k * 64 + lane < valid) {
      rank[k] += s_wave_hist[wave][digit_of(key[k], shift)];
      s_keys[rank[k]] = key[k];
    }
  }
  __syncthreads();
  uint32_t pos[kKpt];
#pragma unroll
  for (int k = 0; k < kKpt; ++k) {
    const uint32_t i = (uint32_t)k * kSortBlock + t;
    pos[k] = 0xFFFFFFFFu;
    if (i < tile_count) {
      const K x = s_keys[i];
      pos[k] = s_adjust[digit_of(x, shift)] + i;
      if (pos[k] < n) out_keys[pos[k]] = x;
    }
  }
  if constexpr (kValues) {
    uint32_t* s_vals = reinterpret_cast<uint32_t*>(s_keys);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kKpt; ++k)
      if ((uint32_t)k * 64 + lane < valid) s_vals[rank[k]] = val[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kKpt; ++k) {
      const uint32_t i = (uint32_t)k * kSortBlock + t;
      if (i < tile_count && pos[k] < n) out_vals[pos[k]] = s_vals[i];
    }
  }
}

// Every pass over a short list in one block: the keys (and values) live in
// registers and LDS from the first pass to the last.
constexpr int kSmallBlock = 1024, kSmallKpt = (int)(kSortSmall / kSmallBlock), kSmallWaves = kSmallBlock / 64;
template <typename K, bool kValues>
__global__ void __launch_bounds__(kSmallBlock) sort_small_kernel(K* __restrict__ keys, uint32_t* __restrict__ vals,
                                                                 uint32_t n, uint32_t begin_bit, uint32_t passes) {
  __shared__ K s_keys[kSortSmall];
  __shared__ uint32_t s_vals[kValues ? kSortSmall : 1];
  __shared__ uint32_t s_hist[kSmallWaves][256];
  __shared__ uint32_t s_tmp[4];
  const uint32_t t = threadIdx.x, lane = lane_id(), wave = t >> 6;
  // a wave takes `span` consecutive keys, 64 at a time
  const uint32_t span = (n + kSmallBlock - 1) / kSmallBlock * 64;
  const uint32_t base = wave * span;
  const uint32_t valid = n > base ? (n - base < span ? n - base : span) : 0u;
  for (uint32_t i = t; i < n; i += kSmallBlock) {
    s_keys[i] = keys[i];
    if constexpr (kValues) s_vals[i] = vals[i];
  }
  for (uint32_t p = 0; p < passes; ++p) {
    const uint32_t shift = begin_bit + 8 * p;
    for (uint32_t i = t; i < kSmallWaves * 256; i += kSmallBlock) (&s_hist[0][0])[i] = 0;
    __syncthreads();
    K key[kSmallKpt];
    uint32_t val[kValues ? kSmallKpt : 1], rank[kSmallKpt];
#pragma unroll
    for (int k = 0; k < kSmallKpt; ++k) {
      const uint32_t o = (uint32_t)k * 64 + lane;
      key[k] = o < valid ? s_keys[base + o] : (K)0;
      if constexpr (kValues) val[k] = o < valid ? s_vals[base + o] : 0u;
    }
#pragma unroll
    for (int k = 0; k < kSmallKpt; ++k) {
      if ((uint32_t)k * 64 < valid) {
        const K one[1] = {key[k]};
        uint32_t r[1];
        rank_keys<K, 1>(one, shift, valid - (uint32_t)k * 64, lane, s_hist[wave], r);
        rank[k] = r[0];
      }
    }
    __syncthreads();
    // digit t's first position, then each wave's
    uint32_t total = 0;
    if (t < 256)
      for (int w = 0; w < kSmallWaves; ++w) total += s_hist[w][t];
    uint32_t x = total;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = __shfl_up(x, off, 64);
      if (lane >= (uint32_t)off) x += y;
    }
    if (t < 256 && lane == 63) s_tmp[wave] = x;
    __syncthreads();
    if (t < 256) {
      uint32_t run = x - total;
      for (uint32_t w = 0; w < wave; ++w) run += s_tmp[w];
      for (int w = 0; w < kSmallWaves; ++w) {
        const uint32_t c = s_hist[w][t];
        s_hist[w][t] = run;
        run += c;
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kSmallKpt; ++k) {
      if ((uint32_t)k * 64 + lane < valid) {
        const uint32_t at = s_hist[wave][digit_of(key[k], shift)] + rank[k];
        s_keys[at] = key[k];
        if constexpr (kValues) s_vals[at] = val[k];
      }
    }
    __syncthreads();
  }
  for (uint32_t i = t; i < n; i += kSmallBlock) {
    keys[i] = s_keys[i];
    if constexpr (kValues) vals[i] = s_vals[i];
  }
}

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

template <typename K, bool kValues, int kKpt>
void launch_bin(bajo_ctx* ctx, const SortPlan& p, const K* src, K* dst, const uint32_t* vsrc, uint32_t* vdst,
                uint32_t shift, const uint32_t* hist, uint32_t* lookback, uint32_t* tickets, uint32_t patience) {
  sort_bin_kernel<K, kValues, kKpt><<<p.tiles, kSortBlock, 0, ctx->stream>>>(
      src, dst, vsrc, vdst, p.n, shift, hist, lookback, tickets, patience);
}

template <typename K, bool kValues>
int32_t run_typed(bajo_ctx* ctx, const SortPlan& p, K* keys, uint32_t* values, char* ws, bool hist_ready) {
  if (p.n <= kSortSmall) {
    sort_small_kernel<K, kValues><<<1, kSmallBlock, 0, ctx->stream>>>(keys, values, (uint32_t)p.n,
                                                                      (uint32_t)p.begin_bit, (uint32_t)p.passes);
    BJ_HIP(hipGetLastError());
    return BAJO_OK;
  }
  K* alt_keys = (K*)(ws + p.off_alt_keys);
  uint32_t* alt_vals = kValues ? (uint32_t*)(ws + p.off_alt_vals) : nullptr;
  uint32_t* hist = (uint32_t*)(ws + p.off_hist);
  uint32_t* lookback = (uint32_t*)(ws + p.off_lookback);
  uint32_t* tickets = (uint32_t*)(ws + p.off_tickets);
  const uint64_t lb_pass_words = p.lookback_words / (uint64_t)p.passes;
  if (!hist_ready) {
    sort_init_kernel<<<1, 256, 0, ctx->stream>>>(hist, (uint32_t)p.passes * 256, tickets,
                                                 (uint32_t)p.passes * kTicketWords);
    BJ_HIP(hipGetLastError());
    unsigned blocks = div_up(p.n, (uint64_t)kHistBlock * 4);
    if (blocks > 256) blocks = 256;
    sort_hist_kernel<K><<<blocks, kHistBlock, 0, ctx->stream>>>(keys, p.n, (uint32_t)p.begin_bit, (uint32_t)p.passes,
                                                                hist, lookback, p.lookback_words);
    BJ_HIP(hipGetLastError());
  }
  K* src = keys;
  K* dst = alt_keys;
  uint32_t* vsrc = values;
  uint32_t* vdst = alt_vals;
  const uint32_t patience = ctx->spin_limit ? ctx->spin_limit : kLookbackPatience;
  for (int pass = 0; pass < p.passes; ++pass) {
    const uint32_t shift = (uint32_t)(p.begin_bit + 8 * pass);
    const uint32_t* h = hist + pass * 256;
    uint32_t* lb = lookback + lb_pass_words * pass;
    uint32_t* tk = tickets + (uint32_t)pass * kTicketWords;
    if (p.kpt == 4) launch_bin<K, kValues, 4>(ctx, p, src, dst, vsrc, vdst, shift, h, lb, tk, patience);
    else if (p.kpt == 8) launch_bin<K, kValues, 8>(ctx, p, src, dst, vsrc, vdst, shift, h, lb, tk, patience);
    else launch_bin<K, kValues, 16>(ctx, p, src, dst, vsrc, vdst, shift, h, lb, tk, patience);
    BJ_HIP(hipGetLastError());
    K* sk = src; src = dst; dst = sk;
    uint32_t* sv = vsrc; vsrc = vdst; vdst = sv;
  }
  if (src != keys) {
    BJ_HIP(hipMemcpyAsync(keys, src, p.n * sizeof(K), hipMemcpyDeviceToDevice, ctx->stream));
    if (kValues) BJ_HIP(hipMemcpyAsync(values, vsrc, p.n * sizeof(uint32_t), hipMemcpyDeviceToDevice, ctx->stream));
  }
  return BAJO_OK;
}

}  // namespace

SortPlan make_sort_plan(uint64_t n, int key_bytes, int has_values, int begin_bit, int end_bit) {
  SortPlan p;
  p.n = n;
  p.key_bytes = key_bytes;
  p.has_values = has_values;
  p.begin_bit = begin_bit;
  p.end_bit = end_bit;
  p.passes = (end_bit - begin_bit + 7) / 8;
  p.kpt = n <= kSortKpt4Keys ? 4 : (n <= kSortKpt8Keys ? 8 : 16);
  p.tiles = div_up(n ? n : 1, (uint64_t)kSortBlock * p.kpt);
  p.lookback_words = (size_t)(p.passes ? p.passes : 1) * (p.tiles + div_up(p.tiles, sort_group(p.kpt))) * 256;
  size_t off = 0;
  p.off_alt_keys = off;
  off = align256(off + n * (size_t)key_bytes);
  p.off_alt_vals = off;
  off = align256(off + (has_values ? n * sizeof(uint32_t) : 0));
  p.off_hist = off;
  off = align256(off + (size_t)(p.passes ? p.passes : 1) * 256 * sizeof(uint32_t));
  p.off_lookback = off;
  off = align256(off + p.lookback_words * sizeof(uint32_t));
  p.off_tickets = off;
  off = align256(off + (size_t)(p.passes ? p.passes : 1) * kTicketWords * sizeof(uint32_t));
  p.total = off;
  return p;
}

size_t sort_workspace_bound(uint64_t n, int key_bytes, int has_values, int begin_bit, int end_bit) {
  size_t most = make_sort_plan(n, key_bytes, has_values, begin_bit, end_bit).total;
  for (const uint64_t m : {kSortKpt4Keys, kSortKpt8Keys}) {
    if (n <= m) break;
    const size_t b = make_sort_plan(m, key_bytes, has_values, begin_bit, end_bit).total;
    if (b > most) most = b;
  }
  return most;
}

int32_t onesweep_run(bajo_ctx* ctx, const SortPlan& plan, void* keys, uint32_t* values, void* ws, bool hist_ready) {
  if (plan.n <= 1 || plan.passes == 0) return BAJO_OK;
  char* w = (char*)ws;
  if (plan.key_bytes == 8)
    return plan.has_values ? run_typed<uint64_t, true>(ctx, plan, (uint64_t*)keys, values, w, hist_ready)
                           : run_typed<uint64_t, false>(ctx, plan, (uint64_t*)keys, values, w, hist_ready);
  return plan.has_values ? run_typed<uint32_t, true>(ctx, plan, (uint32_t*)keys, values, w, hist_ready)
                         : run_typed<uint32_t, false>(ctx, plan, (uint32_t*)keys, values, w, hist_ready);
}

}  // namespace bj

namespace {

int32_t sort_entry(bajo_ctx* ctx, void* keys, uint32_t* values, uint64_t n, int key_bytes, int begin_bit,
                   int end_bit, void* workspace, uint64_t workspace_bytes, const char* name) {
  BJ_REQUIRE(ctx != nullptr, "%s: ctx is NULL", name);
  BJ_REQUIRE(n == 0 || keys != nullptr, "%s: keys is NULL", name);
  BJ_REQUIRE(n <= bj::kSortMaxKeys, "%s: n=%llu exceeds the 2^30-1 key limit", name, (unsigned long long)n);
  BJ_REQUIRE(begin_bit >= 0 && end_bit <= key_bytes * 8 && begin_bit <= end_bit && begin_bit % 8 == 0 &&
                 end_bit % 8 == 0,
             "%s: bit range [%d, %d) must be byte aligned inside the key", name, begin_bit, end_bit);
  if (n <= 1 || begin_bit == end_bit) return BAJO_OK;
  bj::SortPlan plan = bj::make_sort_plan(n, key_bytes, values != nullptr, begin_bit, end_bit);
  void* ws = workspace;
  if (ws) {
    BJ_REQUIRE(workspace_bytes >= plan.total, "%s: workspace of %llu bytes is below the %llu required", name,
               (unsigned long long)workspace_bytes, (unsigned long long)plan.total);
  } else {
    const size_t bytes = bj::sort_workspace_bound(n, key_bytes, values != nullptr, begin_bit, end_bit);
    int32_t rc = bj::ctx_scratch(ctx, bytes, &ws);
    if (rc) return rc;
  }
  return bj::onesweep_run(ctx, plan, keys, values, ws, false);
}

// ---- fixed-scratch sort (no allocation) --------------------------------------
// The workspace of bajo_onesweep_radix_sort_pairs_u64_u32_noalloc lives in a
// file-scope device array: alternate keys and values, digit histograms,
// look-back table and tile tickets of one sort of at most kNoAllocMaxKeys
// pairs.  Each device holds its own copy for the life of the process; host
// code uses the address hipGetSymbolAddress returns for the current device,
// never the array's name.
constexpr uint64_t kNoAllocMaxKeys = 1ull << 20;
constexpr size_t kNoAllocScratchBytes = 20ull << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kNoAllocMaxDevices = 64;
std::mutex g_noalloc_mu;
void* g_noalloc_ptr[kNoAllocMaxDevices] = {};

// The device address of `scratch` on `device`, looked up once per device
// with that device current.
int32_t noalloc_scratch(int device, void** out) {
  BJ_REQUIRE(device >= 0 && device < kNoAllocMaxDevices, "noalloc sort: device %d outside [0, %d)", device,
             kNoAllocMaxDevices);
  std::lock_guard<std::mutex> lock(g_noalloc_mu);
  if (!g_noalloc_ptr[device]) {
    int prev = 0;
    BJ_HIP(hipGetDevice(&prev));
    BJ_HIP(hipSetDevice(device));
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    (void)hipSetDevice(prev);
    if (e != hipSuccess) return bj::hip_fail(e, "hipGetSymbolAddress(scratch)", __FILE__, __LINE__);
    BJ_REQUIRE(ptr != nullptr, "noalloc sort: hipGetSymbolAddress returned NULL");
    g_noalloc_ptr[device] = ptr;
  }
  *out = g_noalloc_ptr[device];
  return BAJO_OK;
}

}  // namespace

extern "C" {

uint64_t bajo_sort_workspace_bytes(uint64_t n, int32_t key_bytes, int32_t has_values) {
  if (key_bytes != 4 && key_bytes != 8) return 0;
  return bj::sort_workspace_bound(n, key_bytes, has_values != 0, 0, key_bytes * 8);
}

int32_t bajo_device_radix_sort_pairs_u64_u32(bajo_ctx* ctx, uint64_t* keys, uint32_t* values, uint64_t n,
                                             void* workspace, uint64_t workspace_bytes) {
  BJ_REQUIRE(n == 0 || values != nullptr, "bajo_device_radix_sort_pairs_u64_u32: values is NULL");
  return sort_entry(ctx, keys, values, n, 8, 0, 64, workspace, workspace_bytes, "bajo_device_radix_sort_pairs_u64_u32");
}

int32_t bajo_device_radix_sort_pairs_u32_u32(bajo_ctx* ctx, uint32_t* keys, uint32_t* values, uint64_t n,
                                             void* workspace, uint64_t workspace_bytes) {
  BJ_REQUIRE(n == 0 || values != nullptr, "bajo_device_radix_sort_pairs_u32_u32: values is NULL");
  return sort_entry(ctx, keys, values, n, 4, 0, 32, workspace, workspace_bytes, "bajo_device_radix_sort_pairs_u32_u32");
}

int32_t bajo_device_radix_sort_keys_u64(bajo_ctx* ctx, uint64_t* keys, uint64_t n, void* workspace,
                                        uint64_t workspace_bytes) {
  return sort_entry(ctx, keys, nullptr, n, 8, 0, 64, workspace, workspace_bytes, "bajo_device_radix_sort_keys_u64");
}

int32_t bajo_device_radix_sort_keys_u32(bajo_ctx* ctx, uint32_t* keys, uint64_t n, void* workspace,
                                        uint64_t workspace_bytes) {
  return sort_entry(ctx, keys, nullptr, n, 4, 0, 32, workspace, workspace_bytes, "bajo_device_radix_sort_keys_u32");
}

int32_t bajo_onesweep_radix_sort_keys_u64(bajo_ctx* ctx, uint64_t* keys, uint64_t n, int32_t begin_bit,
                                          int32_t end_bit, void* workspace, uint64_t workspace_bytes) {
  return sort_entry(ctx, keys, nullptr, n, 8, begin_bit, end_bit, workspace, workspace_bytes,
                    "bajo_onesweep_radix_sort_keys_u64");
}

int32_t bajo_onesweep_radix_sort_pairs_u64_u32(bajo_ctx* ctx, uint64_t* keys, uint32_t* values, uint64_t n,
                                               int32_t begin_bit, int32_t end_bit, void* workspace,
                                               uint64_t workspace_bytes) {
  BJ_REQUIRE(n == 0 || values != nullptr, "bajo_onesweep_radix_sort_pairs_u64_u32: values is NULL");
  return sort_entry(ctx, keys, values, n, 8, begin_bit, end_bit, workspace, workspace_bytes,
                    "bajo_onesweep_radix_sort_pairs_u64_u32");
}
int32_t bajo_onesweep_radix_sort_pairs_u64_u32_noalloc(bajo_ctx* ctx, uint64_t* keys, uint32_t* values, uint64_t n,
                                                       int32_t begin_bit, int32_t end_bit) {
  const char* name = "bajo_onesweep_radix_sort_pairs_u64_u32_noalloc";
  BJ_REQUIRE(ctx != nullptr, "%s: ctx is NULL", name);
  BJ_REQUIRE(n == 0 || (keys != nullptr && values != nullptr), "%s: keys or values is NULL", name);
  BJ_REQUIRE(n <= kNoAllocMaxKeys, "%s: n=%llu exceeds the fixed scratch's limit of %llu pairs", name,
             (unsigned long long)n, (unsigned long long)kNoAllocMaxKeys);
  BJ_REQUIRE(begin_bit >= 0 && end_bit <= 64 && begin_bit <= end_bit && begin_bit % 8 == 0 && end_bit % 8 == 0,
             "%s: bit range [%d, %d) must be byte aligned inside the key", name, begin_bit, end_bit);
  if (n <= 1 || begin_bit == end_bit) return BAJO_OK;
  const bj::SortPlan plan = bj::make_sort_plan(n, 8, 1, begin_bit, end_bit);
  BJ_REQUIRE(plan.total <= kNoAllocScratchBytes, "%s: workspace of %llu bytes exceeds the fixed scratch", name,
             (unsigned long long)plan.total);
  void* ws = nullptr;
  const int32_t rc = noalloc_scratch(ctx->device, &ws);
  if (rc) return rc;
  return bj::onesweep_run(ctx, plan, keys, values, ws, false);
}

}  // extern "C"

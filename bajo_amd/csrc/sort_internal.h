// Internal interface of the onesweep radix sort shared with the LBVH builder.
#pragma once

#include "bajo_common.h"

namespace bj {

constexpr int kSortBlock = 256;             // 4 waves of 64
constexpr int kSortWaves = kSortBlock / 64;
// Tiles per look-back group.  A tile reads the counts of half a group on
// average, and at 16 keys per thread the registers of 15 loads in flight
// spill: 64-bit pairs, 4M 314 us with 16 tiles and 262 with 8, 47.5M 4.16 and
// 3.60 ms.  Shorter lists have registers to spare and fewer, smaller tiles:
// 300K 107 and 110 us.
constexpr uint32_t sort_group(int kpt) { return kpt == 16 ? 8u : 16u; }
// Tile tickets are drawn from eight counters a cache line apart.
constexpr uint32_t kTicketClasses = 8, kTicketStride = 32;
constexpr uint32_t kTicketWords = kTicketClasses * kTicketStride;  // per pass
// Lists one block sorts by itself, in LDS.
constexpr uint64_t kSortSmall = 8192;
constexpr uint32_t kLookbackAgg = 0x40000000u;
constexpr uint32_t kLookbackInc = 0x80000000u;
constexpr uint32_t kLookbackMask = 0x3FFFFFFFu;
constexpr uint64_t kSortMaxKeys = (1ull << 30) - 1;
// Polls of the look-back table (about a microsecond each) before a tile counts
// its missing predecessors itself; a pass alone on the chip waits some tens.
constexpr uint32_t kLookbackPatience = 512;

// Workspace layout of one sort.  All offsets are 256-byte aligned.
struct SortPlan {
  uint64_t n = 0;
  int key_bytes = 8;
  int has_values = 0;
  int begin_bit = 0, end_bit = 64, passes = 0;
  int kpt = 16;          // keys per thread of a tile
  unsigned tiles = 0;
  size_t lookback_words = 0;  // all passes: 256 words per tile and per group of tiles
  size_t off_alt_keys = 0, off_alt_vals = 0, off_hist = 0, off_lookback = 0, off_tickets = 0, total = 0;
};

// Longest lists of tiles with 4 and with 8 keys per thread (longer ones: 16).
// Smaller tiles for shorter lists: a pass lasts as long as a tile's chain, so
// the keys are spread over the chip (64-bit pairs with 16 tiles per group:
// 262,144 keys 105.9 us with 4 keys per thread, 115.3 with 8; 1M 163 with 8,
// 186 with 16; 2M 258 and 262; 4M 451 and 402; the call's own figures are
// lower by now, 4M 262).
constexpr uint64_t kSortKpt4Keys = 262144, kSortKpt8Keys = 1310720;

SortPlan make_sort_plan(uint64_t n, int key_bytes, int has_values, int begin_bit, int end_bit);

// Bytes that hold the workspace of every list of at most n keys: the look-back
// table shrinks where the tiles grow, so a shorter list can need more.
size_t sort_workspace_bound(uint64_t n, int key_bytes, int has_values, int begin_bit, int end_bit);

// Runs the digit-binning passes.  When `hist_ready` is false the plan's
// counters are cleared and the digit histogram is computed first; when true
// the caller has already cleared the tickets, zeroed the look-back table and
// filled the histogram (the LBVH Morton kernel does this in its own pass).
// Lists of at most kSortSmall keys need none of them.
// Sorted output always lands back in `keys` / `values`.
int32_t onesweep_run(bajo_ctx* ctx, const SortPlan& plan, void* keys, uint32_t* values, void* ws, bool hist_ready);

}  // namespace bj

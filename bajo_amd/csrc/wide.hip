// Binary LBVH -> 8-wide BVH with quantized child boxes (gfx950).
//
// Plays the role of bajo's wide collapse and compressed-BVH8 encoding
// (bvh/gpu/builder/wide_collapse.mojo:148-643, bvh/gpu/compressed_bounds_bvh.mojo:
// 84-369): a top-down collapse that opens the child with the largest surface
// area until a node has 8 children -- first among children holding more than
// the leaf size, then among any inner child -- and turns inner children of
// at most the leaf size (1..8 triangles) into leaves.  Child boxes are
// stored as 8-bit offsets on a per-axis power-of-two grid anchored at the
// node's lower corner.
//
// Unlike bajo's persistent work queue with a spin fail-safe, no wave here
// waits on another block.  Two launches build the whole hierarchy:
//   - one block opens the first levels, one per barrier round, until a level
//     holds more nodes than the block has threads, then nodes with more leaves
//     than a block's share, and deals out the nodes still to be opened: every
//     gridDim-th to a block if that spreads the leaves evenly, else a run of
//     them with a share of the leaves;
//   - one block per CU then finishes its nodes' subtrees by itself: it keeps
//     the index ranges of its nodes still to be opened on an LDS stack and
//     reserves the nodes of each batch's children (a contiguous range) with
//     one atomic.
// No block of the second launch gets more than two shares, whatever the
// geometry.  With 80 % of 4M triangles in a cube of 5 % of the scene's width a
// deal by node number alone left 40 % of the nodes to one block: 7.62 ms, now
// 0.28; 4,096 environments of 256 to 65,536 triangles 1.86 -> 1.24 ms.  Opening
// and dealing costs an even mesh 5 us (4M: 177 -> 182; nearly all of it is code
// fetched once: scans unrolled or with LDS atomics took 3 us more, leaf counts
// read from memory instead of kept as nodes are reserved 5 us more).
// A node's children are opened through a chain of up to seven dependent loads,
// so a level costs its latency however few nodes it has.  One launch per level
// (each followed by a launch that opened the next, with four to five spare
// ones for the depth) took 22 launches of 5-31 us: 0.40 ms at 4M triangles
// (LBVH), 0.26 ms at 1M (H-PLOC), where the two launches took 0.24 and 0.15.
// The host reads nothing back, so the collapse is enqueue-only and can be
// captured in a HIP graph.  Leaf children reference ranges of the sorted
// triangle records that the refit already wrote (a subtree covers a contiguous
// sorted range), so no triangle data is copied.
#include "bvh_internal.h"

namespace bj {
namespace {

constexpr int kCollapseBlock = 1024;
// Levels the first launch takes at most, and ranges a block of the second one
// keeps (one per level of its subtrees): a deeper tree raises
// BAJO_STATUS_COLLAPSE_FAILED.
constexpr uint32_t kLevelCap = 4096;
// Leaves of a subtree that one block finishes in a few batches: smaller ones
// are not opened to spread them.
constexpr uint32_t kSmallSubtree = 4096;
// Blocks of the second launch at most: their runs are kept in one hand-over
// slot block of the climb, which is free by then (kHandSlots 32-byte records).
constexpr unsigned kMostBlocks = 1023;
// wide_ctl words: node counter, range still to be opened, status, how the range is dealt
constexpr int kCtlCount = 0, kCtlBegin = 1, kCtlEnd = 2, kCtlStatus = 3, kCtlRuns = 4;
constexpr uint32_t kStatusOutOfNodes = 1, kStatusTooDeep = 2, kStatusBadRoot = 4;

struct Child {
  uint32_t ref, count;
  uint32_t first;  // Karras hierarchies: the first sorted position below
  float b[6];
};

BJ_D float half_area(const float* b) {
  const float dx = b[3] - b[0], dy = b[4] - b[1], dz = b[5] - b[2];
  return dx * dy + dx * dz + dy * dz;
}

// The children of binary node `node`.  In a Karras hierarchy the left child's
// reference is the split position, so with the node's own range (`first`,
// `count`) the children's ranges are known without another load; H-PLOC nodes
// look their counts up.
template <bool kKarras>
BJ_D void load_children(const BjNode* __restrict__ bnodes, const uint32_t* __restrict__ leaf_counts, uint32_t node,
                        uint32_t first, uint32_t count, Child& l, Child& r) {
  const float4* p = reinterpret_cast<const float4*>(bnodes + node);
  const float4 a = p[0], b = p[1], c = p[2];
  const uint4 m = reinterpret_cast<const uint4*>(bnodes + node)[3];
  l.b[0] = a.x; l.b[1] = a.y; l.b[2] = a.z; l.b[3] = a.w; l.b[4] = b.x; l.b[5] = b.y;
  r.b[0] = b.z; r.b[1] = b.w; r.b[2] = c.x; r.b[3] = c.y; r.b[4] = c.z; r.b[5] = c.w;
  l.ref = m.y;
  r.ref = m.z;
  if constexpr (kKarras) {
    l.first = first;
    l.count = (m.y & kIndexMask) - first + 1u;
    r.first = first + l.count;
    r.count = count - l.count;
  } else {
    l.first = r.first = 0u;
    l.count = (l.ref & kLeafFlag) ? 1u : leaf_counts[l.ref];
    r.count = (r.ref & kLeafFlag) ? 1u : leaf_counts[r.ref];
  }
}

// Smallest biased exponent e with o + 254 * 2^(e-127) >= hi (one spare step).
BJ_HD uint32_t grid_exponent(float o, float hi) {
  const float extent = hi - o;
  uint32_t e = 1;
  if (extent > 0.0f) {
    const uint32_t bits = __builtin_bit_cast(uint32_t, extent / 254.0f);
    e = (bits >> 23) & 0xFFu;
    if (bits & 0x7FFFFFu) e += 1;
    if (e < 1) e = 1;
  }
  while (e < 253) {
    const float s = __builtin_bit_cast(float, e << 23);
    if (o + 254.0f * s >= hi) break;
    ++e;
  }
  return e;
}

BJ_HD void quantize(float o, uint32_t e, float lo, float hi, uint8_t& qlo, uint8_t& qhi) {
  const float s = __builtin_bit_cast(float, e << 23);
  const float inv = __builtin_bit_cast(float, (254u - e) << 23);  // exact 2^-(e-127)
  float fl = floorf((lo - o) * inv);
  fl = fl < 0.0f ? 0.0f : (fl > 255.0f ? 255.0f : fl);
  while (fl > 0.0f && o + fl * s > lo) fl -= 1.0f;
  float fh = ceilf((hi - o) * inv);
  fh = fh < 0.0f ? 0.0f : (fh > 255.0f ? 255.0f : fh);
  while (fh < 255.0f && o + fh * s < hi) fh += 1.0f;
  fl = fl > 0.0f ? fl - 1.0f : 0.0f;      // padding: one step below
  fh = fh < 255.0f ? fh + 1.0f : 255.0f;  // and one above
  qlo = (uint8_t)fl;
  qhi = (uint8_t)fh;
}

// Wide node 0's source, written by one thread: the binary root.  `root_dev`
// (H-PLOC: the root its clustering wrote) overrides `root_binary`; a root
// outside the hierarchy raises BAJO_STATUS_COLLAPSE_FAILED and leaves nothing
// to open.  Returns the nodes of level 0 still to be opened.
BJ_D uint32_t collapse_root(const float* __restrict__ scene, uint32_t n, uint32_t root_binary,
                            const uint32_t* __restrict__ root_dev, BjWide* __restrict__ wide,
                            uint32_t* __restrict__ wide_src, uint32_t* __restrict__ ctl,
                            uint32_t* __restrict__ status) {
  ctl[kCtlStatus] = 0;
  if (n == 1) {
    // single triangle: one wide node with one leaf child spanning the scene box
    BjWide w;
    w.ox = scene[0]; w.oy = scene[1]; w.oz = scene[2];
    w.ex = (uint8_t)grid_exponent(scene[0], scene[3]);
    w.ey = (uint8_t)grid_exponent(scene[1], scene[4]);
    w.ez = (uint8_t)grid_exponent(scene[2], scene[5]);
    w.n = 1;
    for (int i = 0; i < 8; ++i) {
      w.lo_x[i] = w.lo_y[i] = w.lo_z[i] = 255;
      w.hi_x[i] = w.hi_y[i] = w.hi_z[i] = 0;
      w.child[i] = 0;
    }
    quantize(scene[0], w.ex, scene[0], scene[3], w.lo_x[0], w.hi_x[0]);
    quantize(scene[1], w.ey, scene[1], scene[4], w.lo_y[0], w.hi_y[0]);
    quantize(scene[2], w.ez, scene[2], scene[5], w.lo_z[0], w.hi_z[0]);
    w.child[0] = kLeafFlag | 0u;
    wide[0] = w;
    return 0;
  }
  const uint32_t root = root_dev ? *root_dev : root_binary;
  if ((root & kLeafFlag) || root >= n - 1) {
    ctl[kCtlStatus] = kStatusBadRoot;
    atomicMax(status, (uint32_t)BAJO_STATUS_COLLAPSE_FAILED);
    return 0;
  }
  wide_src[0] = root;
  return 1;
}

// Segmented builds: wide node s is the root of segment s (S roots form level
// 0).  A one-triangle segment's root is written here, with a single leaf
// child spanning the segment's box; its wide_src entry marks it done.
__global__ void seg_collapse_root_kernel(const float* __restrict__ seg_scene, const uint64_t* __restrict__ off,
                                         uint32_t S, BjWide* __restrict__ wide, uint32_t* __restrict__ wide_src,
                                         uint32_t* __restrict__ ctl) {
  const uint32_t stride = gridDim.x * blockDim.x;
  const uint32_t gtid = blockIdx.x * blockDim.x + threadIdx.x;
  if (gtid == 0) {
    ctl[kCtlStatus] = 0;
    ctl[kCtlCount] = S;
    ctl[kCtlBegin] = 0;
    ctl[kCtlEnd] = S;
  }
  for (uint32_t s = gtid; s < S; s += stride) {
    const uint64_t first = off[s], count = off[s + 1] - first;
    if (count > 1) {
      wide_src[s] = (uint32_t)first;
      continue;
    }
    const float* b = seg_scene + 12 * (uint64_t)s;
    BjWide w;
    w.ox = b[0]; w.oy = b[1]; w.oz = b[2];
    w.ex = (uint8_t)grid_exponent(b[0], b[3]);
    w.ey = (uint8_t)grid_exponent(b[1], b[4]);
    w.ez = (uint8_t)grid_exponent(b[2], b[5]);
    w.n = 1;
    for (int i = 0; i < 8; ++i) {
      w.lo_x[i] = w.lo_y[i] = w.lo_z[i] = 255;
      w.hi_x[i] = w.hi_y[i] = w.hi_z[i] = 0;
      w.child[i] = 0;
    }
    quantize(b[0], w.ex, b[0], b[3], w.lo_x[0], w.hi_x[0]);
    quantize(b[1], w.ey, b[1], b[4], w.lo_y[0], w.hi_y[0]);
    quantize(b[2], w.ez, b[2], b[5], w.lo_z[0], w.hi_z[0]);
    w.child[0] = kLeafFlag | (uint32_t)first;
    wide[s] = w;
    wide_src[s] = kSentinel;
  }
}

// LDS of one block's batch: per-wave totals, then offsets; the range reserved
// for the batch's children.
struct Batch {
  uint32_t wave_total[kCollapseBlock / 64];
  uint32_t first, total;
  uint32_t failed;
};

// Inclusive scan of one value per thread over the block.
BJ_D uint32_t block_inclusive_scan(uint32_t v, uint32_t* __restrict__ wave_total) {
  const uint32_t lane = lane_id(), wave = threadIdx.x >> 6;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(v, off, 64);
    if (lane >= (uint32_t)off) v += y;
  }
  if (lane == 63) wave_total[wave] = v;
  __syncthreads();
  for (uint32_t i = 0; i < wave; ++i) v += wave_total[i];
  __syncthreads();
  return v;
}

// Leaves below a wide node still to be opened (0: opened, or a segment's lone leaf).
BJ_D uint32_t open_leaves(const uint32_t* __restrict__ wide_src, const uint32_t* __restrict__ leaf_counts, uint32_t w) {
  const uint32_t src = wide_src[w];
  return src != kSentinel ? leaf_counts[src] : 0u;
}

// Leaves below the nodes [origin, origin + kKnown) that the first launch has
// reserved, kept in LDS as they are reserved; later ones are looked up.
constexpr uint32_t kKnown = 12288;
struct Leaves {
  uint32_t of[kKnown];
};

// Opens each thread's wide node `w` (where `have`), the whole block together:
// kShared reserves their children with one atomic on
// the node counter (a per-node atomic serializes, about 25 ns each), a lone
// block counts on in bt->first + bt->total and keeps the children's leaves in
// `known`, from `origin` on.  Afterwards [bt->first,
// bt->first + bt->total) are the children to be opened; bt->failed is set if
// they do not fit.
template <bool kKarras, bool kShared>
BJ_D void collapse_batch(const BjNode* __restrict__ bnodes, const uint32_t* __restrict__ leaf_counts,
                         BjWide* __restrict__ wide, uint32_t* __restrict__ wide_src, uint32_t* __restrict__ ctl,
                         uint32_t capacity, uint32_t max_leaf, int max_children, uint32_t w, bool have,
                         Batch* __restrict__ bt, Leaves* __restrict__ known = nullptr, uint32_t origin = 0) {
  const uint32_t lane = lane_id();
  const uint32_t wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  {
    const uint32_t src = have ? wide_src[w] : kSentinel;
    const bool active = src != kSentinel;
    // The children live in registers: every index into ch[] is a compile-time
    // constant (a data-dependent one would place the array in scratch memory).
    // A lane that still opens children in step k has k + 2 of them, so the
    // right child's slot is a constant and only the opened child's slot is
    // selected.  A child's area is formed once, when it is loaded.
    Child ch[8];
    float area[8];
    int n = 0;
    if (active) {
      uint32_t count = 0, first = 0;
      if constexpr (kKarras) {
        count = leaf_counts[src];
        first = bnodes[src].fence + 1u - count;
      }
      load_children<kKarras>(bnodes, leaf_counts, src, first, count, ch[0], ch[1]);
      area[0] = half_area(ch[0].b);
      area[1] = half_area(ch[1].b);
      n = 2;
    }
#pragma unroll
    for (int k = 2; k < 8; ++k) {
      if (k < max_children && n == k) {
        // the largest child too big for a leaf, else the largest inner child
        // (the first of equal ones)
        int pick = -1, pick1 = -1;
        float best = -1.0f, best1 = -1.0f;
#pragma unroll
        for (int i = 0; i < k; ++i) {
          const bool inner = !(ch[i].ref & kLeafFlag) && ch[i].count >= 2;
          if (inner && ch[i].count > max_leaf && area[i] > best) {
            best = area[i];
            pick = i;
          }
          if (inner && area[i] > best1) {
            best1 = area[i];
            pick1 = i;
          }
        }
        if (pick < 0) pick = pick1;
        if (pick >= 0) {
          uint32_t pick_ref = ch[0].ref, pick_first = ch[0].first, pick_count = ch[0].count;
#pragma unroll
          for (int i = 1; i < k; ++i) {
            pick_ref = i == pick ? ch[i].ref : pick_ref;
            pick_first = i == pick ? ch[i].first : pick_first;
            pick_count = i == pick ? ch[i].count : pick_count;
          }
          Child l;
          load_children<kKarras>(bnodes, leaf_counts, pick_ref, pick_first, pick_count, l, ch[k]);
          const float al = half_area(l.b);
          area[k] = half_area(ch[k].b);
#pragma unroll
          for (int i = 0; i < k; ++i) {
            if (i == pick) {
              ch[i] = l;
              area[i] = al;
            }
          }
          n = k + 1;
        }
      }
    }
    // reserve wide nodes for inner children that stay inner (wave-aggregated)
    uint32_t k = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i < n && !(ch[i].ref & kLeafFlag) && ch[i].count > max_leaf) ++k;
    uint32_t incl = k;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = __shfl_up(incl, off, 64);
      if (lane >= (uint32_t)off) incl += y;
    }
    if (lane == 63) bt->wave_total[wave] = incl;
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t sum = 0;
      for (uint32_t i = 0; i < waves; ++i) {
        const uint32_t t = bt->wave_total[i];
        bt->wave_total[i] = sum;
        sum += t;
      }
      if constexpr (kShared) bt->first = sum ? atomicAdd(ctl + kCtlCount, sum) : 0u;
      else bt->first += bt->total;
      bt->total = sum;
      bt->failed = (uint64_t)bt->first + sum > capacity ? 1u : 0u;
    }
    __syncthreads();
    if (!active || bt->failed) return;
    const uint32_t first = bt->first + bt->wave_total[wave] + (incl - k);
    // node box and per-axis grids
    float box[6] = {kFltMax, kFltMax, kFltMax, -kFltMax, -kFltMax, -kFltMax};
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i < n)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          box[a] = fmin_sel(box[a], ch[i].b[a]);
          box[a + 3] = fmax_sel(box[a + 3], ch[i].b[a + 3]);
        }
    const uint32_t e[3] = {grid_exponent(box[0], box[3]), grid_exponent(box[1], box[4]),
                           grid_exponent(box[2], box[5])};
    // packed byte planes: lo_x, lo_y, lo_z, hi_x, hi_y, hi_z, two words each
    uint32_t q[12];
#pragma unroll
    for (int j = 0; j < 12; ++j) q[j] = j < 6 ? 0xFFFFFFFFu : 0u;
    uint32_t child[8];
    uint32_t next = first;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      child[i] = 0;
      if (i < n) {
        const int word = i >> 2, shift = 8 * (i & 3);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          uint8_t ql, qh;
          quantize(box[a], e[a], ch[i].b[a], ch[i].b[a + 3], ql, qh);
          q[2 * a + word] = (q[2 * a + word] & ~(0xFFu << shift)) | ((uint32_t)ql << shift);
          q[6 + 2 * a + word] |= (uint32_t)qh << shift;
        }
        const uint32_t ref = ch[i].ref;
        if (ref & kLeafFlag) {
          child[i] = kLeafFlag | (ref & kIndexMask);  // one triangle
        } else if (ch[i].count <= max_leaf) {
          // inner binary node over sorted range [fence - count + 1, fence]
          const uint32_t start = kKarras ? ch[i].first : bnodes[ref].fence + 1u - ch[i].count;
          child[i] = kLeafFlag | ((ch[i].count - 1u) << 28) | start;
        } else {
          child[i] = next;
          wide_src[next] = ref;
          if constexpr (!kShared)
            if (next - origin < kKnown) known->of[next - origin] = ch[i].count;
          ++next;
        }
      }
    }
    const uint32_t meta = e[0] | (e[1] << 8) | (e[2] << 16) | ((uint32_t)n << 24);
    uint4* dst = reinterpret_cast<uint4*>(wide + w);
    dst[0] = make_uint4(__builtin_bit_cast(uint32_t, box[0]), __builtin_bit_cast(uint32_t, box[1]),
                        __builtin_bit_cast(uint32_t, box[2]), meta);
    dst[1] = make_uint4(q[0], q[1], q[2], q[3]);
    dst[2] = make_uint4(q[4], q[5], q[6], q[7]);
    dst[3] = make_uint4(q[8], q[9], q[10], q[11]);
    dst[4] = make_uint4(child[0], child[1], child[2], child[3]);
    dst[5] = make_uint4(child[4], child[5], child[6], child[7]);
  }
}

// The first levels, in one block.  `segmented`: level 0 (the segment roots)
// is already in ctl.  Opens whole levels until one holds more nodes than the
// block has threads, then nodes with more than `share` leaves (their subtrees
// are disjoint, so fewer than n / share at a time).  Leaves the range that
// holds the nodes still to be opened (or an empty range) in ctl, and how it is
// dealt: every `blocks`-th node to a block if that is even (kCtlRuns 0), else
// runs of equal numbers of leaves, in deal[0 .. blocks].
template <bool kKarras>
__global__ void __launch_bounds__(kCollapseBlock)
collapse_top_kernel(const BjNode* __restrict__ bnodes, const uint32_t* __restrict__ leaf_counts,
                    BjWide* __restrict__ wide, uint32_t* __restrict__ wide_src, uint32_t* __restrict__ ctl,
                    uint32_t capacity, uint32_t max_leaf, int max_children, const float* __restrict__ scene,
                    uint32_t n, uint32_t root_binary, const uint32_t* __restrict__ root_dev, int segmented,
                    uint32_t share, uint32_t* __restrict__ deal, uint32_t blocks, uint32_t* __restrict__ status) {
  __shared__ Batch bt;
  __shared__ Leaves known;
  __shared__ uint32_t s_list[kCollapseBlock], s_word;
  const uint32_t t = threadIdx.x;
  // the level being opened is [bt.first, bt.first + bt.total)
  if (t == 0) {
    bt.first = 0;
    bt.total = segmented ? ctl[kCtlEnd] : collapse_root(scene, n, root_binary, root_dev, wide, wide_src, ctl, status);
    bt.failed = 0;
  }
  __threadfence_block();
  __syncthreads();
  uint32_t level = 0, begin = 0;  // begin: of the nodes still to be opened
  bool levels = true;             // whole levels so far
  const auto leaves_of = [&](uint32_t i) {
    return i < kKnown ? known.of[i] : open_leaves(wide_src, leaf_counts, begin + i);
  };
  for (;;) {
    const uint32_t first = bt.first, len = bt.total;
    if (len == 0 || bt.failed || level == kLevelCap) break;
    uint32_t w = first + t, origin = first + len;
    bool have = t < len;
    if (levels && len > kCollapseBlock) {
      levels = false;
      begin = first;
      if (level == 0)  // segment roots
#pragma unroll 1
        for (uint32_t i = t; i < len && i < kKnown; i += kCollapseBlock)
          known.of[i] = open_leaves(wide_src, leaf_counts, begin + i);
    }
    if (!levels) {
      // the last range's nodes above a share
      if (t == 0) s_word = 0;
      __syncthreads();
#pragma unroll 1
      for (uint32_t i = t; i < len; i += kCollapseBlock)
        if (leaves_of(first - begin + i) > share) {
          const uint32_t at = atomicAdd(&s_word, 1u);
          if (at < kCollapseBlock) s_list[at] = first + i;
        }
      __syncthreads();
      if (s_word == 0) break;
      have = t < s_word;
      w = have ? s_list[t] : first;
      origin = begin;
    }
    ++level;
    __syncthreads();
    collapse_batch<kKarras, false>(bnodes, leaf_counts, wide, wide_src, ctl, capacity, max_leaf, max_children, w,
                                   have, &bt, &known, origin);
    if (!levels && have) {
      wide_src[w] = kSentinel;
      if (w - begin < kKnown) known.of[w - begin] = 0;
    }
    __threadfence_block();
    __syncthreads();
  }
  if (levels) begin = bt.first;
  const bool failed = bt.failed || (bt.total != 0 && level == kLevelCap);
  const uint32_t len = failed ? 0u : bt.first + bt.total - begin;  // from `begin` on
  // whether a block's share is too large when the nodes are dealt by number
  uint32_t load = 0;
  if (t < blocks)
#pragma unroll 1
    for (uint32_t i = t; i < len; i += blocks) load += leaves_of(i);
  const bool runs = __syncthreads_or(load > share + share / 8) != 0;
  if (runs) {
    // node i belongs to block (leaves before i) * blocks / n
    constexpr uint32_t kEach = 8;
    uint32_t carry = 0;
    for (uint32_t base = 0; base < len; base += kEach * kCollapseBlock) {
      const uint32_t mine = base + kEach * t;
      uint32_t leaves[kEach], sum = 0;
#pragma unroll
      for (uint32_t i = 0; i < kEach; ++i) {
        leaves[i] = mine + i < len ? leaves_of(mine + i) : 0u;
        sum += leaves[i];
      }
      const uint32_t incl = block_inclusive_scan(sum, bt.wave_total);
      uint32_t before = carry + incl - sum;
#pragma unroll
      for (uint32_t i = 0; i < kEach; ++i) {
        const uint32_t a = (uint32_t)((uint64_t)before * blocks / n);
        const uint32_t b = (uint32_t)((uint64_t)(before + leaves[i]) * blocks / n);
        for (uint32_t k = a + 1; k <= b && k <= blocks; ++k) deal[k] = begin + mine + i + 1;
        before += leaves[i];
      }
      if (t == kCollapseBlock - 1) s_word = before;
      __syncthreads();
      carry = s_word;
      __syncthreads();
    }
    if (t == 0) {
      deal[0] = begin;
      for (uint32_t k = (uint32_t)((uint64_t)carry * blocks / n) + 1; k <= blocks; ++k) deal[k] = begin + len;
    }
  }
  if (t == 0) {
    if (failed) {
      ctl[kCtlStatus] = bt.failed ? kStatusOutOfNodes : kStatusTooDeep;
      atomicMax(status, (uint32_t)BAJO_STATUS_COLLAPSE_FAILED);
    }
    const uint32_t end = failed ? bt.first : begin + len;
    ctl[kCtlBegin] = end - len;
    ctl[kCtlEnd] = end;
    ctl[kCtlRuns] = runs ? 1u : 0u;
    // a build without nodes to open still has its root record
    ctl[kCtlCount] = end > 0 ? end : 1u;
  }
}

// Every level left, one subtree after another in each block.
template <bool kKarras>
__global__ void __launch_bounds__(kCollapseBlock)
collapse_subtree_kernel(const BjNode* __restrict__ bnodes, const uint32_t* __restrict__ leaf_counts,
                        BjWide* __restrict__ wide, uint32_t* __restrict__ wide_src, uint32_t* __restrict__ ctl,
                        uint32_t capacity, uint32_t max_leaf, int max_children, const uint32_t* __restrict__ deal,
                        uint32_t* __restrict__ status) {
  __shared__ Batch bt;
  __shared__ uint32_t s_first[kLevelCap], s_len[kLevelCap];
  const uint32_t begin = ctl[kCtlBegin], end = ctl[kCtlEnd];
  if (begin == end) return;
  // the block's nodes: share + stride * i, i < count; the bottom of the stack
  // holds the range of i still to be opened, what lies above it node ranges
  uint32_t share = begin + blockIdx.x, stride = gridDim.x, count = 0;
  if (ctl[kCtlRuns]) {
    share = deal[blockIdx.x];
    stride = 1;
    count = deal[blockIdx.x + 1] - share;
  } else if (share < end) {
    count = (end - share + stride - 1) / stride;
  }
  if (count == 0) return;
  if (threadIdx.x == 0) {
    s_first[0] = 0;
    s_len[0] = count;
  }
  __syncthreads();
  int depth = 1, bottom = 1;
  while (depth > 0) {
    // the next batch: up to a block's worth of the range on top
    const uint32_t first = s_first[depth - 1], range = s_len[depth - 1];
    const uint32_t len = range < blockDim.x ? range : blockDim.x;
    const uint32_t w = depth == bottom ? share + stride * (first + threadIdx.x) : first + threadIdx.x;
    __syncthreads();
    if (len == range) {
      if (depth == bottom) bottom = 0;
      --depth;
    } else if (threadIdx.x == 0) {
      s_first[depth - 1] = first + len;
      s_len[depth - 1] = range - len;
    }
    collapse_batch<kKarras, true>(bnodes, leaf_counts, wide, wide_src, ctl, capacity, max_leaf, max_children, w,
                                  threadIdx.x < len, &bt);
    __threadfence_block();
    __syncthreads();
    const bool full = bt.total != 0 && depth == (int)kLevelCap;
    if (bt.failed || full) {
      if (threadIdx.x == 0) {
        atomicOr(ctl + kCtlStatus, full ? kStatusTooDeep : kStatusOutOfNodes);
        atomicMax(status, (uint32_t)BAJO_STATUS_COLLAPSE_FAILED);
      }
      return;
    }
    if (bt.total != 0) {
      if (threadIdx.x == 0) {
        s_first[depth] = bt.first;
        s_len[depth] = bt.total;
      }
      ++depth;
    }
    __syncthreads();
  }
}

template <bool kKarras>
void launch_collapse(bajo_ctx* ctx, bajo_bvh* h, const uint32_t* root_dev, unsigned blocks) {
  const uint32_t n = (uint32_t)h->n, capacity = (uint32_t)h->wide_capacity;
  // a subtree of up to kSmallSubtree leaves is a few batches of one block
  const uint32_t share = n / blocks > kSmallSubtree ? n / blocks : kSmallSubtree;
  uint32_t* deal = static_cast<uint32_t*>(h->hands);  // free once the binary hierarchy stands
  collapse_top_kernel<kKarras><<<1, kCollapseBlock, 0, ctx->stream>>>(
      h->nodes, h->leaf_counts, h->wide, h->wide_src, h->wide_ctl, capacity, h->wide_leaf, h->node_width, h->scene, n,
      n > 1 ? h->root : 0u, root_dev, h->seg_count ? 1 : 0, share, deal, blocks, ctx->status);
  if (n <= kCollapseBlock && !h->seg_count) return;  // no level can outgrow the first launch
  collapse_subtree_kernel<kKarras><<<blocks, kCollapseBlock, 0, ctx->stream>>>(
      h->nodes, h->leaf_counts, h->wide, h->wide_src, h->wide_ctl, capacity, h->wide_leaf, h->node_width, deal,
      ctx->status);
}

}  // namespace

// Builds the W-wide layout of h from its binary hierarchy.  Enqueue-only: the
// host reads nothing back (the node count is read at the first host query,
// H-PLOC's root comes from the device).
int32_t collapse_wide(bajo_ctx* ctx, bajo_bvh* h) {
  hipStream_t st = ctx->stream;
  const uint32_t n = (uint32_t)h->n;
  int dev = 0, cus = 0;
  BJ_HIP(hipGetDevice(&dev));
  BJ_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const uint32_t* root_dev = nullptr;
  if (h->seg_count) {
    const uint32_t S = h->seg_count;
    seg_collapse_root_kernel<<<div_up(S, 256u) < 1024u ? div_up(S, 256u) : 1024u, 256, 0, st>>>(
        h->seg_scene, h->seg_off, S, h->wide, h->wide_src, h->wide_ctl);
    BJ_HIP(hipGetLastError());
  } else if (n > 1 && h->root_on_device) {
    root_dev = h->hp_ctl + kHpCtlRoot;
  }
  const unsigned blocks = (unsigned)cus < kMostBlocks ? (unsigned)cus : kMostBlocks;
  if (h->method == BAJO_BUILD_HPLOC) launch_collapse<false>(ctx, h, root_dev, blocks);
  else launch_collapse<true>(ctx, h, root_dev, blocks);
  BJ_HIP(hipGetLastError());
  h->wide_pending = !(n == 1 && !h->seg_count);
  if (!h->wide_pending) h->wide_count = 1;
  return BAJO_OK;
}

// The node count the last collapse left in wide_ctl (clipped to the capacity).
uint32_t collapse_read_count(const uint32_t* host_ctl, uint64_t capacity) {
  const uint32_t c = host_ctl[kCtlCount];
  return (uint64_t)c > capacity ? (uint32_t)capacity : c;
}

}  // namespace bj

// Closest-hit / any-hit ray launches over the binary or 8-wide BVH (gfx950).
//
// Replaces GpuTriangleBvh.launch_rays / launch_camera /
// launch_camera_instrumented (bvh/gpu/triangle_bvh.mojo:520-614,730-863) and
// the near-first loop of bvh/gpu/trace.mojo:341-552 with its leaf test
// (bvh/gpu/triangle_bvh.mojo:866-959, determinant-scaled Moller-Trumbore in
// FP32, normal = normalize(e1 x e2)).
//
// MI355X design:
//   - persistent waves: the grid is sized to the resident capacity and each
//     wave fetches 64-ray batches from an atomic counter, so the divergent
//     tail of one batch never idles a whole CU;
//   - nodes are 64 B (both child boxes + children) read with four 16-byte
//     loads; sorted leaf triangles are 48 B (three 16-byte loads);
//   - each lane's traversal stack lives in LDS, laid out depth-major across
//     the block so lanes at any depth hit distinct banks.  Entries deeper
//     than kLdsStack spill to a per-thread global area; the Karras hierarchy
//     over 64-bit (code, index) keys is at most 64 levels deep, so 64 entries
//     always suffice.
#include "traverse.h"
#include "rt_math.h"

namespace bj {
namespace {

// Batched camera launches over a BLAS set: camera view e traces segment e,
// whose root follows from the segment offsets (one-triangle segments are a
// single leaf; an 8-wide segment's root is wide node e).
template <bool kWide>
BJ_D uint32_t segment_root(const uint64_t* __restrict__ off, uint64_t e) {
  if constexpr (kWide) return (uint32_t)e;
  const uint64_t first = off[e];
  return off[e + 1] - first == 1 ? (kLeafFlag | (uint32_t)first) : (uint32_t)first;
}

template <int kMode, bool kStats, bool kCamera, bool kWide, bool kSeg, bool kSph>
__global__ void __launch_bounds__(kTraceBlock) trace_kernel(const AccelView av,
                                                            const float* __restrict__ rays,
                                                            const float* __restrict__ cams, uint32_t cam_w,
                                                            uint32_t cam_h, float inv_height,
                                                            float* __restrict__ hits, uint64_t R,
                                                            uint32_t* __restrict__ stats,
                                                            uint32_t* __restrict__ counter,
                                                            uint32_t* __restrict__ spill,
                                                            const uint64_t* __restrict__ seg_off) {
  __shared__ uint32_t s_stack[kLdsStack * kTraceBlock];
  const uint32_t lane = lane_id();
  const uint64_t gtid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  Stack st{s_stack + threadIdx.x, spill + gtid, (uint64_t)gridDim.x * blockDim.x, 0};

  // Batches of 64 rays per atomic while the launch is short; up to eight
  // batches per fetch when every wave would otherwise fetch 8+ times.
  const uint64_t waves = (uint64_t)gridDim.x * (kTraceBlock / 64);
  uint64_t kb = R / (waves * 64u * 8u);
  const uint32_t batch = 64u * (uint32_t)(kb < 1 ? 1 : (kb > 8 ? 8 : kb));
  for (uint32_t base = 0, off = batch;;) {
    if (off >= batch) {
      if (lane == 0) base = atomicAdd(counter, batch);
      base = __shfl(base, 0, 64);
      off = 0;
    }
    if ((uint64_t)base + off >= R) break;
    const uint64_t r = (uint64_t)base + off + lane;
    off += 64;
    if (r >= R) continue;

    Ray ray;
    if constexpr (kCamera) {
      ray = camera_ray(cams, r, cam_w, cam_h, inv_height);
    } else {
      ray.o = mk(rays[0 * R + r], rays[1 * R + r], rays[2 * R + r]);
      ray.tmin = rays[3 * R + r];
      ray.d = mk(rays[4 * R + r], rays[5 * R + r], rays[6 * R + r]);
      ray.tmax = rays[7 * R + r];
    }
    TraceCounters tc;
    AccelView v = av;
    if constexpr (kSeg) {
      const uint32_t root = segment_root<kWide>(seg_off, r / ((uint64_t)cam_w * cam_h));
      if constexpr (kWide) v.wide.root = root;
      else v.bin.root = root;
    }
    Hit hit = trace_accel<kMode, kStats, kWide, kSph>(v, ray, st, &tc);
    store_hit(hits, r, hit);
    if constexpr (kStats) {
      uint32_t* s = stats + 5 * r;
      s[0] = tc.visits; s[1] = tc.inner; s[2] = 0; s[3] = tc.leaves; s[4] = tc.max_sp;
    }
  }
}

// 8-wide launches keep every lane busy: a lane whose ray is finished takes a
// new one as soon as a quarter of the wave is idle, instead of idling until
// the slowest ray of its batch ends (random rays differ in node visits by an
// order of magnitude, so fixed 64-ray batches left most lanes idle).  Each
// wave reserves kRefillChunk ray indices per atomic and hands them to idle
// lanes in lane order; one node visit per loop iteration.
constexpr uint32_t kRefillLanes = 16;
constexpr uint32_t kRefillChunk = 256;

template <int kMode, bool kStats, bool kCamera, bool kSeg, bool kSph>
__global__ void __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(6))) trace_refill_kernel(const WideView wv, const float* __restrict__ rays,
                                                                   const float* __restrict__ cams, uint32_t cam_w,
                                                                   uint32_t cam_h, float inv_height,
                                                                   float* __restrict__ hits, uint64_t R,
                                                                   uint32_t* __restrict__ stats,
                                                                   uint32_t* __restrict__ counter,
                                                                   uint32_t* __restrict__ spill,
                                                                   const uint64_t* __restrict__ seg_off) {
  __shared__ uint32_t s_stack[kLdsStack * kTraceBlock];
  const uint32_t lane = lane_id();
  const uint64_t gtid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  Stack st{s_stack + threadIdx.x, spill + gtid, (uint64_t)gridDim.x * blockDim.x, 0};
  Walk8<kMode, kStats, kSph> w;
  w.cur = kSentinel;
  bool active = false, drained = false;
  uint64_t r = 0, next = 0, stop = 0;  // the wave's reserved, not yet assigned indices [next, stop)
  // short launches are spread one 64-ray batch per wave, long ones take up to
  // kRefillChunk rays per atomic
  const uint64_t waves = ((uint64_t)gridDim.x * blockDim.x) >> 6;
  const uint64_t per_wave = (R / waves + 63u) & ~63ull;
  const uint32_t chunk = per_wave < 64u ? 64u : (per_wave > kRefillChunk ? kRefillChunk : (uint32_t)per_wave);
  for (;;) {
    const uint64_t idle = ballot(!active);
    const uint32_t n_idle = (uint32_t)__builtin_popcountll(idle);
    if (!drained && n_idle >= kRefillLanes) {
      if (next >= stop) {
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(counter, chunk);
        base = __shfl(base, 0, 64);
        next = base;
        stop = (uint64_t)base + chunk < R ? (uint64_t)base + chunk : R;
        if ((uint64_t)base >= R) drained = true;
      }
      if (next < stop) {
        const uint64_t mine = next + mask_rank(idle);
        if (!active && mine < stop) {
          r = mine;
          Ray ray;
          if constexpr (kCamera) {
            ray = camera_ray(cams, r, cam_w, cam_h, inv_height);
          } else {
            ray.o = mk(rays[0 * R + r], rays[1 * R + r], rays[2 * R + r]);
            ray.tmin = rays[3 * R + r];
            ray.d = mk(rays[4 * R + r], rays[5 * R + r], rays[6 * R + r]);
            ray.tmax = rays[7 * R + r];
          }
          if constexpr (kSeg) {
            WideView sv = wv;
            sv.root = segment_root<true>(seg_off, r / ((uint64_t)cam_w * cam_h));
            w.begin(sv, ray, st);
          } else {
            w.begin(wv, ray, st);
          }
          active = true;
        }
        next = next + n_idle < stop ? next + n_idle : stop;
      }
    }
    if (!ballot(active)) {
      if (drained) break;
      continue;
    }
    if (active) {
      if (!w.done()) w.step(wv, st);
      if (w.done()) {
        TraceCounters tc;
        store_hit(hits, r, w.finish(wv, &tc));
        if constexpr (kStats) {
          uint32_t* sp = stats + 5 * r;
          sp[0] = tc.visits; sp[1] = tc.inner; sp[2] = 0; sp[3] = tc.leaves; sp[4] = tc.max_sp;
        }
        active = false;
      }
    }
  }
}

// Short launches: G lanes per ray (OrderedWalk8, GroupWalk8 or GroupWalk2),
// each group taking every `groups`-th ray.  With one lane per ray a launch
// lasts as long as its slowest lane's chain of node and record loads, whatever
// its size: 4,096 closest-hit rays through a 65,536-triangle soup took 377 us
// at widths 2 and 8; with 32 (binary) or 64 (8-wide) lanes per ray 43 and 27.
// Five waves per SIMD: the walk holds about 85 VGPRs, the rare fallback more.
template <int kMode, bool kCamera, bool kWide, bool kSeg, int G>
__global__ void __launch_bounds__(kTraceBlock) __attribute__((amdgpu_waves_per_eu(5)))
trace_group_kernel(const AccelView av, const float* __restrict__ rays,
                                                                  const float* __restrict__ cams, uint32_t cam_w,
                                                                  uint32_t cam_h, float inv_height,
                                                                  float* __restrict__ hits, uint64_t R,
                                                                  const uint64_t* __restrict__ seg_off) {
  constexpr bool kAny = kMode == BAJO_TRACE_ANY_HIT;
  constexpr int kGroups = kTraceBlock / G;
  using Walk = std::conditional_t<kWide, Wide8<G < 8 ? 8 : G, kAny>, GroupWalk2<G, kAny>>;
  __shared__ uint32_t s_stack[kGroups][Walk::kStackWords];
  __shared__ uint32_t s_recs[kWide ? kGroups : 1][kWide ? Wide8<G < 8 ? 8 : G, kAny>::kRecs : 1];
  const uint32_t grp = threadIdx.x / G, gl = lane_id() % G;
  uint32_t* stack = s_stack[grp];
  uint32_t* recs = s_recs[kWide ? grp : 0];
  const uint64_t groups = (uint64_t)gridDim.x * kGroups;
  uint64_t r = (uint64_t)blockIdx.x * kGroups + grp;
  AccelView v = av;
  Walk walk;
  // A finished ray's record and the next ray's start cost a few loads that the
  // other groups of the wave would wait for, so they are done once a quarter
  // of the groups are finished or none is left walking (262,144 closest-hit
  // rays, 8 lanes each: 279 us against 294 with every group on its own).
  constexpr uint32_t kRefill = G < 16 ? 64 / G / 4 : 1;
  bool have = false, walking = false;
  uint32_t visits = 0, tests = 0;
  for (;;) {
    const uint64_t busy = ballot(walking);
    if (64u - (uint32_t)__builtin_popcountll(busy) >= kRefill * G || busy == 0) {
      if (have && !walking) {
        Hit h;
        if constexpr (kWide) {
          h = walk.finish(v.wide, stack, recs, visits, tests);
          if (gl == 0) store_hit(hits, r, h);
        } else if (gl == 0) {
          store_hit(hits, r, walk.finish(v.bin, stack));
        }
        have = false;
        r += groups;
      }
      if (!have && r < R) {
        Ray ray;
        if constexpr (kCamera) {
          ray = camera_ray(cams, r, cam_w, cam_h, inv_height);
        } else {
          ray.o = mk(rays[0 * R + r], rays[1 * R + r], rays[2 * R + r]);
          ray.tmin = rays[3 * R + r];
          ray.d = mk(rays[4 * R + r], rays[5 * R + r], rays[6 * R + r]);
          ray.tmax = rays[7 * R + r];
        }
        if constexpr (kSeg) {
          const uint32_t root = segment_root<kWide>(seg_off, r / ((uint64_t)cam_w * cam_h));
          if constexpr (kWide) v.wide.root = root;
          else v.bin.root = root;
        }
        if constexpr (kWide) walk.begin(v.wide, ray);
        else walk.begin(v.bin, ray);
        have = walking = true;
      }
      if (ballot(have) == 0) break;  // every group of the wave is out of rays
    }
    if (walking) {
      if constexpr (kWide) walking = !walk.step(v.wide, stack, recs, visits, tests);
      else walking = !walk.step(v.bin, stack);
    }
  }
}

__global__ void trace_init_kernel(uint32_t* counter, uint32_t* status) {
  if (threadIdx.x == 0) { *counter = 0; *status = 0; }
}

struct TraceScratch {
  uint32_t* counter;
  uint32_t* status;
  uint32_t* spill;
  unsigned grid;
};

template <int kMode, bool kStats, bool kCamera, bool kWide, bool kSeg, bool kSph>
int32_t occupancy_grid(unsigned* grid) {
  static unsigned cached = 0;
  if (!cached) {
    int dev = 0, cus = 0, per_cu = 0;
    BJ_HIP(hipGetDevice(&dev));
    BJ_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    if constexpr (kWide)
      BJ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, trace_refill_kernel<kMode, kStats, kCamera, kSeg, kSph>,
                                                          kTraceBlock, 0));
    else
      BJ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu,
                                                          trace_kernel<kMode, kStats, kCamera, kWide, kSeg, kSph>,
                                                          kTraceBlock, 0));
    if (per_cu < 1) per_cu = 1;
    cached = (unsigned)(cus * per_cu);
  }
  *grid = cached;
  return BAJO_OK;
}

// Lanes per ray of a launch of R rays (1: the per-lane kernels).  More lanes
// shorten the serial chain of a ray but spend more instructions on it, so
// each width pays until the chip is full.  Measured over 65,536-triangle and
// 1M-triangle soups and 100K / 4M-triangle closed meshes, random and camera
// rays (us, one lane per ray against the choice): 8-wide closest 16,384 rays
// 343 -> 64, 65,536: 293 -> 137, 131,072: 332 -> 249, 262,144: 433 -> 458;
// 8-wide any 16,384: 194 -> 31, 131,072: 214 -> 165, 262,144: 289 -> 306;
// binary closest 4,096: 377 -> 43, 16,384: 395 -> 66, 65,536: 405 -> 160,
// 131,072: 437 -> 306, 262,144: 515 -> 475, 524,288: 471 -> 622 (camera).
// Rays through few triangles have short chains, and the wider form stops
// paying earlier: 22,000 camera rays over a 300-triangle ball 36 us with one
// lane, 46 with 64 and 17 with 8 (12,000 triangles 99, 66 and 34; a million
// scattered 582, 98 and 175); binary, 95,000 rays, 57 us with one lane, 75
// with 8 and 58 with 4 (12,000 triangles 145, 127, 116; a million 907, 361,
// 616 closest).  The last limits are a mean over the hierarchies' sizes: just
// below them 30,000 scattered triangles lose (8-wide, 190,000 rays 275 us with
// one lane, 309 with 8; binary, 290,000 camera rays 280 and 307) and small and
// large ones gain (500: 80 and 42; a million, binary: 966 and 717).
constexpr uint64_t kFewTriangles = 16384;
int lanes_per_ray(bool wide, bool any, uint64_t R, uint64_t triangles) {
  const bool few = triangles <= kFewTriangles;
  if (wide) {
    if (R <= (any ? 32768u : few ? 12288u : 24576u)) return 64;
    return R <= 196608u ? (any ? 16 : 8) : 1;
  }
  if (R <= 8192u) return 32;
  if (R <= 32768u) return 16;
  if (R <= (few ? 65536u : 98304u)) return 8;
  return R <= (any ? 196608u : 294912u) ? 4 : 1;
}

// A launch with G lanes per ray on its resident blocks.
template <int kMode, bool kCamera, bool kWide, bool kSeg, int G>
int32_t launch_groups(bajo_ctx* ctx, const bajo_bvh* h, const float* rays, const float* cams, uint32_t w, uint32_t hh,
                      float* hits, uint64_t R) {
  static unsigned resident = 0;
  if (!resident) {
    int dev = 0, cus = 0, per_cu = 0;
    BJ_HIP(hipGetDevice(&dev));
    BJ_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    BJ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, trace_group_kernel<kMode, kCamera, kWide, kSeg, G>,
                                                        kTraceBlock, 0));
    resident = (unsigned)(cus * (per_cu < 1 ? 1 : per_cu));
  }
  const uint64_t need = (R * G + kTraceBlock - 1) / kTraceBlock;
  const unsigned grid = need < resident ? (unsigned)need : resident;
  void* scratch = nullptr;
  const int32_t rc = ctx_scratch(ctx, 256, &scratch);
  if (rc) return rc;
  const AccelView av = accel_view(h, (uint32_t*)scratch);
  trace_group_kernel<kMode, kCamera, kWide, kSeg, G><<<grid, kTraceBlock, 0, ctx->stream>>>(
      av, rays, cams, w, hh, hh ? 1.0f / (float)hh : 0.0f, hits, R, kSeg ? h->seg_off : nullptr);
  BJ_HIP(hipGetLastError());
  return BAJO_OK;
}

template <int kMode, bool kStats, bool kCamera, bool kWide, bool kSeg = false, bool kSph = false>
int32_t launch_width(bajo_ctx* ctx, const bajo_bvh* h, const float* rays, const float* cams, uint32_t w, uint32_t hh,
                     float* hits, uint64_t R, uint32_t* stats) {
  if constexpr (!kStats && !kSph) {
    switch (lanes_per_ray(kWide, kMode == BAJO_TRACE_ANY_HIT, R, h->n)) {
      case 4:
        if constexpr (!kWide) return launch_groups<kMode, kCamera, kWide, kSeg, 4>(ctx, h, rays, cams, w, hh, hits, R);
        break;
      case 8:
        if constexpr (!kWide || kMode == BAJO_TRACE_CLOSEST_HIT)
          return launch_groups<kMode, kCamera, kWide, kSeg, 8>(ctx, h, rays, cams, w, hh, hits, R);
        break;
      case 16:
        if constexpr (!kWide || kMode == BAJO_TRACE_ANY_HIT)
          return launch_groups<kMode, kCamera, kWide, kSeg, 16>(ctx, h, rays, cams, w, hh, hits, R);
        break;
      case 32:
        if constexpr (!kWide) return launch_groups<kMode, kCamera, kWide, kSeg, 32>(ctx, h, rays, cams, w, hh, hits, R);
        break;
      case 64:
        if constexpr (kWide) return launch_groups<kMode, kCamera, kWide, kSeg, 64>(ctx, h, rays, cams, w, hh, hits, R);
        break;
      default: break;
    }
  }
  unsigned grid = 0;
  int32_t rc = occupancy_grid<kMode, kStats, kCamera, kWide, kSeg, kSph>(&grid);
  if (rc) return rc;
  uint64_t need_blocks = (R + kTraceBlock - 1) / kTraceBlock;
  if ((uint64_t)grid > need_blocks) grid = (unsigned)need_blocks;
  if (grid < 1) grid = 1;
  const uint64_t threads = (uint64_t)grid * kTraceBlock;
  void* scratch = nullptr;
  rc = ctx_scratch(ctx, 256 + threads * kSpill * sizeof(uint32_t), &scratch);
  if (rc) return rc;
  uint32_t* counter = (uint32_t*)scratch;
  uint32_t* status = counter + 1;
  uint32_t* spill = (uint32_t*)((char*)scratch + 256);
  trace_init_kernel<<<1, 64, 0, ctx->stream>>>(counter, status);
  const AccelView av = accel_view(h, status);
  const uint64_t* seg_off = kSeg ? h->seg_off : nullptr;
  if constexpr (kWide)
    trace_refill_kernel<kMode, kStats, kCamera, kSeg, kSph><<<grid, kTraceBlock, 0, ctx->stream>>>(
        av.wide, rays, cams, w, hh, hh ? 1.0f / (float)hh : 0.0f, hits, R, stats, counter, spill, seg_off);
  else
    trace_kernel<kMode, kStats, kCamera, kWide, kSeg, kSph><<<grid, kTraceBlock, 0, ctx->stream>>>(
        av, rays, cams, w, hh, hh ? 1.0f / (float)hh : 0.0f, hits, R, stats, counter, spill, seg_off);
  BJ_HIP(hipGetLastError());
  return BAJO_OK;
}

template <int kMode, bool kStats, bool kCamera>
int32_t launch(bajo_ctx* ctx, const bajo_bvh* h, const float* rays, const float* cams, uint32_t w, uint32_t hh,
               float* hits, uint64_t R, uint32_t* stats) {
  if (h->spheres) {
    if (wide_layout(h->node_width))
      return launch_width<kMode, kStats, kCamera, true, false, true>(ctx, h, rays, cams, w, hh, hits, R, stats);
    return launch_width<kMode, kStats, kCamera, false, false, true>(ctx, h, rays, cams, w, hh, hits, R, stats);
  }
  if (wide_layout(h->node_width))
    return launch_width<kMode, kStats, kCamera, true>(ctx, h, rays, cams, w, hh, hits, R, stats);
  return launch_width<kMode, kStats, kCamera, false>(ctx, h, rays, cams, w, hh, hits, R, stats);
}

// Ambient-occlusion rays of closest hits: bajo's _make_ao_ray
// (rt/gpu/path_shading.mojo:650-665) applied to a ray launch.  AO ray
// j = r * samples + k belongs to primary ray r and draws its direction from
// the Philox stream (seed, path j, stage 1): uniform on the sphere, flipped to
// the side of the normal oriented against the incoming ray
// (rt/geometry.mojo:20-30).  Origin o + t d, t in [0.001, 4.0].  A primary ray
// without a surface hit yields a ray with t_max = -1, which no traversal can
// hit.  Output is field-major like the input rays.
__global__ void __launch_bounds__(256) ao_rays_kernel(const float* __restrict__ rays, const float* __restrict__ hits,
                                                      uint64_t n, uint32_t samples, uint64_t seed,
                                                      float* __restrict__ out) {
  const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t m = n * samples;
  if (j >= m) return;
  const uint64_t r = j / samples;
  const float4* hp = reinterpret_cast<const float4*>(hits + 8 * r);
  const float4 h0 = hp[0], h1 = hp[1];
  const uint32_t prim = __builtin_bit_cast(uint32_t, h0.z);
  const v3 o = mk(rays[r], rays[n + r], rays[2 * n + r]);
  const v3 d = mk(rays[4 * n + r], rays[5 * n + r], rays[6 * n + r]);
  const float tmax = rays[7 * n + r];
  v3 po = mk(0.0f, 0.0f, 0.0f), dir = mk(0.0f, 0.0f, 1.0f);
  float t_hi = -1.0f;
  if (prim != kEmpty && h1.w < tmax) {
    const v3 hn = mk(h1.x, h1.y, h1.z);
    const v3 nn = dot(d, hn) < 0.0f ? hn : mk(-hn.x, -hn.y, -hn.z);
    po = add(o, scale(d, h1.w));
    StageRng rng(seed, (uint32_t)j, 1u);
    float sn, cs;
    sincos_turns(rng.next(), sn, cs);
    const float z = 1.0f - 2.0f * rng.next();
    const float rad = sqrtf(1.0f - z * z);
    dir = mk(rad * cs, rad * sn, z);
    if (dot(dir, nn) < 0.0f) dir = mk(-dir.x, -dir.y, -dir.z);
    t_hi = 4.0f;
  }
  const float f[8] = {po.x, po.y, po.z, 0.001f, dir.x, dir.y, dir.z, t_hi};
#pragma unroll
  for (int k = 0; k < 8; ++k) out[(uint64_t)k * m + j] = f[k];
}

}  // namespace
}  // namespace bj

extern "C" {

int32_t bajo_ao_rays(bajo_ctx* ctx, const float* rays, const float* hits, uint64_t ray_count, uint32_t samples,
                     uint64_t seed, float* ao_rays) {
  BJ_REQUIRE(ctx != nullptr, "bajo_ao_rays: NULL ctx");
  BJ_REQUIRE(rays != nullptr && hits != nullptr && ao_rays != nullptr, "bajo_ao_rays: NULL buffer");
  BJ_REQUIRE(ray_count > 0 && samples > 0, "bajo_ao_rays: ray and sample counts must be positive");
  BJ_REQUIRE(ray_count * samples < (1ull << 31), "bajo_ao_rays: ray_count * samples must be below 2^31");
  const uint64_t m = ray_count * samples;
  bj::ao_rays_kernel<<<(unsigned)((m + 255) / 256), 256, 0, ctx->stream>>>(rays, hits, ray_count, samples, seed,
                                                                          ao_rays);
  BJ_HIP(hipGetLastError());
  return BAJO_OK;
}

int32_t bajo_trace_rays(bajo_ctx* ctx, const bajo_bvh* bvh, int32_t mode, const float* rays, float* hits,
                        uint64_t ray_count, uint32_t* stats) {
  BJ_REQUIRE(ctx != nullptr && bvh != nullptr, "bajo_trace_rays: NULL ctx/bvh");
  BJ_REQUIRE(mode == BAJO_TRACE_CLOSEST_HIT || mode == BAJO_TRACE_ANY_HIT, "bajo_trace_rays: bad mode %d", mode);
  BJ_REQUIRE(ray_count > 0, "bajo_trace_rays: ray count must be positive");
  BJ_REQUIRE(ray_count < (1ull << 31), "bajo_trace_rays: ray count must be below 2^31");
  BJ_REQUIRE(rays != nullptr && hits != nullptr, "bajo_trace_rays: NULL rays/hits");
  BJ_REQUIRE(bvh->n > 0, "bajo_trace_rays: empty BVH");
  BJ_REQUIRE(!bvh->boxes || bvh->spheres, "bajo_trace_rays: the hierarchy was built over boxes, not triangles or spheres");
  BJ_REQUIRE(!bvh->seg_count, "bajo_trace_rays: trace a BLAS set through its segment views (bajo_blas_set_get)");
  if (mode == BAJO_TRACE_ANY_HIT) {
    BJ_REQUIRE(stats == nullptr, "bajo_trace_rays: stats are collected for closest-hit queries only");
    return bj::launch<BAJO_TRACE_ANY_HIT, false, false>(ctx, bvh, rays, nullptr, 0, 0, hits, ray_count, nullptr);
  }
  if (stats) return bj::launch<BAJO_TRACE_CLOSEST_HIT, true, false>(ctx, bvh, rays, nullptr, 0, 0, hits, ray_count, stats);
  return bj::launch<BAJO_TRACE_CLOSEST_HIT, false, false>(ctx, bvh, rays, nullptr, 0, 0, hits, ray_count, nullptr);
}

int32_t bajo_trace_camera(bajo_ctx* ctx, const bajo_bvh* bvh, const float* camera, float* hits, uint64_t ray_count,
                          uint32_t width, uint32_t height, uint32_t* stats) {
  BJ_REQUIRE(ctx != nullptr && bvh != nullptr, "bajo_trace_camera: NULL ctx/bvh");
  BJ_REQUIRE(ray_count > 0 && width > 0 && height > 0, "bajo_trace_camera: launch dimensions must be positive");
  BJ_REQUIRE(ray_count < (1ull << 31), "bajo_trace_camera: ray count must be below 2^31");
  BJ_REQUIRE(camera != nullptr && hits != nullptr, "bajo_trace_camera: NULL camera/hits");
  BJ_REQUIRE(bvh->n > 0, "bajo_trace_camera: empty BVH");
  BJ_REQUIRE(!bvh->boxes || bvh->spheres, "bajo_trace_camera: the hierarchy was built over boxes, not triangles or spheres");
  BJ_REQUIRE(!bvh->seg_count, "bajo_trace_camera: trace a BLAS set through its segment views (bajo_blas_set_get)");
  if (stats)
    return bj::launch<BAJO_TRACE_CLOSEST_HIT, true, true>(ctx, bvh, nullptr, camera, width, height, hits, ray_count, stats);
  return bj::launch<BAJO_TRACE_CLOSEST_HIT, false, true>(ctx, bvh, nullptr, camera, width, height, hits, ray_count,
                                                         nullptr);
}

int32_t bajo_blas_set_trace_camera(bajo_ctx* ctx, const bajo_blas_set* set, const float* cameras, float* hits,
                                   uint32_t width, uint32_t height, uint32_t* stats) {
  BJ_REQUIRE(ctx != nullptr && set != nullptr, "bajo_blas_set_trace_camera: NULL ctx/set");
  BJ_REQUIRE(cameras != nullptr && hits != nullptr, "bajo_blas_set_trace_camera: NULL cameras/hits");
  BJ_REQUIRE(width > 0 && height > 0, "bajo_blas_set_trace_camera: launch dimensions must be positive");
  const bajo_bvh* h = bj::blas_set_store(set);
  const uint64_t R = (uint64_t)h->seg_count * width * height;
  BJ_REQUIRE(R < (1ull << 31), "bajo_blas_set_trace_camera: %u segments x %u x %u rays exceed 2^31", h->seg_count,
             width, height);
  constexpr int kC = BAJO_TRACE_CLOSEST_HIT;
  if (wide_layout(h->node_width)) {
    if (stats) return bj::launch_width<kC, true, true, true, true>(ctx, h, nullptr, cameras, width, height, hits, R, stats);
    return bj::launch_width<kC, false, true, true, true>(ctx, h, nullptr, cameras, width, height, hits, R, nullptr);
  }
  if (stats) return bj::launch_width<kC, true, true, false, true>(ctx, h, nullptr, cameras, width, height, hits, R, stats);
  return bj::launch_width<kC, false, true, false, true>(ctx, h, nullptr, cameras, width, height, hits, R, nullptr);
}

int32_t bajo_camera_make(const float* o3, const float* t3, const float* u3, float fov_scale, float focus_dist,
                         float* out20) {
  BJ_REQUIRE(o3 && t3 && u3 && out20, "bajo_camera_make: NULL argument");
  using namespace bj;
  v3 o = mk(o3[0], o3[1], o3[2]);
  v3 fwd = normalize(sub(mk(t3[0], t3[1], t3[2]), o));
  v3 right = normalize(cross(fwd, mk(u3[0], u3[1], u3[2])));
  v3 up = normalize(cross(right, fwd));
  float v[20] = {o.x, o.y, o.z, fwd.x, fwd.y, fwd.z, right.x, right.y, right.z, up.x, up.y, up.z,
                 fov_scale, focus_dist, 0, 0, 0, 0, 0, 0};
  for (int i = 0; i < 20; ++i) out20[i] = v[i];
  return BAJO_OK;
}

}  // extern "C"

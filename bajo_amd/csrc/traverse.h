// Device-side BVH2 traversal shared by the ray-launch kernels and the
// wavefront renderer.
//
// Follows bajo's near-first loop (bvh/gpu/trace.mojo:341-552) and its
// triangle leaf test (bvh/gpu/triangle_bvh.mojo:866-959: determinant-scaled
// Moller-Trumbore in FP32, normal = normalize(e1 x e2)).  Nodes are 64-byte
// records read with four 16-byte loads, leaf triangles 48-byte records read
// with three.  The per-lane stack lives in LDS (depth-major across the
// block, so lanes at any depth hit distinct banks); entries deeper than
// kLdsStack spill to a per-thread global column.  A Karras hierarchy over
// 64-bit (code, index) keys is at most 64 levels deep, so 64 entries always
// suffice.
#pragma once

#include <type_traits>

#include "bvh_internal.h"

namespace bj {

constexpr int kTraceBlock = 256;
// A third traversal mode chosen per lane at run time (closest or any hit), so
// lanes tracing either kind of ray step through one instruction stream: the
// near-first closest-hit walk, ended at the first hit for an any-hit lane.
constexpr int kTraceEither = 2;
constexpr int kTraceShadow = 3;  // 3..6: any hit through one of the shadow walks (8-wide)
constexpr int kLdsStack = 24;
constexpr int kMaxStack = 64;
constexpr int kSpill = kMaxStack - kLdsStack;
// The shallowest LDS stack a kernel uses (the 8-waves-per-SIMD extension
// kernel, whose LDS must fit eight blocks per CU) and the spill it needs.
constexpr int kLdsStackMin = 16;
constexpr int kLdsStackMax = 32;  // the 4-waves-per-SIMD extension kernel
constexpr int kSpillMax = kMaxStack - kLdsStackMin;

struct Ray {
  v3 o, d;
  float tmin, tmax;
};

struct Hit {
  float u, v;
  uint32_t prim, inst;
  v3 n;
  float t;
};

BJ_D Hit miss(float t) { return Hit{0.0f, 0.0f, kEmpty, kEmpty, mk(0, 0, 0), t}; }

BJ_D void store_hit(float* hits, uint64_t r, const Hit& h) {
  float4* p = reinterpret_cast<float4*>(hits + 8 * r);
  p[0] = make_float4(h.u, h.v, __builtin_bit_cast(float, h.prim), __builtin_bit_cast(float, h.inst));
  p[1] = make_float4(h.n.x, h.n.y, h.n.z, h.t);
}

// core/intersect.mojo:193-215 with select min/max.
BJ_D bool slab(v3 o, v3 rcp, float lx, float ly, float lz, float hx, float hy, float hz, float t_max, float& t_out) {
  float t0x = (lx - o.x) * rcp.x, t0y = (ly - o.y) * rcp.y, t0z = (lz - o.z) * rcp.z;
  float t1x = (hx - o.x) * rcp.x, t1y = (hy - o.y) * rcp.y, t1z = (hz - o.z) * rcp.z;
  float tnx = fmin_sel(t0x, t1x), tny = fmin_sel(t0y, t1y), tnz = fmin_sel(t0z, t1z);
  float tfx = fmax_sel(t0x, t1x), tfy = fmax_sel(t0y, t1y), tfz = fmax_sel(t0z, t1z);
  float tmin = fmax_sel(fmax_sel(tnx, tny), fmax_sel(tnz, 0.0f));
  float tmax = fmin_sel(fmin_sel(tfx, tfy), fmin_sel(tfz, t_max));
  t_out = tmin;
  return tmin <= tmax;
}

struct TriData {
  v3 v0, e1, e2;
  uint32_t prim;
};

BJ_D TriData load_tri(const BjTri* __restrict__ tris, uint32_t s) {
  const float4* p = reinterpret_cast<const float4*>(tris + s);
  float4 a = p[0], b = p[1], c = p[2];
  return TriData{mk(a.x, a.y, a.z), mk(b.x, b.y, b.z), mk(c.x, c.y, c.z), __builtin_bit_cast(uint32_t, a.w)};
}

// core/intersect.mojo:462-508.  Returns the mask; fills the scaled values.
BJ_D bool tri_scaled(const Ray& r, const TriData& tr, float t_max, float& abs_det, float& ts, float& us, float& vs) {
  v3 p = cross(r.d, tr.e2);
  float det = dot(tr.e1, p);
  bool pos = det >= 0.0f;
  abs_det = pos ? det : -det;
  v3 tv = sub(r.o, tr.v0);
  float u_num = dot(tv, p);
  us = pos ? u_num : -u_num;
  v3 q = cross(tv, tr.e1);
  float v_num = dot(r.d, q);
  float t_num = dot(tr.e2, q);
  vs = pos ? v_num : -v_num;
  ts = pos ? t_num : -t_num;
  return abs_det > 1e-8f && us >= 0.0f && us <= abs_det && vs >= 0.0f && (us + vs) <= abs_det &&
         ts > r.tmin * abs_det && ts < t_max * abs_det;
}

// The closest-hit candidate held during a traversal: distance, scaled
// barycentrics, reciprocal determinant and triangle position.  The hit record
// (u = us * inv, v = vs * inv, primitive, unit normal of e1 x e2) is formed
// once at the end from the same values, so it equals the record formed at
// each accepted triangle, at a fraction of the per-triangle work.
struct Closest {
  float t, us, vs, inv;
  uint32_t s;
};

BJ_D Closest no_closest(float t) { return Closest{t, 0.0f, 0.0f, 0.0f, kEmpty}; }

BJ_D bool leaf_closest(const BjTri* __restrict__ tris, uint32_t s, const Ray& r, Closest& c) {
  TriData tr = load_tri(tris, s);
  float ad, ts, us, vs;
  if (!tri_scaled(r, tr, c.t, ad, ts, us, vs)) return false;
  const float inv = 1.0f / ad;
  c.t = ts * inv;
  c.us = us;
  c.vs = vs;
  c.inv = inv;
  c.s = s;
  return true;
}

BJ_D Hit closest_hit(const BjTri* __restrict__ tris, const Closest& c) {
  if (c.s == kEmpty) return miss(c.t);
  const TriData tr = load_tri(tris, c.s);
  return Hit{c.us * c.inv, c.vs * c.inv, tr.prim, kEmpty, normalize(cross(tr.e1, tr.e2)), c.t};
}

BJ_D bool leaf_any(const BjTri* __restrict__ tris, uint32_t s, const Ray& r) {
  TriData tr = load_tri(tris, s);
  float ad, ts, us, vs;
  return tri_scaled(r, tr, r.tmax, ad, ts, us, vs);
}

// ---- sphere leaves (bajo's GpuSphereBvh, bvh/gpu/sphere_bvh.mojo:423-478) ----
// A sphere BVH stores one 48-byte record per sorted leaf like a triangle BVH:
// center.xyz + prim id, then the radius (the rest unused).
struct SphData {
  v3 c;
  float r;
  uint32_t prim;
};

BJ_D SphData load_sphere(const BjTri* __restrict__ recs, uint32_t s) {
  const float4* p = reinterpret_cast<const float4*>(recs + s);
  const float4 a = p[0], b = p[1];
  return SphData{mk(a.x, a.y, a.z), b.x, __builtin_bit_cast(uint32_t, a.w)};
}

// intersect_ray_sphere (core/intersect.mojo:309-350): the nearer root inside
// (t_min, t_max), else the farther one.
BJ_D bool sphere_t(const Ray& r, const SphData& sp, float t_max, float& t) {
  const v3 oc = sub(r.o, sp.c);
  const float a = dot(r.d, r.d), half_b = dot(oc, r.d), c = dot(oc, oc) - sp.r * sp.r;
  const float det = half_b * half_b - a * c;
  const bool ok = det >= 0.0f;
  const float sq = sqrtf(fmax_sel(det, 0.0f));
  const float inv_a = 1.0f / a;
  const float t0 = (-half_b - sq) * inv_a, t1 = (-half_b + sq) * inv_a;
  const bool near = ok && t0 > r.tmin && t0 < t_max;
  const bool far = ok && !near && t1 > r.tmin && t1 < t_max;
  t = near ? t0 : t1;
  return near || far;
}

// Leaf tests and the final hit record for either primitive kind.
template <bool kSph>
BJ_D bool leaf_closest_p(const BjTri* __restrict__ recs, uint32_t s, const Ray& r, Closest& c) {
  if constexpr (kSph) {
    float t;
    if (!sphere_t(r, load_sphere(recs, s), c.t, t)) return false;
    c.t = t;
    c.s = s;
    return true;
  } else {
    return leaf_closest(recs, s, r, c);
  }
}

template <bool kSph>
BJ_D bool leaf_any_p(const BjTri* __restrict__ recs, uint32_t s, const Ray& r) {
  if constexpr (kSph) {
    float t;
    return sphere_t(r, load_sphere(recs, s), r.tmax, t);
  } else {
    return leaf_any(recs, s, r);
  }
}

// Sphere hit: u = v = 0, normal = normalize(o + t d - center).
template <bool kSph>
BJ_D Hit closest_hit_p(const BjTri* __restrict__ recs, const Closest& c, const Ray& r) {
  if constexpr (kSph) {
    if (c.s == kEmpty) return miss(c.t);
    const SphData sp = load_sphere(recs, c.s);
    const v3 p = add(r.o, scale(r.d, c.t));
    return Hit{0.0f, 0.0f, sp.prim, kEmpty, normalize(sub(p, sp.c)), c.t};
  } else {
    return closest_hit(recs, c);
  }
}

// A leaf record held in registers (triangle: v0 + prim, e1, e2; sphere:
// center + prim, radius), so a walk can load the next record before it
// tests the current one.
struct LeafRec {
  float4 a, b, c;
};

template <bool kSph>
BJ_D LeafRec load_rec(const BjTri* __restrict__ recs, uint32_t s) {
  const float4* p = reinterpret_cast<const float4*>(recs + s);
  LeafRec r;
  r.a = p[0];
  r.b = p[1];
  if constexpr (kSph) r.c = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  else r.c = p[2];
  return r;
}

template <bool kSph>
BJ_D bool rec_closest(const LeafRec& rec, uint32_t s, const Ray& r, Closest& c) {
  if constexpr (kSph) {
    const SphData sp{mk(rec.a.x, rec.a.y, rec.a.z), rec.b.x, __builtin_bit_cast(uint32_t, rec.a.w)};
    float t;
    if (!sphere_t(r, sp, c.t, t)) return false;
    c.t = t;
    c.s = s;
    return true;
  } else {
    const TriData tr{mk(rec.a.x, rec.a.y, rec.a.z), mk(rec.b.x, rec.b.y, rec.b.z), mk(rec.c.x, rec.c.y, rec.c.z),
                     __builtin_bit_cast(uint32_t, rec.a.w)};
    float ad, ts, us, vs;
    if (!tri_scaled(r, tr, c.t, ad, ts, us, vs)) return false;
    const float inv = 1.0f / ad;
    c.t = ts * inv;
    c.us = us;
    c.vs = vs;
    c.inv = inv;
    c.s = s;
    return true;
  }
}

template <bool kSph>
BJ_D bool rec_any(const LeafRec& rec, const Ray& r) {
  if constexpr (kSph) {
    const SphData sp{mk(rec.a.x, rec.a.y, rec.a.z), rec.b.x, __builtin_bit_cast(uint32_t, rec.a.w)};
    float t;
    return sphere_t(r, sp, r.tmax, t);
  } else {
    const TriData tr{mk(rec.a.x, rec.a.y, rec.a.z), mk(rec.b.x, rec.b.y, rec.b.z), mk(rec.c.x, rec.c.y, rec.c.z),
                     __builtin_bit_cast(uint32_t, rec.a.w)};
    float ad, ts, us, vs;
    return tri_scaled(r, tr, r.tmax, ad, ts, us, vs);
  }
}

struct Stack {
  uint32_t* lds;       // this lane's column: entry k at lds[k * kTraceBlock]
  uint32_t* spill;     // this thread's column: entry k at spill[k * spill_stride]
  uint64_t spill_stride;
  int sp;
  int lds_depth = kLdsStack;    // entries held in LDS; deeper ones spill
  int lds_stride = kTraceBlock;  // words between LDS entries (a column per lane of a block, or 1)
  BJ_D void push(uint32_t v) {
    if (sp < lds_depth) lds[sp * lds_stride] = v;
    else spill[(uint64_t)(sp - lds_depth) * spill_stride] = v;
    ++sp;
  }
  BJ_D uint32_t pop() {
    --sp;
    return sp < lds_depth ? lds[sp * lds_stride] : spill[(uint64_t)(sp - lds_depth) * spill_stride];
  }
};


struct BvhView {
  const BjNode* nodes;
  const BjTri* tris;
  uint32_t root, node_count, prim_count;
  uint32_t* status;
  const uint32_t* root_dev;  // when set, the root is read here (H-PLOC leaves it on the device)
};

struct TraceCounters {
  uint32_t visits, inner, leaves, max_sp;
};

// Closest hit (kMode == BAJO_TRACE_CLOSEST_HIT) or occlusion (ANY_HIT: the
// returned record is bajo's Hit.shadow_hit() or Hit.miss(t_max)).
template <int kMode, bool kStats, bool kSph = false>
BJ_D Hit traverse(const BvhView& bv, const Ray& ray, Stack& st, TraceCounters* tc, bool any_rt = false) {
  uint32_t n_visit = 0, n_inner = 0, n_leaf = 0, max_sp = 0;
  const BjNode* __restrict__ nodes = bv.nodes;
  const BjTri* __restrict__ tris = bv.tris;
  const uint32_t root = bv.root_dev ? *bv.root_dev : bv.root;
  const uint32_t node_count = bv.node_count, prim_count = bv.prim_count;
  uint32_t* status = bv.status;
  Closest best = no_closest(ray.tmax);
  const v3 rcp = rcp_dir(ray.d);
  st.sp = 0;
  bool occluded = false;

  if ((root & kLeafFlag) && root != kSentinel) {
    n_leaf++;
    if constexpr (kMode == BAJO_TRACE_ANY_HIT) occluded = leaf_any_p<kSph>(tris, root & kIndexMask, ray);
    else if (leaf_closest_p<kSph>(tris, root & kIndexMask, ray, best) && kMode == kTraceEither && any_rt) occluded = true;
  } else if (root != kSentinel) {
    uint32_t cur = root;
    for (;;) {
      // A valid hierarchy visits each node at most once per ray; the cap only
      // ends a ray early (with a status word) if the hierarchy is corrupted.
      if (cur >= node_count || n_visit > node_count) { atomicOr(status, (uint32_t)BAJO_STATUS_BAD_NODE); break; }
      n_visit++;
      const float4* np = reinterpret_cast<const float4*>(nodes + cur);
      float4 q0 = np[0], q1 = np[1], q2 = np[2];
      uint4 m = reinterpret_cast<const uint4*>(nodes + cur)[3];
      const float node_tmax = kMode == BAJO_TRACE_ANY_HIT ? ray.tmax : best.t;
      float t0, t1;
      bool h0 = slab(ray.o, rcp, q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, node_tmax, t0);
      bool h1 = slab(ray.o, rcp, q1.z, q1.w, q2.x, q2.y, q2.z, q2.w, node_tmax, t1);
      const uint32_t c0 = m.y, c1 = m.z;
      const bool l0 = (c0 & kLeafFlag) && (c0 & kIndexMask) < prim_count;
      const bool l1 = (c1 & kLeafFlag) && (c1 & kIndexMask) < prim_count;
      if constexpr (kMode == BAJO_TRACE_ANY_HIT) {
        if (h0) {
          if (l0) {
            n_leaf++;
            if (leaf_any_p<kSph>(tris, c0 & kIndexMask, ray)) { occluded = true; break; }
          } else if (!(c0 & kLeafFlag)) {
            if (st.sp >= kMaxStack) { atomicOr(status, (uint32_t)BAJO_STATUS_STACK_OVERFLOW); break; }
            st.push(c0);
          }
        }
        if (h1) {
          if (l1) {
            n_leaf++;
            if (leaf_any_p<kSph>(tris, c1 & kIndexMask, ray)) { occluded = true; break; }
          } else if (!(c1 & kLeafFlag)) {
            if (st.sp >= kMaxStack) { atomicOr(status, (uint32_t)BAJO_STATUS_STACK_OVERFLOW); break; }
            st.push(c1);
          }
        }
        if (st.sp == 0) break;
        cur = st.pop();
        continue;
      } else {
        bool v0 = false, v1 = false;
        if (h0) {
          if (l0) {
            n_leaf++;
            if (leaf_closest_p<kSph>(tris, c0 & kIndexMask, ray, best) && kMode == kTraceEither && any_rt) {
              occluded = true;
              break;
            }
          } else if (!(c0 & kLeafFlag)) { v0 = true; n_inner++; }
        }
        if (h1) {
          if (l1) {
            n_leaf++;
            if (leaf_closest_p<kSph>(tris, c1 & kIndexMask, ray, best) && kMode == kTraceEither && any_rt) {
              occluded = true;
              break;
            }
          } else if (!(c1 & kLeafFlag)) { v1 = true; n_inner++; }
        }
        // bvh/gpu/trace.mojo:395-426: nearest child first, push the other.
        int near = -1;
        float near_t = kFltMax;
        if (v0) { near = 0; near_t = t0; }
        if (v1 && (near == -1 || t1 < near_t)) { near = 1; near_t = t1; }
        bool overflow = false;
        if (v0 && near != 0 && t0 <= best.t) {
          if (st.sp >= kMaxStack) overflow = true; else st.push(c0);
        }
        if (v1 && near != 1 && t1 <= best.t) {
          if (st.sp >= kMaxStack) overflow = true; else st.push(c1);
        }
        if (overflow) { atomicOr(status, (uint32_t)BAJO_STATUS_STACK_OVERFLOW); break; }
        if (kStats && (uint32_t)st.sp > max_sp) max_sp = (uint32_t)st.sp;
        if (near != -1 && near_t <= best.t) { cur = near == 0 ? c0 : c1; continue; }
        if (st.sp == 0) break;
        cur = st.pop();
      }
    }
  }
  Hit hit;
  if (kMode == BAJO_TRACE_ANY_HIT || (kMode == kTraceEither && any_rt)) {
    // bvh/gpu/trace.mojo:44-59: occlusion is reported as Hit.shadow_hit().
    hit = occluded ? Hit{0.0f, 0.0f, kEmpty, kEmpty, mk(0, 0, 0), 0.0f} : miss(ray.tmax);
  } else {
    hit = closest_hit_p<kSph>(tris, best, ray);
  }
  if constexpr (kStats) {
    tc->visits = n_visit;
    tc->inner = n_inner;
    tc->leaves = n_leaf;
    tc->max_sp = max_sp;
  }
  return hit;
}

// ---- 8-wide traversal -------------------------------------------------------------
// Plays the role of bajo's compressed-BVH8 traversal
// (bvh/gpu/triangle_bvh.mojo:1010-1104, bvh/gpu/compressed_bounds_bvh.mojo:
// 469-576) over the 96-byte quantized nodes built by the collapse.  Per node:
// six 16-byte loads, the ray octant picks the near and far plane bytes, and
// t(q) = (o + q*2^e - ray.o) * rcp is evaluated as fmaf(q, 2^e*rcp,
// (o - ray.o)*rcp).  Leaf children hit by the ray are tested after the box
// loop in one flattened triangle loop (so lanes diverge by the number of
// triangles, not by child slot); inner children continue nearest first with
// the others pushed far-to-near.

struct WideView {
  const BjWide* nodes;
  const BjTri* tris;
  uint32_t node_count, prim_count;
  uint32_t* status;
  uint32_t root;
};

BJ_D float ubyte_f(uint32_t word, int k) { return (float)((word >> (8 * k)) & 0xFFu); }

// Child reference of a one-hot slot mask, as a chain of selects on plain
// register values (an index-based select over an array or struct would be
// folded into a dynamically indexed stack copy, i.e. scratch memory, when the
// index differs between lanes).
BJ_D uint32_t sel8(uint32_t bit, uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t c4, uint32_t c5,
                   uint32_t c6, uint32_t c7) {
  uint32_t r = c0;
  r = (bit & 0x02u) ? c1 : r;
  r = (bit & 0x04u) ? c2 : r;
  r = (bit & 0x08u) ? c3 : r;
  r = (bit & 0x10u) ? c4 : r;
  r = (bit & 0x20u) ? c5 : r;
  r = (bit & 0x40u) ? c6 : r;
  r = (bit & 0x80u) ? c7 : r;
  return r;
}

// The 8-wide traversal as a resumable walk: begin() takes a ray, each step()
// visits one node (its eight slab tests, the triangles of the leaf children
// it enters, the pushes of the inner ones) and moves to the next node;
// done() once the stack is empty, the ray is occluded (any hit) or an error
// ended it.  Launches that refill finished lanes with new rays call the steps
// themselves; traverse8 runs one ray to the end.
template <int kMode, bool kStats, bool kSph = false>
struct Walk8 {
  Ray ray;
  v3 rcp;
  bool px, py, pz, occluded, any_rt;
  Closest best;
  uint32_t cur, n_visit, n_inner, n_leaf, max_sp;

  BJ_D void begin(const WideView& wv, const Ray& r, Stack& st, bool any = false) {
    ray = r;
    any_rt = any;
    best = no_closest(r.tmax);
    rcp = rcp_dir(r.d);
    px = rcp.x >= 0.0f;
    py = rcp.y >= 0.0f;
    pz = rcp.z >= 0.0f;
    occluded = false;
    st.sp = 0;
    cur = wv.node_count == 0 ? kSentinel : wv.root;
    n_visit = n_inner = n_leaf = max_sp = 0;
  }

  BJ_D bool done() const { return cur == kSentinel; }

  BJ_D void step(const WideView& wv, Stack& st) {
    if (cur >= wv.node_count || n_visit > wv.node_count) {
      atomicOr(wv.status, (uint32_t)BAJO_STATUS_BAD_NODE);
      cur = kSentinel;
      return;
    }
    n_visit++;
    const uint4* np = reinterpret_cast<const uint4*>(wv.nodes + cur);
    const uint4 w0 = np[0], w1 = np[1], w2 = np[2], w3 = np[3], w4 = np[4], w5 = np[5];
    const uint32_t meta = w0.w;
    const int n = (int)(meta >> 24);
    const float sx = __builtin_bit_cast(float, (meta & 0xFFu) << 23);
    const float sy = __builtin_bit_cast(float, ((meta >> 8) & 0xFFu) << 23);
    const float sz = __builtin_bit_cast(float, ((meta >> 16) & 0xFFu) << 23);
    const float ax = (__builtin_bit_cast(float, w0.x) - ray.o.x) * rcp.x;
    const float ay = (__builtin_bit_cast(float, w0.y) - ray.o.y) * rcp.y;
    const float az = (__builtin_bit_cast(float, w0.z) - ray.o.z) * rcp.z;
    const float bx = sx * rcp.x, by = sy * rcp.y, bz = sz * rcp.z;
    // near / far plane bytes per axis for this ray octant (words: lo_x w1.xy,
    // lo_y w1.zw, lo_z w2.xy, hi_x w2.zw, hi_y w3.xy, hi_z w3.zw)
    const uint32_t nx0 = px ? w1.x : w2.z, nx1 = px ? w1.y : w2.w, fx0 = px ? w2.z : w1.x, fx1 = px ? w2.w : w1.y;
    const uint32_t ny0 = py ? w1.z : w3.x, ny1 = py ? w1.w : w3.y, fy0 = py ? w3.x : w1.z, fy1 = py ? w3.y : w1.w;
    const uint32_t nz0 = pz ? w2.x : w3.z, nz1 = pz ? w2.y : w3.w, fz0 = pz ? w3.z : w2.x, fz1 = pz ? w3.w : w2.y;
    uint32_t c0 = w4.x, c1 = w4.y, c2 = w4.z, c3 = w4.w, c4 = w5.x, c5 = w5.y, c6 = w5.z, c7 = w5.w;
    asm("" : "+v"(c0), "+v"(c1), "+v"(c2), "+v"(c3), "+v"(c4), "+v"(c5), "+v"(c6), "+v"(c7));
    const float node_tmax = kMode == BAJO_TRACE_ANY_HIT ? ray.tmax : best.t;
    float th[8];
    // slot hits as a bit mask, built without branches (per-slot branches
    // cost more than the slab test itself)
    uint32_t hit_mask = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int bt = i & 3;
      const uint32_t qnx = i < 4 ? nx0 : nx1, qfx = i < 4 ? fx0 : fx1;
      const uint32_t qny = i < 4 ? ny0 : ny1, qfy = i < 4 ? fy0 : fy1;
      const uint32_t qnz = i < 4 ? nz0 : nz1, qfz = i < 4 ? fz0 : fz1;
      const float tnx = fmaf(ubyte_f(qnx, bt), bx, ax), tfx = fmaf(ubyte_f(qfx, bt), bx, ax);
      const float tny = fmaf(ubyte_f(qny, bt), by, ay), tfy = fmaf(ubyte_f(qfy, bt), by, ay);
      const float tnz = fmaf(ubyte_f(qnz, bt), bz, az), tfz = fmaf(ubyte_f(qfz, bt), bz, az);
      const float tmin = fmaxf(fmaxf(tnx, tny), fmaxf(tnz, 0.0f));
      const float tmax = fminf(fminf(tfx, tfy), fminf(tfz, node_tmax));
      th[i] = tmin;
      hit_mask |= tmin <= tmax ? (1u << i) : 0u;
    }
    hit_mask &= n >= 8 ? 0xFFu : (1u << n) - 1u;  // slots past the child count are never entered
    const uint32_t leaf_bits = (c0 >> 31) | ((c1 >> 30) & 2u) | ((c2 >> 29) & 4u) | ((c3 >> 28) & 8u) |
                               ((c4 >> 27) & 16u) | ((c5 >> 26) & 32u) | ((c6 >> 25) & 64u) | ((c7 >> 24) & 128u);
    uint32_t leaf_mask = hit_mask & leaf_bits, inner_mask = hit_mask & ~leaf_bits;
    // leaf children: one record per iteration across all hit leaves, in
    // slot order; the next record's load is issued before the current one
    // is tested, so a leaf's records arrive back to back
    uint32_t tri = 0, tri_end = 0;
    auto advance = [&](uint32_t& t, uint32_t& e) -> bool {
      while (t >= e) {
        if (!leaf_mask) return false;
        const uint32_t bit = leaf_mask & (0u - leaf_mask);
        leaf_mask ^= bit;
        const uint32_t ref = sel8(bit, c0, c1, c2, c3, c4, c5, c6, c7);
        t = ref & kWideLeafStartMask;
        e = t + ((ref >> 28) & 7u) + 1u;
        if (e > wv.prim_count) e = wv.prim_count;
      }
      return true;
    };
    bool have = advance(tri, tri_end);
    LeafRec cur_rec;
    if (have) cur_rec = load_rec<kSph>(wv.tris, tri);
    while (have) {
      uint32_t nt = tri + 1, ne = tri_end;
      const bool nhave = advance(nt, ne);
      LeafRec next_rec;
      if (nhave) next_rec = load_rec<kSph>(wv.tris, nt);
      n_leaf++;
      if constexpr (kMode == BAJO_TRACE_ANY_HIT) {
        if (rec_any<kSph>(cur_rec, ray)) {
          occluded = true;
          break;
        }
      } else if constexpr (kMode == kTraceEither) {
        // best.t stays at t_max on an any-hit lane, so the closest-hit test is its occlusion test
        if (rec_closest<kSph>(cur_rec, tri, ray, best) && any_rt) {
          occluded = true;
          break;
        }
      } else {
        rec_closest<kSph>(cur_rec, tri, ray, best);
      }
      tri = nt;
      tri_end = ne;
      have = nhave;
      cur_rec = next_rec;
    }
    if constexpr (kMode == BAJO_TRACE_ANY_HIT || kMode == kTraceEither) {
      if (occluded) {
        cur = kSentinel;
        return;
      }
    }
    if constexpr (kMode != BAJO_TRACE_ANY_HIT) {
      // children entered beyond the (possibly improved) closest hit are dropped
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (th[i] > best.t) inner_mask &= ~(1u << i);
    }
    if (kStats) n_inner += __builtin_popcount(inner_mask);
    if (inner_mask) {
      // push all but the nearest inner child, farthest first
      bool overflow = false;
      while (inner_mask & (inner_mask - 1u)) {
        uint32_t far_bit = 0, far_ref = 0;
        float far_t = -1.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (((inner_mask >> i) & 1u) && th[i] >= far_t) {
            far_t = th[i];
            far_bit = 1u << i;
            far_ref = sel8(1u << i, c0, c1, c2, c3, c4, c5, c6, c7);
          }
        inner_mask ^= far_bit;
        if (st.sp >= kMaxStack) {
          overflow = true;
          break;
        }
        st.push(far_ref);
      }
      if (overflow) {
        atomicOr(wv.status, (uint32_t)BAJO_STATUS_STACK_OVERFLOW);
        cur = kSentinel;
        return;
      }
      if (kStats && (uint32_t)st.sp > max_sp) max_sp = (uint32_t)st.sp;
      cur = sel8(inner_mask, c0, c1, c2, c3, c4, c5, c6, c7);
      return;
    }
    cur = st.sp == 0 ? kSentinel : st.pop();

}

  BJ_D Hit finish(const WideView& wv, TraceCounters* tc) const {
    Hit hit;
    if (kMode == BAJO_TRACE_ANY_HIT || (kMode == kTraceEither && any_rt)) {
      hit = occluded ? Hit{0.0f, 0.0f, kEmpty, kEmpty, mk(0, 0, 0), 0.0f} : miss(ray.tmax);
    } else {
      hit = closest_hit_p<kSph>(wv.tris, best, ray);
    }
    if constexpr (kStats) {
      tc->visits = n_visit;
      tc->inner = n_inner;
      tc->leaves = n_leaf;
      tc->max_sp = max_sp;
    }
    return hit;
  }
};

template <int kMode, bool kStats, bool kSph = false>
BJ_D Hit traverse8(const WideView& wv, const Ray& ray, Stack& st, TraceCounters* tc, bool any_rt = false) {
  Walk8<kMode, kStats, kSph> w;
  w.begin(wv, ray, st, any_rt);
  while (!w.done()) w.step(wv, st);
  return w.finish(wv, tc);
}

// Child slab tests of one 8-wide node: which slots the ray enters, which of
// those are leaves, their entry distances and references.
struct WideHits {
  uint32_t c[8];
  float th[8];
  uint32_t leaf, inner;
};

BJ_D void wide_node_hits(const uint4 (&w)[6], const Ray& ray, const v3& rcp, bool px, bool py, bool pz,
                         float node_tmax, WideHits& h) {
  const uint32_t meta = w[0].w;
  const int n = (int)(meta >> 24);
  const float sx = __builtin_bit_cast(float, (meta & 0xFFu) << 23);
  const float sy = __builtin_bit_cast(float, ((meta >> 8) & 0xFFu) << 23);
  const float sz = __builtin_bit_cast(float, ((meta >> 16) & 0xFFu) << 23);
  const float ax = (__builtin_bit_cast(float, w[0].x) - ray.o.x) * rcp.x;
  const float ay = (__builtin_bit_cast(float, w[0].y) - ray.o.y) * rcp.y;
  const float az = (__builtin_bit_cast(float, w[0].z) - ray.o.z) * rcp.z;
  const float bx = sx * rcp.x, by = sy * rcp.y, bz = sz * rcp.z;
  const uint32_t nx0 = px ? w[1].x : w[2].z, nx1 = px ? w[1].y : w[2].w, fx0 = px ? w[2].z : w[1].x,
                 fx1 = px ? w[2].w : w[1].y;
  const uint32_t ny0 = py ? w[1].z : w[3].x, ny1 = py ? w[1].w : w[3].y, fy0 = py ? w[3].x : w[1].z,
                 fy1 = py ? w[3].y : w[1].w;
  const uint32_t nz0 = pz ? w[2].x : w[3].z, nz1 = pz ? w[2].y : w[3].w, fz0 = pz ? w[3].z : w[2].x,
                 fz1 = pz ? w[3].w : w[2].y;
  h.c[0] = w[4].x; h.c[1] = w[4].y; h.c[2] = w[4].z; h.c[3] = w[4].w;
  h.c[4] = w[5].x; h.c[5] = w[5].y; h.c[6] = w[5].z; h.c[7] = w[5].w;
  uint32_t hit_mask = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int bt = i & 3;
    const uint32_t qnx = i < 4 ? nx0 : nx1, qfx = i < 4 ? fx0 : fx1;
    const uint32_t qny = i < 4 ? ny0 : ny1, qfy = i < 4 ? fy0 : fy1;
    const uint32_t qnz = i < 4 ? nz0 : nz1, qfz = i < 4 ? fz0 : fz1;
    const float tnx = fmaf(ubyte_f(qnx, bt), bx, ax), tfx = fmaf(ubyte_f(qfx, bt), bx, ax);
    const float tny = fmaf(ubyte_f(qny, bt), by, ay), tfy = fmaf(ubyte_f(qfy, bt), by, ay);
    const float tnz = fmaf(ubyte_f(qnz, bt), bz, az), tfz = fmaf(ubyte_f(qfz, bt), bz, az);
    const float tmin = fmaxf(fmaxf(tnx, tny), fmaxf(tnz, 0.0f));
    const float tmax = fminf(fminf(tfx, tfy), fminf(tfz, node_tmax));
    h.th[i] = tmin;
    hit_mask |= tmin <= tmax ? (1u << i) : 0u;
  }
  hit_mask &= n >= 8 ? 0xFFu : (1u << n) - 1u;
  uint32_t leaf_bits = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) leaf_bits |= (h.c[i] >> 31) << i;
  h.leaf = hit_mask & leaf_bits;
  h.inner = hit_mask & ~leaf_bits;
}

// Moves (t, e) to the next leaf record of the leaf slots left in lm_a, then
// lm_b (slot order); false once both are empty.
BJ_D bool next_leaf_range2(uint32_t& lm_a, uint32_t& lm_b, const WideHits& ha, const WideHits& hb,
                           uint32_t prim_count, uint32_t& t, uint32_t& e) {
  while (t >= e) {
    uint32_t ref;
    if (lm_a) {
      const uint32_t bit = lm_a & (0u - lm_a);
      lm_a ^= bit;
      ref = sel8(bit, ha.c[0], ha.c[1], ha.c[2], ha.c[3], ha.c[4], ha.c[5], ha.c[6], ha.c[7]);
    } else if (lm_b) {
      const uint32_t bit = lm_b & (0u - lm_b);
      lm_b ^= bit;
      ref = sel8(bit, hb.c[0], hb.c[1], hb.c[2], hb.c[3], hb.c[4], hb.c[5], hb.c[6], hb.c[7]);
    } else {
      return false;
    }
    t = ref & kWideLeafStartMask;
    e = t + ((ref >> 28) & 7u) + 1u;
    if (e > prim_count) e = prim_count;
  }
  return true;
}

// Any hit over the 8-wide layout for shadow rays, whose walks are long serial
// chains (they leave a surface and pass many boxes and leaves near it), in
// four forms picked per launch:
//   kTwo: two nodes per step -- the node on top of the stack is loaded and
//     tested together with the current one, so a step waits for one round of
//     node loads for both;
//   kBatch = 4: the leaf records of the entered leaves are loaded four at a
//     time (a 4-triangle leaf costs one load round instead of four);
//     kBatch = 1 keeps one record in flight ahead of the one being tested.
// Whether a ray is occluded does not depend on the order its nodes and
// records are visited in, so every form returns traverse8's result (an
// occluded ray returns the same constant record); only the visit counters
// can differ.
template <bool kStats, bool kSph, bool kTwo, int kBatch>
BJ_D Hit traverse8_any(const WideView& wv, const Ray& ray, Stack& st, TraceCounters* tc) {
  const v3 rcp = rcp_dir(ray.d);
  const bool px = rcp.x >= 0.0f, py = rcp.y >= 0.0f, pz = rcp.z >= 0.0f;
  uint32_t n_visit = 0, n_inner = 0, n_leaf = 0, max_sp = 0;
  bool occluded = false;
  st.sp = 0;
  uint32_t a = wv.node_count == 0 ? kSentinel : wv.root;
  while (a != kSentinel) {
    const uint32_t b = (kTwo && st.sp > 0) ? st.pop() : kSentinel;
    if (a >= wv.node_count || (b != kSentinel && b >= wv.node_count) || n_visit > wv.node_count) {
      atomicOr(wv.status, (uint32_t)BAJO_STATUS_BAD_NODE);
      break;
    }
    uint4 wa[6], wb[6];
    const uint4* pa = reinterpret_cast<const uint4*>(wv.nodes + a);
#pragma unroll
    for (int k = 0; k < 6; ++k) wa[k] = pa[k];
    if (kTwo && b != kSentinel) {
      const uint4* pb = reinterpret_cast<const uint4*>(wv.nodes + b);
#pragma unroll
      for (int k = 0; k < 6; ++k) wb[k] = pb[k];
    }
    WideHits ha, hb;
    // both nodes' loads are in flight; test a, then b (kept apart so the
    // scheduler does not interleave the two sets of slab temporaries)
    __builtin_amdgcn_sched_barrier(0);
    wide_node_hits(wa, ray, rcp, px, py, pz, ray.tmax, ha);
    n_visit++;
    __builtin_amdgcn_sched_barrier(0);
    if (kTwo && b != kSentinel) {
      wide_node_hits(wb, ray, rcp, px, py, pz, ray.tmax, hb);
      n_visit++;
    } else {
      hb.leaf = hb.inner = 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        hb.c[i] = 0;
        hb.th[i] = 0.0f;
      }
    }
    // the leaf records of both nodes (a's leaves first, slot order)
    uint32_t lm_a = ha.leaf, lm_b = hb.leaf;
    uint32_t tri = 0, tri_end = 0;
    if constexpr (kBatch == 4) {
      for (;;) {
        uint32_t r0 = 0, r1 = 0, r2 = 0, r3 = 0;
        const bool h0 = next_leaf_range2(lm_a, lm_b, ha, hb, wv.prim_count, tri, tri_end);
        if (h0) r0 = tri++;
        const bool h1 = h0 && next_leaf_range2(lm_a, lm_b, ha, hb, wv.prim_count, tri, tri_end);
        if (h1) r1 = tri++;
        const bool h2 = h1 && next_leaf_range2(lm_a, lm_b, ha, hb, wv.prim_count, tri, tri_end);
        if (h2) r2 = tri++;
        const bool h3 = h2 && next_leaf_range2(lm_a, lm_b, ha, hb, wv.prim_count, tri, tri_end);
        if (h3) r3 = tri++;
        if (!h0) break;
        LeafRec q0 = load_rec<kSph>(wv.tris, r0), q1, q2, q3;
        if (h1) q1 = load_rec<kSph>(wv.tris, r1);
        if (h2) q2 = load_rec<kSph>(wv.tris, r2);
        if (h3) q3 = load_rec<kSph>(wv.tris, r3);
        n_leaf += 1u + (h1 ? 1u : 0u) + (h2 ? 1u : 0u) + (h3 ? 1u : 0u);
        if (rec_any<kSph>(q0, ray) || (h1 && rec_any<kSph>(q1, ray)) || (h2 && rec_any<kSph>(q2, ray)) ||
            (h3 && rec_any<kSph>(q3, ray))) {
          occluded = true;
          break;
        }
        if (!h3) break;
      }
    } else {
      bool have = next_leaf_range2(lm_a, lm_b, ha, hb, wv.prim_count, tri, tri_end);
      LeafRec cur_rec;
      if (have) cur_rec = load_rec<kSph>(wv.tris, tri);
      while (have) {
        uint32_t nt = tri + 1, ne = tri_end;
        const bool nhave = next_leaf_range2(lm_a, lm_b, ha, hb, wv.prim_count, nt, ne);
        LeafRec next_rec;
        if (nhave) next_rec = load_rec<kSph>(wv.tris, nt);
        n_leaf++;
        if (rec_any<kSph>(cur_rec, ray)) {
          occluded = true;
          break;
        }
        tri = nt;
        tri_end = ne;
        have = nhave;
        cur_rec = next_rec;
      }
    }
    if (occluded) break;
    uint32_t ia = ha.inner, ib = hb.inner;
    if (kStats) n_inner += __builtin_popcount(ia) + __builtin_popcount(ib);
    // push b's inner children, then a's farthest first; continue at a's
    // nearest (or the top of the stack)
    bool overflow = false;
    while (ib) {
      const uint32_t bit = ib & (0u - ib);
      ib ^= bit;
      if (st.sp >= kMaxStack) { overflow = true; break; }
      st.push(sel8(bit, hb.c[0], hb.c[1], hb.c[2], hb.c[3], hb.c[4], hb.c[5], hb.c[6], hb.c[7]));
    }
    while (!overflow && (ia & (ia - 1u))) {
      uint32_t far_bit = 0;
      float far_t = -1.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (((ia >> i) & 1u) && ha.th[i] >= far_t) {
          far_t = ha.th[i];
          far_bit = 1u << i;
        }
      ia ^= far_bit;
      if (st.sp >= kMaxStack) { overflow = true; break; }
      st.push(sel8(far_bit, ha.c[0], ha.c[1], ha.c[2], ha.c[3], ha.c[4], ha.c[5], ha.c[6], ha.c[7]));
    }
    if (overflow) {
      atomicOr(wv.status, (uint32_t)BAJO_STATUS_STACK_OVERFLOW);
      break;
    }
    if (kStats && (uint32_t)st.sp > max_sp) max_sp = (uint32_t)st.sp;
    if (ia) a = sel8(ia, ha.c[0], ha.c[1], ha.c[2], ha.c[3], ha.c[4], ha.c[5], ha.c[6], ha.c[7]);
    else a = st.sp == 0 ? kSentinel : st.pop();
  }
  if constexpr (kStats) {
    tc->visits = n_visit;
    tc->inner = n_inner;
    tc->leaves = n_leaf;
    tc->max_sp = max_sp;
  }
  return occluded ? Hit{0.0f, 0.0f, kEmpty, kEmpty, mk(0, 0, 0), 0.0f} : miss(ray.tmax);
}

// bvh/camera.mojo:137-154, camera record bvh/camera.mojo:19-30.
BJ_D Ray camera_ray(const float* __restrict__ cams, uint64_t r, uint32_t w, uint32_t h, float inv_height) {
  uint64_t ppv = (uint64_t)w * h;
  uint64_t view = r / ppv, local = r - view * ppv;
  const float* c = cams + 20 * view;
  uint32_t px = (uint32_t)(local % w), py = (uint32_t)(local / w);
  float sx = (2.0f * ((float)px + 0.5f) - (float)w) * inv_height;
  float sy = 1.0f - 2.0f * ((float)py + 0.5f) * inv_height;
  float fov = c[12];
  v3 dir = add(add(mk(c[3], c[4], c[5]), scale(mk(c[6], c[7], c[8]), sx * fov)), scale(mk(c[9], c[10], c[11]), sy * fov));
  return Ray{mk(c[0], c[1], c[2]), normalize(dir), 0.0f, kFltMax};
}

// Either layout behind one call: kWide selects the 8-wide traversal.
struct AccelView {
  BvhView bin;
  WideView wide;
};

// Host: the view of a built hierarchy; `status` receives traversal errors.
inline AccelView accel_view(const bajo_bvh* h, uint32_t* status) {
  AccelView av;
  av.bin = BvhView{h->nodes, h->tris, h->root, h->trav_nodes, h->trav_prims, status,
                   h->root_on_device ? h->hp_ctl + kHpCtlRoot : nullptr};
  // a collapse whose node count has not been read back is bounded by its capacity
  const uint32_t wide_nodes = h->wide_pending ? (uint32_t)h->wide_capacity : h->wide_count;
  av.wide = WideView{h->wide, h->tris, wide_layout(h->node_width) ? wide_nodes : 0u, h->trav_prims, status,
                     h->wide_root};
  return av;
}

// Orders one wave's LDS writes before its later LDS reads by other lanes.
BJ_D void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Ballots and lane masks of a group of G lanes: 32 bits wide where they fit.
template <int G>
using GroupBits = std::conditional_t<G == 64, uint64_t, uint32_t>;

template <int G>
BJ_D GroupBits<G> group_ballot(bool p) {
  const uint64_t b = ballot(p);
  if constexpr (G == 64) return b;
  else return (uint32_t)(b >> (lane_id() & (64u - G))) & (uint32_t)((1ull << G) - 1ull);
}
BJ_D uint32_t bit_count(uint32_t m) { return (uint32_t)__builtin_popcount(m); }
BJ_D uint32_t bit_count(uint64_t m) { return (uint32_t)__builtin_popcountll(m); }
BJ_D uint32_t low_bit(uint32_t m) { return (uint32_t)__builtin_ctz(m); }
BJ_D uint32_t low_bit(uint64_t m) { return (uint32_t)__builtin_ctzll(m); }

template <int kCtrl>
BJ_D uint32_t dpp_mov(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kCtrl, 0xF, 0xF, true);
}

// Within each aligned group of 8 lanes: how many lanes with a nonzero key come
// before this one when keys are ordered from the largest down (equal keys:
// higher lane first).  Lanes exchange keys through quad permutes and the
// half-row mirror, so nothing waits on LDS.
BJ_D uint32_t far_rank8(uint32_t key) {
  const uint32_t lane = lane_id();
  // a partner above this lane comes first at an equal key, one below does not
  const uint32_t t1 = key + (lane & 1u), t2 = key + ((lane >> 1) & 1u), t4 = key + ((lane >> 2) & 1u);
  const uint32_t m = dpp_mov<0x141>(key);  // lane ^ 7
  uint32_t r = 0;
  r += dpp_mov<0xB1>(key) >= t1 ? 1u : 0u;  // ^ 1
  r += dpp_mov<0x4E>(key) >= t2 ? 1u : 0u;  // ^ 2
  r += dpp_mov<0x1B>(key) >= t2 ? 1u : 0u;  // ^ 3
  r += dpp_mov<0x1B>(m) >= t4 ? 1u : 0u;    // ^ 4
  r += dpp_mov<0x4E>(m) >= t4 ? 1u : 0u;    // ^ 5
  r += dpp_mov<0xB1>(m) >= t4 ? 1u : 0u;    // ^ 6
  r += m >= t4 ? 1u : 0u;                   // ^ 7
  return r;
}

// The two nearest candidates a group has met.  A one-lane walk accepts a
// triangle when its scaled distance beats the best so far
// (ts < t_best * det) and enters boxes up to the best so far, so which of two
// triangles wins can depend on their order when their distances lie within
// rounding of each other, or when a computed distance lies before the
// triangle's own box; a group visits nodes in another order.  So the group
// keeps the two smallest candidate distances it has seen (t1 with its record,
// t2; candidates pass the walk's own test against the ray's t_max) and hands
// the ray to the one-lane order
//   - if t2 lies within a slack of t1: 4e-6 t1 (ten times the rounding of the
//     scaled test) plus 1e-6 of the origin's coordinates (t of a near triangle
//     carries the rounding of o - v0);
//   - if t1 lies before its triangle's box by more than that slack: the
//     one-lane walk may have closed the box by then;
//   - if t1 < 0 (only rays with a negative t_min have such hits): it closes
//     every box to the one-lane walk, so what that had found decides.
// Else the nearest candidate is what the one-lane walk ends at, provided that
// the group has seen it: it culls boxes entered beyond t1 plus 2^-10 t1, so
// only a triangle whose computed distance lies further than that before its
// box could be missed.  The computed distance errs like 1 / cosine: of 55
// million hits of triangles within 1e-5 to 3e-2 of edge on, 57 came more than
// 4e-6 t before the triangle's box and none 1e-4 t.  The hit record is
// formed by testing the triangle again (the same arithmetic that formed it in
// the walk).
struct NearTwo {
  static constexpr float kRelative = 4e-6f, kAbsolute = 1e-6f, kCull = 0x1p-10f;
  float t1, t2, slack;
  uint32_t best;  // record of t1 (kEmpty: no candidate)
  BJ_D void clear(const Ray& r) {
    t1 = t2 = kFltMax;
    best = kEmpty;
    const float d = fmaxf(fabsf(r.d.x), fmaxf(fabsf(r.d.y), fabsf(r.d.z)));
    slack = kAbsolute * (fabsf(r.o.x) + fabsf(r.o.y) + fabsf(r.o.z)) / d;
  }
  BJ_D float reach() const { return fmaf(t1, kRelative, t1 + slack); }
  BJ_D float cull(float tmax) const { return fminf(tmax, fmaf(t1, kCull, t1 + slack)); }
  BJ_D bool tie() const { return best != kEmpty && (!(t2 > reach()) || t1 < 0.0f); }
  // Whether the nearest candidate lies before its own triangle's box.
  BJ_D bool early(const BjTri* __restrict__ tris, const Ray& r, const v3& rcp) const {
    if (best == kEmpty) return false;
    const TriData tr = load_tri(tris, best);
    const v3 b = add(tr.v0, tr.e1), c = add(tr.v0, tr.e2);
    const v3 lo = vmin(vmin(tr.v0, b), c), hi = vmax(vmax(tr.v0, b), c);
    float enter = 0.0f;
    slab(r.o, rcp, lo.x, lo.y, lo.z, hi.x, hi.y, hi.z, kFltMax, enter);
    return enter > reach();
  }
  // Takes the candidates of the group's lanes (record `s` at distance `t`
  // where `on`); every lane of the group holds the same state.
  template <int G>
  BJ_D void take(bool on, float t, uint32_t s) {
    const uint32_t base = lane_id() & (64u - G);
    for (GroupBits<G> m = group_ballot<G>(on); m; m &= m - 1) {
      const int p = (int)(base + low_bit(m));
      const float tp = __shfl(t, p, 64);
      const uint32_t sp = (uint32_t)__shfl((int)s, p, 64);
      if (best == kEmpty || tp < t1) {
        t2 = t1;
        t1 = tp;
        best = sp;
      } else {
        t2 = fminf(t2, tp);
      }
    }
  }
};

// Lane 8j + i's share of an 8-wide node: the header, child i's six plane bytes
// and its reference.  Each lane loads its own bytes (eight lanes' bytes of a
// plane are contiguous), so nothing is shifted out of wider words.
struct ChildLane {
  uint4 h;
  uint32_t lx, ly, lz, hx, hy, hz, ref;

  BJ_D void load(const BjWide* __restrict__ nodes, uint32_t node) {
    const BjWide* nd = nodes + node;
    const uint32_t i = lane_id() & 7u;
    h = *reinterpret_cast<const uint4*>(nd);
    lx = nd->lo_x[i];
    ly = nd->lo_y[i];
    lz = nd->lo_z[i];
    hx = nd->hi_x[i];
    hy = nd->hi_y[i];
    hz = nd->hi_z[i];
    ref = nd->child[i];
  }

  // The quantized slab test of Walk8: whether the ray enters child i before
  // `limit`, and where.  The planes of a child are ordered, so the smaller
  // of its two distances is the near plane's.
  BJ_D bool enters(const v3& o, const v3& rcp, float limit, float& tin) const {
    const uint32_t meta = h.w;
    const float bx = __builtin_bit_cast(float, (meta & 0xFFu) << 23) * rcp.x;
    const float by = __builtin_bit_cast(float, ((meta >> 8) & 0xFFu) << 23) * rcp.y;
    const float bz = __builtin_bit_cast(float, ((meta >> 16) & 0xFFu) << 23) * rcp.z;
    const float ax = (__builtin_bit_cast(float, h.x) - o.x) * rcp.x;
    const float ay = (__builtin_bit_cast(float, h.y) - o.y) * rcp.y;
    const float az = (__builtin_bit_cast(float, h.z) - o.z) * rcp.z;
    const float x0 = fmaf((float)lx, bx, ax), x1 = fmaf((float)hx, bx, ax);
    const float y0 = fmaf((float)ly, by, ay), y1 = fmaf((float)hy, by, ay);
    const float z0 = fmaf((float)lz, bz, az), z1 = fmaf((float)hz, bz, az);
    tin = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fmaxf(fminf(z0, z1), 0.0f));
    const float tout = fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fminf(fmaxf(z0, z1), limit));
    return (lane_id() & 7u) < (meta >> 24) && tin <= tout;
  }
};

// Writes the records of the entered leaves of a group (`is_leaf`, reference
// `cref`) to the group's LDS list in lane order and returns their number.
// Positions come from one ballot per count bit: a shuffle scan would wait on
// LDS log2(G) times.
template <int G>
BJ_D uint32_t list_records(bool is_leaf, uint32_t cref, uint32_t prim_count, uint32_t gl, uint32_t* recs) {
  const GroupBits<G> leaves = group_ballot<G>(is_leaf);
  if (leaves == 0) return 0;
  const GroupBits<G> below = ((GroupBits<G>)1 << gl) - 1;
  uint32_t start = 0, k = 0;
  if (is_leaf) {
    start = cref & kWideLeafStartMask;
    const uint32_t e = start + ((cref >> 28) & 7u) + 1u;
    k = (e > prim_count ? prim_count : e) - (start < prim_count ? start : prim_count);
  }
  uint32_t first = 0, total = 0;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const GroupBits<G> m = group_ballot<G>((k >> b) & 1u);
    first += bit_count(m & below) << b;
    total += bit_count(m) << b;
  }
  for (uint32_t m = 0; m < k; ++m) recs[first + m] = start + m;
  return total;
}

// Scaled test of a record held in registers.
BJ_D bool rec_scaled(const LeafRec& rec, const Ray& r, float t_max, float& ad, float& ts) {
  const TriData tr{mk(rec.a.x, rec.a.y, rec.a.z), mk(rec.b.x, rec.b.y, rec.b.z), mk(rec.c.x, rec.c.y, rec.c.z),
                   __builtin_bit_cast(uint32_t, rec.a.w)};
  float us, vs;
  return tri_scaled(r, tr, t_max, ad, ts, us, vs);
}

// The closest hit's record from its leaf record: the test that accepted it in
// the walk, done again.
BJ_D Hit record_hit(const BjTri* __restrict__ tris, uint32_t best, const Ray& ray) {
  Closest c = no_closest(ray.tmax);
  if (best != kEmpty) rec_closest<false>(load_rec<false>(tris, best), best, ray, c);
  return closest_hit_p<false>(tris, c, ray);
}

BJ_D Hit shadow_record(bool occluded, float tmax) {
  return occluded ? Hit{0.0f, 0.0f, kEmpty, kEmpty, mk(0, 0, 0), 0.0f} : miss(tmax);
}

// One ray walked by 8 lanes in exactly Walk8's order: lane i tests child i of
// the current node, records are tested one per lane and accepted in slot
// order, the nearest inner child comes next and the others go on the stack,
// farthest first.  So the hit is Walk8's by construction, at an eighth of its
// serial instructions per step.  While the records are tested the expected
// next node (the nearest entered child, else the stack's top) is loaded.
template <bool kAny>
struct OrderedWalk8 {
  static constexpr int G = 8;
  static constexpr int kStackWords = kMaxStack;
  static constexpr int kRecs = 64;
  Ray ray;
  v3 rcp;
  float best_t;
  uint32_t best, cur, steps;
  int sp;
  bool occluded;
  ChildLane nd;

  BJ_D void begin(const WideView& wv, const Ray& r) {
    ray = r;
    rcp = rcp_dir(r.d);
    best_t = r.tmax;
    best = kEmpty;
    occluded = false;
    steps = 0;
    sp = 0;
    cur = wv.node_count == 0 ? kSentinel : wv.root;
    if (cur < wv.node_count) nd.load(wv.nodes, cur);
  }

  // One step; true once the walk is finished (or ended by an error).
  BJ_D bool step(const WideView& wv, uint32_t* stack, uint32_t* recs, uint32_t& visits, uint32_t& tests) {
    if (cur == kSentinel) return true;
    const uint32_t gl = lane_id() & 7u;
    if (cur >= wv.node_count || steps > wv.node_count) {
      if (gl == 0) atomicOr(wv.status, (uint32_t)BAJO_STATUS_BAD_NODE);
      return true;
    }
    ++steps;
    ++visits;
    float tin;
    const bool hit = nd.enters(ray.o, rcp, kAny ? ray.tmax : best_t, tin);
    const uint32_t cref = nd.ref;
    const bool is_inner = hit && (cref & kLeafFlag) == 0;
    const uint32_t total = list_records<G>(hit && (cref & kLeafFlag) != 0, cref, wv.prim_count, gl, recs);
    const uint32_t rank = far_rank8(is_inner ? __builtin_bit_cast(uint32_t, tin) + 1u : 0u);
    const uint32_t inner = group_ballot<G>(is_inner);
    const uint32_t n_inner = bit_count(inner);
    wave_lds_sync();
    LeafRec rec;
    uint32_t s = 0;
    if (gl < total) {
      s = recs[gl];
      rec = load_rec<false>(wv.tris, s);
    }
    // the node to visit next unless a record drops it
    uint32_t next = kSentinel;
    if (n_inner) {
      const uint32_t p = low_bit(group_ballot<G>(is_inner && rank + 1u == n_inner));
      next = (uint32_t)__shfl((int)cref, (int)((lane_id() & 56u) + p), 64);
    } else if (sp > 0) {
      next = stack[sp - 1];
    }
    if (next < wv.node_count) nd.load(wv.nodes, next);
    bool closer = false;
    for (uint32_t base = 0; base < total; base += G) {
      const bool go = base + gl < total;
      if (base > 0 && go) {
        s = recs[base + gl];
        rec = load_rec<false>(wv.tris, s);
      }
      float ad = 0.0f, ts = 0.0f;
      const bool cand = go && rec_scaled(rec, ray, kAny ? ray.tmax : best_t, ad, ts);
      uint32_t m = group_ballot<G>(cand);
      tests += total - base < G ? total - base : G;
      if constexpr (kAny) {
        if (m) {
          occluded = true;
          return true;
        }
      } else {
        const float t = cand ? ts * (1.0f / ad) : 0.0f;
        for (; m; m &= m - 1) {
          const int p = (int)((lane_id() & 56u) + low_bit(m));
          if (__shfl(ts, p, 64) < best_t * __shfl(ad, p, 64)) {
            best_t = __shfl(t, p, 64);
            best = (uint32_t)__shfl((int)s, p, 64);
            closer = true;
          }
        }
      }
    }
    if (n_inner) {
      // children entered beyond the closest hit are dropped: the farthest ones
      uint32_t kept = n_inner;
      bool keep = is_inner;
      if (!kAny && closer) {
        keep = is_inner && !(tin > best_t);
        kept = bit_count(group_ballot<G>(keep));
      }
      if (kept > 1 && sp + (int)kept - 1 > kMaxStack) {
        if (gl == 0) atomicOr(wv.status, (uint32_t)BAJO_STATUS_STACK_OVERFLOW);
        return true;
      }
      if (keep && rank + 1u < n_inner) stack[sp + (int)(rank - (n_inner - kept))] = cref;
      wave_lds_sync();
      if (kept) {
        sp += (int)kept - 1;
        cur = next;
        return false;
      }
      if (sp == 0) {
        cur = kSentinel;
        return true;
      }
      cur = stack[--sp];
      if (cur < wv.node_count) nd.load(wv.nodes, cur);
      return false;
    }
    wave_lds_sync();
    cur = next;
    if (sp > 0) --sp;
    return cur == kSentinel;
  }

  BJ_D Hit finish(const WideView& wv, uint32_t*, uint32_t*, uint32_t&, uint32_t&) const {
    if constexpr (kAny) return shadow_record(occluded, ray.tmax);
    else return record_hit(wv.tris, best, ray);
  }
};

// One ray walked by G lanes (any hit: 8 to 64, closest hit: 16 to 64) over the
// 8-wide layout: the walk of rays whose chains are long and serial when one
// lane carries a ray (shadow rays, the last paths of a chunk, and launches
// with fewer rays than the chip has lanes).  A step holds up to G/8 nodes of
// the frontier, lane 8j + i tests child i of node j, entered inner children
// are pushed on the group's LDS stack, each node's farthest first and the
// nearest node's last, and the records of all entered leaves are tested one
// per lane.  The first round of record loads and the next frontier's node
// loads are issued before the records are tested, so a step waits for one
// round of memory whatever its width.
//
// Any hit: occlusion does not depend on the order of the tests.  Closest hit:
// see NearTwo; stack entries carry their entry distance, and entries beyond
// the nearest candidate are dropped as they come off the stack.
//
// `fallback` set at the end asks for the ordered walk (a near tie, or a
// frontier larger than the group's stack): finish() runs it on the group's
// first eight lanes.  With kFallback off (any hit in the renderer, whose
// shadow kernel would lose a resident wave to the code: 0.87 -> 1.09 ms for
// 416 K rays) a full stack ends the ray with a status word.  Every lane of a group holds the same state, and the
// group's lanes call together; other groups of the wave may be on rays of
// their own.
template <int G, bool kAny, bool kFallback = true>
struct GroupWalk8 {
  static_assert(kAny || kFallback, "closest hits need the ordered walk at near ties");
  static_assert(kAny || G > 8, "eight lanes walk closest hits in order (OrderedWalk8)");
  using Bits = GroupBits<G>;
  static constexpr int kEntry = kAny ? 1 : 2;           // words: node (, entry distance)
  static constexpr int kStackWords = 16 * G;            // per group
  static constexpr int kStack = kStackWords / kEntry;
  static constexpr int kRecs = 8 * G;                   // G entered leaves of up to 8 records
  static constexpr uint32_t kNodes = G / 8;
  static_assert(kStackWords >= OrderedWalk8<kAny>::kStackWords && kRecs >= OrderedWalk8<kAny>::kRecs,
                "the ordered walk uses the group's LDS area");
  Ray ray;
  v3 rcp;
  bool occluded, fallback;
  int sp;
  uint32_t steps;
  NearTwo near;
  // The frontier of the next step, taken off the stack and loaded while the
  // previous step's records were tested: how many nodes it holds, whether
  // this lane's node is one of them, its entry distance and this lane's child.
  // Lanes without a node load their group's first one (the same cache lines),
  // so the loads are unconditional and stay in flight across the record tests.
  uint32_t nf;
  bool mine;
  float te;
  ChildLane nd;

  // Starts a ray with the root as its first frontier (loaded here); a root
  // outside the hierarchy ends the ray at once with a status word.
  BJ_D void begin(const WideView& wv, const Ray& r) {
    ray = r;
    rcp = rcp_dir(r.d);
    occluded = fallback = false;
    steps = 1;
    sp = 0;
    near.clear(r);
    const bool ok = wv.node_count != 0 && wv.root < wv.node_count;
    if (wv.node_count != 0 && !ok && lane_id() % G == 0) atomicOr(wv.status, (uint32_t)BAJO_STATUS_BAD_NODE);
    nf = ok ? 1u : 0u;
    te = 0.0f;
    mine = ok && (lane_id() % G) < 8;
    if (ok) nd.load(wv.nodes, wv.root);
  }

  // Takes the next frontier off the stack and issues its loads.
  BJ_D bool pop(const WideView& wv, const uint32_t* stack, uint32_t gl) {
    const uint32_t j = gl >> 3;
    uint32_t node = 0;
    if constexpr (kAny) {
      nf = sp < (int)kNodes ? (uint32_t)sp : kNodes;
      mine = j < nf;
      const int at = sp - 1 - (mine ? (int)j : 0);
      node = stack[at > 0 ? at : 0];
      sp -= (int)nf;
    } else {
      const float limit = near.cull(ray.tmax);
      nf = 0;
      while (sp > 0) {
        // the top G entries, one per lane; the nearest kNodes still in reach
        const int at = sp - 1 - (int)gl;
        const bool live = at >= 0 && __builtin_bit_cast(float, stack[2 * (at < 0 ? 0 : at) + 1]) <= limit;
        Bits b = group_ballot<G>(live);
        if (b == 0) {
          sp = sp > G ? sp - G : 0;
          continue;
        }
        uint32_t own = low_bit(b), last = own;
        nf = 1;
#pragma unroll
        for (uint32_t q = 1; q < kNodes; ++q) {
          b &= b - 1;
          if (b) {
            last = low_bit(b);
            own = j >= q ? last : own;
            nf = q + 1;
          }
        }
        mine = j < nf;
        const int e = 2 * (sp - 1 - (int)(mine ? own : 0u));
        node = stack[e > 0 ? e : 0];
        te = __builtin_bit_cast(float, stack[e > 0 ? e + 1 : 1]);
        sp -= (int)last + 1;
        break;
      }
      if (nf == 0) mine = false;
    }
    const bool bad = group_ballot<G>(mine && node >= wv.node_count) != 0 || (nf > 0 && ++steps > wv.node_count);
    nd.load(wv.nodes, mine && node < wv.node_count ? node : 0u);
    return bad;
  }

  // One step; true once the walk is finished (or ended by an error).
  BJ_D bool step(const WideView& wv, uint32_t* stack, uint32_t* recs, uint32_t& visits, uint32_t& tests) {
    if (nf == 0) return true;
    const uint32_t gl = lane_id() % G, j = gl >> 3, i = gl & 7;
    const float limit = kAny ? ray.tmax : near.cull(ray.tmax);
    const bool on = mine && (kAny || te <= limit);
    visits += kAny ? nf : bit_count(group_ballot<G>(on && i == 0));
    float tin = 0.0f;
    const bool hit = nd.enters(ray.o, rcp, limit, tin) && on;
    const uint32_t cref = nd.ref;
    const bool is_inner = hit && (cref & kLeafFlag) == 0;
    // entered inner children onto the group's stack
    const Bits inner = group_ballot<G>(is_inner);
    const int n_inner = (int)bit_count(inner);
    if (sp + n_inner > kStack) {
      if constexpr (kFallback) fallback = true;
      else if (gl == 0) atomicOr(wv.status, (uint32_t)BAJO_STATUS_STACK_OVERFLOW);
      nf = 0;
      return true;
    }
    if constexpr (kAny) {
      if (is_inner) stack[sp + (int)bit_count(inner & (((Bits)1 << gl) - 1))] = cref;
    } else {
      const uint32_t rank = far_rank8(is_inner ? __builtin_bit_cast(uint32_t, tin) + 1u : 0u);
      if (is_inner) {
        // nodes off the stack's top come first in the frontier and go back last
        const Bits later = j + 1u < kNodes ? inner >> (8u * (j + 1u)) : 0;
        const int at = sp + (int)(bit_count(later) + rank);
        stack[2 * at] = cref;
        stack[2 * at + 1] = __builtin_bit_cast(uint32_t, tin);
      }
    }
    sp += n_inner;
    // the entered leaves' records, one per lane
    const uint32_t total = list_records<G>(hit && (cref & kLeafFlag) != 0, cref, wv.prim_count, gl, recs);
    wave_lds_sync();
    tests += total;
    LeafRec rec;
    uint32_t s = 0;
    if (gl < total) {
      s = recs[gl];
      rec = load_rec<false>(wv.tris, s);
    }
    const bool bad = pop(wv, stack, gl);
    wave_lds_sync();
    for (uint32_t base = 0; base < total; base += G) {
      const bool go = base + gl < total;
      if (base > 0 && go) {
        s = recs[base + gl];
        rec = load_rec<false>(wv.tris, s);
      }
      float ad = 0.0f, ts = 0.0f;
      const bool cand = go && rec_scaled(rec, ray, ray.tmax, ad, ts);
      if constexpr (kAny) {
        if (group_ballot<G>(cand) != 0) {
          occluded = true;
          nf = 0;
          return true;
        }
      } else {
        near.take<G>(cand, cand ? ts * (1.0f / ad) : 0.0f, s);
      }
    }
    if (total > G) wave_lds_sync();
    if (bad) {
      if (gl == 0) atomicOr(wv.status, (uint32_t)BAJO_STATUS_BAD_NODE);
      nf = 0;
    }
    if (nf == 0 && !kAny && near.tie()) fallback = true;
    return nf == 0;
  }

  // The finished walk's hit record, in the group's first lanes.
  BJ_D Hit finish(const WideView& wv, uint32_t* stack, uint32_t* recs, uint32_t& visits, uint32_t& tests) const {
    if (kFallback && (fallback || (!kAny && near.early(wv.tris, ray, rcp)))) {
      Hit h = miss(ray.tmax);
      if (lane_id() % G < 8) {
        OrderedWalk8<kAny> w;
        w.begin(wv, ray);
        while (!w.step(wv, stack, recs, visits, tests)) {
        }
        h = w.finish(wv, stack, recs, visits, tests);
      }
      return h;
    }
    if constexpr (kAny) return shadow_record(occluded, ray.tmax);
    else return record_hit(wv.tris, near.best, ray);
  }
};

// The group walk of G lanes over the 8-wide layout.
template <int G, bool kAny>
using Wide8 = std::conditional_t<G == 8 && !kAny, OrderedWalk8<false>, GroupWalk8<G == 8 && !kAny ? 16 : G, kAny>>;

// One ray walked by G lanes over the binary layout, as GroupWalk8: a step
// holds up to G/2 nodes, lane 2j + i tests child i of node j against its full
// box (the slab test of traverse()) and, where that child is a leaf, its one
// triangle, so no records are handed between lanes.
template <int G, bool kAny>
struct GroupWalk2 {
  static constexpr int kStackWords = 16 * G;
  static constexpr int kStack = kStackWords / 2;  // (node, entry distance)
  static constexpr uint32_t kNodes = G / 2;
  using Bits = GroupBits<G>;
  Ray ray;
  v3 rcp;
  bool occluded, fallback;
  int sp;
  uint32_t steps;
  NearTwo near;
  uint32_t nf;
  bool mine;
  float te;
  float2 b0, b1, b2;  // this lane's child box
  uint32_t ref;

  BJ_D void load(const BvhView& bv, uint32_t node) {
    const uint32_t i = lane_id() & 1u;
    const float* p = reinterpret_cast<const float*>(bv.nodes + node);
    const float2* q = reinterpret_cast<const float2*>(p + 6 * i);
    b0 = q[0];
    b1 = q[1];
    b2 = q[2];
    ref = reinterpret_cast<const uint32_t*>(p)[13 + i];
  }

  BJ_D void begin(const BvhView& bv, const Ray& r) {
    ray = r;
    rcp = rcp_dir(r.d);
    occluded = fallback = false;
    steps = 1;
    sp = 0;
    near.clear(r);
    const uint32_t root = bv.root_dev ? *bv.root_dev : bv.root;
    // a hierarchy of one leaf, or a root the one-lane walk reports
    fallback = root != kSentinel && ((root & kLeafFlag) != 0 || root >= bv.node_count);
    const bool ok = root != kSentinel && !fallback;
    nf = ok ? 1u : 0u;
    te = 0.0f;
    mine = ok && (lane_id() % G) < 2;
    if (ok) load(bv, root);
  }

  BJ_D bool step(const BvhView& bv, uint32_t* stack) {
    if (nf == 0) return true;
    const uint32_t gl = lane_id() % G, j = gl >> 1;
    const float limit = kAny ? ray.tmax : near.cull(ray.tmax);
    const bool on = mine && te <= limit;
    float tin = 0.0f;
    bool hit = false;
    if (on) hit = slab(ray.o, rcp, b0.x, b0.y, b1.x, b1.y, b2.x, b2.y, limit, tin);
    const uint32_t cref = ref;
    const uint32_t s = cref & kIndexMask;
    const bool is_leaf = hit && (cref & kLeafFlag) != 0 && s < bv.prim_count;
    const bool is_inner = hit && (cref & kLeafFlag) == 0;
    const Bits inner = group_ballot<G>(is_inner);
    const int n_inner = (int)bit_count(inner);
    if (sp + n_inner > kStack) {
      fallback = true;
      nf = 0;
      return true;
    }
    // the nearer of two entered children on top (child 0 at equal distances)
    const uint32_t key = is_inner ? __builtin_bit_cast(uint32_t, tin) + 1u : 0u;
    const uint32_t other = dpp_mov<0xB1>(key);
    if (is_inner) {
      const uint32_t rank = other >= key + (gl & 1u) ? 1u : 0u;
      const Bits later = j + 1u < kNodes ? inner >> (2u * (j + 1u)) : 0;
      const int at = sp + (int)(bit_count(later) + rank);
      stack[2 * at] = cref;
      stack[2 * at + 1] = __builtin_bit_cast(uint32_t, tin);
    }
    sp += n_inner;
    LeafRec rec;
    if (is_leaf) rec = load_rec<false>(bv.tris, s);
    wave_lds_sync();
    // the next frontier: the nearest kNodes of the stack's top G entries still in reach
    nf = 0;
    uint32_t node = 0;
    while (sp > 0) {
      const int at = sp - 1 - (int)gl;
      const bool live = at >= 0 && __builtin_bit_cast(float, stack[2 * (at < 0 ? 0 : at) + 1]) <= limit;
      const Bits b = group_ballot<G>(live);
      if (b == 0) {
        sp = sp > G ? sp - G : 0;
        continue;
      }
      // the j-th live entry belongs to lanes 2j and 2j + 1
      uint32_t own = low_bit(b), last = own;
      Bits m = b;
      nf = 1;
#pragma unroll
      for (uint32_t q = 1; q < kNodes; ++q) {
        m &= m - 1;
        if (m) {
          last = low_bit(m);
          own = j >= q ? last : own;
          nf = q + 1;
        }
      }
      mine = j < nf;
      const int e = 2 * (sp - 1 - (int)(mine ? own : 0u));
      node = stack[e > 0 ? e : 0];
      te = __builtin_bit_cast(float, stack[e > 0 ? e + 1 : 1]);
      sp -= (int)last + 1;
      break;
    }
    if (nf == 0) mine = false;
    const bool bad = group_ballot<G>(mine && node >= bv.node_count) != 0 || (nf > 0 && ++steps > bv.node_count);
    load(bv, mine && node < bv.node_count ? node : 0u);
    wave_lds_sync();
    if constexpr (kAny) {
      if (group_ballot<G>(is_leaf && rec_any<false>(rec, ray)) != 0) {
        occluded = true;
        nf = 0;
        return true;
      }
    } else {
      float ad = 0.0f, ts = 0.0f;
      const bool cand = is_leaf && rec_scaled(rec, ray, ray.tmax, ad, ts);
      near.take<G>(cand, cand ? ts * (1.0f / ad) : 0.0f, s);
    }
    if (bad) {
      if (gl == 0) atomicOr(bv.status, (uint32_t)BAJO_STATUS_BAD_NODE);
      nf = 0;
    }
    if (nf == 0 && !kAny && near.tie()) fallback = true;
    return nf == 0;
  }

  BJ_D Hit finish(const BvhView& bv, uint32_t* stack) const {
    if (fallback || (!kAny && near.early(bv.tris, ray, rcp))) {
      Stack st{stack, nullptr, 0, 0, kMaxStack, 1};
      return traverse<kAny ? BAJO_TRACE_ANY_HIT : BAJO_TRACE_CLOSEST_HIT, false>(bv, ray, st, nullptr);
    }
    if constexpr (kAny) return shadow_record(occluded, ray.tmax);
    else return record_hit(bv.tris, near.best, ray);
  }
};

// kTraceShadow + w (w = 0..3): any hit through a shadow walk -- w = 0 the
// one-node Walk8, else traverse8_any with bit 0 = two nodes per step and
// bit 1 = leaf records four at a time -- the same result as
// BAJO_TRACE_ANY_HIT; the binary layout keeps its one-node walk.
template <int kMode, bool kStats, bool kWide, bool kSph = false>
BJ_D Hit trace_accel(const AccelView& av, const Ray& ray, Stack& st, TraceCounters* tc, bool any_rt = false) {
  if constexpr (kMode >= kTraceShadow) {
    constexpr int w = kMode - kTraceShadow;
    if constexpr (kWide && w == 0) return traverse8<BAJO_TRACE_ANY_HIT, kStats, kSph>(av.wide, ray, st, tc, false);
    else if constexpr (kWide) return traverse8_any<kStats, kSph, (w & 1) != 0, (w & 2) ? 4 : 1>(av.wide, ray, st, tc);
    else return traverse<BAJO_TRACE_ANY_HIT, kStats, kSph>(av.bin, ray, st, tc, false);
  } else if constexpr (kWide) {
    return traverse8<kMode, kStats, kSph>(av.wide, ray, st, tc, any_rt);
  } else {
    return traverse<kMode, kStats, kSph>(av.bin, ray, st, tc, any_rt);
  }
}

}  // namespace bj

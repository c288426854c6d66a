// Learned path guiding on gfx950: the network's forward pass, its fused
// forward + backward pass, the weight gradient and Adam, all hand-written
// for the BF16 matrix cores (v_mfma_f32_16x16x32_bf16, FP32 accumulation).
// bajo has no counterpart; the network and its output are defined in
// guide_math.h.
//
// MI355X design:
// - Weights live in one device image: BF16 rows padded by 8 elements (so
//   16 lanes reading one 16-byte column slice of 16 rows hit different LDS
//   banks), transposed copies of W2..W4 for the backward pass, FP32 biases.
//   A block copies the image into LDS once (55 KB forward, 83 KB training).
// - MFMA operand layout (16x16x32): A[i][k] at lane i + 16 (k / 8), element
//   k % 8; B[k][j] at lane j + 16 (k / 8); D[i][j] at lane j + 16 (i / 4),
//   element i % 4.  Weights are the A operand and samples the B operand's
//   columns, so a lane's results are units 16 t + 4 g .. + 3 of one sample.
//   The rows of W2..W4 hold their inputs in the order in which the lanes
//   then have them (hidden_pos), so a layer's results, rounded to BF16 in
//   registers, are the next layer's operand: activations never pass
//   through LDS, and outputs leave as 16-byte stores.
// - The input encoding is computed straight into the layer-1 operand: lane
//   (i, g) of k-step s needs features 32 s + 8 g .. + 7, i.e. four
//   frequencies of one input.
// - A wave takes 32 samples (two operands) for each weight fragment it reads.
// - Training is one launch: the operands of a product swapped give its
//   transpose (lanes hold units, registers samples), which is the operand
//   form of the weight gradient dW = D^T X with the batch as K.  The eight
//   waves of a block exchange these fragments through LDS and each
//   accumulates 12 to 14 of the 111 gradient tiles; one partial per block
//   of 256 samples goes to memory, summed in fixed order by the Adam kernel
//   (deterministic, no atomics).
#include <math.h>
#include <string.h>

#include <vector>

#include "guide_internal.h"

namespace bj {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

// ---- weight image --------------------------------------------------------------
constexpr int kW1Stride = kGuideK0 + 8;      // 232
constexpr int kRowStride = kGuideHidden + 8;  // 72: rows of 64-wide operands
constexpr int kPackW1 = 0;                                       // [64][232]
constexpr int kPackW2 = kPackW1 + kGuideHidden * kW1Stride;      // [64][72]
constexpr int kPackW3 = kPackW2 + kGuideHidden * kRowStride;     // [64][72]
constexpr int kPackW4 = kPackW3 + kGuideHidden * kRowStride;     // [48][72]
constexpr int kPackFwd = kPackW4 + kGuideOutPad * kRowStride;    // forward weights end
constexpr int kPackW2t = kPackFwd;                               // [64 in][72]: W2^T
constexpr int kPackW3t = kPackW2t + kGuideHidden * kRowStride;   // W3^T
constexpr int kPackW4t = kPackW3t + kGuideHidden * kRowStride;   // [64 hidden][72]: W4^T (outputs < 40)
constexpr int kPackAll = kPackW4t + kGuideHidden * kRowStride;
constexpr int kBiasFloats = 3 * kGuideHidden + kGuideOutPad;     // b1 b2 b3 b4(48)
constexpr size_t kPackBytes = (size_t)kPackAll * 2 + kBiasFloats * 4;
static_assert((kPackAll * 2) % 16 == 0 && (kPackFwd * 2) % 16 == 0, "pack images are 16-byte aligned");

// ---- training layout -----------------------------------------------------------
constexpr int kTrainWaves = 8;
constexpr int kTrainSamples = kTrainWaves * 32;  // samples of one block and pass
constexpr uint32_t kTrainBlocks = 256;           // at most one per CU; larger batches loop
// gradient tiles (16 x 16 of dW[out][in], the bias in the column of the constant input)
constexpr int kT1 = 0, kT2 = 4 * 14, kT3 = kT2 + 4 * 5, kT4 = kT3 + 4 * 5, kTiles = kT4 + 3 * 5;  // 111

BJ_HD uint16_t f2bf(float x) {
  uint32_t u = __builtin_bit_cast(uint32_t, x);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
BJ_HD float bf2f(uint16_t b) { return __builtin_bit_cast(float, (uint32_t)b << 16); }

BJ_D bf16x8 frag16(const uint16_t* p) { return __builtin_bit_cast(bf16x8, *(const uint4*)p); }
BJ_D f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

// Where input k of a 64-wide layer lives in its weight row: lane group g of
// k-step s takes elements 32 s + 8 g .. + 7, and as B operand it has units
// 16 (2 s) + 4 g .. + 3 and 16 (2 s + 1) + 4 g .. + 3 of the layer before.
BJ_HD int hidden_pos(int k) { return 32 * (k >> 5) + 8 * ((k >> 2) & 3) + 4 * ((k >> 4) & 1) + (k & 3); }

// Where parameter p lives in the weight image (forward and, for W2..W4,
// transposed; -1 = none; biases go to the FP32 bias block).
struct ParamSlot {
  int fwd, tr, bias;
};
BJ_HD ParamSlot param_slot(int p) {
  ParamSlot s{-1, -1, -1};
  if (p < kGuideOffB1) {
    const int j = p / kGuideFeatures;
    s.fwd = kPackW1 + j * kW1Stride + (p - j * kGuideFeatures);
    return s;
  }
  if (p < kGuideOffW2) {
    s.bias = p - kGuideOffB1;
    return s;
  }
  int fwd_base, tr_base, bias_base, rows = kGuideHidden;
  if (p < kGuideOffW3) { fwd_base = kPackW2; tr_base = kPackW2t; bias_base = 64; p -= kGuideOffW2; }
  else if (p < kGuideOffW4) { fwd_base = kPackW3; tr_base = kPackW3t; bias_base = 128; p -= kGuideOffW3; }
  else { fwd_base = kPackW4; tr_base = kPackW4t; bias_base = 192; p -= kGuideOffW4; rows = kGuideOut; }
  if (p < rows * kGuideHidden) {
    const int j = p / kGuideHidden, k = p - j * kGuideHidden;
    s.fwd = fwd_base + j * kRowStride + hidden_pos(k);
    s.tr = tr_base + k * kRowStride + hidden_pos(j);
  } else {
    s.bias = bias_base + p - rows * kGuideHidden;
  }
  return s;
}

// The parameter of element e of gradient tile t (lane e / 4 holds four rows
// of one column), or -1: the column after the inputs is the bias.
BJ_HD int slot_param(int t, int e) {
  int base, tiles, rows = kGuideHidden, inputs = kGuideHidden;
  if (t < kT2) { base = kGuideOffW1; tiles = 14; inputs = kGuideFeatures; t -= kT1; }
  else if (t < kT3) { base = kGuideOffW2; tiles = 5; t -= kT2; }
  else if (t < kT4) { base = kGuideOffW3; tiles = 5; t -= kT3; }
  else { base = kGuideOffW4; tiles = 5; rows = kGuideOut; t -= kT4; }
  const int m = t / tiles;
  const int j = 16 * m + 4 * (e >> 6) + (e & 3), k = 16 * (t - m * tiles) + ((e >> 2) & 15);
  if (j >= rows || k > inputs) return -1;
  return k == inputs ? base + rows * inputs + j : base + j * inputs + k;
}

BJ_D void pack_param(uint8_t* pack, const ParamSlot& s, float v) {
  uint16_t* w = (uint16_t*)pack;
  float* b = (float*)(pack + (size_t)kPackAll * 2);
  if (s.bias >= 0) {
    b[s.bias] = v;
    return;
  }
  const uint16_t h = f2bf(v);
  w[s.fwd] = h;
  if (s.tr >= 0) w[s.tr] = h;
}

__global__ void __launch_bounds__(256) guide_pack_kernel(const float* __restrict__ params, uint8_t* __restrict__ pack) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < kGuideParams) pack_param(pack, param_slot(p), params[p]);
}

// ---- layer-1 operand -------------------------------------------------------------
// Chunk q = 4 s + g (0..27) of a sample's features: input d = q / 3,
// frequencies 4 (q % 3) .. + 3, (sin, cos) pairs; chunk 27 is padding, whose
// first element is the constant input (its weights are zero, its gradient is
// the bias's).  The chunks of one k-step lie in two neighbouring inputs.
BJ_D int chunk_input(int s, uint32_t g) {
  const int q = 4 * s + (int)g;
  return q < 27 ? q / 3 : kGuideInputs - 1;
}

// A lane's scales of its chunks' first frequencies: (q % 3) == (s + g) % 3.
BJ_D void chunk_scales(uint32_t g, float (&sc)[3]) {
#pragma unroll
  for (int t = 0; t < 3; ++t) sc[t] = guide_freq_scale(4 * (int)((t + g) % 3));
}

BJ_D bf16x8 encode_chunk(float x, float scale, bool constant) {
  float s[4], c[4];
  guide_encode_scaled(x, scale, s, c);
  // round to nearest even (the hardware conversion equals f2bf for finite values)
  bf16x8 f = {(__bf16)s[0], (__bf16)c[0], (__bf16)s[1], (__bf16)c[1],
              (__bf16)s[2], (__bf16)c[2], (__bf16)s[3], (__bf16)c[3]};
  if (constant) f = __builtin_bit_cast(bf16x8, uint4{0x3F80u, 0u, 0u, 0u});
  return f;
}

// ---- layers ----------------------------------------------------------------------
// ReLU (NaN to 0).
BJ_D float relu(float v) { return __builtin_amdgcn_fmed3f(v, 0.0f, __builtin_inff()); }
BJ_D f32x4 relu4(f32x4 v) { return f32x4{relu(v[0]), relu(v[1]), relu(v[2]), relu(v[3])}; }
BJ_D bf16x8 to_frag(f32x4 a, f32x4 b) {
  return bf16x8{(__bf16)a[0], (__bf16)a[1], (__bf16)a[2], (__bf16)a[3],
                (__bf16)b[0], (__bf16)b[1], (__bf16)b[2], (__bf16)b[3]};
}

// acc[u][t] += (rows 16 t .. + 15 of a 64-wide layer) x (sample tile u).
template <int kT>
BJ_D void layer64(const uint16_t* sw, const bf16x8 (&in)[2][2], f32x4 (&acc)[2][kT], uint32_t lane) {
  const uint32_t i = lane & 15u, g = lane >> 4;
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int t = 0; t < kT; ++t) {
      const bf16x8 w = frag16(sw + (16 * t + i) * kRowStride + 32 * s + 8 * g);
#pragma unroll
      for (int u = 0; u < 2; ++u) acc[u][t] = mfma(w, in[u][s], acc[u][t]);
    }
}

// Biases of a lane's units 16 t + 4 g .. + 3.
template <int kT>
BJ_D void start_bias(const float* bias, f32x4 (&acc)[2][kT], uint32_t g) {
#pragma unroll
  for (int t = 0; t < kT; ++t) acc[0][t] = acc[1][t] = *(const f32x4*)(bias + 16 * t + 4 * g);
}

// Activations as the next layer's operand.
BJ_D void hidden_frags(const f32x4 (&acc)[2][4], bf16x8 (&h)[2][2]) {
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int s = 0; s < 2; ++s) h[u][s] = to_frag(relu4(acc[u][2 * s]), relu4(acc[u][2 * s + 1]));
}

// A value that the compiler takes for a new one: what depends on it is
// computed where it stands.  Loops over sample tiles use it for the lane:
// the weights' addresses and fragments, hoisted out of the loop, would take
// more registers than there are.
BJ_D uint32_t fresh(uint32_t v) {
  asm volatile("" : "+v"(v));
  return v;
}

// Block-wide copy of the first `elems` BF16 weights and the biases into LDS.
BJ_D void load_pack(const uint8_t* __restrict__ pack, uint16_t* sw, int elems, float* sb, uint32_t tid) {
  const uint4* src = (const uint4*)pack;
  uint4* dst = (uint4*)sw;
  for (uint32_t i = tid; i < (uint32_t)elems / 8; i += blockDim.x) dst[i] = src[i];
  const float* bsrc = (const float*)(pack + (size_t)kPackAll * 2);
  for (uint32_t i = tid; i < (uint32_t)kBiasFloats; i += blockDim.x) sb[i] = bsrc[i];
  __syncthreads();
}

// ---- forward ---------------------------------------------------------------------
// Inputs: explicit f32[9 n], or render vertices (their position, normal and
// ray direction planes) normalized against the scene box.
// load: the inputs of row r's seven chunks of lane group g.
struct InputRows {
  const float* x;
  BJ_D void load(uint64_t r, uint32_t g, float (&v)[7]) const {
#pragma unroll
    for (int s = 0; s < 7; ++s) v[s] = x[r * kGuideInputs + chunk_input(s, g)];
  }
};

struct VertexRows {
  const float* f;
  const float* bounds;  // scene box lo.xyz, hi.xyz
  BJ_D void load(uint64_t r, uint32_t g, float (&v)[7]) const {
    const v3 lo = mk(bounds[0], bounds[1], bounds[2]);
    const v3 hi = mk(bounds[3], bounds[4], bounds[5]);
    const v3 ext = sub(hi, lo);
    const v3 inv = mk(ext.x > 0.0f ? 1.0f / ext.x : 0.0f, ext.y > 0.0f ? 1.0f / ext.y : 0.0f,
                      ext.z > 0.0f ? 1.0f / ext.z : 0.0f);
    const v3 p = mk(f[vplane(r, 0)], f[vplane(r, 1)], f[vplane(r, 2)]);
    const v3 n = mk(f[vplane(r, 3)], f[vplane(r, 4)], f[vplane(r, 5)]);
    const v3 d = mk(f[vplane(r, 6)], f[vplane(r, 7)], f[vplane(r, 8)]);
    const GuideInput gi = guide_input(p, n, normalize(mk(-d.x, -d.y, -d.z)), lo, inv);
#pragma unroll
    for (int s = 0; s < 7; ++s) {
      const int first = 4 * s / 3, next = first + 1 < kGuideInputs ? first + 1 : first;
      v[s] = chunk_input(s, g) == first ? gi.v[first] : gi.v[next];
    }
  }
};

// Bound by the encoding's arithmetic (about 400 instructions per lane and 16
// samples) beside the outputs' 160 bytes per sample; 524,309 inputs take
// 48 us, 102 with activations staged through LDS 16 samples at a time,
// element by element.
constexpr int kForwardBlock = 512;

template <typename Rows>
__global__ void __launch_bounds__(kForwardBlock) guide_forward_kernel(const uint8_t* __restrict__ pack, Rows rows,
                                                                      const uint32_t* __restrict__ count_dev,
                                                                      uint64_t count, float* __restrict__ out) {
  // outputs may start at any float
  typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4_any;
  __shared__ __attribute__((aligned(16))) uint16_t s_w[kPackFwd];
  __shared__ __attribute__((aligned(16))) float s_b[kBiasFloats];
  constexpr uint32_t kWaves = kForwardBlock / 64;
  uint64_t n = count;
  if (count_dev) n = *count_dev < count ? *count_dev : count;
  const uint64_t pairs = (n + 31) / 32;
  if ((uint64_t)blockIdx.x >= pairs) return;  // uniform per block: before the barrier
  load_pack(pack, s_w, kPackFwd, s_b, threadIdx.x);
  const uint32_t wave = threadIdx.x >> 6;
  // waves take neighbouring pairs across the grid, so that a short list spreads over the blocks
  for (uint64_t pair = (uint64_t)wave * gridDim.x + blockIdx.x; pair < pairs; pair += (uint64_t)gridDim.x * kWaves) {
    const uint32_t lane = fresh(lane_id());
    const uint32_t i = lane & 15u, g = lane >> 4;
    float sc[3];
    chunk_scales(g, sc);
    float x[2][7];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const uint64_t r = pair * 32 + 16 * u + i;
      rows.load(r < n ? r : n - 1, g, x[u]);
    }
    f32x4 acc[2][4];
    start_bias<4>(s_b, acc, g);
#pragma unroll
    for (int s = 0; s < 7; ++s) {
      bf16x8 f[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) f[u] = encode_chunk(x[u][s], sc[s % 3], s == 6 && g == 3);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const bf16x8 w = frag16(s_w + kPackW1 + (16 * t + i) * kW1Stride + 32 * s + 8 * g);
#pragma unroll
        for (int u = 0; u < 2; ++u) acc[u][t] = mfma(w, f[u], acc[u][t]);
      }
    }
    bf16x8 h[2][2];
    hidden_frags(acc, h);
    start_bias<4>(s_b + 64, acc, g);
    layer64<4>(s_w + kPackW2, h, acc, lane);
    hidden_frags(acc, h);
    start_bias<4>(s_b + 128, acc, g);
    layer64<4>(s_w + kPackW3, h, acc, lane);
    hidden_frags(acc, h);
    f32x4 o[2][3];
    start_bias<3>(s_b + 192, o, g);
    layer64<3>(s_w + kPackW4, h, o, lane);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const uint64_t r = pair * 32 + 16 * u + i;
      if (r >= n) continue;
      float* row = out + r * kGuideOut + 4 * g;
      *(f32x4_any*)row = o[u][0];
      *(f32x4_any*)(row + 16) = o[u][1];
      if (g < 2) *(f32x4_any*)(row + 32) = o[u][2];
    }
  }
}

// ---- loss gradient of one sample (outputs -> d loss / d outputs) ------------------
// Sum and maximum over the four lanes of a sample (the same in each).
BJ_D float sample_sum(float v) {
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}
BJ_D float sample_max(float v) {
  v = fmax_sel(v, __shfl_xor(v, 16, 64));
  return fmax_sel(v, __shfl_xor(v, 32, 64));
}

// Loss -w ln q(dir), q = sum_j pi_j vMF_j(dir) in log space; each of a
// sample's four lanes takes two lobes (`o`: their 10 outputs, `d`: the
// gradients).  Returns the sample's weighted loss.
BJ_D float output_gradient(const float (&o)[10], v3 dir, float w, float (&d)[10]) {
  float lp[2], lc[2], kap[2], mdw[2], len[2], e2v[2];
  v3 mu[2];
  bool inside[2];
  const float amax = sample_max(fmax_sel(o[4], o[9]));
  const float lse_a = amax + ln_f(sample_sum(exp_f(o[4] - amax) + exp_f(o[9] - amax)));
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const float* oj = o + 5 * j;
    const float l2 = oj[0] * oj[0] + oj[1] * oj[1] + oj[2] * oj[2];
    len[j] = sqrtf(l2);
    mu[j] = l2 > 1.0e-24f ? mk(oj[0] / len[j], oj[1] / len[j], oj[2] / len[j]) : mk(0.0f, 0.0f, 1.0f);
    inside[j] = oj[3] > kGuideLogKappaMin && oj[3] < kGuideLogKappaMax;
    const float s = fmin_sel(fmax_sel(oj[3], kGuideLogKappaMin), kGuideLogKappaMax);
    kap[j] = exp_f(s);
    e2v[j] = exp_f(-2.0f * kap[j]);
    mdw[j] = dot(mu[j], dir);
    lp[j] = oj[4] - lse_a;
    lc[j] = lp[j] + (s - kLn2Pi - ln_f(1.0f - e2v[j])) + kap[j] * (mdw[j] - 1.0f);
  }
  const float cmax = sample_max(fmax_sel(lc[0], lc[1]));
  const float lq = cmax + ln_f(sample_sum(exp_f(lc[0] - cmax) + exp_f(lc[1] - cmax)));
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const float r = exp_f(lc[j] - lq);
    const float pi = exp_f(lp[j]);
    d[5 * j + 4] = w * (pi - r);
    const float dlk = 1.0f / kap[j] - 2.0f * e2v[j] / (1.0f - e2v[j]) + (mdw[j] - 1.0f);
    d[5 * j + 3] = inside[j] ? -w * r * dlk * kap[j] : 0.0f;
    const float k = len[j] > 1.0e-12f ? -w * r * kap[j] / len[j] : 0.0f;
    d[5 * j + 0] = k * (dir.x - mdw[j] * mu[j].x);
    d[5 * j + 1] = k * (dir.y - mdw[j] * mu[j].y);
    d[5 * j + 2] = k * (dir.z - mdw[j] * mu[j].z);
  }
  return -w * lq;
}

// ---- training: forward, backward and the weight gradient ----------------------------
// Where the activation was 0 the delta is 0.
BJ_D bf16x8 masked(bf16x8 d, bf16x8 h) {
  const uint4 hw = __builtin_bit_cast(uint4, h);
  uint4 dw = __builtin_bit_cast(uint4, d);
  const auto keep = [](uint32_t v) { return ((v & 0xFFFFu) ? 0xFFFFu : 0u) | ((v >> 16) ? 0xFFFF0000u : 0u); };
  dw.x &= keep(hw.x);
  dw.y &= keep(hw.y);
  dw.z &= keep(hw.z);
  dw.w &= keep(hw.w);
  return __builtin_bit_cast(bf16x8, dw);
}

// The products of row tile k of a 64-wide layer with both sample tiles, in
// both orientations: n as layer64, t its transpose (lane: unit 16 k + i,
// elements: samples 4 g .. + 3).
BJ_D void tile_both(const uint16_t* sw, int k, const bf16x8 (&in)[2][2], f32x4 (&n)[2], f32x4 (&t)[2], uint32_t lane) {
  const uint32_t i = lane & 15u, g = lane >> 4;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const bf16x8 w = frag16(sw + (16 * k + i) * kRowStride + 32 * s + 8 * g);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      n[u] = mfma(w, in[u][s], n[u]);
      t[u] = mfma(in[u][s], w, t[u]);
    }
  }
}

// A hidden layer forward: h the next operand, ht the transposed activations:
// unit 16 k + i of samples 4 g .. + 3 of both sample tiles, one operand of
// the weight gradient (its K order is the same for both operands).  Row tile
// by row tile, so that few products are live beside what the gradient needs.
BJ_D void forward_both(const uint16_t* sw, const float* bias, const bf16x8 (&in)[2][2], bf16x8 (&h)[2][2],
                       bf16x8 (&ht)[4], uint32_t lane) {
  const uint32_t i = lane & 15u, g = lane >> 4;
#pragma unroll
  for (int kp = 0; kp < 2; ++kp) {
    f32x4 n[2][2];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int k = 2 * kp + half;
      const float b = bias[16 * k + i];
      f32x4 t[2] = {f32x4{b, b, b, b}, f32x4{b, b, b, b}};
      n[half][0] = n[half][1] = *(const f32x4*)(bias + 16 * k + 4 * g);
      tile_both(sw, k, in, n[half], t, lane);
      ht[k] = to_frag(relu4(t[0]), relu4(t[1]));
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) h[u][kp] = to_frag(relu4(n[0][u]), relu4(n[1][u]));
  }
}

// A layer backward: the deltas of its inputs, masked by their activations
// (h, ht), as the next operand and transposed.
BJ_D void backward_both(const uint16_t* sw, const bf16x8 (&in)[2][2], const bf16x8 (&h)[2][2], const bf16x8 (&ht)[4],
                        bf16x8 (&d)[2][2], bf16x8 (&dt)[4], uint32_t lane) {
#pragma unroll
  for (int kp = 0; kp < 2; ++kp) {
    f32x4 n[2][2];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int k = 2 * kp + half;
      const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
      f32x4 t[2] = {zero, zero};
      n[half][0] = n[half][1] = zero;
      tile_both(sw, k, in, n[half], t, lane);
      dt[k] = masked(to_frag(t[0], t[1]), ht[k]);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) d[u][kp] = masked(to_frag(n[0][u], n[1][u]), h[u][kp]);
  }
}

struct TrainArgs {
  const float* samples;  // f32[13 * src_count]
  // batch row r is sample (src_offset + r * src_stride) % src_count
  uint64_t src_count, src_offset, src_stride;
  uint64_t n;            // samples
  float* part;           // [block][kTiles][256] weight gradients
  double* loss_part;     // per block: sum of weights, weighted loss
};

// Fragments of the weight gradient in LDS: [fragment][wave of the samples][lane].
constexpr int kExchangeFrags = 14 + 4;  // layer 1, the largest: features and deltas
constexpr size_t kExchangeBytes = (size_t)kExchangeFrags * kTrainWaves * 64 * 16;
constexpr int kOutRow = 44;             // floats of a sample's outputs (16-byte rows)
constexpr size_t kOutBytes = (size_t)kTrainWaves * 32 * kOutRow * 4;
static_assert((size_t)kPackAll * 2 + kOutBytes <= kExchangeBytes, "weights and outputs share the exchange's LDS");

// kN gradient tiles (first, first + 1, ...) over the block's samples: deltas
// at fragment `a`, inputs at fragments `b`, `b` + 1, ...; fragment index -1 is
// the constant input in column `i == 0`.
template <int kN>
BJ_D void gradient_tiles(const uint4* ex, int a, const int (&b)[kN], float* part, int first, bool add, uint32_t lane) {
  f32x4 acc[kN];
  float* at = part + (size_t)first * 256 + lane * 4;
#pragma unroll
  for (int t = 0; t < kN; ++t) acc[t] = add ? *(const f32x4*)(at + 256 * t) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const uint32_t one = (lane & 15u) == 0 ? 0x3F803F80u : 0u;
#pragma unroll 2
  for (int w = 0; w < kTrainWaves; ++w) {
    const bf16x8 d = __builtin_bit_cast(bf16x8, ex[(a * kTrainWaves + w) * 64 + lane]);
#pragma unroll
    for (int t = 0; t < kN; ++t) {
      const uint4 x = b[t] >= 0 ? ex[(b[t] * kTrainWaves + w) * 64 + lane] : uint4{one, one, one, one};
      acc[t] = mfma(d, __builtin_bit_cast(bf16x8, x), acc[t]);
    }
  }
#pragma unroll
  for (int t = 0; t < kN; ++t) *(f32x4*)(at + 256 * t) = acc[t];
}

// Inputs below this have finite features at every frequency.
constexpr float kLargeInput = 1e30f;

// One launch per batch, 256 samples per block and pass.  Latency bound: one
// wave's chain of four layers, the loss and three layers back, then three
// exchanges.  65,521 samples: 38 us; 85 + 62 us as a pass that wrote
// every activation and delta to memory in BF16 (92 MB) and a batch-reduction
// kernel that read them.
__global__ void __launch_bounds__(kTrainWaves * 64) guide_train_kernel(const uint8_t* __restrict__ pack, TrainArgs ta) {
  __shared__ __attribute__((aligned(16))) uint8_t s_mem[kExchangeBytes];
  __shared__ __attribute__((aligned(16))) float s_b[kBiasFloats];
  __shared__ float s_loss[kTrainWaves * 2][2];
  __shared__ uint32_t s_nan;  // chunks of the features that were not numbers
  if (threadIdx.x == 0) s_nan = 0;
  uint16_t* s_w = (uint16_t*)s_mem;
  uint4* ex = (uint4*)s_mem;
  float* part = ta.part + (size_t)blockIdx.x * kTiles * 256;
  double block_w = 0.0, block_l = 0.0;
  for (uint64_t base = (uint64_t)blockIdx.x * kTrainSamples; base < ta.n; base += (uint64_t)gridDim.x * kTrainSamples) {
    const bool add = base != (uint64_t)blockIdx.x * kTrainSamples;
    const uint32_t tid = fresh(threadIdx.x), lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t i = lane & 15u, g = lane >> 4;
    float* s_out = (float*)(s_mem + (size_t)kPackAll * 2) + wave * 32 * kOutRow;
    float sc[3];
    chunk_scales(g, sc);
    load_pack(pack, s_w, kPackAll, s_b, tid);
    const float* sp[2];
    bool real[2];
    float x[2][7];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const uint64_t r = base + wave * 32 + 16 * u + i;
      real[u] = r < ta.n;
      const uint64_t row = real[u] ? (ta.src_offset + r * ta.src_stride) % ta.src_count : 0;
      sp[u] = ta.samples + row * kGuideSampleFloats;
#pragma unroll
      for (int s = 0; s < 7; ++s) x[u][s] = real[u] ? sp[u][chunk_input(s, g)] : 0.0f;
    }
    // Chunks of features that are not numbers are marked.  Their sample's
    // hidden units are off (ReLU of a NaN is 0), so nothing but the weights of
    // the chunk's own columns depends on them.
    bool large = false;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int s = 0; s < 7; ++s) large = large || !(fabsf(x[u][s]) < kLargeInput);
    if (ballot(large) != 0) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int s = 0; s < 7; ++s)
          if (!(fabsf(x[u][s] * sc[s % 3]) < __builtin_inff()) && 4 * s + (int)g < 27)
            atomicOr(&s_nan, 1u << (4 * s + g));
    }
    bf16x8 h1t[4], h2t[4], h3t[4];
    bf16x8 h1[2][2], h2[2][2], h3[2][2];
    {
      f32x4 n[2][4], t[2][4];
      start_bias<4>(s_b, n, g);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float b = s_b[16 * k + i];
        t[0][k] = t[1][k] = f32x4{b, b, b, b};
      }
#pragma unroll
      for (int s = 0; s < 7; ++s) {
        bf16x8 f[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) f[u] = encode_chunk(x[u][s], sc[s % 3], s == 6 && g == 3);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const bf16x8 w = frag16(s_w + kPackW1 + (16 * k + i) * kW1Stride + 32 * s + 8 * g);
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            n[u][k] = mfma(w, f[u], n[u][k]);
            t[u][k] = mfma(f[u], w, t[u][k]);
          }
        }
      }
      hidden_frags(n, h1);
#pragma unroll
      for (int k = 0; k < 4; ++k) h1t[k] = to_frag(relu4(t[0][k]), relu4(t[1][k]));
    }
    forward_both(s_w + kPackW2, s_b + 64, h1, h2, h2t, lane);
    forward_both(s_w + kPackW3, s_b + 128, h2, h3, h3t, lane);
    f32x4 o[2][3];
    start_bias<3>(s_b + 192, o, g);
    layer64<3>(s_w + kPackW4, h3, o, lane);
    __builtin_amdgcn_sched_barrier(0);
    // outputs to rows of samples; a sample's four lanes take two lobes each
    bf16x8 dof[2][2], dot[3], d3t[4], d2t[4], d1t[4];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float* row = s_out + (16 * u + i) * kOutRow;
#pragma unroll
      for (int k = 0; k < 3; ++k)
        if (k < 2 || g < 2) *(f32x4*)(row + 16 * k + 4 * g) = o[u][k];
      __builtin_amdgcn_wave_barrier();
      float lobe[10], d[10];
#pragma unroll
      for (int k = 0; k < 10; ++k) lobe[k] = row[10 * g + k];
      const v3 dir = real[u] ? mk(sp[u][9], sp[u][10], sp[u][11]) : mk(0.0f, 0.0f, 1.0f);
      const float w = real[u] ? sp[u][12] : 0.0f;
      const float loss = output_gradient(lobe, dir, w, d);
#pragma unroll
      for (int k = 0; k < 10; ++k) row[10 * g + k] = d[k];
      float wsum = w, lsum = w > 0.0f ? loss : 0.0f;
#pragma unroll
      for (int off = 8; off >= 1; off >>= 1) {
        wsum += __shfl_xor(wsum, off, 64);
        lsum += __shfl_xor(lsum, off, 64);
      }
      if (lane == 0) {
        s_loss[2 * wave + u][0] = wsum;
        s_loss[2 * wave + u][1] = lsum;
      }
    }
    __builtin_amdgcn_wave_barrier();
    {
      const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const float* row = s_out + (16 * u + i) * kOutRow + 4 * g;
        dof[u][0] = to_frag(*(const f32x4*)row, *(const f32x4*)(row + 16));
        dof[u][1] = to_frag(g < 2 ? *(const f32x4*)(row + 32) : zero, zero);
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        f32x4 c[2] = {zero, zero};
        if (k < 2 || i < 8)
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < 4; ++r) c[u][r] = s_out[(16 * u + 4 * g + r) * kOutRow + 16 * k + i];
        dot[k] = to_frag(c[0], c[1]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // backward: d3 = W4^T dO, masked by h3; then d2, d1 (its transpose only)
    bf16x8 d3[2][2], d2[2][2];
    backward_both(s_w + kPackW4t, dof, h3, h3t, d3, d3t, lane);
    backward_both(s_w + kPackW3t, d3, h2, h2t, d2, d2t, lane);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
      f32x4 t[2] = {zero, zero};
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const bf16x8 w = frag16(s_w + kPackW2t + (16 * k + i) * kRowStride + 32 * s + 8 * g);
#pragma unroll
        for (int u = 0; u < 2; ++u) t[u] = mfma(d2[u][s], w, t[u]);
      }
      d1t[k] = masked(to_frag(t[0], t[1]), h1t[k]);
    }
    __builtin_amdgcn_sched_barrier(0);
    // weight gradients; each exchange waits for the last one's readers
    const auto put = [&](int f, bf16x8 v) { ex[(f * kTrainWaves + wave) * 64 + lane] = __builtin_bit_cast(uint4, v); };
    __syncthreads();
    if (threadIdx.x == 0)
      for (int k = 0; k < 2 * kTrainWaves; ++k) {
        block_w += (double)s_loss[k][0];
        block_l += (double)s_loss[k][1];
      }
    // the features' transpose is their product with unit columns (encoded
    // again: kept from layer 1 they would not fit the registers).  It would
    // spread a feature that is not a number over its block of 32: an input
    // that has some counts as 0 here (from 2^24 turns on the finite features
    // are those of 0), and the columns marked above are set below.
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int s = 0; s < 7; ++s) {
        asm volatile("" : "+v"(x[u][s]));
        x[u][s] = fabsf(x[u][s]) < kLargeInput ? x[u][s] : 0.0f;
      }
    bf16x8 unit[2];
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int e = 0; e < 8; ++e) unit[half][e] = (__bf16)(8 * g + e == 16 * half + i ? 1.0f : 0.0f);
#pragma unroll
    for (int s = 0; s < 7; ++s) {
      bf16x8 f[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) f[u] = encode_chunk(x[u][s], sc[s % 3], s == 6 && g == 3);
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
        put(2 * s + half, to_frag(mfma(f[0], unit[half], zero), mfma(f[1], unit[half], zero)));
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) put(14 + k, d1t[k]);
    __syncthreads();
    {  // layer 1: wave w takes rows 16 (w % 4) .. + 15, seven of the 14 column tiles
      const int m = (int)wave & 3, c = 7 * ((int)wave >> 2);
      const int b[7] = {c, c + 1, c + 2, c + 3, c + 4, c + 5, c + 6};
      gradient_tiles<7>(ex, 14 + m, b, part, kT1 + 14 * m + c, add, lane);
      const uint32_t nans = s_nan;
      if (nans)
        for (int t = 0; t < 7; ++t)
          if ((nans >> (2u * (uint32_t)(c + t) + (i >> 3))) & 1u)  // chunk of column 16 (c + t) + i
            for (int r = 0; r < 4; ++r) part[(size_t)(kT1 + 14 * m + c + t) * 256 + lane * 4 + r] = __builtin_nanf("");
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      __builtin_amdgcn_sched_barrier(0);
      put(k, h1t[k]);
      put(4 + k, h2t[k]);
      put(8 + k, d2t[k]);
      put(12 + k, d3t[k]);
    }
    __syncthreads();
    {  // layers 2 and 3: one row of five tiles (the last holds the biases) per wave
      const int m = (int)wave & 3, c = 4 * ((int)wave >> 2);
      const int b[5] = {c, c + 1, c + 2, c + 3, -1};
      gradient_tiles<5>(ex, 8 + c + m, b, part, (wave < 4 ? kT2 : kT3) + 5 * m, add, lane);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) put(k, h3t[k]);
#pragma unroll
    for (int k = 0; k < 3; ++k) put(4 + k, dot[k]);
    __syncthreads();
    if (wave < 6) {  // layer 4: three rows of five tiles, two waves per row
      const int m = (int)wave >> 1;
      if (wave & 1u) {
        const int b[2] = {3, -1};
        gradient_tiles<2>(ex, 4 + m, b, part, kT4 + 5 * m + 3, add, lane);
      } else {
        const int b[3] = {0, 1, 2};
        gradient_tiles<3>(ex, 4 + m, b, part, kT4 + 5 * m, add, lane);
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    ta.loss_part[2 * blockIdx.x] = block_w;
    ta.loss_part[2 * blockIdx.x + 1] = block_l;
  }
}

// ---- reduce + Adam ----------------------------------------------------------------
struct AdamArgs {
  float* params;
  float* m;
  float* v;
  uint8_t* pack;
  float* ema;            // moving average of the weights and its weight images
  uint8_t* infer_pack;
  float ema_decay;
  const float* part;
  const double* loss_part;
  uint32_t blocks;       // partials
  float lr, beta1, beta2, eps, bias1, bias2;  // bias1/2 = 1 - beta^t
  float* grad_out;  // gradient mode: write the gradient, no update
};

// Decay of the weights' moving average that renders sample from: the last
// steps of a frame are noisy (lr 1e-2 on one frame's samples), and the
// average over about 100 steps is the steadier guide.
constexpr float kEmaDecay = 0.99f;

// One block per 64 elements of a gradient tile (elements that are no
// parameter's are skipped at the end): its 16 waves sum every 16th partial
// each, so that up to 256 partials (29 MB) are read with 16 loads in flight
// per wave; 7.7 us, 16.5 with one thread per parameter over 32 partials.
constexpr int kAdamWaves = 16;

__global__ void __launch_bounds__(kAdamWaves * 64) guide_adam_kernel(AdamArgs aa) {
  __shared__ float s_sum[kAdamWaves][64];
  const uint32_t lane = lane_id(), wave = threadIdx.x >> 6;
  const uint32_t at = blockIdx.x * 64 + lane;  // tile * 256 + element
  float acc = 0.0f;
#pragma unroll 16
  for (uint32_t b = wave; b < aa.blocks; b += kAdamWaves) acc += aa.part[(uint64_t)b * (kTiles * 256) + at];
  s_sum[wave][lane] = acc;
  __syncthreads();
  if (wave) return;
  double weights = 0.0;
  for (uint32_t b = lane; b < aa.blocks; b += 64) weights += aa.loss_part[2 * b];
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) weights += __shfl_xor(weights, off, 64);
  const float wsum = (float)weights;
  const int p = slot_param((int)(at >> 8), (int)(at & 255u));
  if (p < 0) return;
  float gsum = 0.0f;
#pragma unroll
  for (int w = 0; w < kAdamWaves; ++w) gsum += s_sum[w][lane];
  const ParamSlot sl = param_slot(p);
  const float grad = wsum > 0.0f ? gsum / wsum : 0.0f;
  if (aa.grad_out) {
    aa.grad_out[p] = grad;
    return;
  }
  const float m = aa.beta1 * aa.m[p] + (1.0f - aa.beta1) * grad;
  const float v = aa.beta2 * aa.v[p] + (1.0f - aa.beta2) * grad * grad;
  aa.m[p] = m;
  aa.v[p] = v;
  const float mh = m / aa.bias1, vh = v / aa.bias2;
  const float w = aa.params[p] - aa.lr * mh / (sqrtf(vh) + aa.eps);
  aa.params[p] = w;
  pack_param(aa.pack, sl, w);
  const float e = aa.ema_decay * aa.ema[p] + (1.0f - aa.ema_decay) * w;
  aa.ema[p] = e;
  pack_param(aa.infer_pack, sl, e);
}

// ---- mixture sampling (tests and tools) ---------------------------------------------
__global__ void __launch_bounds__(256) guide_mixture_kernel(const float* __restrict__ outputs, uint64_t n,
                                                            const float* __restrict__ u, float* __restrict__ dirs,
                                                            float* __restrict__ pdfs) {
  const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  GuideMixture m;
  guide_decode(outputs + r * kGuideOut, m);
  const v3 d = guide_sample(m, outputs + r * kGuideOut, u[3 * r], u[3 * r + 1], u[3 * r + 2]);
  dirs[3 * r] = d.x;
  dirs[3 * r + 1] = d.y;
  dirs[3 * r + 2] = d.z;
  pdfs[r] = guide_pdf(m, d);
}

// ---- host -------------------------------------------------------------------------
struct Pcg32 {
  uint64_t state = 0, inc = 0;
  Pcg32(uint64_t initstate, uint64_t initseq) {
    inc = (initseq << 1u) | 1u;
    next();
    state += initstate;
    next();
  }
  uint32_t next() {
    const uint64_t old = state;
    state = old * 6364136223846793005ULL + inc;
    const uint32_t xs = (uint32_t)(((old >> 18u) ^ old) >> 27u);
    const uint32_t rot = (uint32_t)(old >> 59u);
    return (xs >> rot) | (xs << ((-rot) & 31));
  }
  float uniform() { return (float)(next() >> 8) * (1.0f / 16777216.0f); }
};

// He-uniform weights (bound sqrt(6 / fan_in)), output layer scaled by 0.1,
// zero biases, drawn in parameter order from PCG32(seed, 54).
void init_params(uint64_t seed, std::vector<float>& p) {
  p.assign(kGuideParams, 0.0f);
  Pcg32 rng(seed, 54);
  auto fill = [&](int off, int rows, int fan_in, float gain) {
    const float bound = gain * sqrtf(6.0f / (float)fan_in);
    for (int k = 0; k < rows * fan_in; ++k) p[off + k] = (2.0f * rng.uniform() - 1.0f) * bound;
  };
  fill(kGuideOffW1, kGuideHidden, kGuideFeatures, 1.0f);
  fill(kGuideOffW2, kGuideHidden, kGuideHidden, 1.0f);
  fill(kGuideOffW3, kGuideHidden, kGuideHidden, 1.0f);
  fill(kGuideOffW4, kGuideOut, kGuideHidden, 0.1f);
}

int32_t upload_params(bajo_ctx* ctx, bajo_guide* g, const float* host) {
  BJ_HIP(hipMemcpyAsync(g->params, host, kGuideParams * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
  BJ_HIP(hipMemsetAsync(g->adam_m, 0, kGuideParams * sizeof(float), ctx->stream));
  BJ_HIP(hipMemsetAsync(g->adam_v, 0, kGuideParams * sizeof(float), ctx->stream));
  BJ_HIP(hipMemcpyAsync(g->ema, g->params, kGuideParams * sizeof(float), hipMemcpyDeviceToDevice, ctx->stream));
  guide_pack_kernel<<<div_up(kGuideParams, 256), 256, 0, ctx->stream>>>(g->params, g->pack);
  guide_pack_kernel<<<div_up(kGuideParams, 256), 256, 0, ctx->stream>>>(g->params, g->infer_pack);
  BJ_HIP(hipGetLastError());
  g->step = 0;
  return BAJO_OK;
}

void free_guide(bajo_guide* g) {
  if (!g) return;
  (void)hipFree(g->params); (void)hipFree(g->adam_m); (void)hipFree(g->adam_v); (void)hipFree(g->pack);
  (void)hipFree(g->ema); (void)hipFree(g->infer_pack);
  (void)hipFree(g->loss_part); (void)hipFree(g->grad_part);
  (void)hipFree(g->records); (void)hipFree(g->contrib); (void)hipFree(g->samples); (void)hipFree(g->sample_count);
  (void)hipFree(g->block_counts);
  (void)hipFree(g->vertices); (void)hipFree(g->outputs);
  delete g;
}

template <typename K>
int32_t blocks_per_cu(K kernel, int* out) {
  int dev = 0, cus = 0, per_cu = 0;
  BJ_HIP(hipGetDevice(&dev));
  BJ_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  BJ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kForwardBlock, 0));
  *out = cus * (per_cu < 1 ? 1 : per_cu);
  return BAJO_OK;
}

// Blocks of one training pass over n samples.
uint32_t train_blocks(uint64_t n) {
  const uint64_t need = (n + kTrainSamples - 1) / kTrainSamples;
  return (uint32_t)(need < kTrainBlocks ? need : kTrainBlocks);
}

// Weight-gradient and loss partials of one batch (n <= batch_cap), one per block.
int32_t run_backward(hipStream_t stream, bajo_guide* g, const float* samples, uint64_t src_count, uint64_t src_offset,
                     uint64_t src_stride, uint64_t n, uint32_t* blocks) {
  *blocks = train_blocks(n);
  TrainArgs ta{samples, src_count, src_offset, src_stride, n, g->grad_part, g->loss_part};
  guide_train_kernel<<<*blocks, kTrainWaves * 64, 0, stream>>>(g->pack, ta);
  BJ_HIP(hipGetLastError());
  return BAJO_OK;
}

// The batch's mean loss from its partials (synchronizes).
int32_t read_loss(hipStream_t stream, const bajo_guide* g, uint32_t blocks, float* loss) {
  double part[2 * kTrainBlocks];
  BJ_HIP(hipMemcpyAsync(part, g->loss_part, 2 * blocks * sizeof(double), hipMemcpyDeviceToHost, stream));
  BJ_HIP(hipStreamSynchronize(stream));
  double ws = 0.0, ls = 0.0;
  for (uint32_t k = 0; k < blocks; ++k) {
    ws += part[2 * k];
    ls += part[2 * k + 1];
  }
  *loss = ws > 0.0 ? (float)(ls / ws) : 0.0f;
  return BAJO_OK;
}

int32_t run_adam(hipStream_t stream, bajo_guide* g, uint32_t blocks, float* grad_out) {
  AdamArgs aa;
  aa.params = g->params;
  aa.m = g->adam_m;
  aa.v = g->adam_v;
  aa.pack = g->pack;
  aa.ema = g->ema;
  aa.infer_pack = g->infer_pack;
  aa.part = g->grad_part;
  aa.loss_part = g->loss_part;
  aa.blocks = blocks;
  aa.lr = g->opt.learning_rate;
  aa.beta1 = g->opt.beta1;
  aa.beta2 = g->opt.beta2;
  aa.eps = g->opt.epsilon;
  aa.grad_out = grad_out;
  aa.ema_decay = 0.0f;
  if (!grad_out) {
    g->step += 1;
    aa.bias1 = 1.0f - powf(g->opt.beta1, (float)g->step);
    aa.bias2 = 1.0f - powf(g->opt.beta2, (float)g->step);
    // the average follows the first steps closely, then settles at kEmaDecay
    const float warm = (1.0f + (float)g->step) / (10.0f + (float)g->step);
    aa.ema_decay = warm < kEmaDecay ? warm : kEmaDecay;
  } else {
    aa.bias1 = aa.bias2 = 1.0f;
  }
  guide_adam_kernel<<<kTiles * 4, kAdamWaves * 64, 0, stream>>>(aa);
  BJ_HIP(hipGetLastError());
  return BAJO_OK;
}

}  // namespace

int32_t guide_train_samples(hipStream_t stream, bajo_guide* g, const float* samples, uint64_t n) {
  for (uint64_t b = 0; b < n; b += g->batch_cap) {
    const uint64_t m = n - b < g->batch_cap ? n - b : g->batch_cap;
    uint32_t blocks = 0;
    int32_t rc = run_backward(stream, g, samples, n, b, 1, m, &blocks);
    if (rc) return rc;
    rc = run_adam(stream, g, blocks, nullptr);
    if (rc) return rc;
  }
  return BAJO_OK;
}

namespace {

// The training sample of path p at bounce k, if it has one: the vertex's
// inputs, the direction taken, and as weight the radiance added at bounces
// after it over the throughput the path carried out of it (per channel), as
// luminance over the density its direction was drawn with.
BJ_D bool collect_sample(const float* __restrict__ records, const float* __restrict__ contrib, uint64_t p,
                         uint32_t k, uint32_t depth, v3 lo, v3 inv, float* out) {
  const float* r = records + (p * depth + k) * kRecordPlanes;
  const float pdf = r[12];
  if (!(pdf > 0.0f)) return false;
  v3 L = mk(0.0f, 0.0f, 0.0f);
  for (uint32_t j = k + 1; j < depth; ++j) {
    const float* c = contrib + 3 * (p * depth + j);
    L = add(L, mk(c[0], c[1], c[2]));
  }
  const v3 T = mk(r[13], r[14], r[15]);
  L = mk(T.x > 0.0f ? L.x / T.x : 0.0f, T.y > 0.0f ? L.y / T.y : 0.0f, T.z > 0.0f ? L.z / T.z : 0.0f);
  const float lum = 0.2126f * L.x + 0.7152f * L.y + 0.0722f * L.z;
  if (!(lum > 0.0f)) return false;
  const GuideInput gi = guide_input(mk(r[0], r[1], r[2]), mk(r[3], r[4], r[5]), mk(r[6], r[7], r[8]), lo, inv);
#pragma unroll
  for (int a = 0; a < kGuideInputs; ++a) out[a] = gi.v[a];
  out[9] = r[9];
  out[10] = r[10];
  out[11] = r[11];
  out[12] = lum / pdf;
  return true;
}

BJ_D void bounds_frame(const float* __restrict__ bounds, v3& lo, v3& inv) {
  lo = mk(bounds[0], bounds[1], bounds[2]);
  const v3 ext = sub(mk(bounds[3], bounds[4], bounds[5]), lo);
  inv = mk(ext.x > 0.0f ? 1.0f / ext.x : 0.0f, ext.y > 0.0f ? 1.0f / ext.y : 0.0f, ext.z > 0.0f ? 1.0f / ext.z : 0.0f);
}

// The frame's samples are stored in a fixed order -- block by block (256
// paths each), bounce by bounce within a block, then path order -- so the
// training batches, and the trained network, do not depend on the order in
// which waves run.  Pass 1 counts each block's samples.
__global__ void __launch_bounds__(256) guide_count_kernel(const float* __restrict__ records,
                                                          const float* __restrict__ contrib, uint64_t paths,
                                                          uint32_t depth, const float* __restrict__ bounds,
                                                          uint32_t* __restrict__ block_counts) {
  __shared__ uint32_t s_wave[4];
  const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  v3 lo, inv;
  bounds_frame(bounds, lo, inv);
  uint32_t mine = 0;
  float out[kGuideSampleFloats];
  if (p < paths)
    for (uint32_t k = 0; k < depth; ++k) mine += collect_sample(records, contrib, p, k, depth, lo, inv, out) ? 1u : 0u;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) mine += (uint32_t)__shfl_xor((int)mine, off, 64);
  if (lane_id() == 0) s_wave[threadIdx.x >> 6] = mine;
  __syncthreads();
  if (threadIdx.x == 0) block_counts[blockIdx.x] = s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
}

// Pass 2 (one block): exclusive prefix of the block counts, in place; the
// total becomes the frame's sample count.
__global__ void __launch_bounds__(1024) guide_offsets_kernel(uint32_t* __restrict__ block_counts, uint32_t blocks,
                                                             uint32_t* __restrict__ count) {
  __shared__ uint32_t s_wave[16];
  __shared__ uint32_t s_carry;
  if (threadIdx.x == 0) s_carry = 0;
  __syncthreads();
  const uint32_t lane = lane_id(), wave = threadIdx.x >> 6;
  for (uint32_t base = 0; base < blocks; base += blockDim.x) {
    const uint32_t i = base + threadIdx.x;
    const uint32_t v = i < blocks ? block_counts[i] : 0u;
    uint32_t incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = (uint32_t)__shfl_up((int)incl, off, 64);
      if (lane >= (uint32_t)off) incl += y;
    }
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    uint32_t before = s_carry;
    for (uint32_t w = 0; w < wave; ++w) before += s_wave[w];
    if (i < blocks) block_counts[i] = before + incl - v;
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t t = 0;
      for (uint32_t w = 0; w < blockDim.x / 64; ++w) t += s_wave[w];
      s_carry += t;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) count[0] = s_carry;
}

// Pass 3: each block writes its samples from its offset, bounce by bounce,
// in path order.
__global__ void __launch_bounds__(256) guide_collect_kernel(const float* __restrict__ records,
                                                            const float* __restrict__ contrib, uint64_t paths,
                                                            uint32_t depth, const float* __restrict__ bounds,
                                                            const uint32_t* __restrict__ block_offsets,
                                                            float* __restrict__ samples, uint64_t cap) {
  __shared__ uint32_t s_wave[4];
  const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t lane = lane_id(), wave = threadIdx.x >> 6;
  v3 lo, inv;
  bounds_frame(bounds, lo, inv);
  uint64_t next = block_offsets[blockIdx.x];
  for (uint32_t k = 0; k < depth; ++k) {
    float out[kGuideSampleFloats];
    const bool want = p < paths && collect_sample(records, contrib, p, k, depth, lo, inv, out);
    const uint64_t m = ballot(want);
    if (lane == 0) s_wave[wave] = (uint32_t)__builtin_popcountll(m);
    __syncthreads();
    uint32_t before = 0, total = 0;
    for (uint32_t w = 0; w < 4; ++w) {
      if (w < wave) before += s_wave[w];
      total += s_wave[w];
    }
    const uint64_t slot = next + before + mask_rank(m);
    if (want && slot < cap)
#pragma unroll
      for (int a = 0; a < kGuideSampleFloats; ++a) samples[slot * kGuideSampleFloats + a] = out[a];
    next += total;
    __syncthreads();
  }
}

uint64_t gcd_u64(uint64_t a, uint64_t b) {
  while (b) {
    const uint64_t t = a % b;
    a = b;
    b = t;
  }
  return a;
}

}  // namespace

int32_t guide_infer_vertices(hipStream_t stream, const bajo_guide* g, const float* vertex_fields,
                             const uint32_t* count_dev, uint64_t cap, const float* scene_bounds, float* outputs) {
  int grid = 0;
  int32_t rc = blocks_per_cu(guide_forward_kernel<VertexRows>, &grid);
  if (rc) return rc;
  const uint64_t need = (cap + 31) / 32;
  if ((uint64_t)grid > need) grid = (int)need;
  guide_forward_kernel<VertexRows><<<grid, kForwardBlock, 0, stream>>>(g->infer_pack, VertexRows{vertex_fields, scene_bounds},
                                                             count_dev, cap, outputs);
  BJ_HIP(hipGetLastError());
  return BAJO_OK;
}

int32_t guide_prepare_frame(hipStream_t stream, bajo_guide* g, uint64_t paths, uint32_t depth, bool train) {
  if (paths > g->vertex_cap) {
    BJ_HIP(hipStreamSynchronize(stream));
    (void)hipFree(g->vertices);
    (void)hipFree(g->outputs);
    g->vertices = g->outputs = nullptr;
    g->vertex_cap = 0;
    const uint64_t tiles = (paths + 63) / 64;
    BJ_HIP(hipMalloc(&g->vertices, tiles * 64 * kVertexPlanes * sizeof(float)));
    BJ_HIP(hipMalloc(&g->outputs, paths * kGuideOut * sizeof(float)));
    g->vertex_cap = paths;
  }
  if (!train) return BAJO_OK;
  const uint64_t slots = paths * depth;
  if (slots > g->record_cap) {
    BJ_HIP(hipStreamSynchronize(stream));
    (void)hipFree(g->records);
    (void)hipFree(g->contrib);
    (void)hipFree(g->samples);
    g->records = g->contrib = g->samples = nullptr;
    g->record_cap = g->sample_cap = 0;
    BJ_HIP(hipMalloc(&g->records, slots * kRecordPlanes * sizeof(float)));
    BJ_HIP(hipMalloc(&g->contrib, slots * 3 * sizeof(float)));
    BJ_HIP(hipMalloc(&g->samples, slots * kGuideSampleFloats * sizeof(float)));
    g->record_cap = g->sample_cap = slots;
  }
  const uint64_t blocks = (paths + 255) / 256;
  if (blocks > g->block_cap) {
    BJ_HIP(hipStreamSynchronize(stream));
    (void)hipFree(g->block_counts);
    g->block_counts = nullptr;
    g->block_cap = 0;
    BJ_HIP(hipMalloc(&g->block_counts, blocks * sizeof(uint32_t)));
    g->block_cap = blocks;
  }
  BJ_HIP(hipMemsetAsync(g->records, 0, slots * kRecordPlanes * sizeof(float), stream));
  BJ_HIP(hipMemsetAsync(g->contrib, 0, slots * 3 * sizeof(float), stream));
  BJ_HIP(hipMemsetAsync(g->sample_count, 0, sizeof(uint32_t), stream));
  return BAJO_OK;
}

int32_t guide_collect(hipStream_t stream, bajo_guide* g, uint64_t paths, uint32_t depth, const float* scene_bounds) {
  const unsigned blocks = div_up(paths, 256);
  BJ_REQUIRE(blocks <= g->block_cap, "guide_collect: %u blocks, room for %llu", blocks,
             (unsigned long long)g->block_cap);
  guide_count_kernel<<<blocks, 256, 0, stream>>>(g->records, g->contrib, paths, depth, scene_bounds, g->block_counts);
  guide_offsets_kernel<<<1, 1024, 0, stream>>>(g->block_counts, blocks, g->sample_count);
  guide_collect_kernel<<<blocks, 256, 0, stream>>>(g->records, g->contrib, paths, depth, scene_bounds,
                                                  g->block_counts, g->samples, g->sample_cap);
  BJ_HIP(hipGetLastError());
  return BAJO_OK;
}

int32_t guide_train_collected(hipStream_t stream, bajo_guide* g, uint64_t* samples_out, uint32_t* steps_out,
                              float* loss_out) {
  uint32_t count = 0;
  BJ_HIP(hipMemcpyAsync(&count, g->sample_count, sizeof(count), hipMemcpyDeviceToHost, stream));
  BJ_HIP(hipStreamSynchronize(stream));
  const uint64_t total = count < g->sample_cap ? count : g->sample_cap;
  *samples_out = total;
  *steps_out = 0;
  *loss_out = 0.0f;
  if (total == 0) return BAJO_OK;
  const uint64_t n = total < g->batch_cap ? total : g->batch_cap;
  // a stride coprime with the set's size spreads each batch over the whole frame
  uint64_t stride = total / n;
  if (stride < 1) stride = 1;
  while (gcd_u64(stride, total) != 1) ++stride;
  uint32_t blocks = 0;
  for (uint32_t k = 0; k < g->opt.steps_per_frame; ++k) {
    const uint64_t offset = g->sample_cursor++ % total;
    int32_t rc = run_backward(stream, g, g->samples, total, offset, stride, n, &blocks);
    if (rc) return rc;
    rc = run_adam(stream, g, blocks, nullptr);
    if (rc) return rc;
    *steps_out += 1;
  }
  return read_loss(stream, g, blocks, loss_out);
}

}  // namespace bj

extern "C" {

int32_t bajo_guide_create(bajo_ctx* ctx, const bajo_guide_options* options, bajo_guide** out) {
  BJ_REQUIRE(ctx != nullptr && out != nullptr, "bajo_guide_create: NULL argument");
  *out = nullptr;
  bajo_guide_options o{};
  if (options) o = *options;
  if (!(o.learning_rate > 0.0f)) o.learning_rate = 1.0e-2f;
  if (!(o.beta1 > 0.0f)) o.beta1 = 0.9f;
  if (!(o.beta2 > 0.0f)) o.beta2 = 0.999f;
  if (!(o.epsilon > 0.0f)) o.epsilon = 1.0e-8f;
  if (o.batch_size == 0) o.batch_size = 65536;
  if (o.steps_per_frame == 0) o.steps_per_frame = 4;
  BJ_REQUIRE(o.batch_size % 32 == 0 && o.batch_size <= (1u << 22),
             "bajo_guide_create: batch_size %u must be a multiple of 32 and at most 2^22", o.batch_size);
  BJ_REQUIRE(o.beta1 < 1.0f && o.beta2 < 1.0f, "bajo_guide_create: Adam decays must be below 1");
  bajo_guide* g = new bajo_guide();
  g->device = ctx->device;
  g->opt = o;
  g->batch_cap = (o.batch_size + 2047) / 2048 * 2048;
  const uint32_t blocks = bj::train_blocks(g->batch_cap);
  auto fail = [&](hipError_t e, const char* what) {
    bj::free_guide(g);
    return bj::hip_fail(e, what, __FILE__, __LINE__);
  };
  hipError_t e = hipSuccess;
  if (e == hipSuccess) e = hipMalloc(&g->params, bj::kGuideParams * sizeof(float));
  if (e == hipSuccess) e = hipMalloc(&g->adam_m, bj::kGuideParams * sizeof(float));
  if (e == hipSuccess) e = hipMalloc(&g->adam_v, bj::kGuideParams * sizeof(float));
  if (e == hipSuccess) e = hipMalloc(&g->pack, bj::kPackBytes);
  if (e == hipSuccess) e = hipMalloc(&g->ema, bj::kGuideParams * sizeof(float));
  if (e == hipSuccess) e = hipMalloc(&g->infer_pack, bj::kPackBytes);
  if (e == hipSuccess) e = hipMalloc(&g->loss_part, (size_t)blocks * 2 * sizeof(double));
  if (e == hipSuccess) e = hipMalloc(&g->grad_part, (size_t)blocks * bj::kTiles * 256 * sizeof(float));
  if (e == hipSuccess) e = hipMalloc(&g->sample_count, 4 * sizeof(uint32_t));
  if (e != hipSuccess) return fail(e, "hipMalloc(guide)");
  // padding entries of the weight image stay zero
  e = hipMemsetAsync(g->pack, 0, bj::kPackBytes, ctx->stream);
  if (e == hipSuccess) e = hipMemsetAsync(g->infer_pack, 0, bj::kPackBytes, ctx->stream);
  if (e == hipSuccess) e = hipMemsetAsync(g->sample_count, 0, 4 * sizeof(uint32_t), ctx->stream);
  if (e != hipSuccess) return fail(e, "hipMemsetAsync(guide)");
  std::vector<float> p;
  bj::init_params(o.seed, p);
  int32_t rc = bj::upload_params(ctx, g, p.data());
  if (rc == BAJO_OK) {
    e = hipStreamSynchronize(ctx->stream);  // the host vector dies here
    if (e != hipSuccess) return fail(e, "hipStreamSynchronize(guide)");
  }
  if (rc) {
    bj::free_guide(g);
    return rc;
  }
  *out = g;
  return BAJO_OK;
}

int32_t bajo_guide_free(bajo_guide* guide) {
  if (guide) {
    (void)hipDeviceSynchronize();
    bj::free_guide(guide);
  }
  return BAJO_OK;
}

int32_t bajo_guide_get_params(bajo_ctx* ctx, const bajo_guide* guide, float* params) {
  BJ_REQUIRE(ctx && guide && params, "bajo_guide_get_params: NULL argument");
  BJ_HIP(hipMemcpyAsync(params, guide->params, bj::kGuideParams * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
  BJ_HIP(hipStreamSynchronize(ctx->stream));
  return BAJO_OK;
}

int32_t bajo_guide_set_params(bajo_ctx* ctx, bajo_guide* guide, const float* params) {
  BJ_REQUIRE(ctx && guide && params, "bajo_guide_set_params: NULL argument");
  int32_t rc = bj::upload_params(ctx, guide, params);
  if (rc) return rc;
  BJ_HIP(hipStreamSynchronize(ctx->stream));
  return BAJO_OK;
}

int32_t bajo_guide_forward(bajo_ctx* ctx, const bajo_guide* guide, const float* inputs, uint64_t n, float* outputs) {
  BJ_REQUIRE(ctx && guide, "bajo_guide_forward: NULL argument");
  BJ_REQUIRE(n == 0 || (inputs && outputs), "bajo_guide_forward: NULL buffer");
  if (n == 0) return BAJO_OK;
  int grid = 0;
  int32_t rc = bj::blocks_per_cu(bj::guide_forward_kernel<bj::InputRows>, &grid);
  if (rc) return rc;
  const uint64_t need = (n + 31) / 32;
  if ((uint64_t)grid > need) grid = (int)need;
  bj::guide_forward_kernel<bj::InputRows><<<grid, bj::kForwardBlock, 0, ctx->stream>>>(guide->pack, bj::InputRows{inputs}, nullptr,
                                                                         n, outputs);
  BJ_HIP(hipGetLastError());
  return BAJO_OK;
}

int32_t bajo_guide_gradient(bajo_ctx* ctx, bajo_guide* guide, const float* samples, uint64_t n, float* gradient,
                            float* loss) {
  BJ_REQUIRE(ctx && guide && gradient, "bajo_guide_gradient: NULL argument");
  BJ_REQUIRE(n > 0 && samples, "bajo_guide_gradient: empty batch");
  BJ_REQUIRE(n <= guide->batch_cap, "bajo_guide_gradient: %llu samples exceed the batch size %u",
             (unsigned long long)n, guide->batch_cap);
  uint32_t blocks = 0;
  int32_t rc = bj::run_backward(ctx->stream, guide, samples, n, 0, 1, n, &blocks);
  if (rc) return rc;
  rc = bj::run_adam(ctx->stream, guide, blocks, gradient);
  if (rc) return rc;
  return loss ? bj::read_loss(ctx->stream, guide, blocks, loss) : BAJO_OK;
}

int32_t bajo_guide_train(bajo_ctx* ctx, bajo_guide* guide, const float* samples, uint64_t n) {
  BJ_REQUIRE(ctx && guide, "bajo_guide_train: NULL argument");
  BJ_REQUIRE(n == 0 || samples, "bajo_guide_train: samples is NULL");
  return bj::guide_train_samples(ctx->stream, guide, samples, n);
}

int32_t bajo_guide_training_samples(bajo_ctx* ctx, const bajo_guide* guide, float* samples, uint64_t cap,
                                    uint64_t* count) {
  BJ_REQUIRE(ctx && guide && count, "bajo_guide_training_samples: NULL argument");
  BJ_REQUIRE(cap == 0 || samples, "bajo_guide_training_samples: samples is NULL");
  uint32_t c = 0;
  if (guide->sample_count) {
    BJ_HIP(hipMemcpyAsync(&c, guide->sample_count, sizeof(c), hipMemcpyDeviceToHost, ctx->stream));
    BJ_HIP(hipStreamSynchronize(ctx->stream));
  }
  uint64_t have = c < guide->sample_cap ? c : guide->sample_cap;
  *count = have;
  if (have > cap) have = cap;
  if (have) {
    BJ_HIP(hipMemcpyAsync(samples, guide->samples, have * bj::kGuideSampleFloats * sizeof(float),
                          hipMemcpyDeviceToHost, ctx->stream));
    BJ_HIP(hipStreamSynchronize(ctx->stream));
  }
  return BAJO_OK;
}

int32_t bajo_guide_mixture_sample(bajo_ctx* ctx, const float* outputs, uint64_t n, const float* uniforms, float* dirs,
                                  float* pdfs) {
  BJ_REQUIRE(ctx != nullptr, "bajo_guide_mixture_sample: ctx is NULL");
  BJ_REQUIRE(n == 0 || (outputs && uniforms && dirs && pdfs), "bajo_guide_mixture_sample: NULL buffer");
  if (n == 0) return BAJO_OK;
  bj::guide_mixture_kernel<<<bj::div_up(n, 256), 256, 0, ctx->stream>>>(outputs, n, uniforms, dirs, pdfs);
  BJ_HIP(hipGetLastError());
  return BAJO_OK;
}

}  // extern "C"

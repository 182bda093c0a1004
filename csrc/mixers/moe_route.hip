// Mixture-of-experts routing: softmax over all experts (fp32), an additive selection
// bias that does not enter the weights, group-limited selection (only the experts of
// the `keep` best of `groups` equal groups of neighbours stay eligible; a group's score
// is its best biased score; excluded experts count as -infinity), then the `top`
// eligible experts with the largest biased scores.  Weights = the chosen experts'
// unbiased softmax scores, not renormalised.  One wave per token; ties go to the lower
// index.  A second router (moe_top_logits) chooses on the logits and weights the chosen ones
// by the softmax over just those, or by their sigmoids divided by the sum of those, times a
// factor; there, too, the choice may be limited to the best groups, a group's score being the
// sum of its two largest sigmoids.
#include "route_choice.h"

namespace mx {

struct Best {
  float v;
  int i;
};

__device__ __forceinline__ Best better(Best a, Best b) {
  return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a;
}

__device__ __forceinline__ Best wave_best(Best x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    Best y;
    y.v = __shfl_xor(x.v, o, 64);
    y.i = __shfl_xor(x.i, o, 64);
    x = better(x, y);
  }
  return x;
}

// One wave: s [experts] holds a row's logits; its choice (see above).  ch [experts] and gs [groups] are scratch.
__device__ __forceinline__ void choose_softmax_all(int* idx, float* wts, float* s, float* ch, float* gs,
                                                   const float* corr, int experts, int top, int groups, int keep,
                                                   int lane) {
  float mx_ = -INFINITY;
  for (int e = lane; e < experts; e += 64) mx_ = fmaxf(mx_, s[e]);
  mx_ = ft::wave_max(mx_);
  float sum = 0.f;
  for (int e = lane; e < experts; e += 64) {
    const float p = expf(s[e] - mx_);
    s[e] = p;
    sum += p;
  }
  sum = ft::wave_sum(sum);
  for (int e = lane; e < experts; e += 64) {
    const float p = s[e] / sum;
    s[e] = p;                       // softmax scores
    ch[e] = p + corr[e];            // biased scores, -inf once excluded or taken
  }
  wave_lds_fence();
  if (groups > 1 && keep < groups) {
    const int gsz = experts / groups;
    for (int g = lane; g < groups; g += 64) {
      float b = -INFINITY;
      for (int e = g * gsz; e < (g + 1) * gsz; ++e) b = fmaxf(b, ch[e]);
      gs[g] = b;
    }
    wave_lds_fence();
    // the keep best groups get +inf as a mark; the others' experts are excluded
    for (int k = 0; k < keep; ++k) {
      Best b{-INFINITY, 1 << 30};
      for (int g = lane; g < groups; g += 64)
        if (gs[g] != INFINITY) b = better(b, Best{gs[g], g});
      b = wave_best(b);
      if (lane == 0 && b.i < groups) gs[b.i] = INFINITY;
      wave_lds_fence();
    }
    for (int e = lane; e < experts; e += 64)
      if (gs[e / gsz] != INFINITY) ch[e] = -INFINITY;
    wave_lds_fence();
  }
  for (int k = 0; k < top; ++k) {
    Best b{-INFINITY, 1 << 30};
    for (int e = lane; e < experts; e += 64) b = better(b, Best{ch[e], e});
    b = wave_best(b);
    const int e = b.i < experts ? b.i : 0;
    if (lane == 0) {
      idx[k] = e;
      wts[k] = s[e];
      ch[e] = -INFINITY;
    }
    wave_lds_fence();
  }
}

__global__ void __launch_bounds__(64)
moe_topk_kernel(int* __restrict__ idx, float* __restrict__ wts, const float* __restrict__ z,
                const float* __restrict__ corr, int experts, int top, int groups, int keep) {
  extern __shared__ float sm[];
  const long row = blockIdx.x;
  const int lane = threadIdx.x;
  for (int e = lane; e < experts; e += 64) sm[e] = z[row * experts + e];
  wave_lds_fence();
  choose_softmax_all(idx + row * top, wts + row * top, sm, sm + experts, sm + 2 * experts, corr, experts, top, groups,
                     keep, lane);
}

// One wave: the logits ch of every expert outside the `keep` best of `groups` equal groups
// become -inf.  A group's score is the sum of the sigmoids of its two largest logits (of its
// only one in a group of one); gs holds `groups` scores.
__device__ __forceinline__ void limit_to_best_groups(float* ch, float* gs, int experts, int groups, int keep, int lane) {
  const int gsz = experts / groups;
  for (int g = lane; g < groups; g += 64) {
    float a = -INFINITY, b = -INFINITY;
    for (int e = g * gsz; e < (g + 1) * gsz; ++e) {
      const float v = ch[e];
      if (v > a) { b = a; a = v; }
      else b = fmaxf(b, v);
    }
    gs[g] = sigmoidf_(a) + (gsz > 1 ? sigmoidf_(b) : 0.f);
  }
  wave_lds_fence();
  for (int k = 0; k < keep; ++k) {       // a kept group is marked by +inf
    Best b{-INFINITY, 1 << 30};
    for (int g = lane; g < groups; g += 64)
      if (gs[g] != INFINITY) b = better(b, Best{gs[g], g});
    b = wave_best(b);
    if (lane == 0 && b.i < groups) gs[b.i] = INFINITY;
    wave_lds_fence();
  }
  for (int e = lane; e < experts; e += 64)
    if (gs[e / gsz] != INFINITY) ch[e] = -INFINITY;
  wave_lds_fence();
}

// weights of the chosen logits val[0 .. top) (largest first), one wave
__device__ __forceinline__ void chosen_weights(float* w, const float* val, int top, int lane, int sigmoid, float scale) {
  auto f = [&](int k) { return sigmoid ? sigmoidf_(val[k]) : expf(val[k] - val[0]); };
  float sum = 0.f;
  for (int k = lane; k < top; k += 64) sum += f(k);
  sum = ft::wave_sum(sum);
  if (sigmoid) sum += 1e-20f;
  for (int k = lane; k < top; k += 64) w[k] = f(k) / sum * scale;
}

// Routing on the logits themselves: the `top` largest logits of a row are chosen (ties to
// the lower index) and weighted by chosen_weights.  One wave per token.
__global__ void __launch_bounds__(64)
moe_top_logits_kernel(int* __restrict__ idx, float* __restrict__ wts, const float* __restrict__ z, int experts,
                      int top, int sigmoid, float scale, int groups, int keep) {
  extern __shared__ float sm[];
  float* ch = sm;                   // logits, -inf once taken
  float* val = sm + experts;        // the chosen logits, largest first
  const long row = blockIdx.x;
  const int lane = threadIdx.x;
  const float* zr = z + row * experts;
  for (int e = lane; e < experts; e += 64) ch[e] = zr[e];
  __syncthreads();
  if (keep < groups) limit_to_best_groups(ch, val + top, experts, groups, keep, lane);
  for (int k = 0; k < top; ++k) {
    Best b{-INFINITY, 1 << 30};
    for (int e = lane; e < experts; e += 64) b = better(b, Best{ch[e], e});
    b = wave_best(b);
    const int e = b.i < experts ? b.i : 0;
    if (lane == 0) {
      idx[row * top + k] = e;
      val[k] = b.v;
      ch[e] = -INFINITY;
    }
    __syncthreads();
  }
  chosen_weights(wts + row * top, val, top, lane, sigmoid, scale);
}

// One wave: ch [experts] holds a row's logits; its choice by any of the routers, one expert after the other.  val
// [top, or experts for softmax over all, + groups] is scratch.  Lane 0's LDS writes are made visible to the wave's other lanes
// by a wave-level fence.
__device__ __forceinline__ void choose_in_turn(int* idx, float* wts, float* ch, float* val, const float* bias, int experts,
                                               int top, int mode, float scale, int groups, int keep, int lane) {
  if (mode == kRouteSoftmaxAll) {
    choose_softmax_all(idx, wts, ch, val, val + experts, bias, experts, top, groups, keep, lane);
    return;
  }
  if (keep < groups) limit_to_best_groups(ch, val + top, experts, groups, keep, lane);
  for (int k = 0; k < top; ++k) {
    Best b{-INFINITY, 1 << 30};
    for (int e = lane; e < experts; e += 64) b = better(b, Best{ch[e], e});
    b = wave_best(b);
    const int e = b.i < experts ? b.i : 0;
    if (lane == 0) {
      idx[k] = e;
      val[k] = b.v;
      ch[e] = -INFINITY;
    }
    wave_lds_fence();
  }
  chosen_weights(wts, val, top, lane, mode == kRouteSigmoid, scale);
}

// four consecutive activations as fp32
__device__ __forceinline__ void load4(const float* p, float* v) {
  const float4 u = *reinterpret_cast<const float4*>(p);
  v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w;
}
__device__ __forceinline__ void load4(const bf16_t* p, float* v) {
  const uint2 u = *reinterpret_cast<const uint2*>(p);
  v[0] = __uint_as_float(u.x << 16);
  v[1] = __uint_as_float(u.x & 0xffff0000u);
  v[2] = __uint_as_float(u.y << 16);
  v[3] = __uint_as_float(u.y & 0xffff0000u);
}

// The routers with their logits computed here, for few rows (decode steps): z = W h + b
// in fp32 (W, b fp32; h fp32 or bf16), one workgroup of sixteen waves per token, a wave
// per expert in turn with the lanes along the width (four elements per lane and pass when
// the rows allow 16-byte loads, several passes in flight); then wave 0 chooses as above.
constexpr int kRouteWaves = 16;

template <typename T>
__global__ void __launch_bounds__(64 * kRouteWaves)
moe_route_top_logits_kernel(int* __restrict__ idx, float* __restrict__ wts, const T* __restrict__ h, long h_stride,
                            const float* __restrict__ router, const float* __restrict__ bias, int experts,
                            int width, int top, int vec, int mode, float scale, int groups, int keep) {
  extern __shared__ float sm[];
  float* ch = sm;
  float* val = sm + experts;
  const long row = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const T* hr = h + row * h_stride;
  for (int e = wave; e < experts; e += kRouteWaves) {
    const float* wr = router + (long)e * width;
    float acc = 0.f;
    if (vec) {
#pragma unroll 4
      for (int i = lane * 4; i < width; i += 256) {
        float x[4];
        load4(hr + i, x);
        const float4 w4 = *reinterpret_cast<const float4*>(wr + i);
        acc += x[0] * w4.x + x[1] * w4.y + x[2] * w4.z + x[3] * w4.w;
      }
    } else {
      for (int i = lane; i < width; i += 64) acc += ld(hr, i) * wr[i];
    }
    acc = ft::wave_sum(acc);
    if (lane == 0) ch[e] = acc + (bias != nullptr && mode != kRouteSoftmaxAll ? bias[e] : 0.f);
  }
  __syncthreads();
  if (wave != 0) return;
  choose_in_turn(idx + row * top, wts + row * top, ch, val, bias, experts, top, mode, scale, groups, keep, lane);
}

// The same for bf16 rows of whole 256 and up to 64 experts, optionally behind the norm step that makes the rows: one workgroup of
// sixteen waves per row.  A wave's router rows (an expert in turn, the lanes along the width) are on their way while the
// norm's reductions run, and a row passes to the products through LDS.
//   NORM 0: h given;  1: x += rms_norm(y) * wb (y as it is without wb), h = rms_norm(x) * w;  2: x += layer_norm(y) * w + b, h = x
// Bound by what one CU draws of the router (256 KB for 32 experts of 2048) behind that chain, then by the choice.  Width 2048, 32
// experts, in a decode step: layer norm and router of 32 rows 10.4 us (4.7 + 10.4 in two launches), RMS norms and router of 8
// rows with groups 12.9 (3.9 + 12.7); with the router asked for before the row 1.2 more.
constexpr int kRoutePieces = 8;              // 16-byte pieces of the router a lane asks for at a time; two such in flight

struct RouteRows {
  int* idx;
  float* wts;
  bf16_t* h;                                 // read (NORM 0), else written, dense
  long h_stride;
  float* x;
  const void* y;                             // TY; PARTS of them a row: dense, and their sum is the row
  long y_stride;
  const float *wb, *w, *b;
  const float *router, *bias;
  int experts, width, top, mode, groups, keep;
  float eps, scale;
  int in_turn;                               // rows with logits that are no finite numbers: experts by choose_in_turn
};
// Which experts such a row names does not hang on the kernel that its step takes: up to 64 rows those of the routers above, beyond
// those of the router for sixteen rows a workgroup where that serves (widths of whole 2048)
static bool route_in_turn(long rows, int width) { return rows <= 64 || width % 2048 != 0; }

template <int NORM, int C, typename TY, int PARTS = 1>
__global__ void __launch_bounds__(64 * kRouteWaves)
route_rows_kernel(RouteRows R) {
  constexpr int NT = 64 * kRouteWaves;
  extern __shared__ __attribute__((aligned(16))) float row_s[];
  __shared__ float red[kRouteWaves], z_s[64];
  const long row = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), width = R.width;
  const int passes = width / 256;
  using Raw = typename std::conditional<sizeof(TY) == 2, uint2, float4>::type;
  // (loads come back in the order they were asked for: the row's before the router's)
  float v[C][4], t[C][4], w[C][4], u[C][4];
  Raw yr[C][PARTS];
  uint2 hr[C];
  const float* wb = NORM == 2 ? R.w : R.wb;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int i = min((c * NT + tid) * 4, width - 4);
    if constexpr (NORM == 0) {
      hr[c] = *reinterpret_cast<const uint2*>(R.h + row * R.h_stride + i);
    } else {
#pragma unroll
      for (int p = 0; p < PARTS; ++p)
        yr[c][p] = *reinterpret_cast<const Raw*>((const TY*)R.y + (PARTS > 1 ? (row * PARTS + p) * width : row * R.y_stride) + i);
      load4(R.x + row * width + i, v[c]);
      load4((wb != nullptr ? wb : R.w) + i, w[c]);
      load4((NORM == 2 ? R.b : R.w) + i, u[c]);
    }
  }
  const bool biased = R.bias != nullptr && R.mode != kRouteSoftmaxAll;
  const float bias = (biased ? R.bias : R.router)[min(lane, R.experts - 1)];
  float4 ahead[2][kRoutePieces];
  int fe = wave, fp = 0;                     // the expert and piece to ask for next
  // (no branch around a load: behind one the wait for the row would be a wait for all; pieces past an end are read twice)
  auto fetch = [&](float4 (&a)[kRoutePieces]) {
    const float* p = R.router + (long)min(fe, R.experts - 1) * width + lane * 4;
#pragma unroll
    for (int i = 0; i < kRoutePieces; ++i) a[i] = *reinterpret_cast<const float4*>(p + min(fp + i, passes - 1) * 256);
    fp += kRoutePieces;
    if (fp >= passes) fp = 0, fe += kRouteWaves;
  };
  fetch(ahead[0]);
  fetch(ahead[1]);
  __builtin_amdgcn_sched_barrier(0);
  auto keep_row = [&](int i, const float (&v)[4]) {
    *reinterpret_cast<float4*>(row_s + i) = make_float4(v[0], v[1], v[2], v[3]);
  };
  if constexpr (NORM == 0) {
#pragma unroll
    for (int c = 0; c < C; ++c)
      if ((c * NT + tid) * 4 < width) {
        ft::unpack2(hr[c].x, v[c][0], v[c][1]);
        ft::unpack2(hr[c].y, v[c][2], v[c][3]);
        keep_row((c * NT + tid) * 4, v[c]);
      }
  } else {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if constexpr (sizeof(TY) == 2) {
        ft::unpack2(yr[c][0].x, t[c][0], t[c][1]);
        ft::unpack2(yr[c][0].y, t[c][2], t[c][3]);
      } else {
        t[c][0] = yr[c][0].x, t[c][1] = yr[c][0].y, t[c][2] = yr[c][0].z, t[c][3] = yr[c][0].w;
#pragma unroll
        for (int p = 1; p < PARTS; ++p) t[c][0] += yr[c][p].x, t[c][1] += yr[c][p].y, t[c][2] += yr[c][p].z, t[c][3] += yr[c][p].w;
      }
      if ((c * NT + tid) * 4 >= width)
#pragma unroll
        for (int k = 0; k < 4; ++k) v[c][k] = t[c][k] = w[c][k] = u[c][k] = 0.f;
    }
    float sum = 0.f;
    if constexpr (NORM == 2) {
#pragma unroll
      for (int c = 0; c < C; ++c) sum += (t[c][0] + t[c][1]) + (t[c][2] + t[c][3]);
      const float mean = block_sum<NT>(sum, red) / (float)width;
      sum = 0.f;
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          t[c][k] = (c * NT + tid) * 4 < width ? t[c][k] - mean : 0.f;
          sum += t[c][k] * t[c][k];
        }
    } else if (wb != nullptr) {
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int k = 0; k < 4; ++k) sum += t[c][k] * t[c][k];
    }
    if (wb != nullptr) {
      const float r = 1.0f / sqrtf(block_sum<NT>(sum, red) / (float)width + R.eps);
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int k = 0; k < 4; ++k) t[c][k] = NORM == 2 ? t[c][k] * r * w[c][k] + u[c][k] : t[c][k] * (r * w[c][k]);
    }
    sum = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        v[c][k] += t[c][k];
        sum += v[c][k] * v[c][k];
      }
    const float r = NORM == 2 ? 1.f : 1.0f / sqrtf(block_sum<NT>(sum, red) / (float)width + R.eps);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int i = (c * NT + tid) * 4;
      if (i >= width) continue;
      *reinterpret_cast<float4*>(R.x + row * width + i) = make_float4(v[c][0], v[c][1], v[c][2], v[c][3]);
      uint2 o;
      if constexpr (NORM == 2) {
        o = make_uint2(ft::pack2(v[c][0], v[c][1]), ft::pack2(v[c][2], v[c][3]));
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) v[c][k] *= r * u[c][k];
        o = make_uint2(ft::pack2(v[c][0], v[c][1]), ft::pack2(v[c][2], v[c][3]));
      }
      *reinterpret_cast<uint2*>(R.h + row * width + i) = o;
      float q[4];                            // (the router reads the rounded row)
      ft::unpack2(o.x, q[0], q[1]);
      ft::unpack2(o.y, q[2], q[3]);
      keep_row(i, q);
    }
  }
  __syncthreads();
  int e = wave, pass = 0;
  float acc = 0.f;
  auto products = [&](const float4 (&a)[kRoutePieces]) {
#pragma unroll
    for (int i = 0; i < kRoutePieces; ++i) {
      if (pass + i >= passes) break;
      const float4 x = *reinterpret_cast<const float4*>(row_s + (pass + i) * 256 + lane * 4);
      acc += x.x * a[i].x + x.y * a[i].y + x.z * a[i].z + x.w * a[i].w;
    }
    pass += kRoutePieces;
    if (pass < passes) return;
    acc = ft::wave_sum(acc);
    if (lane == 0) z_s[e] = acc;
    acc = 0.f;
    pass = 0;
    e += kRouteWaves;
  };
  while (e < R.experts) {
    products(ahead[0]);
    if (e >= R.experts) break;
    if (fe < R.experts) fetch(ahead[0]);
    products(ahead[1]);
    if (fe < R.experts) fetch(ahead[1]);
  }
  __syncthreads();
  if (wave != 0) return;
  const float z = lane < R.experts ? z_s[lane] + (biased ? bias : 0.f) : 0.f;
  if (lane < R.experts) z_s[lane] = z;       // (for the choice in turn)
  wave_lds_fence();
  // (ties and NaN have another order there)
  const bool odd = !(fabsf(z) < INFINITY) || (R.mode == kRouteSoftmaxAll && !(fabsf(R.bias[min(lane, R.experts - 1)]) < INFINITY));
  if (R.in_turn && __any(odd))
    choose_in_turn(R.idx + row * R.top, R.wts + row * R.top, z_s, row_s, R.bias, R.experts, R.top, R.mode, R.scale, R.groups,
                   R.keep, lane);
  else
    choose_in_lanes(R.idx + row * R.top, R.wts + row * R.top, z, R.bias, R.experts, R.top, R.mode, R.scale, R.groups, R.keep,
                    lane);
}

// All routers with their logits computed here, for any number of bf16 rows: one workgroup of sixteen waves per 16
// rows.  Logits z = W h (+ bias) with the fp32 router given as three bf16 parts (hi + mid + lo: exactly it), three
// v_mfma_f32_16x16x32_bf16 per operand pair (the fp32 ones take five times as long), a wave a sixteenth of the
// width, partial sums through LDS; then a wave a row, a lane an expert, every lane its expert's place in the order
// (ties to the lower index) by comparing with all others, so no choice waits for the one before.
// The parts lie in operand order, [width / 32][tile of 16 experts][part][lane][8], and the rows pass through LDS,
// so that neighbouring lanes load neighbouring bytes: with a row or expert per lane the load unit took a line per
// lane and 8 rows 17 us.
// Bound by a CU's read of the router (12 KB an expert) behind a chain of load, product and choice: 2000 rows of
// 2048, 32 experts 13 us; 4096 16 (rows widened, a library product and a choice kernel: 25 and 34 us in three
// launches).  Up to 512 rows the kernel above, a workgroup per row, is faster: 9 us for 8 to 256 rows, 13 for 512.
constexpr int kTileRows = 16, kRouteStep = 128;      // width of a wave's turn

template <int NE>
__global__ void __launch_bounds__(64 * kRouteWaves)
moe_route_tile_kernel(int* __restrict__ idx, float* __restrict__ wts, const bf16_t* __restrict__ h, long h_stride,
                      const bf16_t* __restrict__ router, const float* __restrict__ bias, long rows, int experts, int width,
                      int top, int mode, float scale, int groups, int keep) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
  __shared__ __attribute__((aligned(16))) uint4 strip[kRouteWaves][kTileRows][kRouteStep / 8];
  __shared__ float part[kRouteWaves][kTileRows][16 * NE + 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 15, g4 = lane >> 4;
  const long row0 = (long)blockIdx.x * kTileRows;
  {
    f32x4 acc[NE][3];
#pragma unroll
    for (int t = 0; t < NE; ++t)
#pragma unroll
      for (int p = 0; p < 3; ++p) acc[t][p] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k0 = wave * kRouteStep; k0 < width; k0 += kRouteWaves * kRouteStep) {
      uint4 x[4];
      constexpr int kAhead = NE <= 2 ? 2 : 1;         // steps of 32 whose experts are loaded ahead (registers)
      bf16x8 w[kAhead][NE][3];
      auto fetch = [&](int j) {
#pragma unroll
        for (int t = 0; t < NE; ++t)
#pragma unroll
          for (int p = 0; p < 3; ++p)
            w[j % kAhead][t][p] = *reinterpret_cast<const bf16x8*>(router + (((long)(k0 / 32 + j) * NE + t) * 3 + p) * 512 + lane * 8);
      };
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const long r = row0 + 4 * i + g4;
        x[i] = *reinterpret_cast<const uint4*>(h + (r < rows ? r : rows - 1) * h_stride + k0 + 8 * n);
      }
#pragma unroll
      for (int j = 0; j < kAhead; ++j) fetch(j);
      wave_lds_fence();
#pragma unroll
      for (int i = 0; i < 4; ++i) strip[wave][4 * i + g4][n ^ (4 * i + g4)] = x[i];
      wave_lds_fence();
#pragma unroll
      for (int j = 0; j < kRouteStep / 32; ++j) {
        const bf16x8 a = __builtin_bit_cast(bf16x8, strip[wave][n][(4 * j + g4) ^ n]);
#pragma unroll
        for (int t = 0; t < NE; ++t)
#pragma unroll
          for (int p = 0; p < 3; ++p) acc[t][p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w[j % kAhead][t][p], acc[t][p], 0, 0, 0);
        if (j + kAhead < kRouteStep / 32) fetch(j + kAhead);
      }
    }
#pragma unroll
    for (int t = 0; t < NE; ++t) {
      const f32x4 z = acc[t][2] + acc[t][1] + acc[t][0];
#pragma unroll
      for (int v = 0; v < 4; ++v) part[wave][4 * g4 + v][16 * t + n] = z[v];
    }
  }
  __syncthreads();
  const long row = row0 + wave;
  if (row >= rows) return;
  float z = 0.f;
#pragma unroll
  for (int w = 0; w < kRouteWaves; ++w) z += part[w][wave][min(lane, 16 * NE - 1)];
  if (mode != kRouteSoftmaxAll && bias != nullptr && lane < experts) z += bias[lane];
  choose_in_lanes(idx + row * top, wts + row * top, z, bias, experts, top, mode, scale, groups, keep, lane);
}

// (rows of 32 KB in LDS at most)
static bool route_rows_fit(int width, int experts) {
  return width >= 256 && width <= 8192 && width % 256 == 0 && experts >= 1 && experts <= 64;
}

}  // namespace mx

extern "C" int mx_norm_route_fits(int width, int experts) { return mx::route_rows_fit(width, experts); }

// The norm step in front of a router and the router, bf16 rows out: layer 0: x += rms_norm(y) * wb (wb null: y), h = rms_norm(x) * w;
// 1: x += layer_norm(y) * w + b, h = x.  parts 2 or 4: y [rows][parts][width] fp32, rows the sums of their parts.  Modes as below.
extern "C" int mx_norm_route(int* idx, float* wts, void* h, float* x, const void* y, int y_bf16, long y_stride, int parts,
                             int layer, const float* wb, const float* w, const float* b, float eps, const float* router, const float* bias, long rows,
                             int experts, int width, int top, int mode, float scale, int groups, int keep, hipStream_t s) {
  if (rows <= 0) return 0;
  if (!mx::route_rows_fit(width, experts) || top < 1 || top > experts || mode < 0 || mode > 2 || (mode == 2 && bias == nullptr) ||
      rows > 0x7fffffffL || y_stride % 4 || !(parts == 1 || ((parts == 2 || parts == 4) && !y_bf16))) return -1;
  if (groups < 1 || experts % groups || keep < 1 || keep > groups || top > experts / groups * keep) return -1;
  if (((uintptr_t)h | (uintptr_t)x | (uintptr_t)wb | (uintptr_t)w | (uintptr_t)b | (uintptr_t)router) % 16 || ((uintptr_t)y) % (y_bf16 ? 8 : 16))
    return -2;
  const mx::RouteRows R{idx, wts, (mx::bf16_t*)h, width, x, y, y_stride, wb, w, b, router, bias, experts, width,
                        top, mode, groups, keep, eps, scale, mx::route_in_turn(rows, width)};
#define MX_NR(NORM, C)                                                                                                     \
  MX_DISPATCH_T(y_bf16, hipLaunchKernelGGL((mx::route_rows_kernel<NORM, C, T>), dim3((unsigned)rows), dim3(64 * mx::kRouteWaves), \
                                           width * 4, s, R))
#define MX_NR_PARTS(NORM, C, PARTS)                                                                                  \
  hipLaunchKernelGGL((mx::route_rows_kernel<NORM, C, float, PARTS>), dim3((unsigned)rows), dim3(64 * mx::kRouteWaves), \
                     width * 4, s, R)
#define MX_NR_P(NORM, C)                            \
  do {                                              \
    if (parts == 4) MX_NR_PARTS(NORM, C, 4);        \
    else if (parts == 2) MX_NR_PARTS(NORM, C, 2);   \
    else MX_NR(NORM, C);                            \
  } while (0)
#define MX_NR_C(NORM)                    \
  do {                                   \
    if (width <= 4096) MX_NR_P(NORM, 1); \
    else MX_NR_P(NORM, 2);               \
  } while (0)
  if (layer) MX_NR_C(2);
  else MX_NR_C(1);
#undef MX_NR_C
#undef MX_NR_P
#undef MX_NR_PARTS
#undef MX_NR
  return (int)hipGetLastError();
}

// mode 0: moe_top_logits by softmax, 1: by sigmoids, 2: moe_topk (bias: the selection bias)
extern "C" int mx_moe_route_few(int* idx, float* wts, const void* h, int bf16, long h_stride,
                                const float* router, const float* bias, long rows, int experts, int width,
                                int top, int mode, float scale, int groups, int keep, hipStream_t s) {
  if (rows <= 0) return 0;
  if (experts < 1 || top < 1 || top > experts || width < 1 || mode < 0 || mode > 2 || (mode == 2 && bias == nullptr)) return -1;
  if (groups < 1 || experts % groups || keep < 1 || keep > groups || top > experts / groups * keep) return -1;
  const size_t lds = (size_t)(experts + (mode == 2 ? experts : top) + groups) * sizeof(float);
  if (lds > 60 * 1024) return -2;
  const long es = bf16 ? 2 : 4;
  const int vec = width % 4 == 0 && h_stride % 4 == 0 && ((uintptr_t)h) % (4 * es) == 0 &&
                  ((uintptr_t)router) % 16 == 0;
  if (bf16 && vec && mx::route_rows_fit(width, experts)) {
    const mx::RouteRows R{idx, wts, (mx::bf16_t*)const_cast<void*>(h), h_stride, nullptr, nullptr, 0, nullptr, nullptr, nullptr,
                          router, bias, experts, width, top, mode, groups, keep, 0.f, scale,
                          mx::route_in_turn(rows, width)};
    if (width <= 4096)
      hipLaunchKernelGGL((mx::route_rows_kernel<0, 1, mx::bf16_t>), dim3((unsigned)rows), dim3(64 * mx::kRouteWaves), width * 4, s, R);
    else
      hipLaunchKernelGGL((mx::route_rows_kernel<0, 2, mx::bf16_t>), dim3((unsigned)rows), dim3(64 * mx::kRouteWaves), width * 4, s, R);
    return (int)hipGetLastError();
  }
  MX_DISPATCH_T(bf16, hipLaunchKernelGGL((mx::moe_route_top_logits_kernel<T>), dim3((unsigned)rows),
                                         dim3(64 * mx::kRouteWaves), lds, s, idx, wts, (const T*)h, h_stride, router,
                                         bias, experts, width, top, vec, mode, scale, groups, keep));
  return (int)hipGetLastError();
}

extern "C" int mx_moe_route_fits(const void* h, long h_stride, const void* parts, int experts, int width) {
  return experts >= 1 && experts <= 64 && width >= 1 && width % (mx::kRouteStep * mx::kRouteWaves) == 0 && h_stride % 8 == 0 &&
         (((uintptr_t)h) | ((uintptr_t)parts)) % 16 == 0;
}

// parts: the router's three bf16 parts in operand order, whole tiles of experts; modes as mx_moe_route_few
extern "C" int mx_moe_route(int* idx, float* wts, const void* h, long h_stride, const void* parts, const float* bias,
                            long rows, int experts, int width, int top, int mode, float scale, int groups, int keep,
                            hipStream_t s) {
  if (rows <= 0) return 0;
  if (!mx_moe_route_fits(h, h_stride, parts, experts, width) || top < 1 || mode < 0 || mode > 2 ||
      (mode == 2 && bias == nullptr)) return -1;
  if (groups < 1 || experts % groups || keep < 1 || keep > groups || top > experts / groups * keep) return -1;
  const long tiles = (rows + mx::kTileRows - 1) / mx::kTileRows;
  if (tiles > 0x7fffffffL) return -2;
#define MX_ROUTE(NE)                                                                                         \
  hipLaunchKernelGGL((mx::moe_route_tile_kernel<NE>), dim3((unsigned)tiles), dim3(64 * mx::kRouteWaves), 0, s, \
                     idx, wts, (const mx::bf16_t*)h, h_stride, (const mx::bf16_t*)parts, bias, rows, experts, width, top, \
                     mode, scale, groups, keep)
  if (experts <= 16) MX_ROUTE(1);
  else if (experts <= 32) MX_ROUTE(2);
  else if (experts <= 48) MX_ROUTE(3);
  else MX_ROUTE(4);
#undef MX_ROUTE
  return (int)hipGetLastError();
}

extern "C" int mx_moe_top_logits(int* idx, float* wts, const float* z, long rows, int experts, int top,
                                 int sigmoid, float scale, int groups, int keep, hipStream_t s) {
  if (rows <= 0) return 0;
  if (experts < 1 || top < 1 || top > experts) return -1;
  if (groups < 1 || experts % groups || keep < 1 || keep > groups || top > experts / groups * keep) return -1;
  const size_t lds = (size_t)(experts + top + groups) * sizeof(float);
  if (lds > 60 * 1024) return -2;
  hipLaunchKernelGGL(mx::moe_top_logits_kernel, dim3((unsigned)rows), dim3(64), lds, s, idx, wts, z, experts, top,
                     sigmoid, scale, groups, keep);
  return (int)hipGetLastError();
}

extern "C" int mx_moe_topk(int* idx, float* wts, const float* z, const float* corr, long rows, int experts,
                           int top, int groups, int keep, hipStream_t s) {
  if (rows <= 0) return 0;
  if (experts < 1 || top < 1 || top > experts || groups < 1 || experts % groups || keep < 1 || keep > groups)
    return -1;
  const size_t lds = (size_t)(2 * experts + groups) * sizeof(float);
  if (lds > 60 * 1024) return -2;
  hipLaunchKernelGGL(mx::moe_topk_kernel, dim3((unsigned)rows), dim3(64), lds, s, idx, wts, z, corr, experts,
                     top, groups, keep);
  return (int)hipGetLastError();
}

// Shared helpers of the sequence-mixer / MoE kernels (extension `_C_mixers`).
//
// Every kernel is instantiated for fp32 and bf16 activations (`T` = float or
// ft::bf16_raw); statistics, scores, recurrent state and gates are fp32 in both.
// Launchers take `int bf16` flags and void pointers, and the caller's stream.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "ft_common.h"
#include <type_traits>

namespace mx {

using bf16_t = ft::bf16_raw;

__device__ __forceinline__ float ld(const float* p, long i) { return p[i]; }
__device__ __forceinline__ float ld(const bf16_t* p, long i) { return ft::bf16_to_f32(p[i]); }
__device__ __forceinline__ void st(float* p, long i, float v) { p[i] = v; }
__device__ __forceinline__ void st(bf16_t* p, long i, float v) { p[i] = ft::f32_to_bf16(v); }

// 1 / (1 + e^-x), as exact as the library's exponential and division (2.7 units in the last place at most, 0.45 on average in
// -8 .. 8, the same in both) in half their instructions.  The denominator is formed 2^-24 times as large: e^104 has a
// reciprocal, so results are right down to the smallest numbers, and 0 below.
__device__ __forceinline__ float sigmoidf_(float x) {
  const float c = fminf(fmaxf(x, -104.f), 88.f);                 // (NaN: below)
  float t, f;                                                    // e^-x = 2^(t + r), r what t's rounding lost
  {
#pragma clang fp contract(off)
    t = c * -1.44269502f;
  }
  const float r = fmaf(c, -1.44269502f, -t) - c * 1.92596303e-8f, n = rintf(t);
  {
#pragma clang fp contract(off)
    f = t - n;
  }
  const float d = 0x1p-24f + __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(f + r), (int)n - 24);
  const float q = __builtin_amdgcn_rcpf(d);
  return x == x ? 0x1p-24f * fmaf(fmaf(-d, q, 1.f), q, q) : x;
}

__device__ __forceinline__ float gelu_tanh_(float z) {
  return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

// softplus with the usual linear branch for large arguments
__device__ __forceinline__ float softplusf_(float x) { return x > 20.0f ? x : log1pf(expf(x)); }

// entry d < dims of a head x after rotary positions, cs = [cos | sin] of the position: pairs
// (i, i + dims/2), or (2i, 2i + 1) if interleaved
template <typename T>
__device__ __forceinline__ float rope_at(const T* x, int d, int dims, const float* cs, int interleaved) {
  const int half = dims / 2;
  const int i = interleaved ? d >> 1 : (d < half ? d : d - half);
  const bool second = interleaved ? (d & 1) : d >= half;
  const int other = interleaved ? d ^ 1 : (second ? d - half : d + half);
  const float v = ld(x, d), w = ld(x, other), c = cs[i], s = cs[half + i];
  return second ? v * c + w * s : v * c - w * s;
}

// sum / maximum over the 16 lanes of a row (quad swaps, mirrored half row, mirrored row): every
// lane gets it
__device__ __forceinline__ float sum16(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xF, 0xF, true));
  return v;
}
__device__ __forceinline__ float max16(float v) {
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, true)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xF, 0xF, true)));
  return v;
}

// v plus the v of the lane 16 / 32 away (row swaps instead of the LDS permute path)
__device__ __forceinline__ float add_row_pair(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float add_halves(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// sigmoid(z)^(1/tau) = exp(-softplus(-z) / tau) in fp32 on the hardware's exp2 / log2:
// softplus(-z) = log(1 + e) with e = exp(-z); for small e the series e - e^2/2 keeps the
// digits that 1 + e would drop.  The absolute error of the decay's logarithm stays near
// 1e-7, the spacing of fp32 numbers below 1.
__device__ __forceinline__ float gla_decay(float z, float inv_tau) {
  const float e = __expf(-z);
  const float sp = e < 1e-3f ? e * (1.0f - 0.5f * e) : __logf(1.0f + e);
  return __expf(-sp * inv_tau);
}

// exp(-rate softplus(z)) on the hardware's exp2 and log2, a third of the instructions of the library's expf and log1pf and nearer:
// softplus(z) = max(z, 0) + log(1 + e), e = exp(-|z|), with what 1 + e drops of e added back; what the roundings of that sum and of
// the products with rate and log2 e drop goes into the result at the end.  Largest and mean error in units in the last place, z in
// -12 .. 12, rate in e^-3 .. e^3: 46 and 0.6 (library: 138 and 2.4).  channel_prep, 4096 rows of 16 heads of 128: 134 us and now 109.
__device__ __forceinline__ float delta_decay(float z, float rate) {
  constexpr float kL = 1.4426950408889634f, kLo = 1.925963033500e-8f, kLn2 = 0.6931471805599453f;
  const float e = __builtin_amdgcn_exp2f(-kL * fabsf(z)), u = 1.0f + e, m = fmaxf(z, 0.0f);
  const float l = fmaf(__builtin_amdgcn_logf(u), kLn2, (e - (u - 1.0f)) * __builtin_amdgcn_rcpf(u));
  const float sp = m + l;
  float y = rate * sp, low = fmaf(rate, sp, -y) + rate * (l - (sp - m));
  if (!(y <= 200.0f)) y = y > 200.0f ? 200.0f : y, low = 0.f;          // (a NaN stays one)
  const float t = y * -kL;
  low = fmaf(y, -kLo, fmaf(y, -kL, -t)) - kL * low;
  const int down = t < -100.0f ? 64 : 0;            // (exp2 has no denormal results)
  const float r = __builtin_amdgcn_exp2f(t + (float)down);
  return ldexpf(fmaf(r * kLn2, low, r), -down);
}

// tanh without branches: the Taylor polynomial up to |x| = 1/4, (1 - e^-2|x|) / (1 + e^-2|x|) beyond
__device__ __forceinline__ float tanh_(float x) {
  const float a = fabsf(x), q = a * a;
  const float p = a + a * q * (-1.f / 3 + q * (2.f / 15 + q * (-17.f / 315 + q * (62.f / 2835 - q * (1382.f / 155925)))));
  const float t = __builtin_amdgcn_exp2f(-2.8853900817779268f * a);
  const float r = (1.f - t) / (1.f + t);
  return copysignf(a < 0.25f ? p : r, x);
}

// two fp32 values -> their hi, mid and lo bf16 parts (24 bits: the sum is the value)
__device__ __forceinline__ void split_bf16x3(float a, float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  hi = ft::pack2(a, b);
  const float a1 = a - __uint_as_float(hi << 16), b1 = b - __uint_as_float(hi & 0xffff0000u);
  mid = ft::pack2(a1, b1);
  lo = ft::pack2(a1 - __uint_as_float(mid << 16), b1 - __uint_as_float(mid & 0xffff0000u));
}

// the same for any two values: of one that is infinite, or that bf16 would round to infinity, the largest finite hi part, and
// what is left is mid (infinite itself, with nothing in lo, or exact)
__device__ __forceinline__ void split_any_bf16x3(float a, float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  constexpr float kMax = 3.38953139e38f;
  const auto cut = [](float x) { return fminf(fmaxf(x, -kMax), kMax); };
  hi = ft::pack2(cut(a), cut(b));
  const float a1 = a - __uint_as_float(hi << 16), b1 = b - __uint_as_float(hi & 0xffff0000u);
  mid = ft::pack2(a1, b1);
  const float a2 = cut(a1), b2 = cut(b1);
  const uint32_t m = ft::pack2(a2, b2);
  lo = ft::pack2(a2 - __uint_as_float(m << 16), b2 - __uint_as_float(m & 0xffff0000u));
}

// the parts of this lane's 8 entries of each of KS pieces of 32 (src: the lane's first), as matrix operands.  (Any value, with no
// question asked: a branch between this and the short form has the entries waited for behind the keys' loads, a decode
// row of 540 keys 19 to 20 us, 18.3 so and with the short form alone.)
template <int KS>
__device__ __forceinline__ void split_queries(const float4 (&src)[KS][2], uint4 (&part)[3][KS]) {
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const float4 u = src[s][0], v = src[s][1];
    split_any_bf16x3(u.x, u.y, part[0][s].x, part[1][s].x, part[2][s].x);
    split_any_bf16x3(u.z, u.w, part[0][s].y, part[1][s].y, part[2][s].y);
    split_any_bf16x3(v.x, v.y, part[0][s].z, part[1][s].z, part[2][s].z);
    split_any_bf16x3(v.z, v.w, part[0][s].w, part[1][s].w, part[2][s].w);
  }
}

template <int KS>
__device__ __forceinline__ void split_queries(const float* src, uint4 (&part)[3][KS]) {
  float4 raw[KS][2];
#pragma unroll
  for (int s = 0; s < KS; ++s)
#pragma unroll
    for (int y = 0; y < 2; ++y) raw[s][y] = *reinterpret_cast<const float4*>(src + 32 * s + 4 * y);
  split_queries<KS>(raw, part);
}

// a wave's own LDS writes, to be read by its other lanes
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// the segment that owns a row: the last s with start[s] <= row.  Decode rows come first in a
// step, one row each: for them one look at two neighbouring entries is enough.
__device__ __forceinline__ int segment_of(const int* __restrict__ start, int num_segs, int row) {
  if (row < num_segs && start[row] == row && start[row + 1] == row + 1) return row;
  int lo = 0, hi = num_segs;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (start[mid] <= row) lo = mid; else hi = mid;
  }
  return lo;
}

// A short causal convolution over time of one wave's channels c0 + lane + 64 u (u < NU, below
// c0 + len), walked row by row: taps (<= TAPS) weights and the last taps - 1 inputs in
// registers, fp32.  Missing taps in front count as zeros.
template <int TAPS, int NU>
struct ConvWalk {
  float w[NU][TAPS], win[NU][TAPS];            // win[u][TAPS - 1] is the current row's input

  __device__ __forceinline__ void weights(const float* __restrict__ conv_w, int taps, int c0, int len, int lane) {
    const int pad = TAPS - taps;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int i = lane + 64 * u;
      const float* p = conv_w + (long)(c0 + (i < len ? i : 0)) * taps;
      if (TAPS == 4 && pad == 0 && ((uintptr_t)conv_w) % 16 == 0) {
        const float4 v = *reinterpret_cast<const float4*>(p);
        w[u][0] = v.x; w[u][1] = v.y; w[u][TAPS == 4 ? 2 : 0] = v.z; w[u][TAPS == 4 ? 3 : 0] = v.w;
      } else {
#pragma unroll
        for (int j = 0; j < TAPS; ++j) w[u][j] = j >= pad ? p[j - pad] : 0.f;
      }
    }
  }
  // the inputs before row rel of the segment that starts at row r0: rows of x, further back the
  // history h [taps - 1][channels] (null: zeros)
  template <typename T>
  __device__ __forceinline__ void begin(const T* __restrict__ x, long stride, long r0, int rel, const float* h,
                                        int channels, int taps, int c0, int len, int lane) {
    const int pad = TAPS - taps;
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j) {
      const int src = rel - (TAPS - 1) + j;
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const int i = lane + 64 * u, c = c0 + (i < len ? i : 0);
        float v = 0.f;
        if (j >= pad) {
          if (src >= 0) v = ld(x, (r0 + src) * stride + c);
          else if (h != nullptr) v = h[(long)(taps - 1 + src) * channels + c];
        }
        win[u][j] = v;
      }
    }
  }
  __device__ __forceinline__ float step(int u, float v) {
    win[u][TAPS - 1] = v;
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < TAPS; ++j) acc += win[u][j] * w[u][j];
    return acc;
  }
  // to the next row
  __device__ __forceinline__ void shift(int u) {
#pragma unroll
    for (int j = 0; j + 1 < TAPS; ++j) win[u][j] = win[u][j + 1];
  }
  // after shift(): the last taps - 1 inputs, as a history
  __device__ __forceinline__ void store(float* h, int channels, int taps, int c0, int len, int lane) const {
    const int pad = TAPS - taps;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int i = lane + 64 * u;
#pragma unroll
      for (int j = 0; j + 1 < TAPS; ++j)
        if (j >= pad && i < len) h[(long)(j - pad) * channels + c0 + i] = win[u][j];
    }
  }
};

// sum_sp w[sp] acc[sp * stride + c] for a wave that owns columns [c0, c0 + 256) of n: w, from weight(c), is lane
// sp's value (slices <= 64, 0 beyond them; a slice of weight 0 adds nothing).  VEC (n and stride multiples of 4,
// 16-byte aligned): several slices per pass, 16-byte loads, the first ones asked for before the weights, which wait for
// loads of their own; c is the first column that the lane may leave.  out(c, values, count) is called once per
// column by one lane, four columns at a time (VEC) or one.
template <bool VEC, typename W, typename F>
__device__ __forceinline__ void merge_slices(const float* __restrict__ acc, long stride, W weight, int slices, int c0,
                                             int n, int lane, F out) {
  const int cols = min(256, n - c0);
  if constexpr (VEC) {
    const int pieces = cols / 4;
    int lpp = 1;
    while (lpp < pieces) lpp <<= 1;              // lanes per slice
    const int per = 64 / lpp, sub = lane / lpp, pc = lane & (lpp - 1);
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    float4 a[8];
    auto load = [&](int s0) {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        a[u] = *reinterpret_cast<const float4*>(acc + min(s0 + u * per + sub, slices - 1) * stride + c0 + 4 * min(pc, pieces - 1));
    };
    load(0);
    const float w = weight(c0 + 4 * min(pc, pieces - 1));
    // eight passes' loads at a time without a branch among them (with one per slice 32 slices of 512 columns took 14 us,
    // so 6); a slice of weight 0 may hold anything and adds nothing
    const unsigned long long some = __builtin_amdgcn_ballot_w64(w != 0.f);
    for (int s0 = 0; s0 < slices; s0 += 8 * per) {
      if (((some >> s0) & (8 * per < 64 ? (1ull << (8 * per)) - 1 : ~0ull)) == 0) continue;
      if (s0 > 0) load(s0);
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int sp = s0 + u * per + sub;
        const float ws = __shfl(w, min(sp, 63));
        const bool on = sp < slices && ws != 0.f;
        v[0] = on ? v[0] + ws * a[u].x : v[0];
        v[1] = on ? v[1] + ws * a[u].y : v[1];
        v[2] = on ? v[2] + ws * a[u].z : v[2];
        v[3] = on ? v[3] + ws * a[u].w : v[3];
      }
    }
    for (int off = lpp; off < 64; off <<= 1) {
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] += __shfl_xor(v[k], off);
    }
    if (sub == 0 && pc < pieces) out(c0 + 4 * pc, v, std::integral_constant<int, 4>{});
  } else {
    const float w = weight(c0);
    for (int c = lane; c - lane < cols; c += 64) {
      float v = 0.f;
#pragma unroll 4
      for (int sp = 0; sp < slices; ++sp) {
        const float ws = __shfl(w, sp);
        if (c < cols && ws != 0.f) v += ws * acc[sp * stride + c0 + c];
      }
      if (c < cols) out(c0 + c, &v, std::integral_constant<int, 1>{});
    }
  }
}

// sum over a block of NT threads (NT multiple of 64, <= 1024); every thread gets it
template <int NT>
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = ft::wave_sum(v);
  constexpr int NW = NT / 64;
  if constexpr (NW == 1) return v;
  __syncthreads();   // red may still be read from a previous call
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float s = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) s += red[w];
  return s;
}

// the work item: segment and block of `per` pairs within it, `rep` pairs a row (false: none), of the segments
// of at least min_rows rows.  Later blocks, which see more keys, come first.
__device__ __forceinline__ bool segment_block(const int* start, int num_segs, int min_rows, int rep, int per, int item,
                                              int& seg, int& block) {
  const int lane = threadIdx.x & 63;
  for (int s0 = 0; s0 < num_segs; s0 += 64) {
    const int s = s0 + lane;
    int n = 0;
    if (s < num_segs) n = start[s + 1] - start[s];
    const int cnt = n >= min_rows ? (n * rep + per - 1) / per : 0;
    int sum = cnt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(sum, o);
      if (lane >= o) sum += v;
    }
    const uint64_t m = __ballot(sum > item);
    if (m) {
      const int l = __builtin_ctzll(m);
      seg = s0 + l;
      const int c = __shfl(cnt, l);
      block = c - 1 - (item - (__shfl(sum, l) - c));
      return true;
    }
    item -= __shfl(sum, 63);
  }
  return false;
}

}  // namespace mx

#define MX_DISPATCH_T(bf16, ...)            \
  do {                                      \
    if (bf16) {                             \
      using T = ::mx::bf16_t;               \
      __VA_ARGS__;                          \
    } else {                                \
      using T = float;                      \
      __VA_ARGS__;                          \
    }                                       \
  } while (0)

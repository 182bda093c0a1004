// The matrix-unit core of products with few rows (decode steps): C[r, n] = sum_k X[r, k] W[n, k],
// bf16 in, fp32 accumulate, at most 64 rows of X against many rows of W.
//
// Such a product is bound by the stream of W, and at decode sizes by the latency of getting that
// stream going: W is read once, straight from its rows into operand registers (no packed copy of
// the weights), and every wave has U steps of loads in flight before its first multiply.  A step
// is 64 elements of k: lane (quarter q, row n) takes 32 contiguous bytes at k = 64 s + 16 q of its
// row, so a wave's step covers whole 128-byte lines of 16 weight rows, and the two 16x16x32
// products of a step see k in the order {16 q + 0..7}, {16 q + 8..15} on both operands (a sum
// over k does not mind the order).  The waves of a workgroup own contiguous ranges of k, and their
// partial sums meet in LDS in wave order (fixed, so results do not depend on timing).
//
// X goes through the wave's own corner of LDS: read in operand order straight from memory, 16 rows
// a load, it costs the L1 one line a lane (64 rows of 8192 columns against 2048 weight rows took 38
// us, 12 us of it W); read along its rows it costs a quarter of that.  No workgroup barrier: a wave
// reads back only what it wrote.
#pragma once

#include "mx_common.h"

namespace mx {

typedef __bf16 fr_bf16x8 __attribute__((ext_vector_type(8)));
typedef float fr_f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ fr_f32x4 fr_mfma(const uint4& a, const uint4& b, fr_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(fr_bf16x8, a), __builtin_bit_cast(fr_bf16x8, b), c,
                                                 0, 0, 0);
}

// bytes of a staged X row of U steps (16 more: the 16 rows of an operand read fall on all banks)
template <int U>
constexpr int kFrRow = U * 128 + 16;
// bytes of LDS per wave
template <int NB, int U>
constexpr int kFrStage = NB * 16 * kFrRow<U>;

// acc[t][b] += W rows of tile t times X rows of block b, over this wave's share of k.  wp: the lane's
// row of each tile; xrow(r): row r < rows of X; stage: this wave's kFrStage bytes.  All pieces are 16
// bytes (K a multiple of 8); those past the wave's share count as zeros.
template <int NT, int NB, int WV, int U, typename XR>
__device__ __forceinline__ void few_rows_core(fr_f32x4 (&acc)[NT][NB], const bf16_t* const (&wp)[NT], XR xrow, int rows,
                                              int K, char* stage, int wave, int lane) {
  constexpr int LPR = U * 8, RPI = 64 / LPR, XI = NB * 16 / RPI;   // lanes a row, rows a load, loads a round
  const int n = lane & 15, q = lane >> 4;
  const int per = (((K + 63) >> 6) + WV - 1) / WV * 64;
  const int kend = min((wave + 1) * per, K);
  const int sr = lane / LPR, sk = (lane % LPR) * 8;
  for (int k0 = wave * per; k0 < kend; k0 += 64 * U) {
    uint4 x[XI], w[U][NT][2];
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int r = i * RPI + sr;
      x[i] = uint4{0, 0, 0, 0};
      if (r < rows && k0 + sk < kend) x[i] = *reinterpret_cast<const uint4*>(xrow(r) + k0 + sk);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int k = k0 + 64 * u + 16 * q + 8 * j;
          w[u][t][j] = uint4{0, 0, 0, 0};
          if (k < kend) w[u][t][j] = *reinterpret_cast<const uint4*>(wp[t] + k);
        }
    wave_lds_fence();                            // the last round's operands have been read
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int r = i * RPI + sr;
      if (r < rows) *reinterpret_cast<uint4*>(stage + r * kFrRow<U> + sk * 2) = x[i];
    }
    wave_lds_fence();
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        uint4 xb[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b)
          xb[b] = *reinterpret_cast<const uint4*>(stage + (16 * b + n) * kFrRow<U> + u * 128 + q * 32 + j * 16);
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int b = 0; b < NB; ++b) acc[t][b] = fr_mfma(w[u][t][j], xb[b], acc[t][b]);
      }
  }
}

// The same with a round's loads in flight under the products of the one before, for workgroups that have a CU to themselves.  Written
// out beside the other: one loop with a switch, or parts that both call, are scheduled otherwise and take 5.07 to 5.11 us of 1 to
// 8 rows of 2048 -> 2048 where these take 4.97 to 5.05.
template <int NT, int NB, int WV, int U, typename XR>
__device__ __forceinline__ void few_rows_core_ahead(fr_f32x4 (&acc)[NT][NB], const bf16_t* const (&wp)[NT], XR xrow, int rows,
                                                    int K, char* stage, int wave, int lane) {
  constexpr int LPR = U * 8, RPI = 64 / LPR, XI = NB * 16 / RPI;   // lanes a row, rows a load, loads a round
  const int n = lane & 15, q = lane >> 4;
  const int per = (((K + 63) >> 6) + WV - 1) / WV * 64;
  const int kend = min((wave + 1) * per, K);
  const int sr = lane / LPR, sk = (lane % LPR) * 8;
  uint4 x[XI], w[U][NT][2];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int r = i * RPI + sr;
      x[i] = uint4{0, 0, 0, 0};
      if (r < rows && k0 + sk < kend) x[i] = *reinterpret_cast<const uint4*>(xrow(r) + k0 + sk);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int k = k0 + 64 * u + 16 * q + 8 * j;
          w[u][t][j] = uint4{0, 0, 0, 0};
          if (k < kend) w[u][t][j] = *reinterpret_cast<const uint4*>(wp[t] + k);
        }
  };
  fetch(wave * per);
  for (int k0 = wave * per; k0 < kend; k0 += 64 * U) {
    wave_lds_fence();                            // the last round's operands have been read
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const int r = i * RPI + sr;
      if (r < rows) *reinterpret_cast<uint4*>(stage + r * kFrRow<U> + sk * 2) = x[i];
    }
    uint4 now[U][NT][2];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j) now[u][t][j] = w[u][t][j];
    if (k0 + 64 * U < kend) fetch(k0 + 64 * U);
    wave_lds_fence();
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        uint4 xb[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b)
          xb[b] = *reinterpret_cast<const uint4*>(stage + (16 * b + n) * kFrRow<U> + u * 128 + q * 32 + j * 16);
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int b = 0; b < NB; ++b) acc[t][b] = fr_mfma(now[u][t][j], xb[b], acc[t][b]);
      }
  }
}

// what is done to a column's sum(s)
enum { kFrStore = 0, kFrGelu = 1, kFrRelu = 2, kFrSilu = 3, kFrClamp = 4, kFrReluSq = 5, kFrTanhCap = 6 };

// gated forms take the gate's and the up matrix's sums; relu^2 takes one.  0.5 (1 + tanh z) = sigmoid(2 z).  One sigmoid for
// all: with one in each case of a switch tile_gemm.hip's epilogue is too long for the compiler to unroll, its sums lie in
// memory, and 2048 x 2048 -> 2 x 8192 takes 189 us instead of 113.
__device__ __forceinline__ float fr_act(int act, float limit, float g, float u) {
  if (act == kFrReluSq) {
    const float r = fmaxf(g, 0.f);
    return r * r;
  }
  float a = g, z = g, b = u;
  if (act == kFrGelu) z = 1.5957691216057308f * (g + 0.044715f * g * g * g);
  if (act == kFrClamp) {
    a = fminf(g, limit);
    z = 1.702f * a;
    b = fminf(fmaxf(u, -limit), limit) + 1.0f;
  }
  return (act == kFrRelu ? fmaxf(g, 0.f) : a * sigmoidf_(z)) * b;
}

// four neighbouring columns n0 .. n0 + 3 of one output row
template <typename TO>
__device__ __forceinline__ void fr_store4(TO* row, int n0, int N, bool vec, const float (&v)[4]) {
  if (vec && n0 + 3 < N) {
    if constexpr (sizeof(TO) == 2) {
      *reinterpret_cast<uint2*>(row + n0) = make_uint2(ft::pack2(v[0], v[1]), ft::pack2(v[2], v[3]));
    } else {
      *reinterpret_cast<float4*>(row + n0) = make_float4(v[0], v[1], v[2], v[3]);
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (n0 + i < N) st(row, n0 + i, v[i]);
}

}  // namespace mx

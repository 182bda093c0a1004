// Products with few rows (decode steps) on the matrix units, weights read in place:
//   few_rows_gemm   Y[r, n] = sum_k X[r, k] W[n, k] (+ bias[n]), bf16 or fp32 out; or, gated,
//                   Y[r, c] = act(X W_gate^T, X W_up^T), W = [gate | up]; or relu(X W^T)^2
//   few_rows_parts  the same product with k cut into parts, a workgroup each: fp32 sums of the parts, which the step behind adds
//   experts_first   the chosen experts' first matrices (and the shared expert's) with the
//                   activation, one read of an expert's matrix for all rows that chose it
//   experts_down    their second matrices, one fp32 row per (row, chosen expert)
//   experts_combine out[r] = sum_k w[r, k] d[r, k] + shared part
// The core and its layout: few_rows.h.
#include "few_rows.h"

#include <type_traits>

namespace mx {

constexpr int kFewRows = 64;       // most rows of X

// partial sums of the waves -> one sum per (tile, block, lane), in wave order.  red: [WV][NT * NB][64] float4
template <int NT, int NB, int WV>
__device__ __forceinline__ void few_rows_park(float4* red, const fr_f32x4 (&acc)[NT][NB], int wave, int lane) {
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int b = 0; b < NB; ++b)
      red[(wave * NT * NB + t * NB + b) * 64 + lane] = make_float4(acc[t][b][0], acc[t][b][1], acc[t][b][2], acc[t][b][3]);
}
template <int NT, int NB, int WV>
__device__ __forceinline__ void few_rows_sum(const float4* red, int t, int b, int lane, float (&v)[4]) {
  v[0] = v[1] = v[2] = v[3] = 0.f;
#pragma unroll
  for (int w = 0; w < WV; ++w) {
    const float4 p = red[(w * NT * NB + t * NB + b) * 64 + lane];
    v[0] += p.x;
    v[1] += p.y;
    v[2] += p.z;
    v[3] += p.w;
  }
}

// What rides in a launch of a plain product, which at decode sizes is 4.6 us by itself: a second product of the same sizes and
// strides (workgroups of blockIdx.y = 1), or a token-side gate behind the sums, gelu(v) * table[ids[row], column].
struct FewRowsRider {
  const bf16_t *X2, *W2;
  void* Y2;
  const bf16_t* table;
  const int* ids;
  long table_stride;
  int vocab;
};

// ---------------------------------------------------------------------------------
// one workgroup of WV waves per P tiles of 16 output columns (GLU: P tiles of the gate and the
// same of the up matrix).
// ---------------------------------------------------------------------------------
template <int P, bool GLU, int NB, int WV, int U, typename TO, bool RIDE>
__global__ void __launch_bounds__(64 * WV)
few_rows_gemm_kernel(TO* __restrict__ Y, long y_stride, const bf16_t* __restrict__ X, long x_stride, int rows,
                     const bf16_t* __restrict__ W, const bf16_t* __restrict__ bias, int N, int K, int act, float limit,
                     int vec, FewRowsRider R) {
  if constexpr (RIDE) {
    if (blockIdx.y != 0) X = R.X2, W = R.W2, Y = (TO*)R.Y2;
  }
  constexpr int NT = GLU ? 2 * P : P;
  extern __shared__ float4 red[];                // few_rows_lds bytes: X stages, then partial sums
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.x * 16 * P;
  const bf16_t* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) wp[t] = W + ((long)min(n0 + 16 * (t % P) + (lane & 15), N - 1) + (t / P) * (long)N) * K;
  fr_f32x4 acc[NT][NB];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[t][b] = fr_f32x4{0.f, 0.f, 0.f, 0.f};
  few_rows_core<NT, NB, WV, U>(acc, wp, [&](int r) { return X + r * x_stride; }, rows, K,
                               reinterpret_cast<char*>(red) + wave * kFrStage<NB, U>, wave, lane);
  __syncthreads();
  few_rows_park<NT, NB, WV>(red, acc, wave, lane);
  __syncthreads();
  // entry (tile, block, lane'): lane' = 16 q' + row, columns 4 q' .. 4 q' + 3
  for (int e = tid; e < P * NB * 64; e += 64 * WV) {
    const int el = e & 63, b = (e >> 6) % NB, t = (e >> 6) / NB;
    const int r = 16 * b + (el & 15), c = n0 + 16 * t + 4 * (el >> 4);
    if (r >= rows || c >= N) continue;
    float v[4];
    few_rows_sum<NT, NB, WV>(red, t, b, el, v);
    if constexpr (GLU) {
      float u[4];
      few_rows_sum<NT, NB, WV>(red, t + P, b, el, u);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = fr_act(act, limit, v[i], u[i]);
    } else {
      if (bias != nullptr) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += c + i < N ? ft::bf16_to_f32(bias[c + i]) : 0.f;
      }
      if (act == kFrReluSq) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = fr_act(act, limit, v[i], 0.f);
      }
      if constexpr (RIDE) {
        if (R.table != nullptr) {
          const int id = R.ids[r];
          const bf16_t* g = R.table + (long)(id < 0 || id >= R.vocab ? 0 : id) * R.table_stride + c;
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = c + i < N ? gelu_tanh_(v[i]) * ft::bf16_to_f32(g[i]) : 0.f;
        }
      }
      if constexpr (sizeof(TO) == 4) {           // logits: as tanh_cap_kernel, 5 us less than behind the product
        if (act == kFrTanhCap) {
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = isfinite(v[i]) ? limit * tanhf(v[i] / limit) : v[i];
        }
      }
    }
    fr_store4(Y + r * y_stride, c, N, vec != 0, v);
  }
}

// ---------------------------------------------------------------------------------
// D[r, p, n] = the sum over part p of k (the first: + bias[n]), blockIdx.y: products of few columns, whose tiles are half the chip's CUs and each a chain
// along k.  What reads Y there is a norm, which adds the parts as it reads them (rows.hip: ExpertRows; moe_route.hip).
// Bound by the read of W, and by the latency of the first loads.  N = 2048, weights from HBM, us at 1 / 16 / 32 / 64 rows, a
// workgroup a tile beside it:
//   K = 2048, two parts, 8 waves       4.4 4.4 5.2 6.3    (5.2 5.8 6.9 8.6)
//   K = 4096, four parts               5.4 6.0 7.2 9.1    (7.3 8.4 10.5 14.0)
//   K = 8192, four parts               8.4 9.4 11.4 15.2  (11.4 13.5 17.6 24.5)
//   K = 14336, four parts              12.2 15.4 18.4 25.1 (18.1 23.3 31.2 43.3)
// ---------------------------------------------------------------------------------
template <int NB, int WV, int U>
__global__ void __launch_bounds__(64 * WV)
few_rows_parts_kernel(float* __restrict__ D, const bf16_t* __restrict__ X, long x_stride, int rows, const bf16_t* __restrict__ W,
                      const bf16_t* __restrict__ bias, int N, int K, int part) {
  extern __shared__ float4 red[];                // X stages, then partial sums
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.x * 16, k0 = blockIdx.y * part;
  const bf16_t* wp[1] = {W + (long)min(n0 + (lane & 15), N - 1) * K + k0};
  fr_f32x4 acc[1][NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[0][b] = fr_f32x4{0.f, 0.f, 0.f, 0.f};
  few_rows_core<1, NB, WV, U>(acc, wp, [&](int r) { return X + r * x_stride + k0; }, rows, min(part, K - k0),
                              reinterpret_cast<char*>(red) + wave * kFrStage<NB, U>, wave, lane);
  __syncthreads();
  few_rows_park<1, NB, WV>(red, acc, wave, lane);
  __syncthreads();
  for (int e = tid; e < NB * 64; e += 64 * WV) {
    const int el = e & 63, b = e >> 6, r = 16 * b + (el & 15), c = n0 + 4 * (el >> 4);
    if (r >= rows || c >= N) continue;
    float v[4];
    few_rows_sum<1, NB, WV>(red, 0, b, el, v);
    if (bias != nullptr && blockIdx.y == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] += ft::bf16_to_f32(bias[c + i]);      // (N: whole fours)
    }
    fr_store4(D + ((long)r * gridDim.y + blockIdx.y) * N, c, N, true, v);
  }
}

template <int NB, int WV, int U>
int few_rows_parts_launch(float* D, const void* X, long x_stride, int rows, const void* W, const void* bias, int N, int K, int parts, hipStream_t s) {
  constexpr int kRed = WV * NB * 1024, kX = WV * kFrStage<NB, U>, lds = kRed > kX ? kRed : kX;
  static_assert(lds <= 160 * 1024, "");
  auto kernel = few_rows_parts_kernel<NB, WV, U>;
  if constexpr (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return (int)e;
  }
  const int part = ((K + 63) / 64 + parts - 1) / parts * 64;
  hipLaunchKernelGGL(kernel, dim3((unsigned)((N + 15) / 16), (unsigned)parts), dim3(64 * WV), lds, s, D, (const bf16_t*)X, x_stride,
                     rows, (const bf16_t*)W, (const bf16_t*)bias, N, K, part);
  return (int)hipGetLastError();
}

// Parts of k (1: few_rows_gemm is as fast): until there are two to three workgroups a CU.  From a grid of N = 1280 to 6144, K = 1024 to
// 14336 and 1 to 64 rows, us of one / two / four / eight parts at 16 rows: N = 1280, K = 8192 13.3 - 8.5 7.2; 2048, 1024 3.7
// 3.3; 3072, 1024 4.2 4.3; 3072, 4096 9.0 8.4 7.5; 4096, 2048 6.7 6.3 6.2; 4096, 8192 15.6 15.6 16.3.  Every part is a row more
// for the step behind to read, so where a few per cent are all there is to gain (4096 columns on) k stays whole.
int few_rows_parts(int N, int K) {
  if (N > 3584 || K < 1024 || (N > 2048 && K < 2048)) return 1;
  return K >= 4096 || N > 2048 ? 4 : 2;
}

// Waves and steps in flight: where the columns fill the chip four waves with one step are the best at all rows; below, shares of k of
// 512 or less are one round of loads for eight waves, and with more rows X's way through LDS counts (four waves).
template <int NB>
int few_rows_parts_pick(float* D, const void* X, long x_stride, int rows, const void* W, const void* bias, int N, int K, int parts, hipStream_t s) {
#define FR_PARTS(WV, U) few_rows_parts_launch<NB, WV, U>(D, X, x_stride, rows, W, bias, N, K, parts, s)
  if (N > 2048) return FR_PARTS(4, 1);
  if (parts <= 2) return K < 2048 || NB == 4 ? FR_PARTS(8, 1) : FR_PARTS(8, 2);
  return NB == 1 ? FR_PARTS(8, 1) : FR_PARTS(4, 2);
#undef FR_PARTS
}

// ---------------------------------------------------------------------------------
// Experts of few rows.  A workgroup owns one tile of 16 (two) columns of one expert's matrix and
// serves every row that chose the expert: the matrix is read once however many rows share it.
// blockIdx.y: the shared expert, which serves all rows and whose down matrix may have the longest rows, where there is one; then
// the experts (expert_in_slot).
// Bound by the stream of the chosen experts' matrices.  us of the first and the down matrices (forms: mx_experts_few), alone with
// weights from HBM, as before / now (one form for all with the shared expert last): 32 rows, top 4 of 32 experts of 1536 (relu^2) and a shared one of 3072,
// 214 MB each 52 + 51, 41 + 41; 16 rows, top 6 of 32 gated experts of 1024 48 + 26, 47 + 25; 8 rows, top 4 of them and a shared one
// of 2048 37 + 24, 36 + 20; 3 rows 24 + 17, 24 + 14.
// ---------------------------------------------------------------------------------
struct ExpertSet {
  const bf16_t* w;        // [experts][rows_w][K]
  const bf16_t* shared;   // [shared rows][K_shared], or null
  int experts, K, N;      // N: output columns (GLU: of gate and of up each)
  int shared_K, shared_N;
  int slots;              // workgroups' rows of the grid before the shared expert's: the experts, or the most that can be chosen
};

__device__ __forceinline__ int expert_of(int v, int experts) { return v < 0 || v >= experts ? 0 : v; }

// Expert of a row of the grid: itself, or where there are fewer rows than experts the slot-th of the chosen ones (none: -1).
// One row, top 6 of 32 experts: 6 x 64 workgroups instead of 32 x 64, most of which end after they have read the choices.
__device__ __forceinline__ int expert_in_slot(const int* __restrict__ idx, int pairs, const ExpertSet& E, int slot) {
  if (E.slots == E.experts) return slot;         // (E.experts <= 64 otherwise)
  const int lane = threadIdx.x & 63;
  uint64_t m = 0;
  for (int p = lane; p < pairs; p += 64) m |= 1ull << expert_of(idx[p], E.experts);
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) m |= __shfl_xor((unsigned long long)m, o, 64);
  for (int i = 0; i < slot; ++i) m &= m - 1;
  return m != 0 ? __builtin_amdgcn_readfirstlane(__builtin_ctzll(m)) : -1;
}

// the (row, choice) pairs that chose expert e -> list, ascending, the first `room` of them; returns how many there are.
// `once`: a row's first pair only.  All threads of the workgroup call it.
template <int WV>
__device__ __forceinline__ int pairs_of(const int* __restrict__ idx, int pairs, int top, int experts, int e, bool once,
                                        int room, int* list, int* counts) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int total = 0;
  for (int p0 = 0; p0 < pairs; p0 += 64 * WV) {
    const int p = p0 + tid;
    bool mine = p < pairs && expert_of(idx[p], experts) == e;
    if (once && mine)
      for (int q = p / top * top; q < p; ++q) mine = mine && expert_of(idx[q], experts) != e;
    const uint64_t m = __ballot(mine);
    if (lane == 0) counts[wave] = __popcll(m);
    __syncthreads();
    int before = total;
    for (int w = 0; w < WV; ++w) {
      if (w < wave) before += counts[w];
      total += counts[w];
    }
    const int at = before + __popcll(m & ((1ull << lane) - 1));
    if (mine && at < room) list[at] = p;
    __syncthreads();
  }
  return total;
}

// The same for a tile with room for all rows.  A router names an expert once per row, except for a row of NaN, whose choices
// are all the same, and an index outside the experts counts as the first's.  Where that makes more pairs than there
// is room, the list has a row's first pair and the others take its results (`shared`).  (Walking a longer list in turns
// cost the products 2 to 15%, in registers; looking for repeated choices always, 1 to 5 us.)
template <int WV>
__device__ __forceinline__ int rows_of(const int* __restrict__ idx, int pairs, int top, int experts, int e, int room, int* list,
                                       int* counts, bool& shared) {
  int count = pairs_of<WV>(idx, pairs, top, experts, e, false, room, list, counts);
  shared = count > room;
  if (shared) count = pairs_of<WV>(idx, pairs, top, experts, e, true, room, list, counts);
  return count;
}

// the tile's sums for the listed rows: f(entry row in the list, column, sums, up sums)
template <int P, bool GLU, int NB, int WV, int U, bool AHEAD, typename F>
__device__ __forceinline__ void expert_tile(float4* red, const bf16_t* W, int N, int K, int n0, const bf16_t* X,
                                            long x_stride, const int* list, int count, int div, int wave, int lane,
                                            F out) {
  constexpr int NT = GLU ? 2 * P : P;
  const bf16_t* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) wp[t] = W + ((long)min(n0 + 16 * (t % P) + (lane & 15), N - 1) + (t / P) * (long)N) * K;
  fr_f32x4 acc[NT][NB];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[t][b] = fr_f32x4{0.f, 0.f, 0.f, 0.f};
  const auto row = [&](int r) { return X + (long)(list[r] / div) * x_stride; };
  char* const stage = reinterpret_cast<char*>(red) + wave * kFrStage<NB, U>;
  if constexpr (AHEAD) few_rows_core_ahead<NT, NB, WV, U>(acc, wp, row, count, K, stage, wave, lane);
  else few_rows_core<NT, NB, WV, U>(acc, wp, row, count, K, stage, wave, lane);
  __syncthreads();
  few_rows_park<NT, NB, WV>(red, acc, wave, lane);
  __syncthreads();
  for (int e = threadIdx.x; e < P * NB * 64; e += 64 * WV) {
    const int el = e & 63, b = (e >> 6) % NB, t = (e >> 6) / NB;
    const int r = 16 * b + (el & 15), c = n0 + 16 * t + 4 * (el >> 4);
    if (r >= count || c >= N) continue;
    float v[4], u[4] = {0.f, 0.f, 0.f, 0.f};
    few_rows_sum<NT, NB, WV>(red, t, b, el, v);
    if constexpr (GLU) few_rows_sum<NT, NB, WV>(red, t + P, b, el, u);
    out(r, c, v, u);
  }
}

// blocks of 16 rows that the listed rows fill, at most MB
template <int P, bool GLU, int WV, int MB, int U, bool AHEAD, typename F>
__device__ __forceinline__ void expert_tile_any(float4* red, const bf16_t* W, int N, int K, int n0, const bf16_t* X,
                                                long x_stride, const int* list, int count, int div, int wave, int lane,
                                                F out) {
  if (MB == 1 || count <= 16) expert_tile<P, GLU, 1, WV, U, AHEAD>(red, W, N, K, n0, X, x_stride, list, count, div, wave, lane, out);
  else if (MB == 2 || count <= 32) expert_tile<P, GLU, 2, WV, U, AHEAD>(red, W, N, K, n0, X, x_stride, list, count, div, wave, lane, out);
  else expert_tile<P, GLU, MB, WV, U, AHEAD>(red, W, N, K, n0, X, x_stride, list, count, div, wave, lane, out);
}

// float4s of X stages and partial sums of WV waves' NT tiles with MB blocks of rows
template <int NT, int MB, int WV, int U>
constexpr int kExpLds = WV * (kFrStage<MB, U> > 1024 * NT * MB ? kFrStage<MB, U> : 1024 * NT * MB) / 16;

// y[pair] = act(first matrices of the pair's expert times its row of h); ys[row] the same of the
// shared expert; with a shared gate (one more row of its matrix) sg[row] = that row's product, by
// the workgroup past the shared expert's last tile.
template <bool GLU, int P, int MB, int WV, int U, bool AHEAD>
__global__ void __launch_bounds__(64 * WV)
experts_first_kernel(bf16_t* __restrict__ y, bf16_t* __restrict__ ys, float* __restrict__ sg,
                     const bf16_t* __restrict__ h, long h_stride, int rows, const int* __restrict__ idx, int top,
                     ExpertSet E, int act, float limit, float shared_limit) {
  __shared__ float4 red[kExpLds<GLU ? 2 * P : P, MB, WV, U>];
  __shared__ int list[kFewRows], counts[WV];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.x * 16 * P, slot = (int)blockIdx.y - (E.shared != nullptr ? 1 : 0);
  if (slot >= 0) {
    if (n0 >= E.N) return;
    const int e = expert_in_slot(idx, rows * top, E, slot);
    if (e < 0) return;
    bool shared;
    const int count = rows_of<WV>(idx, rows * top, top, E.experts, e, 16 * MB, list, counts, shared);
    if (count == 0) return;
    const bf16_t* W = E.w + (long)e * E.N * (GLU ? 2 : 1) * E.K;
    expert_tile_any<P, GLU, WV, MB, U, AHEAD>(red, W, E.N, E.K, n0, h, h_stride, list, count, top, wave, lane,
                                       [&](int r, int c, float (&v)[4], float (&u)[4]) {
#pragma unroll
                                         for (int i = 0; i < 4; ++i) v[i] = fr_act(act, limit, v[i], u[i]);
                                         fr_store4(y + (long)list[r] * E.N, c, E.N, true, v);
                                       });
    return;
  }
  const int tiles = (E.shared_N + 16 * P - 1) / (16 * P);
  if ((int)blockIdx.x > tiles || ((int)blockIdx.x == tiles && sg == nullptr)) return;
  if (tid < rows) list[tid] = tid;
  __syncthreads();
  if ((int)blockIdx.x == tiles) {
    const bf16_t* W = E.shared + (long)E.shared_N * (GLU ? 2 : 1) * E.K;
    expert_tile_any<1, false, WV, MB, U, AHEAD>(red, W, 1, E.K, 0, h, h_stride, list, rows, 1, wave, lane,
                                         [&](int r, int c, float (&v)[4], float (&)[4]) { if (c == 0) sg[r] = v[0]; });
    return;
  }
  expert_tile_any<P, GLU, WV, MB, U, AHEAD>(red, E.shared, E.shared_N, E.K, n0, h, h_stride, list, rows, 1, wave, lane,
                                     [&](int r, int c, float (&v)[4], float (&u)[4]) {
#pragma unroll
                                       for (int i = 0; i < 4; ++i) v[i] = fr_act(act, shared_limit, v[i], u[i]);
                                       fr_store4(ys + (long)r * E.shared_N, c, E.shared_N, true, v);
                                     });
}

// d[pair] = W_down of the pair's expert times y[pair], ds[row] the shared expert's, fp32
template <int P, int MB, int WV, int U>
__global__ void __launch_bounds__(64 * WV)
experts_down_kernel(float* __restrict__ d, float* __restrict__ ds, const bf16_t* __restrict__ y,
                    const bf16_t* __restrict__ ys, int rows, const int* __restrict__ idx, int top, ExpertSet E) {
  __shared__ float4 red[kExpLds<P, MB, WV, U>];
  __shared__ int list[kFewRows], counts[WV];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.x * 16 * P, slot = (int)blockIdx.y - (E.shared != nullptr ? 1 : 0);
  const bool routed = slot >= 0;
  const int e = routed ? expert_in_slot(idx, rows * top, E, slot) : 0;
  if (e < 0) return;
  float* dst = d;
  const bf16_t *W = E.w + (long)e * E.N * E.K, *X = y;
  int K = E.K, count = rows;
  bool shared = false;
  if (routed) {
    count = rows_of<WV>(idx, rows * top, top, E.experts, e, 16 * MB, list, counts, shared);
    if (count == 0) return;
  } else {
    if (tid < rows) list[tid] = tid;
    __syncthreads();
    dst = ds;
    W = E.shared;
    X = ys;
    K = E.shared_K;
  }
  expert_tile_any<P, false, WV, MB, U, false>(red, W, E.N, K, n0, X, K, list, count, 1, wave, lane,
                                       [&](int r, int c, float (&v)[4], float (&)[4]) {
                                         const int p = list[r];
                                         fr_store4(dst + (long)p * E.N, c, E.N, true, v);
                                         if (!shared) return;
                                         for (int q = p + 1; q % top != 0; ++q)
                                           if (expert_of(idx[q], E.experts) == e) fr_store4(dst + (long)q * E.N, c, E.N, true, v);
                                       });
}

// out[row] = sum_k wts[row, k] d[row, k] + shared[row] * (sigmoid(sg[row]) or 1)
__global__ void __launch_bounds__(256)
experts_combine_kernel(float* __restrict__ out, const float* __restrict__ d, const float* __restrict__ wts,
                       const float* __restrict__ ds, const float* __restrict__ sg, int top, int width) {
  const long row = blockIdx.y;
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= width) return;
  float v = 0.f;
#pragma unroll 4
  for (int k = 0; k < top; ++k) v += wts[row * top + k] * d[(row * top + k) * width + c];
  if (ds != nullptr) v += ds[row * width + c] * (sg != nullptr ? sigmoidf_(sg[row]) : 1.f);
  out[row * width + c] = v;
}

template <int P, bool GLU, int NB, int WV, int U, typename TO, bool RIDE>
int few_rows_launch(void* Y, long y_stride, const void* X, long x_stride, int rows, const void* W, const void* bias,
                    int N, int K, int act, float limit, int vec, const FewRowsRider& R, hipStream_t s) {
  constexpr int NT = GLU ? 2 * P : P;
  constexpr int kRed = WV * NT * NB * 1024, kX = WV * kFrStage<NB, U>, lds = kRed > kX ? kRed : kX;
  auto kernel = few_rows_gemm_kernel<P, GLU, NB, WV, U, TO, RIDE>;
  if constexpr (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return (int)e;
  }
  hipLaunchKernelGGL(kernel, dim3((unsigned)((N + 16 * P - 1) / (16 * P)), R.W2 != nullptr ? 2 : 1), dim3(64 * WV), lds, s,
                     (TO*)Y, y_stride, (const bf16_t*)X, x_stride, rows, (const bf16_t*)W, (const bf16_t*)bias, N, K, act, limit, vec,
                     R);
  return (int)hipGetLastError();
}

// Tiles per workgroup, waves and steps in flight, measured with weights that come from HBM (K = 2048
// unless said; us at 1 / 16 / 32 / 64 rows, the vendor's product beside it):
//   N = 2048 and 3072: 8 waves, two steps       5.3 5.9 7.0 8.6      (vendor 11.0 11.0 11.1 11.6)
//   N = 2048, K = 8192                          11.6 13.8 18.0 24.6  (13.1 13.2 16.0 22.6)
//   N = 10272: 4 waves, one step, more groups   11.8 11.7 14.8 22.1  (16.4 14.3 14.3 15.7)
//   N = 32768: four tiles share an X fragment   26.9 27.7 29.0 34.2  (35.1 33.5 35.2 36.2; 24.0 at 5.6 TB/s)
//   gated, 2 x 8192: 4 waves                    15.7 15.7 17.5 21.8  (18 + 5 for the activation)
// Below 1024 columns of X a wave has one step or none: four waves.
template <bool GLU, int NB, typename TO, bool RIDE = false>
int few_rows_pick(void* Y, long y_stride, const void* X, long x_stride, int rows, const void* W, const void* bias,
                  int N, int K, int act, float limit, int vec, const FewRowsRider& R, hipStream_t s) {
#define FR_RUN(P, WV, U) \
  few_rows_launch<P, GLU, NB, WV, U, TO, RIDE>(Y, y_stride, X, x_stride, rows, W, bias, N, K, act, limit, vec, R, s)
  if constexpr (GLU) {
    return FR_RUN(1, 4, NB == 4 ? 2 : 1);
  } else {
    if (N >= 16384 || (NB == 4 && N > 4096)) return FR_RUN(4, 4, 1);
    return N > 4096 || K < 1024 ? FR_RUN(1, 4, 1) : FR_RUN(1, 8, 2);
  }
#undef FR_RUN
}

}  // namespace mx

using namespace mx;

extern "C" int mx_few_rows_max() { return kFewRows; }

extern "C" int mx_few_rows_gemm(void* Y, int y_f32, long y_stride, const void* X, long x_stride, int rows,
                                const void* W, const void* bias, int N, int K, int act, float limit, hipStream_t s) {
  if (rows <= 0 || N <= 0) return 0;
  if (rows > kFewRows || K < 8 || K % 8 || x_stride % 8 || act < kFrStore || act > kFrTanhCap || (act == kFrTanhCap && !y_f32))
    return -1;
  if (((uintptr_t)X) % 16 || ((uintptr_t)W) % 16) return -2;
  const bool glu = act >= kFrGelu && act <= kFrClamp;
  if (glu && (bias != nullptr || y_f32)) return -3;
  const int es = y_f32 ? 4 : 2;
  const int vec = y_stride % 4 == 0 && ((uintptr_t)Y) % (4 * es) == 0;
  const int nb = rows <= 16 ? 1 : rows <= 32 ? 2 : 4;
  const FewRowsRider R{};
#define FR_GO(GLU, TO)                                                                                               \
  (nb == 1   ? few_rows_pick<GLU, 1, TO>(Y, y_stride, X, x_stride, rows, W, bias, N, K, act, limit, vec, R, s)       \
   : nb == 2 ? few_rows_pick<GLU, 2, TO>(Y, y_stride, X, x_stride, rows, W, bias, N, K, act, limit, vec, R, s)       \
             : few_rows_pick<GLU, 4, TO>(Y, y_stride, X, x_stride, rows, W, bias, N, K, act, limit, vec, R, s))
  if (glu) return FR_GO(true, bf16_t);
  return y_f32 ? FR_GO(false, float) : FR_GO(false, bf16_t);
#undef FR_GO
}

extern "C" int mx_few_rows_parts(int N, int K) { return few_rows_parts(N, K); }

// D [rows][parts][N]: parts as mx_few_rows_parts says, or fewer than K has steps of 64
extern "C" int mx_few_rows_gemm_parts(float* D, const void* X, long x_stride, int rows, const void* W, const void* bias,
                                      int N, int K, int parts, hipStream_t s) {
  if (rows <= 0 || N <= 0) return 0;
  if (rows > kFewRows || K < 8 || K % 8 || x_stride % 8 || N % 4 || parts < 1 || parts > 65535) return -1;
  if (((((K + 63) / 64) + parts - 1) / parts) * 64L * (parts - 1) >= K) return -1;       // (a part without any k)
  if (((uintptr_t)X | (uintptr_t)W | (uintptr_t)D) % 16) return -2;
  if (rows <= 16) return few_rows_parts_pick<1>(D, X, x_stride, rows, W, bias, N, K, parts, s);
  if (rows <= 32) return few_rows_parts_pick<2>(D, X, x_stride, rows, W, bias, N, K, parts, s);
  return few_rows_parts_pick<4>(D, X, x_stride, rows, W, bias, N, K, parts, s);
}

// bf16 products with a rider: Y = X W^T and Y2 = X2 W2^T, of the same sizes and strides
extern "C" int mx_few_rows_pair(void* Y, void* Y2, long y_stride, const void* X, const void* X2, long x_stride, int rows,
                                const void* W, const void* W2, int N, int K, hipStream_t s) {
  if (rows <= 0 || N <= 0) return 0;
  if (rows > kFewRows || K < 8 || K % 8 || x_stride % 8 || W2 == nullptr) return -1;
  if (((uintptr_t)X | (uintptr_t)X2 | (uintptr_t)W | (uintptr_t)W2) % 16) return -2;
  const int vec = y_stride % 4 == 0 && ((uintptr_t)Y | (uintptr_t)Y2) % 8 == 0;
  const FewRowsRider R{(const bf16_t*)X2, (const bf16_t*)W2, Y2, nullptr, nullptr, 0, 0};
  if (rows <= 16) return few_rows_pick<false, 1, bf16_t, true>(Y, y_stride, X, x_stride, rows, W, nullptr, N, K, kFrStore, 0.f, vec, R, s);
  if (rows <= 32) return few_rows_pick<false, 2, bf16_t, true>(Y, y_stride, X, x_stride, rows, W, nullptr, N, K, kFrStore, 0.f, vec, R, s);
  return few_rows_pick<false, 4, bf16_t, true>(Y, y_stride, X, x_stride, rows, W, nullptr, N, K, kFrStore, 0.f, vec, R, s);
}

// Y = gelu(X W^T) * table[ids[row], 0 .. N), ids outside 0 .. vocab as 0
extern "C" int mx_few_rows_side_gate(void* Y, long y_stride, const void* X, long x_stride, int rows, const void* W, int N, int K,
                                     const void* table, long table_stride, const int* ids, int vocab, hipStream_t s) {
  if (rows <= 0 || N <= 0) return 0;
  if (rows > kFewRows || K < 8 || K % 8 || x_stride % 8 || table == nullptr || vocab < 1) return -1;
  if (((uintptr_t)X | (uintptr_t)W) % 16) return -2;
  const int vec = y_stride % 4 == 0 && ((uintptr_t)Y) % 8 == 0;
  const FewRowsRider R{nullptr, nullptr, nullptr, (const bf16_t*)table, ids, table_stride, vocab};
  if (rows <= 16) return few_rows_pick<false, 1, bf16_t, true>(Y, y_stride, X, x_stride, rows, W, nullptr, N, K, kFrStore, 0.f, vec, R, s);
  if (rows <= 32) return few_rows_pick<false, 2, bf16_t, true>(Y, y_stride, X, x_stride, rows, W, nullptr, N, K, kFrStore, 0.f, vec, R, s);
  return few_rows_pick<false, 4, bf16_t, true>(Y, y_stride, X, x_stride, rows, W, nullptr, N, K, kFrStore, 0.f, vec, R, s);
}

extern "C" int mx_experts_few(float* out, void* y, float* d, const void* h, long h_stride, const int* idx,
                              const float* wts, const void* wgu, const void* wdown, int rows, int top, int experts,
                              int ff, int width, float limit, int act, void* ys, float* ds, float* sg,
                              const void* shared_w, const void* shared_down, int shared_ff, float shared_limit,
                              hipStream_t s) {
  if (rows <= 0) return 0;
  if (rows > kFewRows || experts < 1 || experts > 65534 || top < 1 || ff % 8 || width % 8 ||
      ff < 8 || width < 8 || h_stride % 8 || shared_ff % 8 || act < kFrGelu || act > kFrReluSq ||
      (shared_w == nullptr) != (shared_down == nullptr)) return -1;
  if (((uintptr_t)h) % 16 || ((uintptr_t)wgu) % 16 || ((uintptr_t)wdown) % 16 || ((uintptr_t)shared_w) % 16 ||
      ((uintptr_t)shared_down) % 16) return -2;
  const bool glu = act != kFrReluSq, sh = shared_w != nullptr;
  // Forms by the rows, us of 32 experts and a shared one (rows of the comment above), tiles a workgroup x waves x steps of k a round:
  //   first, gated      1 x 4 x 1   1 x 4 x 2, the next round's loads under a round   1 x 8 x 1    (4096 wide, 32 rows: 1 x 8 x 2 241, x 1 248)
  //     8 rows          41.1        36.4                                               37.9
  //     32 rows         56.2        -                                                  52.8
  //     64 rows         61.2        -                                                  64.3
  //   first, relu^2     2 x 4 x 1   1 x 4 x 2, loads ahead    1 x 8 x 1   1 x 4 x 1
  //     8 rows          39.5        29.6                      29.6        30.5
  //     32 rows         50.2        -                         40.8        43.4
  //     64 rows         55.7        -                         60.9        56.4
  //   down              2 x 4 x 1   1 x 4 x 2                 2 x 8 x 1   (of 1024 / 1536)
  //     8 rows          21.7 33     19.8 29.9                 20.4 30.4
  //     32 rows         29.0 43.4   - 44.6                    29.0 41.3
  //     64 rows         33.5 48.0   -                         36.7 51.0
  const bool many = rows > 32;
  const int p1 = glu || !many ? 1 : 2, p2 = rows <= 16 ? 1 : 2, cols = 16 * p1;
  const int tiles = (ff + cols - 1) / cols, tiles_s = sh ? (shared_ff + cols - 1) / cols + (sg != nullptr) : 0;
  const int tiles_d = (width + 16 * p2 - 1) / (16 * p2);
  // The lines below are from 700 layers of at most 16 rows, 4 to 128 experts, sizes at random.  Rows of the grid per pair: less than 150
  // workgroups spared cost up to 0.9 us (the choices are read first), 150 to 300 are level (-3 to 1), 300 to 600 save 0.5, 1000 1.2 and
  // more 2 to 5.  Loads ahead: 1.01 to 1.12 of the time at 1 to 3 steps of k a wave, whatever the grid; from 4 on 0.94 to 0.99 up to a
  // workgroup a CU, 0.96 to 0.99 with three and more, between these 1.00 to 1.03 (up to 1.2).
  const int pairs = rows * top;
  const auto slots = [&](int cols) { return experts <= 64 && pairs < experts && (long)(experts - pairs) * cols >= 150 ? pairs : experts; };
  // workgroups that have rows, where the rows choose their experts independently
  const float groups = experts * (1.f - powf(1.f - (float)(top < experts ? top : experts) / experts, (float)rows)) * tiles + tiles_s;
  const bool ahead = (width + 63) / 64 > 12 && (groups <= 256.f || groups > 700.f);
  ExpertSet first{(const bf16_t*)wgu, (const bf16_t*)shared_w, experts, width, ff, width, shared_ff, slots(tiles)};
  ExpertSet down{(const bf16_t*)wdown, (const bf16_t*)shared_down, experts, ff, width, shared_ff, width, slots(tiles_d)};
  const dim3 g1((unsigned)(tiles > tiles_s ? tiles : tiles_s), (unsigned)(first.slots + (sh ? 1 : 0)));
  const dim3 g2((unsigned)tiles_d, (unsigned)(down.slots + (sh ? 1 : 0)));
#define EX_FIRST(GLU, P, MB, WV, U, AHEAD)                                                                                \
  hipLaunchKernelGGL((experts_first_kernel<GLU, P, MB, WV, U, AHEAD>), g1, dim3(64 * WV), 0, s, (bf16_t*)y, (bf16_t*)ys, sg, \
                     (const bf16_t*)h, h_stride, rows, idx, top, first, act, limit, shared_limit)
#define EX_DOWN(P, MB, WV, U)                                                                                          \
  hipLaunchKernelGGL((experts_down_kernel<P, MB, WV, U>), g2, dim3(64 * WV), 0, s, d, ds, (const bf16_t*)y, (const bf16_t*)ys, \
                     rows, idx, top, down)
#define EX_FIRST_ROWS(GLU)                                \
  do {                                                    \
    if (many) EX_FIRST(GLU, GLU ? 1 : 2, 4, 4, 1, false); \
    else if (rows > 16 && width >= 4096) EX_FIRST(GLU, 1, 2, 8, 2, false); \
    else if (rows > 16) EX_FIRST(GLU, 1, 2, 8, 1, false); \
    else if (ahead) EX_FIRST(GLU, 1, 1, 4, 2, true);      \
    else EX_FIRST(GLU, 1, 1, 4, 1, false);                \
  } while (0)
  if (glu) EX_FIRST_ROWS(true);
  else EX_FIRST_ROWS(false);
  if (many) EX_DOWN(2, 4, 4, 1);
  else if (rows > 16) EX_DOWN(2, 2, 8, 1);
  else EX_DOWN(1, 1, 4, 2);
#undef EX_FIRST_ROWS
#undef EX_FIRST
#undef EX_DOWN
  if (out == nullptr) return (int)hipGetLastError();       // (the step behind sums them: rows.hip, ExpertRows)
  hipLaunchKernelGGL(experts_combine_kernel, dim3((unsigned)((width + 255) / 256), (unsigned)rows), dim3(256), 0, s,
                     out, d, wts, sh ? ds : nullptr, sg, top, width);
  return (int)hipGetLastError();
}

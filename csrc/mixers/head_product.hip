// Products of few rows with a matrix per head, in fp32: what a decode step of latent attention needs around its attention,
// q W_uk (into latent space, with the rotation of the queries' other part) and o W_uv (to the values, gated and rounded).
//   y[t, h, :] = x[t, h, :] W[h]      W fp32 [heads][K][N]
// A workgroup owns 4 Q columns of one head: a lane a quad of columns and eight rows of W, whose 16-byte loads are all under
// way before the rows of x have arrived in LDS; the lanes' sums over K meet by shuffles and through LDS.
// Bound by latency, a chain of load, products and two exchanges; W is read once for eight rows.  Q is 16 where that makes 128
// workgroups and 4 otherwise (64-byte pieces of W's rows).
// 8 rows of 16 heads, 128 -> 512 in 4.7 us (rotation and library product 8.8), 512 -> 128 with gate in 6.0 (14.5).
#include "mx_common.h"

namespace mx {

constexpr int kHpRows = 8;       // rows of x at a time
constexpr int kHpK = 8;          // rows of W a thread holds

struct HeadProduct {
  const float* w;
  int K, N, rows, heads;
  const void* x;                 // x[t * x_t + h * x_h + k]
  long x_t, x_h;
  void* y;                       // y[t * y_t + h * y_h + n]
  long y_t, y_h;
  const void* gate;              // y times sigmoid(gate[t * gate_t + h]), or null
  long gate_t;
  // ROPE: x's rows are [K | dr]; the rotated dr -> qr [rows][heads][dr], by one more workgroup a head
  float* qr;
  const float* table;
  const int* positions;
  int table_rows, dims, dr, interleaved;
};

template <int Q, typename TX, typename TO, bool ROPE>
__global__ void __launch_bounds__(256)
head_product_kernel(HeadProduct P) {
  constexpr int KG = 256 / Q, LG = 64 / Q;             // groups along K: of the workgroup, of a wave
  extern __shared__ __attribute__((aligned(16))) float xs[];          // [kHpRows][K], then [4][kHpRows][4 Q] sums
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = blockIdx.y, K = P.K;
  const TX* x = (const TX*)P.x + h * P.x_h;
  if (ROPE && blockIdx.x + 1 == gridDim.x) {
    for (int e = tid; e < P.rows * P.dr; e += 256) {
      const int t = e / P.dr, j = e % P.dr;
      int p = P.positions[t];
      p = p < 0 ? 0 : (p >= P.table_rows ? P.table_rows - 1 : p);
      const TX* u = x + t * P.x_t + K;
      P.qr[((long)t * P.heads + h) * P.dr + j] =
          j < P.dims ? rope_at(u, j, P.dims, P.table + (long)p * P.dims, P.interleaved) : ld(u, j);
    }
    return;
  }
  const int n = (blockIdx.x * Q + tid % Q) * 4, kg = tid / Q, nl = min(n, P.N - 4);
  const float* w = P.w + (long)h * K * P.N + nl;
  float* sums = xs + kHpRows * K;
  float4 wr[kHpK];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < kHpK; ++i) wr[i] = *reinterpret_cast<const float4*>(w + (long)min(k0 + kg * kHpK + i, K - 1) * P.N);
  };
  fetch(0);
  for (int t0 = 0; t0 < P.rows; t0 += kHpRows) {
    const int nt = min(kHpRows, P.rows - t0);
    for (int e = tid * 4; e < nt * K; e += 1024) {
      const int t = e / K, k = e % K;
      float v[4];
      if constexpr (sizeof(TX) == 2) {
        const uint2 u = *reinterpret_cast<const uint2*>(x + (t0 + t) * P.x_t + k);
        ft::unpack2(u.x, v[0], v[1]);
        ft::unpack2(u.y, v[2], v[3]);
      } else {
        const float4 u = *reinterpret_cast<const float4*>(x + (t0 + t) * P.x_t + k);
        v[0] = u.x, v[1] = u.y, v[2] = u.z, v[3] = u.w;
      }
      *reinterpret_cast<float4*>(xs + e) = make_float4(v[0], v[1], v[2], v[3]);
    }
    __syncthreads();
    float acc[kHpRows][4] = {};
    for (int k0 = 0; k0 < K; k0 += kHpK * KG) {
      if (k0 > 0) fetch(k0);
      const int k = k0 + kg * kHpK;
      if (k < K) {                                     // (K in whole eights)
#pragma unroll
        for (int t = 0; t < kHpRows; ++t) {
          if (t >= nt) break;
          const float4 a = *reinterpret_cast<const float4*>(xs + t * K + k), b = *reinterpret_cast<const float4*>(xs + t * K + k + 4);
          const float xv[kHpK] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
          for (int i = 0; i < kHpK; ++i) {
            acc[t][0] += xv[i] * wr[i].x;
            acc[t][1] += xv[i] * wr[i].y;
            acc[t][2] += xv[i] * wr[i].z;
            acc[t][3] += xv[i] * wr[i].w;
          }
        }
      }
    }
    if (t0 + kHpRows < P.rows && K > kHpK * KG) fetch(0);
#pragma unroll
    for (int t = 0; t < kHpRows; ++t) {
      if (t >= nt) break;
#pragma unroll
      for (int o = Q; o < 64; o <<= 1)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[t][c] += __shfl_xor(acc[t][c], o, 64);
      if (lane < Q) *reinterpret_cast<float4*>(sums + (wave * kHpRows + t) * 4 * Q + 4 * lane) = make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
    }
    __syncthreads();
    static_assert(kHpRows * Q <= 256, "a thread a row and quad");
    const int t = tid / Q;
    if (t < nt && n < P.N) {
      float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float4 s = *reinterpret_cast<const float4*>(sums + (u * kHpRows + t) * 4 * Q + 4 * (tid % Q));
        v[0] += s.x, v[1] += s.y, v[2] += s.z, v[3] += s.w;
      }
      const long row = t0 + t;
      if (P.gate != nullptr) {
        const float g = sigmoidf_(ld((const TO*)P.gate, row * P.gate_t + h));
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] *= g;
      }
      TO* y = (TO*)P.y + row * P.y_t + h * P.y_h + n;
      if constexpr (sizeof(TO) == 2)
        *reinterpret_cast<uint2*>(y) = make_uint2(ft::pack2(v[0], v[1]), ft::pack2(v[2], v[3]));
      else
        *reinterpret_cast<float4*>(y) = make_float4(v[0], v[1], v[2], v[3]);
    }
    if (t0 + kHpRows < P.rows) __syncthreads();
  }
}

template <typename TX, typename TO, bool ROPE>
static int launch_head_product(const HeadProduct& P, hipStream_t s) {
  const size_t lds = (size_t)(kHpRows * P.K) * sizeof(float);
  if ((long)P.heads * (P.N / 64) >= 128)
    hipLaunchKernelGGL((head_product_kernel<16, TX, TO, ROPE>), dim3((P.N + 63) / 64 + ROPE, P.heads), dim3(256),
                       lds + 4 * kHpRows * 64 * sizeof(float), s, P);
  else
    hipLaunchKernelGGL((head_product_kernel<4, TX, TO, ROPE>), dim3((P.N + 15) / 16 + ROPE, P.heads), dim3(256),
                       lds + 4 * kHpRows * 16 * sizeof(float), s, P);
  return (int)hipGetLastError();
}

}  // namespace mx

using namespace mx;

// K in whole eights up to 1024 (a block of rows in LDS), N in whole fours
extern "C" int mx_head_product_fits(int K, int N) { return K >= 8 && K % 8 == 0 && K <= 1024 && N >= 4 && N % 4 == 0; }

// qa [heads][rows][N] = q's first K of a head times wuk; qr [rows][heads][dr]: its other dr rotated.  q bf16 or fp32, heads
// K + dr apart
extern "C" int mx_latent_q_absorb(float* qa, float* qr, const void* q, int bf16, long stride, const float* wuk, const float* table,
                                  int table_rows, int dims, const int* positions, int rows, int heads, int K, int N, int dr,
                                  int interleaved, hipStream_t s) {
  if (rows <= 0) return 0;
  const int es = bf16 ? 2 : 4;
  if (!mx_head_product_fits(K, N) || heads < 1 || heads > 65535 || stride % 4 || (K + dr) % 4) return -1;
  if (((uintptr_t)wuk | (uintptr_t)qa) % 16 || ((uintptr_t)q) % (4 * es)) return -2;
  const HeadProduct P{wuk, K, N, rows, heads, q, stride, K + dr, qa, N, (long)rows * N, nullptr, 0, qr, table, positions,
                      table_rows, dims, dr, interleaved};
  if (bf16) return launch_head_product<bf16_t, float, true>(P, s);
  return launch_head_product<float, float, true>(P, s);
}

// out [rows][heads * N] = o [heads][rows][K] times wuv per head, times sigmoid(gate[t, h]) if there is a gate (of out's type)
extern "C" int mx_head_values(void* out, int out_bf16, const float* o, const float* wuv, const void* gate, long gate_stride,
                              int rows, int heads, int K, int N, hipStream_t s) {
  if (rows <= 0) return 0;
  if (!mx_head_product_fits(K, N) || heads < 1 || heads > 65535) return -1;
  if (((uintptr_t)wuv | (uintptr_t)o) % 16 || ((uintptr_t)out) % (out_bf16 ? 8 : 16)) return -2;
  const HeadProduct P{wuv, K, N, rows, heads, o, K, (long)rows * K, out, (long)heads * N, N, gate, gate_stride, nullptr, nullptr,
                      nullptr, 0, 0, 0, 0};
  if (out_bf16) return launch_head_product<float, bf16_t, false>(P, s);
  return launch_head_product<float, float, false>(P, s);
}

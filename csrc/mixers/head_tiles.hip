// Products of many rows with a matrix per head whose values are bf16 ones (a checkpoint's): q W_uk with the rotation of the
// queries' other part, and o W_uv, gated and rounded, as rows.  fp32 results and rows are kept at their precision on the bf16
// matrix units: a bf16 row times a bf16 weight is exact in fp32, an fp32 row goes as three bf16 parts (24 bits).
// A wave owns 32 rows and 32 C columns of one head.  The matrix is laid out once per wave's load (a step of 32 along K and 16
// columns are 1 KB in a row), rows are read where they lie; no LDS and no barrier but in the sum of SPLIT, where few rows leave
// most of the chip idle and a workgroup's four waves share K instead of owning rows each.
// Bound by memory, the results of the first and the rows of the second product (4 bytes of rank 512 a row and head): 4096 rows of 16
// heads, 128 -> 512 with the rotation in 44 us (4.0 TB/s; the library's fp32 product and the rotation's launch 104, the same stores
// in 64-byte pieces 48), 512 -> 128 with gate and rows in 34 us (4.4 TB/s; the library's, the gate's and the rows' launch 105), on their own
// buffers again and again; in a model's pass, from and to memory that others have used since, 67 and 45.
// Error against 64 bits 6.0e-8 and 2.4e-7 (library 7.3e-8 and 4.1e-7), SPLIT 4.8e-8 and 8.4e-8 (head_product.hip 4.9e-8, 9.7e-8).
#include "mx_common.h"

namespace mx {

typedef __attribute__((ext_vector_type(8))) __bf16 ht_bf16x8;
typedef __attribute__((ext_vector_type(4))) float ht_f32x4;

struct HeadTiles {
  const uint4* w;                // [heads][N / 32][K / 32][2][64]: ht_weight's order
  int K, N, rows, heads;
  const void* x;                 // x[t * x_t + h * x_h + k]
  long x_t, x_h;
  void* y;                       // y[t * y_t + h * y_h + n]
  long y_t, y_h;
  const void* gate;              // y times sigmoid(gate[t * gate_t + h]), or null
  long gate_t;
  // ROPE: x's rows are [K | dr]; the rotated dr -> qr [rows][heads][dr], by the workgroups from rope_from on
  float* qr;
  const float* table;
  const int* positions;
  int table_rows, dims, dr, interleaved;
  int chunks, row_tiles, rope_from;
};

__device__ __forceinline__ void ht_mfma(ht_f32x4& c, const uint4& a, const uint4& b) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ht_bf16x8, a), __builtin_bit_cast(ht_bf16x8, b), c, 0, 0, 0);
}

// a lane's 8 entries of a row
template <typename T> struct HtRow;
template <> struct HtRow<bf16_t> {
  static constexpr int kParts = 1;
  uint4 u;
  __device__ __forceinline__ void load(const bf16_t* p) { u = *reinterpret_cast<const uint4*>(p); }
  __device__ __forceinline__ void parts(uint4 (&o)[1]) const { o[0] = u; }
};
template <> struct HtRow<float> {
  static constexpr int kParts = 3;
  float4 u, v;
  __device__ __forceinline__ void load(const float* p) {
    u = *reinterpret_cast<const float4*>(p);
    v = *reinterpret_cast<const float4*>(p + 4);
  }
  __device__ __forceinline__ void parts(uint4 (&o)[3]) const {
    split_any_bf16x3(u.x, u.y, o[0].x, o[1].x, o[2].x);
    split_any_bf16x3(u.z, u.w, o[0].y, o[1].y, o[2].y);
    split_any_bf16x3(v.x, v.y, o[0].z, o[1].z, o[2].z);
    split_any_bf16x3(v.z, v.w, o[0].w, o[1].w, o[2].w);
  }
};

constexpr int kHtRows = 32;      // rows of a wave: two tiles
constexpr int kHtCols = 4;        // pairs of tiles of columns of a wave, but 1 of SPLIT
constexpr int kHtXcds = 8;
constexpr int kHtRopeHeads = 4;

template <int C, bool SPLIT, typename TX, typename TO, bool ROPE>
__global__ void __launch_bounds__(256, SPLIT ? 4 : 2)
head_tiles_kernel(HeadTiles P) {
  constexpr bool kRows = !SPLIT && sizeof(TO) == 4;        // results leave through LDS, whole pieces of a row at once
  constexpr int kPitch = 32 * C + 4;
  __shared__ __attribute__((aligned(16))) float sums[SPLIT ? 4 * C * 16 * 64 : kRows ? 4 * 16 * kPitch : 4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, hi = lane >> 4, lo = lane & 15;
  if (ROPE && (int)blockIdx.x >= P.rope_from) {
    // a wave the heads of a row, up to kHtRopeHeads: its lanes' angles are loaded once
    const int groups = (P.heads + kHtRopeHeads - 1) / kHtRopeHeads, u = ((int)blockIdx.x - P.rope_from) * 4 + wave;
    const int t = u / groups, h0 = u % groups * kHtRopeHeads, h1 = min(h0 + kHtRopeHeads, P.heads);
    if (t >= P.rows) return;
    int p = P.positions[t];
    p = p < 0 ? 0 : (p >= P.table_rows ? P.table_rows - 1 : p);
    const TX* xr = (const TX*)P.x + t * P.x_t + P.K;
    float* out = P.qr + (long)t * P.heads * P.dr;
    for (int j = lane; j < P.dr; j += 64) {
#pragma unroll 4
      for (int h = h0; h < h1; ++h)
        out[h * P.dr + j] = j < P.dims ? rope_at(xr + h * P.x_h, j, P.dims, P.table + (long)p * P.dims, P.interleaved)
                                       : ld(xr + h * P.x_h, j);
    }
    return;
  }
  // the workgroups of one tile of rows lie eight apart: they read the same rows through the same L2
  const int b = blockIdx.x, chunk = (b / kHtXcds) % P.chunks, unit = b % kHtXcds + b / (kHtXcds * P.chunks) * kHtXcds;
  if (unit >= P.row_tiles * P.heads) return;
  const int h = unit / P.row_tiles, t0 = (unit % P.row_tiles * (SPLIT ? 1 : 4) + (SPLIT ? 0 : wave)) * kHtRows;
  if (!SPLIT && t0 >= P.rows) return;
  const int steps = P.K / 32, pairs = P.N / 32, p0 = chunk * C;
  const TX* x[2];
#pragma unroll
  for (int r = 0; r < 2; ++r) x[r] = (const TX*)P.x + (long)min(t0 + 16 * r + lo, P.rows - 1) * P.x_t + h * P.x_h + 8 * hi;
  const uint4* w[C];
#pragma unroll
  for (int c = 0; c < C; ++c) w[c] = P.w + ((long)h * pairs + min(p0 + c, pairs - 1)) * steps * 128 + lane;
  constexpr int kParts = HtRow<TX>::kParts;
  struct Step { HtRow<TX> x[2]; uint4 w[C][2]; };
  auto fetch = [&](Step& s, int k) {
#pragma unroll
    for (int r = 0; r < 2; ++r) s.x[r].load(x[r] + 32 * k);
#pragma unroll
    for (int c = 0; c < C; ++c) s.w[c][0] = w[c][k * 128], s.w[c][1] = w[c][k * 128 + 64];
  };
  // (four sums are nearer than one; of the other form's they cost the registers of its second wave: 52 us instead of 44)
  constexpr int kSums = SPLIT ? 4 : 1;
  ht_f32x4 sum[kSums][2][C][2] = {}, (&acc)[2][C][2] = sum[0];
  const int first = SPLIT ? wave : 0;
  constexpr int kStride = SPLIT ? 4 : 1, kUnroll = SPLIT ? 4 : 2;
  if (first < steps) {
    Step cur, next;
    fetch(cur, first);
    for (int k = first; k < steps; k += kStride * kUnroll) {
#pragma unroll
      for (int i = 0; i < kUnroll; ++i) {
        if (i > 0 && k + kStride * i >= steps) break;
        fetch(next, min(k + kStride * (i + 1), steps - 1));
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          uint4 part[kParts];
          cur.x[r].parts(part);
#pragma unroll
          for (int q = kParts - 1; q >= 0; --q)           // the smallest first
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
              for (int j = 0; j < 2; ++j) ht_mfma(sum[i % kSums][r][c][j], cur.w[c][j], part[q]);
        }
        cur = next;
      }
    }
  }
  if constexpr (SPLIT)
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[r][c][j] = (sum[0][r][c][j] + sum[1][r][c][j]) + (sum[2][r][c][j] + sum[3][r][c][j]);
  if constexpr (SPLIT) {
    // [wave][value][lane]; wave u then adds and stores the values of tile r = u / 2, its columns' tile j = u % 2
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) sums[((wave * 4 + r * 2 + j) * C * 4 + c * 4 + e) * 64 + lane] = acc[r][c][j][e];
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    if (SPLIT && r != wave >> 1) continue;
    const long t = t0 + 16 * r + lo;
    if (!kRows && t >= P.rows) continue;
    const float g = P.gate != nullptr && t < P.rows ? sigmoidf_(ld((const TO*)P.gate, t * P.gate_t + h)) : 1.0f;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if (p0 + c >= pairs) break;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (SPLIT && j != (wave & 1)) continue;
        ht_f32x4 v;
        if constexpr (SPLIT) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float* s = sums + ((r * 2 + j) * C * 4 + c * 4 + e) * 64 + lane;
            constexpr int kWave = 4 * C * 4 * 64;
            v[e] = (s[0] + s[kWave]) + (s[2 * kWave] + s[3 * kWave]);
          }
        } else {
          v = acc[r][c][j];
        }
        if (P.gate != nullptr) v *= g;
        if constexpr (kRows) {
          *reinterpret_cast<float4*>(sums + (wave * 16 + lo) * kPitch + 32 * c + 16 * j + 4 * hi) = make_float4(v[0], v[1], v[2], v[3]);
          continue;
        }
        TO* y = (TO*)P.y + t * P.y_t + h * P.y_h + (p0 + c) * 32 + 16 * j + 4 * hi;
        if constexpr (sizeof(TO) == 2)
          *reinterpret_cast<uint2*>(y) = make_uint2(ft::pack2(v[0], v[1]), ft::pack2(v[2], v[3]));
        else
          *reinterpret_cast<float4*>(y) = make_float4(v[0], v[1], v[2], v[3]);
      }
    }
    if constexpr (kRows) {
      wave_lds_fence();
      constexpr int kQuads = 8 * C;
#pragma unroll
      for (int i = 0; i < 16 * kQuads / 64; ++i) {
        const int e = 64 * i + lane, row = e / kQuads, n = p0 * 32 + e % kQuads * 4;
        if (t0 + 16 * r + row < P.rows && n < P.N)
          *reinterpret_cast<float4*>((float*)P.y + (long)(t0 + 16 * r + row) * P.y_t + h * P.y_h + n) =
              *reinterpret_cast<const float4*>(sums + (wave * 16 + row) * kPitch + e % kQuads * 4);
      }
      wave_lds_fence();
    }
  }
}

template <typename TX, typename TO, bool ROPE>
static int launch_head_tiles(HeadTiles P, hipStream_t s) {
  // SPLIT while its workgroups, of 32 rows and 32 columns, make two rounds over the chip's CUs, four where K is long enough to hide
  // one another's loads: 100 rows of 16 heads 128 -> 512 (1024 of them) 7.7 us so and 6.0 in whole tiles, 64 rows (512) 4.9 and 4.8;
  // 512 -> 128, 300 rows (640) 11.2 and 16, 777 (1600) 22.9 and 20.9, of 128 heads 64 rows (1024) 14.9 and 19.5.  Up to 16 rows
  // always, for its sums.
  const long parts = (long)((P.rows + kHtRows - 1) / kHtRows) * P.heads * (P.N / 32);
  const bool split = P.rows <= 16 || parts <= (P.K >= 256 ? 1024 : 512);
  const int cols = 32 * (split ? 1 : kHtCols), rows = split ? kHtRows : 4 * kHtRows;
  P.chunks = (P.N + cols - 1) / cols;
  P.row_tiles = (P.rows + rows - 1) / rows;
  const long units = ((long)P.row_tiles * P.heads + kHtXcds - 1) / kHtXcds * kHtXcds * P.chunks;
  const long rope = ROPE ? ((long)P.rows * ((P.heads + kHtRopeHeads - 1) / kHtRopeHeads) + 3) / 4 : 0;
  if (units + rope > 0x7fffffffL) return -1;
  P.rope_from = (int)units;
  const dim3 grid((unsigned)(units + rope));
  if (split)
    hipLaunchKernelGGL((head_tiles_kernel<1, true, TX, TO, ROPE>), grid, dim3(256), 0, s, P);
  else
    hipLaunchKernelGGL((head_tiles_kernel<kHtCols, false, TX, TO, ROPE>), grid, dim3(256), 0, s, P);
  return (int)hipGetLastError();
}

}  // namespace mx

using namespace mx;

// K and N in whole steps and pairs of tiles
extern "C" int mx_head_tiles_fits(int K, int N) { return K >= 32 && K % 32 == 0 && N >= 32 && N % 32 == 0; }

// mx_latent_q_absorb for wuk in bf16 and the order of HeadTiles::w; q's rows and heads at multiples of 16 bytes
extern "C" int mx_latent_q_tiles(float* qa, float* qr, const void* q, int bf16, long stride, const void* wuk, const float* table,
                                 int table_rows, int dims, const int* positions, int rows, int heads, int K, int N, int dr,
                                 int interleaved, hipStream_t s) {
  if (rows <= 0) return 0;
  const int in16 = bf16 ? 8 : 4;
  if (!mx_head_tiles_fits(K, N) || heads < 1 || stride % in16 || (K + dr) % in16) return -1;
  if (((uintptr_t)wuk | (uintptr_t)qa | (uintptr_t)q) % 16) return -2;
  const HeadTiles P{(const uint4*)wuk, K, N, rows, heads, q, stride, K + dr, qa, N, (long)rows * N, nullptr, 0, qr, table, positions,
                    table_rows, dims, dr, interleaved, 0, 0, 0};
  if (bf16) return launch_head_tiles<bf16_t, float, true>(P, s);
  return launch_head_tiles<float, float, true>(P, s);
}

// mx_head_values for wuv in bf16 and the order of HeadTiles::w
extern "C" int mx_head_values_tiles(void* out, int out_bf16, const float* o, const void* wuv, const void* gate, long gate_stride,
                                    int rows, int heads, int K, int N, hipStream_t s) {
  if (rows <= 0) return 0;
  if (!mx_head_tiles_fits(K, N) || heads < 1) return -1;
  if (((uintptr_t)wuv | (uintptr_t)o) % 16 || ((uintptr_t)out) % (out_bf16 ? 8 : 16)) return -2;
  const HeadTiles P{(const uint4*)wuv, K, N, rows, heads, o, K, (long)rows * K, out, (long)heads * N, N, gate, gate_stride, nullptr,
                    nullptr, nullptr, 0, 0, 0, 0, 0, 0, 0};
  if (out_bf16) return launch_head_tiles<float, bf16_t, false>(P, s);
  return launch_head_tiles<float, float, false>(P, s);
}

// Latent attention of decode rows and short segments over the paged bf16 cache of [c (512) | rotated key (64)]:
// the split-key form (latent_attn.hip latent_split_kernel, any sizes) on the matrix units.
//
// fp32 queries and weights stay fp32: each is the exact sum of three bf16 parts, the cache is bf16 already, so
// three v_mfma_f32_16x16x32_bf16 per operand pair form the products of an fp32 multiply, summed in fp32.
//
// A workgroup of eight waves owns one row, up to 16 heads (one tile of the products) and one slice of its
// keys, 64 at a time through LDS.  Scores: a wave takes 32 keys and a quarter of the 576 dimensions (so the
// queries are split once per workgroup), partial sums meet in LDS, where four waves turn 16 keys each into
// weights; sums: a wave takes 64 columns.  The slices' (maximum, sum, sums) are merged by the caller's kernel.
// Bound by the chain of one slice (load, scores, softmax, sums) up to a few rows, by the read of the rows beyond.
// 16 heads, with the merge: 3 rows of 500 keys 16 us, of 4000 26; 8 rows of 1000 20; 64 rows of 2000 50 (147 MB:
// 2.9 TB/s).  The general kernel, multiplying on the vector units: 47, 257, 78, 505.
#include "latent_tile.h"

namespace mx {

constexpr int kLdKeys = 64;

__global__ void __launch_bounds__(512, 1)
latent_decode_kernel(float* __restrict__ ws_acc, float* __restrict__ ws_ml, const float* __restrict__ qa,
                     const float* __restrict__ qr, const bf16_t* __restrict__ cache, const int* __restrict__ start,
                     const int* __restrict__ pos0, const int* __restrict__ kv_len, const int* __restrict__ bt,
                     int bt_stride, int heads, long total_rows, int block_size, int num_blocks, float scale,
                     int skip_from, int splits) {
  __shared__ __attribute__((aligned(1024))) uint8_t tiles[2 * kLpTile];
  __shared__ __attribute__((aligned(16))) float4 part[4][4][64];            // [dimensions][key tile][lane]
  __shared__ __attribute__((aligned(16))) uint32_t wts[2][3][64][4];        // [32 keys][part][lane]
  __shared__ float tile_max[4][16], tile_sum[4][16];
  const int s = blockIdx.z;
  const int r0 = start[s], n_rows = start[s + 1] - r0, rel = blockIdx.y;
  if (rel >= n_rows || (skip_from > 0 && n_rows >= skip_from)) return;
  const long row = r0 + rel;
  const int sp = blockIdx.x % splits, h0 = (blockIdx.x / splits) * 16;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g4 = lane >> 4;
  const int head = min(h0 + n, heads - 1);
  const bool live = h0 + n < heads;
  const int nk = min(pos0[s] + rel + 1, kv_len[s]);
  const int per = (nk + splits - 1) / splits, chunk = (per + kLdKeys - 1) / kLdKeys * kLdKeys;
  const int k_begin = sp * chunk, k_end = min(nk, k_begin + chunk);
  const long base = (row * splits + sp) * heads + h0 + n;
  if (k_begin >= k_end) {                     // no key: weight zero, the sums are not read
    if (wave == 0 && g4 == 0 && live) ws_ml[base * 2] = -INFINITY, ws_ml[base * 2 + 1] = 0.f;
    return;
  }
  const int* tab = bt + (long)s * bt_stride;
  const uint32_t lds0 = ft::lds_off(tiles);
  auto issue = [&](int k0) {                  // this wave's eight keys (past the last: repeated, weight zero)
    const int key = min(k0 + 8 * wave + (lane >> 3), k_end - 1);
    int blk = tab[key / block_size];
    if (blk < 0 || blk >= num_blocks) blk = 0;
    lp_issue(cache + ((long)blk * block_size + key % block_size) * kLpWidth, wave & 3, lane,
             lds0 + (wave >> 2) * kLpTile);
  };

  // this wave's share of the queries: 32-dimension steps s0 .. s0 + steps - 1 of 18
  constexpr int KS = kLpWidth / 32, QS = (KS + 3) / 4;
  const int dq = wave & 3, kh = wave >> 2, s0 = dq < 2 ? QS * dq : 2 * QS + (QS - 1) * (dq - 2), steps = dq < 2 ? QS : QS - 1;
  static_assert(2 * QS + 2 * (QS - 1) == KS, "queries' shares");
  float4 qf[QS][2];
  const float* a = qa + ((long)head * total_rows + row) * kLpRank;
  const float* r = qr + (row * heads + head) * kLpRot;
#pragma unroll
  for (int i = 0; i < QS; ++i) {
    const int d = 32 * (s0 + min(i, steps - 1)) + 8 * g4;
    const float* src = d < kLpRank ? a + d : r + (d - kLpRank);
    qf[i][0] = *reinterpret_cast<const float4*>(src);
    qf[i][1] = *reinterpret_cast<const float4*>(src + 4);
  }
  issue(k_begin);
  uint4 q[QS][3];
#pragma unroll
  for (int i = 0; i < QS; ++i) {
    const float4 x = qf[i][0], y = qf[i][1];
    split_bf16x3(x.x, x.y, q[i][0].x, q[i][1].x, q[i][2].x);
    split_bf16x3(x.z, x.w, q[i][0].y, q[i][1].y, q[i][2].y);
    split_bf16x3(y.x, y.y, q[i][0].z, q[i][1].z, q[i][2].z);
    split_bf16x3(y.z, y.w, q[i][0].w, q[i][1].w, q[i][2].w);
  }
  int k_off[2], v_off[4];
  lp_offsets(n, g4, k_off, v_off);

  float m = -INFINITY, l = 0.f;               // of head n, alike in all waves and lane groups
  lp_f32x4 o[4];                              // columns 64 wave + 16 u + 4 g4 .. of head n
#pragma unroll
  for (int u = 0; u < 4; ++u) o[u] = lp_f32x4{0.f, 0.f, 0.f, 0.f};

  for (int k0 = k_begin; k0 < k_end; k0 += kLdKeys) {
    ft::vm_wait<0>();
    __syncthreads();
    const uint8_t* tile = tiles + kh * kLpTile;
    lp_f32x4 sc[2][3];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int p = 0; p < 3; ++p) sc[i][p] = lp_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < QS; ++j) {
      if (j >= steps) break;
      const int ks = s0 + j;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint4 k = *reinterpret_cast<const uint4*>(tile + (ks >> 1) * 4096 + i * 2048 + (ks & 1 ? k_off[1] : k_off[0]));
#pragma unroll
        for (int p = 0; p < 3; ++p) sc[i][p] = lp_mfma(k, q[j][p], sc[i][p]);
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const lp_f32x4 v = sc[i][2] + sc[i][1] + sc[i][0];
      part[dq][2 * kh + i][lane] = make_float4(v[0], v[1], v[2], v[3]);
    }
    __syncthreads();
    float x[4];
    if (wave < 4) {                           // keys 16 wave + 4 g4 .. of head n
      float top = -INFINITY;
      float4 v = part[0][wave][lane];
      x[0] = v.x, x[1] = v.y, x[2] = v.z, x[3] = v.w;
#pragma unroll
      for (int d = 1; d < 4; ++d) {
        v = part[d][wave][lane];
        x[0] += v.x, x[1] += v.y, x[2] += v.z, x[3] += v.w;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = k0 + 16 * wave + 4 * g4 + e < k_end ? x[e] * scale : -INFINITY;
        top = fmaxf(top, x[e]);
      }
      top = ft::kgroups_max(top);
      if (g4 == 0) tile_max[wave][n] = top;
    }
    __syncthreads();
    const float mn = fmaxf(fmaxf(m, fmaxf(tile_max[0][n], tile_max[1][n])), fmaxf(tile_max[2][n], tile_max[3][n]));
    const float mu = mn == -INFINITY ? 0.f : mn;      // (scores of -inf, sums that overflow, have weight 0, also alone)
    const float alpha = expf(m - mu);         // 0 at the first tile (m = -inf)
    if (wave < 4) {
      float sum = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = expf(x[e] - mu);               // exp(-inf) = 0 for the masked keys
        sum += x[e];
      }
      uint2 hi, mid, lo;
      split_bf16x3(x[0], x[1], hi.x, mid.x, lo.x);
      split_bf16x3(x[2], x[3], hi.y, mid.y, lo.y);
      *reinterpret_cast<uint2*>(&wts[wave >> 1][0][lane][2 * (wave & 1)]) = hi;
      *reinterpret_cast<uint2*>(&wts[wave >> 1][1][lane][2 * (wave & 1)]) = mid;
      *reinterpret_cast<uint2*>(&wts[wave >> 1][2][lane][2 * (wave & 1)]) = lo;
      sum = ft::kgroups_sum(sum);
      if (g4 == 0) tile_sum[wave][n] = sum;
    }
    __syncthreads();
    l = l * alpha + ((tile_sum[0][n] + tile_sum[1][n]) + (tile_sum[2][n] + tile_sum[3][n]));
    m = mn;
#pragma unroll
    for (int u = 0; u < 4; ++u) o[u] *= alpha;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint4 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = lp_values(tiles + h * kLpTile, 4 * wave + u, v_off);
#pragma unroll
      for (int p = 2; p >= 0; --p) {
        const uint4 w = *reinterpret_cast<const uint4*>(wts[h][p][lane]);
#pragma unroll
        for (int u = 0; u < 4; ++u) o[u] = lp_mfma(v[u], w, o[u]);
      }
    }
    if (k0 + kLdKeys < k_end) {
      __syncthreads();                        // the tile is no longer read
      issue(k0 + kLdKeys);
    }
  }
  if (!live) return;
#pragma unroll
  for (int u = 0; u < 4; ++u)
    *reinterpret_cast<float4*>(ws_acc + base * kLpRank + 64 * wave + 16 * u + 4 * g4) = make_float4(o[u][0], o[u][1], o[u][2], o[u][3]);
  if (wave == 0 && g4 == 0) ws_ml[base * 2] = m, ws_ml[base * 2 + 1] = l;
}

}  // namespace mx

using namespace mx;

extern "C" int mx_latent_decode_fits(int rank, int dr, int cache_bf16) {
  return rank == kLpRank && dr == kLpRot && cache_bf16;
}

// the slices of mx_latent_attention_split (checked there) for sizes that fit
extern "C" int mx_latent_decode(float* ws_acc, float* ws_ml, const float* qa, const float* qr, const void* cache,
                                const int* start, const int* pos0, const int* kv_len, const int* bt, int bt_stride,
                                int num_segs, int max_rows, int heads, long total_rows, int block_size, int num_blocks,
                                float scale, int skip_from, int splits, hipStream_t s) {
  const dim3 grid(splits * ((heads + 15) / 16), max_rows, num_segs);
  hipLaunchKernelGGL(latent_decode_kernel, grid, dim3(512), 0, s, ws_acc, ws_ml, qa, qr, (const bf16_t*)cache, start,
                     pos0, kv_len, bt, bt_stride, heads, total_rows, block_size, num_blocks, scale, skip_from, splits);
  return (int)hipGetLastError();
}

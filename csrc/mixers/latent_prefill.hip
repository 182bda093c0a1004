// Latent attention of long row segments (prefill chunks) over the paged bf16 cache of [c (512) | rotated key
// (64)], in one pass: scores, causal softmax (optionally with a learned number per head in the denominator)
// and weighted sums of the c parts, no scores in memory.
//
// Numbers as in the two products of the general path: queries and weights rounded to bf16, cache rows bf16
// as they are, fp32 sums, fp32 softmax statistics.
//
// Shape of the work: all heads share the cached rows, so a segment is rows x heads pairs; a workgroup of
// four waves owns 128 consecutive pairs (heads fastest), a wave 32 of them with their queries and
// sums (256 registers) resident, one wave per SIMD.  Everything is transposed: S^T = K Q^T and
// O^T = C^T P^T on v_mfma_f32_16x16x32_bf16, a column per pair, so the first product's result is the second
// one's operand with no exchange between lanes.  Tiles of 32 keys go to LDS by global_load_lds_dwordx4 into
// a ring of four, two in flight; both products read the same rows, the second one through
// ds_read_b64_tr_b16.
// The running maximum is a reference: it moves (and the sums are rescaled) only when a score exceeds it by a
// factor of 2^8, so the weights stay within fp32 and bf16 range and their relative rounding is the same.
//
// The chain of one wave per SIMD is hidden by order: a tile's weights are computed under the next tile's
// scores and its sums run over the next tile's exponents (without that 380 us for the first size below).
// Nearly all sums are in accumulation registers, the rest in vector ones; a ninth of the queries stays in LDS,
// the registers are full.
//
// 16 heads, from position 0: 4096 rows 305 us (0.95 PFLOP/s, of 1.46 for a large product; what is left is the
// wait at each tile's barrier), 2048 rows 141, 777 rows 70, 300 rows 41.  Two products through memory with a
// softmax kernel between them: 1360, 428, 126, 93 us and 9 launches per segment.
#include "latent_tile.h"

namespace mx {

constexpr int kLpPairs = 128, kLpSlots = 4;
constexpr int kLpInReg = 16;                          // query steps of 32 in registers, the rest in LDS
constexpr int kLpAhead = 3;

struct LatPreArgs {
  float* out;
  const float *qa, *qr;
  const bf16_t* cache;
  const int *start, *pos0, *kv_len, *bt;
  int bt_stride, num_segs, heads;
  long total_rows;
  int page_shift, num_blocks, min_rows;
  float scale;
  const float* sink;
};

// d += a b with d in the accumulation registers (the compiler's own choice is one kind of register for every
// product of a kernel, and a wave's sums alone take 256).  The wait states cover operands that a vector
// instruction has just written.
__device__ __forceinline__ void lp_mfma_acc(lp_f32x4& d, const uint4& a, const uint4& b) {
  asm("s_nop 1\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
      : "+a"(d)
      : "v"(__builtin_bit_cast(lp_bf16x8, a)), "v"(__builtin_bit_cast(lp_bf16x8, b)));
}
// ... and before d is read by anything else
__device__ __forceinline__ void lp_acc_done(lp_f32x4& d) { asm volatile("s_nop 15" : "+a"(d)); }

__device__ __forceinline__ void lp_acc_scale(lp_f32x4& d, float f) {
  lp_acc_done(d);
  float x = d[0], y = d[1], z = d[2], w = d[3];
  x *= f, y *= f, z *= f, w *= f;
  d = lp_f32x4{x, y, z, w};
  asm volatile("" : "+a"(d));
}

__global__ void __launch_bounds__(256, 1)
latent_prefill_kernel(LatPreArgs A) {
  constexpr int KS = kLpWidth / 32, CT = kLpRank / 16, QL = KS - kLpInReg, CA = 30;
  __shared__ __attribute__((aligned(1024))) uint8_t ring[kLpSlots * kLpTile];
  __shared__ __attribute__((aligned(16))) uint4 q_lds[4 * 2 * QL * 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g4 = lane >> 4;
  int seg, block;
  if (!segment_block(A.start, A.num_segs, A.min_rows, A.heads, kLpPairs, blockIdx.x, seg, block)) return;
  seg = __builtin_amdgcn_readfirstlane(seg);
  block = __builtin_amdgcn_readfirstlane(block);
  const int r0 = A.start[seg], rows = A.start[seg + 1] - r0, p0 = A.pos0[seg], kv = A.kv_len[seg];
  const int pairs = rows * A.heads, m0 = block * kLpPairs;
  const int* table = A.bt + (long)seg * A.bt_stride;

  // this lane's two pairs: queries (bf16) and number of keys
  uint4 q[2][kLpInReg], *q_rest = q_lds + wave * 2 * QL * 64 + lane;
  int nk[2], row[2], head[2];
  bool live[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int m = m0 + wave * 32 + p * 16 + n;
    live[p] = m < pairs;
    const int mc = min(m, pairs - 1);
    row[p] = mc / A.heads;
    head[p] = mc - row[p] * A.heads;
    nk[p] = min(p0 + row[p] + 1, kv);
    const float* a = A.qa + ((long)head[p] * A.total_rows + r0 + row[p]) * kLpRank;
    const float* r = A.qr + ((long)(r0 + row[p]) * A.heads + head[p]) * kLpRot;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const float* src = s < kLpRank / 32 ? a + 32 * s + 8 * g4 : r + 32 * (s - kLpRank / 32) + 8 * g4;
      const float4 x = *reinterpret_cast<const float4*>(src), y = *reinterpret_cast<const float4*>(src + 4);
      const uint4 v = make_uint4(ft::pack2(x.x, x.y), ft::pack2(x.z, x.w), ft::pack2(y.x, y.y), ft::pack2(y.z, y.w));
      if (s < kLpInReg) q[p][s] = v;
      else q_rest[(p * QL + s - kLpInReg) * 64] = v;         // (read by this lane alone)
    }
  }
  // keys of this workgroup (its last row sees most) and of this wave's first pair (which sees fewest)
  const int keys = min(p0 + min(m0 + kLpPairs - 1, pairs - 1) / A.heads + 1, kv);
  const int sure = min(p0 + min(m0 + wave * 32, pairs - 1) / A.heads + 1, kv);
  const int tiles = keys > 0 ? (keys + kLpKeys - 1) / kLpKeys : 0;

  lp_f32x4 o[2][CT];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int t = 0; t < CT; ++t) o[p][t] = lp_f32x4{0.f, 0.f, 0.f, 0.f};
  // (the reference starts below every score, but finite: scores of -inf, sums that overflow, have weight 0)
  float ref[2] = {-1e38f, -1e38f}, sum[2] = {0.f, 0.f};
  const float c = A.scale * 1.44269504f;

  // page ids, a lane each, of 64 pages from page0 on
  int page0 = 0;
  auto pages = [&](int from) {
    page0 = from;
    const int p = min(from + lane, (keys - 1) >> A.page_shift);
    int b = table[p];
    return b < 0 || b >= A.num_blocks ? 0 : b;
  };
  int ids = tiles > 0 ? pages(0) : 0;
  const uint32_t lds0 = ft::lds_off(ring);
  // this wave's eight keys of tile t -> its slot (keys past the last repeat it: finite, weight zero)
  auto issue = [&](int t) {
    const int k0 = t * kLpKeys + 8 * wave;
    const int page = min(k0, keys - 1) >> A.page_shift;
    if (page - page0 >= 64) ids = pages(page);
    const int key = min(k0 + (lane >> 3), keys - 1);
    const long at = ((long)__builtin_amdgcn_readlane(ids, page - page0) << A.page_shift) + (key & ((1 << A.page_shift) - 1));
    lp_issue(A.cache + at * kLpWidth, wave, lane, lds0 + (t % kLpSlots) * kLpTile);
  };
  for (int t = 0; t < 2 && t < tiles; ++t) issue(t);

  int k_off[2], v_off[4];
  lp_offsets(n, g4, k_off, v_off);

  lp_f32x4 s[2][2];                       // a tile's scores, [key tile][pair tile]
  float x[2][8], top;                     // exponents (base 2) relative to the reference, then weights
  uint32_t w[2][4];                       // weights in bf16
  uint4 ops[kLpAhead + 1][2], kq[2][2];   // operands read kLpAhead steps before their products
  auto slot = [&](int t) { return ring + (t % kLpSlots) * kLpTile; };
  auto arrive = [&](int t) {              // tile t is whole (younger: t + 1), and no wave still reads t - 2's slot
    if (t + 1 < tiles) ft::vm_wait<kLpDma>();
    else ft::vm_wait<0>();
    __syncthreads();
    if (t + 2 < tiles) issue(t + 2);
  };
  // S^T of a tile; `with` is run a step at a time under the products
  auto scores = [&](const uint8_t* tile, auto with) {
    auto k_read = [&](int ks) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
        ops[ks % (kLpAhead + 1)][i] = *reinterpret_cast<const uint4*>(tile + (ks >> 1) * 4096 + i * 2048 + k_off[ks & 1]);
    };
#pragma unroll
    for (int ks = 0; ks < kLpAhead; ++ks) k_read(ks);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int p = 0; p < 2; ++p) s[i][p] = lp_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (ks + 1 < KS && ks + 1 >= kLpInReg) {
#pragma unroll
        for (int p = 0; p < 2; ++p) kq[(ks + 1) & 1][p] = q_rest[(p * QL + ks + 1 - kLpInReg) * 64];
      }
      if (ks + kLpAhead < KS) k_read(ks + kLpAhead);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int p = 0; p < 2; ++p)
          s[i][p] = lp_mfma(ops[ks % (kLpAhead + 1)][i], ks < kLpInReg ? q[p][ks] : kq[ks & 1][p], s[i][p]);
      with(ks);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // O^T += C^T P^T of a tile, `with` likewise
  auto sums = [&](const uint8_t* tile, auto with) {
    auto v_read = [&](int step) {         // column tiles 2 step, 2 step + 1
#pragma unroll
      for (int d = 0; d < 2; ++d) ops[step % (kLpAhead + 1)][d] = lp_values(tile, 2 * step + d, v_off);
    };
#pragma unroll
    for (int step = 0; step < kLpAhead; ++step) v_read(step);
    __builtin_amdgcn_sched_barrier(0);
    const uint4 w4[2] = {make_uint4(w[0][0], w[0][1], w[0][2], w[0][3]), make_uint4(w[1][0], w[1][1], w[1][2], w[1][3])};
#pragma unroll
    for (int step = 0; step < CT / 2; ++step) {
      if (step + kLpAhead < CT / 2) v_read(step + kLpAhead);
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const int u = 2 * step + d;
          if (u < CA) lp_mfma_acc(o[p][u], ops[step % (kLpAhead + 1)][d], w4[p]);
          else o[p][u] = lp_mfma(ops[step % (kLpAhead + 1)][d], w4[p], o[p][u]);
        }
      with(step);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto exponents = [&](int e) {           // of key 16 (e / 4) + 4 g4 + e % 4
    if (e >= 8) return;
    if (e == 0) top = -INFINITY;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      x[p][e] = fmaf(s[e >> 2][p][e & 3], c, -ref[p]);
      top = fmaxf(top, x[p][e]);
    }
  };
  auto weights = [&](int e) {
    if (e >= 8) return;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      x[p][e] = __builtin_amdgcn_exp2f(x[p][e]);
      sum[p] += x[p][e];
      if (e & 1) w[p][e >> 1] = ft::pack2(x[p][e - 1], x[p][e]);
    }
  };
  // after a tile's exponents: the reference, if a score is far above it; keys a row does not see: none
  auto settle = [&](int k0) {
    if (__any(top > 8.f)) {
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        float mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (k0 + 16 * (e >> 2) + 4 * g4 + (e & 3) < nk[p]) mx = fmaxf(mx, s[e >> 2][p][e & 3] * c);
        const float to = fmaxf(ref[p], ft::kgroups_max(mx));
        const float f = to > ref[p] ? __builtin_amdgcn_exp2f(ref[p] - to) : 1.f;
        ref[p] = to;
        sum[p] *= f;
#pragma unroll
        for (int u = 0; u < CT; ++u) {
          if (u < CA) lp_acc_scale(o[p][u], f);
          else o[p][u] *= f;
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) x[p][e] = fmaf(s[e >> 2][p][e & 3], c, -ref[p]);
      }
    }
    if (k0 + kLpKeys > sure) {
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (k0 + 16 * (e >> 2) + 4 * g4 + (e & 3) >= nk[p]) x[p][e] = -INFINITY;
    }
  };
  const auto nothing = [](int) {};
  if (tiles > 0) {
    arrive(0);
    scores(slot(0), nothing);
#pragma unroll
    for (int e = 0; e < 8; ++e) exponents(e);
    settle(0);
    // a tile's weights under the next tile's scores, its sums over the next tile's exponents
    for (int t = 0; t + 1 < tiles; ++t) {
      arrive(t + 1);
      scores(slot(t + 1), weights);
      sums(slot(t), exponents);
      settle((t + 1) * kLpKeys);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) weights(e);
    sums(slot(tiles - 1), nothing);
  }
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    float l = ft::kgroups_sum(sum[p]), f = 1.f;
    if (A.sink != nullptr && nk[p] > 0) {             // one more term of the denominator
      const float sk = A.sink[head[p]] * 1.44269504f, to = fmaxf(ref[p], sk);
      f = __builtin_amdgcn_exp2f(ref[p] - to);
      l = l * f + __builtin_amdgcn_exp2f(sk - to);
    }
    f = l > 0.f ? f / l : (l == 0.f ? 0.f : l);       // (NaN stays)
    if (!live[p]) continue;
    float* dst = A.out + ((long)head[p] * A.total_rows + r0 + row[p]) * kLpRank + 4 * g4;
#pragma unroll
    for (int u = 0; u < CT; ++u) {
      if (u < CA) lp_acc_done(o[p][u]);
      *reinterpret_cast<float4*>(dst + 16 * u) = make_float4(o[p][u][0] * f, o[p][u][1] * f, o[p][u][2] * f, o[p][u][3] * f);
    }
  }
}

}  // namespace mx

using namespace mx;

// pages of at least 8 keys, a power of two: eight neighbouring keys lie in one page
extern "C" int mx_latent_prefill_fits(int rank, int dr, int block_size) {
  return rank == kLpRank && dr == kLpRot && block_size >= 8 && (block_size & (block_size - 1)) == 0;
}

// segments of at least min_rows rows (long_segs of them with long_rows rows); the others are left alone
extern "C" int mx_latent_prefill(float* out, const float* qa, const float* qr, const void* cache, const int* start,
                                 const int* pos0, const int* kv_len, const int* bt, int bt_stride, int num_segs,
                                 int long_segs, long long_rows, int heads, long total_rows, int rank, int dr,
                                 int block_size, int num_blocks, float scale, int min_rows, const float* sink,
                                 hipStream_t s) {
  if (num_segs <= 0 || long_segs <= 0 || long_rows <= 0) return 0;
  if (!mx_latent_prefill_fits(rank, dr, block_size) || heads < 1 || min_rows < 1) return -1;
  if (((uintptr_t)out) % 16 || ((uintptr_t)qa) % 16 || ((uintptr_t)qr) % 16 || ((uintptr_t)cache) % 16) return -2;
  if (long_rows * heads > 0x3fffffffL) return -3;
  const LatPreArgs A{out, qa, qr, (const bf16_t*)cache, start, pos0, kv_len, bt, bt_stride, num_segs, heads, total_rows,
                     __builtin_ctz((unsigned)block_size), num_blocks, min_rows, scale, sink};
  const long items = long_rows * heads / kLpPairs + long_segs;
  hipLaunchKernelGGL(latent_prefill_kernel, dim3((unsigned)items), dim3(256), 0, s, A);
  return (int)hipGetLastError();
}

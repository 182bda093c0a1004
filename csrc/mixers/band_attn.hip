// Attention of long row segments (prefill chunks) over paged bf16 keys and values, in one pass: the
// masks, score terms and weights of the windowed attentions (window_attn.hip) with scores and sums on
// the matrix units and no scores in memory.
//
// Exactness: queries and weights are fp32 and stay fp32.  An fp32 value is the sum of three bf16 parts
// (hi + mid + lo, 24 bits), keys and values are bf16 already, so three v_mfma_f32_16x16x32_bf16 per
// operand pair form the same products as an fp32 multiply, summed in fp32, smallest parts first.
//
// Shape of the work: a workgroup of WV waves owns one key head (and score map) and 16 WV consecutive
// (row, query head of the group) pairs of one segment, a wave 16 of them, so the tile of 64 keys that
// is staged in LDS serves all query heads that share it.  Everything is transposed: S^T = K Q^T and
// O^T = V^T P^T, a column per pair.  The result layout of the first product (lane (g, n): keys 4 g ..
// 4 g + 3 of pair n) is the operand layout of the second one, up to the order of the keys within 32,
// and V is staged in that order; a pair's maximum and sum need two lane swaps.  Keys and values of the
// next tile are loaded during the products of the current one.
//
// Bound by the vector units (per score: exponential, cap or bias, the three-way split) beside 96 MFMAs
// per 64 keys and wave.  16 heads of 128 on 4 key heads: 2048 rows causal 124 us (0.42 PFLOP/s of bf16
// products), 777 rows in blocks of 1024 38 us, with a distance table 56 us, five prompts of 200 to 542
// rows with a cap 47 us; two fp32 products through memory with a weights kernel between them, gathers
// and layout changes around them, took 400 to 550 us and 25 launches per segment.
#include "mx_common.h"

namespace mx {

typedef __bf16 ba_bf16x8 __attribute__((ext_vector_type(8)));
typedef float ba_f32x4 __attribute__((ext_vector_type(4)));

constexpr int kBandTile = 64;

struct BandArgs {
  void* out;                                  // fp32, or bf16 (rounded once, here)
  int out_bf16;
  const float* q;
  const bf16_t *kc, *vc;
  const int *start, *pos0, *kv_len, *bt;
  int bt_stride, num_segs, heads, maps, kv_heads, window;
  float scale;
  int sigmoid;
  const float *r1, *r2, *pb;
  int page_shift, num_blocks, min_rows;       // pages of 1 << page_shift keys
  float softcap;
  int has_sink;
  float sink_all;
  const float* sinks;
  int blocks, keep_first;
  const float* dist_bias;
  int nd;
};

__device__ __forceinline__ ba_f32x4 ba_mfma(const uint4& a, const uint4& b, ba_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ba_bf16x8, a), __builtin_bit_cast(ba_bf16x8, b), c,
                                                 0, 0, 0);
}

// e^x for x <= 0, the argument's rounding in base 2 made good; 0 far below; NaN stays NaN
__device__ __forceinline__ float ba_exp(float x) {
  x = x < -150.f ? -150.f : x;
  const float t = x * 1.44269502f;
  const float r = fmaf(x, 1.44269502f, -t) + x * 1.92596303e-8f;
  const float e = __builtin_amdgcn_exp2f(t);
  return fmaf(e, r * 0.693147181f, e);
}

// the score terms a kernel is built for (run-time tests per score cost as much as the products: a
// block-masked 777-row layer took 70 us with them)
enum { kBandPlain = 0, kBandCap = 1, kBandDist = 2, kBandSigmoid = 3, kBandAny = 4 };

template <int DK, int DV, int WV, int KIND>
__global__ void __launch_bounds__(64 * WV, 2)
band_attn_kernel(BandArgs A) {
  constexpr bool kAny = KIND == kBandAny;
  const bool use_cap = KIND == kBandCap || (kAny && A.softcap > 0.f);
  const bool use_terms = (KIND == kBandSigmoid || kAny) && A.r1 != nullptr;
  const bool use_dist = KIND == kBandDist || (kAny && A.dist_bias != nullptr);
  const bool sigmoid = KIND == kBandSigmoid || (kAny && A.sigmoid);
  constexpr int KS = DK / 32, DT = DV / 16, NTHR = 64 * WV;
  constexpr int KROW = DK + 8;                                   // bf16 per staged key
  constexpr int TASKS_K = 16 * (DK / 8), TASKS = TASKS_K + 16 * (DV / 8), NT = (TASKS + NTHR - 1) / NTHR;
  __shared__ __attribute__((aligned(16))) bf16_t Ks[kBandTile * KROW];
  __shared__ __attribute__((aligned(16))) bf16_t Vt[DV * kBandTile];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g4 = lane >> 4;
  const int rep = A.heads / A.kv_heads, gk = blockIdx.y, kvh = gk / A.maps, map = gk % A.maps;
  int seg, block;
  if (!segment_block(A.start, A.num_segs, A.min_rows, rep, 16 * WV, blockIdx.x, seg, block)) return;
  seg = __builtin_amdgcn_readfirstlane(seg);
  block = __builtin_amdgcn_readfirstlane(block);
  const int r0 = A.start[seg], rows = A.start[seg + 1] - r0, p0 = A.pos0[seg];
  const int pairs = rows * rep, m0 = block * 16 * WV;
  const int* table = A.bt + (long)seg * A.bt_stride;
  const int hq = A.heads * A.maps;
  const long nk = (long)A.kv_heads * A.maps * DK, nv = (long)A.kv_heads * DV;

  // this lane's pair
  const int m = m0 + 16 * wave + n, mc = min(m, pairs - 1);
  const int row = mc / rep, a = (kvh * rep + mc % rep) * A.maps + map;
  const int i = p0 + row;
  auto first_of = [&](int p) {
    return A.window > 0 ? (A.blocks ? p / A.window * A.window : max(0, p - A.window + 1)) : 0;
  };
  const int first_i = first_of(i), keep = A.window > 0 ? A.keep_first : 0;
  // positions of the workgroup's and of the wave's first and last pair (uniform)
  const int i_lo = p0 + m0 / rep, i_hi = p0 + (min(m0 + 16 * WV, pairs) - 1) / rep;
  const int w_lo = p0 + min(m0 + 16 * wave, pairs - 1) / rep, w_hi = p0 + min(m0 + 16 * wave + 15, pairs - 1) / rep;
  const int last = min(i_hi, A.kv_len[seg] - 1), i_vis = min(i, last);
  const int lo = first_of(i_lo), w_first = first_of(w_lo), w_first_hi = first_of(w_hi);
  const int head_tiles = (min(keep, lo) + kBandTile - 1) / kBandTile;   // tiles of the kept first positions
  const int band0 = max(head_tiles, lo / kBandTile), tiles = last / kBandTile + 1;

  // the queries' parts, as right operands: pair n, elements 32 s + 8 g4 .. + 7
  uint4 qp[3][KS];
  split_queries<KS>(A.q + ((long)(r0 + row) * hq + a) * DK + 8 * g4, qp);
  const float c1 = use_terms ? A.r1[a] : 0.f, c2 = use_terms ? A.r2[a] : 0.f;
  const float pbias = A.pb != nullptr ? A.pb[a] : 0.f;
  const float cap = A.softcap, icap = cap > 0.f ? 1.f / cap : 0.f;
  const float sink = A.sinks != nullptr ? A.sinks[a] : A.sink_all;
  float mx_ = A.has_sink ? sink : -INFINITY, l_ = A.has_sink && g4 == 0 ? 1.f : 0.f;
  ba_f32x4 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = ba_f32x4{0.f, 0.f, 0.f, 0.f};

  // a task loads 16 bytes of four neighbouring keys (of K, then of V), which share a page; the page of
  // the tile after next is looked up a tile ahead, so no load waits for a table entry
  uint4 st_[NT][4];
  int blk[NT];
  auto key_of = [&](int u, int tile) {
    const int task = tid + NTHR * u, e = task < TASKS_K ? task / (DK / 8) : (task - TASKS_K) / (DV / 8);
    return tile * kBandTile + 4 * e;
  };
  auto pages = [&](int tile) {
#pragma unroll
    for (int u = 0; u < NT; ++u) blk[u] = table[max(min(key_of(u, tile), last), 0) >> A.page_shift];   // (last: -1 without keys)
  };
  auto fetch = [&](int tile) {
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const int task = tid + NTHR * u, j0 = key_of(u, tile);
      const bool isk = task < TASKS_K;
      const int pc = isk ? task % (DK / 8) : (task - TASKS_K) % (DV / 8);
      const bool ok = task < TASKS && blk[u] >= 0 && blk[u] < A.num_blocks;
      const long slot = ((long)blk[u] << A.page_shift) + (j0 & ((1 << A.page_shift) - 1));
      const bf16_t* p = isk ? A.kc + slot * nk + (long)gk * DK + 8 * pc : A.vc + slot * nv + (long)kvh * DV + 8 * pc;
      const long step = isk ? nk : nv;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        st_[u][x] = uint4{0, 0, 0, 0};
        if (ok && j0 + x <= last) st_[u][x] = *reinterpret_cast<const uint4*>(p + x * step);
      }
    }
  };
  auto park = [&]() {
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const int task = tid + NTHR * u;
      if (task < TASKS_K) {
        const int kg = task / (DK / 8), pc = task % (DK / 8);
#pragma unroll
        for (int x = 0; x < 4; ++x) *reinterpret_cast<uint4*>(Ks + (4 * kg + x) * KROW + 8 * pc) = st_[u][x];
      } else if (task < TASKS) {
        // rows of V^T: keys in the order the weights come in, 16-byte pieces rotated by the row
        const int e = task - TASKS_K, kg = e / (DV / 8), pc = e % (DV / 8);
        const int piece = (kg >> 3) * 4 + (kg & 3), half = (kg >> 2) & 1;
        uint32_t w[4][4];
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          w[x][0] = st_[u][x].x; w[x][1] = st_[u][x].y; w[x][2] = st_[u][x].z; w[x][3] = st_[u][x].w;
        }
#pragma unroll
        for (int d = 0; d < 8; ++d) {
          const uint32_t sel = d & 1 ? 0x07060302u : 0x05040100u;
          const uint2 v = make_uint2(__builtin_amdgcn_perm(w[1][d >> 1], w[0][d >> 1], sel),
                                     __builtin_amdgcn_perm(w[3][d >> 1], w[2][d >> 1], sel));
          const int dv = 8 * pc + d;
          *reinterpret_cast<uint2*>(Vt + dv * kBandTile + ((piece ^ ((pc ^ d) & 7)) * 8) + 4 * half) = v;
        }
      }
    }
  };

  auto after = [&](int t) { return t + 1 < head_tiles || t >= band0 ? t + 1 : band0; };
  int tile = head_tiles > 0 ? 0 : band0;
  pages(tile);
  fetch(tile);
  pages(after(tile));
  while (tile < tiles) {
    __syncthreads();                                       // the last tile has been read
    park();
    __syncthreads();
    const int t0 = tile * kBandTile;
    tile = after(tile);
    if (tile < tiles) {
      fetch(tile);
      pages(after(tile));
    }
    // no pair of this wave sees the tile
    if (t0 > w_hi || (t0 + kBandTile <= w_first && t0 >= keep)) continue;
    ba_f32x4 sc[4];
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) sc[kt] = ba_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      uint4 kf[4];
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) kf[kt] = *reinterpret_cast<const uint4*>(Ks + (16 * kt + n) * KROW + 32 * s + 8 * g4);
#pragma unroll
      for (int p = 2; p >= 0; --p)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) sc[kt] = ba_mfma(kf[kt], qp[p][s], sc[kt]);
    }
    // scores of pair n: keys t0 + 16 kt + 4 g4 + v
    const bool whole = t0 + kBandTile - 1 <= min(w_lo, last) && (t0 >= w_first_hi || t0 + kBandTile <= keep);
    float tmax = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int j = t0 + 16 * kt + 4 * g4 + v, d = i - j;
        float z = sc[kt][v] * A.scale;
        if (use_cap) z = cap * tanh_(z * icap);
        if (use_terms) z -= c1 * logf(1.0f + c2 * (float)max(d, 0));
        if (use_dist) z += A.dist_bias[min(max(d, 0), A.nd - 1) * hq + a];
        if (sigmoid) z = sigmoidf_(z + pbias);
        if (!whole && !(j <= i_vis && (j >= first_i || j < keep))) z = sigmoid ? 0.f : -INFINITY;
        sc[kt][v] = z;
        tmax = fmaxf(tmax, z);
      }
    if (!sigmoid) {
      tmax = ft::kgroups_max(tmax);
      if (__ballot(tmax > mx_)) {                          // (rare once the first tiles have been seen)
        const float nm = fmaxf(mx_, tmax), f = mx_ == -INFINITY ? 0.f : ba_exp(mx_ - nm);
        l_ *= f;
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int v = 0; v < 4; ++v) o[t][v] *= f;
        mx_ = nm;
      }
      const float mu = mx_ == -INFINITY ? 0.f : mx_;
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          sc[kt][v] = ba_exp(sc[kt][v] - mu);
          l_ += sc[kt][v];
        }
    }
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      uint4 pp[3];
      split_bf16x3(sc[2 * kb][0], sc[2 * kb][1], pp[0].x, pp[1].x, pp[2].x);
      split_bf16x3(sc[2 * kb][2], sc[2 * kb][3], pp[0].y, pp[1].y, pp[2].y);
      split_bf16x3(sc[2 * kb + 1][0], sc[2 * kb + 1][1], pp[0].z, pp[1].z, pp[2].z);
      split_bf16x3(sc[2 * kb + 1][2], sc[2 * kb + 1][3], pp[0].w, pp[1].w, pp[2].w);
      uint4 vf[DT];
#pragma unroll
      for (int t = 0; t < DT; ++t)
        vf[t] = *reinterpret_cast<const uint4*>(Vt + (16 * t + n) * kBandTile + 8 * ((4 * kb + g4) ^ (((2 * t + (n >> 3)) ^ n) & 7)));
#pragma unroll
      for (int p = 2; p >= 0; --p)
#pragma unroll
        for (int t = 0; t < DT; ++t) o[t] = ba_mfma(vf[t], pp[p], o[t]);
    }
  }
  float f = 1.f;
  if (!sigmoid) {
    l_ = ft::kgroups_sum(l_);
    f = l_ > 0.f ? 1.0f / l_ : (l_ == 0.f ? 0.f : l_);     // (NaN stays)
  }
  if (m < pairs) {
    const long at = ((long)(r0 + row) * hq + a) * DV + 4 * g4;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      const float4 y = make_float4(o[t][0] * f, o[t][1] * f, o[t][2] * f, o[t][3] * f);
      if (A.out_bf16) *reinterpret_cast<uint2*>((bf16_t*)A.out + at + 16 * t) = make_uint2(ft::pack2(y.x, y.y), ft::pack2(y.z, y.w));
      else *reinterpret_cast<float4*>((float*)A.out + at + 16 * t) = y;
    }
  }
}

}  // namespace mx

using namespace mx;

// whether the sizes fit the kernel's tiles (otherwise: banded products)
extern "C" int mx_band_attn_fits(int dk, int dv, int block_size) {
  return (dk == 64 || dk == 128) && (dv == 64 || dv == 128) && block_size >= 4 &&
         (block_size & (block_size - 1)) == 0;
}

// pairs: (row, query head of a group) pairs over all segments of at least min_rows rows; segments of
// fewer rows are left alone
extern "C" int mx_band_attn(void* out, int out_bf16, const float* q, const void* k_cache, const void* v_cache, const int* start,
                            const int* pos0, const int* kv_len, const int* bt, int bt_stride, int num_segs,
                            int long_segs, long long_rows, int heads, int maps, int kv_heads, int dk, int dv, int window,
                            float scale, int sigmoid, const float* r1, const float* r2, const float* pb, int block_size,
                            int num_blocks, int min_rows, float softcap, int has_sink, float sink, const float* sinks,
                            int blocks, int keep_first, const float* dist_bias, int nd, hipStream_t s) {
  if (num_segs <= 0 || long_segs <= 0 || long_rows <= 0) return 0;
  if (!mx_band_attn_fits(dk, dv, block_size) || heads % kv_heads || maps < 1 || kv_heads * maps > 65535 ||
      min_rows < 1 || keep_first < 0 || (dist_bias != nullptr && nd < 1) || (blocks && window < 1)) return -1;
  if (((uintptr_t)q) % 16 || ((uintptr_t)out) % 16 || ((uintptr_t)k_cache) % 16 || ((uintptr_t)v_cache) % 16) return -2;
  const long rep = heads / kv_heads, gk = (long)kv_heads * maps;
  if (long_rows * rep > 0x3fffffffL || (long)nd * heads * maps > 0x7fffffffL) return -3;
  const BandArgs A{out, out_bf16, q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, start, pos0, kv_len, bt, bt_stride, num_segs,
                   heads, maps, kv_heads, window, scale, sigmoid, r1, r2, pb, __builtin_ctz((unsigned)block_size), num_blocks, min_rows, softcap,
                   has_sink, sink, sinks, blocks, keep_first, dist_bias, nd};
  // eight waves share a staged tile once that leaves two workgroups per CU; fewer pairs: four
  const bool wide = long_rows * rep * gk >= 2L * 256 * 128;
  const long items = long_rows * rep / (wide ? 128 : 64) + long_segs;
  const dim3 grid((unsigned)items, (unsigned)gk);
  const bool terms = r1 != nullptr, cap = softcap > 0.f, dist = dist_bias != nullptr;
  const int kind = sigmoid && !cap && !dist ? kBandSigmoid : sigmoid || terms || (cap && dist) ? kBandAny
                   : cap ? kBandCap : dist ? kBandDist : kBandPlain;
#define BA_KIND(DK, DV, KIND)                                                                       \
  do {                                                                                              \
    if (wide) hipLaunchKernelGGL((band_attn_kernel<DK, DV, 8, KIND>), grid, dim3(512), 0, s, A);     \
    else hipLaunchKernelGGL((band_attn_kernel<DK, DV, 4, KIND>), grid, dim3(256), 0, s, A);          \
  } while (0)
#define BA_GO(DK, DV)                                                                               \
  do {                                                                                              \
    if (kind == kBandPlain) BA_KIND(DK, DV, kBandPlain);                                            \
    else if (kind == kBandCap) BA_KIND(DK, DV, kBandCap);                                           \
    else if (kind == kBandDist) BA_KIND(DK, DV, kBandDist);                                         \
    else if (kind == kBandSigmoid) BA_KIND(DK, DV, kBandSigmoid);                                   \
    else BA_KIND(DK, DV, kBandAny);                                                                 \
  } while (0)
  if (dk == 128 && dv == 128) BA_GO(128, 128);
  else if (dk == 64 && dv == 128) BA_GO(64, 128);
  else if (dk == 128) BA_GO(128, 64);
  else BA_GO(64, 64);
#undef BA_GO
#undef BA_KIND
  return (int)hipGetLastError();
}

// Attention of long row segments (prefill chunks) over paged bf16 keys and values, in one pass: the
// masks, score terms and weights of the windowed attentions (window_attn.hip) with scores and sums on
// the matrix units and no scores in memory.
//
// Exactness: queries and weights are fp32 and stay fp32.  An fp32 value is the sum of three bf16 parts
// (hi + mid + lo, 24 bits), keys and values are bf16 already, so three v_mfma_f32_16x16x32_bf16 per
// operand pair form the same products as an fp32 multiply, summed in fp32, smallest parts first.
//
// Shape of the work: a workgroup owns one key head (and score map) and 64 consecutive (row, query head of
// the group) pairs of one segment, a wave 16 of them, so the tile of 64 keys that is staged in LDS serves
// all query heads that share it.  Everything is transposed: S^T = K Q^T and O^T = V^T P^T, a column per
// pair.  The result layout of the first product (lane (g, n): keys 4 g .. 4 g + 3 of pair n) is the operand
// layout of the second one, up to the order of the keys within 32, and V is staged in that order; a pair's
// maximum and sum need two lane swaps.  Rows of the next tile are on their way during the current one.
// A workgroup is one group of four waves, or two that take the tiles in turn, half a step apart (one in
// the first product while the other is in its weights and the second), and join their sums at the end.
//
// Vector work beside 96 MFMAs per 64 keys and wave: exponential, the three-way split, staging, about 300
// instructions (the score times log2(e) in one fused step, masks only on tiles that need them, loads
// without branches; 1150 before that, which took three times the products' time).  16 heads of 128 on 4
// key heads, us, before -> now: 2048 rows causal 115 -> 70, 4096 334 -> 206 (0.5 PFLOP/s of bf16 products),
// 777 37 -> 28, with a distance table 51 -> 32, with sigmoids of 2048 159 -> 83, five prompts of 258 to 542
// with a cap 51 -> 39; two fp32 products through memory with a weights kernel between them, gathers
// and layout changes around them, take 140 to 500 us and 25 launches per segment.
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
  float scale, scale2;                        // scale2: scale log2(e)
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

constexpr int kBandPairs = 64;                // pairs of a workgroup: 16 for each wave of a group

template <int DK, int DV, int KIND, int G>
__global__ void __launch_bounds__(256 * G, 2)
band_attn_kernel(BandArgs A) {
  constexpr bool kAny = KIND == kBandAny;
  const bool use_cap = kAny && A.softcap > 0.f;
  const bool use_terms = (KIND == kBandSigmoid || kAny) && A.r1 != nullptr;
  const bool use_dist = KIND == kBandDist || (kAny && A.dist_bias != nullptr);
  const bool sigmoid = KIND == kBandSigmoid || (kAny && A.sigmoid);
  constexpr bool kHalves = KIND == kBandSigmoid;                 // half of the weights beside the second products
  constexpr int KS = DK / 32, DT = DV / 16;
  constexpr int KROW = DK + 8;                                   // bf16 per staged key
  constexpr int kKeyBytes = kBandTile * KROW * 2, kValBytes = DV * kBandTile * 2, kGroup = kKeyBytes + kValBytes;
  static_assert(G == 1 || 2 * kGroup >= DT * 256 * 16 + 2 * 256 * 4, "the second group's results fit the tiles");
  __shared__ __attribute__((aligned(16))) char smem[G * kGroup];
  const int tid = threadIdx.x & 255, lane = tid & 63;
  const int grp = G > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  bf16_t* const Ks = reinterpret_cast<bf16_t*>(smem + grp * kGroup);
  bf16_t* const Vt = reinterpret_cast<bf16_t*>(smem + grp * kGroup + kKeyBytes);
  const int n = lane & 15, g4 = lane >> 4;
  const int rep = A.heads / A.kv_heads, gks = A.kv_heads * A.maps, gk = blockIdx.x % gks, kvh = gk / A.maps, map = gk % A.maps;
  int seg, block;
  if (!segment_block(A.start, A.num_segs, A.min_rows, rep, kBandPairs, blockIdx.x / gks, seg, block)) return;
  seg = __builtin_amdgcn_readfirstlane(seg);
  block = __builtin_amdgcn_readfirstlane(block);
  const int r0 = A.start[seg], rows = A.start[seg + 1] - r0, p0 = A.pos0[seg];
  const int pairs = rows * rep, m0 = block * kBandPairs;
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
  const int i_lo = p0 + m0 / rep, i_hi = p0 + (min(m0 + kBandPairs, pairs) - 1) / rep;
  const int w_lo = p0 + min(m0 + 16 * wave, pairs - 1) / rep, w_hi = p0 + min(m0 + 16 * wave + 15, pairs - 1) / rep;
  const int last = min(i_hi, A.kv_len[seg] - 1), i_vis = min(i, last);
  const int lo = first_of(i_lo), w_first = first_of(w_lo), w_first_hi = first_of(w_hi);
  const int head_tiles = (min(keep, lo) + kBandTile - 1) / kBandTile;   // tiles of the kept first positions
  const int band0 = max(head_tiles, lo / kBandTile), tiles = last / kBandTile + 1;
  // the tiles in turn: group g takes those of numbers G s + g
  const int count = min(head_tiles, tiles) + max(0, tiles - band0);
  auto tile_of = [&](int q) {
    q = min(q, count - 1);
    return q < head_tiles ? q : band0 + q - head_tiles;
  };

  const float c1 = use_terms ? A.r1[a] : 0.f, c2 = use_terms ? A.r2[a] : 0.f;
  const float pbias = A.pb != nullptr ? A.pb[a] : 0.f;
  const float cap = A.softcap, icap = cap > 0.f ? (KIND == kBandCap ? A.scale / cap : 1.f / cap) : 0.f;
  const float sink = A.sinks != nullptr ? A.sinks[a] : A.sink_all;
  // Without terms a score is v vmul in base 2, v the product or tanh.  With terms it stays as it is: a bias may be the type's
  // lowest value, which has no multiple, and log2(e) rounded once for all would be a larger error than ba_exp's.
  constexpr bool kTwo = KIND == kBandPlain || KIND == kBandCap;
  constexpr float kLog2e = 1.44269502f;
  const float vmul = KIND == kBandPlain ? A.scale2 : KIND == kBandCap ? cap * kLog2e : 1.f;
  auto weight = [](float x) { return kTwo ? __builtin_amdgcn_exp2f(x) : ba_exp(x); };
  const bool sinks = A.has_sink && grp == 0;
  float mx_ = sinks ? (kTwo ? sink * kLog2e : sink) : -INFINITY, l_ = sinks && g4 == 0 ? 1.f : 0.f;
  ba_f32x4 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = ba_f32x4{0.f, 0.f, 0.f, 0.f};

  // A thread of a group loads 16 bytes of four neighbouring keys, which share a page, of K and of V; the page of a tile is
  // looked up a tile ahead, so no load waits for a table entry.  Past the last tile that one again.
  constexpr int PK = DK / 8, PV = DV / 8;
  const int k_key = 4 * min(tid / PK, 15), v_key = 4 * min(tid / PV, 15);
  const bf16_t* const k_base = A.kc + (long)gk * DK + 8 * (tid % PK);
  const bf16_t* const v_base = A.vc + (long)kvh * DV + 8 * (tid % PV);
  auto page = [&](int q, int key) {
    return table[max(min(tile_of(q) * kBandTile + key, last), 0) >> A.page_shift];       // (last: -1 without keys)
  };
  // whether any of the wave's keys is past the last or has no page
  auto fetch = [&](uint4 (&st)[4], int q, int key, int blk, const bf16_t* base, long step) {
    const int j = tile_of(q) * kBandTile + key;
    const bool bad = (unsigned)blk >= (unsigned)A.num_blocks;
    const bf16_t* p = base + (((long)(bad ? 0 : blk) << A.page_shift) + (j & ((1 << A.page_shift) - 1))) * step;
#pragma unroll
    for (int x = 0; x < 4; ++x) st[x] = *reinterpret_cast<const uint4*>(p + x * step);
    return __ballot(bad || j + 3 > last) != 0;
  };
  // those are zeros (a page may hold anything there)
  auto clear = [&](uint4 (&st)[4], int q, int key, int blk) {
    const int j = tile_of(q) * kBandTile + key;
#pragma unroll
    for (int x = 0; x < 4; ++x)
      if ((unsigned)blk >= (unsigned)A.num_blocks || j + x > last) st[x] = uint4{0, 0, 0, 0};
  };
  uint4 ks[4], vs[4];
  auto park_k = [&]() {
    if (tid < 16 * PK)
#pragma unroll
      for (int x = 0; x < 4; ++x) *reinterpret_cast<uint4*>(Ks + (k_key + x) * KROW + 8 * (tid % PK)) = ks[x];
  };
  auto park_v = [&]() {
    if (tid >= 16 * PV) return;
    // rows of V^T: keys in the order the weights come in, 16-byte pieces rotated by the row
    const int kg = tid / PV, pc = tid % PV;
    const int piece = (kg >> 3) * 4 + (kg & 3), half = (kg >> 2) & 1;
    uint32_t w[4][4];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      w[x][0] = vs[x].x; w[x][1] = vs[x].y; w[x][2] = vs[x].z; w[x][3] = vs[x].w;
    }
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      const uint32_t sel = d & 1 ? 0x07060302u : 0x05040100u;
      const uint2 v = make_uint2(__builtin_amdgcn_perm(w[1][d >> 1], w[0][d >> 1], sel),
                                 __builtin_amdgcn_perm(w[3][d >> 1], w[2][d >> 1], sel));
      *reinterpret_cast<uint2*>(Vt + (8 * pc + d) * kBandTile + ((piece ^ ((pc ^ d) & 7)) * 8) + 4 * half) = v;
    }
  };

  // the score terms of keys 16 kt .. of a tile; sigmoids are weights already
  auto terms = [&](ba_f32x4 (&sc)[4], int t0, bool whole, int kt0, int kt1) {
#pragma unroll
    for (int kt = kt0; kt < kt1; ++kt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int d = i - (t0 + 16 * kt + 4 * g4 + v);
        float z = sc[kt][v];
        if constexpr (KIND == kBandCap) z = tanh_(z * icap);
        if constexpr (KIND != kBandPlain && KIND != kBandCap) z *= A.scale;
        if constexpr (kAny) {
          if (use_cap) z = cap * tanh_(z * icap);
        }
        if (use_terms) z -= c1 * logf(1.0f + c2 * (float)max(d, 0));
        if (use_dist) z += A.dist_bias[min(max(d, 0), A.nd - 1) * hq + a];
        if (sigmoid) z = sigmoidf_(z + pbias);
        sc[kt][v] = z;
      }
    if (whole) return;
    const float none = sigmoid ? 0.f : -INFINITY;
#pragma unroll
    for (int kt = kt0; kt < kt1; ++kt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int j = t0 + 16 * kt + 4 * g4 + v;
        sc[kt][v] = j <= i_vis && (j >= first_i || j < keep) ? sc[kt][v] : none;
      }
  };

  if (count > 0) {
    const int steps = (count + G - 1) / G;
    int k_blk = page(grp, k_key), v_blk = page(grp, v_key), k_next = page(grp + G, k_key), v_next = page(grp + G, v_key);
    bool k_holes = fetch(ks, grp, k_key, k_blk, k_base, nk), v_holes = fetch(vs, grp, v_key, v_blk, v_base, nv);
    // the queries' parts, as right operands: pair n, elements 32 s + 8 g4 .. + 7 (behind the tiles, which are two loads away)
    uint4 qp[3][KS];
    split_queries<KS>(A.q + ((long)(r0 + row) * hq + a) * DK + 8 * g4, qp);
    if (k_holes) clear(ks, grp, k_key, k_blk);
    park_k();
    __syncthreads();
    if (G > 1 && grp != 0) __syncthreads();                // half a step behind
    for (int s = 0; s < steps; ++s) {
      const int q = G * s + grp, t0 = tile_of(q) * kBandTile;
      // whether a pair of this wave sees the tile
      const bool seen = q < count && t0 <= w_hi && !(t0 + kBandTile <= w_first && t0 >= keep);
      // (loads come back in order: the pages, which the next step copies, before the rows)
      const int v_at = v_next;
      k_blk = k_next;
      k_next = page(q + 2 * G, k_key);
      v_next = page(q + 2 * G, v_key);
      k_holes = fetch(ks, q + G, k_key, k_blk, k_base, nk);
      ba_f32x4 sc[4];
      const bool whole = t0 + kBandTile - 1 <= min(w_lo, last) && (t0 >= w_first_hi || t0 + kBandTile <= keep);
      if (seen) {
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) sc[kt] = ba_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s_ = 0; s_ < KS; ++s_) {
          uint4 kf[4];
#pragma unroll
          for (int kt = 0; kt < 4; ++kt)
            kf[kt] = *reinterpret_cast<const uint4*>(Ks + (16 * kt + n) * KROW + 32 * s_ + 8 * g4);
#pragma unroll
          for (int p = 2; p >= 0; --p)
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) sc[kt] = ba_mfma(kf[kt], qp[p][s_], sc[kt]);
        }
        // scores of pair n: keys t0 + 16 kt + 4 g4 + v
        terms(sc, t0, whole, 0, kHalves ? 2 : 4);
        if (!sigmoid) {
          float tmax = sc[0][0];
#pragma unroll
          for (int e = 1; e < 16; ++e) tmax = fmaxf(tmax, sc[e >> 2][e & 3]);
          tmax = ft::kgroups_max(tmax) * vmul;
          if (__ballot(tmax > mx_)) {                          // (rare once the first tiles have been seen)
            const float nm = fmaxf(mx_, tmax), f = mx_ == -INFINITY ? 0.f : weight(mx_ - nm);
            l_ *= f;
#pragma unroll
            for (int t = 0; t < DT; ++t)
#pragma unroll
              for (int v = 0; v < 4; ++v) o[t][v] *= f;
            mx_ = nm;
          }
        }
      }
      if (v_holes) clear(vs, q, v_key, v_blk);
      park_v();
      __syncthreads();
      v_blk = v_at;
      v_holes = fetch(vs, q + G, v_key, v_blk, v_base, nv);
      if (seen) {
        if constexpr (kHalves) terms(sc, t0, whole, 2, 4);
        if (!sigmoid) {
          const float mu = mx_ == -INFINITY ? 0.f : mx_;
#pragma unroll
          for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              sc[kt][v] = weight(kTwo ? fmaf(sc[kt][v], vmul, -mu) : sc[kt][v] - mu);
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
      if (s + 1 < steps) {                                 // (nor waited for past the last)
        if (k_holes) clear(ks, q + G, k_key, k_blk);
        park_k();
      }
      __syncthreads();
    }
    if (G > 1 && grp == 0) __syncthreads();
  }
  if (!sigmoid) l_ = ft::kgroups_sum(l_);
  // the second group's results through LDS; the first writes
  float4* const part = reinterpret_cast<float4*>(smem);
  float f = 1.f, f2 = 1.f;
  if constexpr (G > 1) {
    float* const ml = reinterpret_cast<float*>(smem + DT * 256 * 16);
    __syncthreads();
    if (grp != 0) {
#pragma unroll
      for (int t = 0; t < DT; ++t) part[256 * t + tid] = make_float4(o[t][0], o[t][1], o[t][2], o[t][3]);
      ml[tid] = mx_, ml[256 + tid] = l_;
    }
    __syncthreads();
    if (grp != 0) return;
    if (!sigmoid) {
      const float m2 = ml[tid], l2 = ml[256 + tid], nm = fmaxf(mx_, m2), mu = nm == -INFINITY ? 0.f : nm;
      f = mx_ == mu ? 1.f : weight(mx_ - mu), f2 = m2 == mu ? 1.f : weight(m2 - mu);     // (a sink may be infinite)
      l_ = l_ * f + l2 * f2;
    }
  }
  if (!sigmoid) {
    const float inv = l_ > 0.f ? 1.0f / l_ : (l_ == 0.f ? 0.f : l_);         // (NaN stays)
    f *= inv, f2 *= inv;
  }
  if (m < pairs) {
    const long at = ((long)(r0 + row) * hq + a) * DV + 4 * g4;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      float4 y = make_float4(o[t][0] * f, o[t][1] * f, o[t][2] * f, o[t][3] * f);
      if constexpr (G > 1) {
        const float4 u = part[256 * t + tid];
        y.x += u.x * f2, y.y += u.y * f2, y.z += u.z * f2, y.w += u.w * f2;
      }
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
// fewer rows are left alone.  groups: 1 or 2 groups of waves to a workgroup, with the same results up to fp32 sums
extern "C" int mx_band_attn(void* out, int out_bf16, const float* q, const void* k_cache, const void* v_cache, const int* start,
                            const int* pos0, const int* kv_len, const int* bt, int bt_stride, int num_segs,
                            int long_segs, long long_rows, int heads, int maps, int kv_heads, int dk, int dv, int window,
                            float scale, int sigmoid, const float* r1, const float* r2, const float* pb, int block_size,
                            int num_blocks, int min_rows, float softcap, int has_sink, float sink, const float* sinks,
                            int blocks, int keep_first, const float* dist_bias, int nd, int groups, hipStream_t s) {
  if (num_segs <= 0 || long_segs <= 0 || long_rows <= 0) return 0;
  if (!mx_band_attn_fits(dk, dv, block_size) || heads % kv_heads || maps < 1 || kv_heads * maps > 65535 ||
      groups < 1 || groups > 2 || min_rows < 1 || keep_first < 0 || (dist_bias != nullptr && nd < 1) || (blocks && window < 1)) return -1;
  if (((uintptr_t)q) % 16 || ((uintptr_t)out) % 16 || ((uintptr_t)k_cache) % 16 || ((uintptr_t)v_cache) % 16) return -2;
  const long rep = heads / kv_heads, gk = (long)kv_heads * maps;
  if (long_rows * rep > 0x3fffffffL || (long)nd * heads * maps > 0x7fffffffL) return -3;
  const BandArgs A{out, out_bf16, q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, start, pos0, kv_len, bt, bt_stride, num_segs,
                   heads, maps, kv_heads, window, scale, (float)(scale * 1.4426950408889634), sigmoid, r1, r2, pb, __builtin_ctz((unsigned)block_size), num_blocks, min_rows, softcap,
                   has_sink, sink, sinks, blocks, keep_first, dist_bias, nd};
  const long items = long_rows * rep / kBandPairs + long_segs;
  if (items * gk > 0x7fffffffL) return -3;
  const dim3 grid((unsigned)(items * gk));                               // the longest blocks of all heads first
  const bool two = groups == 2;
  const bool terms = r1 != nullptr, cap = softcap > 0.f, dist = dist_bias != nullptr;
  const int kind = sigmoid && !cap && !dist ? kBandSigmoid : sigmoid || terms || (cap && dist) ? kBandAny
                   : cap ? kBandCap : dist ? kBandDist : scale > 0.f ? kBandPlain : kBandAny;
#define BA_KIND(DK, DV, KIND)                                                                       \
  do {                                                                                              \
    if (two) hipLaunchKernelGGL((band_attn_kernel<DK, DV, KIND, 2>), grid, dim3(512), 0, s, A);     \
    else hipLaunchKernelGGL((band_attn_kernel<DK, DV, KIND, 1>), grid, dim3(256), 0, s, A);         \
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

// Windowed attention of decode rows and short segments over paged bf16 keys and values (window_attn.hip's masks,
// score terms and weights) on the matrix units.
//
// fp32 queries and weights stay fp32: each is the exact sum of three bf16 parts, keys and values are bf16 already,
// so three v_mfma_f32_16x16x32_bf16 per operand pair form the products of an fp32 multiply, summed in fp32.
//
// A workgroup owns one row and one key head (and score map) with the up to 16 query heads that share it; its waves
// (eight, fewer where there are many groups) take 32 keys in turn, so a key is read once for all its heads.
// S^T = K Q^T and O^T = V^T P^T, a column per head: keys go straight from memory to operands, values through a wave's
// own LDS strip (ds_read_b64_tr_b16), and weights need no exchange.  The next 32 keys load under the softmax and the
// sums.  The waves' (maximum, sum, sums) meet in LDS at the end: one launch, whatever the length.
// Bound by the vector units for few rows (a step of 32 keys is 700 instructions of a wave beside 48 products, two waves a unit),
// by the read of the keys for many: so terms that a row has not are skipped for all of its keys at once, whole steps ask for no
// key's presence, and blocks of a power of two are shifted.  us in a graph at 30 / 300 / 540 / 1024 keys, 16 heads of 128 on 4 key
// heads: one row 7.4 11 13 18, 64 rows 8.2 16 23 33; two maps of 64, one row 6.9 9.9 11 14 (a look at every term and key by
// itself: 8.1 13 16 23, 8.6 18 25 36 and 7.3 12 14 19; general kernel, a workgroup per head: 50 a row of 900).  Two steps of keys
// on their way were no sooner.  One query head a key head wastes fifteen columns of sixteen: 64 rows of 16 such heads 10 us at 30
// keys, 61 at 540, 328 at 3300.  Lengths are not known on the host where a step is replayed, so sizes alone choose.
// (Eight waves for all of them and a merge that read every wave's part, an entry a thread: 32 at 100 keys; 16 heads a
// group, one key: 12.4, now 9.3.)  Lengths are not known on the host where a step is replayed, so sizes alone choose.
#include "mx_common.h"

#include <type_traits>

namespace mx {

typedef __bf16 wd_bf16x8 __attribute__((ext_vector_type(8)));
typedef float wd_f32x4 __attribute__((ext_vector_type(4)));
typedef short wd_i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) wd_i16x4 wd_lds_i16x4;

struct WindowArgs {
  void* out;                                  // fp32, or bf16 (rounded once, here)
  int out_bf16;
  const float* q;
  const bf16_t *kc, *vc;
  const int *start, *pos0, *kv_len, *bt;
  int bt_stride, num_segs, heads, maps, kv_heads, window;
  float scale;
  int sigmoid;
  const float *r1, *r2, *pb;
  int block_size, num_blocks, skip_from;
  float softcap;
  int has_sink;
  float sink_all;
  const float* sinks;
  int blocks, keep_first;
  const float* dist_bias;
  int nd, block_shift;                        // block_size as a power of two, or -1
};

__device__ __forceinline__ wd_f32x4 wd_mfma(const uint4& a, const uint4& b, wd_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(wd_bf16x8, a), __builtin_bit_cast(wd_bf16x8, b), c,
                                                 0, 0, 0);
}

constexpr int kWdKeys = 32, kWdMaxRep = 16;

// e^x, x <= 0: 2^(x log2 e) with the rounding of that product, and of log2 e, in a first-order term; a unit in the last place or so
__device__ __forceinline__ float wd_exp(float x) {
  constexpr float kLog2e = 1.44269504f, kLow = 1.92596299e-8f, kLn2 = 0.693147181f;   // (kLow: log2 e - kLog2e)
  x = fmaxf(x, -160.f);                       // (there 0 already)
  const float t = x * kLog2e, low = fmaf(x, kLow, fmaf(x, kLog2e, -t)), e = __builtin_amdgcn_exp2f(t);
  return fmaf(e * low, kLn2, e);
}

template <int DK, int DV, int WV>
__global__ void __launch_bounds__(64 * WV, 2)
window_decode_kernel(WindowArgs A) {
  constexpr int KS = DK / 32, DT = DV / 16, PV = DV / 8, VL = kWdKeys * PV / 64;
  constexpr int kStrip = kWdKeys * DV * 2, kMerge = kWdMaxRep * DV * 4;      // bytes per wave
  __shared__ __attribute__((aligned(16))) uint8_t lds[WV * (kStrip > kMerge ? kStrip : kMerge)];
  __shared__ float ml[WV][2][kWdMaxRep];
  const int row = blockIdx.x, gk = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g4 = lane >> 4;
  const int s = segment_of(A.start, A.num_segs, row);
  const int r0 = A.start[s], rows = A.start[s + 1] - r0;
  if (row >= A.start[A.num_segs] || (A.skip_from > 0 && rows >= A.skip_from)) return;
  const int rep = A.heads / A.kv_heads, kvh = gk / A.maps, map = gk % A.maps, hq = A.heads * A.maps;
  const int a = (kvh * rep + min(n, rep - 1)) * A.maps + map;
  const long nk = (long)A.kv_heads * A.maps * DK, nv = (long)A.kv_heads * DV;
  const int i = A.pos0[s] + (row - r0), last = min(i, A.kv_len[s] - 1);
  const int first = A.window > 0 ? (A.blocks ? i / A.window * A.window : max(0, i - A.window + 1)) : 0;
  // kept first positions that lie before the window go in front of it
  const int ext = A.window > 0 ? max(0, min(min(A.keep_first, first), last + 1)) : 0;
  const int nkeys = ext + max(0, last - first + 1);
  const int* table = A.bt + (long)s * A.bt_stride;

  // No load of the keys' loop stands behind a branch or is looked at before the next step: the loads come back in order, so
  // a table entry whose range was checked at once waited for the keys asked for before it, twice a step (22.7 us a row of 1024
  // keys, 21.2 so).  Keys that there are not read slot 0 and count for nothing.
  uint4 k[2][KS], v[VL];
  constexpr int kStep = WV * kWdKeys;
  int slot[2], vslot[VL], blk[2], off[2];      // this step's slots (none: -1), the next one's table entries and places in them
  auto look = [&](int c0) {                    // lane n of each group: keys n and 16 + n
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int c = c0 + 16 * t + n, in = min(c, nkeys - 1), j = in < ext ? in : first + in - ext;
      const int b = A.block_shift >= 0 ? j >> A.block_shift : j / A.block_size;
      blk[t] = table[b];
      off[t] = c < nkeys ? j - b * A.block_size : -1;
    }
  };
  auto fetch = [&]() {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      slot[t] = off[t] >= 0 && blk[t] >= 0 && blk[t] < A.num_blocks ? blk[t] * A.block_size + off[t] : -1;
      const bf16_t* p = A.kc + max(slot[t], 0) * nk + (long)gk * DK + 8 * g4;
#pragma unroll
      for (int x = 0; x < KS; ++x) k[t][x] = *reinterpret_cast<const uint4*>(p + 32 * x);
    }
#pragma unroll
    for (int x = 0; x < VL; ++x) {
      vslot[x] = __shfl(slot[x < VL / 2 ? 0 : 1], ((64 * x + lane) / PV) & 15);
      v[x] = *reinterpret_cast<const uint4*>(A.vc + max(vslot[x], 0) * nv + (long)kvh * DV + (lane % PV) * 8);
    }
  };
  const float* q = A.q + ((long)row * hq + a) * DK + 8 * g4;
  float4 raw[KS][2];
#pragma unroll
  for (int x = 0; x < KS; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) raw[x][y] = *reinterpret_cast<const float4*>(q + 32 * x + 4 * y);
  const float c1 = A.r1 != nullptr ? A.r1[a] : 0.f, c2 = A.r1 != nullptr ? A.r2[a] : 0.f;
  const float bias = A.sigmoid && A.pb != nullptr ? A.pb[a] : 0.f;
  const bool sinks = A.has_sink && !A.sigmoid && wave == 0;
  float mx_ = sinks ? (A.sinks != nullptr ? A.sinks[a] : A.sink_all) : -INFINITY, l_ = sinks && g4 == 0 ? 1.f : 0.f;
  if (nkeys > 0) {
    look(wave * kWdKeys);
    fetch();
    look(wave * kWdKeys + kStep);
  }

  // the queries' parts, as right operands: head n, elements 32 x + 8 g4 .. + 7
  uint4 qp[3][KS];
  split_queries<KS>(raw, qp);
  wd_f32x4 o[DT];                              // columns 16 t + 4 g4 .. of head n
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = wd_f32x4{0.f, 0.f, 0.f, 0.f};
  // values in LDS: rows of PV pieces, piece p of key j at p ^ swap(j) (no bank conflicts in the transposed read)
  uint8_t* strip = lds + wave * kStrip;
  const auto swap = [](int j) { return DV == 128 ? 2 * (j & 7) : 2 * ((j >> 1) & 3); };
  const int vkey = 4 * g4 + (n >> 2);

  for (int c0 = wave * kWdKeys; c0 < nkeys; c0 += kStep) {
    wave_lds_fence();                          // (the last strip has been read)
    const bool whole = __all(slot[0] >= 0 && slot[1] >= 0);
    if (!whole) {
#pragma unroll
      for (int x = 0; x < VL; ++x)
        if (vslot[x] < 0) v[x] = uint4{0, 0, 0, 0};
    }
#pragma unroll
    for (int x = 0; x < VL; ++x) {
      const int key = (64 * x + lane) / PV;
      *reinterpret_cast<uint4*>(strip + key * DV * 2 + ((lane % PV) ^ swap(key)) * 16) = v[x];
    }
    // (loads come back in order: the bias of this step is asked for before the next step's keys)
    float db[2][4];
    if (A.dist_bias != nullptr) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int c = c0 + 16 * t + 4 * g4 + e, d = i - (c < ext ? c : first + c - ext);
          db[t][e] = A.dist_bias[(long)min(max(d, 0), A.nd - 1) * hq + a];
        }
    }
    wd_f32x4 sp[3][2], sc[2];                  // (a chain per part)
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int t = 0; t < 2; ++t) sp[p][t] = wd_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < KS; ++x)
#pragma unroll
      for (int p = 2; p >= 0; --p)
#pragma unroll
        for (int t = 0; t < 2; ++t) sp[p][t] = wd_mfma(k[t][x], qp[p][x], sp[p][t]);
#pragma unroll
    for (int t = 0; t < 2; ++t) sc[t] = sp[2][t] + sp[1][t] + sp[0][t];
    // which of keys 16 t + 4 g4 + e there are
    bool has[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) has[t][e] = whole || __shfl(slot[t], 4 * g4 + e) >= 0;
    fetch();
    look(c0 + 2 * kStep);
    auto scores = [&](auto f) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[t][e] = f(sc[t][e], t, e);
    };
    // (a look at each term for all of them: the vector units bound a step, and most rows have none)
    scores([&](float z, int, int) { return z * A.scale; });
    if (A.softcap > 0.f) scores([&](float z, int, int) { return A.softcap * tanhf(z / A.softcap); });
    if (A.r1 != nullptr)
      scores([&](float z, int t, int e) {
        const int c = c0 + 16 * t + 4 * g4 + e, d = i - (c < ext ? c : first + c - ext);
        return z - c1 * logf(1.0f + c2 * (float)max(d, 0));
      });
    if (A.dist_bias != nullptr) scores([&](float z, int t, int e) { return z + db[t][e]; });
    if (A.sigmoid) scores([&](float z, int, int) { return sigmoidf_(z + bias); });
    if (!whole) {
      const float none = A.sigmoid ? 0.f : -INFINITY;
      scores([&](float z, int t, int e) { return has[t][e] ? z : none; });
    }
    if (!A.sigmoid) {
      const float top = fmaxf(fmaxf(fmaxf(sc[0][0], sc[0][1]), fmaxf(sc[0][2], sc[0][3])),
                              fmaxf(fmaxf(sc[1][0], sc[1][1]), fmaxf(sc[1][2], sc[1][3])));
      const float mn = fmaxf(mx_, ft::kgroups_max(top)), mu = mn == -INFINITY ? 0.f : mn;
      const float f = mx_ == -INFINITY ? 0.f : wd_exp(mx_ - mu);
      l_ *= f;
#pragma unroll
      for (int t = 0; t < DT; ++t) o[t] *= f;
      mx_ = mn;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          sc[t][e] = wd_exp(sc[t][e] - mu);
          l_ += sc[t][e];
        }
    }
    uint4 pp[3];
    split_bf16x3(sc[0][0], sc[0][1], pp[0].x, pp[1].x, pp[2].x);
    split_bf16x3(sc[0][2], sc[0][3], pp[0].y, pp[1].y, pp[2].y);
    split_bf16x3(sc[1][0], sc[1][1], pp[0].z, pp[1].z, pp[2].z);
    split_bf16x3(sc[1][2], sc[1][3], pp[0].w, pp[1].w, pp[2].w);
    wave_lds_fence();
    uint4 vt[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      const uint8_t* at = strip + vkey * DV * 2 + ((2 * t + ((n >> 1) & 1)) ^ swap(vkey)) * 16 + (n & 1) * 8;
      const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((wd_lds_i16x4*)at));
      const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((wd_lds_i16x4*)(at + 16 * DV * 2)));
      vt[t] = make_uint4(lo.x, lo.y, hi.x, hi.y);
    }
#pragma unroll
    for (int p = 2; p >= 0; --p)
#pragma unroll
      for (int t = 0; t < DT; ++t) o[t] = wd_mfma(vt[t], pp[p], o[t]);
  }
  // the waves' parts
  __syncthreads();
  const int waves = max(1, min(WV, (nkeys + kWdKeys - 1) / kWdKeys));       // that have seen a key
  l_ = ft::kgroups_sum(l_);
  float* mine = reinterpret_cast<float*>(lds) + (long)wave * rep * DV;
  if (n < rep && wave < waves) {
#pragma unroll
    for (int t = 0; t < DT; ++t)
      *reinterpret_cast<float4*>(mine + n * DV + 16 * t + 4 * g4) = make_float4(o[t][0], o[t][1], o[t][2], o[t][3]);
    if (g4 == 0) ml[wave][0][n] = mx_, ml[wave][1][n] = l_;
  }
  __syncthreads();
  // (all of the waves: a constant, every read in flight; four columns a thread where the entries are more than the threads)
  auto merge = [&](auto count, auto cols) {
    constexpr int C = decltype(cols)::value;
    for (int e = tid; e < rep * (DV / C); e += 64 * WV) {
      const int h = e / (DV / C);
      float top = -INFINITY, l = 0.f, y[C];
#pragma unroll
      for (int c = 0; c < C; ++c) y[c] = 0.f;
#pragma unroll
      for (int w = 0; w < count; ++w) top = fmaxf(top, ml[w][0][h]);
#pragma unroll
      for (int w = 0; w < count; ++w) {
        const float f = A.sigmoid ? 1.f : ml[w][0][h] == -INFINITY ? 0.f : expf(ml[w][0][h] - top);
        const float* p = reinterpret_cast<const float*>(lds) + (long)w * rep * DV + e * C;
        l += f * ml[w][1][h];
#pragma unroll
        for (int c = 0; c < C; ++c) y[c] += f * p[c];
      }
#pragma unroll
      for (int c = 0; c < C; ++c) y[c] = A.sigmoid ? y[c] : l > 0.f ? y[c] / l : 0.f;
      const long at = ((long)row * hq + (kvh * rep + h) * A.maps + map) * DV + C * (e % (DV / C));
      if constexpr (C == 4) {
        if (A.out_bf16) *reinterpret_cast<uint2*>((bf16_t*)A.out + at) = make_uint2(ft::pack2(y[0], y[1]), ft::pack2(y[2], y[3]));
        else *reinterpret_cast<float4*>((float*)A.out + at) = make_float4(y[0], y[1], y[2], y[3]);
      } else {
        if (A.out_bf16) st((bf16_t*)A.out, at, y[0]);
        else ((float*)A.out)[at] = y[0];
      }
    }
  };
  const std::integral_constant<int, 1> one;
  const std::integral_constant<int, 4> four;
  const std::integral_constant<int, WV> all;
  if (rep * DV > 64 * WV) {
    if (waves == WV) merge(all, four);
    else merge(waves, four);
  } else {
    if (waves == WV) merge(all, one);
    else merge(waves, one);
  }
}

}  // namespace mx

using namespace mx;

// whether the sizes and addresses fit the kernel's tiles
extern "C" int mx_window_decode_fits(const void* out, const void* q, const void* k_cache, const void* v_cache,
                                     int cache_bf16, int heads, int maps, int kv_heads, int dk, int dv, int block_size,
                                     int num_blocks) {
  return cache_bf16 && maps >= 1 && kv_heads >= 1 && (dk == 64 || dk == 128) && (dv == 64 || dv == 128) && heads / kv_heads <= kWdMaxRep &&
         (long)kv_heads * maps <= 65535 && (long)block_size * num_blocks <= 0x7fffffffL &&
         ((((uintptr_t)out) | ((uintptr_t)q) | ((uintptr_t)k_cache) | ((uintptr_t)v_cache)) % 16) == 0;
}

// arguments as mx_window_attention (checked there)
extern "C" int mx_window_decode(void* out, int out_bf16, const float* q, const void* k_cache, const void* v_cache, const int* start,
                                const int* pos0, const int* kv_len, const int* bt, int bt_stride, int num_segs,
                                long total_rows, int heads, int maps, int kv_heads, int dk, int dv, int window, float scale,
                                int sigmoid, const float* r1, const float* r2, const float* pb, int block_size,
                                int num_blocks, int skip_from, float softcap, int has_sink, float sink,
                                const float* sinks, int blocks, int keep_first, const float* dist_bias, int nd,
                                hipStream_t s) {
  const WindowArgs A{out, out_bf16, q, (const bf16_t*)k_cache, (const bf16_t*)v_cache, start, pos0, kv_len, bt, bt_stride, num_segs,
                     heads, maps, kv_heads, window, scale, sigmoid, r1, r2, pb, block_size, num_blocks, skip_from, softcap,
                     has_sink, sink, sinks, blocks, keep_first, dist_bias, nd,
                     block_size & (block_size - 1) ? -1 : __builtin_ctz(block_size)};
  const long groups = total_rows * kv_heads * maps;
  const dim3 grid((unsigned)total_rows, (unsigned)(kv_heads * maps));
  // eight waves are a CU's registers: fewer share a group's keys where that leaves groups waiting.  us with 8 / 4 / 2 waves,
  // 16 heads of 128 with a key head each: 64 rows (1024 groups) of 30 keys 27 15 9, of 300 56 42 34, of 1500 178 173 155; 32
  // rows (512) of 20 15 9 9, of 600 41 34 47; 4 key heads, 64 rows (256) of 30 9 9 9, of 400 20 23 30, of 6000 161 226 331
  const int wv = groups <= 256 ? 8 : groups <= 512 ? 4 : 2;
#define WD_WAVES(DK, DV, WV) hipLaunchKernelGGL((window_decode_kernel<DK, DV, WV>), grid, dim3(64 * WV), 0, s, A)
#define WD_GO(DK, DV)                     \
  do {                                    \
    if (wv == 8) WD_WAVES(DK, DV, 8);     \
    else if (wv == 4) WD_WAVES(DK, DV, 4); \
    else WD_WAVES(DK, DV, 2);             \
  } while (0)
  if (dk == 128 && dv == 128) WD_GO(128, 128);
  else if (dk == 64 && dv == 128) WD_GO(64, 128);
  else if (dk == 128) WD_GO(128, 64);
  else WD_GO(64, 64);
#undef WD_GO
#undef WD_WAVES
  return (int)hipGetLastError();
}

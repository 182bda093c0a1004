// Recurrences with a decay per head and key channel, long segments, in chunk form: the gated delta rule
// (delta_rule.hip) and gated linear attention (linear_attn.hip) as fp32 matrix products over chunks of 64
// rows (see chunk_state.hip for the form and the workspace layout).
//
// With decays g_t (a vector over the channels) the pair weights of a chunk are
//   sum_d k_td k_jd prod_{j < s <= t} g_sd,
// no longer a product of two numbers, and the factored form (k_t e^{G_t}) . (k_j e^{-G_j}) overflows where
// a channel forgets quickly.  So a chunk is cut into four blocks of 16 rows:
//   * block below the diagonal (I, J): prod = c_t . B_{J+1} .. B_{I-1} . u_j with c_t the product of the
//     decays of block I up to t, u_j that of block J after j, B a block's whole product.  All three are at
//     most one: the rows k_t c_t (times B's) against k_j u_j, on the matrix units.
//   * diagonal block: the product walked row by row in registers, a lane per (j, quarter of the channels).
// Nothing is divided and no logarithms are taken; what underflows is zero.
//
// Kernels:
//   channel_prep  per (chunk, head), parallel: the pair weights of q (P), the rows q_t e^{G_t}, the rows
//                 k_j e^{G_63 - G_j}, e^{G_63}; for the delta rule also the pair weights of k, their
//                 inverse and U, -W
//   chunk_carry   chunk_common.h, decays by row of the state
//   channel_out   per (chunk, head, 64 columns), parallel: o = (q e^G) S + P w
// channel_prep is bound by the vector units (the diagonal blocks) and one workgroup a CU (139 KB of LDS);
// the carry by its chain.  4096 rows, 16 heads of 128 x 128, delta rule: 173 + 156 + 46 us, the walk 2080;
// 777 rows, linear attention: 30 + 19 + 16 us, the walk 245.
#include "chunk_common.h"

namespace mx {

struct ChannelIn {
  const void *q, *k, *v;
  long q_stride, k_stride, v_stride;       // elements between rows
  int rep;                                 // heads per q / k head
  const void* g;                           // DELTA: decays fp32 [T, heads * dk]; else their pre-activation
  long g_stride;
  const float* a_bias;                     // [heads * dk] (pre-activation form)
  float inv_tau, q_scale;
  const float* beta;                       // DELTA: [T, heads]
};

// floats of dynamic LDS of channel_prep
template <int DKT>
constexpr int kPrepFloats = 3 * kC * (16 * DKT + 4) + 2 * kC * kPLD + 4 * 16 * DKT + kC;

// fragments of P: piece (row block m, key block b), lane: rows 16 m + lo, keys 16 b + 4 e + hi, e = 0 .. 3;
// of q e^G: piece (m, 16 channels i), lane: rows 16 m + lo, channels 16 i + 4 e + hi

template <int DKT, bool DELTA, typename TQ, typename TV>
__global__ void __launch_bounds__(256)
channel_prep_kernel(float* __restrict__ ws_p, float* __restrict__ ws_q, float* __restrict__ ws_k,
                    float* __restrict__ ws_g, float* __restrict__ ws_w, float* __restrict__ ws_u, ChannelIn in,
                    const int* __restrict__ start, const int* __restrict__ pos0, const int* __restrict__ slot, int heads,
                    int dk, int dv, int num_slots, int min_rows) {
  constexpr int DKP = 16 * DKT, LDK = DKP + 4, CH = DKP / 4;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float *kb = lds, *qb = kb + kC * LDK, *gb = qb + kC * LDK;       // rows of k, q, decays; later k u, q c, k c
  float *ab = gb + kC * LDK, *pb = ab + kC * kPLD;                 // pair weights of k (times beta) and of q
  float *bt = pb + kC * kPLD, *bs = bt + 4 * DKP;                  // block products, beta
  Chunk c;
  if (!find_chunk(c, blockIdx.x, blockIdx.z, start, pos0, slot, min_rows, num_slots)) return;
  const int h = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lo = lane & 15, hi = lane >> 4;
  {
    const long kh = (long)(h / in.rep) * dk;
    const TQ *qp = (const TQ*)in.q + c.row0 * in.q_stride + kh, *kp = (const TQ*)in.k + c.row0 * in.k_stride + kh;
    const TQ* gp = (const TQ*)in.g + c.row0 * in.g_stride + (long)h * dk;
#pragma unroll 4
    for (int e = tid; e < kC * DKP; e += 256) {
      const int t = e / DKP, i = e % DKP;
      float k = 0.f, q = 0.f, g = 1.f;
      if (t < c.cnt && i < dk) {
        k = ld(kp, t * in.k_stride + i);
        q = ld(qp, t * in.q_stride + i) * in.q_scale;
        g = ld(gp, t * in.g_stride + i);
        if constexpr (!DELTA) g = gla_decay(g + in.a_bias[(long)h * dk + i], in.inv_tau);
      }
      kb[t * LDK + i] = k;
      qb[t * LDK + i] = q;
      gb[t * LDK + i] = g;
    }
    if (DELTA && tid < kC) bs[tid] = tid < c.cnt ? in.beta[(c.row0 + tid) * heads + h] : 0.f;
  }
  __syncthreads();
  // diagonal blocks: lane (j = lo, channels 16 i + 4 hi + e) walks the rows after j
  {
    const int r0 = 16 * wave;
    float m[CH];
#pragma unroll
    for (int i = 0; i < CH / 4; ++i) {
      const float4 u = *reinterpret_cast<const float4*>(kb + (r0 + lo) * LDK + 16 * i + 4 * hi);
      m[4 * i] = u.x; m[4 * i + 1] = u.y; m[4 * i + 2] = u.z; m[4 * i + 3] = u.w;
    }
    for (int t = 0; t < 16; ++t) {
      float sk = 0.f, sq = 0.f;
      if (t >= lo) {
        const float *kr = kb + (r0 + t) * LDK + 4 * hi, *qr = qb + (r0 + t) * LDK + 4 * hi, *gr = gb + (r0 + t) * LDK + 4 * hi;
        float s0[4] = {0.f, 0.f, 0.f, 0.f}, s1[4] = {0.f, 0.f, 0.f, 0.f};
        const bool first = t == lo;
#pragma unroll
        for (int i = 0; i < CH / 4; ++i) {
          const float4 q4 = *reinterpret_cast<const float4*>(qr + 16 * i), g4 = *reinterpret_cast<const float4*>(gr + 16 * i);
          const float qv[4] = {q4.x, q4.y, q4.z, q4.w}, gv[4] = {g4.x, g4.y, g4.z, g4.w};
          float kv[4];
          if constexpr (DELTA) {
            const float4 k4 = *reinterpret_cast<const float4*>(kr + 16 * i);
            kv[0] = k4.x; kv[1] = k4.y; kv[2] = k4.z; kv[3] = k4.w;
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float& x = m[4 * i + e];
            x *= first ? 1.f : gv[e];
            s1[e] += qv[e] * x;
            if constexpr (DELTA) s0[e] += kv[e] * x;
          }
        }
        sq = (s1[0] + s1[1]) + (s1[2] + s1[3]);
        sk = (s0[0] + s0[1]) + (s0[2] + s0[3]);
      }
      sq = add_halves(add_row_pair(sq));
      if constexpr (DELTA) sk = add_halves(add_row_pair(sk));
      if (hi == 0) {
        pb[(r0 + t) * kPLD + r0 + lo] = sq;                       // (0 where j > t)
        if constexpr (DELTA) ab[(r0 + t) * kPLD + r0 + lo] = t > lo ? bs[r0 + t] * sk : 0.f;
      }
    }
  }
  __syncthreads();
  // per channel: products within the blocks
  for (int e = tid; e < 4 * DKP; e += 256) {
    const int d = e % DKP, r0 = 16 * (e / DKP);
    float g[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) g[t] = gb[(r0 + t) * LDK + d];
    float p = 1.f;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      p *= g[t];
      const int at = (r0 + t) * LDK + d;
      qb[at] *= p;
      if constexpr (DELTA) gb[at] = kb[at] * p;
    }
    bt[e] = p;
    p = 1.f;
#pragma unroll
    for (int t = 15; t >= 0; --t) {
      kb[(r0 + t) * LDK + d] *= p;
      p *= g[t];
    }
  }
  __syncthreads();
  const long cs = c.ws * heads + h;
  {
    float kf[4 * DKT], qf[4 * DKT];
#pragma unroll
    for (int s = 0; s < 4 * DKT; ++s) {
      qf[s] = qb[(16 * wave + lo) * LDK + 4 * s + hi];
      if constexpr (DELTA) kf[s] = gb[(16 * wave + lo) * LDK + 4 * s + hi];
    }
    for (int jt = wave - 1; jt >= 0; --jt) {
      const float* kr = kb + (16 * jt + lo) * LDK + hi;
      const f32x4 p = dot_steps<4 * DKT>([&](int s) { return qf[s]; }, [&](int s) { return kr[4 * s]; });
#pragma unroll
      for (int r = 0; r < 4; ++r) pb[(16 * wave + 4 * hi + r) * kPLD + 16 * jt + lo] = p[r];
      if constexpr (DELTA) {
        const f32x4 a = dot_steps<4 * DKT>([&](int s) { return kf[s]; }, [&](int s) { return kr[4 * s]; });
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * wave + 4 * hi + r;
          ab[i * kPLD + 16 * jt + lo] = bs[i] * a[r];
        }
      }
#pragma unroll
      for (int s = 0; s < 4 * DKT; ++s) {
        const float b = bt[jt * DKP + 4 * s + hi];
        qf[s] *= b;
        if constexpr (DELTA) kf[s] *= b;
      }
    }
    f32x4* wq = (f32x4*)ws_q + cs * (4 * DKT * 64) + wave * DKT * 64 + lane;
#pragma unroll
    for (int i = 0; i < DKT; ++i) wq[i * 64] = f32x4{qf[4 * i], qf[4 * i + 1], qf[4 * i + 2], qf[4 * i + 3]};
    if constexpr (DELTA) {
#pragma unroll
      for (int s = 0; s < 4 * DKT; ++s) gb[(16 * wave + lo) * LDK + 4 * s + hi] = kf[s];   // k e^G
    }
  }
  wave_lds_fence();
  {
    f32x4* wp = (f32x4*)ws_p + cs * (4 * 4 * 64) + wave * 4 * 64 + lane;
    for (int b = 0; b <= wave; ++b) {
      f32x4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = pb[(16 * wave + lo) * kPLD + 16 * b + 4 * e + hi];
      wp[b * 64] = x;
    }
    // k e^{G_63 - G}: tile (i, m) columns 16 i + lo, rows 16 m + 4 hi + r
    f32x4* wk = (f32x4*)ws_k + cs * (4 * DKT * 64) + lane;
    for (int e = wave; e < 4 * DKT; e += 4) {
      const int i = e / 4, m = e % 4;
      float f = 1.f;
      for (int b = m + 1; b < 4; ++b) f *= bt[b * DKP + 16 * i + lo];
      f32x4 x;
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = kb[(16 * m + 4 * hi + r) * LDK + 16 * i + lo] * f;
      wk[e * 64] = x;
    }
    if (tid < DKP) ws_g[cs * DKP + tid] = (bt[tid] * bt[DKP + tid]) * (bt[2 * DKP + tid] * bt[3 * DKP + tid]);
  }
  if constexpr (DELTA) {
    invert_unit_lower(ab, wave, lo, hi);
    // [W | U] = T [beta e^G k | beta v], column tiles dealt out to the waves (the inverse's barriers have
    // made every wave's rows of k e^G visible)
    float tf[4][16], fu[16];
    load_inverse(tf, ab, lo, hi);
#pragma unroll
    for (int s = 0; s < 16; ++s) fu[s] = bs[4 * s + hi];
    f32x4* ww = (f32x4*)ws_w + cs * (4 * DKT * 64);
    for (int ct = wave; ct < DKT; ct += 4) {
      float b[16];
      f32x4 x[4];
#pragma unroll
      for (int s = 0; s < 16; ++s) b[s] = -fu[s] * gb[(4 * s + hi) * LDK + 16 * ct + lo];
      inverse_column<true>(tf, b, x);
#pragma unroll
      for (int m = 0; m < 4; ++m) ww[(m * DKT + ct) * 64 + lane] = x[m];
    }
    const int vtiles = (dv + 15) / 16;
    f32x4* wu = (f32x4*)ws_u + cs * (long)vtiles * 256;
    for (int ct = wave; ct < vtiles; ct += 4) {
      float b[16];
      f32x4 x[4];
      const TV* vp = (const TV*)in.v + c.row0 * in.v_stride + (long)h * dv + min(16 * ct + lo, dv - 1);
#pragma unroll
      for (int s = 0; s < 16; ++s) b[s] = fu[s] * ld(vp, min(4 * s + hi, c.cnt - 1) * in.v_stride);   // beta is 0 past cnt
      inverse_column<false>(tf, b, x);
#pragma unroll
      for (int m = 0; m < 4; ++m) wu[(ct * 4 + m) * 64 + lane] = x[m];
    }
  }
}

// grid (chunks, heads * ceil(dv / 64), segments): o of the chunk's rows, wave w rows 16 w .. 16 w + 15
template <int DKT, bool DELTA, typename TV>
__global__ void __launch_bounds__(256)
channel_out_kernel(float* __restrict__ o, ChannelIn in, const float* __restrict__ ws_s, const float* __restrict__ ws_p,
                   const float* __restrict__ ws_q, const float* __restrict__ ws_u, const int* __restrict__ start,
                   const int* __restrict__ pos0, const int* __restrict__ slot, int heads, int dk, int dv, int num_slots,
                   int min_rows, int vec) {
  __shared__ __attribute__((aligned(16))) float vb[2][kC * kVLD];
  const int vt = (dv + 63) / 64;
  const int h = blockIdx.y / vt, col0 = blockIdx.y % vt * 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lo = lane & 15, hi = lane >> 4;
  Chunk c;
  if (!find_chunk(c, blockIdx.x, blockIdx.z, start, pos0, slot, min_rows, num_slots)) {
    // a padding segment's rows are zeros
    const int s = blockIdx.z, r0 = start[s], n = start[s + 1] - r0;
    if (n >= min_rows && (slot[s] < 0 || slot[s] >= num_slots))
      for (int e = tid; e < kC * 64; e += 256) {
        const int t = blockIdx.x * kC + (e >> 6), cc = col0 + (e & 63);
        if (t < n && cc < dv) o[((long)(r0 + t) * heads + h) * dv + cc] = 0.f;
      }
    return;
  }
  const long cs = c.ws * heads + h;
  const float* S = ws_s + cs * dk * (long)dv;
  const int svec = dv % 4 == 0;
  stage_cols<float>(vb[0], S, dv, min(dk, kC), col0, dv, svec);
  if constexpr (DKT > 4) stage_cols<float>(vb[1], S + (long)kC * dv, dv, dk - kC, col0, dv, svec);
  f32x4 qf[DKT], pf[4];
  {
    const f32x4* wq = (const f32x4*)ws_q + cs * (4 * DKT * 64) + wave * DKT * 64 + lane;
#pragma unroll
    for (int i = 0; i < DKT; ++i) qf[i] = wq[i * 64];
    const f32x4* wp = (const f32x4*)ws_p + cs * (4 * 4 * 64) + wave * 4 * 64 + lane;
#pragma unroll
    for (int b = 0; b < 4; ++b) pf[b] = wp[min(b, wave) * 64];
  }
  __syncthreads();
  f32x4 O[4];
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) O[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < DKT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int ct = 0; ct < 4; ++ct)
        O[ct] = mma(qf[i][e], vb[i / 4][(16 * (i % 4) + 4 * e + hi) * kVLD + 16 * ct + lo], O[ct]);
  __syncthreads();
  float* wb = vb[0];
  if constexpr (DELTA) {
    const int tiles = (dv + 15) / 16;
    const f32x4* fp = (const f32x4*)ws_u + cs * (long)tiles * 256;
    const int tile = min(col0 / 16 + wave, tiles - 1);             // columns past dv are not stored
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const f32x4 u = fp[(tile * 4 + m) * 64 + lane];
#pragma unroll
      for (int r = 0; r < 4; ++r) wb[(16 * m + 4 * hi + r) * kVLD + 16 * wave + lo] = u[r];
    }
  } else {
    stage_cols<TV>(wb, (const TV*)in.v + c.row0 * in.v_stride + (long)h * dv, in.v_stride, c.cnt, col0, dv, vec);
  }
  __syncthreads();
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    if (b > wave) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) O[ct] = mma(pf[b][e], wb[(16 * b + 4 * e + hi) * kVLD + 16 * ct + lo], O[ct]);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int t = 16 * wave + 4 * hi + r;
    if (t >= c.cnt) continue;
    float* op = o + ((c.row0 + t) * heads + h) * dv;
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
      if (col0 + 16 * ct + lo < dv) op[col0 + 16 * ct + lo] = O[ct][r];
  }
}

struct ChannelWs {
  float *s, *p, *q, *k, *g, *w, *u;
};

template <bool DELTA, typename TQ, typename TV>
int channel_run(float* o, const ChannelIn& in, const ChannelWs& ws, float* state, const int* start, const int* pos0,
                const int* slot, int num_segs, int max_rows, int heads, int dk, int dv, int num_slots, int min_rows,
                int vec, hipStream_t s) {
  const int chunks = (max_rows + kC - 1) / kC;
  const long outs = (long)heads * ((dv + 63) / 64);
  if (heads > 65535 || outs > 65535 || num_segs > 65535) return -2;
  int rc = 0;
  key_tiles(dk, [&](auto t) {
    constexpr int DKT = decltype(t)::value, lds = kPrepFloats<DKT> * 4;
    auto prep = channel_prep_kernel<DKT, DELTA, TQ, TV>;
    if constexpr (lds > 64 * 1024) {
      rc = (int)hipFuncSetAttribute(reinterpret_cast<const void*>(prep), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      if (rc != 0) return;
    }
    hipLaunchKernelGGL(prep, dim3(chunks, heads, num_segs), dim3(256), lds, s, ws.p, ws.q, ws.k, ws.g, ws.w, ws.u, in,
                       start, pos0, slot, heads, dk, dv, num_slots, min_rows);
    const dim3 cgrid(heads, (dv + 15) / 16, num_segs);
    if (dk == 16 * DKT && dv % 16 == 0)
      hipLaunchKernelGGL((chunk_carry_kernel<DKT, true, true, DELTA, TV>), cgrid, dim3(256), 0, s, ws.s, ws.w, ws.k, ws.u,
                         ws.g, (const TV*)in.v, in.v_stride, state, start, pos0, slot, heads, dk, dv, num_slots, min_rows);
    else
      hipLaunchKernelGGL((chunk_carry_kernel<DKT, false, true, DELTA, TV>), cgrid, dim3(256), 0, s, ws.s, ws.w, ws.k, ws.u,
                         ws.g, (const TV*)in.v, in.v_stride, state, start, pos0, slot, heads, dk, dv, num_slots, min_rows);
    hipLaunchKernelGGL((channel_out_kernel<DKT, DELTA, TV>), dim3(chunks, (unsigned)outs, num_segs), dim3(256), 0, s, o, in,
                       ws.s, ws.p, ws.q, ws.u, start, pos0, slot, heads, dk, dv, num_slots, min_rows, vec);
  });
  return rc != 0 ? rc : (int)hipGetLastError();
}

}  // namespace mx

using namespace mx;

// Workspaces, floats per (chunk, head): s dk dv, p 4096, q and k 64 times the padded key size, g the padded
// key size; delta rule: w as k, u 64 times dv up to a multiple of 16.
extern "C" int mx_channel_delta_chunks(float* o, const float* qn, const float* kn, const float* g, const float* beta,
                                       const void* v, int v_bf16, long v_stride, float* state, float* ws_s, float* ws_p,
                                       float* ws_q, float* ws_k, float* ws_g, float* ws_w, float* ws_u, const int* start,
                                       const int* pos0, const int* slot, int num_segs, int max_rows, int heads,
                                       int kv_heads, int dk, int dv, int num_slots, int min_rows, hipStream_t s) {
  if (num_segs <= 0 || max_rows < min_rows) return 0;
  if (dk < 1 || dk > 128 || dv < 1 || kv_heads < 1 || heads % kv_heads || min_rows < 1) return -1;
  if (((uintptr_t)ws_p | (uintptr_t)ws_q | (uintptr_t)ws_k | (uintptr_t)ws_g | (uintptr_t)ws_w | (uintptr_t)ws_u) % 16) return -3;
  ChannelIn in{};
  in.q = qn; in.k = kn; in.v = v; in.g = g;
  in.q_stride = in.k_stride = (long)kv_heads * dk;
  in.g_stride = (long)heads * dk;
  in.v_stride = v_stride;
  in.rep = heads / kv_heads;
  in.q_scale = 1.f;
  in.beta = beta;
  const ChannelWs ws{ws_s, ws_p, ws_q, ws_k, ws_g, ws_w, ws_u};
  if (v_bf16)
    return channel_run<true, float, bf16_t>(o, in, ws, state, start, pos0, slot, num_segs, max_rows, heads, dk, dv,
                                            num_slots, min_rows, 0, s);
  return channel_run<true, float, float>(o, in, ws, state, start, pos0, slot, num_segs, max_rows, heads, dk, dv, num_slots,
                                         min_rows, 0, s);
}

extern "C" int mx_channel_linear_chunks(float* o, const void* qkv, int bf16, long stride, const void* a, long a_stride,
                                        const float* a_bias, float tau, float* state, float* ws_s, float* ws_p,
                                        float* ws_q, float* ws_k, float* ws_g, const int* start, const int* pos0,
                                        const int* slot, int num_segs, int max_rows, int heads, int dk, int dv,
                                        int num_slots, int min_rows, hipStream_t s) {
  if (num_segs <= 0 || max_rows < min_rows) return 0;
  if (dk < 1 || dk > 128 || dv < 1 || heads < 1 || min_rows < 1 || !(tau > 0.f)) return -1;
  if (((uintptr_t)ws_p | (uintptr_t)ws_q | (uintptr_t)ws_k | (uintptr_t)ws_g) % 16) return -3;
  const long es = bf16 ? 2 : 4;
  ChannelIn in{};
  in.q = qkv;
  in.k = (const char*)qkv + es * heads * dk;
  in.v = (const char*)qkv + es * 2 * heads * dk;
  in.g = a;
  in.q_stride = in.k_stride = in.v_stride = stride;
  in.g_stride = a_stride;
  in.rep = 1;
  in.a_bias = a_bias;
  in.inv_tau = 1.0f / tau;
  in.q_scale = 1.0f / sqrtf((float)dk);
  const int vec = dk % 4 == 0 && dv % 4 == 0 && stride % 4 == 0 && ((uintptr_t)qkv) % (4 * es) == 0;
  const ChannelWs ws{ws_s, ws_p, ws_q, ws_k, ws_g, nullptr, nullptr};
  MX_DISPATCH_T(bf16, return (channel_run<false, T, T>(o, in, ws, state, start, pos0, slot, num_segs, max_rows, heads, dk,
                                                       dv, num_slots, min_rows, vec, s)));
}

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
//   * diagonal block: the product walked row by row in registers, a lane per (two j, sixteenth of the channels).
// Nothing is divided and no logarithms are taken; what underflows is zero.
//
// Kernels:
//   channel_prep  per (chunk, head), parallel: the pair weights of q (P), the rows q_t e^{G_t}, the rows
//                 k_j e^{G_63 - G_j}, e^{G_63}; for the delta rule also the pair weights of k, their
//                 inverse and U, -W
//   chunk_carry   chunk_common.h, decays by row of the state
//   channel_out   per (chunk, head, 64 columns), parallel: o = (q e^G) S + P w
// channel_prep is bound by its phases' latencies (loads, LDS, the inverse's substitution), which follow one
// another in the one workgroup a CU that 139 KB of LDS leave room for: hence eight waves and all of a row's
// loads in flight (four waves, loads of one entry, a key per lane on the diagonal: 174 us where this takes
// 101, and 30 where it takes 17); the carry by its chain.  4096 rows, 16 heads of 128 x 128, delta rule:
// 101 + 159 + 46 us, the walk 2080; 777 rows, linear attention: 17 + 19 + 16 us, the walk 245.
// Where no segment of a step is walked, the delta rule's rows come as the projections left them and are normed
// and their decays formed here (113 us; 129 before delta_decay, when a kernel of its own, which writes and reads them again,
// made it 101 + 56).
#include "chunk_common.h"

namespace mx {

struct ChannelIn {
  const void *q, *k, *v;
  long q_stride, k_stride, v_stride;       // elements between rows
  int rep;                                 // heads per q / k head
  const void* g;                           // pre-activations of the decays, heads * dk columns
  long g_stride;
  const float* a_bias;                     // [heads * dk]
  float inv_tau, q_scale;
  // delta rule: q and k become unit vectors (q times q_scale), decays e^{-e^{a_log} softplus}, beta a sigmoid;
  // or (a_log null) q, k, decays and beta as they stand, in fp32: where a step's short segments are walked, they
  // have been prepared for all of its rows
  const float* a_log;                      // [heads]
  const void* b;                           // (pre-activations of) beta, heads columns
  long b_stride;
};

enum ChannelRows { kLinear, kDelta, kReady };      // what channel_prep does to its rows

// floats of dynamic LDS of channel_prep
template <int DKT>
constexpr int kPrepFloats = 3 * kC * (16 * DKT + 4) + 2 * kC * kPLD + 4 * 16 * DKT + kC;

// fragments of P: piece (row block m, key block b), lane: rows 16 m + lo, keys 16 b + 4 e + hi, e = 0 .. 3;
// of q e^G: piece (m, 16 channels i), lane: rows 16 m + lo, channels 16 i + 4 e + hi

// Eight waves, two a SIMD (the LDS leaves room for one workgroup a CU): row blocks are dealt out so that
// both waves of a SIMD together have the same work whichever SIMD it is.  vec: 16-byte loads of q, k, g.
constexpr int kPrepThreads = 512;

// the value of the lane `ctrl` names (a permutation within 16 lanes)
template <int ctrl>
__device__ __forceinline__ float dpp(float x) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), ctrl, 0xf, 0xf, true));
}
constexpr int kSwap1 = 0xB1, kSwap2 = 0x4E, kHalfMirror = 0x141, kMirror = 0x140, kRor4 = 0x124, kRor8 = 0x128;

// sums over 16 lanes: a, b, c, d land in lanes 0, 1, 2, 3 (mod 4) of the sixteen
__device__ __forceinline__ float sum16(float a, float b, float c, float d, int lane) {
  const bool odd = lane & 1, two = lane & 2;
  const float ab = (odd ? b : a) + dpp<kSwap1>(odd ? a : b), cd = (odd ? d : c) + dpp<kSwap1>(odd ? c : d);
  float x = (two ? cd : ab) + dpp<kSwap2>(two ? ab : cd);
  x += dpp<kRor4>(x);
  return x + dpp<kRor8>(x);
}

// sum over LPR lanes in a row (4 to 32, a power of two)
template <int LPR>
__device__ __forceinline__ float sum_lanes(float x) {
  x += dpp<kSwap1>(x);
  x += dpp<kSwap2>(x);
  if constexpr (LPR > 4) x += dpp<kHalfMirror>(x);
  if constexpr (LPR > 8) x += dpp<kMirror>(x);
  if constexpr (LPR > 16) x = add_row_pair(x);
  return x;
}

template <int DKT, bool DELTA, typename T>
__global__ void __launch_bounds__(kPrepThreads)
channel_prep_kernel(float* __restrict__ ws_p, float* __restrict__ ws_q, float* __restrict__ ws_k,
                    float* __restrict__ ws_g, float* __restrict__ ws_w, float* __restrict__ ws_u, ChannelIn in,
                    const int* __restrict__ start, const int* __restrict__ pos0, const int* __restrict__ slot, int heads,
                    int dk, int dv, int num_slots, ChunkSteps st, int vec) {
  constexpr int DKP = 16 * DKT, LDK = DKP + 4;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float *kb = lds, *qb = kb + kC * LDK, *gb = qb + kC * LDK;       // rows of k, q, decays; later k u, q c, k c
  float *ab = gb + kC * LDK, *pb = ab + kC * kPLD;                 // pair weights of k (times beta) and of q
  float *bt = pb + kC * kPLD, *bs = bt + 4 * DKP;                  // block products, beta
  Chunk c;
  int seg, idx;
  if (!find_chunk(c, blockIdx.x / heads, st, seg, idx, start, pos0, slot, num_slots)) return;
  const int h = blockIdx.x % heads;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lo = lane & 15, hi = lane >> 4, half = wave >> 2;
  auto stage = [&](auto type, auto rows) {
    using TQ = decltype(type);
    constexpr ChannelRows R = decltype(rows)::value;
    const long kh = (long)(h / in.rep) * dk;
    const TQ *qp = (const TQ*)in.q + c.row0 * in.q_stride + kh, *kp = (const TQ*)in.k + c.row0 * in.k_stride + kh;
    const TQ* gp = (const TQ*)in.g + c.row0 * in.g_stride + (long)h * dk;
    const float* bias = in.a_bias + (long)h * dk;
    const float rate = R == kDelta ? expf(in.a_log[h]) : 0.f;
    auto decay = [&](float z, int i) {
      if constexpr (R == kReady) return z;
      else if constexpr (R == kDelta) return delta_decay(z + bias[i], rate);
      else return gla_decay(z + bias[i], in.inv_tau);
    };
    auto unit = [](float square) { return 1.0f / sqrtf(square + 1e-6f); };
    if (vec) {                                                     // dk a multiple of 4; addresses stay inside the rows
      constexpr int LPR = DKP / 4, QUADS = kC * LPR, N = (QUADS + kPrepThreads - 1) / kPrepThreads;
      float k[N][4], q[N][4], g[N][4];
      const int i = tid % LPR * 4, ic = min(i, dk - 4);            // the same columns every time
#pragma unroll
      for (int n = 0; n < N; ++n) {
        const int t = min((tid + n * kPrepThreads) / LPR, c.cnt - 1);
        load4(kp + t * in.k_stride + ic, k[n]);
        load4(qp + t * in.q_stride + ic, q[n]);
        load4(gp + t * in.g_stride + ic, g[n]);
      }
#pragma unroll
      for (int n = 0; n < N; ++n) {
        const int e = tid + n * kPrepThreads, t = e / LPR;
        if (QUADS % kPrepThreads != 0 && e >= QUADS) continue;     // (whole waves)
        const bool live = t < c.cnt && i < dk;
        float rk = 1.f, rq = in.q_scale;
        if constexpr (R == kDelta) {
          const float sk = (k[n][0] * k[n][0] + k[n][1] * k[n][1]) + (k[n][2] * k[n][2] + k[n][3] * k[n][3]);
          const float sq = (q[n][0] * q[n][0] + q[n][1] * q[n][1]) + (q[n][2] * q[n][2] + q[n][3] * q[n][3]);
          rk = unit(sum_lanes<LPR>(i < dk ? sk : 0.f));
          rq *= unit(sum_lanes<LPR>(i < dk ? sq : 0.f));
        }
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          k[n][x] = live ? k[n][x] * rk : 0.f;
          q[n][x] = live ? q[n][x] * rq : 0.f;
          g[n][x] = live ? decay(g[n][x], ic + x) : 1.f;
        }
        *reinterpret_cast<float4*>(kb + t * LDK + i) = make_float4(k[n][0], k[n][1], k[n][2], k[n][3]);
        *reinterpret_cast<float4*>(qb + t * LDK + i) = make_float4(q[n][0], q[n][1], q[n][2], q[n][3]);
        *reinterpret_cast<float4*>(gb + t * LDK + i) = make_float4(g[n][0], g[n][1], g[n][2], g[n][3]);
      }
    } else {
#pragma unroll 4
      for (int e = tid; e < kC * DKP; e += kPrepThreads) {
        const int t = e / DKP, i = e % DKP;
        float k = 0.f, q = 0.f, g = 1.f;
        if (t < c.cnt && i < dk) {
          k = ld(kp, t * in.k_stride + i);
          q = ld(qp, t * in.q_stride + i);
          g = decay(ld(gp, t * in.g_stride + i), i);
          if constexpr (R != kDelta) q *= in.q_scale;
        }
        kb[t * LDK + i] = k;
        qb[t * LDK + i] = q;
        gb[t * LDK + i] = g;
      }
      if constexpr (R == kDelta) {                                       // eight threads a row
        __syncthreads();
        float *kr = kb + (tid >> 3) * LDK, *qr = qb + (tid >> 3) * LDK, sk = 0.f, sq = 0.f;
        for (int i = tid & 7; i < DKP; i += 8) {
          sk += kr[i] * kr[i];
          sq += qr[i] * qr[i];
        }
        const float rk = unit(sum_lanes<8>(sk)), rq = unit(sum_lanes<8>(sq)) * in.q_scale;
        for (int i = tid & 7; i < DKP; i += 8) {
          kr[i] *= rk;
          qr[i] *= rq;
        }
      }
    }
    if (R != kLinear && tid < kC) {
      float x = 0.f;
      if (tid < c.cnt) {
        x = ld((const TQ*)in.b, (c.row0 + tid) * in.b_stride + h);
        if constexpr (R == kDelta) x = sigmoidf_(x);
      }
      bs[tid] = x;
    }
  };
  if constexpr (!DELTA) stage(T{}, std::integral_constant<ChannelRows, kLinear>{});
  else if (in.a_log != nullptr) stage(T{}, std::integral_constant<ChannelRows, kDelta>{});
  else stage(float{}, std::integral_constant<ChannelRows, kReady>{});
  __syncthreads();
  // diagonal blocks: wave (block, half) has the keys 8 half .. 8 half + 7 of a block and walks the rows from
  // there; a lane two keys and DKT channels, so that a row read from LDS serves two keys and sixteen lanes add up
  {
    constexpr int VW = DKT < 4 ? DKT : 4, NV = DKT / VW;
    typedef float vec_t __attribute__((ext_vector_type(VW)));
    const int r0 = 16 * (wave & 3), j0 = 8 * half + 2 * hi;        // lane's channels: VW lo + 16 VW i + e
    float m[2][DKT];
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const vec_t u = *reinterpret_cast<const vec_t*>(kb + (r0 + j0 + y) * LDK + 16 * VW * i + VW * lo);
#pragma unroll
        for (int e = 0; e < VW; ++e) m[y][VW * i + e] = u[e];
      }
    if (half == 1) pb[(r0 + (lane >> 3)) * kPLD + r0 + 8 + (lane & 7)] = 0.f;     // keys behind the rows
#pragma unroll 2
    for (int t = 8 * half; t < 16; ++t) {
      const float *kr = kb + (r0 + t) * LDK + VW * lo, *qr = qb + (r0 + t) * LDK + VW * lo, *gr = gb + (r0 + t) * LDK + VW * lo;
      float sq[2][2] = {{0.f, 0.f}, {0.f, 0.f}}, sk[2][2] = {{0.f, 0.f}, {0.f, 0.f}};
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const vec_t qv = *reinterpret_cast<const vec_t*>(qr + 16 * VW * i), gv = *reinterpret_cast<const vec_t*>(gr + 16 * VW * i);
        vec_t kv = qv;
        if constexpr (DELTA) kv = *reinterpret_cast<const vec_t*>(kr + 16 * VW * i);
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
          for (int e = 0; e < VW; ++e) {
            float& x = m[y][VW * i + e];
            x *= t > j0 + y ? gv[e] : 1.f;
            sq[y][e & 1] += qv[e] * x;
            if constexpr (DELTA) sk[y][e & 1] += kv[e] * x;
          }
      }
      const float s = sum16(sq[0][0] + sq[0][1], sk[0][0] + sk[0][1], sq[1][0] + sq[1][1], sk[1][0] + sk[1][1], lane);
      const int j = j0 + (lo >> 1);
      if (lo < 4) {
        if ((lo & 1) == 0) pb[(r0 + t) * kPLD + r0 + j] = t >= j ? s : 0.f;
        else if constexpr (DELTA) ab[(r0 + t) * kPLD + r0 + j] = t > j ? bs[r0 + t] * s : 0.f;
      }
    }
  }
  __syncthreads();
  // per channel: products within the blocks
  for (int e = tid; e < 4 * DKP; e += kPrepThreads) {
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
  // below the diagonal blocks: the first four waves the rows of q, the others (delta rule) those of k, blocks
  // in opposite order
  if (half == 0 || DELTA) {
    const int blk = half == 0 ? wave : 7 - wave;
    const float* rows = half == 0 ? qb : gb;
    float* dst = half == 0 ? pb : ab;
    float f[4 * DKT];
#pragma unroll
    for (int s = 0; s < 4 * DKT; ++s) f[s] = rows[(16 * blk + lo) * LDK + 4 * s + hi];
    for (int jt = blk - 1; jt >= 0; --jt) {
      const float* kr = kb + (16 * jt + lo) * LDK + hi;
      const f32x4 p = dot_steps<4 * DKT>([&](int s) { return f[s]; }, [&](int s) { return kr[4 * s]; });
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * blk + 4 * hi + r;
        dst[i * kPLD + 16 * jt + lo] = half == 0 ? p[r] : bs[i] * p[r];
      }
#pragma unroll
      for (int s = 0; s < 4 * DKT; ++s) f[s] *= bt[jt * DKP + 4 * s + hi];
    }
    if (half == 0) {
      f32x4* wq = (f32x4*)ws_q + cs * (4 * DKT * 64) + blk * DKT * 64 + lane;
#pragma unroll
      for (int i = 0; i < DKT; ++i) wq[i * 64] = f32x4{f[4 * i], f[4 * i + 1], f[4 * i + 2], f[4 * i + 3]};
      wave_lds_fence();
      f32x4* wp = (f32x4*)ws_p + cs * (4 * 4 * 64) + blk * 4 * 64 + lane;
      for (int b = 0; b <= blk; ++b) {
        f32x4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = pb[(16 * blk + lo) * kPLD + 16 * b + 4 * e + hi];
        wp[b * 64] = x;
      }
    } else {
#pragma unroll
      for (int s = 0; s < 4 * DKT; ++s) gb[(16 * blk + lo) * LDK + 4 * s + hi] = f[s];     // k e^G
    }
  }
  // k e^{G_63 - G}: tile (i, m) columns 16 i + lo, rows 16 m + 4 hi + r (delta rule: by the waves that have no
  // part in the inverse)
  if (half == 1 || !DELTA) {
    f32x4* wk = (f32x4*)ws_k + cs * (4 * DKT * 64) + lane;
    for (int e = DELTA ? wave - 4 : wave; e < 4 * DKT; e += DELTA ? 4 : 8) {
      const int i = e / 4, m = e % 4;
      float f = 1.f;
      for (int b = m + 1; b < 4; ++b) f *= bt[b * DKP + 16 * i + lo];
      f32x4 x;
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = kb[(16 * m + 4 * hi + r) * LDK + 16 * i + lo] * f;
      wk[e * 64] = x;
    }
    const int d = tid - 256;
    if (d >= 0 && d < DKP) ws_g[cs * DKP + d] = (bt[d] * bt[DKP + d]) * (bt[2 * DKP + d] * bt[3 * DKP + d]);
  }
  if constexpr (DELTA) {
    const int vtiles = (dv + 15) / 16;
    float vr[16];
    auto fetch_v = [&](int ct) {                                   // rows past cnt: beta is 0; columns past dv are not used
      const T* vp = (const T*)in.v + c.row0 * in.v_stride + (long)h * dv + min(16 * ct + lo, dv - 1);
#pragma unroll
      for (int s = 0; s < 16; ++s) vr[s] = ld(vp, min(4 * s + hi, c.cnt - 1) * in.v_stride);
    };
    fetch_v(wave);                                                 // on their way during the inverse
    invert_unit_lower<8>(ab, wave, lo, hi);
    // [W | U] = T [beta e^G k | beta v], column tiles dealt out to the waves (the inverse's barriers have
    // made every wave's rows of k e^G visible)
    float tf[4][16], fu[16];
    load_inverse(tf, ab, lo, hi);
#pragma unroll
    for (int s = 0; s < 16; ++s) fu[s] = bs[4 * s + hi];
    f32x4* ww = (f32x4*)ws_w + cs * (4 * DKT * 64);
    for (int ct = wave; ct < DKT; ct += 8) {
      float b[16];
      f32x4 x[4];
#pragma unroll
      for (int s = 0; s < 16; ++s) b[s] = -fu[s] * gb[(4 * s + hi) * LDK + 16 * ct + lo];
      inverse_column<true>(tf, b, x);
#pragma unroll
      for (int m = 0; m < 4; ++m) ww[(m * DKT + ct) * 64 + lane] = x[m];
    }
    f32x4* wu = (f32x4*)ws_u + cs * (long)vtiles * 256;
    for (int ct = wave; ct < vtiles; ct += 8) {
      float b[16];
      f32x4 x[4];
#pragma unroll
      for (int s = 0; s < 16; ++s) b[s] = fu[s] * vr[s];
      if (ct + 8 < vtiles) fetch_v(ct + 8);
      inverse_column<false>(tf, b, x);
#pragma unroll
      for (int m = 0; m < 4; ++m) wu[(ct * 4 + m) * 64 + lane] = x[m];
    }
  }
}

// a workgroup per chunk, head and 64 columns: o of the chunk's rows, wave w rows 16 w .. 16 w + 15
template <int DKT, bool DELTA, typename TV>
__global__ void __launch_bounds__(256)
channel_out_kernel(float* __restrict__ o, ChannelIn in, const float* __restrict__ ws_s, const float* __restrict__ ws_p,
                   const float* __restrict__ ws_q, const float* __restrict__ ws_u, const int* __restrict__ start,
                   const int* __restrict__ pos0, const int* __restrict__ slot, int heads, int dk, int dv, int num_slots,
                   ChunkSteps st, int vec) {
  __shared__ __attribute__((aligned(16))) float vb[2][kC * kVLD];
  const int vt = (dv + 63) / 64, unit = blockIdx.x % (heads * vt);
  const int h = unit / vt, col0 = unit % vt * 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lo = lane & 15, hi = lane >> 4;
  Chunk c;
  int s, idx;
  if (!find_chunk(c, blockIdx.x / (heads * vt), st, s, idx, start, pos0, slot, num_slots)) {
    if (s < 0) return;
    // a padding segment's rows are zeros
    const int r0 = start[s], n = start[s + 1] - r0;
    if (n >= st.min_rows && (slot[s] < 0 || slot[s] >= num_slots))
      for (int e = tid; e < kC * 64; e += 256) {
        const int t = idx * kC + (e >> 6), cc = col0 + (e & 63);
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
        O[ct] = mma(qf[i][e], vb[i / 4][swizzled<kVLD>(16 * (i % 4) + 4 * e + hi, 16 * ct + lo)], O[ct]);
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
      for (int r = 0; r < 4; ++r) wb[swizzled<kVLD>(16 * m + 4 * hi + r, 16 * wave + lo)] = u[r];
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
      for (int ct = 0; ct < 4; ++ct) O[ct] = mma(pf[b][e], wb[swizzled<kVLD>(16 * b + 4 * e + hi, 16 * ct + lo)], O[ct]);
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

template <bool DELTA, typename T>
int channel_run(float* o, const ChannelIn& in, const ChannelWs& ws, float* state, const int* start, const int* pos0,
                const int* slot, long rows, int num_segs, int max_rows, int heads, int dk, int dv, int num_slots, int min_rows,
                int vec, hipStream_t s) {
  const ChunkGrid g(rows, max_rows, min_rows, num_segs);
  const long outs = (long)heads * ((dv + 63) / 64);
  if (!g.fits(outs)) return -2;
  // whole quads of q, k and g at aligned addresses
  const int quads = dk % 4 == 0 && in.q_stride % 4 == 0 && in.k_stride % 4 == 0 && in.g_stride % 4 == 0 &&
                    ((uintptr_t)in.q | (uintptr_t)in.k | (uintptr_t)in.g) % (4 * (DELTA && in.a_log == nullptr ? sizeof(float) : sizeof(T))) == 0;
  int rc = 0;
  key_tiles(dk, [&](auto tiles) {
    constexpr int DKT = decltype(tiles)::value, lds = kPrepFloats<DKT> * 4;
    auto prep = channel_prep_kernel<DKT, DELTA, T>;
    if constexpr (lds > 64 * 1024) {
      rc = (int)hipFuncSetAttribute(reinterpret_cast<const void*>(prep), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      if (rc != 0) return;
    }
    hipLaunchKernelGGL(prep, g.grid(heads), dim3(kPrepThreads), lds, s, ws.p, ws.q, ws.k, ws.g, ws.w,
                       ws.u, in, start, pos0, slot, heads, dk, dv, num_slots, g.steps, quads);
    const dim3 cgrid(heads, (dv + 15) / 16, g.longs);
    if (dk == 16 * DKT && dv % 16 == 0)
      hipLaunchKernelGGL((chunk_carry_kernel<DKT, true, true, DELTA, T>), cgrid, dim3(256), 0, s, ws.s, ws.w, ws.k, ws.u,
                         ws.g, (const T*)in.v, in.v_stride, state, start, pos0, slot, heads, dk, dv, num_slots, g.steps);
    else
      hipLaunchKernelGGL((chunk_carry_kernel<DKT, false, true, DELTA, T>), cgrid, dim3(256), 0, s, ws.s, ws.w, ws.k, ws.u,
                         ws.g, (const T*)in.v, in.v_stride, state, start, pos0, slot, heads, dk, dv, num_slots, g.steps);
    hipLaunchKernelGGL((channel_out_kernel<DKT, DELTA, T>), g.grid(outs), dim3(256), 0, s, o, in,
                       ws.s, ws.p, ws.q, ws.u, start, pos0, slot, heads, dk, dv, num_slots, g.steps, vec);
  });
  return rc != 0 ? rc : (int)hipGetLastError();
}

}  // namespace mx

using namespace mx;

// Workspaces, floats per (chunk, head): s dk dv, p 4096, q and k 64 times the padded key size, g the padded
// key size; delta rule: w as k, u 64 times dv up to a multiple of 16.
// qn, kn, g, beta: the rows prepared (mx_delta_prep), or null.
extern "C" int mx_channel_delta_chunks(float* o, const float* qn, const float* kn, const float* g, const float* beta,
                                       const void* qkv, int bf16, long stride, const void* a, long a_stride,
                                       const void* b, long b_stride, const float* a_log, const float* dt_bias,
                                       float* state, float* ws_s, float* ws_p, float* ws_q, float* ws_k, float* ws_g,
                                       float* ws_w, float* ws_u, const int* start, const int* pos0, const int* slot,
                                       long rows, int num_segs, int max_rows, int heads, int kv_heads, int dk, int dv,
                                       int num_slots, int min_rows, hipStream_t s) {
  if (num_segs <= 0 || max_rows < min_rows) return 0;
  if (dk < 1 || dk > 128 || dv < 1 || kv_heads < 1 || heads % kv_heads || min_rows < 1) return -1;
  if (((uintptr_t)ws_p | (uintptr_t)ws_q | (uintptr_t)ws_k | (uintptr_t)ws_g | (uintptr_t)ws_w | (uintptr_t)ws_u) % 16) return -3;
  const long es = bf16 ? 2 : 4;
  ChannelIn in{};
  in.q = qkv;
  in.k = (const char*)qkv + es * kv_heads * dk;
  in.v = (const char*)qkv + es * 2 * kv_heads * dk;
  in.g = a;
  in.q_stride = in.k_stride = in.v_stride = stride;
  in.g_stride = a_stride;
  in.rep = heads / kv_heads;
  in.a_bias = dt_bias;
  in.q_scale = 1.0f / sqrtf((float)dk);
  in.a_log = a_log;
  in.b = b;
  in.b_stride = b_stride;
  if (qn != nullptr) {
    in.q = qn; in.k = kn; in.g = g; in.b = beta;
    in.q_stride = in.k_stride = (long)kv_heads * dk;
    in.g_stride = (long)heads * dk;
    in.b_stride = heads;
    in.a_log = nullptr;
    in.q_scale = 1.f;
  }
  const ChannelWs ws{ws_s, ws_p, ws_q, ws_k, ws_g, ws_w, ws_u};
  MX_DISPATCH_T(bf16, return (channel_run<true, T>(o, in, ws, state, start, pos0, slot, rows, num_segs, max_rows, heads, dk, dv,
                                                   num_slots, min_rows, 0, s)));
}

extern "C" int mx_channel_linear_chunks(float* o, const void* qkv, int bf16, long stride, const void* a, long a_stride,
                                        const float* a_bias, float tau, float* state, float* ws_s, float* ws_p,
                                        float* ws_q, float* ws_k, float* ws_g, const int* start, const int* pos0,
                                        const int* slot, long rows, int num_segs, int max_rows, int heads, int dk, int dv,
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
  MX_DISPATCH_T(bf16, return (channel_run<false, T>(o, in, ws, state, start, pos0, slot, rows, num_segs, max_rows, heads, dk,
                                                       dv, num_slots, min_rows, vec, s)));
}

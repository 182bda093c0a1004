// One row per sequence (decode) of a recurrent mixer in one launch, from its projection to the rows of the output product:
//   kind 0  delta rule, a decay per head and key channel: short causal convolution and silu over q, k and v, unit q and k,
//           S <- diag(g) S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q
//   kind 1  the same with one decay per head
//   kind 2  gated linear attention, no convolution: S <- diag(g) S + k v^T;  o = S^T q
// and of each, per head, out = o / rms(o) * w * sigmoid(gate), or * silu(gate).  Formulas as in delta_rule.hip, head_state.hip,
// linear_attn.hip and rows.hip, with nothing rounded between them; the history of the convolution and the state are left behind.
//
// A workgroup owns a head of a sequence, a wave 16 columns of its state, a lane four of them (16 bytes) in every 16th row: the sums
// over the rows stay in a wave, and only the head's vectors and the output's square cross it.  All loads are asked for
// before any is waited for, the projection's and the convolution's first, since they come back in order.
// Bound by the read and write of the states for many sequences, by the launch and one chain of loads for few.  In running models, 16
// heads of 128 x 128, us a layer, with a launch each for the convolution or preparation, the state and the norm with its gate
// beside it: a decay per channel, 8 sequences 9.5 (6.4 + 8.7 + 4.5); per head, 16 sequences 11.1 (6.0 + 12.0 + 4.6).
#include "mx_common.h"

namespace mx {

enum { kRowChannel = 0, kRowHead = 1, kRowLinear = 2 };
constexpr int kRsWaves = 8, kRsDv = 16 * kRsWaves, kRsMaxDk = 256, kRsTaps = 4;

struct RowStepArgs {
  void* out;                         // [T, heads * dv], dense
  const void* x;                     // rows q | k | v
  long x_stride;
  const void *a, *b, *gate;          // decay (per channel or per head) and beta before their activations; the output's gate
  long a_stride, b_stride, gate_stride;
  const float *conv_w, *a_log, *dt_bias, *norm;
  float *hist, *state;
  const int *start, *pos0, *slot;
  int heads, dk, dv, num_slots, silu;
  float eps, inv_tau;
};

// sum over the 16 lanes of a wave that share lane % 4
__device__ __forceinline__ float sum_fours(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xF, 0xF, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, true));
  return add_halves(add_row_pair(v));
}

// TAPS: of the convolution (0: none); NR: rows of the state a lane, dk <= 16 NR
template <typename T, int KIND, int TAPS, int NR>
__global__ void __launch_bounds__(64 * kRsWaves)
row_step_kernel(RowStepArgs A) {
  constexpr int NP = 16 * NR, NT = 64 * kRsWaves, CE = (2 * NP + kRsDv + NT - 1) / NT, kOld = TAPS > 1 ? TAPS - 1 : 0;
  __shared__ float q_s[NP], k_s[NP], g_s[NP], v_s[kRsDv], sq_s[kRsWaves];
  const int h = blockIdx.x, s = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = A.start[s], rows = A.start[s + 1] - row, sl = A.slot[s];
  if (rows <= 0) return;
  const int dk = A.dk, dv = A.dv, rg = lane >> 2, col = 16 * wave + 4 * (lane & 3);
  const bool live = col < dv, first = live && rg == 0;
  T* out = (T*)A.out + (long)row * A.heads * dv + (long)h * dv + col;
  if (sl < 0 || sl >= A.num_slots) {
    if (first)
#pragma unroll
      for (int j = 0; j < 4; ++j) st(out, j, 0.f);
    return;
  }
  const bool fresh = A.pos0[s] <= 0;
  const T* x = (const T*)A.x + (long)row * A.x_stride;
  const int n = 2 * dk + dv, channels = A.heads * n;
  // entry e of the head's q | k | v: its channel
  auto channel = [&](int e) {
    return e < dk ? h * dk + e : e < 2 * dk ? (A.heads - 1) * dk + h * dk + e : 2 * A.heads * dk + h * dv + e - 2 * dk;
  };
  float xin[CE], old[CE][kOld + 1], cw[CE][TAPS + 1];
  float* hist[CE];
#pragma unroll
  for (int c = 0; c < CE; ++c) {
    const int ch = channel(min(tid + c * NT, n - 1));
    xin[c] = ld(x, ch);
    if constexpr (TAPS > 0) {
      hist[c] = A.hist + (long)sl * kOld * channels + ch;
#pragma unroll
      for (int m = 0; m < kOld; ++m) old[c][m] = hist[c][(long)m * channels];
#pragma unroll
      for (int j = 0; j < TAPS; ++j) cw[c][j] = A.conv_w[(long)ch * TAPS + j];
    }
  }
  const int i0 = min(tid, dk - 1), at = KIND == kRowHead ? h : h * dk + i0;
  const float az = ld((const T*)A.a + (long)row * A.a_stride, at) + A.dt_bias[at];
  const float rate = KIND == kRowLinear ? 0.f : A.a_log[h];
  const float bz = KIND == kRowLinear ? 0.f : ld((const T*)A.b + (long)row * A.b_stride, h);
  float gz[4], nw[4];
  const int c0 = live ? col : 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    gz[j] = ld((const T*)A.gate + (long)row * A.gate_stride + (long)h * dv, c0 + j);
    nw[j] = A.norm[c0 + j];
  }
  float* S = A.state + ((long)sl * A.heads + h) * dk * dv + c0;
  float4 e[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int i = rg + 16 * r;
    e[r] = live && !fresh && i < dk ? *reinterpret_cast<const float4*>(S + (long)i * dv) : make_float4(0.f, 0.f, 0.f, 0.f);
  }

#pragma unroll
  for (int c = 0; c < CE; ++c) {
    const int i = tid + c * NT;
    float y = xin[c];
    if constexpr (TAPS > 0) {
      y = 0.f;
#pragma unroll
      for (int m = 0; m < kOld; ++m) {
        old[c][m] = fresh ? 0.f : old[c][m];
        y += old[c][m] * cw[c][m];
      }
      y += xin[c] * cw[c][TAPS - 1];
      y *= sigmoidf_(y);
      if (i < n)
#pragma unroll
        for (int m = 0; m < kOld; ++m) hist[c][(long)m * channels] = m + 1 < kOld ? old[c][m + 1] : xin[c];
    }
    if (i < dk) q_s[i] = y;
    else if (i < 2 * dk) k_s[i - dk] = y;
    else if (i < n) v_s[i - 2 * dk] = y;
  }
  if (tid < NP) {
    if (tid >= dk) q_s[tid] = 0.f, k_s[tid] = 0.f;
    g_s[tid] = KIND == kRowLinear ? gla_decay(az, A.inv_tau) : expf(-expf(rate) * softplusf_(az));
  }
  __syncthreads();
  float rq = 1.0f / sqrtf((float)dk), rk = 1.f, qk = 0.f, beta = 0.f;
  if constexpr (KIND != kRowLinear) {        // (every wave for itself)
    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int u = 0; u < (NP + 63) / 64; ++u) {
      const int i = lane + 64 * u;
      const float q = i < NP ? q_s[i] : 0.f, k = i < NP ? k_s[i] : 0.f;
      sq += q * q, sk += k * k, qk += q * k;
    }
    sq = ft::wave_sum(sq), sk = ft::wave_sum(sk), qk = ft::wave_sum(qk);
    rq *= 1.0f / sqrtf(sq + 1e-6f);
    rk = 1.0f / sqrtf(sk + 1e-6f);
    qk *= rq * rk;
    beta = sigmoidf_(bz);
  }
  float v[4], sum[4] = {0.f, 0.f, 0.f, 0.f}, del[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = v_s[c0 + j];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int i = rg + 16 * r;
    const float q = q_s[i] * rq, k = k_s[i] * rk, g = g_s[i];
    float* f = reinterpret_cast<float*>(&e[r]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (KIND == kRowLinear) {
        f[j] = g * f[j] + k * v[j];
      } else {
        f[j] *= g;
        del[j] += f[j] * k;
      }
      sum[j] += f[j] * q;
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    sum[j] = sum_fours(sum[j]);
    if constexpr (KIND != kRowLinear) {
      const float u = beta * (v[j] - sum_fours(del[j]));
#pragma unroll
      for (int r = 0; r < NR; ++r) reinterpret_cast<float*>(&e[r])[j] += k_s[rg + 16 * r] * rk * u;
      sum[j] += u * qk;
    }
  }
  if (live)
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int i = rg + 16 * r;
      if (i < dk) *reinterpret_cast<float4*>(S + (long)i * dv) = e[r];
    }
  float ss = live ? (sum[0] * sum[0] + sum[1] * sum[1]) + (sum[2] * sum[2] + sum[3] * sum[3]) : 0.f;
  ss += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(ss), 0xB1, 0xF, 0xF, true));
  ss += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(ss), 0x4E, 0xF, 0xF, true));
  if (lane == 0) sq_s[wave] = ss;
  __syncthreads();
  if (!first) return;
  ss = 0.f;
#pragma unroll
  for (int w = 0; w < kRsWaves; ++w) ss += sq_s[w];
  const float r = 1.0f / sqrtf(ss / (float)dv + A.eps);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float g = sigmoidf_(gz[j]);
    sum[j] *= r * nw[j] * (A.silu ? gz[j] * g : g);
  }
  if constexpr (sizeof(T) == 2)
    *reinterpret_cast<uint2*>(out) = make_uint2(ft::pack2(sum[0], sum[1]), ft::pack2(sum[2], sum[3]));
  else
    *reinterpret_cast<float4*>(out) = make_float4(sum[0], sum[1], sum[2], sum[3]);
}

// The same of a state-space mixer (ssd.hip): convolution with a bias and silu over x, B and C, S <- g S + B (step x)^T,
// y = S^T C + skip x, and out = y silu(z) / rms * w over a group of heads.  B and C, their history and the norm belong to a group,
// so a workgroup owns all heads of one; a wave 32 columns of one head, a lane four of them in every 8th row.
// Bound for few sequences by what one CU reads and writes (256 KB each of 4 heads of 128 x 128; the chain before the state's
// loads arrive, convolution and history, costs nothing when it is asked for first: 13.5 us with the compiler's order), for many by
// the states' bytes.  In running models, 32 heads of 128 x 128 in 8 groups, us a layer at 1 / 8 / 16 / 32 / 48 / 64 sequences:
// 11.8 14.6 17.8 27 45 52, with a launch each for convolution, state and norm 15.7 21 27 40 57 69.
constexpr int kGsWaves = 16, kGsCols = 32, kGsMaxDk = 128;

struct GroupStepArgs {
  void* out;                         // [T, heads * dv], dense
  const void *x, *z, *dt;            // rows x (heads * dv) | B | C (groups * dk each); the gate; steps, one a head
  long x_stride, z_stride, dt_stride;
  const float *conv_w, *conv_b, *a_log, *dt_bias, *skip, *norm;      // conv_b may be null
  float *hist, *state;
  const int *start, *pos0, *slot;
  int heads, groups, dk, dv, num_slots;
  float eps;
};

// NR: rows of the state a lane, dk <= 8 NR (FULL: dk = 8 NR)
template <typename T, int TAPS, int NR, bool FULL>
__global__ void __launch_bounds__(64 * kGsWaves)
group_step_kernel(GroupStepArgs A) {
  constexpr int kOld = TAPS - 1;
  __shared__ float x_s[kGsWaves * kGsCols], b_s[kGsMaxDk], c_s[kGsMaxDk], sq_s[kGsWaves];
  const int grp = blockIdx.x, s = blockIdx.y, tid = threadIdx.x, lane = tid & 63, waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = A.start[s], rows = A.start[s + 1] - row, sl = A.slot[s];
  if (rows <= 0) return;
  const int dk = A.dk, dv = A.dv, gs = waves * kGsCols, inner = A.heads * dv, rg = lane >> 3;
  const int col = wave * kGsCols + 4 * (lane & 7), hd = wave * kGsCols / dv, h = grp * (A.heads / A.groups) + hd;
  T* out = (T*)A.out + (long)row * inner + (long)grp * gs + col;
  if (sl < 0 || sl >= A.num_slots) {
    if (rg == 0)
#pragma unroll
      for (int j = 0; j < 4; ++j) st(out, j, 0.f);
    return;
  }
  const bool fresh = A.pos0[s] <= 0;
  // entry e of the group's x | B | C: its channel, a thread each (2 dk <= gs)
  const int n = gs + 2 * dk, channels = inner + 2 * A.groups * dk, e = min(tid, n - 1);
  const int ch = e < gs ? grp * gs + e : e < gs + dk ? inner + grp * dk + e - gs : inner + (A.groups + grp - 1) * dk + e - gs;
  const T xr = ((const T*)A.x + (long)row * A.x_stride)[ch];       // (widened behind the state's loads)
  float* hist = A.hist + (long)sl * kOld * channels + ch;
  float old[kOld], cw[TAPS];
#pragma unroll
  for (int m = 0; m < kOld; ++m) old[m] = hist[(long)m * channels];
#pragma unroll
  for (int j = 0; j < TAPS; ++j) cw[j] = A.conv_w[(long)ch * TAPS + j];
  const float cb = (A.conv_b != nullptr ? A.conv_b : A.conv_w)[ch];
  const T dr = ((const T*)A.dt + (long)row * A.dt_stride)[h];
  float bias = A.dt_bias[h], rate = A.a_log[h], skip = A.skip[h];
  float nw[4];
  T zr[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    zr[j] = ((const T*)A.z + (long)row * A.z_stride + (long)grp * gs)[col + j];
    nw[j] = A.norm[(long)grp * gs + col + j];
  }
  float* S = A.state + ((long)sl * A.heads + h) * dk * dv + (col - hd * dv);
  float4 st_[NR];
  // (the compiler would move the loads before this behind the state's, to where they are used)
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int r = 0; r < NR; ++r) st_[r] = *reinterpret_cast<const float4*>(S + (long)(FULL ? rg + 8 * r : min(rg + 8 * r, dk - 1)) * dv);
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" : "+s"(bias), "+s"(rate), "+s"(skip));
#pragma unroll
  for (int m = 0; m < kOld; ++m) asm volatile("" : "+v"(old[m]));

  const float xin = ld(&xr, 0), dz = ld(&dr, 0);
  float y = 0.f;
#pragma unroll
  for (int m = 0; m < kOld; ++m) {
    old[m] = fresh ? 0.f : old[m];
    y += old[m] * cw[m];
  }
  y += xin * cw[TAPS - 1];
  if (A.conv_b != nullptr) y += cb;
  y *= sigmoidf_(y);
  if (tid < n) {
#pragma unroll
    for (int m = 0; m < kOld; ++m) hist[(long)m * channels] = m + 1 < kOld ? old[m + 1] : xin;
    if (tid < gs) x_s[tid] = y;
    else if (tid < gs + dk) b_s[tid - gs] = y;
    else c_s[tid - gs - dk] = y;
  }
  const float step = softplusf_(dz + bias), decay = expf(-expf(rate) * step);
  __syncthreads();
  float v[4], sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = x_s[col + j];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int i = rg + 8 * r;
    const bool in = FULL || i < dk;
    const float b = in ? b_s[min(i, kGsMaxDk - 1)] : 0.f, c = in ? c_s[min(i, kGsMaxDk - 1)] : 0.f;
    float* f = reinterpret_cast<float*>(&st_[r]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f[j] = (fresh || !in ? 0.f : decay * f[j]) + b * (step * v[j]);
      sum[j] += f[j] * c;
    }
    if (in) *reinterpret_cast<float4*>(S + (long)i * dv) = st_[r];
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    sum[j] = ft::kgroups_sum(sum[j] + __shfl_xor(sum[j], 8)) + skip * v[j];
    const float gz = ld(&zr[j], 0);
    sum[j] *= gz * sigmoidf_(gz);
    ss += sum[j] * sum[j];
  }
  ss += __shfl_xor(ss, 1);
  ss += __shfl_xor(ss, 2);
  ss += __shfl_xor(ss, 4);
  if (lane == 0) sq_s[wave] = ss;
  __syncthreads();
  if (rg != 0) return;
  ss = 0.f;
  for (int w = 0; w < waves; ++w) ss += sq_s[w];
  const float r = 1.0f / sqrtf(ss / (float)gs + A.eps);
#pragma unroll
  for (int j = 0; j < 4; ++j) sum[j] *= r * nw[j];
  if constexpr (sizeof(T) == 2)
    *reinterpret_cast<uint2*>(out) = make_uint2(ft::pack2(sum[0], sum[1]), ft::pack2(sum[2], sum[3]));
  else
    *reinterpret_cast<float4*>(out) = make_float4(sum[0], sum[1], sum[2], sum[3]);
}

}  // namespace mx

using namespace mx;

// whether group_step_kernel takes the sizes: a group's heads in one workgroup, no wave's columns in two of them
extern "C" int mx_group_step_fits(int taps, int heads, int groups, int dk, int dv) {
  if (groups < 1 || heads < groups || heads % groups || dk < 1 || dv < kGsCols || dv % kGsCols) return 0;
  const long gs = (long)(heads / groups) * dv;
  return gs <= kGsWaves * kGsCols && dk <= kGsMaxDk && 2 * dk <= gs && taps >= 2 && taps <= kRsTaps;
}

// out and state at 16-byte addresses; every segment has one row at most
extern "C" int mx_group_step(void* out, int bf16, const void* x, long x_stride, const void* z, long z_stride, const void* dt,
                             long dt_stride, const float* conv_w, const float* conv_b, int taps, float* hist, const float* a_log,
                             const float* dt_bias, const float* skip, const float* norm, float eps, float* state,
                             const int* start, const int* pos0, const int* slot, int num_segs, int heads, int groups, int dk,
                             int dv, int num_slots, hipStream_t s) {
  if (num_segs <= 0) return 0;
  if (!mx_group_step_fits(taps, heads, groups, dk, dv)) return -1;
  if ((((uintptr_t)out) | ((uintptr_t)state)) % 16 || num_segs > 65535) return -2;
  const GroupStepArgs A{out, x, z, dt, x_stride, z_stride, dt_stride, conv_w, conv_b, a_log, dt_bias, skip, norm, hist, state,
                        start, pos0, slot, heads, groups, dk, dv, num_slots, eps};
  const dim3 grid((unsigned)groups, (unsigned)num_segs), block((unsigned)(64 * (heads / groups * dv / kGsCols)));
#define MX_GS(TAPS, NR)                                                                                                       \
  do {                                                                                                                        \
    if (dk == 8 * NR) MX_DISPATCH_T(bf16, hipLaunchKernelGGL((group_step_kernel<T, TAPS, NR, true>), grid, block, 0, s, A));   \
    else MX_DISPATCH_T(bf16, hipLaunchKernelGGL((group_step_kernel<T, TAPS, NR, false>), grid, block, 0, s, A));               \
  } while (0)
#define MX_GS_DK(TAPS)                \
  do {                                \
    if (dk <= 32) MX_GS(TAPS, 4);     \
    else if (dk <= 64) MX_GS(TAPS, 8); \
    else MX_GS(TAPS, 16);             \
  } while (0)
  if (taps == 4) MX_GS_DK(4);
  else if (taps == 3) MX_GS_DK(3);
  else MX_GS_DK(2);
#undef MX_GS_DK
#undef MX_GS
  return (int)hipGetLastError();
}

// whether the kernel takes the sizes: whole fours of columns that one workgroup holds, a convolution of two to four taps (kind 2: none)
extern "C" int mx_row_step_fits(int kind, int taps, int dk, int dv) {
  return dk >= 1 && dk <= kRsMaxDk && dv >= 4 && dv <= kRsDv && dv % 4 == 0 && (kind == kRowLinear ? taps == 0 : taps >= 2 && taps <= kRsTaps);
}

// out and state at 16-byte addresses; every segment has one row at most
extern "C" int mx_row_step(int kind, void* out, int bf16, const void* x, long x_stride, const void* a, long a_stride, const void* b,
                           long b_stride, const void* gate, long gate_stride, const float* conv_w, int taps, float* hist,
                           const float* a_log, const float* dt_bias, float inv_tau, const float* norm, float eps, int silu,
                           float* state, const int* start, const int* pos0, const int* slot, int num_segs, int heads, int dk,
                           int dv, int num_slots, hipStream_t s) {
  if (num_segs <= 0) return 0;
  if (!mx_row_step_fits(kind, taps, dk, dv) || heads < 1 || kind < 0 || kind > kRowLinear) return -1;
  if ((((uintptr_t)out) | ((uintptr_t)state)) % 16 || num_segs > 65535) return -2;
  const RowStepArgs A{out, x, x_stride, a, b, gate, a_stride, b_stride, gate_stride, conv_w, a_log, dt_bias, norm, hist, state,
                      start, pos0, slot, heads, dk, dv, num_slots, silu, eps, inv_tau};
  const dim3 grid((unsigned)heads, (unsigned)num_segs);
#define MX_RS(KIND, TAPS, NR) \
  MX_DISPATCH_T(bf16, hipLaunchKernelGGL((row_step_kernel<T, KIND, TAPS, NR>), grid, dim3(64 * kRsWaves), 0, s, A))
#define MX_RS_DK(KIND, TAPS)               \
  do {                                     \
    if (dk <= 32) MX_RS(KIND, TAPS, 2);    \
    else if (dk <= 64) MX_RS(KIND, TAPS, 4); \
    else if (dk <= 128) MX_RS(KIND, TAPS, 8); \
    else MX_RS(KIND, TAPS, 16);            \
  } while (0)
#define MX_RS_CONV(KIND)                   \
  do {                                     \
    if (taps == 4) MX_RS_DK(KIND, 4);      \
    else if (taps == 3) MX_RS_DK(KIND, 3); \
    else MX_RS_DK(KIND, 2);                \
  } while (0)
  if (kind == kRowChannel) MX_RS_CONV(kRowChannel);
  else if (kind == kRowHead) MX_RS_CONV(kRowHead);
  else MX_RS_DK(kRowLinear, 0);
#undef MX_RS_CONV
#undef MX_RS_DK
#undef MX_RS
  return (int)hipGetLastError();
}

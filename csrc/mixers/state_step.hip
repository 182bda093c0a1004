// One row per sequence (decode) of the recurrences over fp32 state slots: the gated delta rule with a decay per
// head and key channel (delta_rule.hip), gated linear attention (linear_attn.hip) and the state-space scan
// (ssd.hip), whose walks over longer segments stay there.  Formulas as there; S is [dk, dv] per head:
//   delta:   S <- diag(g) S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q, as  S_g^T q + u (q . k)
//   linear:  S <- diag(g) S + k v^T;  o = S^T q
//   scan:    S <- g S + B (step x)^T;  y = S^T C + skip x
// A workgroup owns 32 columns of one head of one sequence: a thread four neighbouring columns (16 bytes) of every
// 32nd row, all loads in flight before the head's vectors are prepared (so no launch and no fp32 copies for
// those), both dot products of the delta rule in one reduction.
// Bound by the read and write of the states.  In running models: delta rule, 16 heads of 128 x 128, 64 sequences
// 33 us (134 MB: 4.1 TB/s), 8 sequences 8.4; linear attention, same heads, 32 sequences 14, one 5; scan, 32 heads of
// 128 x 128, 32 sequences 28, one 5.5.  The walks, whose lanes read a column's rows and not a row's columns, with
// the launch that prepared the vectors: 103, 22; 48, 7; 77, 7.
#include "mx_common.h"

namespace mx {

enum { kStepDelta = 0, kStepLinear = 1, kStepScan = 2 };
constexpr int kStepCols = 32, kStepRows = 32, kStepMaxDk = 256;

struct StepArgs {
  float* o;
  const void* x;
  long x_stride;
  const void *a, *b;                 // decay (per channel or per head) and beta before their activations
  long a_stride, b_stride;
  const float *a_log, *dt_bias, *skip;
  float inv_tau;
  float* state;
  const int *start, *pos0, *slot;
  int heads, kv_heads, dk, dv, num_slots;
};

template <typename T, int KIND, int NR>
__global__ void __launch_bounds__(256)
state_step_kernel(StepArgs A) {
  __shared__ float q_s[kStepRows * NR], k_s[kStepRows * NR], g_s[kStepRows * NR], norm[4][3], red[4][8][8];
  const int s = blockIdx.z, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int row = A.start[s], rows = A.start[s + 1] - row, sl = A.slot[s];
  if (rows <= 0) return;
  const int dk = A.dk, dv = A.dv, heads = A.heads, c4 = tid & 7, rg = tid >> 3;
  const int col = blockIdx.x * kStepCols + 4 * c4;
  const bool live = col < dv;
  float* out = A.o + (long)row * heads * dv + (long)h * dv + col;
  if (sl < 0 || sl >= A.num_slots) {
    if (live && rg == 0) *reinterpret_cast<float4*>(out) = make_float4(0.f, 0.f, 0.f, 0.f);
    return;
  }
  float* S = A.state + ((long)sl * heads + h) * dk * dv + col;
  const bool load = live && A.pos0[s] > 0;
  float4 st_[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int i = rg + kStepRows * r;
    st_[r] = load && i < dk ? *reinterpret_cast<const float4*>(S + (long)i * dv) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  const T* x = (const T*)A.x + (long)row * A.x_stride;
  const T* a = (const T*)A.a + (long)row * A.a_stride;
  const int kh = h / (heads / A.kv_heads);
  long q0, k0, v0;
  if constexpr (KIND == kStepDelta) {
    q0 = (long)kh * dk, k0 = q0 + (long)A.kv_heads * dk, v0 = 2L * A.kv_heads * dk + (long)h * dv;
  } else if constexpr (KIND == kStepLinear) {
    q0 = (long)h * dk, k0 = q0 + (long)heads * dk, v0 = 2L * heads * dk + (long)h * dv;
  } else {
    k0 = (long)heads * dv + (long)kh * dk, q0 = k0 + (long)A.kv_heads * dk, v0 = (long)h * dv;
  }
  float v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = live ? ld(x, v0 + col + j) : 0.f;

  // the head's vectors, a thread an entry
  float sq = 0.f, sk = 0.f, qk = 0.f;
  if (tid < kStepRows * NR) {
    const int i = tid;
    float q = 0.f, k = 0.f, g = 0.f;
    if (i < dk) {
      q = ld(x, q0 + i), k = ld(x, k0 + i);
      if constexpr (KIND == kStepDelta)
        g = expf(-expf(A.a_log[h]) * softplusf_(ld(a, (long)h * dk + i) + A.dt_bias[(long)h * dk + i]));
      else if constexpr (KIND == kStepLinear)
        g = gla_decay(ld(a, (long)h * dk + i) + A.dt_bias[(long)h * dk + i], A.inv_tau);
    }
    q_s[i] = q, k_s[i] = k, g_s[i] = g;
    sq = q * q, sk = k * k, qk = q * k;
  }
  float rq = 1.f, rk = 1.f, beta = 0.f, decay = 0.f;
  if constexpr (KIND == kStepDelta) {
    sq = ft::wave_sum(sq), sk = ft::wave_sum(sk), qk = ft::wave_sum(qk);
    if (lane == 0) norm[wave][0] = sq, norm[wave][1] = sk, norm[wave][2] = qk;
    beta = sigmoidf_(ld((const T*)A.b, (long)row * A.b_stride + h));
  } else if constexpr (KIND == kStepLinear) {
    rq = 1.0f / sqrtf((float)dk);
  } else {
    const float step = softplusf_(ld(a, h) + A.dt_bias[h]);
    decay = expf(-expf(A.a_log[h]) * step);
    beta = step;
  }
  __syncthreads();
  if constexpr (KIND == kStepDelta) {
    sq = norm[0][0] + norm[1][0] + norm[2][0] + norm[3][0];
    sk = norm[0][1] + norm[1][1] + norm[2][1] + norm[3][1];
    rq = 1.0f / sqrtf(sq + 1e-6f) * (1.0f / sqrtf((float)dk));
    rk = 1.0f / sqrtf(sk + 1e-6f);
    qk = (norm[0][2] + norm[1][2] + norm[2][2] + norm[3][2]) * rq * rk;
  }
  constexpr int NS = KIND == kStepDelta ? 8 : 4;
  float sum[NS];
#pragma unroll
  for (int j = 0; j < NS; ++j) sum[j] = 0.f;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int i = rg + kStepRows * r;
    const float q = q_s[i] * rq, k = k_s[i] * rk, g = KIND == kStepScan ? decay : g_s[i];
    float* e = reinterpret_cast<float*>(&st_[r]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (KIND == kStepDelta) {
        e[j] *= g;
        sum[4 + j] += e[j] * k;
      } else {
        e[j] = g * e[j] + k * (KIND == kStepScan ? beta * v[j] : v[j]);
      }
      sum[j] += e[j] * q;
    }
  }
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    sum[j] = ft::kgroups_sum(sum[j] + __shfl_xor(sum[j], 8));
    if (lane < 8) red[wave][lane][j] = sum[j];
  }
  if constexpr (KIND != kStepDelta) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int i = rg + kStepRows * r;
      if (live && i < dk) *reinterpret_cast<float4*>(S + (long)i * dv) = st_[r];
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NS; ++j) sum[j] = (red[0][c4][j] + red[1][c4][j]) + (red[2][c4][j] + red[3][c4][j]);
  if (!live) return;
  if constexpr (KIND == kStepDelta) {
    float u[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) u[j] = beta * (v[j] - sum[4 + j]);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const int i = rg + kStepRows * r;
      if (i >= dk) continue;
      const float k = k_s[i] * rk;
      *reinterpret_cast<float4*>(S + (long)i * dv) = make_float4(st_[r].x + k * u[0], st_[r].y + k * u[1],
                                                                 st_[r].z + k * u[2], st_[r].w + k * u[3]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) sum[j] += u[j] * qk;
  } else if constexpr (KIND == kStepScan) {
    const float skip = A.skip[h];
#pragma unroll
    for (int j = 0; j < 4; ++j) sum[j] += skip * v[j];
  }
  if (rg == 0) *reinterpret_cast<float4*>(out) = make_float4(sum[0], sum[1], sum[2], sum[3]);
}

}  // namespace mx

using namespace mx;

// rows of 16-byte pieces of the states
extern "C" int mx_state_step_fits(const float* o, const float* state, int dk, int dv) {
  return dk >= 1 && dk <= kStepMaxDk && dv % 4 == 0 && (((uintptr_t)o) | ((uintptr_t)state)) % 16 == 0;
}

// kind 0: delta rule (x: q | k | v), 1: linear attention (x: q | k | v), 2: scan (x: v | B | C, kv_heads: groups);
// every segment has one row at most
extern "C" int mx_state_step(int kind, float* o, const void* x, int bf16, long x_stride, const void* a, long a_stride,
                             const void* b, long b_stride, const float* a_log, const float* dt_bias, const float* skip,
                             float inv_tau, float* state, const int* start, const int* pos0, const int* slot,
                             int num_segs, int heads, int kv_heads, int dk, int dv, int num_slots, hipStream_t s) {
  if (num_segs <= 0) return 0;
  if (!mx_state_step_fits(o, state, dk, dv) || heads < 1 || kv_heads < 1 || heads % kv_heads || kind < 0 || kind > 2)
    return -1;
  const dim3 grid((dv + kStepCols - 1) / kStepCols, heads, num_segs);
  if (grid.z > 65535 || grid.y > 65535) return -2;
  const StepArgs A{o, x, x_stride, a, b, a_stride, b_stride, a_log, dt_bias, skip, inv_tau, state, start, pos0, slot,
                   heads, kv_heads, dk, dv, num_slots};
#define MX_STEP_R(KIND, NR) \
  MX_DISPATCH_T(bf16, hipLaunchKernelGGL((state_step_kernel<T, KIND, NR>), grid, dim3(256), 0, s, A))
#define MX_STEP(KIND)                       \
  do {                                      \
    if (dk <= 32) MX_STEP_R(KIND, 1);       \
    else if (dk <= 64) MX_STEP_R(KIND, 2);  \
    else if (dk <= 128) MX_STEP_R(KIND, 4); \
    else MX_STEP_R(KIND, 8);                \
  } while (0)
  if (kind == kStepDelta) MX_STEP(kStepDelta);
  else if (kind == kStepLinear) MX_STEP(kStepLinear);
  else MX_STEP(kStepScan);
#undef MX_STEP
#undef MX_STEP_R
  return (int)hipGetLastError();
}

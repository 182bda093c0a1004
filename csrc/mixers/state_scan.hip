// The selective state-space scan's long segments with bf16 rows and 128 state entries, in chunks of 64 rows (chunk_state.hip has the
// form): the chunks' pair weights at once (state_pairs), then a workgroup per (head, 16 columns of the state, segment) that walks
// its chunks with the state in registers (state_scan).
//
// Rows of bf16 are operands of the bf16 matrix units as they are, and what is fp32 is the exact sum of three bf16 parts: q . k is one
// product, q . S and (pair weights) . v are three, where the fp32 units take sixteen times as long for each.  So cheap, neither
// a chunk's own contribution to the state nor its incoming state goes through memory, which is what the chunk-parallel form is
// bound by (state_add, state_carry and chunk_out of 2048 rows, 32 heads of 128 x 128: 44 + 30 + 78 us, 67 MB written, read, written
// and read again); the weights are 18 KB a chunk and head.
//
// state_scan: waves 4 .. 7 hold the state, 32 rows each, and make the next chunk's of it; waves 0 .. 3 the outputs of 16 rows each,
// from the state's parts that the others left in LDS; waves 8 .. 11 bring rows, and scale and split v.  A barrier a chunk: while one's
// outputs are formed, the state of the next is, and the chunks after that are on their way.  Bound by the state's chain and the
// issue of all of them: 1.4 us a chunk; those 2048 rows take 59 us back to back, 15 + 50 in a model's pass.  (All of it in one launch,
// weights and sums of decays by other waves of the same workgroup, which every 16 columns repeat: 87 us; by the output waves: 86 to 97.)
//
// A value of v that is not finite reaches its own row and later ones only: a weight of 0 would take it to the rows before it in its block of
// 16, so blocks with such a value (`loose`) have them apart from the products (2048 rows 58.8 us so and 59.3
// without, 777 30.9 and 30.1, 2000 of 8 heads, a chain that leaves most of the chip idle, 49.0 and 47.0).
//
// Operand layouts (v_mfma_f32_16x16x32_bf16): lane (hi, lo) = (lane / 16, lane % 16) holds row or column lo, inner entries 8 hi ..
// 8 hi + 7; accumulators hold row 4 hi + r, column lo.  Sums over rows j take j in the order in which accumulators lie, entry i < 4
// of (hi) row 4 hi + i of a tile of 16, i >= 4 of the next one.
#include "chunk_common.h"

namespace mx {

typedef __bf16 ss_bf16x8 __attribute__((ext_vector_type(8)));
typedef short ss_i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) ss_i16x4 ss_lds_i16x4;

__device__ __forceinline__ f32x4 ss_mma(const uint4& a, const uint4& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ss_bf16x8, a), __builtin_bit_cast(ss_bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ uint2 ss_read_tr(const char* p) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((ss_lds_i16x4*)p));
}
__device__ __forceinline__ void ss_split(float a, float b, float c, float d, uint2 (&p)[3]) {
  split_any_bf16x3(a, b, p[0].x, p[1].x, p[2].x);
  split_any_bf16x3(c, d, p[0].y, p[1].y, p[2].y);
}
// which of two bf16 are infinite or NaN: in the bits of their signs alone, and as 0xffff of theirs
__device__ __forceinline__ uint32_t ss_loose(uint32_t u) { return (u & 0x7f807f80u) + 0x00800080u; }
__device__ __forceinline__ uint32_t ss_not_finite(uint32_t u) { return (ss_loose(u) >> 15 & 0x00010001u) * 0xffffu; }
// e^x of a sum of log decays, x <= 0, within 2 units in the last place of fp32 (which are larger below its smallest normal number)
__device__ __forceinline__ float ss_exp(double x) {
  constexpr float kL = 1.4426950408889634f, kLo = 1.925963033500e-8f, kLn2 = 0.6931471805599453f;
  x = x < -200.0 ? -200.0 : x;                     // (a NaN stays one)
  const float y = (float)x, rest = (float)(x - (double)y), t = y * kL;
  const int down = t < -100.0f ? 64 : 0;           // (exp2 has no denormal results)
  const float r = __builtin_amdgcn_exp2f(t + (float)down);
  // what t dropped of x in units of log2; the sum with `down` is exact
  const float low = fmaf(rest, kL, fmaf(y, kLo, fmaf(y, kL, -t)));
  return ldexpf(fmaf(r * kLn2, low, r), -down);
}

constexpr int kSsKeys = 128, kSsCols = 16;

struct ScanIn {
  const bf16_t *q, *k, *v;             // rows; head h's columns at h / rep * kSsKeys (q, k) and h * dv (v)
  long stride;
  int rep;
  const bf16_t* dt;                    // step pre-activations
  long dt_stride;
  const float *a_log, *dt_bias, *skip; // [heads]
};

// a chunk and head's workspace: the pair weights as right operands, six pieces of 32 rows j (block of rows 0, 1: one each; 2, 3: two)
// of three parts; then, per row, e^{G_t} and (step e^{G_63 - G_t}), and e^{G_63}
constexpr int kSsPairs = 6 * 3 * 64 * 4, kSsFloats = kSsPairs + 2 * kC + 4;
__device__ __forceinline__ int ss_piece(int block, int p, int z) { return ((block < 2 ? block : 2 * block - 2 + p) * 3 + z) * 64; }

// ---------------------------------------------------------------------------------
// a workgroup per chunk and head: pair weights e^{G_t - G_j} step_j (q_t . k_j), j <= t, wave w rows 16 w ..; sums of decays
// ---------------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
state_pairs_kernel(float* __restrict__ ws, ScanIn in, const int* __restrict__ start, const int* __restrict__ pos0,
                   const int* __restrict__ slot, int heads, int num_slots, ChunkSteps st) {
  __shared__ double G[kC];
  __shared__ float step[kC];
  Chunk c;
  int seg, idx;
  if (!find_chunk(c, blockIdx.x / heads, st, seg, idx, start, pos0, slot, num_slots)) return;
  const int h = blockIdx.x % heads, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lo = lane & 15, hi = lane >> 4;
  const long at = c.row0 * in.stride + (long)(h / in.rep) * kSsKeys + 8 * hi;
  uint4 q[4], k[4][4];
  {
    const bf16_t* p = in.q + at + (long)min(16 * wave + lo, c.cnt - 1) * in.stride;
#pragma unroll
    for (int x = 0; x < 4; ++x) q[x] = *reinterpret_cast<const uint4*>(p + 32 * x);
  }
#pragma unroll
  for (int J = 0; J < 4; ++J) {
    if (J > wave) continue;
    const bf16_t* p = in.k + at + (long)min(16 * J + lo, c.cnt - 1) * in.stride;
#pragma unroll
    for (int x = 0; x < 4; ++x) k[J][x] = *reinterpret_cast<const uint4*>(p + 32 * x);
  }
  float* const out = ws + (c.ws * heads + h) * (long)kSsFloats;
  if (wave == 0) {
    // sums of log decays in double precision (their differences are rounded, not they), a row a lane
    const int t = lane;
    const bool live = t < c.cnt;
    const float s = softplusf_(ld(in.dt, (c.row0 + min(t, c.cnt - 1)) * in.dt_stride + h) + in.dt_bias[h]), lf = -expf(in.a_log[h]) * s;
    double g = live ? (double)(lf < -3e38f ? -3e38f : lf) : 0.0;             // (subtracted: -inf would become NaN)
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const double u = __shfl_up(g, off, 64);
      if (t >= off) g += u;
    }
    G[t] = g;
    const float w = live ? s : 0.f;
    step[t] = w;
    const double last = __shfl(g, 63, 64);
    out[kSsPairs + t] = ss_exp(g);
    out[kSsPairs + kC + t] = ss_exp(last - g) * w;
    if (t == 0) out[kSsPairs + 2 * kC] = ss_exp(last);
  }
  __syncthreads();
  const int t = 16 * wave + lo;
  const double gt = G[t];
  uint4* const pieces = (uint4*)out + lane;
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    if (2 * p > wave) continue;
    uint2 half[2][3];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int J = 2 * p + e;
      if (J > wave) {                              // (a block behind all rows: no weights)
#pragma unroll
        for (int z = 0; z < 3; ++z) half[e][z] = uint2{0, 0};
        continue;
      }
      f32x4 a[4];                                  // (four sums: nearer than one)
#pragma unroll
      for (int x = 0; x < 4; ++x) a[x] = ss_mma(k[J][x], q[x], f32x4{0.f, 0.f, 0.f, 0.f});
      f32x4 w = (a[0] + a[1]) + (a[2] + a[3]);
      const int j0 = 16 * J + 4 * hi;
#pragma unroll
      for (int r = 0; r < 4; ++r) w[r] = j0 + r <= t ? w[r] * (ss_exp(gt - G[j0 + r]) * step[j0 + r]) : 0.f;
      ss_split(w[0], w[1], w[2], w[3], half[e]);
    }
#pragma unroll
    for (int z = 0; z < 3; ++z)
      pieces[ss_piece(wave, p, z)] = make_uint4(half[0][z].x, half[0][z].y, half[1][z].x, half[1][z].y);
  }
}

// ---------------------------------------------------------------------------------
// grid (heads, dv / 16, long segments)
// ---------------------------------------------------------------------------------
constexpr int kSsThreads = 768;

__global__ void __launch_bounds__(kSsThreads, 3)
state_scan_kernel(float* __restrict__ o, const float* __restrict__ ws, ScanIn in, float* __restrict__ state,
                  const int* __restrict__ start, const int* __restrict__ pos0, const int* __restrict__ slot, int heads, int dv,
                  int num_slots, ChunkSteps st) {
  // rows of k: 16 pieces of 16 bytes, piece p of row j at p ^ (j & 15); of v: 32 bytes; three chunks of them
  __shared__ __attribute__((aligned(16))) char ks[3][kC * 256], vs[3][kC * 32];
  __shared__ __attribute__((aligned(16))) uint2 parts[2][3][4][64][2];       // the state's, as left operands (columns) of q . S
  __shared__ __attribute__((aligned(16))) uint4 scaled[2][2][3][64];         // step e^{G_63 - G_j} v_j's, as right operands (columns)
  __shared__ uint32_t loose[3][4];                      // lanes with a value of v that is not finite, a block of 16 rows each
  const int h = blockIdx.x, c0 = blockIdx.y * kSsCols;
  const int seg = long_segment(blockIdx.z, gridDim.z, st, start);
  if (seg < 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lo = lane & 15, hi = lane >> 4;
  const int row0 = start[seg], rows = start[seg + 1] - row0;
  Chunk c;
  if (!find_chunk(c, 0, seg, start, pos0, slot, st.min_rows, num_slots)) {
    // a padding segment's rows are zeros
    if (rows >= st.min_rows && (slot[seg] < 0 || slot[seg] >= num_slots))
      for (int e = tid; e < rows * kSsCols; e += kSsThreads) o[((long)(row0 + e / kSsCols) * heads + h) * dv + c0 + e % kSsCols] = 0.f;
    return;
  }
  const float* const wsh = ws + (c.ws * heads + h) * (long)kSsFloats;
  const long ws_step = (long)heads * kSsFloats;
  // transposed reads: lane (hi, lo) asks for row 4 hi + lo / 4, four columns from 4 (lo % 4) on, and gets column lo of four rows
  const int tr_row = 4 * hi + (lo >> 2), tr_half = (lo & 1) * 8, tr_piece = (lo >> 1) & 1;
  // v, 32 rows a piece, as a left or right operand (its columns)
  auto read_v = [&](const char* vb, int p) {
    const uint2 x = ss_read_tr(vb + (32 * p + tr_row) * 32 + tr_piece * 16 + tr_half);
    const uint2 y = ss_read_tr(vb + (32 * p + 16 + tr_row) * 32 + tr_piece * 16 + tr_half);
    return make_uint4(x.x, x.y, y.x, y.y);
  };
  // chunk i lies in copy i mod 3; before each turn: what the turn before made is there, and nobody reads what this one writes
  auto turns = [&](auto turn) {
    int b = 2;
    for (int idx = -1; idx < c.num; ++idx) {
      turn(idx, b);
      b = b == 2 ? 0 : b + 1;
      __syncthreads();
    }
  };
  auto next = [](int b) { return b == 2 ? 0 : b + 1; };

  if (wave >= 8) {
    // ---- rows of k and v into LDS two chunks ahead, loads three; the next chunk's scaled v
    const int lt = tid - 512;
    const bf16_t* const kp = in.k + (long)row0 * in.stride + (long)(h / in.rep) * kSsKeys + (lt & 15) * 8;
    const bf16_t* const vp = in.v + (long)row0 * in.stride + (long)h * dv + c0 + (lt & 1) * 8;
    uint4 kr[4], vr;
    float4 f[2];
    auto fetch = [&](int idx) {        // (rows past the end: the last one, put as zeros)
      idx = min(idx, c.num - 1);
      const int left = min(kC, rows - idx * kC) - 1;
#pragma unroll
      for (int n = 0; n < 4; ++n) kr[n] = *reinterpret_cast<const uint4*>(kp + (long)(idx * kC + min((lt >> 4) + 16 * n, left)) * in.stride);
      vr = *reinterpret_cast<const uint4*>(vp + (long)(idx * kC + min((lt >> 1) & 63, left)) * in.stride);
    };
    auto fetch_f = [&](int idx) {
      const float* p = wsh + min(idx, c.num - 1) * ws_step + kSsPairs + kC + 32 * (wave & 1) + 4 * hi;
      f[0] = *reinterpret_cast<const float4*>(p);
      f[1] = *reinterpret_cast<const float4*>(p + 16);
    };
    auto put = [&](int idx, int b) {
      const int left = rows - idx * kC;
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        const int j = (lt >> 4) + 16 * n;
        uint4 x = kr[n];
        if (j >= left) x = uint4{0, 0, 0, 0};
        *reinterpret_cast<uint4*>(ks[b] + j * 256 + ((lt & 15) ^ (j & 15)) * 16) = x;
      }
      if ((lt >> 1) >= left) vr = uint4{0, 0, 0, 0};
      if (lt < 2 * kC) {
        *reinterpret_cast<uint4*>(vs[b] + lt * 16) = vr;
        const uint64_t m = __ballot(((ss_loose(vr.x) | ss_loose(vr.y) | ss_loose(vr.z) | ss_loose(vr.w)) & 0x80008000u) != 0);
        if ((lane & 31) == 0) loose[b][lt >> 5] = (uint32_t)(m >> lane);
      }
    };
    fetch(0);
    put(0, 0);
    fetch(1);
    if (wave >= 10) fetch_f(0);
    __syncthreads();
    turns([&](int idx, int b) {
      if (idx + 2 < c.num) put(idx + 2, next(next(b)));
      if (wave >= 10 && idx + 1 < c.num) {
        const int p = wave & 1;
        const uint4 v = read_v(vs[next(b)], p);
        float x[8];
        ft::unpack2(v.x, x[0], x[1]);
        ft::unpack2(v.y, x[2], x[3]);
        ft::unpack2(v.z, x[4], x[5]);
        ft::unpack2(v.w, x[6], x[7]);
        uint2 u[3], w[3];
        ss_split(x[0] * f[0].x, x[1] * f[0].y, x[2] * f[0].z, x[3] * f[0].w, u);
        ss_split(x[4] * f[1].x, x[5] * f[1].y, x[6] * f[1].z, x[7] * f[1].w, w);
#pragma unroll
        for (int z = 0; z < 3; ++z) scaled[(idx + 1) & 1][p][z][lane] = make_uint4(u[z].x, u[z].y, w[z].x, w[z].y);
        fetch_f(idx + 2);
      }
      fetch(idx + 3);
      asm volatile("" ::: "memory");     // the loads stay here: they are not moved to their uses, a chunk on
    });
  } else if (wave >= 4) {
    // ---- the state: rows 32 (wave - 4) .. of it, S <- total S + sum_j k_j (to_end_j v_j)^T
    const int w4 = wave - 4;
    float* const sp = state + (((long)c.slot * heads + h) * kSsKeys) * dv + c0 + lo;
    f32x4 S[2];
    auto publish = [&](int b) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        uint2 p[3];
        ss_split(S[i][0], S[i][1], S[i][2], S[i][3], p);
        // entries 32 w4 + 16 i + 4 hi ..: inner step w4, of lane (2 i + hi / 2, lo) half hi % 2
#pragma unroll
        for (int t = 0; t < 3; ++t) parts[b][t][w4][(2 * i + (hi >> 1)) * 16 + lo][hi & 1] = p[t];
      }
    };
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[i][r] = c.pos > 0 ? sp[(long)(32 * w4 + 16 * i + 4 * hi + r) * dv] : 0.f;
    publish(0);
    float gn = wsh[kSsPairs + 2 * kC];
    __syncthreads();
    turns([&](int idx, int b) {
      if (idx < 0) return;
      const char* kb = ks[b];
      const float g = gn;
      gn = wsh[min(idx + 1, c.num - 1) * ws_step + kSsPairs + 2 * kC];
      f32x4 acc[2][3];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int z = 0; z < 3; ++z) acc[i][z] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        uint4 w[3];
#pragma unroll
        for (int z = 0; z < 3; ++z) w[z] = scaled[idx & 1][p][z][lane];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int piece = 4 * w4 + 2 * i + tr_piece, j = 32 * p + tr_row;
          const uint2 k0 = ss_read_tr(kb + j * 256 + (piece ^ (j & 15)) * 16 + tr_half);
          const uint2 k1 = ss_read_tr(kb + (j + 16) * 256 + (piece ^ (j & 15)) * 16 + tr_half);
          const uint4 a = make_uint4(k0.x, k0.y, k1.x, k1.y);
#pragma unroll
          for (int z = 2; z >= 0; --z) acc[i][z] = ss_mma(a, w[z], acc[i][z]);
        }
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) S[i] = S[i] * g + ((acc[i][2] + acc[i][1]) + acc[i][0]);
      if (idx + 1 < c.num) publish((idx + 1) & 1);
    });
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) sp[(long)(32 * w4 + 16 * i + 4 * hi + r) * dv] = S[i][r];
  } else {
    // ---- outputs: rows 16 wave + lo, columns c0 + 4 hi ..
    const float skip = in.skip[h];
    const int t = 16 * wave + lo;
    const bf16_t* const qp = in.q + (long)row0 * in.stride + (long)(h / in.rep) * kSsKeys + 8 * hi;
    uint4 q[4], qn[4], w[2][3], wn[2][3];
    float f0, fn;
    auto fetch = [&](int idx) {
      idx = min(idx, c.num - 1);
      const bf16_t* p = qp + (long)min(idx * kC + t, rows - 1) * in.stride;
#pragma unroll
      for (int x = 0; x < 4; ++x) qn[x] = *reinterpret_cast<const uint4*>(p + 32 * x);
      const float* f = wsh + idx * ws_step;
      const uint4* g = (const uint4*)f + lane;
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int z = 0; z < 3; ++z) wn[p][z] = g[ss_piece(wave, wave < 2 ? 0 : p, z)];
      fn = f[kSsPairs + t];
      asm volatile("" ::: "memory");
    };
    fetch(0);
    __syncthreads();
    turns([&](int idx, int b) {
      if (idx < 0) return;
      const char* vb = vs[b];
      const int from = idx & 1;
#pragma unroll
      for (int x = 0; x < 4; ++x) q[x] = qn[x];
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int z = 0; z < 3; ++z) w[p][z] = wn[p][z];
      f0 = fn;
      fetch(idx + 1);
      f32x4 O[3], pv[3];
      const uint32_t apart = loose[b][wave];
#pragma unroll
      for (int z = 0; z < 3; ++z) O[z] = pv[z] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int z = 2; z >= 0; --z) O[z] = ss_mma(*reinterpret_cast<const uint4*>(&parts[from][z][x][lane][0]), q[x], O[z]);
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        if (2 * p > wave) continue;
        uint4 v = read_v(vb, p);
        if (2 * p + 1 > wave) v.z = v.w = 0;       // (rows behind all of these: nothing of theirs, were it infinite)
#pragma unroll
        for (int z = 2; z >= 0; --z) pv[z] = ss_mma(v, w[p][z], pv[z]);
      }
      const bool again = __builtin_amdgcn_readfirstlane(apart) != 0;
      if (again) {
        // One of the block's own rows is not finite, and a weight of 0 takes it to the rows before it: the sums again without such
        // values of the block, which then go to the rows from them on.
#pragma unroll
        for (int z = 0; z < 3; ++z) pv[z] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          if (2 * p > wave) continue;
          uint4 v = read_v(vb, p);
          if (2 * p + 1 > wave) v.z = v.w = 0;
          if (p == wave >> 1) {
            if (wave & 1) v.z &= ~ss_not_finite(v.z), v.w &= ~ss_not_finite(v.w);
            else v.x &= ~ss_not_finite(v.x), v.y &= ~ss_not_finite(v.y);
          }
#pragma unroll
          for (int z = 2; z >= 0; --z) pv[z] = ss_mma(v, w[p][z], pv[z]);
        }
      }
      f32x4 y = ((O[2] + O[1]) + O[0]) * f0 + ((pv[2] + pv[1]) + pv[0]);
      if (again) {
        // lane (hi, lo) has the weights of row t and rows 4 hi .. 4 hi + 3 of the block
        float own[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          own[r] = 0.f;
#pragma unroll
          for (int z = 2; z >= 0; --z) {
            const uint32_t first = wave >> 1 ? (r < 2 ? w[1][z].x : w[1][z].y) : r < 2 ? w[0][z].x : w[0][z].y;
            const uint32_t second = wave >> 1 ? (r < 2 ? w[1][z].z : w[1][z].w) : r < 2 ? w[0][z].z : w[0][z].w;
            const uint32_t x = wave & 1 ? second : first;
            own[r] += __uint_as_float(r & 1 ? x & 0xffff0000u : x << 16);
          }
        }
#pragma unroll 1
        for (int g = 0; g < 4; ++g) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int j = 4 * g + r;
            const float wj = __shfl(own[r], 16 * g + lo, 64);
            const uint2 u = *reinterpret_cast<const uint2*>(vb + (16 * wave + j) * 32 + 8 * hi);
            const uint32_t m[2] = {ss_not_finite(u.x), ss_not_finite(u.y)}, x[2] = {u.x, u.y};
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (j <= lo && (m[e >> 1] >> (16 * (e & 1)) & 1)) y[e] += wj * __uint_as_float(e & 1 ? x[e >> 1] & 0xffff0000u : x[e >> 1] << 16);
          }
        }
      }
      if (t < rows - idx * kC) {
        const uint2 own = *reinterpret_cast<const uint2*>(vb + t * 32 + 8 * hi);
        float x[4];
        ft::unpack2(own.x, x[0], x[1]);
        ft::unpack2(own.y, x[2], x[3]);
        *reinterpret_cast<float4*>(o + ((long)(row0 + idx * kC + t) * heads + h) * dv + c0 + 4 * hi) =
            make_float4(y[0] + skip * x[0], y[1] + skip * x[1], y[2] + skip * x[2], y[3] + skip * x[3]);
      }
    });
  }
}

}  // namespace mx

using namespace mx;

// floats of workspace per chunk and head
extern "C" int mx_state_scan_floats() { return kSsFloats; }

// Whether these rows are the kernels': bf16, 128 entries of the state a column, whole 16-byte pieces, and workgroups enough or
// chunks few enough that the chain of chunks is not what a segment waits for.  us, beside the chunk-parallel form: 16 workgroups (4
// heads of 128 x 64), 500 / 1000 / 2000 / 4000 rows 21 31 47 94 (32 35 38 53); 32 (4 of 128 x 128), 2000 49 (46); 64 (8 of 128 x
// 128), 2000 and 4000 49 96 (60 104); 256 (32 of 128 x 128), 64 / 200 / 777 / 2048 / 4096 12 17 32 59 106 (34 40 82 149 251), five of
// 400 73 (158), 64 of 100 390 (704).
extern "C" int mx_state_scan_takes(const void* y, const void* xbc, int bf16, long stride, int heads, int groups, int n, int dv,
                                   int max_rows) {
  return bf16 && n == kSsKeys && dv >= 1 && dv % kSsCols == 0 && stride % 8 == 0 && ((uintptr_t)xbc) % 16 == 0 &&
         ((uintptr_t)y) % 16 == 0 && dv / kSsCols <= 65535 && heads >= 1 && heads <= 65535 && groups >= 1 && heads % groups == 0 &&
         ((long)heads * (dv / kSsCols) >= 64 || max_rows <= 1000);
}

// segments of min_rows rows or more; arguments as mx_ssd_chunks
extern "C" int mx_state_scan(float* y, float* ws, const void* xbc, long stride, const void* dt, long dt_stride, const float* a_log,
                             const float* dt_bias, const float* d_skip, float* state, long rows, const int* start, const int* pos0,
                             const int* slot, int num_segs, int max_rows, int heads, int groups, int n, int dv, int num_slots,
                             int min_rows, hipStream_t s) {
  if (num_segs <= 0 || max_rows < min_rows || rows <= 0) return 0;
  if (min_rows < 1 || !mx_state_scan_takes(y, xbc, 1, stride, heads, groups, n, dv, max_rows)) return -1;
  const ChunkGrid g(rows, max_rows, min_rows, num_segs);
  const bf16_t* x = (const bf16_t*)xbc;
  const ScanIn in{x + (long)heads * dv + (long)groups * n, x + (long)heads * dv, x, stride, heads / groups,
                  (const bf16_t*)dt, dt_stride, a_log, dt_bias, d_skip};
  if (!g.fits(heads) || ((uintptr_t)ws) % 16) return -2;
  hipLaunchKernelGGL(state_pairs_kernel, g.grid(heads), dim3(256), 0, s, ws, in, start, pos0, slot, heads, num_slots, g.steps);
  hipLaunchKernelGGL(state_scan_kernel, dim3(heads, dv / kSsCols, g.longs), dim3(kSsThreads), 0, s, y, ws, in, state, start, pos0, slot, heads,
                     dv, num_slots, g.steps);
  return (int)hipGetLastError();
}

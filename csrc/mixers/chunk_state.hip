// Recurrences with one decay per head, long segments: the gated delta rule, retention and the selective
// state-space scan (a retention whose decay changes by row) in chunk form, as fp32 matrix products (v_mfma_f32_16x16x4_f32) over chunks of 64 rows, so
// that only one small step per chunk is sequential.
//
// With the rows of a chunk t = 0 .. 63, their log decays l_t, G_t = l_0 + .. + l_t and the
// state S before the chunk:
//   o_t = e^{G_t} S^T q_t + sum_{j <= t} e^{G_t - G_j} (q_t.k_j) w_j
//   S' = e^{G_63} S + sum_j e^{G_63 - G_j} k_j w_j^T
// where w_j = v_j for retention.  For the delta rule w solves
//   w_t = beta_t (v_t - e^{G_t} S^T k_t - sum_{j < t} e^{G_t - G_j} (k_t.k_j) w_j),
// which is linear in S: w = U - W S with (I + A) [U | W] = [beta v | beta e^G k] and A_tj =
// beta_t e^{G_t - G_j} (k_t.k_j) for j < t.
//
// Kernels:
//   delta_solve   per (chunk, head), parallel: A, (I + A)^-1 (16-row diagonal blocks by
//                 substitution, the rest by block products) and [U | W] on the matrix units;
//                 leaves U, -W and e^{G_63 - G_j} k_j.  (The inverse is harmless numerically:
//                 its entries are -beta k^T (products of I - beta k k^T) k, at most one in size.)
//   chunk_carry   per (head, 16 columns of the state), chunk after chunk: the state stays in the
//                 accumulators of four waves (16-row tiles dealt out), whose register layout is
//                 that of a right-hand operand; leaves w and every chunk's incoming state
//   state_add     retention, state space, per (chunk, head), parallel: a chunk's own contribution to the state
//   state_carry   retention, state space: elementwise scan over the chunks
//   chunk_out     both, per (chunk, head, 64 columns), parallel: o from the incoming state
// Sums of log decays are formed in double precision and only their differences are rounded, so
// a chunk's decay ratios are as exact as a row-by-row walk's.
//
// delta_solve leaves -W, the keys and U as fragments: for every 16 x 16 tile one 16-byte piece per
// lane (hi, lo) = (lane / 16, lane % 16), in the lanes' order, so that delta_carry's operand
// loads are whole kilobytes: -W tile (m, i) holds rows 16 m + lo, columns 16 i + 4 hi + r; key
// tile (i, m) columns 16 i + lo, rows 16 m + 4 hi + r; U tile (ct, m) rows 16 m + 4 hi + r, column
// 16 ct + lo (r = 0 .. 3 the piece's entries).
//
// A chunk's workspace index is start[s] / 64 + s + its number within the segment: distinct
// for all chunks of a step, below rows / 64 + segments.  Rows of a last, partial chunk past the
// segment's end count as k = v = 0, beta = 0, l = 0.
#include "chunk_common.h"

namespace mx {

struct ChunkIn {
  const void* q;
  const void* k;
  const void* v;
  long q_stride, k_stride, v_stride;   // elements between rows
  int rep;                             // heads per q / k head
  const float* lg;                     // log decays [T, heads], null: log_decay per head
  const double* log_decay;             // [heads]
  const float* table;                  // rotation of q and k, null: none
  int table_rows, rot_dims, interleaved;
  float k_scale;
  int v_frags;                         // v: fragments by workspace chunk (below) instead of rows
  const float* v_scale;                // factor of each row of v in the state [T, heads], null: 1
  const float* skip;                   // o += skip[h] v, null: none
};

// rows [0, cnt) of one head of q or k (dk in whole fours, DKP of them padded), by 256 threads; rows past the end read the last
template <typename T, int DKP>
__device__ __forceinline__ void fetch_head(Four<T> (&u)[DKP / 16], const T* src, long stride, int cnt, int dk) {
#pragma unroll
  for (int n = 0; n < DKP / 16; ++n) {
    const int e = threadIdx.x + 256 * n, t = min(e / (DKP / 4), cnt - 1), i = min(e % (DKP / 4) * 4, dk - 4);
    u[n] = *reinterpret_cast<const Four<T>*>(src + t * stride + i);
  }
}
// times scale into LDS, entry (row, column) at `at`, zeros elsewhere
template <typename F, int DKP, typename At>
__device__ __forceinline__ void put_head(float* dst, At at, const F (&u)[DKP / 16], int cnt, int dk, float scale) {
#pragma unroll
  for (int n = 0; n < DKP / 16; ++n) {
    const int e = threadIdx.x + 256 * n, t = e / (DKP / 4), i = e % (DKP / 4) * 4;
    const float4 v = widen(u[n]);
    const float f = t < cnt && i < dk ? scale : 0.f;
    *reinterpret_cast<float4*>(dst + at(t, i)) = f != 0.f ? make_float4(v.x * f, v.y * f, v.z * f, v.w * f) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
}

// rows [0, cnt) of one head of q or k into LDS, rotated, times scale; zeros past cnt
// and past dk (up to DKP)
template <typename T, int DKP, typename At>
__device__ __forceinline__ void stage_head(float* dst, At at, const T* src, long stride, int cnt, int dk,
                                           const float* table, int table_rows, int rot, int interleaved, int pos,
                                           float scale, int vec) {
  const int tid = threadIdx.x;
  const int t0 = tid >> 5, l0 = tid & 31;   // without 16-byte pieces: 32 lanes per row, 8 rows at a time
  int d0 = 0;                       // entries below are rotated pairs
  if (table != nullptr && rot > 0) {
    d0 = rot;
    const int half = rot / 2;
#pragma unroll 4
    for (int t = t0; t < kC; t += 8) {
      // rows past cnt read the last row and count as zeros
      const int tt = min(t, cnt - 1);
      int p = pos + tt;
      if (p < 0 || p >= table_rows) p = 0;
      const float* cs = table + (long)p * rot;
      const float f = t < cnt ? scale : 0.f;
      for (int i = l0; i < half; i += 32) {
        const int a = interleaved ? 2 * i : i, b = interleaved ? 2 * i + 1 : i + half;
        const float c = cs[i], sn = cs[half + i];
        const float x = ld(src, tt * stride + a), y = ld(src, tt * stride + b);
        dst[at(t, a)] = (x * c - y * sn) * f;
        dst[at(t, b)] = (y * c + x * sn) * f;
      }
    }
  }
  if (vec && d0 == 0) {
    Four<T> u[DKP / 16];
    fetch_head<T, DKP>(u, src, stride, cnt, dk);
    put_head<Four<T>, DKP>(dst, at, u, cnt, dk, scale);
    return;
  }
  for (int t = t0; t < kC; t += 8)
    for (int i = d0 + l0; i < DKP; i += 32) dst[at(t, i)] = t < cnt && i < dk ? ld(src, t * stride + i) * scale : 0.f;
}

// G[t] = sum of the chunk's log decays up to t (wave 0; 64 rows)
__device__ __forceinline__ void stage_log_decay(double* G, const ChunkIn& in, long row0, int cnt, int heads, int h) {
  if (threadIdx.x >= 64) return;
  const int t = threadIdx.x;
  double l = 0.0;
  if (t < cnt) l = in.lg != nullptr ? (double)in.lg[(row0 + t) * heads + h] : in.log_decay[h];
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double u = __shfl_up(l, off, 64);
    if (t >= off) l += u;
  }
  G[t] = l;
}

// rs[t] = the factor of row t of v (0 past cnt: v counts as zeros there)
__device__ __forceinline__ void stage_row_scale(float* rs, const ChunkIn& in, long row0, int cnt, int heads, int h) {
  const int t = threadIdx.x;
  if (t < kC) rs[t] = t >= cnt ? 0.f : in.v_scale != nullptr ? in.v_scale[(row0 + t) * heads + h] : 1.f;
}

// ---------------------------------------------------------------------------------
// a workgroup per chunk, head and 64 columns: L = sum_j e^{G_last - G_j} k_j v_j^T into the
// chunk's workspace [dk, dv] (v times its row factor); totals[chunk, head] = e^{G_last} if wanted.
// Wave w: columns 16 w .. 16 w + 15 of the 64, all rows.
// ---------------------------------------------------------------------------------
template <typename T, int DKT>
__global__ void __launch_bounds__(256)
state_add_kernel(float* __restrict__ ws_s, float* __restrict__ totals, ChunkIn in, const int* __restrict__ start,
                 const int* __restrict__ pos0, const int* __restrict__ slot, int heads, int dk, int dv, int num_slots,
                 ChunkSteps st, int vec) {
  constexpr int DKP = 16 * DKT, LDK = DKT >= 4 ? DKP : DKP + 16;       // (fewer blocks than there are to exchange: padded)
  auto at = [](int row, int col) { return DKT >= 4 ? swizzled<LDK>(row, col) : row * LDK + col; };
  __shared__ __attribute__((aligned(16))) float kb[kC * LDK], vb[kC * kVLD];
  __shared__ double G[kC];
  __shared__ float rs[kC];
  const int vt = (dv + 63) / 64, unit = blockIdx.x % (heads * vt);
  const int h = unit / vt, col0 = unit % vt * 64;
  Chunk c;
  int seg, idx;
  if (!find_chunk(c, blockIdx.x / (heads * vt), st, seg, idx, start, pos0, slot, num_slots)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lo = lane & 15, hi = lane >> 4;
  stage_log_decay(G, in, c.row0, c.cnt, heads, h);
  stage_row_scale(rs, in, c.row0, c.cnt, heads, h);
  stage_head<T, DKP>(kb, at, (const T*)in.k + c.row0 * in.k_stride + (long)(h / in.rep) * dk, in.k_stride, c.cnt, dk,
                     in.table, in.table_rows, in.rot_dims, in.interleaved, c.pos, in.k_scale, vec);
  stage_cols<T>(vb, (const T*)in.v + c.row0 * in.v_stride + (long)h * dv, in.v_stride, c.cnt, col0, dv, vec);
  __syncthreads();
  const double gl = G[kC - 1];
  if (totals != nullptr && col0 == 0 && tid == 0) totals[c.ws * heads + h] = expf((float)gl);
  f32x4 acc[DKT];
#pragma unroll
  for (int i = 0; i < DKT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < kC / 4; ++s) {
    const int j = 4 * s + hi;
    const float b = vb[swizzled<kVLD>(j, 16 * wave + lo)] * (expf((float)(gl - G[j])) * rs[j]);
#pragma unroll
    for (int i = 0; i < DKT; ++i) acc[i] = mma(kb[at(j, 16 * i + lo)], b, acc[i]);
  }
  const int col = col0 + 16 * wave + lo;
  if (col >= dv) return;
  float* out = ws_s + ((c.ws * heads + h) * dk) * dv + col;
#pragma unroll
  for (int i = 0; i < DKT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * i + 4 * hi + r;
      if (row < dk) out[(long)row * dv] = acc[i][r];
    }
}

// grid (ceil(dk dv / 256), heads, long segments): workspaces hold every chunk's own contribution L_c
// and become its incoming state; the last one goes to the slot.  A chunk's decay: totals[chunk, head],
// or the head's fixed one per row.
__global__ void __launch_bounds__(256)
state_carry_kernel(float* __restrict__ ws_s, const double* __restrict__ log_decay, const float* __restrict__ totals,
                   float* __restrict__ state, const int* __restrict__ start, const int* __restrict__ pos0,
                   const int* __restrict__ slot, int heads, int size, int num_slots, ChunkSteps st) {
  Chunk c;
  const int seg = long_segment(blockIdx.z, gridDim.z, st, start);
  if (seg < 0 || !find_chunk(c, 0, seg, start, pos0, slot, st.min_rows, num_slots)) return;
  const int h = blockIdx.y, e = blockIdx.x * 256 + threadIdx.x;
  if (e >= size) return;
  const int n = start[seg + 1] - start[seg];
  float* sp = state + ((long)c.slot * heads + h) * size + e;
  float S = c.pos > 0 ? *sp : 0.f;
  float full = 0.f, last = 0.f;
  if (totals == nullptr) {
    full = (float)exp(log_decay[h] * kC);
    last = (float)exp(log_decay[h] * (n - (c.num - 1) * kC));
  }
  float* w = ws_s + (c.ws * heads + h) * (long)size + e;
  const long step = (long)heads * size;
  constexpr int AHEAD = 8;            // contributions in flight
  for (int i0 = 0; i0 < c.num; i0 += AHEAD) {
    float l[AHEAD], g[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      l[u] = i0 + u < c.num ? w[(i0 + u) * step] : 0.f;
      g[u] = totals == nullptr ? (i0 + u + 1 < c.num ? full : last) : totals[(c.ws + min(i0 + u, c.num - 1)) * heads + h];
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      if (i0 + u < c.num) {
        w[(i0 + u) * step] = S;
        S = g[u] * S + l[u];
      }
    }
  }
  *sp = S;
}

// ---------------------------------------------------------------------------------
// a workgroup per chunk, head and 64 columns: o of the chunk's rows.  Wave w: rows 16 w ..
// 16 w + 15, 64 columns; its q rows stay in registers as left-hand operands.
// ---------------------------------------------------------------------------------
template <typename T, int DKT>
__global__ void __launch_bounds__(256)
chunk_out_kernel(float* __restrict__ o, ChunkIn in, const float* __restrict__ ws_s, const int* __restrict__ start,
                 const int* __restrict__ pos0, const int* __restrict__ slot, int heads, int dk, int dv, int num_slots,
                 ChunkSteps st, int vec) {
  constexpr int DKP = 16 * DKT, LDK = DKP + 4;
  auto at = [](int row, int col) { return row * LDK + col; };
  constexpr int KB = kC * LDK > 64 * kPLD ? kC * LDK : 64 * kPLD;
  __shared__ __attribute__((aligned(16))) float kb[KB], vb[kC * kVLD];
  __shared__ double G[kC];
  __shared__ float rs[kC];
  const int vt = (dv + 63) / 64, unit = blockIdx.x % (heads * vt);
  const int h = unit / vt, col0 = unit % vt * 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lo = lane & 15, hi = lane >> 4;
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
  const long hoff = (long)(h / in.rep) * dk;
  const float* S = ws_s + ((c.ws * heads + h) * dk) * (long)dv;
  stage_log_decay(G, in, c.row0, c.cnt, heads, h);
  stage_row_scale(rs, in, c.row0, c.cnt, heads, h);
  stage_head<T, DKP>(kb, at, (const T*)in.q + c.row0 * in.q_stride + hoff, in.q_stride, c.cnt, dk, in.table,
                     in.table_rows, in.rot_dims, in.interleaved, c.pos, 1.f, vec);
  const int svec = dv % 4 == 0;
  stage_cols<float>(vb, S, dv, min(dk, kC), col0, dv, svec);         // rows 0 .. 63 of the incoming state
  // what follows is asked for now: rows 64 .. of the state, the keys and the values
  const T* const kp = (const T*)in.k + c.row0 * in.k_stride + hoff;
  const T* const vp = (const T*)in.v + c.row0 * in.v_stride + (long)h * dv;
  const bool plain = vec && (in.table == nullptr || in.rot_dims == 0), rows_v = vec && !in.v_frags;
  Four<float> s_next[4];
  Four<T> k_next[DKT], v_next[4];
  if constexpr (DKT > 4) {
    if (svec) fetch_cols<float>(s_next, S + 64L * dv, dv, dk - 64, col0, dv);
  }
  if (plain) fetch_head<T, DKP>(k_next, kp, in.k_stride, c.cnt, dk);
  if (rows_v) fetch_cols<T>(v_next, vp, in.v_stride, c.cnt, col0, dv);
  __syncthreads();
  float qf[4 * DKT];
#pragma unroll
  for (int s = 0; s < 4 * DKT; ++s) qf[s] = kb[(16 * wave + lo) * LDK + 4 * s + hi];
  f32x4 O[4];
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) O[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < (DKT < 4 ? 4 * DKT : 16); ++s)
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) O[ct] = mma(qf[s], vb[swizzled<kVLD>(4 * s + hi, 16 * ct + lo)], O[ct]);
  __syncthreads();
  if constexpr (DKT > 4) {                                   // rows 64 .. of the state
    if (svec) put_cols(vb, s_next, dk - 64, col0, dv);
    else stage_cols<float>(vb, S + 64L * dv, dv, dk - 64, col0, dv, 0);
    __syncthreads();
#pragma unroll
    for (int s = 16; s < 4 * DKT; ++s)
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) O[ct] = mma(qf[s], vb[swizzled<kVLD>(4 * (s - 16) + hi, 16 * ct + lo)], O[ct]);
    __syncthreads();
  }
  if (plain)
    put_head<Four<T>, DKP>(kb, at, k_next, c.cnt, dk, in.k_scale);
  else
    stage_head<T, DKP>(kb, at, kp, in.k_stride, c.cnt, dk, in.table, in.table_rows, in.rot_dims, in.interleaved, c.pos,
                       in.k_scale, vec);
  if (in.v_frags) {
    const int tiles = (dv + 15) / 16;
    const float4* fp = (const float4*)in.v + (c.ws * heads + h) * (long)tiles * 256;
    for (int ct = wave; ct < 4; ct += 4) {
      const int tile = min(col0 / 16 + ct, tiles - 1);       // columns past dv are not stored
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const float4 u = fp[(tile * 4 + m) * 64 + lane];
        const float v[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) vb[swizzled<kVLD>(16 * m + 4 * hi + r, 16 * ct + lo)] = v[r];
      }
    }
  } else if (rows_v) {
    put_cols(vb, v_next, c.cnt, col0, dv);
  } else {
    stage_cols<T>(vb, vp, in.v_stride, c.cnt, col0, dv, 0);
  }
  double gr[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    gr[r] = G[16 * wave + 4 * hi + r];
    const float e = expf((float)gr[r]);
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) O[ct][r] *= e;
  }
  __syncthreads();
  f32x4 P[4];
#pragma unroll
  for (int jt = 0; jt < 4; ++jt) {
    if (jt > wave) continue;                                 // keys behind every row of this wave
    const float* kr = kb + (16 * jt + lo) * LDK + hi;
    f32x4 a = dot_steps<4 * DKT>([&](int s) { return qf[s]; }, [&](int s) { return kr[4 * s]; });
    const double gj = G[16 * jt + lo];
    const float rj = rs[16 * jt + lo];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      a[r] = 16 * jt + lo <= 16 * wave + 4 * hi + r ? a[r] * expf((float)(gr[r] - gj)) * rj : 0.f;
    P[jt] = a;
  }
  __syncthreads();                                           // kb becomes four [16][64] strips
  float* strip = kb + wave * 16 * kPLD;
#pragma unroll
  for (int jt = 0; jt < 4; ++jt) {
    if (jt > wave) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) strip[(4 * hi + r) * kPLD + 16 * jt + lo] = P[jt][r];
  }
  wave_lds_fence();
#pragma unroll
  for (int jt = 0; jt < 4; ++jt) {
    if (jt > wave) continue;
#pragma unroll
    for (int s = 4 * jt; s < 4 * jt + 4; ++s) {
      const float a = strip[lo * kPLD + 4 * s + hi];
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) O[ct] = mma(a, vb[swizzled<kVLD>(4 * s + hi, 16 * ct + lo)], O[ct]);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int t = 16 * wave + 4 * hi + r;
    if (t >= c.cnt) continue;
    float* op = o + ((c.row0 + t) * heads + h) * dv;
    const float sk = in.skip != nullptr ? in.skip[h] : 0.f;
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
      if (col0 + 16 * ct + lo < dv)
        op[col0 + 16 * ct + lo] = in.skip != nullptr ? O[ct][r] + sk * vb[swizzled<kVLD>(t, 16 * ct + lo)] : O[ct][r];
  }
}

// ---------------------------------------------------------------------------------
// a workgroup per chunk and head, 256 threads.  Leaves per chunk and head, as fragments: -W,
// e^{G_last - G_j} k_j and U; and e^{G_last}.
// ---------------------------------------------------------------------------------
template <int DKT>
__global__ void __launch_bounds__(256)
delta_solve_kernel(float* __restrict__ ws_w, float* __restrict__ ws_k, float* __restrict__ ws_u,
                   float* __restrict__ ws_g, ChunkIn in, const float* __restrict__ beta, const int* __restrict__ start,
                   const int* __restrict__ pos0, const int* __restrict__ slot, int heads, int dk, int dv, int num_slots,
                   ChunkSteps st, int vec) {
  constexpr int DKP = 16 * DKT, LDK = DKP + 4;
  auto at = [](int row, int col) { return row * LDK + col; };
  // ab: A, block by block replaced by T = (I + A)^-1 (blocks above the diagonal are never read)
  __shared__ __attribute__((aligned(16))) float kb[kC * LDK], ab[kC * kPLD];
  __shared__ double G[kC];
  __shared__ float bs[kC], eg[kC], el[kC];
  Chunk c;
  int seg, idx;
  if (!find_chunk(c, blockIdx.x / heads, st, seg, idx, start, pos0, slot, num_slots)) return;
  const int h = blockIdx.x % heads;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lo = lane & 15, hi = lane >> 4;
  stage_log_decay(G, in, c.row0, c.cnt, heads, h);
  if (tid >= 64 && tid < 128) bs[tid - 64] = tid - 64 < c.cnt ? beta[(c.row0 + tid - 64) * heads + h] : 0.f;
  stage_head<float, DKP>(kb, at, (const float*)in.k + c.row0 * in.k_stride + (long)(h / in.rep) * dk, in.k_stride, c.cnt,
                         dk, nullptr, 0, 0, 0, 0, 1.f, vec);
  __syncthreads();
  if (tid < kC) {
    eg[tid] = expf((float)G[tid]) * bs[tid];
    el[tid] = expf((float)(G[kC - 1] - G[tid]));
    if (tid == 0) ws_g[c.ws * heads + h] = expf((float)G[kC - 1]);
  }
  {
    float kf[4 * DKT];
#pragma unroll
    for (int s = 0; s < 4 * DKT; ++s) kf[s] = kb[(16 * wave + lo) * LDK + 4 * s + hi];
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) {
      if (jt > wave) continue;
      const float* kr = kb + (16 * jt + lo) * LDK + hi;
      const f32x4 a = dot_steps<4 * DKT>([&](int s) { return kf[s]; }, [&](int s) { return kr[4 * s]; });
      const int j = 16 * jt + lo;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 16 * wave + 4 * hi + r;
        ab[i * kPLD + j] = j < i ? bs[i] * a[r] * expf((float)(G[i] - G[j])) : 0.f;
      }
    }
  }
  invert_unit_lower(ab, wave, lo, hi);
  // [W | U] = T [beta e^G k | beta v], column tiles dealt out to the waves
  float tf[4][16], fw[16], fu[16];
  load_inverse(tf, ab, lo, hi);
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    fw[s] = eg[4 * s + hi];
    fu[s] = bs[4 * s + hi];
  }
  f32x4* ww = (f32x4*)ws_w + (c.ws * heads + h) * (long)(4 * DKT * 64);
  for (int ct = wave; ct < DKT; ct += 4) {
    float b[16];
    f32x4 x[4];
#pragma unroll
    for (int s = 0; s < 16; ++s) b[s] = -fw[s] * kb[(4 * s + hi) * LDK + 16 * ct + lo];
    inverse_column<true>(tf, b, x);
#pragma unroll
    for (int m = 0; m < 4; ++m) ww[(m * DKT + ct) * 64 + lane] = x[m];
  }
  const int vtiles = (dv + 15) / 16;
  f32x4* wu = (f32x4*)ws_u + (c.ws * heads + h) * (long)vtiles * 256;
  for (int ct = wave; ct < vtiles; ct += 4) {
    float b[16];
    f32x4 x[4];
    const int col = 16 * ct + lo;
    const float* vp = (const float*)in.v + c.row0 * in.v_stride + (long)h * dv + min(col, dv - 1);
#pragma unroll
    for (int s = 0; s < 16; ++s) b[s] = fu[s] * vp[min(4 * s + hi, c.cnt - 1) * in.v_stride];   // beta is 0 past cnt
    inverse_column<false>(tf, b, x);
#pragma unroll
    for (int m = 0; m < 4; ++m) wu[(ct * 4 + m) * 64 + lane] = x[m];
  }
  f32x4* wk = (f32x4*)ws_k + (c.ws * heads + h) * (long)(4 * DKT * 64);
  for (int e = wave; e < 4 * DKT; e += 4) {
    const int i = e / 4, m = e % 4;
    f32x4 x;
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] = kb[(16 * m + 4 * hi + r) * LDK + 16 * i + lo] * el[16 * m + 4 * hi + r];
    wk[e * 64 + lane] = x;
  }
}

}  // namespace mx

using namespace mx;

extern "C" int mx_chunk_rows() { return kC; }
extern "C" int mx_chunk_max_dk() { return 128; }
// key size up to the kernels' whole tiles (rows of the -W and key workspaces)
extern "C" int mx_chunk_key_pad(int dk) { return dk <= 16 ? 16 : dk <= 32 ? 32 : dk <= 64 ? 64 : 128; }

template <typename T>
static void launch_out(float* o, const ChunkIn& in, const float* ws_s, const int* start, const int* pos0,
                       const int* slot, const ChunkGrid& g, int heads, int dk, int dv, int num_slots, int vec,
                       hipStream_t s) {
  key_tiles(dk, [&](auto t) {
    hipLaunchKernelGGL((chunk_out_kernel<T, decltype(t)::value>), g.grid((long)heads * ((dv + 63) / 64)), dim3(256), 0, s, o, in,
                       ws_s, start, pos0, slot, heads, dk, dv, num_slots, g.steps, vec);
  });
}

extern "C" int mx_retention_chunks(float* o, const void* p, int bf16, long stride, const float* table, int table_rows,
                                   int rot_dims, int interleaved, const double* log_decay, float* state, float* ws_s,
                                   const int* start, const int* pos0, const int* slot, long rows, int num_segs, int max_rows,
                                   int heads, int dk, int dv, int num_slots, int min_rows, hipStream_t s) {
  if (num_segs <= 0 || max_rows < min_rows) return 0;
  if (dk < 1 || dk > mx_chunk_max_dk() || dv < 1 || heads < 1 || min_rows < 1) return -1;
  ChunkIn in{};
  const long es = bf16 ? 2 : 4;
  in.q = p;
  in.k = (const char*)p + es * heads * dk;
  in.v = (const char*)p + es * 2 * heads * dk;
  in.q_stride = in.k_stride = in.v_stride = stride;
  in.rep = 1;
  in.log_decay = log_decay;
  in.table = rot_dims > 0 ? table : nullptr;
  in.table_rows = table_rows; in.rot_dims = rot_dims; in.interleaved = interleaved;
  in.k_scale = 1.0f / sqrtf((float)dk);
  const int vec = dk % 4 == 0 && dv % 4 == 0 && stride % 4 == 0 && ((uintptr_t)p) % (4 * es) == 0;
  const ChunkGrid g(rows, max_rows, min_rows, num_segs);
  const long units = (long)heads * ((dv + 63) / 64);
  if (!g.fits(units)) return -2;
  MX_DISPATCH_T(bf16, key_tiles(dk, [&](auto t) {
    hipLaunchKernelGGL((state_add_kernel<T, decltype(t)::value>), g.grid(units), dim3(256), 0, s, ws_s, nullptr, in, start, pos0,
                       slot, heads, dk, dv, num_slots, g.steps, vec);
  }));
  hipLaunchKernelGGL(state_carry_kernel, dim3((dk * dv + 255) / 256, heads, g.longs), dim3(256), 0, s, ws_s, log_decay,
                     nullptr, state, start, pos0, slot, heads, dk * dv, num_slots, g.steps);
  MX_DISPATCH_T(bf16, (launch_out<T>(o, in, ws_s, start, pos0, slot, g, heads, dk, dv, num_slots, vec, s)));
  return (int)hipGetLastError();
}

// step = softplus(dt + dt_bias) and the log decay -exp(a_log) step of every row and head
template <typename T>
__global__ void ssd_steps_kernel(float* __restrict__ step, float* __restrict__ lg, const T* __restrict__ dt,
                                 long dt_stride, const float* __restrict__ a_log, const float* __restrict__ dt_bias,
                                 long rows, int heads) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= rows * heads) return;
  const long row = e / heads;
  const int h = (int)(e % heads);
  const float v = softplusf_(ld(dt, row * dt_stride + h) + dt_bias[h]);
  const float l = -expf(a_log[h]) * v;
  step[e] = v;
  lg[e] = l < -3e38f ? -3e38f : l;         // (sums of these are subtracted: -inf would become NaN; the decay is 0)
}

// The selective state-space scan's long segments: q = C and k = B (one per group of heads), v = x times
// its step, a decay per row and head, o += D x.  ws_h: 2 rows * heads floats (steps, log decays).
extern "C" int mx_ssd_chunks(float* y, const void* xbc, int bf16, long stride, const void* dt, long dt_stride,
                             const float* a_log, const float* dt_bias, const float* d_skip, float* state, float* ws_s,
                             float* ws_g, float* ws_h, long rows, const int* start, const int* pos0, const int* slot,
                             int num_segs, int max_rows, int heads, int groups, int n, int dv, int num_slots,
                             int min_rows, hipStream_t s) {
  if (num_segs <= 0 || max_rows < min_rows || rows <= 0) return 0;
  if (n < 1 || n > mx_chunk_max_dk() || dv < 1 || groups < 1 || heads % groups || min_rows < 1) return -1;
  const long es = bf16 ? 2 : 4;
  ChunkIn in{};
  in.v = xbc;
  in.k = (const char*)xbc + es * heads * dv;
  in.q = (const char*)xbc + es * ((long)heads * dv + (long)groups * n);
  in.q_stride = in.k_stride = in.v_stride = stride;
  in.rep = heads / groups;
  in.v_scale = ws_h;
  in.lg = ws_h + rows * heads;
  in.skip = d_skip;
  in.k_scale = 1.f;
  const int vec = n % 4 == 0 && dv % 4 == 0 && stride % 4 == 0 && ((uintptr_t)xbc) % (4 * es) == 0;
  const ChunkGrid g(rows, max_rows, min_rows, num_segs);
  const long units = (long)heads * ((dv + 63) / 64);
  if (!g.fits(units)) return -2;
  MX_DISPATCH_T(bf16, hipLaunchKernelGGL((ssd_steps_kernel<T>), dim3((unsigned)((rows * heads + 255) / 256)), dim3(256),
                                         0, s, ws_h, ws_h + rows * heads, (const T*)dt, dt_stride, a_log, dt_bias, rows,
                                         heads));
  MX_DISPATCH_T(bf16, key_tiles(n, [&](auto t) {
    hipLaunchKernelGGL((state_add_kernel<T, decltype(t)::value>), g.grid(units), dim3(256), 0, s, ws_s, ws_g, in, start, pos0,
                       slot, heads, n, dv, num_slots, g.steps, vec);
  }));
  hipLaunchKernelGGL(state_carry_kernel, dim3((n * dv + 255) / 256, heads, g.longs), dim3(256), 0, s, ws_s, nullptr,
                     ws_g, state, start, pos0, slot, heads, n * dv, num_slots, g.steps);
  MX_DISPATCH_T(bf16, (launch_out<T>(y, in, ws_s, start, pos0, slot, g, heads, n, dv, num_slots, vec, s)));
  return (int)hipGetLastError();
}

extern "C" int mx_head_delta_chunks(float* o, const float* q, const float* k, const float* v, const float* lg,
                                    const float* beta, float* state, float* ws_s, float* ws_w, float* ws_k, float* ws_u,
                                    float* ws_g, const int* start, const int* pos0, const int* slot, long rows, int num_segs,
                                    int max_rows, int heads, int kv_heads, int dk, int dv, int num_slots, int min_rows,
                                    hipStream_t s) {
  if (num_segs <= 0 || max_rows < min_rows) return 0;
  if (dk < 1 || dk > mx_chunk_max_dk() || dv < 1 || kv_heads < 1 || heads % kv_heads || min_rows < 1) return -1;
  ChunkIn in{};
  in.q = q; in.k = k; in.v = v;
  in.q_stride = in.k_stride = (long)kv_heads * dk;
  in.v_stride = (long)heads * dv;
  in.rep = heads / kv_heads;
  in.lg = lg;
  in.k_scale = 1.f;
  const int vec = dk % 4 == 0 && dv % 4 == 0 && (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) % 16) == 0;
  if (((uintptr_t)ws_w | (uintptr_t)ws_k | (uintptr_t)ws_u) % 16) return -3;
  const ChunkGrid g(rows, max_rows, min_rows, num_segs);
  if (!g.fits((long)heads * ((dv + 63) / 64))) return -2;
  key_tiles(dk, [&](auto t) {
    hipLaunchKernelGGL((delta_solve_kernel<decltype(t)::value>), g.grid(heads), dim3(256), 0, s, ws_w,
                       ws_k, ws_u, ws_g, in, beta, start, pos0, slot, heads, dk, dv, num_slots, g.steps, vec);
    constexpr int DKT = decltype(t)::value;
    const dim3 cgrid(heads, (dv + 15) / 16, g.longs);
    if (dk == 16 * DKT && dv % 16 == 0)
      hipLaunchKernelGGL((chunk_carry_kernel<DKT, true, false, true, float>), cgrid, dim3(256), 0, s, ws_s, ws_w, ws_k,
                         ws_u, ws_g, (const float*)nullptr, 0L, state, start,
                         pos0, slot, heads, dk, dv, num_slots, g.steps);
    else
      hipLaunchKernelGGL((chunk_carry_kernel<DKT, false, false, true, float>), cgrid, dim3(256), 0, s, ws_s, ws_w, ws_k,
                         ws_u, ws_g, (const float*)nullptr, 0L, state, start,
                         pos0, slot, heads, dk, dv, num_slots, g.steps);
  });
  in.v = ws_u;                     // the solved rows take the values' place
  in.v_frags = 1;
  launch_out<float>(o, in, ws_s, start, pos0, slot, g, heads, dk, dv, num_slots, vec, s);
  return (int)hipGetLastError();
}

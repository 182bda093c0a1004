// Shared pieces of the chunk forms of the recurrences: chunks of 64 rows, fp32 matrix products
// (v_mfma_f32_16x16x4_f32), where a chunk lies, staging, and the inverse of a chunk's unit lower
// triangular matrix.
#pragma once

#include <algorithm>
#include <type_traits>

#include "mx_common.h"

namespace mx {

typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kC = 64;          // rows per chunk
// entry (row, col) of a staged tile of `ld` floats a row, 16-column blocks exchanged by the row: lanes (hi, lo) that read rows
// 4 s + hi, columns lo fall on all 64 banks, without padding (which cost chunk_out and state_add the third workgroup a CU)
template <int LD>
__device__ __forceinline__ int swizzled(int row, int col) { return row * LD + (col ^ ((row & 3) << 4)); }
constexpr int kVLD = 64;        // of a [rows][64 columns] tile
constexpr int kPLD = 68;        // floats between rows of a staged [16][64] strip

__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// a product over N inner steps of 4, a(s) and b(s) the operands of step s: four sums in turn, so
// that no product waits for the one before
template <int N, typename A, typename B>
__device__ __forceinline__ f32x4 dot_steps(A a, B b) {
  f32x4 p[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) p[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < N; ++s) p[s & 3] = mma(a(s), b(s), p[s & 3]);
  return (p[0] + p[1]) + (p[2] + p[3]);
}

// four consecutive entries as fp32 (16- or 8-byte load)
__device__ __forceinline__ void load4(const float* p, float* v) {
  const float4 u = *reinterpret_cast<const float4*>(p);
  v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w;
}
__device__ __forceinline__ void load4(const bf16_t* p, float* v) {
  const uint2 u = *reinterpret_cast<const uint2*>(p);
  ft::unpack2(u.x, v[0], v[1]);
  ft::unpack2(u.y, v[2], v[3]);
}

// Four neighbouring entries of a row on their way to LDS: what is fetched is put later, so a workgroup asks for all of a tile
// at once, and for the next one before it needs it (chunk_out of 2048 rows, 64 heads of 128 x 64, with loads behind a branch
// each, one after the other, 104 us; so 81; with three workgroups a CU 73).
template <typename T>
using Four = typename std::conditional<sizeof(T) == 2, uint2, float4>::type;
__device__ __forceinline__ float4 widen(const float4& u) { return u; }
__device__ __forceinline__ float4 widen(const uint2& u) {
  float4 v;
  ft::unpack2(u.x, v.x, v.y);
  ft::unpack2(u.y, v.z, v.w);
  return v;
}

// rows [0, cnt) x 64 columns from col0 of a [., dv] array (dv in whole fours), by 256 threads; rows past the end read the last
template <typename T>
__device__ __forceinline__ void fetch_cols(Four<T> (&u)[4], const T* src, long stride, int cnt, int col0, int dv) {
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const int e = threadIdx.x + 256 * n, t = min(e >> 4, cnt - 1), c = min(col0 + (e & 15) * 4, dv - 4);
    u[n] = *reinterpret_cast<const Four<T>*>(src + t * stride + c);
  }
}
// into LDS [kC][kVLD] (swizzled), zeros elsewhere
template <typename F>
__device__ __forceinline__ void put_cols(float* dst, const F (&u)[4], int cnt, int col0, int dv) {
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const int e = threadIdx.x + 256 * n, t = e >> 4, c = (e & 15) * 4;
    *reinterpret_cast<float4*>(dst + swizzled<kVLD>(t, c)) = t < cnt && col0 + c < dv ? widen(u[n]) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
}
template <typename T>
__device__ __forceinline__ void stage_cols(float* dst, const T* src, long stride, int cnt, int col0, int dv, int vec) {
  if (vec) {
    Four<T> u[4];
    fetch_cols<T>(u, src, stride, cnt, col0, dv);
    put_cols(dst, u, cnt, col0, dv);
  } else {
    for (int e = threadIdx.x; e < kC * 64; e += 256) {
      const int t = e >> 6, c = e & 63;
      dst[swizzled<kVLD>(t, c)] = t < cnt && col0 + c < dv ? ld(src, t * stride + col0 + c) : 0.f;
    }
  }
}

// the chunk of this workgroup: false if the segment has no such chunk (or is left to the walk)
struct Chunk {
  int cnt, num, pos, slot;
  long row0, ws;
};
__device__ __forceinline__ bool find_chunk(Chunk& c, int idx, int s, const int* start, const int* pos0, const int* slot,
                                           int min_rows, int num_slots) {
  const int r0 = start[s], n = start[s + 1] - r0;
  c.slot = slot[s];
  if (n < min_rows || n <= 0 || c.slot < 0 || c.slot >= num_slots) return false;
  c.num = (n + kC - 1) / kC;
  if (idx >= c.num) return false;
  c.cnt = min(kC, n - idx * kC);
  c.row0 = r0 + (long)idx * kC;
  c.pos = pos0[s] + idx * kC;
  c.ws = r0 / kC + s + idx;
  return true;
}

// A step's chunk kernels run over its chunks and not over as many per segment as its longest one has: a prompt beside 64
// decode rows would be one chunk in a hundred, and every empty workgroup waits for the LDS of a full one.  The counts are
// bounds from the step's rows; which segment a workgroup has it finds itself, unless all have the same number.
struct ChunkSteps {
  int num_segs, min_rows, per_seg;     // per_seg: chunks of every segment, or 0
};
// workgroup `item` of a unit: its segment and chunk; false if there is none (s: -1 if there is no such segment)
__device__ __forceinline__ bool find_chunk(Chunk& c, int item, const ChunkSteps& st, int& s, int& idx, const int* start,
                                           const int* pos0, const int* slot, int num_slots) {
  if (st.per_seg > 0) {
    s = item / st.per_seg, idx = item % st.per_seg;
  } else {
    s = -1;
    if (!segment_block(start, st.num_segs, st.min_rows, 1, kC, item, s, idx)) return false;
    s = __builtin_amdgcn_readfirstlane(s), idx = __builtin_amdgcn_readfirstlane(idx);
  }
  return find_chunk(c, idx, s, start, pos0, slot, st.min_rows, num_slots);
}
// the i-th of `longs` segments that have chunks (-1: none)
__device__ __forceinline__ int long_segment(int i, int longs, const ChunkSteps& st, const int* start) {
  if (longs == st.num_segs) return i;
  int s = -1, block;
  if (!segment_block(start, st.num_segs, st.min_rows, 1, 1 << 30, i, s, block)) return -1;
  return __builtin_amdgcn_readfirstlane(s);
}

// ab [kC][kPLD]: A below the diagonal (nothing else is read) -> T = (I + A)^-1, the blocks above the
// diagonal blocks left as they are.  The first four of WAVES waves work; what they read of the diagonal
// blocks of A has been written by the wave itself or before a barrier.
template <int WAVES = 4>
__device__ __forceinline__ void invert_unit_lower(float* ab, int wave, int lo, int hi) {
  wave_lds_fence();
  if (WAVES == 4 || wave < 4) {
    // the wave's own diagonal block: lane lo holds column lo of its inverse (the four quarters
    // of the wave do the same work)
    float* d = ab + 16 * wave * kPLD + 16 * wave;
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = i == lo ? 1.f : 0.f;
#pragma unroll
    for (int j = 0; j < 15; ++j)
#pragma unroll
      for (int i = j + 1; i < 16; ++i) x[i] -= d[i * kPLD + j] * x[j];
    wave_lds_fence();
    if (hi == 0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) d[i * kPLD + lo] = x[i];
    }
  }
  __syncthreads();
  // below the diagonal, one row of blocks after the other: T_ij = -T_ii sum_{j <= k < i} A_ik T_kj
#pragma unroll
  for (int i = 1; i < 4; ++i) {
    f32x4 t = f32x4{0.f, 0.f, 0.f, 0.f};
    const int j = wave;
    if (j < i) {
      f32x4 m = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < i; ++k) {
        if (k < j) continue;
#pragma unroll
        for (int s = 0; s < 4; ++s)
          m = mma(ab[(16 * i + lo) * kPLD + 16 * k + 4 * s + hi], ab[(16 * k + 4 * s + hi) * kPLD + 16 * j + lo], m);
      }
      // m in accumulator layout is a right-hand operand with inner index 4 hi + r
#pragma unroll
      for (int r = 0; r < 4; ++r) t = mma(-ab[(16 * i + lo) * kPLD + 16 * i + 4 * hi + r], m[r], t);
    }
    __syncthreads();
    if (j < i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) ab[(16 * i + 4 * hi + r) * kPLD + 16 * j + lo] = t[r];
    }
    __syncthreads();
  }
}

// operands of products T b with T (I + A)^-1: row tile m, inner step s (up to the tile's diagonal)
__device__ __forceinline__ void load_inverse(float (&tf)[4][16], const float* ab, int lo, int hi) {
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int s = 0; s < 4 * m + 4; ++s) tf[m][s] = ab[(16 * m + lo) * kPLD + 4 * s + hi];
}

// four row tiles of T b, or of its transpose (the operands in turn: their layouts are alike)
template <bool TRANSPOSED>
__device__ __forceinline__ void inverse_column(const float (&tf)[4][16], const float (&b)[16], f32x4 (&x)[4]) {
#pragma unroll
  for (int m = 0; m < 4; ++m) x[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < 16; ++s)
#pragma unroll
    for (int m = s / 4; m < 4; ++m) x[m] = TRANSPOSED ? mma(b[s], tf[m][s], x[m]) : mma(tf[m][s], b[s], x[m]);
}

// ---------------------------------------------------------------------------------
// grid (heads, ceil(dv / 16), long segments), four waves: the state's 16 columns, chunk after chunk.
// (Heads come first so that, 8 XCDs taking workgroups in turn, the column tiles of a head
// tend to share one XCD's L2: they all read the same operands.)
// Wave w holds the 16-row tiles w IT .. w IT + IT - 1 in accumulators; accumulator register r of
// lane (hi, lo) is row 4 hi + r, column lo, which is also a right-hand operand whose inner index
// 4 hi + r the left-hand operands (16-byte loads) follow.  Per chunk: every wave's part of
// -W S for all 64 rows, the parts added through LDS (wave w adds U and owns rows 16 w ..), w left
// in place of U, then S <- e^{G_last} S + K^T w.  Two register sets keep a chunk's operands
// on their way while the chunk before is computed.  FULL (whole tiles: dk = 16 DKT, dv a multiple of
// 16): no access is conditional, so nothing in the loop waits for more than it uses.
// CHANNEL: e^{G_last} per row of the state (ws_g [16 DKT] per chunk and head) instead of one number.
// SOLVED: as above; otherwise w is the rows of v themselves (linear attention, nothing to solve).
// ---------------------------------------------------------------------------------
template <int DKT, bool FULL, bool CHANNEL, bool SOLVED, typename TV>
__global__ void __launch_bounds__(256)
chunk_carry_kernel(float* __restrict__ ws_s, const float* __restrict__ ws_w, const float* __restrict__ ws_k,
                   float* __restrict__ ws_u, const float* __restrict__ ws_g, const TV* __restrict__ v_rows,
                   long v_stride, float* __restrict__ state, const int* __restrict__ start, const int* __restrict__ pos0, const int* __restrict__ slot, int heads,
                   int dk, int dv, int num_slots, ChunkSteps st) {
  constexpr int IT = DKT < 4 ? 1 : DKT / 4;
  __shared__ f32x4 part[SOLVED ? 4 : 1][4][64], whole[2][4][64];
  Chunk c;
  const int seg = long_segment(blockIdx.z, gridDim.z, st, start);
  if (seg < 0 || !find_chunk(c, 0, seg, start, pos0, slot, st.min_rows, num_slots)) return;
  const int h = blockIdx.x, rows = start[seg + 1] - start[seg];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lo = lane & 15, hi = lane >> 4;
  const int col = blockIdx.y * 16 + lo;
  const bool live = FULL || col < dv;
  const bool mine = DKT >= 4 || wave * IT < DKT;     // few tiles: some waves only add
  float* sp = state + (((long)c.slot * heads + h) * dk) * dv + col;
  f32x4 S[IT];
#pragma unroll
  for (int ii = 0; ii < IT; ++ii)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * (wave * IT + ii) + 4 * hi + r;
      S[ii][r] = c.pos > 0 && mine && live && row < dk ? sp[(long)row * dv] : 0.f;
    }
  struct Ops {
    f32x4 w[4][IT], k[IT][4], u, gr[IT];
    float g;
  };
  auto fetch = [&](Ops& f, int idx) {
    idx = min(idx, c.num - 1);         // past the end: loaded again, not used
    const long cs = (c.ws + idx) * heads + h;
    const f32x4* k = (const f32x4*)ws_k + cs * (4 * DKT * 64) + lane;
    if (mine) {
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int ii = 0; ii < IT; ++ii) {
          const int i = wave * IT + ii;
          if constexpr (SOLVED) f.w[m][ii] = ((const f32x4*)ws_w + cs * (4 * DKT * 64) + lane)[(m * DKT + i) * 64];
          f.k[ii][m] = k[(i * 4 + m) * 64];
        }
    }
    if constexpr (SOLVED) {
      f.u = ((const f32x4*)ws_u)[((cs * gridDim.y + blockIdx.y) * 4 + wave) * 64 + lane];
    } else {
      const int left = min(kC, rows - idx * kC);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * wave + 4 * hi + r;      // rows past the end read the last row and count as zeros
        const float x = ld(v_rows, (c.row0 + (long)idx * kC + min(t, left - 1)) * v_stride + (long)h * dv + (live ? col : dv - 1));
        f.u[r] = t < left ? x : 0.f;
      }
    }
    if constexpr (CHANNEL) {
#pragma unroll
      for (int ii = 0; ii < IT; ++ii)
        f.gr[ii] = *(const f32x4*)(ws_g + cs * (16 * DKT) + 16 * (mine ? wave * IT + ii : 0) + 4 * hi);
    } else {
      f.g = ws_g[cs];
    }
    asm volatile("" ::: "memory");     // the loads stay here: they are not moved to their uses, two chunks on
  };
  auto turn = [&](const Ops& f, int idx) {
    float* so = ws_s + (((c.ws + idx) * heads + h) * dk) * (long)dv + col;
    if (mine && live) {
#pragma unroll
      for (int ii = 0; ii < IT; ++ii)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 16 * (wave * IT + ii) + 4 * hi + r;
          if (FULL || row < dk) so[(long)row * dv] = S[ii][r];
        }
    }
    f32x4 v = f.u;
    if constexpr (SOLVED) {
      f32x4 a[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) a[m] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (mine) {
#pragma unroll
        for (int ii = 0; ii < IT; ++ii)
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int m = 0; m < 4; ++m) a[m] = mma(f.w[m][ii][r], S[ii][r], a[m]);
      }
#pragma unroll
      for (int m = 0; m < 4; ++m) part[m][wave][lane] = a[m];
      __syncthreads();
      {
        const f32x4 v0 = part[wave][0][lane], v1 = part[wave][1][lane], v2 = part[wave][2][lane], v3 = part[wave][3][lane];
        v = (f.u + v0) + (v1 + (v2 + v3));
      }
    }
    whole[idx & 1][wave][lane] = v;          // (two copies: a wave may still read the last chunk's)
    if constexpr (SOLVED) ((f32x4*)ws_u)[((((c.ws + idx) * heads + h) * gridDim.y + blockIdx.y) * 4 + wave) * 64 + lane] = v;
    __syncthreads();
    if (mine) {
      f32x4 vm[4], e[IT][2];             // two sums per tile in turn
#pragma unroll
      for (int m = 0; m < 4; ++m) vm[m] = whole[idx & 1][m][lane];
#pragma unroll
      for (int ii = 0; ii < IT; ++ii) {
        if constexpr (CHANNEL) e[ii][0] = S[ii] * f.gr[ii];
        else e[ii][0] = S[ii] * f.g;
        e[ii][1] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int ii = 0; ii < IT; ++ii) e[ii][r & 1] = mma(f.k[ii][m][r], vm[m][r], e[ii][r & 1]);
#pragma unroll
      for (int ii = 0; ii < IT; ++ii) S[ii] = e[ii][0] + e[ii][1];
    }
  };
  Ops fa, fb;
  fetch(fa, 0);
  fetch(fb, 1);
  for (int idx = 0; idx < c.num; idx += 2) {
    turn(fa, idx);
    fetch(fa, idx + 2);
    if (idx + 1 >= c.num) break;
    turn(fb, idx + 1);
    fetch(fb, idx + 3);
  }
  if (mine && live) {
#pragma unroll
    for (int ii = 0; ii < IT; ++ii)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * (wave * IT + ii) + 4 * hi + r;
        if (row < dk) sp[(long)row * dv] = S[ii][r];
      }
  }
}

}  // namespace mx

// The launches of a step of `rows` rows, segments of up to max_rows, those of at least min_rows in chunks.  grid(units): a
// workgroup per chunk and unit (head, or head and 64 columns), units fastest: workgroups go to the 8 XCDs in turn, so with
// chunks fastest segments of a multiple of eight put their first chunks, a short one's only ones, on the same XCD.  us, delta
// rule / linear attention / scan: 64 heads of 128 x 64, a segment of 1000 rows and ten of 100 436 261 221, with chunks
// fastest 1533 834 223 (walks 688 428 222); 128 of 64 x 32, one of 1000 beside 64 of one row 365 255 163, with a workgroup
// for every chunk that a segment could have 574 458 298 (429 253 181).
struct ChunkGrid {
  mx::ChunkSteps steps;
  long items;
  int longs;
  ChunkGrid(long rows, int max_rows, int min_rows, int num_segs) {
    const int most = (max_rows + mx::kC - 1) / mx::kC;
    longs = (int)std::max(1L, std::min((long)num_segs, rows / min_rows));
    items = std::min((long)most * num_segs, rows / mx::kC + longs);
    steps = {num_segs, min_rows, items == (long)most * num_segs ? most : 0};
  }
  bool fits(long units) const { return units <= 65535 && longs <= 65535 && items * units <= 0x7fffffffL; }
  dim3 grid(long units) const { return dim3((unsigned)(items * units)); }
};

// calls f with the key size's tile count as a constant
template <typename F>
static void key_tiles(int dk, F f) {
  const int t = (dk + 15) / 16;
  if (t <= 1) f(std::integral_constant<int, 1>{});
  else if (t <= 2) f(std::integral_constant<int, 2>{});
  else if (t <= 4) f(std::integral_constant<int, 4>{});
  else f(std::integral_constant<int, 8>{});
}


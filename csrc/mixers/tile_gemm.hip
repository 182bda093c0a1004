// Products of many bf16 rows with bf16 weights on the matrix units, fp32 accumulation:
//   C[r] = act(A[r] . W^T + bias), or, grouped, C[rows of g] = act(A[rows of g] . W[g]^T): rows sorted by group, group g's up
//   to offs[g]; A's rows optionally through an index (a row that several experts chose is read in place).
// W [groups, N, K] in the checkpoint's rows; gated forms: [gate | up] rows, 2 N of them.
//
// Both operands go from memory straight to LDS (global_load_lds, 16 bytes a lane), 64 elements of k a stage: rows of 128
// bytes whose 16-byte piece c lies at slot c ^ ((row >> 1) & 5), so the fragment reads hit all banks.  The weight is the left
// operand: a lane ends with four neighbouring columns of one row.  Gated: the staged columns alternate 16 of the gate and
// the same 16 of the up matrix, so a lane has both sums and the activation is part of the epilogue.  Results leave through
// LDS, whole rows of the tile at a time (written four columns a lane, 4096 x 4096 -> 2 x 14336 takes 700 us instead of 656).
//
// Five kernels, for different numbers of tiles (the table of forms below has the times of three):
//   tile_phase_kernel  256 x 256, eight waves in two groups half a phase apart: while one group's products run, the other's
//                      LDS reads and loads do (all eight in step, 4096 x 2048 -> 2 x 8192 takes 259 us instead of 225).
//                      Bound by the matrix units at the clock that the card's power leaves them: 4096 x 4096 -> 2 x 14336
//                      gated 656 us (1467 TFLOP/s; the vendor's product alone the same), or 700 with eight, four, eight and
//                      four reads a phase instead of six, as the LDS takes longer for eight than their products.
//   tile_ring_kernel   256 x 128 to 64 x 128, a ring of three to six stages: too few tiles for the large ones.  Bound by the
//                      LDS (16 fragment reads and a fifth of that written for 32 products).
//   tile_split_kernel  64 x 64 and smaller, eight waves that share a tile and split its k, each staging its own: few tiles,
//                      where the chain of stages with a barrier each is what takes the time (300 x 2048 -> 2048: 10 us, the ring
//                      14, the vendor 11).
//   tile_groups_kernel 256 x 256 for the whole tiles of each group and 128 or 64 x 256 for what is left of it, the whole ones
//                      first: 512 rows an expert are two tiles and a few rows for every other expert.  Bound by the matrix units or,
//                      up to a hundred rows a group, by the read of the matrices (5.4 TB/s).  us before and now, 32 experts: 4096
//                      rows, top 4, of 2048 -> 2 x 1024 and back 186 + 104, 145 + 86; 1872, of 2048 -> 1536 and back 65 + 92, 61 + 71;
//                      300, top 6, of 2048 -> 2 x 1024 71, 53.
//   tile_tail_kernel   256 x 256 while they fill all CUs, the rest of them as halves (below).
#include "few_rows.h"
#include "ft_lds.h"

#include <type_traits>

namespace mx {

constexpr int kTK = 64;              // k of a stage

struct TileArgs {
  bf16_t* C;
  const bf16_t* A;
  const int* rows;                   // A's row of every row, or null
  const bf16_t* W;
  const bf16_t* bias;
  const int* offs;                   // null: one group of all M rows
  long c_stride;
  unsigned a_bytes, w_bytes;         // between rows
  int groups, M, N, K, col_tiles, act, vec;
  float limit;
  float* parts;                      // PARTS kernels: [M][gridDim.y][N], the sums over a part of k each, instead of C
  int part_stages;                   // of k in a part
};

// a workgroup's group, rows row0 .. end - 1 of it and column tile
struct TileAt {
  int g, row0, end, ct;
};

// Tiles run group by group, in bands of eight row tiles with their columns after each other, and each XCD (workgroup id mod
// 8) takes a contiguous eighth of that order: the tiles in flight on an XCD share rows and columns in its L2.
template <int BM>
__device__ __forceinline__ bool tile_at(const TileArgs& P, int lane, TileAt& at) {
  const int x = blockIdx.x & 7, i = blockIdx.x >> 3, cols = P.col_tiles;
  int g = 0, lo = 0, hi = P.M, n = (P.M + BM - 1) / BM, first = 0;
  long t;
  if (P.offs == nullptr) {
    const int all = n * cols, q = all / 8, r = all % 8;
    if (i >= q + (x < r ? 1 : 0)) return false;
    t = x * q + min(x, r) + i;
  } else {
    // every wave sums the groups' row tiles, a lane a group
    auto span = [&](int k) {
      lo = k > 0 && k < P.groups ? min(max(P.offs[k - 1], 0), P.M) : 0;
      hi = k < P.groups ? min(max(P.offs[k], lo), P.M) : lo;
      n = (hi - lo + BM - 1) / BM;
      int upto = n;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(upto, o, 64);
        upto += lane >= o ? y : 0;
      }
      return upto;
    };
    int total = 0, upto = 0;
    for (int g0 = 0; g0 < P.groups; g0 += 64) {
      upto = span(g0 + lane);
      total += __shfl(upto, 63, 64);
    }
    const long all = (long)total * cols, per = (all + 7) / 8;
    t = x * per + i;
    if (i >= per || t >= all) return false;
    const int tile = (int)(t / cols);
    int base = 0;
    uint64_t past = 0;
    for (g = 0;; g += 64) {                     // (ends: tile < total)
      if (P.groups > 64) upto = span(g + lane);
      past = __ballot(base + upto > tile);
      if (past != 0 || g + 64 >= P.groups) break;
      base += __shfl(upto, 63, 64);
    }
    const int k = past != 0 ? __builtin_ctzll(past) : 63;
    g += k;
    lo = __builtin_amdgcn_readlane(lo, k);
    hi = __builtin_amdgcn_readlane(hi, k);
    n = __builtin_amdgcn_readlane(n, k);
    first = base + __builtin_amdgcn_readlane(upto, k) - n;
  }
  const int r = (int)(t - (long)first * cols), band = r / (8 * cols), in = r - band * 8 * cols, tall = min(8, n - 8 * band);
  at.g = __builtin_amdgcn_readfirstlane(g);
  at.ct = __builtin_amdgcn_readfirstlane(in / tall);
  at.row0 = __builtin_amdgcn_readfirstlane(lo + (8 * band + in % tall) * BM);
  at.end = __builtin_amdgcn_readfirstlane(hi);
  return true;
}

// 64 lanes' 16 bytes at base + off -> LDS at dst, lane after lane (base, dst: wave-uniform).  Not seen by the compiler's own
// waits: the kernels count them (vmcnt).
__device__ __forceinline__ void tile_dma(const void* base, unsigned off, uint32_t dst) {
  const uint64_t b = reinterpret_cast<uintptr_t>(base);
  const uint64_t from = (uint64_t)__builtin_amdgcn_readfirstlane((unsigned)(b >> 32)) << 32 |
                        (unsigned)__builtin_amdgcn_readfirstlane((unsigned)b);
  uint32_t keep;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %3\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(keep)
      : "v"(off), "s"(from), "s"(__builtin_amdgcn_readfirstlane(dst))
      : "memory");
}

// all but `ahead` (at most MOST) of a wave's stages of PW loads have landed
template <int PW, int MOST>
__device__ __forceinline__ void tile_wait(int ahead) {
  if constexpr (MOST >= 1) {
    static_assert(MOST * PW < 64, "vmcnt");
    if (ahead >= MOST) ft::vm_wait<MOST * PW>();
    else tile_wait<PW, MOST - 1>(ahead);
  } else {
    ft::vm_wait<0>();
  }
}

// byte offsets of a lane's piece of row r of the tile: rows past the group's end and columns past N repeat the last one
// (not stored)
__device__ __forceinline__ unsigned tile_a_off(const TileArgs& P, const TileAt& at, int r, int lane) {
  const int row = min(at.row0 + r, at.end - 1);
  return (unsigned)(P.rows != nullptr ? P.rows[row] : row) * P.a_bytes + (unsigned)(((lane & 7) ^ ((r >> 1) & 5)) * 16);
}
template <bool GLU>
__device__ __forceinline__ unsigned tile_w_off(const TileArgs& P, int n0, int r, int lane) {
  const int col = min(n0 + (GLU ? (r >> 5) * 16 + (r & 15) : r), P.N - 1);
  return (unsigned)((GLU && (r & 16) ? P.N : 0) + col) * P.w_bytes + (unsigned)(((lane & 7) ^ ((r >> 1) & 5)) * 16);
}

// SPREAD: the groups begin k at its eighths in turn.  Rows of 4 KB put one stage of all rows into few of the memory's channels,
// and with the workgroups all at the same stage those are what the read waits for: 32 matrices of 2 x 1024 x 2048 with up to 64 rows
// each 71 us (3.8 TB/s) in step, 50 (5.4) spread; 234 rows each 97 and 84.  A group's tiles stay in step, since they share rows in
// an L2 (by columns as well: both products of 2000 rows, top 4, 172 to 200 us).  By the group and not by the XCD: a row's sum is the
// same wherever its tile lies and whatever rows the other groups have.  Three eighths from a group to the next: an XCD
// has one or two of them under way, the next one the two after (us of both products, 32 experts of 1024, by XCD / one eighth on / three /
// g of n at the 8 g / n-th: 4096 rows 262 262 260 266; 300 rows, top 6 95 97 97 95; 64 experts of 1408 256 258 253 257; a group alone of
// 4096 rows, 2048 -> 2048 45 44 43 46).  Products of one matrix read it at that rate from a few rows on and gain nothing.
__device__ __forceinline__ int tile_first_stage(int g, int nk) { return (3 * g & 7) * nk / 8; }
template <bool SPREAD>
__device__ __forceinline__ int tile_stage_at(int t, int k0, int nk) {
  if constexpr (!SPREAD) return t;
  t += k0;
  return t >= nk ? t - nk : t;
}

template <bool GLU>
__device__ __forceinline__ void tile_result(const TileArgs& P, int col, const fr_f32x4& x, const fr_f32x4& up, float (&v)[4]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = x[e];
    if constexpr (GLU) {
      v[e] = fr_act(P.act, P.limit, v[e], up[e]);
    } else {
      if (P.bias != nullptr) v[e] += col + e < P.N ? ft::bf16_to_f32(P.bias[col + e]) : 0.f;
      if (P.act == kFrReluSq) v[e] = fr_act(P.act, P.limit, v[e], 0.f);
    }
  }
}

// a part's sums out, four columns a lane (N in whole fours); the bias goes with the first part
template <typename F>
__device__ __forceinline__ void tile_part_out(const TileArgs& P, int row0, int end, int n0, F put) {
  put([&](int r, int c, const fr_f32x4& x, const fr_f32x4&) {
    if (row0 + r >= end || n0 + c >= P.N) return;
    float v[4] = {x[0], x[1], x[2], x[3]};
    if (P.bias != nullptr && blockIdx.y == 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += ft::bf16_to_f32(P.bias[n0 + c + e]);
    }
    *reinterpret_cast<float4*>(P.parts + ((long)(row0 + r) * gridDim.y + blockIdx.y) * P.N + n0 + c) = make_float4(v[0], v[1], v[2], v[3]);
  });
}

// ROWS rows of OC results out: put(write) hands every lane's (row of the tile, column of the tile, sums, up sums) to `write`.  Where
// rows are whole 16-byte pieces through LDS (all of the workgroup's waves are past their last read of it), else directly.
template <int ROWS, int OC, int WAVES, bool GLU, typename F>
__device__ __forceinline__ void tile_out(const TileArgs& P, char* smem, int row0, int end, int n0, int tid, F put) {
  if (P.vec == 2) {
    constexpr int kRow = OC * 2 + 16, CPR = OC / 8;
    put([&](int r, int c, const fr_f32x4& x, const fr_f32x4& up) {
      float v[4];
      tile_result<GLU>(P, n0 + c, x, up, v);
      *reinterpret_cast<uint2*>(smem + r * kRow + c * 2) = make_uint2(ft::pack2(v[0], v[1]), ft::pack2(v[2], v[3]));
    });
    __syncthreads();
#pragma unroll
    for (int e = tid; e < ROWS * CPR; e += 64 * WAVES) {
      const int r = e / CPR, c = (e % CPR) * 8;
      const uint4 x = *reinterpret_cast<const uint4*>(smem + r * kRow + c * 2);
      if (row0 + r < end && n0 + c < P.N) *reinterpret_cast<uint4*>(P.C + (row0 + r) * P.c_stride + n0 + c) = x;
    }
    return;
  }
  put([&](int r, int c, const fr_f32x4& x, const fr_f32x4& up) {
    if (row0 + r >= end || n0 + c >= P.N) return;
    float v[4];
    tile_result<GLU>(P, n0 + c, x, up, v);
    fr_store4(P.C + (row0 + r) * P.c_stride, n0 + c, P.N, P.vec != 0, v);
  });
}

// ---------------------------------------------------------------------------------
// 256 rows x 256 staged columns, waves 2 (rows) x 4 (columns); a wave owns 64 rows x 32 columns of each quarter of the tile
// (halves lo / hi of either operand).  A stage takes four phases, a quarter's products each:
//   phase      0               1               2               3
//   quarter    A lo, W lo      A lo, W hi      A hi, W lo      A hi, W hi
//   reads      A lo (3 of 4)   W hi, A hi's 4th  A hi (3 of 4)   W lo, A lo's 4th of stage t + 1
//   loads      W lo            A lo            W hi            A hi        of stage t + 2
// A half is loaded into where the phase before read last, so four to six phases lie between a load and its read, with two
// slots.  Every phase: the loads that the next one reads have landed (counted; a barrier lies between), reads, loads,
// barrier, products, barrier.  The second group of waves runs one barrier behind the first.
// ---------------------------------------------------------------------------------
constexpr int kPhaseLds = 131072;

template <bool GLU, bool SPREAD = false>
__device__ __forceinline__ void tile_phase(const TileArgs& P, const TileAt& at, char* smem) {
  constexpr int QM = 4, QN = 2, HM = 32 * QM, HN = 64 * QN, BN = 2 * HN;
  constexpr int PA = HM / 64, PB = HN / 64;                         // loads a wave and half
  constexpr int kA = HM * 128, kB = HN * 128, kSlot = 2 * (kA + kB);
  constexpr int OC = GLU ? BN / 2 : BN;
  static_assert(2 * kSlot == kPhaseLds && HM * (OC * 2 + 16) <= 2 * kSlot, "results fit");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3, l15 = lane & 15, g4 = lane >> 4;
  const int n0 = at.ct * OC;
  const bf16_t* W = P.W + (long)at.g * P.N * (GLU ? 2 : 1) * P.K;
  const int nk = P.K / kTK, k0 = SPREAD ? tile_first_stage(at.g, nk) : 0;
  const uint32_t lds0 = ft::lds_off(smem);
  unsigned ap[2][PA], wp[2][PB];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int p = 0; p < PA; ++p) ap[h][p] = tile_a_off(P, at, h * HM + (wave + 8 * p) * 8 + (lane >> 3), lane);
#pragma unroll
    for (int p = 0; p < PB; ++p) wp[h][p] = tile_w_off<GLU>(P, n0, h * HN + (wave + 8 * p) * 8 + (lane >> 3), lane);
  }
  auto load_a = [&](int h, int t) {
    const int k = tile_stage_at<SPREAD>(t, k0, nk);
    const uint32_t dst = lds0 + (t & 1) * kSlot + h * kA + wave * 1024;
#pragma unroll
    for (int p = 0; p < PA; ++p) tile_dma(P.A + k * kTK, ap[h][p], dst + p * 8192);
  };
  auto load_w = [&](int h, int t) {
    const int k = tile_stage_at<SPREAD>(t, k0, nk);
    const uint32_t dst = lds0 + (t & 1) * kSlot + 2 * kA + h * kB + wave * 1024;
#pragma unroll
    for (int p = 0; p < PB; ++p) tile_dma(W + k * kTK, wp[h][p], dst + p * 8192);
  };
  fr_f32x4 acc[2][2][QN][QM];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int n = 0; n < QN; ++n)
#pragma unroll
        for (int m = 0; m < QM; ++m) acc[i][j][n][m] = fr_f32x4{0.f, 0.f, 0.f, 0.f};
  const int swz = (l15 >> 1) & 5;
  const int get[2] = {l15 * 128 + ((2 * g4) ^ swz) * 16, l15 * 128 + ((2 * g4 + 1) ^ swz) * 16};
  const char* as = smem + wm * QM * 2048;
  const char* ws = smem + 2 * kA + wn * QN * 2048;
  uint4 a[QM - 1][2], last[2][2], wl[QN][2], wh[QN][2];     // (last: the fourth row tile of A's lo and hi half)
  auto read_a = [&](int h, int t) {
    const char* s = as + (t & 1) * kSlot + h * kA;
#pragma unroll
    for (int m = 0; m < QM - 1; ++m)
#pragma unroll
      for (int k = 0; k < 2; ++k) a[m][k] = *reinterpret_cast<const uint4*>(s + get[k] + m * 2048);
  };
  auto read_last = [&](int h, int t) {
    const char* s = as + (t & 1) * kSlot + h * kA + (QM - 1) * 2048;
#pragma unroll
    for (int k = 0; k < 2; ++k) last[h][k] = *reinterpret_cast<const uint4*>(s + get[k]);
  };
  auto read_w = [&](uint4 (&w)[QN][2], int h, int t) {
    const char* s = ws + (t & 1) * kSlot + h * kB;
#pragma unroll
    for (int n = 0; n < QN; ++n)
#pragma unroll
      for (int k = 0; k < 2; ++k) w[n][k] = *reinterpret_cast<const uint4*>(s + get[k] + n * 2048);
  };
  auto products = [&](uint4 (&w)[QN][2], int mq, int nq) {
    ft::lgkm_wait<0>();           // (before the barrier: what these reads read is loaded over behind it)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int m = 0; m < QM; ++m)
#pragma unroll
        for (int n = 0; n < QN; ++n)
          acc[mq][nq][n][m] = fr_mfma(w[n][k], m == QM - 1 ? last[mq][k] : a[m < QM - 1 ? m : 0][k], acc[mq][nq][n][m]);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  // LEFT: stages behind this one (2: two or more)
  auto stage = [&](auto left, int t) {
    constexpr int LEFT = decltype(left)::value;
    ft::vm_wait<LEFT >= 1 ? 2 * PA + 2 * PB : 0>();           // A hi and W hi of t
    read_a(0, t);
    if constexpr (LEFT >= 2) load_w(0, t + 2);
    products(wl, 0, 0);
    read_w(wh, 1, t);
    read_last(1, t);
    if constexpr (LEFT >= 2) load_a(0, t + 2);
    products(wh, 0, 1);
    if constexpr (LEFT >= 1) ft::vm_wait<LEFT >= 2 ? 2 * PA + 2 * PB : PA + PB>();      // W lo and A lo of t + 1
    read_a(1, t);
    if constexpr (LEFT >= 2) load_w(1, t + 2);
    products(wl, 1, 0);
    if constexpr (LEFT >= 1) read_w(wl, 0, t + 1), read_last(0, t + 1);
    if constexpr (LEFT >= 2) load_a(1, t + 2);
    products(wh, 1, 1);
  };
  load_w(0, 0), load_a(0, 0), load_w(1, 0), load_a(1, 0);
  if (nk > 1) {
    load_w(0, 1), load_a(0, 1), load_w(1, 1), load_a(1, 1);
    ft::vm_wait<3 * PA + 3 * PB>();
  } else {
    ft::vm_wait<PA + PB>();
  }
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  read_w(wl, 0, 0);
  read_last(0, 0);
  ft::lgkm_wait<0>();
  if (wm == 1) __builtin_amdgcn_s_barrier();
  for (int t = 0; t + 2 < nk; ++t) stage(std::integral_constant<int, 2>{}, t);
  if (nk > 1) stage(std::integral_constant<int, 1>{}, nk - 2);
  stage(std::integral_constant<int, 0>{}, nk - 1);
  if (wm == 0) __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int mq = 0; mq < 2; ++mq) {
    if (mq) __syncthreads();
    tile_out<HM, OC, 8, GLU>(P, smem, at.row0 + mq * HM, at.end, n0, tid, [&](auto write) {
#pragma unroll
      for (int m = 0; m < QM; ++m)
#pragma unroll
        for (int nq = 0; nq < 2; ++nq)
#pragma unroll
          for (int n = 0; n < QN; n += GLU ? 2 : 1)
            write((wm * QM + m) * 16 + l15, (nq * HN + (wn * QN + n) * 16) / (GLU ? 2 : 1) + 4 * g4, acc[mq][nq][n][m],
                  acc[mq][nq][GLU ? n + 1 : n][m]);
    });
  }
}

template <bool GLU>
__global__ void __launch_bounds__(512, 1)
tile_phase_kernel(TileArgs P) {
  __shared__ __attribute__((aligned(16))) char smem[kPhaseLds];
  TileAt at;
  if (tile_at<256>(P, threadIdx.x & 63, at)) tile_phase<GLU>(P, at, smem);
}

// ---------------------------------------------------------------------------------
// WM x WN waves of MT x NT tiles of 16, a ring of S stages.  The operands of a stage's second half are read under its first
// half's products and the next stage's first half under the second's, a barrier a stage.
// ---------------------------------------------------------------------------------
template <int WM, int WN, int MT, int NT, int S>
constexpr int kRingLds = S * (WM * MT + WN * NT) * 16 * 128;

template <int WM, int WN, int MT, int NT, int S, bool GLU, bool SPREAD = false, bool PARTS = false>
__device__ __forceinline__ void tile_ring(const TileArgs& P, const TileAt& at, char* smem) {
  constexpr int NW = WM * WN, BM = WM * MT * 16, BN = WN * NT * 16;
  constexpr int PA = BM / (8 * NW), PB = BN / (8 * NW), PW = PA + PB;
  constexpr int kStage = (BM + BN) * 128, OC = GLU ? BN / 2 : BN;
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0 && (!GLU || NT % 2 == 0), "");
  static_assert(BM * (OC * 2 + 16) <= S * kStage && S >= 3, "");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN, l15 = lane & 15, g4 = lane >> 4;
  const int n0 = at.ct * OC;
  const int t0 = PARTS ? (int)blockIdx.y * P.part_stages : 0;
  const bf16_t *A = P.A + t0 * kTK, *W = P.W + (long)at.g * P.N * (GLU ? 2 : 1) * P.K + t0 * kTK;
  const int nk = PARTS ? min(P.part_stages, P.K / kTK - t0) : P.K / kTK, k0 = SPREAD ? tile_first_stage(at.g, nk) : 0;
  const uint32_t lds0 = ft::lds_off(smem);
  unsigned ap[PA], wp[PB];
#pragma unroll
  for (int p = 0; p < PA; ++p) ap[p] = tile_a_off(P, at, (wave + NW * p) * 8 + (lane >> 3), lane);
#pragma unroll
  for (int p = 0; p < PB; ++p) wp[p] = tile_w_off<GLU>(P, n0, (wave + NW * p) * 8 + (lane >> 3), lane);
  auto load1 = [&](int t, int slot, int p) {
    const uint32_t dst = lds0 + slot * kStage + wave * 1024;
    const int k = tile_stage_at<SPREAD>(t, k0, nk);
    if (p < PA) tile_dma(A + k * kTK, ap[p < PA ? p : 0], dst + p * NW * 1024);
    else tile_dma(W + k * kTK, wp[p < PA ? 0 : p - PA], dst + BM * 128 + (p - PA) * NW * 1024);
  };
  fr_f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = fr_f32x4{0.f, 0.f, 0.f, 0.f};
  const int swz = (l15 >> 1) & 5;
  const int get[2] = {l15 * 128 + ((2 * g4) ^ swz) * 16, l15 * 128 + ((2 * g4 + 1) ^ swz) * 16};
  const int a0 = wm * MT * 2048, w0 = BM * 128 + wn * NT * 2048;
  uint4 a[MT], w[2][NT];
  const std::integral_constant<int, 0> h0;
  const std::integral_constant<int, 1> h1;
  auto read_w = [&](auto half, int slot) {
    constexpr int H = decltype(half)::value;
#pragma unroll
    for (int i = 0; i < NT; ++i) w[H][i] = *reinterpret_cast<const uint4*>(smem + slot * kStage + get[H] + w0 + i * 2048);
  };
  auto read_a = [&](auto half, int slot, int j) {
    a[j] = *reinterpret_cast<const uint4*>(smem + slot * kStage + get[decltype(half)::value] + a0 + j * 2048);
  };
  auto product = [&](auto half, int j) {
    constexpr int H = decltype(half)::value;
#pragma unroll
    for (int i = 0; i < NT; ++i) acc[i][j] = fr_mfma(w[H][i], a[j], acc[i][j]);
  };
  // a's registers take the second half's operands as the first half's products are done with them
  auto first_half = [&](int slot) {
    __builtin_amdgcn_sched_barrier(0);
    read_w(h1, slot);
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      __builtin_amdgcn_sched_barrier(0);
      product(h0, j);
      read_a(h1, slot, j);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int t = 0; t < S; ++t)
    if (t < nk) {
#pragma unroll
      for (int p = 0; p < PW; ++p) load1(t, t, p);
    }
  tile_wait<PW, S - 1>(min(S - 1, nk - 1));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  read_w(h0, 0);
#pragma unroll
  for (int j = 0; j < MT; ++j) read_a(h0, 0, j);
  // products of the second half before the barrier, to cover the last reads
  constexpr int EARLY = (MT * 3 + 7) / 8, REST = MT - EARLY;
  int slot = 0;
  for (int t = 0; t + 1 < nk; ++t) {
    first_half(slot);
#pragma unroll
    for (int j = 0; j < EARLY; ++j) product(h1, j);
    __builtin_amdgcn_sched_barrier(0);
    tile_wait<PW, S - 2>(min(S - 2, nk - 2 - t));
    ft::lgkm_wait<0>();
    __builtin_amdgcn_s_barrier();
    const int old = slot;
    slot = slot + 1 == S ? 0 : slot + 1;
    __builtin_amdgcn_sched_barrier(0);
    read_w(h0, slot);
#pragma unroll
    for (int j = 0; j < EARLY; ++j) read_a(h0, slot, j);
    const bool more = t + S < nk;
#pragma unroll
    for (int j = EARLY; j < MT; ++j) {
      __builtin_amdgcn_sched_barrier(0);
      if (more) {
#pragma unroll
        for (int p = PW * (j - EARLY) / REST; p < PW * (j - EARLY + 1) / REST; ++p) load1(t + S, old, p);
      }
      __builtin_amdgcn_sched_barrier(0);
      product(h1, j);
      read_a(h0, slot, j);
    }
  }
  first_half(slot);
#pragma unroll
  for (int j = 0; j < MT; ++j) product(h1, j);
  const auto put = [&](auto write) {
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int i = 0; i < NT; i += GLU ? 2 : 1)
        write((wm * MT + j) * 16 + l15, (wn * NT + i) * 16 / (GLU ? 2 : 1) + 4 * g4, acc[i][j], acc[GLU ? i + 1 : i][j]);
  };
  if constexpr (PARTS) {
    tile_part_out(P, at.row0, at.end, n0, put);
    return;
  }
  __syncthreads();
  tile_out<BM, OC, NW, GLU>(P, smem, at.row0, at.end, n0, tid, put);
}

template <int WM, int WN, int MT, int NT, int S, bool GLU, bool PARTS = false>
__global__ void __launch_bounds__(64 * WM * WN, 1)
tile_ring_kernel(TileArgs P) {
  __shared__ __attribute__((aligned(16))) char smem[kRingLds<WM, WN, MT, NT, S>];
  TileAt at;
  if (tile_at<WM * MT * 16>(P, threadIdx.x & 63, at)) tile_ring<WM, WN, MT, NT, S, GLU, false, PARTS>(P, at, smem);
}

// ---------------------------------------------------------------------------------
// Groups in tiles of 256 rows and, for a last piece of at most 128 or 64 rows, of that many, which take half and a third of
// a whole one's time.
// ---------------------------------------------------------------------------------
// As tile_at, the groups' whole tiles (a last piece of more than 128 rows is one) before all shorter ones: the workgroups
// that are dispatched last take the least time.
__device__ __forceinline__ bool tile_at_groups(const TileArgs& P, int lane, TileAt& at, bool& shorter) {
  const int x = blockIdx.x & 7, cols = P.col_tiles;
  int i = blockIdx.x >> 3, lo = 0, hi = 0, whole = 0, part = 0;
  // lane's group's whole and short tiles; the sums over lanes up to it come back as whole * 128 + short (at most 64 of them)
  auto span = [&](int k) {
    lo = k > 0 && k < P.groups ? min(max(P.offs[k - 1], 0), P.M) : 0;
    hi = k < P.groups ? min(max(P.offs[k], lo), P.M) : lo;
    const int last = (hi - lo) & 255;
    whole = ((hi - lo) >> 8) + (last > 128 ? 1 : 0);
    part = last > 0 && last <= 128 ? 1 : 0;
    int upto = whole * 128 + part;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(upto, o, 64);
      upto += lane >= o ? y : 0;
    }
    return upto;
  };
  int wholes = 0, parts = 0, upto = 0;
  for (int g0 = 0; g0 < P.groups; g0 += 64) {
    upto = span(g0 + lane);
    const int sum = __shfl(upto, 63, 64);
    wholes += sum >> 7, parts += sum & 127;
  }
  long all = (long)wholes * cols, per = (all + 7) / 8;
  shorter = i >= per;
  if (shorter) i -= (int)per, all = (long)parts * cols, per = (all + 7) / 8;
  const long t = x * per + i;
  if (i >= per || t >= all) return false;
  const int tile = (int)(t / cols);
  int base = 0, g = 0;
  uint64_t past = 0;
  auto mine = [&](int v) { return shorter ? v & 127 : v >> 7; };
  for (;; g += 64) {                            // (ends: tile < the sum of all)
    if (P.groups > 64) upto = span(g + lane);
    past = __ballot(base + mine(upto) > tile);
    if (past != 0 || g + 64 >= P.groups) break;
    base += mine(__shfl(upto, 63, 64));
  }
  const int k = past != 0 ? __builtin_ctzll(past) : 63;
  lo = __builtin_amdgcn_readlane(lo, k);
  hi = __builtin_amdgcn_readlane(hi, k);
  const int n = __builtin_amdgcn_readlane(shorter ? part : whole, k);
  const int first = base + mine(__builtin_amdgcn_readlane(upto, k)) - n;
  const int r = (int)(t - (long)first * cols), band = r / (8 * cols), in = r - band * 8 * cols, tall = min(8, n - 8 * band);
  at.g = __builtin_amdgcn_readfirstlane(g + k);
  at.ct = __builtin_amdgcn_readfirstlane(in / tall);
  at.row0 = __builtin_amdgcn_readfirstlane(shorter ? hi - ((hi - lo) & 255) : lo + (8 * band + in % tall) * 256);
  at.end = __builtin_amdgcn_readfirstlane(hi);
  return true;
}

template <bool GLU>
__global__ void __launch_bounds__(512, 1)
tile_groups_kernel(TileArgs P) {
  constexpr int k64 = kRingLds<1, 8, 4, 2, 4>, k128 = kRingLds<2, 4, 4, 4, 3>;
  constexpr int kRing = k64 > k128 ? k64 : k128;
  __shared__ __attribute__((aligned(16))) char smem[kRing > kPhaseLds ? kRing : kPhaseLds];
  TileAt at;
  bool shorter;
  if (!tile_at_groups(P, threadIdx.x & 63, at, shorter)) return;
  if (!shorter) tile_phase<GLU, true>(P, at, smem);
  else if (at.end - at.row0 > 64) tile_ring<2, 4, 4, 4, 3, GLU, true>(P, at, smem);
  else tile_ring<1, 8, 4, 2, 4, GLU, true>(P, at, smem);
}

// ---------------------------------------------------------------------------------
// One group's tiles of 256 x 256 while they make whole rounds over the chip's 256 CUs, and the last ones, up to 128, as halves of
// 128 rows, a CU each: a round of those takes 0.7 of a whole one (their fragment reads bind them, as the ring's).  Bit for bit
// the whole tiles' results.  us, whole tiles alone and the vendor's product beside it: 4096 x 2048 -> 6144 87 (96, 89), 2048 x 2048 ->
// 10272 82 (90, 96), 2002 x 512 -> 9568 31 (36, 46).
// ---------------------------------------------------------------------------------
constexpr int kCus = 256;

template <bool GLU>
__global__ void __launch_bounds__(512, 1)
tile_tail_kernel(TileArgs P) {
  constexpr int kRing = kRingLds<2, 4, 4, 4, 3>;
  __shared__ __attribute__((aligned(16))) char smem[kRing > kPhaseLds ? kRing : kPhaseLds];
  const int n = (P.M + 255) / 256, cols = P.col_tiles, all = n * cols, whole = all / kCus * kCus, halves = 2 * (all - whole);
  const int x = blockIdx.x & 7, per = (halves + 7) / 8;
  int i = blockIdx.x >> 3, t, down = 0;
  const bool half = i >= whole / 8;
  if (half) {
    i -= whole / 8;
    const int u = x * per + i;
    if (i >= per || u >= halves) return;
    t = whole + u / 2, down = u % 2 * 128;
  } else {
    t = x * (whole / 8) + i;
  }
  const int band = t / (8 * cols), in = t - band * 8 * cols, tall = min(8, n - 8 * band);
  TileAt at;
  at.g = 0;
  at.ct = __builtin_amdgcn_readfirstlane(in / tall);
  at.row0 = __builtin_amdgcn_readfirstlane((8 * band + in % tall) * 256 + down);
  at.end = P.M;
  if (at.row0 >= P.M) return;
  if (half) tile_ring<2, 4, 4, 4, 3, GLU>(P, at, smem);
  else tile_phase<GLU, false>(P, at, smem);
}

// ---------------------------------------------------------------------------------
// KW waves that share a tile of MT x NT tiles of 16: wave w takes the stages w, w + KW, .. and stages its own operands
// (no barrier before the sums meet in LDS, in wave order).
// ---------------------------------------------------------------------------------
template <int KW, int MT, int NT, bool GLU, bool PARTS = false>
__global__ void __launch_bounds__(64 * KW, 1)
tile_split_kernel(TileArgs P) {
  constexpr int BM = MT * 16, BN = NT * 16, PA = BM / 8, PB = BN / 8;
  constexpr int kStage = (BM + BN) * 128, kRed = KW * MT * NT * 1024, OC = GLU ? BN / 2 : BN;
  static_assert(!GLU || NT % 2 == 0, "");
  constexpr int kLds = KW * kStage > kRed ? KW * kStage : kRed;
  __shared__ __attribute__((aligned(16))) char smem[kLds];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l15 = lane & 15, g4 = lane >> 4;
  TileAt at;
  if (!tile_at<BM>(P, lane, at)) return;
  const int n0 = at.ct * OC;
  const int t0 = PARTS ? (int)blockIdx.y * P.part_stages : 0;
  const bf16_t *A = P.A + t0 * kTK, *W = P.W + (long)at.g * P.N * (GLU ? 2 : 1) * P.K + t0 * kTK;
  const int nk = PARTS ? min(P.part_stages, P.K / kTK - t0) : P.K / kTK;
  const char* mine = smem + wave * kStage;
  const uint32_t lds0 = ft::lds_off(mine);
  unsigned ap[PA], wp[PB];
#pragma unroll
  for (int p = 0; p < PA; ++p) ap[p] = tile_a_off(P, at, p * 8 + (lane >> 3), lane);
#pragma unroll
  for (int p = 0; p < PB; ++p) wp[p] = tile_w_off<GLU>(P, n0, p * 8 + (lane >> 3), lane);
  auto load = [&](int t) {
#pragma unroll
    for (int p = 0; p < PA; ++p) tile_dma(A + t * kTK, ap[p], lds0 + p * 1024);
#pragma unroll
    for (int p = 0; p < PB; ++p) tile_dma(W + t * kTK, wp[p], lds0 + BM * 128 + p * 1024);
  };
  fr_f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = fr_f32x4{0.f, 0.f, 0.f, 0.f};
  const int swz = (l15 >> 1) & 5;
  const int get[2] = {l15 * 128 + ((2 * g4) ^ swz) * 16, l15 * 128 + ((2 * g4 + 1) ^ swz) * 16};
  if (wave < nk) load(wave);
  for (int t = wave; t < nk; t += KW) {
    ft::vm_wait<0>();
    __builtin_amdgcn_sched_barrier(0);
    uint4 a[2][MT], w[2][NT];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
#pragma unroll
      for (int n = 0; n < NT; ++n) w[k][n] = *reinterpret_cast<const uint4*>(mine + get[k] + BM * 128 + n * 2048);
#pragma unroll
      for (int m = 0; m < MT; ++m) a[k][m] = *reinterpret_cast<const uint4*>(mine + get[k] + m * 2048);
    }
    ft::lgkm_wait<0>();
    __builtin_amdgcn_sched_barrier(0);
    if (t + KW < nk) load(t + KW);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n][m] = fr_mfma(w[k][n], a[k][m], acc[n][m]);
    __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();
  float4* red = reinterpret_cast<float4*>(smem);
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m)
      red[((wave * NT + n) * MT + m) * 64 + lane] = make_float4(acc[n][m][0], acc[n][m][1], acc[n][m][2], acc[n][m][3]);
  __syncthreads();
  auto sum = [&](int n, int m, int l) {
    fr_f32x4 v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KW; ++k) {
      const float4 x = red[((k * NT + n) * MT + m) * 64 + l];
      v[0] += x.x, v[1] += x.y, v[2] += x.z, v[3] += x.w;
    }
    return v;
  };
  constexpr int NO = GLU ? NT / 2 : NT;
  for (int e = tid; e < NO * MT * 64; e += 64 * KW) {
    const int l = e & 63, m = (e >> 6) % MT, n = (e >> 6) / MT;
    const int row = at.row0 + 16 * m + (l & 15), col = n0 + 16 * n + 4 * (l >> 4);
    if (row >= at.end || col >= P.N) continue;
    const fr_f32x4 x = sum(GLU ? 2 * n : n, m, l);
    fr_f32x4 up = x;
    if constexpr (GLU) up = sum(2 * n + 1, m, l);
    if constexpr (PARTS) {
      tile_part_out(P, row, at.end, col, [&](auto write) { write(0, 0, x, up); });
      continue;
    }
    float v[4];
    tile_result<GLU>(P, col, x, up, v);
    fr_store4(P.C + row * P.c_stride, col, P.N, P.vec != 0, v);
  }
}

// A form's tile and its time, us, by the tiles a CU takes (r = tiles / 256, R = r rounded up; a workgroup a CU), each of nk stages:
//   begin + R (tile + nk * stage) + r (all_tile + nk * all_stage)
// the second part for what all CUs share (rates of the L2 and of memory, the card's power).  Fitted to 504 products of 65 to 4096
// rows, weights from HBM, N and K of 64 to 14336 (residuals 4 to 11 %); the form chosen takes 1.006 times the best one's
// time in the mean, 1.2 times at most.  kTileTail: whole tiles' rounds, and its last one's fitted beside them.
enum TileForm { kTile256x256, kTile256x128, kTile192x128, kTile128x128, kTile64x128, kTile64x64, kTile64x32, kTile32x64, kTileForms, kTileGroups = kTileForms, kTileTail };
struct TileSize {
  int rows, cols;
  float begin, tile, stage, all_stage, all_tile;
  float us(long tiles, float nk) const {
    return begin + (float)((tiles + 255) / 256) * (tile + nk * stage) + tiles / 256.f * (all_tile + nk * all_stage);
  }
};
constexpr TileSize kTileSizes[kTileForms] = {
    {256, 256, 1.7f, 5.8f, 0.885f, 0.503f, 5.6f}, {256, 128, 2.5f, 2.0f, 0.681f, 0.235f, 3.3f},
    {192, 128, 1.5f, 2.5f, 0.554f, 0.159f, 2.2f}, {128, 128, 2.1f, 1.2f, 0.461f, 0.094f, 1.8f},
    {64, 128, 2.4f, 0.3f, 0.326f, 0.059f, 1.5f},  {64, 64, 3.2f, 0.5f, 0.184f, 0.050f, 1.4f},
    {64, 32, 2.0f, 1.1f, 0.107f, 0.054f, 0.6f},   {32, 64, 2.0f, 0.9f, 0.127f, 0.040f, 0.8f}};

// (groups: of unknown rows, in the forms that take them)
int tile_pick(long M, int N, int K, bool glu, bool groups, float* us) {
  int best = 0;
  float least = 3e38f;
  for (int f = 0; f < kTileForms; ++f) {
    const TileSize& z = kTileSizes[f];
    const int oc = z.cols / (glu ? 2 : 1);
    const long tiles = ((M + z.rows - 1) / z.rows) * ((N + oc - 1) / oc);
    const float t = z.us(tiles, K / 64.f);
    if (t < least) least = t, best = f;
  }
  const long tiles = ((M + 255) / 256) * ((N + (glu ? 127 : 255)) / (glu ? 128 : 256)), last = tiles % kCus;
  if (!groups && tiles > kCus && last > 0 && last <= kCus / 2) {
    const TileSize& z = kTileSizes[kTile256x256];
    const float r = tiles / 256.f, nk = K / 64.f;
    const float t = z.begin + (tiles / kCus) * (z.tile + nk * z.stage) + 3.8f + nk * 0.685f + r * (z.all_tile + nk * z.all_stage);
    if (t < least) least = t, best = kTileTail;
  }
  if (us != nullptr) *us = least;
  return best;
}

// A product of few columns and long sums leaves most of the chip idle: up to 1024 rows of 2048 columns are 16 to 128 tiles.  With
// k in parts, as fp32 sums that the norm step behind adds, every CU has a tile of a shorter chain.  By the forms' times, which the
// parts' kernels keep to (60 products of 65 to 1024 rows: 0.6 to 1.08 of the estimate at whole parts), and what the norm step reads
// beside them, at 6 TB/s.  us in a graph with the norm step, weights from HBM, at 65 / 130 / 300 / 600 / 777 / 1024 rows
// (the sooner of the whole tiles and the vendor's beside them):
//   n = 2048, k = 4096    12 15 18 24 28 32 (16 16 23 30 31 34)     k = 8192   18 21 28 36 44 50 (25 25 36 47 52 56)
//   n = 3072, k = 8192    20 24 35 48 58 69 (26 29 37 56 67 71)     n = 4096, k = 14336   35 38 60 97 116 120 (47 59 79 117 120 134)
// Left whole: k below 4096 (n = k = 2048: 11 13 18 20 22 beside 11 14 18 19 21), more than 1024 rows, whose parts leave the
// caches (n = 2048, k = 8192, 2048 rows: 87 beside 76), and less than a tenth to gain (n = k = 4096, 777 rows: 48 beside 43).
int tile_parts(long M, int N, int K, int* form) {
  if (M > 1024 || K < 4096 || N % 4) return 1;
  float least;
  tile_pick(M, N, K, false, false, &least);
  least *= 0.9f;
  int best = 1;
  for (int f : {kTile256x128, kTile192x128, kTile128x128, kTile64x128, kTile64x64}) {
    const TileSize& z = kTileSizes[f];
    const long tiles = ((M + z.rows - 1) / z.rows) * ((N + z.cols - 1) / z.cols);
    for (int p : {2, 3, 4}) {
      const int stages = (K / 64 + p - 1) / p;       // (64 at least: no part is without any)
      if (M <= 256 && p == 3) continue;              // (a norm step that also routes takes two or four)
      const float t = z.us(tiles * p, (float)stages) + (float)M * N * 4 * (p - 1) / 6e6f;
      if (t < least) least = t, best = p, *form = f;
    }
  }
  return best;
}

template <bool GLU>
int tile_launch(TileArgs& P, int form, hipStream_t s) {
  if (form == kTileGroups) {
    P.col_tiles = (P.N + (GLU ? 127 : 255)) / (GLU ? 128 : 256);
    const long tiles = (P.M / 256 + (long)P.groups) * P.col_tiles;       // (a group has n / 256 rounded up)
    if (P.offs == nullptr || tiles > 0x7fffff00L) return -3;
    // (both sorts of tiles are eighths, rounded up)
    hipLaunchKernelGGL((tile_groups_kernel<GLU>), dim3((unsigned)((tiles + 21) / 8 * 8)), dim3(512), 0, s, P);
    return (int)hipGetLastError();
  }
  if (form == kTileTail) {
    P.col_tiles = (P.N + (GLU ? 127 : 255)) / (GLU ? 128 : 256);
    const long tiles = (P.M + 255L) / 256 * P.col_tiles, whole = tiles / kCus * kCus;
    if (P.offs != nullptr || tiles > 0x3fffff00L) return -3;
    hipLaunchKernelGGL((tile_tail_kernel<GLU>), dim3((unsigned)(whole + (2 * (tiles - whole) + 7) / 8 * 8)), dim3(512), 0, s, P);
    return (int)hipGetLastError();
  }
  const TileSize& z = kTileSizes[form];
  const int oc = z.cols / (GLU ? 2 : 1);
  P.col_tiles = (P.N + oc - 1) / oc;
  const long tiles = ((P.M + z.rows - 1L) / z.rows + (P.offs != nullptr ? P.groups : 0)) * (long)P.col_tiles;
  if (tiles > 0x7ffffff0L) return -3;
  const dim3 grid((unsigned)((tiles + 7) / 8 * 8)), block(512);
#define TG_GO(...) hipLaunchKernelGGL((__VA_ARGS__), grid, block, 0, s, P)
  switch (form) {
    case kTile256x256: TG_GO(tile_phase_kernel<GLU>); break;
    case kTile256x128: TG_GO(tile_ring_kernel<4, 2, 4, 4, 3, GLU>); break;
    case kTile192x128: TG_GO(tile_ring_kernel<4, 2, 3, 4, 3, GLU>); break;
    case kTile128x128: TG_GO(tile_ring_kernel<2, 4, 4, 2, 4, GLU>); break;
    case kTile64x128: TG_GO(tile_ring_kernel<2, 4, 2, 2, 6, GLU>); break;
    case kTile64x64: TG_GO(tile_split_kernel<8, 4, 4, GLU>); break;
    case kTile64x32: TG_GO(tile_split_kernel<8, 4, 2, GLU>); break;
    case kTile32x64: TG_GO(tile_split_kernel<8, 2, 4, GLU>); break;
    default: return -5;
  }
#undef TG_GO
  return (int)hipGetLastError();
}

}  // namespace mx

using namespace mx;

// us that a product is expected to take, and (tail, if not null) whether its last round of tiles is done in halves
extern "C" float mx_tile_gemm_us(long M, int N, int K, int glu, int* tail) {
  float us;
  const int form = tile_pick(M, N, K, glu != 0, false, &us);
  if (tail != nullptr) *tail = form == kTileTail;
  return us;
}

// Whether operands of these sizes are taken: rows of whole stages, offsets of 32 bits
extern "C" int mx_tile_gemm_fits(long M, int N, int K, long a_stride, int glu) {
  return K >= kTK && K % kTK == 0 && a_stride >= K && a_stride % 8 == 0 && M > 0 && N > 0 &&
         M * a_stride * 2 <= 0xffffffffL && (glu ? 2L : 1L) * N * K * 2 <= 0xffffffffL;
}

// C[r] = act(A[rows ? rows[r] : r] W[g]^T + bias), a_rows rows of A; act: few_rows.h; form < 0: by tile_pick
extern "C" int mx_tile_gemm(void* C, long c_stride, const void* A, long a_stride, long a_rows, const int* rows, const void* W,
                            const void* bias, const int* offs, int groups, long M, int N, int K, int act, float limit, int form,
                            hipStream_t s) {
  if (M <= 0 || N <= 0 || groups <= 0) return 0;
  const bool glu = act >= kFrGelu && act <= kFrClamp;
  if (act < kFrStore || act > kFrReluSq || form > kTileTail || M > 0x3fffffffL) return -1;
  if (!mx_tile_gemm_fits(a_rows, N, K, a_stride, glu)) return -1;
  if (((uintptr_t)A) % 16 || ((uintptr_t)W) % 16) return -2;
  if (glu && bias != nullptr) return -4;
  TileArgs P{(bf16_t*)C, (const bf16_t*)A, rows, (const bf16_t*)W, (const bf16_t*)bias, offs, c_stride,
             (unsigned)(a_stride * 2), (unsigned)(K * 2), groups, (int)M, N, K, 0, act, 0, limit};
  P.vec = c_stride % 8 == 0 && N % 8 == 0 && ((uintptr_t)C) % 16 == 0 ? 2 : c_stride % 4 == 0 && ((uintptr_t)C) % 8 == 0 ? 1 : 0;
  if (form < 0) form = tile_pick(M, N, K, glu, offs != nullptr, nullptr);
  return glu ? tile_launch<true>(P, form, s) : tile_launch<false>(P, form, s);
}

// into how many parts of k a product whose norm step adds them is cut; 1: not
extern "C" int mx_tile_parts(long M, int N, int K) {
  int form;
  return mx_tile_gemm_fits(M, N, K, K, 0) ? tile_parts(M, N, K, &form) : 1;
}

// D [M][mx_tile_parts][N] fp32: the sums of A W^T over parts of k (the first: + bias)
extern "C" int mx_tile_gemm_parts(float* D, const void* A, long a_stride, const void* W, const void* bias, long M, int N, int K,
                                  hipStream_t s) {
  if (M <= 0 || N <= 0) return 0;
  if (!mx_tile_gemm_fits(M, N, K, a_stride, 0)) return -1;
  if (((uintptr_t)A | (uintptr_t)W | (uintptr_t)D) % 16) return -2;
  int form;
  const int parts = tile_parts(M, N, K, &form);
  if (parts < 2) return -1;
  TileArgs P{nullptr, (const bf16_t*)A, nullptr, (const bf16_t*)W, (const bf16_t*)bias, nullptr, 0, (unsigned)(a_stride * 2),
             (unsigned)(K * 2), 1, (int)M, N, K, 0, kFrStore, 0, 0.f, D, (K / kTK + parts - 1) / parts};
  const TileSize& z = kTileSizes[form];
  P.col_tiles = (N + z.cols - 1) / z.cols;
  const long tiles = ((M + z.rows - 1L) / z.rows) * P.col_tiles;
  if (tiles > 0x7ffffff0L) return -3;
  const dim3 grid((unsigned)((tiles + 7) / 8 * 8), (unsigned)parts), block(512);
#define TG_GO(...) hipLaunchKernelGGL((__VA_ARGS__), grid, block, 0, s, P)
  switch (form) {
    case kTile256x128: TG_GO(tile_ring_kernel<4, 2, 4, 4, 3, false, true>); break;
    case kTile192x128: TG_GO(tile_ring_kernel<4, 2, 3, 4, 3, false, true>); break;
    case kTile128x128: TG_GO(tile_ring_kernel<2, 4, 4, 2, 4, false, true>); break;
    case kTile64x128: TG_GO(tile_ring_kernel<2, 4, 2, 2, 6, false, true>); break;
    case kTile64x64: TG_GO(tile_split_kernel<8, 4, 4, false, true>); break;
    default: return -5;
  }
#undef TG_GO
  return (int)hipGetLastError();
}

// the forms that grouped_gemm.hip takes
extern "C" int mx_tile_form_128() { return kTile128x128; }
extern "C" int mx_tile_form_256() { return kTile256x256; }
extern "C" int mx_tile_form_groups() { return kTileGroups; }

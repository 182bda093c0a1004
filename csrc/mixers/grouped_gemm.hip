// Mixture-of-experts on many rows (prefill), bf16, nothing read back on the host:
//   pair_sort        (row, choice) pairs in order of their expert: where each expert's pairs end, the row
//                    of every sorted pair and the place of every pair, one launch
//   grouped_gemm     C[rows of g] = act(A[rows of g] . W[g]^T), rows sorted by group, group g's rows up to
//                    offs[g]; W [G, N, K], fp32 accumulate; A's rows optionally through an index (a row that
//                    several experts chose is read in place), the activation in the epilogue
//   experts_merge    out[r] = sum_k w[r, k] d[place of pair (r, k)] + shared part
//
// grouped_gemm: a workgroup of four waves owns BM rows x 128 columns of one group, k in steps of 64 through
// two LDS copies (v_mfma_f32_16x16x32_bf16; a wave owns BM / 2 x 64).  Two steps of 16-byte loads are in
// flight in registers; the LDS reads of one half step run under the products of the other, one barrier a step.
// The weight is the left operand, so a lane ends with four neighbouring columns of a row.  Gated: the staged
// columns alternate 16 of the gate and the same 16 of the up matrix, so a lane has both sums.  Rows past a
// group's end and columns past N repeat the last one and are not stored; k past K counts as zero.
// LDS rows are 128 bytes with 16-byte pieces swapped by row (no bank conflicts; rows padded to 144 bytes:
// a third of the LDS cycles were conflicts).
// Tiles of 128 rows once the groups hold 96 on average, below that 64 (an expert's few rows leave most of a
// taller tile empty).  The tiles run group by group, bands of eight row tiles with their columns after each
// other, and each XCD (workgroup id mod 8) takes one contiguous eighth of that order, so the tiles in flight on
// an XCD share an expert's rows and columns in its L2.
// Serves short groups that do not fill the card otherwise, where it is bound by the read of the matrices, and rows that are no whole
// stages of tile_gemm.hip's: the others go there (grouped_form has the lines and both sides).  1800 pairs of 32 experts, 2048 -> 2 x 1024 gated (268 MB):
// 78 us in a model, with one step of loads in flight, a barrier between reads and products and tiles in grid order 98.
#include "few_rows.h"

#include <type_traits>

namespace mx {

constexpr int kGK = 64;

// 2 x 2 waves, each MT x 4 tiles of 16 x 16: BM = 32 MT rows, 128 staged columns
template <int MT, bool GLU>
__global__ void __launch_bounds__(256, 2)
grouped_gemm_kernel(bf16_t* __restrict__ C, const bf16_t* __restrict__ A, const int* __restrict__ rows,
                    const bf16_t* __restrict__ W, const int* __restrict__ offs, int groups, int M, int N, int K,
                    int col_tiles, int act, float limit, int vec) {
  constexpr int NT = 4, BM = 32 * MT, BN = 32 * NT;
  constexpr int PA = BM / 32, PW = BN / 32;
  constexpr int kStep = (BM + BN) * kGK;
  __shared__ __attribute__((aligned(16))) bf16_t stage[2 * kStep];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1, l15 = lane & 15, g4 = lane >> 4;

  // this workgroup's group, row tile and column tile: every wave sums the groups' row tiles, a lane a group
  int g, row0, end, ct;
  {
    auto span = [&](int i, int& lo, int& hi) {
      lo = i > 0 && i < groups ? min(max(offs[i - 1], 0), M) : 0;
      hi = i < groups ? min(max(offs[i], lo), M) : lo;
      return (hi - lo + BM - 1) / BM;
    };
    int total = 0, lo = 0, hi = 0, n = 0, upto = 0;
    for (int g0 = 0; g0 < groups; g0 += 64) {
      n = span(g0 + lane, lo, hi);
      upto = n;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int x = __shfl_up(upto, o, 64);
        upto += lane >= o ? x : 0;
      }
      total += __shfl(upto, 63, 64);
    }
    const long all = (long)total * col_tiles, per = (all + 7) / 8;
    const long t = (long)(blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per || t >= all) return;
    const int tile = (int)(t / col_tiles);
    int base = 0;
    uint64_t past = 0;
    for (g = 0;; g += 64) {                     // (ends: tile < total)
      if (groups > 64) {
        n = span(g + lane, lo, hi);
        upto = n;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const int x = __shfl_up(upto, o, 64);
          upto += lane >= o ? x : 0;
        }
      }
      past = __ballot(base + upto > tile);
      if (past != 0 || g + 64 >= groups) break;
      base += __shfl(upto, 63, 64);
    }
    const int at = past != 0 ? __builtin_ctzll(past) : 63;
    g += at;
    lo = __builtin_amdgcn_readlane(lo, at);
    hi = __builtin_amdgcn_readlane(hi, at);
    n = __builtin_amdgcn_readlane(n, at);
    const int first = base + __builtin_amdgcn_readlane(upto, at) - n;
    // inside the group: bands of eight row tiles, column tiles after each other, rows fastest
    const int r = (int)(t - (long)first * col_tiles), band = r / (8 * col_tiles);
    const int in = r - band * 8 * col_tiles, tall = min(8, n - 8 * band);
    ct = in / tall;
    row0 = lo + (8 * band + in % tall) * BM;
    end = hi;
  }
  const int n0 = ct * (GLU ? BN / 2 : BN);
  const bf16_t* Wg = W + (long)g * N * (GLU ? 2 : 1) * K;

  // a thread's pieces: row tid / 8 + 32 p of the tile, 8 elements at 8 (tid % 8); rows past the group's end
  // and columns past N repeat the last one (not stored)
  const int kp = (tid & 7) * 8;
  const bf16_t *ap[PA], *wp[PW];
#pragma unroll
  for (int p = 0; p < PA; ++p) {
    const int r = min(row0 + (tid >> 3) + 32 * p, end - 1);
    ap[p] = A + (long)(rows != nullptr ? rows[r] : r) * K;
  }
#pragma unroll
  for (int p = 0; p < PW; ++p) {
    const int r = (tid >> 3) + 32 * p;
    const int col = min(n0 + (GLU ? (r >> 5) * 16 + (r & 15) : r), N - 1);
    wp[p] = Wg + ((long)(GLU && (r & 16) ? N : 0) + col) * K;
  }
  uint4 ra[2][PA], rw[2][PW];
  auto fetch = [&](auto set, int k0) {
    constexpr int S = decltype(set)::value;
    const int k = min(k0 + kp, K - 8);        // (past K: loaded again, zeroed when staged)
#pragma unroll
    for (int p = 0; p < PA; ++p) ra[S][p] = *reinterpret_cast<const uint4*>(ap[p] + k);
#pragma unroll
    for (int p = 0; p < PW; ++p) rw[S][p] = *reinterpret_cast<const uint4*>(wp[p] + k);
  };
  fr_f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = fr_f32x4{0.f, 0.f, 0.f, 0.f};

  // LDS: rows of 128 bytes, 16-byte piece c of row r at slot c ^ swz(r); a lane's fragment of half h of a
  // step is piece 2 g4 + h of its row, for both operands
  const auto swz = [](int r) { return (r >> 1) & 5; };
  const int put = (tid >> 3) * kGK + ((tid & 7) ^ swz(tid >> 3)) * 8;
  const int get[2] = {l15 * kGK + ((2 * g4) ^ swz(l15)) * 8, l15 * kGK + ((2 * g4 + 1) ^ swz(l15)) * 8};
  uint4 a[2][MT], b[2][NT];
  auto stage_in = [&](auto set, int k0) {       // registers of step k0 -> LDS copy `set`
    constexpr int S = decltype(set)::value;
    if (k0 + kGK > K && k0 + kp >= K) {
#pragma unroll
      for (int p = 0; p < PA; ++p) ra[S][p] = uint4{0, 0, 0, 0};
#pragma unroll
      for (int p = 0; p < PW; ++p) rw[S][p] = uint4{0, 0, 0, 0};
    }
#pragma unroll
    for (int p = 0; p < PA; ++p) *reinterpret_cast<uint4*>(stage + S * kStep + put + 32 * p * kGK) = ra[S][p];
#pragma unroll
    for (int p = 0; p < PW; ++p) *reinterpret_cast<uint4*>(stage + S * kStep + BM * kGK + put + 32 * p * kGK) = rw[S][p];
  };
  auto read = [&](auto set, auto half) {
    constexpr int S = decltype(set)::value, H = decltype(half)::value;
#pragma unroll
    for (int j = 0; j < MT; ++j)
      a[H][j] = *reinterpret_cast<const uint4*>(stage + S * kStep + (wm * MT + j) * 16 * kGK + get[H]);
#pragma unroll
    for (int i = 0; i < NT; ++i)
      b[H][i] = *reinterpret_cast<const uint4*>(stage + S * kStep + (BM + (wn * NT + i) * 16) * kGK + get[H]);
  };
  auto product = [&](auto half) {
    constexpr int H = decltype(half)::value;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[i][j] = fr_mfma(b[H][i], a[H][j], acc[i][j]);
  };
  const std::integral_constant<int, 0> even, lo_half;
  const std::integral_constant<int, 1> odd, hi_half;
  // Step k0 (copy `set` staged, its low half in registers): the high half's reads under the low half's
  // products, the next step's staging, one barrier, the next low half's reads under the high half's products.
  // The barrier also ends every wave's reads of a copy before its next writes, a step later.
  auto step = [&](auto set, auto next, auto last, int k0) {
    read(set, hi_half);
    __builtin_amdgcn_sched_barrier(0);
    product(lo_half);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!decltype(last)::value) {
      stage_in(next, k0 + kGK);
      fetch(next, k0 + 3 * kGK);
      __syncthreads();
      read(next, lo_half);
      __builtin_amdgcn_sched_barrier(0);
    }
    product(hi_half);
    __builtin_amdgcn_sched_barrier(0);
  };
  fetch(even, 0);
  __builtin_amdgcn_sched_barrier(0);        // (loads in the order they are waited for)
  fetch(odd, kGK);
  __builtin_amdgcn_sched_barrier(0);
  stage_in(even, 0);
  fetch(even, 2 * kGK);
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();
  read(even, lo_half);
  int k0 = 0;
  for (; k0 + 2 * kGK < K; k0 += 2 * kGK) {
    step(even, odd, std::false_type{}, k0);
    step(odd, even, std::false_type{}, k0 + kGK);
  }
  if (k0 + kGK < K) {
    step(even, odd, std::false_type{}, k0);
    step(odd, even, std::true_type{}, k0 + kGK);
  } else {
    step(even, odd, std::true_type{}, k0);
  }
  // lane (g4, l15) holds columns 4 g4 .. 4 g4 + 3 of row l15 of each 16 x 16 tile
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int row = row0 + (wm * MT + j) * 16 + l15;
    if (row >= end) continue;
#pragma unroll
    for (int i = 0; i < NT; i += GLU ? 2 : 1) {
      const int col = n0 + (GLU ? (wn * NT + i) * 8 : (wn * NT + i) * 16) + 4 * g4;
      if (col >= N) continue;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = acc[i][j][e];
        if constexpr (GLU) v[e] = fr_act(act, limit, v[e], acc[i + 1][j][e]);
        else if (act == kFrReluSq) v[e] = fr_act(act, limit, v[e], 0.f);
      }
      fr_store4(C + (long)row * N, col, N, vec != 0, v);
    }
  }
}

__device__ __forceinline__ void mx_unpack4(const bf16_t* p, float (&x)[4]) {
  const uint2 u = *reinterpret_cast<const uint2*>(p);
  ft::unpack2(u.x, x[0], x[1]);
  ft::unpack2(u.y, x[2], x[3]);
}

// Bound by one pass over the indices per expert, all workgroups at once: 6 us for 8000 pairs of 32 experts
// (a radix sort, count, running sum and scatter of the library: ~45 us in 12 launches).
// One workgroup per expert: the pairs of smaller experts (counted first) lie before its own, which keep
// their order.  A thread takes four neighbouring pairs a turn.
constexpr int kSortThreads = 1024, kSortWaves = kSortThreads / 64;

__global__ void __launch_bounds__(kSortThreads)
pair_sort_kernel(int* __restrict__ offs, int* __restrict__ sorted_row, int* __restrict__ place,
                 const int* __restrict__ idx, int pairs, int top, int experts, int vec) {
  __shared__ int less_s[kSortWaves], same_s[2][kSortWaves];
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // (an index outside the experts counts as the first's, so every pair has one place; past the end: -1)
  auto four = [&](int p, int (&x)[4]) {
    if (vec && p + 3 < pairs) {
      const int4 v = *reinterpret_cast<const int4*>(idx + p);
      x[0] = v.x, x[1] = v.y, x[2] = v.z, x[3] = v.w;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = p + i < pairs ? idx[p + i] : 0;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = p + i >= pairs ? -1 : x[i] < 0 || x[i] >= experts ? 0 : x[i];
  };
  int less = 0;
  for (int p = 4 * tid; p < pairs; p += 4 * kSortThreads) {
    int x[4];
    four(p, x);
#pragma unroll
    for (int i = 0; i < 4; ++i) less += x[i] >= 0 && x[i] < e;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) less += __shfl_xor(less, o, 64);
  if (lane == 0) less_s[wave] = less;
  __syncthreads();
  int at = 0;
#pragma unroll
  for (int w = 0; w < kSortWaves; ++w) at += less_s[w];
  int turn = 0;
  for (int p0 = 0; p0 < pairs; p0 += 4 * kSortThreads, turn ^= 1) {
    const int p = p0 + 4 * tid;
    int x[4], lower = 0, all = 0;
    four(p, x);
    const uint64_t below = (1ull << lane) - 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint64_t m = __ballot(x[i] == e);
      lower += __popcll(m & below);
      all += __popcll(m);
    }
    if (lane == 0) same_s[turn][wave] = all;
    __syncthreads();        // (two copies: a wave a turn ahead writes the other one)
    int pos = at + lower;
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) {
      const int n = same_s[turn][w];
      pos += w < wave ? n : 0;
      at += n;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (x[i] == e) {
        sorted_row[pos] = (p + i) / top;
        place[p + i] = pos++;
      }
  }
  if (tid == 0) offs[e] = at;
}

// Bound by reading d once: 13 us for 2000 rows of 2048, 4 experts and a shared one (the rows filled, added and
// the shared part added in passes of their own: 45 us).
// One workgroup per row: out[row] = sum_k wts[row, k] d[place[row, k]] (+ shared[row], times
// sigmoid(h[row] . gate_w) if there is a gate), fp32.
__global__ void __launch_bounds__(256)
experts_merge_kernel(float* __restrict__ out, const bf16_t* __restrict__ d, const int* __restrict__ place,
                     const float* __restrict__ wts, const bf16_t* __restrict__ shared, const bf16_t* __restrict__ h,
                     long h_stride, const bf16_t* __restrict__ gate_w, int top, int width) {
  __shared__ float part[4];
  const long row = blockIdx.x;
  const int tid = threadIdx.x;
  float gate = 1.f;
  if (gate_w != nullptr) {
    float dot = 0.f;
    for (int c = tid * 4; c < width; c += 1024) {
      float x[4], w[4];
      mx_unpack4(h + row * h_stride + c, x);
      mx_unpack4(gate_w + c, w);
#pragma unroll
      for (int i = 0; i < 4; ++i) dot += x[i] * w[i];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) dot += __shfl_xor(dot, o, 64);
    if ((tid & 63) == 0) part[tid >> 6] = dot;
    __syncthreads();
    gate = sigmoidf_(part[0] + part[1] + part[2] + part[3]);
  }
  for (int c = tid * 4; c < width; c += 1024) {
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    auto add = [&](const bf16_t* p, float w) {
      float x[4];
      mx_unpack4(p, x);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] += w * x[i];
    };
#pragma unroll 4
    for (int k = 0; k < top; ++k) add(d + (long)place[row * top + k] * width + c, wts[row * top + k]);
    if (shared != nullptr) add(shared + row * width + c, gate);
    *reinterpret_cast<float4*>(out + row * width + c) = make_float4(v[0], v[1], v[2], v[3]);
  }
}

}  // namespace mx

using namespace mx;

extern "C" int mx_tile_gemm_fits(long M, int N, int K, long a_stride, int glu);
extern "C" int mx_tile_gemm(void* C, long c_stride, const void* A, long a_stride, long a_rows, const int* rows, const void* W,
                            const void* bias, const int* offs, int groups, long M, int N, int K, int act, float limit, int form,
                            hipStream_t s);
extern "C" int mx_tile_form_128();
extern "C" int mx_tile_form_256();
extern "C" int mx_tile_form_groups();

enum { kTilesHere = 1000 };

// The form for rows of whole stages, by rows a group on average and by how far the tiles fill the card (a workgroup a CU in tile_gemm.hip's).
//
// By rows alone: 64-row tiles here, 128 x 128 from 50, 256 x 256 from 120.  Short pieces beside whole tiles (tile_groups_kernel) instead
// while columns do not leave a quarter of the tiles empty, and:
//  * up to 120 rows, a piece a group: where the last round of pieces over the 256 CUs is full to 144 of them or there are two before it.  Its
//    time over the other form's, by pieces (groups that have rows, times columns of tiles) 60-100 100-128 150-200 225-256 256-350 350-420
//    420-512 more:  50 to 90 rows 1.38 1.24 0.86 0.92 1.04 1.00 0.89 0.90;  20 to 50 rows 1.27 1.14 0.89 0.95 1.10 1.00 0.95 1.01;
//    below 20 1.30 1.18 0.91 1.01 1.12 1.05 1.02 1.07.  In the last two rows only where it is below 1.
//  * so too with more pieces where a matrix's rows are whole 4 KB, which meet on few of the memory's channels in the other forms (tile_first_stage):
//    0.80 to 0.95, with more than 768 pieces of below 20 rows 1.07.
//  * from 120 rows on while whole tiles leave a short last piece or a few groups end just past one: up to 128 rows past whole tiles 0.86 to
//    0.97, 220 to 255 0.95 to 1.0, between these all are whole tiles and it is behind by the rounding of both sorts (1.01 to 1.04, up to
//    1.5; rows of 4 KB 0.94).  Of sets of 256 MB and more, which the last level cache does not hold, the short pieces read the matrices a
//    second time: at 24 to 128 rows past a whole tile 1.05 (320 to 384), 1.05 (560 to 640).
// Over 4300 products of 2 to 256 groups, 1 to 900 rows each, sizes at random (1500 of them after the lines were drawn): 0.982 of the time by
// rows alone in the mean, above 1.03 in 68 and above 1.1 in 12 of them.
static int grouped_form(int groups, long M, int N, int K, bool glu) {
  const int width = glu ? 128 : 256, cols = (N + width - 1) / width;
  const float mean = (float)M / groups;
  const int by_rows = mean >= 120.f ? mx_tile_form_256() : mean >= 50.f ? mx_tile_form_128() : kTilesHere;
  if (4L * N < 3L * cols * width) return by_rows;
  const bool in_step = K % 2048 == 0;
  if (mean < 120.f) {
    const float pieces = groups * (1.f - expf(-mean)) * cols;              // (rows that choose their groups independently)
    const int rounds = (int)ceilf(pieces / 256.f);
    if (rounds <= 2 && pieces - 256.f * (rounds - 1) < 144.f) return by_rows;
    const bool few = mean >= 20.f ? rounds <= (in_step ? rounds : 2) : in_step ? rounds <= 3 : pieces <= 200.f;
    return mean >= 50.f || few ? mx_tile_form_groups() : by_rows;
  }
  if ((long)groups * cols < 128) return by_rows;
  const long past = M / groups % 256;
  if (past >= 128 && past < 220) return in_step ? mx_tile_form_groups() : by_rows;
  const bool twice = 2L * groups * N * K * (glu ? 2 : 1) >= 256L << 20 && M > 256L * groups && past > 24 && past <= 128;
  return twice ? by_rows : mx_tile_form_groups();
}

// act: few_rows.h (0: none).  a_rows: rows of A (M without an index).  rows: A's row of every sorted row, or null.  form: one of
// tile_gemm.hip's for groups, kTilesHere for the kernel above, or below 0 the one that is taken by itself.
extern "C" int mx_grouped_gemm(void* C, const void* A, long a_rows, const int* rows, const void* W, const int* offs, int groups,
                               long M, int N, int K, int act, float limit, int form, hipStream_t s) {
  if (M <= 0 || N <= 0 || groups <= 0) return 0;
  if (K < 8 || K % 8 || M > 0x7fffffffL || act < kFrStore || act > kFrReluSq) return -1;
  if (((uintptr_t)A) % 16 || ((uintptr_t)W) % 16) return -2;
  const bool glu = act >= kFrGelu && act <= kFrClamp;
  const int vec = N % 4 == 0 && ((uintptr_t)C) % 8 == 0;
  if ((M + 63) / 64 + groups > 65535) return -3;
  if (form < 0 && mx_tile_gemm_fits(a_rows, N, K, K, glu)) form = grouped_form(groups, M, N, K, glu);
  if (form >= 0 && form != kTilesHere && form != mx_tile_form_groups() && form != mx_tile_form_256() && form != mx_tile_form_128()) return -4;
  if (form >= 0 && form != kTilesHere)
    return mx_tile_gemm(C, N, A, K, a_rows, rows, W, nullptr, offs, groups, M, N, K, act, limit, form, s);
  // 128-row tiles once the groups fill them on average
  const bool tall = M >= 96L * groups;
  const int cols = 128 / (glu ? 2 : 1), col_tiles = (N + cols - 1) / cols;
  const long tiles = ((M + (tall ? 127 : 63)) / (tall ? 128 : 64) + groups) * col_tiles;
  if (tiles > 0x7ffffff0L) return -3;
  const dim3 grid((unsigned)((tiles + 7) / 8 * 8));
#define GG_GO(MT, GLU)                                                                                       \
  hipLaunchKernelGGL((grouped_gemm_kernel<MT, GLU>), grid, dim3(256), 0, s, (bf16_t*)C, (const bf16_t*)A, rows, \
                     (const bf16_t*)W, offs, groups, (int)M, N, K, col_tiles, act, limit, vec)
  if (tall) {
    if (glu) GG_GO(4, true); else GG_GO(4, false);
  } else {
    if (glu) GG_GO(2, true); else GG_GO(2, false);
  }
#undef GG_GO
  return (int)hipGetLastError();
}

// idx int32 [rows, top] -> offs [experts], sorted_row and place [rows * top]
extern "C" int mx_pair_sort(int* offs, int* sorted_row, int* place, const int* idx, long rows, int top, int experts,
                            hipStream_t s) {
  if (rows <= 0) return 0;
  if (experts < 1 || top < 1 || rows * top > 0x3fffffffL) return -1;
  hipLaunchKernelGGL(pair_sort_kernel, dim3((unsigned)experts), dim3(kSortThreads), 0, s, offs, sorted_row, place, idx,
                     (int)(rows * top), top, experts, (int)(((uintptr_t)idx) % 16 == 0));
  return (int)hipGetLastError();
}

extern "C" int mx_experts_merge(float* out, const void* d, const int* place, const float* wts, const void* shared,
                                const void* h, long h_stride, const void* gate_w, long rows, int top, int width,
                                hipStream_t s) {
  if (rows <= 0) return 0;
  if (width % 4 || top < 1 || rows > 0x7fffffffL) return -1;
  if (((uintptr_t)out) % 16 || ((uintptr_t)d) % 8 || ((uintptr_t)shared) % 8) return -2;
  if (gate_w != nullptr && (h_stride % 4 || ((uintptr_t)h) % 8 || ((uintptr_t)gate_w) % 8)) return -2;
  hipLaunchKernelGGL(experts_merge_kernel, dim3((unsigned)rows), dim3(256), 0, s, out, (const bf16_t*)d, place, wts,
                     (const bf16_t*)shared, (const bf16_t*)h, h_stride, (const bf16_t*)gate_w, top, width);
  return (int)hipGetLastError();
}

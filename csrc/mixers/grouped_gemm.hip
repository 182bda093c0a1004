// Mixture-of-experts on many rows (prefill), bf16, nothing read back on the host:
//   pair_sort        (row, choice) pairs in order of their expert: where each expert's pairs end, the row
//                    of every sorted pair and the place of every pair, one launch
//   grouped_gemm     C[rows of g] = act(A[rows of g] . W[g]^T), rows sorted by group, group g's rows up to
//                    offs[g]; W [G, N, K], fp32 accumulate; A's rows optionally through an index (a row that
//                    several experts chose is read in place), the activation in the epilogue
//   experts_merge    out[r] = sum_k w[r, k] d[place of pair (r, k)] + shared part
//
// grouped_gemm: a workgroup of four waves owns BM rows x BN columns of one group (blockIdx.y walks the
// groups' row tiles; slots past the last tile exit at once), k in steps of 64 through two LDS copies
// with the next step's 16-byte loads in flight during the products (v_mfma_f32_16x16x32_bf16).  The weight
// is the left operand, so a lane ends with four neighbouring columns of a row.  Gated: the staged columns
// alternate 16 of the gate and the same 16 of the up matrix, so a lane has both sums.  Rows past a
// group's end, columns past N and k past K are zero-filled on load and not stored.
// Tiles of 128 rows once the groups hold 96 on average, below that 64 (an expert's few rows leave most of a
// taller tile empty).  16384 pairs of 32 experts, 2048 -> 2 x 1024 gated: 242 us (570 TFLOP/s), 64 x 64 tiles
// with the gathered rows, the activation and its round trip in kernels of their own 270 + 60 + 50; whole
// layers of 2000 rows, 32 experts: 0.95 -> 0.50 ms and 24 -> 8 launches.
// The column tiles come first in the grid: with eight XCDs taking workgroups in turn, an expert's
// column tile stays in one XCD's L2 for all of the expert's row tiles.
#include "few_rows.h"

namespace mx {

constexpr int kGK = 64;
constexpr int kGLd = kGK + 8;        // LDS row stride (bf16): 144 bytes, keeps 16-byte alignment

template <int BM, int BN, bool GLU>
__global__ void __launch_bounds__(256, 2)
grouped_gemm_kernel(bf16_t* __restrict__ C, const bf16_t* __restrict__ A, const int* __restrict__ rows,
                    const bf16_t* __restrict__ W, const int* __restrict__ offs, int groups, int M, int N, int K, int act,
                    float limit, int vec) {
  constexpr int MT = BM / 32, NT = BN / 32;          // 16-wide tiles of a wave (2 x 2 waves)
  constexpr int PA = BM * 8 / 256, PW = BN * 8 / 256;
  constexpr int kStep = (BM + BN) * kGLd;
  __shared__ __attribute__((aligned(16))) bf16_t stage[2 * kStep];
  // this workgroup's group and row tile
  int g = 0, row0 = 0, end = 0;
  {
    int t = blockIdx.y, prev = 0;
    bool found = false;
    for (g = 0; g < groups; ++g) {
      end = min(max(offs[g], prev), M);
      const int tiles = (end - prev + BM - 1) / BM;
      if (t < tiles) {
        row0 = prev + t * BM;
        found = true;
        break;
      }
      t -= tiles;
      prev = end;
    }
    if (!found) return;
  }
  const int n0 = blockIdx.x * (GLU ? BN / 2 : BN);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1, l15 = lane & 15, g4 = lane >> 4;
  const bf16_t* Wg = W + (long)g * N * (GLU ? 2 : 1) * K;

  // a thread's pieces: row tid / 8 + 32 p of the tile, 8 elements at 8 (tid % 8)
  const int kp = (tid & 7) * 8;
  const bf16_t *ap[PA], *wp[PW];
#pragma unroll
  for (int p = 0; p < PA; ++p) {
    const int r = row0 + (tid >> 3) + 32 * p;
    ap[p] = r < end ? A + (long)(rows != nullptr ? rows[r] : r) * K + kp : nullptr;
  }
#pragma unroll
  for (int p = 0; p < PW; ++p) {
    const int r = (tid >> 3) + 32 * p;
    const int col = n0 + (GLU ? (r >> 5) * 16 + (r & 15) : r);
    wp[p] = col < N ? Wg + ((long)(GLU && (r & 16) ? N : 0) + col) * K + kp : nullptr;
  }
  uint4 ra[PA], rw[PW];
  auto fetch = [&](int k0) {
    const bool in = k0 + kp < K;
#pragma unroll
    for (int p = 0; p < PA; ++p) {
      ra[p] = uint4{0, 0, 0, 0};
      if (in && ap[p] != nullptr) ra[p] = *reinterpret_cast<const uint4*>(ap[p] + k0);
    }
#pragma unroll
    for (int p = 0; p < PW; ++p) {
      rw[p] = uint4{0, 0, 0, 0};
      if (in && wp[p] != nullptr) rw[p] = *reinterpret_cast<const uint4*>(wp[p] + k0);
    }
  };
  fr_f32x4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = fr_f32x4{0.f, 0.f, 0.f, 0.f};

  fetch(0);
  int buf = 0;
  for (int k0 = 0; k0 < K; k0 += kGK, buf ^= 1) {
    bf16_t *As = stage + buf * kStep, *Ws = As + BM * kGLd;
    const int off = (tid >> 3) * kGLd + kp;
#pragma unroll
    for (int p = 0; p < PA; ++p) *reinterpret_cast<uint4*>(As + off + 32 * p * kGLd) = ra[p];
#pragma unroll
    for (int p = 0; p < PW; ++p) *reinterpret_cast<uint4*>(Ws + off + 32 * p * kGLd) = rw[p];
    __syncthreads();          // (the other copy's readers have passed the barrier before this one's writes)
    if (k0 + kGK < K) fetch(k0 + kGK);
#pragma unroll
    for (int ks = 0; ks < kGK / 32; ++ks) {
      uint4 a[MT], b[NT];
#pragma unroll
      for (int j = 0; j < MT; ++j)
        a[j] = *reinterpret_cast<const uint4*>(As + (wm * (BM / 2) + j * 16 + l15) * kGLd + ks * 32 + g4 * 8);
#pragma unroll
      for (int i = 0; i < NT; ++i)
        b[i] = *reinterpret_cast<const uint4*>(Ws + (wn * (BN / 2) + i * 16 + l15) * kGLd + ks * 32 + g4 * 8);
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = fr_mfma(b[i], a[j], acc[i][j]);
    }
  }
  // lane (g4, l15) holds columns 4 g4 .. 4 g4 + 3 of row l15 of each 16 x 16 tile
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int row = row0 + wm * (BM / 2) + j * 16 + l15;
    if (row >= end) continue;
#pragma unroll
    for (int i = 0; i < NT; i += GLU ? 2 : 1) {
      const int col = n0 + (GLU ? wn * (BN / 4) + i * 8 : wn * (BN / 2) + i * 16) + 4 * g4;
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

// act: few_rows.h (0: none).  rows: A's row of every sorted row, or null.
extern "C" int mx_grouped_gemm(void* C, const void* A, const int* rows, const void* W, const int* offs, int groups, long M,
                               int N, int K, int act, float limit, hipStream_t s) {
  if (M <= 0 || N <= 0 || groups <= 0) return 0;
  if (K < 8 || K % 8 || M > 0x7fffffffL || act < kFrStore || act > kFrReluSq) return -1;
  if (((uintptr_t)A) % 16 || ((uintptr_t)W) % 16) return -2;
  const bool glu = act >= kFrGelu && act <= kFrClamp;
  const int vec = N % 4 == 0 && ((uintptr_t)C) % 8 == 0;
  // 128-row tiles once the groups fill them on average
  const bool tall = M >= 96L * groups;
  const int bm = tall ? 128 : 64, bn = 128;
  const long tiles = (M + bm - 1) / bm + groups;
  if (tiles > 65535) return -3;
  const int cols = glu ? bn / 2 : bn;
  const dim3 grid((unsigned)((N + cols - 1) / cols), (unsigned)tiles), block(256);
#define GG_GO(BM, GLU)                                                                                               \
  hipLaunchKernelGGL((grouped_gemm_kernel<BM, 128, GLU>), grid, block, 0, s, (bf16_t*)C, (const bf16_t*)A, rows,      \
                     (const bf16_t*)W, offs, groups, (int)M, N, K, act, limit, vec)
  if (tall) {
    if (glu) GG_GO(128, true); else GG_GO(128, false);
  } else {
    if (glu) GG_GO(64, true); else GG_GO(64, false);
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

// Row-wise kernels around an fp32 residual stream: embedding rows (optionally with a
// sinusoidal position vector), the fused "post-norm add + next pre-norm" step (also with a
// token shift of the normed row), the layer
// norm (weight and bias) that adds a sublayer's output to the residual, the tanh cap of
// the logits, per-head gated output norm (alone, or beside a second mixer's scaled rows), activations
// (relu^2, clamped / gelu / relu / silu GLU, gelu * token-side embedding) and the weighted row scatter-add
// that combines expert outputs.
#include <type_traits>

#include "mx_common.h"

namespace mx {

// out = table[id] * scale (+ a sinusoidal position vector when freqs is given: column 2i
// gets sin(p f_i), column 2i+1 cos(p f_i), with the angle p f_i formed in fp32)
template <typename T>
__global__ void embed_rows_kernel(float* __restrict__ out, const int* __restrict__ ids,
                                  const T* __restrict__ table, int width, int vocab, float scale,
                                  const int* __restrict__ positions, const float* __restrict__ freqs) {
  const int row = blockIdx.x;
  int id = ids[row];
  if (id < 0 || id >= vocab) id = 0;
  const float p = freqs != nullptr ? (float)positions[row] : 0.f;
  for (int i = threadIdx.x; i < width; i += blockDim.x) {
    float v = ld(table, (long)id * width + i) * scale;
    if (freqs != nullptr) {
      const float a = p * freqs[i >> 1];
      v += (i & 1) ? cosf(a) : sinf(a);
    }
    out[(long)row * width + i] = v;
  }
}

// a value of a row that is fp32 or bf16, decided at run time (uniform over the launch)
__device__ __forceinline__ float ldx(const void* p, int bf16, long i) {
  return bf16 ? ft::bf16_to_f32(((const bf16_t*)p)[i]) : ((const float*)p)[i];
}

// What a row adds from the table of token pairs: entry hash = (prev * mul_prev + cur * mul_cur) mod buckets, prev the token
// before the row's own in its sequence: the row above within a segment, last_tok[slot] for a segment's first row (pos0 > 0),
// and for a sequence's first token entry `buckets` instead.  That first row's workgroup, the only reader of the slot, then
// leaves the segment's last token there.  -1: none (padding rows).  Every thread of a workgroup calls it.
struct PairArgs {
  const void* table;                          // null: no pairs
  long mul_prev, mul_cur;
  int buckets, num_segs, num_slots;
  const int *start, *pos0, *slot;
  int* last_tok;
};
__device__ __forceinline__ long pair_entry(const PairArgs& P, const int* __restrict__ ids, int row) {
  if (row >= P.start[P.num_segs]) return -1;
  const int sg = segment_of(P.start, P.num_segs, row), first = P.start[sg], end = P.start[sg + 1], sl = P.slot[sg];
  if (sl < 0 || sl >= P.num_slots) return -1;
  long prev = row > first ? ids[row - 1] : P.pos0[sg] > 0 ? P.last_tok[sl] : -1;
  if (row == first) {
    __syncthreads();                          // (all have read it)
    if (threadIdx.x == 0) P.last_tok[sl] = ids[end - 1];
  }
  if (prev < 0) return P.buckets;
  long idx = (prev * P.mul_prev + (long)ids[row] * P.mul_cur) % P.buckets;
  return idx < 0 ? idx + P.buckets : idx;
}

// x (fp32 residual) = embed[cur] * scale + table[hash] per row (without `embed`: x += table[hash]).  One workgroup per row.
template <typename T>
__global__ void pair_embed_add_kernel(float* __restrict__ x, const int* __restrict__ ids, PairArgs P, int width,
                                      const T* __restrict__ embed, int vocab, float scale) {
  const int row = blockIdx.x;
  if (embed != nullptr) {                 // every row gets its embedding row, padding rows too
    int id = ids[row];
    if (id < 0 || id >= vocab) id = 0;
    for (int i = threadIdx.x; i < width; i += blockDim.x)
      x[(long)row * width + i] = ld(embed, (long)id * width + i) * scale;
  }
  const long idx = pair_entry(P, ids, row);
  if (idx < 0) return;
  for (int i = threadIdx.x; i < width; i += blockDim.x) x[(long)row * width + i] += ld((const T*)P.table, idx * width + i);
}

// residual (fp32, in place): x += mult * (y1 + y2);  out = rms_norm(x) * next_w (TO).
// y1 / y2 are fp32 or bf16 each and optional, as is out.
template <typename TO, int NT>
__global__ void add_scaled_rms_norm_kernel(float* __restrict__ x, const void* __restrict__ y1, int y1_bf16,
                                           long y1_stride, const void* __restrict__ y2, int y2_bf16,
                                           long y2_stride, float mult, const float* __restrict__ next_w,
                                           TO* __restrict__ out, int width, float eps) {
  __shared__ float red[NT / 64];
  const long row = blockIdx.x;
  float* xr = x + row * width;
  float ss = 0.f;
  for (int i = threadIdx.x; i < width; i += NT) {
    float v = xr[i];
    if (y1 != nullptr) {
      float y = ldx(y1, y1_bf16, row * y1_stride + i);
      if (y2 != nullptr) y += ldx(y2, y2_bf16, row * y2_stride + i);
      v += mult * y;
      xr[i] = v;
    }
    ss += v * v;
  }
  if (out == nullptr) return;
  ss = block_sum<NT>(ss, red);
  const float r = 1.0f / sqrtf(ss / (float)width + eps);
  // each thread re-reads only what it wrote itself
  for (int i = threadIdx.x; i < width; i += NT) st(out, row * width + i, xr[i] * r * next_w[i]);
}

// out (fp32) = scale * (a / rms(a) * wa + b / rms(b) * wb), one workgroup per row
template <typename T, int NT>
__global__ void dual_rms_mean_kernel(float* __restrict__ out, const T* __restrict__ a, long a_stride,
                                     const T* __restrict__ b, long b_stride, const float* __restrict__ wa,
                                     const float* __restrict__ wb, int width, float eps, float scale) {
  __shared__ float red[NT / 64];
  const long row = blockIdx.x;
  const T* ar = a + row * a_stride;
  const T* br = b + row * b_stride;
  float sa = 0.f, sb = 0.f;
  for (int i = threadIdx.x; i < width; i += NT) {
    const float u = ld(ar, i), v = ld(br, i);
    sa += u * u;
    sb += v * v;
  }
  sa = block_sum<NT>(sa, red);
  sb = block_sum<NT>(sb, red);
  const float ra = 1.0f / sqrtf(sa / (float)width + eps), rb = 1.0f / sqrtf(sb / (float)width + eps);
  for (int i = threadIdx.x; i < width; i += NT)
    out[row * width + i] = scale * (ld(ar, i) * ra * wa[i] + ld(br, i) * rb * wb[i]);
}

// out = o * sigmoid(g), o fp32 dense rows, g rows g_stride apart
template <typename TG, typename TO>
__global__ void sigmoid_gate_kernel(TO* __restrict__ out, const float* __restrict__ o, const TG* __restrict__ g,
                                    long g_stride, long rows, int n) {
  const long total = rows * n;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const long r = i / n;
    const int c = (int)(i % n);
    st(out, i, o[i] * sigmoidf_(ld(g, r * g_stride + c)));
  }
}

// layer norm with weight and bias, ln(u) = (u - mean) / sqrt(var + eps) * w + b with var
// the mean squared deviation (two passes), around an fp32 residual x:
//   y given:            x += ln(y);  cast = x
//   y null, out null:   x  = ln(x);  cast = x
//   y null, out given:  out = ln(x)  (x untouched)
template <typename TY, typename TO, int NT>
__global__ void layer_norm_kernel(float* __restrict__ x, const TY* __restrict__ y, long y_stride,
                                  const float* __restrict__ w, const float* __restrict__ b,
                                  TO* __restrict__ out, TO* __restrict__ cast, int width, float eps) {
  __shared__ float red[NT / 64];
  const long row = blockIdx.x;
  float* xr = x + row * width;
  const TY* yr = y != nullptr ? y + row * y_stride : nullptr;
  auto src = [&](int i) { return yr != nullptr ? ld(yr, i) : xr[i]; };
  float sum = 0.f;
  for (int i = threadIdx.x; i < width; i += NT) sum += src(i);
  const float mean = block_sum<NT>(sum, red) / (float)width;
  float ss = 0.f;
  for (int i = threadIdx.x; i < width; i += NT) {
    const float d = src(i) - mean;
    ss += d * d;
  }
  const float r = 1.0f / sqrtf(block_sum<NT>(ss, red) / (float)width + eps);
  for (int i = threadIdx.x; i < width; i += NT) {
    const float v = (src(i) - mean) * r * w[i] + b[i];
    if (out != nullptr) {
      st(out, row * width + i, v);
    } else {
      const float nx = yr != nullptr ? xr[i] + v : v;
      xr[i] = nx;
      if (cast != nullptr) st(cast, row * width + i, nx);
    }
  }
}

// x <- cap * tanh(x / cap); infinite entries stay
__global__ void tanh_cap_kernel(float* __restrict__ x, long n, float cap) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const float v = x[i];
    if (isfinite(v)) x[i] = cap * tanhf(v / cap);
  }
}

// A row of a workgroup in registers: 4 C entries per thread, four neighbours at a time, width <= 4 C NT.  A kernel asks for
// all rows that it will need and only then looks at the first: `ask` loads, `get` waits and widens.  VEC (16-byte fp32 or
// 8-byte bf16 pieces, width of whole fours): no load stands behind a branch, since the compiler has every load wait that
// may write the registers of another side of a branch; columns past the width read the row's last four and count as zeros.
// (With a branch, one load behind the other: a decode step's add and norm 4.7 us, 4.4 now, with a token shift 6.4 and 4.8.)
// Rows of more than 8192 have no registers for that: they load where they are got.
template <int C>
constexpr bool kAskAhead = C <= 4;
template <typename T, bool VEC, int NT, int C>
struct AskedRow {
  using Raw = typename std::conditional<!VEC, float4, typename std::conditional<sizeof(T) == 2, uint2, float4>::type>::type;
  Raw r[C];
  const T* from;
  __device__ __forceinline__ void ask(const T* p, int width) {
    if constexpr (kAskAhead<C>) load(p, width);
    else from = p;
  }
  __device__ __forceinline__ void load(const T* p, int width) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int i = (c * NT + threadIdx.x) * 4;
      if constexpr (VEC) {
        r[c] = *reinterpret_cast<const Raw*>(p + min(i, width - 4));
      } else {
        float v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = i + k < width ? ld(p, i + k) : 0.f;
        r[c] = make_float4(v[0], v[1], v[2], v[3]);
      }
    }
  }
  __device__ __forceinline__ void get(float (&v)[C][4], int width) {
    if constexpr (!kAskAhead<C>) load(from, width);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if constexpr (VEC && sizeof(T) == 2) {
        ft::unpack2(r[c].x, v[c][0], v[c][1]);
        ft::unpack2(r[c].y, v[c][2], v[c][3]);
      } else {
        v[c][0] = r[c].x, v[c][1] = r[c].y, v[c][2] = r[c].z, v[c][3] = r[c].w;
      }
      if constexpr (VEC)
        if ((c * NT + (int)threadIdx.x) * 4 >= width)
#pragma unroll
          for (int k = 0; k < 4; ++k) v[c][k] = 0.f;
    }
  }
};

template <typename T, bool VEC, int NT, int C>
__device__ __forceinline__ void store_row(T* p, const float (&v)[C][4], int width) {
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int i = (c * NT + threadIdx.x) * 4;
    if constexpr (VEC) {
      if (i >= width) continue;
      if constexpr (sizeof(T) == 2) {
        *reinterpret_cast<uint2*>(p + i) = make_uint2(ft::pack2(v[c][0], v[c][1]), ft::pack2(v[c][2], v[c][3]));
      } else {
        *reinterpret_cast<float4*>(p + i) = make_float4(v[c][0], v[c][1], v[c][2], v[c][3]);
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (i + k < width) st(p, i + k, v[c][k]);
    }
  }
}

// What a norm kernel adds to the residual: a row of a tensor, or of the experts' results not yet summed
// (few_rows.hip: experts_down), sum_k w[row, k] d[row, k] + shared[row] * (sigmoid(gate[row]) or 1), which saves
// a launch and its rows' way through memory (4.6 us a layer of a decode step); or, without weights, of a product's parts
// (few_rows.hip: few_rows_parts).  Asked<>: as AskedRow; `other` is read in the place of what there is not.
template <typename T>
struct RowsOf {
  static constexpr bool kOneRow = false;
  const T* p;
  long stride;
  __device__ __forceinline__ bool any() const { return p != nullptr; }
  template <bool VEC, int NT, int C>
  struct Asked {
    AskedRow<T, VEC, NT, C> r;
    __device__ __forceinline__ void ask(const RowsOf& y, long row, int width, const float* other) {
      r.ask(y.p != nullptr ? y.p + row * y.stride : (const T*)other, width);
    }
    __device__ __forceinline__ void pin(const RowsOf&, int, float*) {}
    __device__ __forceinline__ void get(const RowsOf&, float (&v)[C][4], long, int width) { r.get(v, width); }
  };
};
struct ExpertRows {
  static constexpr bool kOneRow = true;       // (a token shift's: decode rows, segments of one row)
  const float *d, *wts, *shared, *gate;       // [rows * top, width], [rows, top] or null, [rows, width] or null, [rows] or null
  int top;
  __device__ __forceinline__ bool any() const { return true; }
  // (its rows are whole fours at 16 bytes whatever the others are)
  template <bool VEC, int NT, int C>
  struct Asked {
    static constexpr int A = C <= 2 ? 4 : 1;  // of the `top` rows so many at once
    float4 d[A][C], shared[C];
    float w[A], gate;
    __device__ __forceinline__ void ask(const ExpertRows& y, long row, int width, const float*) {
      if constexpr (kAskAhead<C>) load(y, row, width);
    }
    // behind all that is asked for: the compiler moves scalar loads to their use, one wait behind the other
    __device__ __forceinline__ void pin(const ExpertRows&, int, float*) {
      if constexpr (kAskAhead<C>) {
#pragma unroll
        for (int k = 0; k < A; ++k) asm volatile("" : "+s"(w[k]));
        asm volatile("" : "+s"(gate));
      }
    }
    __device__ __forceinline__ void load(const ExpertRows& y, long row, int width) {
      const float* wp = y.wts != nullptr ? y.wts + row * y.top : y.d;
      gate = *(y.gate != nullptr ? y.gate + row : y.d);
#pragma unroll
      for (int k = 0; k < A; ++k) w[k] = wp[min(k, y.top - 1)];
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int i = min((c * NT + (int)threadIdx.x) * 4, width - 4);
#pragma unroll
        for (int k = 0; k < A; ++k)
          d[k][c] = *reinterpret_cast<const float4*>(y.d + (row * y.top + min(k, y.top - 1)) * width + i);
        shared[c] = *reinterpret_cast<const float4*>((y.shared != nullptr ? y.shared + row * width : y.d) + i);
      }
    }
    __device__ __forceinline__ void get(const ExpertRows& y, float (&v)[C][4], long row, int width) {
      if constexpr (!kAskAhead<C>) load(y, row, width);
      const float g = y.gate != nullptr ? sigmoidf_(gate) : 1.f;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int i = (c * NT + (int)threadIdx.x) * 4;
        const bool in = i < width;
        v[c][0] = v[c][1] = v[c][2] = v[c][3] = 0.f;
        auto add = [&](const float4& u, float f) {
          v[c][0] += f * u.x, v[c][1] += f * u.y, v[c][2] += f * u.z, v[c][3] += f * u.w;
        };
#pragma unroll
        for (int k = 0; k < A; ++k)
          if (in && k < y.top) add(d[k][c], y.wts != nullptr ? w[k] : 1.f);
        if (in)
#pragma unroll 4
          for (int k = A; k < y.top; ++k)
            add(*reinterpret_cast<const float4*>(y.d + (row * y.top + k) * width + i), y.wts != nullptr ? y.wts[row * y.top + k] : 1.f);
        if (in && y.shared != nullptr) add(shared[c], g);
      }
    }
  };
};
// The same of many rows, from the grouped products (grouped_gemm.hip): sum_k w[row, k] d[place[row, k]] + shared[row] * (sigmoid(h[row] .
// gate_w) or 1) of bf16 rows, which saves the launch that writes the sums as fp32 rows and the norm's read of those: 2000 rows of
// 2048, 4 experts, layer norm 19.2 us (12.2 + 12.9 in two launches), 4096 rows with a gated shared expert, RMS norms 31.7 (23.2 +
// 18.5), 300 rows 5.8 (5.0 + 4.6).
struct SortedRows {
  static constexpr bool kOneRow = false;
  const bf16_t *d, *shared, *h, *gate_w;      // [pairs, width], [rows, width] or null, [rows, width], [width] or null
  const int* place;                           // [rows, top]
  const float* wts;                           // [rows, top]
  long h_stride;
  int top;
  __device__ __forceinline__ bool any() const { return true; }
  // (its rows are whole fours at 8 bytes whatever the others are)
  template <bool VEC, int NT, int C>
  struct Asked {
    static constexpr int A = C <= 2 ? 4 : 1;  // of the `top` rows so many at once
    uint2 d[A][C], shared[C], h[C], gw[C];
    float w[A], gate;
    __device__ __forceinline__ void ask(const SortedRows& y, long row, int width, const float*) {
      if constexpr (kAskAhead<C>) load(y, row, width);
    }
    __device__ __forceinline__ void load(const SortedRows& y, long row, int width) {
      const bf16_t* p[A];
#pragma unroll
      for (int k = 0; k < A; ++k) {
        const long at = row * y.top + min(k, y.top - 1);
        p[k] = y.d + (long)y.place[at] * width;
        w[k] = y.wts[at];
      }
      const bf16_t* sp = y.shared != nullptr ? y.shared + row * width : p[0];
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int i = min((c * NT + (int)threadIdx.x) * 4, width - 4);
        h[c] = *reinterpret_cast<const uint2*>(y.h + row * y.h_stride + i);
        gw[c] = *reinterpret_cast<const uint2*>((y.gate_w != nullptr ? y.gate_w : p[0]) + i);
#pragma unroll
        for (int k = 0; k < A; ++k) d[k][c] = *reinterpret_cast<const uint2*>(p[k] + i);
        shared[c] = *reinterpret_cast<const uint2*>(sp + i);
      }
    }
    // behind all that is asked for: the shared expert's gate, a sum over the block
    __device__ __forceinline__ void pin(const SortedRows& y, int width, float* red) {
      gate = 1.f;
      if (y.gate_w == nullptr) return;
      float dot = 0.f;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int i = (c * NT + (int)threadIdx.x) * 4;
        uint2 hv = h[c], gv = gw[c];
        if constexpr (!kAskAhead<C>) {
          hv = *reinterpret_cast<const uint2*>(y.h + (long)blockIdx.x * y.h_stride + min(i, width - 4));
          gv = *reinterpret_cast<const uint2*>(y.gate_w + min(i, width - 4));
        }
        float a[4], b[4];
        ft::unpack2(hv.x, a[0], a[1]);
        ft::unpack2(hv.y, a[2], a[3]);
        ft::unpack2(gv.x, b[0], b[1]);
        ft::unpack2(gv.y, b[2], b[3]);
        if (i < width) dot += (a[0] * b[0] + a[1] * b[1]) + (a[2] * b[2] + a[3] * b[3]);
      }
      gate = sigmoidf_(block_sum<NT>(dot, red));
    }
    __device__ __forceinline__ void get(const SortedRows& y, float (&v)[C][4], long row, int width) {
      if constexpr (!kAskAhead<C>) load(y, row, width);
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int i = (c * NT + (int)threadIdx.x) * 4;
        const bool in = i < width;
        v[c][0] = v[c][1] = v[c][2] = v[c][3] = 0.f;
        auto add = [&](const uint2& u, float f) {
          float x[4];
          ft::unpack2(u.x, x[0], x[1]);
          ft::unpack2(u.y, x[2], x[3]);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[c][e] += f * x[e];
        };
#pragma unroll
        for (int k = 0; k < A; ++k)
          if (in && k < y.top) add(d[k][c], w[k]);
        if (in)
#pragma unroll 4
          for (int k = A; k < y.top; ++k)
            add(*reinterpret_cast<const uint2*>(y.d + (long)y.place[row * y.top + k] * width + i), y.wts[row * y.top + k]);
        if (in && y.shared != nullptr) add(shared[c], gate);
      }
    }
  };
};
constexpr int kAskedParts = 4;                // of a product's parts so many at once (no product here has more)
struct AnyRows {                              // either, by the launch: bf16 or fp32 rows, or a product's parts, A at once
  const void* p;
  int bf16, parts;
  long stride;
  __device__ __forceinline__ bool any() const { return p != nullptr; }
  template <bool VEC, int NT, int C, int A>
  struct Asked {
    uint2 lo[A][C], hi[A][C];
    const float* from;
    __device__ __forceinline__ void ask(const AnyRows& y, long row, int width, const float* other) {
      if constexpr (kAskAhead<C>) load(y, row, width, other);
      else from = other;
    }
    __device__ __forceinline__ void load(const AnyRows& y, long row, int width, const float* other) {
      const bool two = y.bf16 && y.p != nullptr, parts = y.parts > 1;
      const long es = two ? 2 : 4, rest = two ? 0 : 8;       // (half an fp32 piece; a bf16 piece is read twice)
#pragma unroll
      for (int k = 0; k < A; ++k) {
        const char* q = y.p == nullptr ? (const char*)other
                                       : (const char*)y.p + (parts ? (row * y.parts + min(k, y.parts - 1)) * width : row * y.stride) * es;
#pragma unroll
        for (int c = 0; c < C; ++c) {
          const int i = (c * NT + (int)threadIdx.x) * 4;
          if (VEC || parts) {
            const char* at = q + min(i, width - 4) * es;
            lo[k][c] = *reinterpret_cast<const uint2*>(at);
            hi[k][c] = *reinterpret_cast<const uint2*>(at + rest);
          } else {
            uint32_t u[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              u[e] = 0;
              if (i + e < width) u[e] = two ? (uint32_t)((const uint16_t*)q)[i + e] << 16 : ((const uint32_t*)q)[i + e];
            }
            lo[k][c] = make_uint2(u[0], u[1]);
            hi[k][c] = make_uint2(u[2], u[3]);
          }
        }
      }
    }
    __device__ __forceinline__ void get(const AnyRows& y, float (&v)[C][4], long row, int width) {
      if constexpr (!kAskAhead<C>) load(y, row, width, from);
      const bool parts = y.parts > 1, packed = VEC && y.bf16 && !parts;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        auto four = [&](int k, float (&u)[4]) {
          float b[4];
          ft::unpack2(lo[k][c].x, b[0], b[1]);
          ft::unpack2(lo[k][c].y, b[2], b[3]);
          u[0] = packed ? b[0] : __uint_as_float(lo[k][c].x);
          u[1] = packed ? b[1] : __uint_as_float(lo[k][c].y);
          u[2] = packed ? b[2] : __uint_as_float(hi[k][c].x);
          u[3] = packed ? b[3] : __uint_as_float(hi[k][c].y);
        };
        four(0, v[c]);
#pragma unroll
        for (int k = 1; k < A; ++k)
          if (parts && k < y.parts) {
            float u[4];
            four(k, u);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[c][e] += u[e];
          }
        if (parts)
          for (int k = A; k < y.parts; ++k) {
            const float4 u = *reinterpret_cast<const float4*>((const float*)y.p + (row * y.parts + k) * width +
                                                              min((c * NT + (int)threadIdx.x) * 4, width - 4));
            v[c][0] += u.x, v[c][1] += u.y, v[c][2] += u.z, v[c][3] += u.w;
          }
        if ((VEC || parts) && (c * NT + (int)threadIdx.x) * 4 >= width) v[c][0] = v[c][1] = v[c][2] = v[c][3] = 0.f;
      }
    }
  };
};

// sums of two values over a block; every thread gets both
template <int NT>
__device__ __forceinline__ void block_sum2(float& a, float& b, float (*red)[2]) {
  a = ft::wave_sum(a);
  b = ft::wave_sum(b);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6][0] = a;
    red[threadIdx.x >> 6][1] = b;
  }
  __syncthreads();
  a = b = 0.f;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) {
    a += red[w][0];
    b += red[w][1];
  }
}

template <int C>
__device__ __forceinline__ float sum_sq(const float (&v)[C][4]) {
  float s = 0.f;
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int k = 0; k < 4; ++k) s += v[c][k] * v[c][k];
  return s;
}

// layer_norm_kernel, add_scaled_rms_norm_kernel and dual_rms_mean_kernel for rows that row_in_registers() takes: the row in
// registers, all its loads in flight at once and no value read twice.  Bound by that one latency and the
// reductions for few rows, by the rows' bytes for many.  Width 2048: layer norm of 32 rows 4.7 us, of 2000 12
// (values read entry by entry, again for each pass: 10 and 16); scaled add and norm of 777 rows 6 (10); mean of two norms
// 5 (9).
template <typename Y, typename TO, bool VEC, int NT, int C>
__global__ void __launch_bounds__(NT)
layer_norm_row_kernel(float* __restrict__ x, Y y, const float* __restrict__ w,
                      const float* __restrict__ b, TO* __restrict__ out, TO* __restrict__ cast,
                      const float* __restrict__ next_w, const float* __restrict__ next_b, int width, float eps) {
  __shared__ float red[NT / 64];
  const long row = blockIdx.x;
  float v[C][4], u[C][4], wv[C][4], bv[C][4];
  AskedRow<float, VEC, NT, C> xa, wa, ba, nwa, nba;
  typename Y::template Asked<VEC, NT, C> ya;
  const bool next = next_w != nullptr;
  xa.ask(x + row * width, width);
  ya.ask(y, row, width, x + row * width);
  wa.ask(w, width);
  ba.ask(b, width);
  nwa.ask(next ? next_w : w, width);
  nba.ask(next ? next_b : b, width);
  ya.pin(y, width, red);
  auto norm = [&] {                          // u <- its layer norm, times wv plus bv
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c) sum += (u[c][0] + u[c][1]) + (u[c][2] + u[c][3]);
    const float mean = block_sum<NT>(sum, red) / (float)width;
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const bool in = (c * NT + (int)threadIdx.x) * 4 + k < width;
        u[c][k] = in ? u[c][k] - mean : 0.f;
        ss += u[c][k] * u[c][k];
      }
    const float r = 1.0f / sqrtf(block_sum<NT>(ss, red) / (float)width + eps);
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) u[c][k] = u[c][k] * r * wv[c][k] + bv[c][k];
  };
  xa.get(v, width);
  if (y.any()) {
    ya.get(y, u, row, width);
  } else {
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) u[c][k] = v[c][k];
  }
  wa.get(wv, width);
  ba.get(bv, width);
  norm();
  if (out == nullptr && y.any())
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) u[c][k] += v[c][k];
  if (out != nullptr) {
    store_row<TO, VEC, NT, C>(out + row * width, u, width);
  } else {
    store_row<float, VEC, NT, C>(x + row * width, u, width);
    if (next) {
      nwa.get(wv, width);
      nba.get(bv, width);
      norm();
    }
    if (cast != nullptr) store_row<TO, VEC, NT, C>(cast + row * width, u, width);
  }
}

// A: parts of y1 and y2 (1: neither is in parts)
template <typename TO, bool VEC, int A, int NT, int C>
__global__ void __launch_bounds__(NT)
add_scaled_rms_norm_row_kernel(float* __restrict__ x, AnyRows y1, AnyRows y2, float mult,
                               const float* __restrict__ next_w, TO* __restrict__ out, int width, float eps) {
  __shared__ float red[NT / 64];
  const long row = blockIdx.x;
  float v[C][4], a[C][4], b[C][4], w[C][4];
  AskedRow<float, VEC, NT, C> xa, wa;
  AnyRows::Asked<VEC, NT, C, kAskAhead<C> ? A : 1> ya, yb;
  xa.ask(x + row * width, width);
  ya.ask(y1, row, width, x + row * width);
  yb.ask(y2, row, width, x + row * width);
  wa.ask(out != nullptr ? next_w : x + row * width, width);
  xa.get(v, width);
  ya.get(y1, a, row, width);
  yb.get(y2, b, row, width);
  wa.get(w, width);
  if (y1.any()) {
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) v[c][k] += mult * (y2.any() ? a[c][k] + b[c][k] : a[c][k]);
    store_row<float, VEC, NT, C>(x + row * width, v, width);
  }
  if (out == nullptr) return;
  const float r = 1.0f / sqrtf(block_sum<NT>(sum_sq<C>(v), red) / (float)width + eps);
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int k = 0; k < 4; ++k) v[c][k] *= r * w[c][k];
  store_row<TO, VEC, NT, C>(out + row * width, v, width);
}

template <bool VEC, int A, int NT, int C>
__global__ void __launch_bounds__(NT)
dual_rms_mean_row_kernel(float* __restrict__ out, AnyRows a, AnyRows b, const float* __restrict__ wa,
                         const float* __restrict__ wb, int width, float eps, float scale) {
  __shared__ float red[NT / 64][2];
  const long row = blockIdx.x;
  float u[C][4], v[C][4], p[C][4], q[C][4];
  AskedRow<float, VEC, NT, C> pa, qa;
  AnyRows::Asked<VEC, NT, C, kAskAhead<C> ? A : 1> ya, yb;
  ya.ask(a, row, width, wa);
  yb.ask(b, row, width, wa);
  pa.ask(wa, width);
  qa.ask(wb, width);
  ya.get(a, u, row, width);
  yb.get(b, v, row, width);
  pa.get(p, width);
  qa.get(q, width);
  float sa = sum_sq<C>(u), sb = sum_sq<C>(v);
  block_sum2<NT>(sa, sb, red);
  const float ra = 1.0f / sqrtf(sa / (float)width + eps), rb = 1.0f / sqrtf(sb / (float)width + eps);
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int k = 0; k < 4; ++k) u[c][k] = scale * (u[c][k] * ra * p[c][k] + v[c][k] * rb * q[c][k]);
  store_row<float, VEC, NT, C>(out + row * width, u, width);
}

// A step's first rows and the norm that reads them, in one launch: x = embed[id] * scale (+ the position's sines and
// cosines) (+ the row of the pair), then out = rms_norm(x) * w (NORM 1), or x = layer_norm(x) * w + b, out = x (NORM 2),
// or nothing (0).  A row in registers, as the kernels below: all of an embedding row's reads in flight at once, and a sine and
// a cosine share their angle's reduction.  Bound by the chain of id, row and sums for few rows, by the rows' bytes for many.
// In running models, us beside embedding, pairs' last tokens and norm in launches of their own: 1 row 4.4 (8.6), 16 with pairs
// 7.0 (19), 32 with positions 5.6 (16), 2048 10.8 (17.7).
struct EmbedArgs {
  const int* ids;
  const void* table;
  int vocab;
  float scale;
  const int* positions;                       // with freqs
  const float* freqs;
};
template <typename T, typename TO, int NT, int C, int NORM>
__global__ void __launch_bounds__(NT)
embed_norm_kernel(EmbedArgs E, PairArgs P, float* __restrict__ x, TO* __restrict__ out, const float* __restrict__ w,
                  const float* __restrict__ b, int width, float eps) {
  __shared__ float red[NT / 64];
  const int row = blockIdx.x;
  int id = E.ids[row];
  if (id < 0 || id >= E.vocab) id = 0;
  float v[C][4], t[C][4], wv[C][4], bv[C][4];
  AskedRow<T, true, NT, C> va, ta;
  AskedRow<float, true, NT, C> wa, ba;
  if constexpr (NORM > 0) wa.ask(w, width);
  if constexpr (NORM == 2) ba.ask(b, width);
  va.ask((const T*)E.table + (long)id * width, width);
  long pair = -1;
  if (P.table != nullptr) {
    pair = pair_entry(P, E.ids, row);
    ta.ask((const T*)P.table + max(pair, 0L) * width, width);
    ta.get(t, width);
  }
  va.get(v, width);
  if constexpr (NORM > 0) wa.get(wv, width);
  if constexpr (NORM == 2) ba.get(bv, width);
  const float p = E.freqs != nullptr ? (float)E.positions[row] : 0.f;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int i = (c * NT + threadIdx.x) * 4;
#pragma unroll
    for (int k = 0; k < 4; ++k) v[c][k] *= E.scale;
    if (E.freqs != nullptr && i < width) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        float sn, cs;
        sincosf(p * E.freqs[i / 2 + k], &sn, &cs);
        v[c][2 * k] += sn;
        v[c][2 * k + 1] += cs;
      }
    }
    if (pair >= 0)
#pragma unroll
      for (int k = 0; k < 4; ++k) v[c][k] += t[c][k];
  }
  if constexpr (NORM < 2) store_row<float, true, NT, C>(x + (long)row * width, v, width);
  if constexpr (NORM == 1) {
    const float r = 1.0f / sqrtf(block_sum<NT>(sum_sq<C>(v), red) / (float)width + eps);
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) v[c][k] *= r * wv[c][k];
  } else if constexpr (NORM == 2) {
    float sum = 0.f, ss = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c) sum += (v[c][0] + v[c][1]) + (v[c][2] + v[c][3]);
    const float mean = block_sum<NT>(sum, red) / (float)width;
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        v[c][k] = (c * NT + (int)threadIdx.x) * 4 + k < width ? v[c][k] - mean : 0.f;
        ss += v[c][k] * v[c][k];
      }
    const float r = 1.0f / sqrtf(block_sum<NT>(ss, red) / (float)width + eps);
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) v[c][k] = v[c][k] * r * wv[c][k] + bv[c][k];
    store_row<float, true, NT, C>(x + (long)row * width, v, width);
  }
  if constexpr (NORM > 0)
    if (out != nullptr) store_row<TO, true, NT, C>(out + (long)row * width, v, width);
}

// residual (fp32, in place): x += rms_norm(y) * wb (y as it is without wb) (+ add_vec);
// out = rms_norm(x) * next_w (TO);  cast = x (TO).  Every part is optional.
// Bound by one latency of memory and the reductions for few rows, by the rows' bytes for many.
template <typename Y, typename TO, bool VEC, int NT, int C>
__global__ void __launch_bounds__(NT)
add_rms_norm_kernel(float* __restrict__ x, Y y, const float* __restrict__ wb,
                    const float* __restrict__ add_vec, const float* __restrict__ next_w, TO* __restrict__ out,
                    TO* __restrict__ cast, int width, float eps) {
  __shared__ float red[NT / 64];
  const long row = blockIdx.x;
  float v[C][4], t[C][4], w[C][4];
  AskedRow<float, VEC, NT, C> xa, wa, aa, na;
  typename Y::template Asked<VEC, NT, C> ya;
  const float* xr = x + row * width;
  xa.ask(xr, width);
  ya.ask(y, row, width, xr);
  wa.ask(wb != nullptr ? wb : xr, width);
  aa.ask(add_vec != nullptr ? add_vec : xr, width);
  na.ask(out != nullptr ? next_w : xr, width);
  ya.pin(y, width, red);
  xa.get(v, width);
  if (y.any()) {
    ya.get(y, t, row, width);
    if (wb != nullptr) {
      wa.get(w, width);
      const float r = 1.0f / sqrtf(block_sum<NT>(sum_sq<C>(t), red) / (float)width + eps);
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int k = 0; k < 4; ++k) t[c][k] *= r * w[c][k];
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) v[c][k] += t[c][k];
  }
  if (add_vec != nullptr) {
    aa.get(w, width);
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) v[c][k] += w[c][k];
  }
  if (y.any() || add_vec != nullptr) store_row<float, VEC, NT, C>(x + row * width, v, width);
  if (cast != nullptr) store_row<TO, VEC, NT, C>(cast + row * width, v, width);
  if (out != nullptr) {
    na.get(w, width);
    const float r = 1.0f / sqrtf(block_sum<NT>(sum_sq<C>(v), red) / (float)width + eps);
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) v[c][k] *= r * w[c][k];
    store_row<TO, VEC, NT, C>(out + row * width, v, width);
  }
}

// ---------------------------------------------------------------------------------
// the step between layers with a token shift, one workgroup per row:
//   x_out = x_in + rms_norm(y) * wb (without y: x_out = x_in, not written)
//   h = rms_norm(x_out) * w;  out = h + (h' - h) * shift
// with h' the h of the token before: of the row above within a segment (recomputed here from
// that row's x_in and y, so x_out must be another buffer than x_in when a segment has several
// rows), of the state slot for a segment's first row, zeros for a sequence's first token.  A
// one-row segment also leaves its h in the slot; shift_state_kernel does that for longer ones
// afterwards (a slot may still be read by the segment's first row here).
// ---------------------------------------------------------------------------------
template <typename Y, typename TO, bool VEC, int NT, int C>
__global__ void __launch_bounds__(NT)
add_norm_shift_kernel(float* x_out, const float* x_in, Y y, const float* __restrict__ wb, const float* __restrict__ w,
                      const float* __restrict__ shift,
                      TO* __restrict__ out, float* state, int num_slots, const int* __restrict__ start,
                      const int* __restrict__ pos0, const int* __restrict__ slot, int num_segs, int width,
                      float eps) {
  __shared__ float red[NT / 64][2];
  const long row = blockIdx.x;
  AskedRow<float, VEC, NT, C> xr, pr, wbr, wr, sr;
  typename Y::template Asked<VEC, NT, C> yr, ypr;
  xr.ask(x_in + row * width, width);
  yr.ask(y, row, width, x_in + row * width);
  wbr.ask(wb != nullptr ? wb : w, width);
  wr.ask(w, width);
  sr.ask(shift, width);
  int sl = -1, rel = 0, n = 1;
  bool old = false;
  if (row < start[num_segs]) {
    const int sg = segment_of(start, num_segs, (int)row);
    if constexpr (!Y::kOneRow) rel = (int)row - start[sg];
    n = start[sg + 1] - start[sg];
    sl = slot[sg];
    if (sl >= num_slots) sl = -1;
    old = sl >= 0 && pos0[sg] > 0;
  }
  // the row above, or what the state slot holds of it
  pr.ask(rel > 0 ? x_in + (row - 1) * width : old ? state + (long)sl * width : x_in + row * width, width);
  float xa[C][4], xp[C][4], t[C][4];
  if (rel > 0 && y.any()) ypr.ask(y, row - 1, width, x_in);
  yr.pin(y, width, nullptr);
  xr.get(xa, width);
  pr.get(xp, width);
  if (y.any()) {
    float yp[C][4], wv[C][4];
    yr.get(y, t, row, width);
    if (rel > 0) ypr.get(y, yp, row - 1, width);
    float sa = sum_sq<C>(t), sb = rel > 0 ? sum_sq<C>(yp) : 0.f;
    block_sum2<NT>(sa, sb, red);
    const float ra = 1.0f / sqrtf(sa / (float)width + eps), rb = 1.0f / sqrtf(sb / (float)width + eps);
    wbr.get(wv, width);
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        xa[c][k] += t[c][k] * ra * wv[c][k];
        if (rel > 0) xp[c][k] += yp[c][k] * rb * wv[c][k];
      }
    store_row<float, VEC, NT, C>(x_out + row * width, xa, width);
  }
  float sa = sum_sq<C>(xa), sb = rel > 0 ? sum_sq<C>(xp) : 0.f;
  block_sum2<NT>(sa, sb, red);
  const float ra = 1.0f / sqrtf(sa / (float)width + eps), rb = 1.0f / sqrtf(sb / (float)width + eps);
  wr.get(t, width);
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      xa[c][k] *= ra * t[c][k];
      xp[c][k] = rel > 0 ? xp[c][k] * (rb * t[c][k]) : old ? xp[c][k] : 0.f;
    }
  if (sl >= 0 && n == 1) store_row<float, VEC, NT, C>(state + (long)sl * width, xa, width);
  sr.get(t, width);
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int k = 0; k < 4; ++k) xa[c][k] += (xp[c][k] - xa[c][k]) * t[c][k];
  store_row<TO, VEC, NT, C>(out + row * width, xa, width);
}

// the h of each longer segment's last row, from its x, into the segment's slot; grid segments
template <bool VEC, int NT, int C>
__global__ void __launch_bounds__(NT)
shift_state_kernel(float* __restrict__ state, int num_slots, const float* __restrict__ x, const float* __restrict__ w,
                   const int* __restrict__ start, const int* __restrict__ slot, int width, float eps) {
  __shared__ float red[NT / 64][2];
  const int s = blockIdx.x;
  const int n = start[s + 1] - start[s], sl = slot[s];
  if (n < 2 || sl < 0 || sl >= num_slots) return;
  float xa[C][4], t[C][4];
  AskedRow<float, VEC, NT, C> xr, wr;
  xr.ask(x + (long)(start[s + 1] - 1) * width, width);
  wr.ask(w, width);
  xr.get(xa, width);
  float sa = sum_sq<C>(xa), sb = 0.f;
  block_sum2<NT>(sa, sb, red);
  const float ra = 1.0f / sqrtf(sa / (float)width + eps);
  wr.get(t, width);
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int k = 0; k < 4; ++k) xa[c][k] *= ra * t[c][k];
  store_row<float, VEC, NT, C>(state + (long)sl * width, xa, width);
}

// one wave per (row, head): out = o / rms(o) * w * sigmoid(gate), or * silu(gate)
template <typename TG, typename TO>
__global__ void head_rms_gate_kernel(TO* __restrict__ out, const float* __restrict__ o,
                                     const float* __restrict__ w, const TG* __restrict__ gate,
                                     long gate_stride, long pairs, int heads, int dv, float eps, int silu) {
  const long pair = (long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (pair >= pairs) return;
  const int lane = threadIdx.x & 63;
  const long row = pair / heads;
  const int h = (int)(pair % heads);
  const float* op = o + (row * heads + h) * dv;
  float ss = 0.f;
  for (int i = lane; i < dv; i += 64) ss += op[i] * op[i];
  ss = ft::wave_sum(ss);
  const float r = 1.0f / sqrtf(ss / (float)dv + eps);
  for (int i = lane; i < dv; i += 64) {
    const float gp = ld(gate, row * gate_stride + (long)h * dv + i);
    const float g = silu ? gp * sigmoidf_(gp) : sigmoidf_(gp);
    st(out, (row * heads + h) * dv + i, op[i] * r * w[i] * g);
  }
}

// The same for heads of 16 to 256 in whole fours: a lane four neighbours, LPR lanes a head, the loads of U heads on their way
// at once.  Bound by the bytes: 4096 rows of 16 heads of 128 14 us (67 MB;
// a wave a head and two entries a lane 32).
template <typename TG, typename TO, int LPR, int U>
__global__ void __launch_bounds__(256)
head_rms_gate_fours_kernel(TO* __restrict__ out, const float* __restrict__ o, const float* __restrict__ w,
                           const TG* __restrict__ gate, long gate_stride, int pairs, int heads, float eps, int silu) {
  constexpr int PER = 64 / LPR, dv = 4 * LPR;
  const int lane = threadIdx.x & 63, sub = lane / LPR, i = lane % LPR * 4;
  const int first = (blockIdx.x * 4 + (threadIdx.x >> 6)) * PER * U + sub;
  float v[U][4], g[U][4], wv[4];
  auto four = [](const auto* p, float (&x)[4]) {
    if constexpr (sizeof(*p) == 2) {
      const uint2 u = *reinterpret_cast<const uint2*>(p);
      ft::unpack2(u.x, x[0], x[1]);
      ft::unpack2(u.y, x[2], x[3]);
    } else {
      const float4 u = *reinterpret_cast<const float4*>(p);
      x[0] = u.x, x[1] = u.y, x[2] = u.z, x[3] = u.w;
    }
  };
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int p = min(first + u * PER, pairs - 1), row = p / heads;
    four(o + (long)p * dv + i, v[u]);
    four(gate + row * gate_stride + (long)(p - row * heads) * dv + i, g[u]);
  }
  four(w + i, wv);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    float ss = (v[u][0] * v[u][0] + v[u][1] * v[u][1]) + (v[u][2] * v[u][2] + v[u][3] * v[u][3]);
#pragma unroll
    for (int off = 1; off < LPR; off <<= 1) ss += __shfl_xor(ss, off, 64);
    const float r = 1.0f / sqrtf(ss / (float)dv + eps);
    float y[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float s = sigmoidf_(g[u][k]);
      y[k] = v[u][k] * r * wv[k] * (silu ? g[u][k] * s : s);
    }
    const int p = first + u * PER;
    if (p >= pairs) continue;
    if constexpr (sizeof(TO) == 2)
      *reinterpret_cast<uint2*>(out + (long)p * dv + i) = make_uint2(ft::pack2(y[0], y[1]), ft::pack2(y[2], y[3]));
    else
      *reinterpret_cast<float4*>(out + (long)p * dv + i) = make_float4(y[0], y[1], y[2], y[3]);
  }
}

// rows [a_scale * a (n) | o_scale * o / rms(o) per head * silu(gate)]: one wave per (row, item),
// items are the heads of o, then pieces of 256 columns of a
template <typename T>
__global__ void scaled_pair_rows_kernel(T* __restrict__ out, const float* __restrict__ a, int n, float a_scale,
                                        const float* __restrict__ o, const T* __restrict__ gate, long gate_stride,
                                        float o_scale, long waves, int items, int heads, int dv, float eps) {
  const long w = (long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (w >= waves) return;
  const int lane = threadIdx.x & 63;
  const long row = w / items;
  const int it = (int)(w % items);
  T* orow = out + row * (n + (long)heads * dv);
  if (it >= heads) {
    const int c0 = (it - heads) * 256;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int c = c0 + lane + 64 * u;
      if (c < n) st(orow, c, a[row * n + c] * a_scale);
    }
    return;
  }
  const float* op = o + (row * heads + it) * dv;
  float ss = 0.f;
  for (int i = lane; i < dv; i += 64) ss += op[i] * op[i];
  const float r = 1.0f / sqrtf(ft::wave_sum(ss) / (float)dv + eps) * o_scale;
  for (int i = lane; i < dv; i += 64) {
    const float g = ld(gate, row * gate_stride + (long)it * dv + i);
    st(orow, n + (long)it * dv + i, op[i] * r * (g * sigmoidf_(g)));
  }
}

template <typename T>
__global__ void relu_sq_kernel(T* __restrict__ x, long n) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const float v = fmaxf(ld(x, i), 0.f);
    st(x, i, v * v);
  }
}

// out[r, c] = relu(u[r, c])^2 for the first ff columns of wider rows
template <typename T>
__global__ void relu_sq_rows_kernel(T* __restrict__ out, const T* __restrict__ u, long u_stride, long rows, int ff) {
  const long n = rows * ff;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const float v = fmaxf(ld(u, (i / ff) * u_stride + i % ff), 0.f);
    st(out, i, v * v);
  }
}

// out[row] += sum_k w[row, k] * y[idx[row, k]]: combines the outputs of the experts each
// row chose, y being in another row order (sorted by expert).  grid rows.
template <typename TY>
__global__ void gather_add_rows_kernel(float* __restrict__ out, const TY* __restrict__ y,
                                       const int* __restrict__ idx, const float* __restrict__ w, int top,
                                       int width, long y_rows) {
  const long row = blockIdx.x;
  for (int c = threadIdx.x; c < width; c += blockDim.x) {
    float acc = 0.f;
    for (int k = 0; k < top; ++k) {
      const long src = idx[row * top + k];
      if (src >= 0 && src < y_rows) acc += w[row * top + k] * ld(y, src * width + c);
    }
    out[row * width + c] += acc;
  }
}

// Gated linear units on rows [gate (ff) | up (ff) | ...], activation by a functor; VEC: eight
// neighbouring bf16 (four fp32) entries per thread, 16-byte accesses
template <typename T> struct GluVec;
template <> struct GluVec<float> { static constexpr int N = 4; };
template <> struct GluVec<bf16_t> { static constexpr int N = 8; };

__device__ __forceinline__ void load16(const float* p, float (&v)[4]) {
  const float4 u = *reinterpret_cast<const float4*>(p);
  v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w;
}
__device__ __forceinline__ void load16(const bf16_t* p, float (&v)[8]) { ft::load8(*reinterpret_cast<const uint4*>(p), v); }
__device__ __forceinline__ void store16(float* p, const float (&v)[4]) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void store16(bf16_t* p, const float (&v)[8]) {
  *reinterpret_cast<uint4*>(p) =
      make_uint4(ft::pack2(v[0], v[1]), ft::pack2(v[2], v[3]), ft::pack2(v[4], v[5]), ft::pack2(v[6], v[7]));
}

template <typename T, typename F>
__device__ __forceinline__ void glu_rows(T* __restrict__ out, const T* __restrict__ gu, long gu_stride, long rows, int ff,
                                         int vec, F act) {
  constexpr int N = GluVec<T>::N;
  const long step = (long)gridDim.x * blockDim.x, i0 = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (vec) {
    const int per = ff / N;
    for (long i = i0; i < rows * per; i += step) {
      const long r = i / per;
      const int c = (int)(i - r * per) * N;
      float g[N], u[N];
      load16(gu + r * gu_stride + c, g);
      load16(gu + r * gu_stride + ff + c, u);
#pragma unroll
      for (int k = 0; k < N; ++k) g[k] = act(g[k], u[k]);
      store16(out + r * ff + c, g);
    }
    return;
  }
  for (long i = i0; i < rows * ff; i += step) {
    const long r = i / ff;
    const int c = (int)(i % ff);
    st(out, i, act(ld(gu, r * gu_stride + c), ld(gu, r * gu_stride + ff + c)));
  }
}

// rows [gate (ff) | up (ff) | ...]: g = min(gate, limit), u = clamp(up, +-limit),
// out = g * sigmoid(1.702 g) * (u + 1)
template <typename T>
__global__ void clamp_swiglu_kernel(T* __restrict__ out, const T* __restrict__ gu, long gu_stride,
                                    long rows, int ff, float limit, int vec) {
  glu_rows(out, gu, gu_stride, rows, ff, vec, [=](float g, float u) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g * sigmoidf_(1.702f * g) * (u + 1.0f);
  });
}


// rows [gate (ff) | up (ff)]: out = act(gate) * up, act = gelu_tanh (0), relu (1) or silu (2)
template <typename T>
__global__ void act_glu_kernel(T* __restrict__ out, const T* __restrict__ gu, long gu_stride, long rows, int ff,
                               int act, int vec) {
  glu_rows(out, gu, gu_stride, rows, ff, vec, [=](float g, float u) {
    return (act == 2 ? g * sigmoidf_(g) : act == 1 ? fmaxf(g, 0.f) : gelu_tanh_(g)) * u;
  });
}

template <typename T>
__global__ void side_gate_kernel(T* __restrict__ out, const T* __restrict__ gpre,
                                 const T* __restrict__ table, long table_stride,
                                 const int* __restrict__ ids, int col0, long rows, int sd, int vocab) {
  const long n = rows * sd;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const long r = i / sd;
    const int c = (int)(i % sd);
    int id = ids[r];
    if (id < 0 || id >= vocab) id = 0;
    st(out, i, gelu_tanh_(ld(gpre, i)) * ld(table, (long)id * table_stride + col0 + c));
  }
}

// out[rows[i]] += w_i * y[i]; rows == nullptr: identity.  No row repeats within a call.
template <typename TY, typename TW>
__global__ void scale_add_rows_kernel(float* __restrict__ out, const TY* __restrict__ y,
                                      const int* __restrict__ rows, const TW* __restrict__ weights,
                                      int sigmoid, int width, int out_rows) {
  const long i = blockIdx.x;
  const long dst = rows != nullptr ? rows[i] : i;
  if (dst < 0 || dst >= out_rows) return;
  float w = ld(weights, i);
  if (sigmoid) w = sigmoidf_(w);
  for (int c = threadIdx.x; c < width; c += blockDim.x)
    out[dst * width + c] += w * ld(y, i * width + c);
}

}  // namespace mx

using namespace mx;

constexpr int kRowThreads = 512;
constexpr int kRowMaxWidth = kRowThreads * 4 * 8;

// calls f with the number of register chunks a row of this width takes, as a constant
template <typename F>
static void row_chunks(int width, F f) {
  const int chunks = (width + kRowThreads * 4 - 1) / (kRowThreads * 4);
  if (chunks <= 1) f(std::integral_constant<int, 1>{});
  else if (chunks <= 2) f(std::integral_constant<int, 2>{});
  else if (chunks <= 4) f(std::integral_constant<int, 4>{});
  else f(std::integral_constant<int, 8>{});
}
// the same and whether rows are read in pieces of four (vec: width of whole fours, all rows aligned)
template <typename F>
static void row_chunks(int width, int vec, F f) {
  row_chunks(width, [&](auto c) {
    if (vec) f(c, std::true_type{});
    else f(c, std::false_type{});
  });
}

// x = embed[id] * scale (+ positions) (+ pairs), then the norm: 0 none, 1 out = rms_norm(x) * w, 2 x = layer_norm(x) * w + b and
// out (if any) = x; rows that are no whole fours or too wide: only without a norm
extern "C" int mx_embed_norm_fits(int width) { return width % 4 == 0 && width <= kRowMaxWidth; }
extern "C" int mx_embed_norm(float* x, const int* ids, const void* table, int bf16, int rows, int width, int vocab, float scale,
                             const int* positions, const float* freqs, const void* pairs, long mul_prev, long mul_cur, int buckets,
                             const int* start, const int* pos0, const int* slot, int num_segs, int* last_tok, int num_slots,
                             int norm, void* out, int out_bf16, const float* w, const float* b, float eps, hipStream_t s) {
  if (rows <= 0) return 0;
  if ((freqs != nullptr && positions == nullptr) || norm < 0 || norm > 2 || (pairs != nullptr && buckets < 1)) return -1;
  if (num_segs < 1) pairs = nullptr;          // (padding rows only)
  const PairArgs P{pairs, mul_prev, mul_cur, buckets, num_segs, num_slots, start, pos0, slot, last_tok};
  const int vec = mx_embed_norm_fits(width) && ((uintptr_t)table | (uintptr_t)pairs) % (bf16 ? 8 : 16) == 0 &&
                  ((uintptr_t)x | (uintptr_t)w | (uintptr_t)b) % 16 == 0 && ((uintptr_t)out) % (out_bf16 ? 8 : 16) == 0;
  if (!vec) {
    if (norm != 0) return -2;
    if (pairs != nullptr && freqs != nullptr) return -3;
    if (pairs != nullptr) {
      MX_DISPATCH_T(bf16, hipLaunchKernelGGL((pair_embed_add_kernel<T>), dim3(rows), dim3(256), 0, s, x, ids, P, width,
                                             (const T*)table, vocab, scale));
    } else {
      MX_DISPATCH_T(bf16, hipLaunchKernelGGL((embed_rows_kernel<T>), dim3(rows), dim3(256), 0, s, x, ids, (const T*)table, width,
                                             vocab, scale, positions, freqs));
    }
    return (int)hipGetLastError();
  }
  const EmbedArgs E{ids, table, vocab, scale, positions, freqs};
#define MX_EN(TO, NORM)                                                                                                    \
  MX_DISPATCH_T(bf16, hipLaunchKernelGGL((embed_norm_kernel<T, TO, kRowThreads, decltype(c)::value, NORM>), dim3(rows),    \
                                         dim3(kRowThreads), 0, s, E, P, x, (TO*)out, w, b, width, eps))
  row_chunks(width, [&](auto c) {
    if (norm == 0) MX_EN(float, 0);
    else if (norm == 1 && out_bf16) MX_EN(bf16_t, 1);
    else if (norm == 1) MX_EN(float, 1);
    else if (out_bf16) MX_EN(bf16_t, 2);
    else MX_EN(float, 2);
  });
#undef MX_EN
  return (int)hipGetLastError();
}

// whether these rows go to the kernels that hold a row in registers (layer norm, scaled add, mean of two norms), 512 threads a
// row.  Below 1024 entries most of those have nothing to do, which many rows feel: layer norm of 2000 rows of 256, 1024 and
// 2048 6.6 6.9 7.4 us (entry by entry 4.1 5.4 7.6), of 64 rows 3.1 3.1 3.1 (2.8 3.7 4.8).  Rows that are no whole fours are
// loaded entry by entry here, too, four neighbours a thread: 2050 entries, 64 rows 4.3 (5.1), 300 5.9 (5.5), 2000 15.6 (7.9).
static bool row_in_registers(int rows, int width, int vec) {
  if (width > kRowMaxWidth) return false;
  return vec ? width > 1024 || (width > 512 && rows <= 512) : width > 1024 && rows <= 64;
}

template <typename TY, typename TO>
static void launch_layer_norm(float* x, const void* y, long ys, const float* w, const float* b, void* out,
                              void* cast, const float* nw, const float* nb, int rows, int width, float eps,
                              hipStream_t s) {
  const int vec = width % 4 == 0 && (y == nullptr || (ys % 4 == 0 && ((uintptr_t)y) % (4 * sizeof(TY)) == 0)) &&
                  ((uintptr_t)x | (uintptr_t)w | (uintptr_t)b | (uintptr_t)nw | (uintptr_t)nb) % 16 == 0 &&
                  ((uintptr_t)out | (uintptr_t)cast) % (4 * sizeof(TO)) == 0;
  if (row_in_registers(rows, width, vec)) {
    row_chunks(width, vec, [&](auto c, auto v4) {
      hipLaunchKernelGGL((layer_norm_row_kernel<RowsOf<TY>, TO, decltype(v4)::value, kRowThreads, decltype(c)::value>), dim3(rows),
                         dim3(kRowThreads), 0, s, x, RowsOf<TY>{(const TY*)y, ys}, w, b, (TO*)out, (TO*)cast, nw, nb,
                         width, eps);
    });
    return;
  }
  hipLaunchKernelGGL((layer_norm_kernel<TY, TO, 256>), dim3(rows), dim3(256), 0, s, x, (const TY*)y, ys, w, b,
                     (TO*)out, nw != nullptr ? (TO*)nullptr : (TO*)cast, width, eps);
  if (nw != nullptr)
    hipLaunchKernelGGL((layer_norm_kernel<float, TO, 256>), dim3(rows), dim3(256), 0, s, x, (const float*)nullptr, 0L, nw, nb,
                       (TO*)cast, (TO*)nullptr, width, eps);
}

// next_w, next_b: cast is the layer norm by these of the new residual
extern "C" int mx_layer_norm(float* x, const void* y, int y_bf16, long y_stride, const float* w, const float* b,
                             void* out, void* cast, int out_bf16, const float* next_w,
                             const float* next_b, int rows, int width, float eps, hipStream_t s) {
  if (rows <= 0) return 0;
  if ((y != nullptr && out != nullptr) || (next_w != nullptr && (next_b == nullptr || cast == nullptr || out != nullptr)))
    return -1;
  if (y_bf16) {
    if (out_bf16) launch_layer_norm<bf16_t, bf16_t>(x, y, y_stride, w, b, out, cast, next_w, next_b, rows, width, eps, s);
    else launch_layer_norm<bf16_t, float>(x, y, y_stride, w, b, out, cast, next_w, next_b, rows, width, eps, s);
  } else {
    if (out_bf16) launch_layer_norm<float, bf16_t>(x, y, y_stride, w, b, out, cast, next_w, next_b, rows, width, eps, s);
    else launch_layer_norm<float, float>(x, y, y_stride, w, b, out, cast, next_w, next_b, rows, width, eps, s);
  }
  return (int)hipGetLastError();
}

template <typename TY, typename TO>
static void launch_add_rms(float* x, const void* y, long ys, const float* wb, const float* av,
                           const float* nw, void* out, void* cast, int rows, int width, float eps,
                           hipStream_t s) {
  const int vec = width % 4 == 0 && (y == nullptr || (ys % 4 == 0 && ((uintptr_t)y) % (4 * sizeof(TY)) == 0)) &&
                  ((uintptr_t)x | (uintptr_t)wb | (uintptr_t)av | (uintptr_t)nw) % 16 == 0 &&
                  ((uintptr_t)out | (uintptr_t)cast) % (4 * sizeof(TO)) == 0;
  row_chunks(width, vec, [&](auto c, auto v4) {
    hipLaunchKernelGGL((add_rms_norm_kernel<RowsOf<TY>, TO, decltype(v4)::value, kRowThreads, decltype(c)::value>), dim3(rows),
                       dim3(kRowThreads), 0, s, x, RowsOf<TY>{(const TY*)y, ys}, wb, av, nw, (TO*)out, (TO*)cast, width, eps);
  });
}

extern "C" int mx_add_rms_norm(float* x, const void* y, int y_bf16, long y_stride, const float* wb,
                               const float* add_vec, const float* next_w, void* out, void* cast,
                               int out_bf16, int rows, int width, float eps, hipStream_t s) {
  if (rows <= 0) return 0;
  if (width < 1 || width > kRowMaxWidth) return -1;
  if (y_bf16) {
    if (out_bf16) launch_add_rms<bf16_t, bf16_t>(x, y, y_stride, wb, add_vec, next_w, out, cast, rows, width, eps, s);
    else launch_add_rms<bf16_t, float>(x, y, y_stride, wb, add_vec, next_w, out, cast, rows, width, eps, s);
  } else {
    if (out_bf16) launch_add_rms<float, bf16_t>(x, y, y_stride, wb, add_vec, next_w, out, cast, rows, width, eps, s);
    else launch_add_rms<float, float>(x, y, y_stride, wb, add_vec, next_w, out, cast, rows, width, eps, s);
  }
  return (int)hipGetLastError();
}

// widths of the forms below
extern "C" int mx_expert_rows_fit(int width) { return width % 8 == 0 && width > 1024 && width <= kRowMaxWidth; }

// the three norm steps with the experts' unsummed results as y; bf16 (cast, out) or fp32 results
extern "C" int mx_add_rms_norm_experts(float* x, const float* d, const float* wts, const float* shared, const float* gate,
                                       int top, const float* wb, const float* add_vec, const float* next_w, void* out,
                                       void* cast, int out_bf16, int rows, int width, float eps, hipStream_t s) {
  if (rows <= 0) return 0;
  if (!mx_expert_rows_fit(width) || top < 1) return -1;
  if (((uintptr_t)d | (uintptr_t)shared) % 16) return -2;
  const int vec = ((uintptr_t)x | (uintptr_t)wb | (uintptr_t)add_vec | (uintptr_t)next_w | (uintptr_t)out | (uintptr_t)cast) % 16 == 0;
  const ExpertRows y{d, wts, shared, gate, top};
  row_chunks(width, vec, [&](auto c, auto v4) {
    if (out_bf16)
      hipLaunchKernelGGL((add_rms_norm_kernel<ExpertRows, bf16_t, decltype(v4)::value, kRowThreads, decltype(c)::value>), dim3(rows),
                         dim3(kRowThreads), 0, s, x, y, wb, add_vec, next_w, (bf16_t*)out, (bf16_t*)cast, width, eps);
    else
      hipLaunchKernelGGL((add_rms_norm_kernel<ExpertRows, float, decltype(v4)::value, kRowThreads, decltype(c)::value>), dim3(rows),
                         dim3(kRowThreads), 0, s, x, y, wb, add_vec, next_w, (float*)out, (float*)cast, width, eps);
  });
  return (int)hipGetLastError();
}

extern "C" int mx_layer_norm_experts(float* x, const float* d, const float* wts, const float* shared, const float* gate,
                                     int top, const float* w, const float* b, void* cast, const float* next_w,
                                     const float* next_b, int rows, int width, float eps, hipStream_t s) {
  if (rows <= 0) return 0;
  if (!mx_expert_rows_fit(width) || top < 1) return -1;
  if (((uintptr_t)d | (uintptr_t)shared) % 16) return -2;
  const int vec = ((uintptr_t)x | (uintptr_t)w | (uintptr_t)b | (uintptr_t)next_w | (uintptr_t)next_b | (uintptr_t)cast) % 16 == 0;
  const ExpertRows y{d, wts, shared, gate, top};
  row_chunks(width, vec, [&](auto c, auto v4) {
    hipLaunchKernelGGL((layer_norm_row_kernel<ExpertRows, bf16_t, decltype(v4)::value, kRowThreads, decltype(c)::value>), dim3(rows),
                       dim3(kRowThreads), 0, s, x, y, w, b, (bf16_t*)nullptr, (bf16_t*)cast, next_w, next_b, width, eps);
  });
  return (int)hipGetLastError();
}

// the two norm steps with the grouped products' rows as y (see SortedRows); bf16 results
static int sorted_ok(const SortedRows& y, int width) {
  return mx_expert_rows_fit(width) && y.top >= 1 && y.h_stride % 4 == 0 &&
         ((uintptr_t)y.d | (uintptr_t)y.shared | (uintptr_t)y.h | (uintptr_t)y.gate_w) % 8 == 0;
}

extern "C" int mx_add_rms_norm_sorted(float* x, const void* d, const int* place, const float* wts, const void* shared, const void* h,
                                      long h_stride, const void* gate_w, int top, const float* wb, const float* add_vec,
                                      const float* next_w, void* out, void* cast, int rows, int width, float eps, hipStream_t s) {
  if (rows <= 0) return 0;
  const SortedRows y{(const bf16_t*)d, (const bf16_t*)shared, (const bf16_t*)h, (const bf16_t*)gate_w, place, wts, h_stride, top};
  if (!sorted_ok(y, width)) return -1;
  const int vec = ((uintptr_t)x | (uintptr_t)wb | (uintptr_t)add_vec | (uintptr_t)next_w | (uintptr_t)out | (uintptr_t)cast) % 16 == 0;
  row_chunks(width, vec, [&](auto c, auto v4) {
    hipLaunchKernelGGL((add_rms_norm_kernel<SortedRows, bf16_t, decltype(v4)::value, kRowThreads, decltype(c)::value>), dim3(rows),
                       dim3(kRowThreads), 0, s, x, y, wb, add_vec, next_w, (bf16_t*)out, (bf16_t*)cast, width, eps);
  });
  return (int)hipGetLastError();
}

extern "C" int mx_layer_norm_sorted(float* x, const void* d, const int* place, const float* wts, const void* shared, const void* h,
                                    long h_stride, const void* gate_w, int top, const float* w, const float* b, void* cast,
                                    const float* next_w, const float* next_b, int rows, int width, float eps, hipStream_t s) {
  if (rows <= 0) return 0;
  const SortedRows y{(const bf16_t*)d, (const bf16_t*)shared, (const bf16_t*)h, (const bf16_t*)gate_w, place, wts, h_stride, top};
  if (!sorted_ok(y, width)) return -1;
  const int vec = ((uintptr_t)x | (uintptr_t)w | (uintptr_t)b | (uintptr_t)next_w | (uintptr_t)next_b | (uintptr_t)cast) % 16 == 0;
  row_chunks(width, vec, [&](auto c, auto v4) {
    hipLaunchKernelGGL((layer_norm_row_kernel<SortedRows, bf16_t, decltype(v4)::value, kRowThreads, decltype(c)::value>), dim3(rows),
                       dim3(kRowThreads), 0, s, x, y, w, b, (bf16_t*)nullptr, (bf16_t*)cast, next_w, next_b, width, eps);
  });
  return (int)hipGetLastError();
}

// decode rows: segments of one row at most, x in place
extern "C" int mx_add_norm_shift_experts(float* x, const float* d, const float* wts, const float* shared, const float* gate,
                                         int top, const float* wb, const float* w, const float* shift, void* out,
                                         float* state, int num_slots, const int* start, const int* pos0, const int* slot,
                                         int num_segs, int rows, int width, float eps, hipStream_t s) {
  if (rows <= 0 || num_segs <= 0) return 0;
  if (!mx_expert_rows_fit(width) || top < 1) return -1;
  if (((uintptr_t)d | (uintptr_t)shared) % 16) return -2;
  const int vec = ((uintptr_t)x | (uintptr_t)wb | (uintptr_t)w | (uintptr_t)shift | (uintptr_t)out | (uintptr_t)state) % 16 == 0;
  const ExpertRows y{d, wts, shared, gate, top};
  row_chunks(width, vec, [&](auto c, auto v4) {
    hipLaunchKernelGGL((add_norm_shift_kernel<ExpertRows, bf16_t, decltype(v4)::value, kRowThreads, decltype(c)::value>), dim3(rows),
                       dim3(kRowThreads), 0, s, x, x, y, wb, w, shift, (bf16_t*)out, state, num_slots, start, pos0, slot,
                       num_segs, width, eps);
  });
  return (int)hipGetLastError();
}

extern "C" int mx_head_rms_gate(void* out, int out_bf16, const float* o, const float* w,
                                const void* gate, int gate_bf16, long gate_stride, long rows, int heads,
                                int dv, float eps, int silu, hipStream_t s) {
  const long pairs = rows * heads;
  if (pairs <= 0) return 0;
  const dim3 grid((unsigned)((pairs + 3) / 4)), block(256);
  const int es = gate_bf16 ? 2 : 4;
  if (gate_bf16 == out_bf16 && pairs < (1L << 30) && gate_stride % 4 == 0 && (((uintptr_t)o | (uintptr_t)w) % 16) == 0 &&
      (((uintptr_t)gate | (uintptr_t)out) % (4 * es)) == 0) {
    bool done = true;
    auto go = [&](auto lpr) {
      constexpr int LPR = decltype(lpr)::value, PER = 64 / LPR;
      // four heads' loads a lane once that leaves waves for the whole chip
      MX_DISPATCH_T(gate_bf16, {
        if (pairs >= 4096L * PER)
          hipLaunchKernelGGL((head_rms_gate_fours_kernel<T, T, LPR, 4>), dim3((unsigned)((pairs + 16 * PER - 1) / (16 * PER))), block, 0,
                             s, (T*)out, o, w, (const T*)gate, gate_stride, (int)pairs, heads, eps, silu);
        else
          hipLaunchKernelGGL((head_rms_gate_fours_kernel<T, T, LPR, 1>), dim3((unsigned)((pairs + 4 * PER - 1) / (4 * PER))), block, 0,
                             s, (T*)out, o, w, (const T*)gate, gate_stride, (int)pairs, heads, eps, silu);
      });
    };
    if (dv == 16) go(std::integral_constant<int, 4>{});
    else if (dv == 32) go(std::integral_constant<int, 8>{});
    else if (dv == 64) go(std::integral_constant<int, 16>{});
    else if (dv == 128) go(std::integral_constant<int, 32>{});
    else if (dv == 256) go(std::integral_constant<int, 64>{});
    else done = false;
    if (done) return (int)hipGetLastError();
  }
  if (gate_bf16 && out_bf16)
    hipLaunchKernelGGL((head_rms_gate_kernel<bf16_t, bf16_t>), grid, block, 0, s, (bf16_t*)out, o, w,
                       (const bf16_t*)gate, gate_stride, pairs, heads, dv, eps, silu);
  else if (!gate_bf16 && !out_bf16)
    hipLaunchKernelGGL((head_rms_gate_kernel<float, float>), grid, block, 0, s, (float*)out, o, w,
                       (const float*)gate, gate_stride, pairs, heads, dv, eps, silu);
  else
    return -1;
  return (int)hipGetLastError();
}

extern "C" int mx_scaled_pair_rows(void* out, int bf16, const float* a, int n, float a_scale, const float* o,
                                   const void* gate, long gate_stride, float o_scale, long rows, int heads, int dv,
                                   float eps, hipStream_t s) {
  const int items = heads + (n + 255) / 256;
  const long waves = rows * items;
  if (waves <= 0) return 0;
  const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
  MX_DISPATCH_T(bf16, hipLaunchKernelGGL((scaled_pair_rows_kernel<T>), grid, block, 0, s, (T*)out, a, n, a_scale, o,
                                         (const T*)gate, gate_stride, o_scale, waves, items, heads, dv, eps));
  return (int)hipGetLastError();
}

static inline unsigned ew_grid(long n) {
  long g = (n + 255) / 256;
  return (unsigned)(g < 1 ? 1 : g > 65535 ? 65535 : g);
}

// whole 16-byte pieces in every row of gate, up and out
static inline int glu_vec(const void* out, const void* gu, int bf16, long gu_stride, int ff) {
  const int n = bf16 ? 8 : 4;
  return ff % n == 0 && gu_stride % n == 0 && ((uintptr_t)out | (uintptr_t)gu) % 16 == 0;
}

extern "C" int mx_tanh_cap(float* x, long n, float cap, hipStream_t s) {
  if (n <= 0) return 0;
  if (!(cap > 0.f)) return -1;
  hipLaunchKernelGGL(tanh_cap_kernel, dim3(ew_grid(n)), dim3(256), 0, s, x, n, cap);
  return (int)hipGetLastError();
}

extern "C" int mx_relu_sq(void* x, int bf16, long n, hipStream_t s) {
  if (n <= 0) return 0;
  MX_DISPATCH_T(bf16, hipLaunchKernelGGL((relu_sq_kernel<T>), dim3(ew_grid(n)), dim3(256), 0, s, (T*)x, n));
  return (int)hipGetLastError();
}

extern "C" int mx_relu_sq_rows(void* out, const void* u, int bf16, long u_stride, long rows, int ff, hipStream_t s) {
  if (rows * ff <= 0) return 0;
  MX_DISPATCH_T(bf16, hipLaunchKernelGGL((relu_sq_rows_kernel<T>), dim3(ew_grid(rows * ff)), dim3(256), 0, s,
                                         (T*)out, (const T*)u, u_stride, rows, ff));
  return (int)hipGetLastError();
}

extern "C" int mx_gather_add_rows(float* out, const void* y, int y_bf16, const int* idx, const float* w, long rows,
                                  int top, int width, long y_rows, hipStream_t s) {
  if (rows <= 0 || top <= 0) return 0;
  if (rows > 0x7fffffffL) return -1;
  MX_DISPATCH_T(y_bf16, hipLaunchKernelGGL((gather_add_rows_kernel<T>), dim3((unsigned)rows), dim3(256), 0, s, out,
                                           (const T*)y, idx, w, top, width, y_rows));
  return (int)hipGetLastError();
}

extern "C" int mx_clamp_swiglu(void* out, const void* gu, int bf16, long gu_stride, long rows, int ff,
                               float limit, hipStream_t s) {
  if (rows * ff <= 0) return 0;
  const int vec = glu_vec(out, gu, bf16, gu_stride, ff);
  MX_DISPATCH_T(bf16, hipLaunchKernelGGL((clamp_swiglu_kernel<T>), dim3(ew_grid(vec ? rows * (ff / GluVec<T>::N) : rows * ff)),
                                         dim3(256), 0, s, (T*)out, (const T*)gu, gu_stride, rows, ff, limit, vec));
  return (int)hipGetLastError();
}

extern "C" int mx_act_glu(void* out, const void* gu, int bf16, long gu_stride, long rows, int ff, int act,
                          hipStream_t s) {
  if (rows * ff <= 0) return 0;
  if (act < 0 || act > 2) return -1;
  const int vec = glu_vec(out, gu, bf16, gu_stride, ff);
  MX_DISPATCH_T(bf16, hipLaunchKernelGGL((act_glu_kernel<T>), dim3(ew_grid(vec ? rows * (ff / GluVec<T>::N) : rows * ff)),
                                         dim3(256), 0, s, (T*)out, (const T*)gu, gu_stride, rows, ff, act, vec));
  return (int)hipGetLastError();
}

extern "C" int mx_side_gate(void* out, const void* gpre, const void* table, int bf16, long table_stride,
                            const int* ids, int col0, long rows, int sd, int vocab, hipStream_t s) {
  if (rows * sd <= 0) return 0;
  MX_DISPATCH_T(bf16, hipLaunchKernelGGL((side_gate_kernel<T>), dim3(ew_grid(rows * sd)), dim3(256), 0, s,
                                         (T*)out, (const T*)gpre, (const T*)table, table_stride, ids, col0,
                                         rows, sd, vocab));
  return (int)hipGetLastError();
}

extern "C" int mx_scale_add_rows(float* out, const void* y, int y_bf16, const int* rows,
                                 const void* weights, int w_bf16, int sigmoid, long n, int width,
                                 int out_rows, hipStream_t s) {
  if (n <= 0) return 0;
  const dim3 grid((unsigned)n), block(256);
  if (y_bf16 && w_bf16)
    hipLaunchKernelGGL((scale_add_rows_kernel<bf16_t, bf16_t>), grid, block, 0, s, out, (const bf16_t*)y,
                       rows, (const bf16_t*)weights, sigmoid, width, out_rows);
  else if (y_bf16)
    hipLaunchKernelGGL((scale_add_rows_kernel<bf16_t, float>), grid, block, 0, s, out, (const bf16_t*)y,
                       rows, (const float*)weights, sigmoid, width, out_rows);
  else if (w_bf16)
    return -1;
  else
    hipLaunchKernelGGL((scale_add_rows_kernel<float, float>), grid, block, 0, s, out, (const float*)y,
                       rows, (const float*)weights, sigmoid, width, out_rows);
  return (int)hipGetLastError();
}

// x (fp32 residual) += table[hash]
extern "C" int mx_pair_embed_add(float* x, const int* ids, const void* table, int bf16, int rows, int width,
                                 long mul_prev, long mul_cur, int buckets, const int* start, const int* pos0,
                                 const int* slot, int num_segs, int* last_tok, int num_slots, hipStream_t s) {
  if (rows <= 0 || num_segs <= 0) return 0;
  if (buckets < 1 || width < 1) return -1;
  const PairArgs P{table, mul_prev, mul_cur, buckets, num_segs, num_slots, start, pos0, slot, last_tok};
  MX_DISPATCH_T(bf16, hipLaunchKernelGGL((pair_embed_add_kernel<T>), dim3(rows), dim3(256), 0, s, x, ids, P, width,
                                         (const T*)nullptr, 0, 1.f));
  return (int)hipGetLastError();
}

// whether AnyRows may be read four entries at a time; parts: -1 if they cannot be read
static int any_rows_vec(const AnyRows& y, int width) {
  if (y.parts > 1) return y.p != nullptr && !y.bf16 && mx_expert_rows_fit(width) && ((uintptr_t)y.p) % 16 == 0 ? 1 : -1;
  return y.p == nullptr || (y.stride % 4 == 0 && ((uintptr_t)y.p) % (y.bf16 ? 8 : 16) == 0);
}

// y1, y2: rows of their stride, or (parts > 1) fp32 [rows * parts, width] whose sums over the parts are the rows
extern "C" int mx_add_scaled_rms_norm(float* x, const void* y1, int y1_bf16, long y1_stride, int y1_parts, const void* y2,
                                      int y2_bf16, long y2_stride, int y2_parts, float mult, const float* next_w, void* out,
                                      int out_bf16, int rows, int width, float eps, hipStream_t s) {
  if (rows <= 0) return 0;
  if (y1 == nullptr && (y2 != nullptr || out == nullptr)) return -1;
  const AnyRows a{y1, y1_bf16, y1_parts, y1_stride}, b{y2, y2_bf16, y2_parts, y2_stride};
  const int va = any_rows_vec(a, width), vb = any_rows_vec(b, width);
  if (va < 0 || vb < 0) return -2;
  const int vec = width % 4 == 0 && va && vb &&
                  ((uintptr_t)x | (uintptr_t)next_w) % 16 == 0 && ((uintptr_t)out) % (out_bf16 ? 8 : 16) == 0;
  if (row_in_registers(rows, width, vec) || y1_parts > 1 || y2_parts > 1) {
    auto go = [&](auto parts) {
      row_chunks(width, vec, [&](auto c, auto v4) {
        constexpr int A = decltype(parts)::value, C = decltype(c)::value;
        if (out_bf16)
          hipLaunchKernelGGL((add_scaled_rms_norm_row_kernel<bf16_t, decltype(v4)::value, A, kRowThreads, C>), dim3(rows),
                             dim3(kRowThreads), 0, s, x, a, b, mult, next_w, (bf16_t*)out, width, eps);
        else
          hipLaunchKernelGGL((add_scaled_rms_norm_row_kernel<float, decltype(v4)::value, A, kRowThreads, C>), dim3(rows),
                             dim3(kRowThreads), 0, s, x, a, b, mult, next_w, (float*)out, width, eps);
      });
    };
    if (y1_parts > 1 || y2_parts > 1) go(std::integral_constant<int, kAskedParts>{});
    else go(std::integral_constant<int, 1>{});
    return (int)hipGetLastError();
  }
  if (out_bf16)
    hipLaunchKernelGGL((add_scaled_rms_norm_kernel<bf16_t, 256>), dim3(rows), dim3(256), 0, s, x, y1, y1_bf16,
                       y1_stride, y2, y2_bf16, y2_stride, mult, next_w, (bf16_t*)out, width, eps);
  else
    hipLaunchKernelGGL((add_scaled_rms_norm_kernel<float, 256>), dim3(rows), dim3(256), 0, s, x, y1, y1_bf16,
                       y1_stride, y2, y2_bf16, y2_stride, mult, next_w, (float*)out, width, eps);
  return (int)hipGetLastError();
}

// a, b: as mx_add_scaled_rms_norm's, both bf16 or both fp32 unless in parts
extern "C" int mx_dual_rms_mean(float* out, const void* a, int a_bf16, long a_stride, int a_parts, const void* b, int b_bf16,
                                long b_stride, int b_parts, const float* wa, const float* wb, int rows, int width, float eps,
                                float scale, hipStream_t s) {
  if (rows <= 0) return 0;
  const AnyRows ra{a, a_bf16, a_parts, a_stride}, rb{b, b_bf16, b_parts, b_stride};
  const int va = any_rows_vec(ra, width), vb = any_rows_vec(rb, width);
  if (va < 0 || vb < 0) return -2;
  const int vec = width % 4 == 0 && va && vb && ((uintptr_t)out | (uintptr_t)wa | (uintptr_t)wb) % 16 == 0;
  if (row_in_registers(rows, width, vec) || a_parts > 1 || b_parts > 1) {
    auto go = [&](auto parts) {
      row_chunks(width, vec, [&](auto c, auto v4) {
        hipLaunchKernelGGL((dual_rms_mean_row_kernel<decltype(v4)::value, decltype(parts)::value, kRowThreads, decltype(c)::value>),
                           dim3(rows), dim3(kRowThreads), 0, s, out, ra, rb, wa, wb, width, eps, scale);
      });
    };
    if (a_parts > 1 || b_parts > 1) go(std::integral_constant<int, kAskedParts>{});
    else go(std::integral_constant<int, 1>{});
    return (int)hipGetLastError();
  }
  if (a_bf16 != b_bf16) return -1;
  MX_DISPATCH_T(a_bf16, hipLaunchKernelGGL((dual_rms_mean_kernel<T, 256>), dim3(rows), dim3(256), 0, s, out,
                                           (const T*)a, a_stride, (const T*)b, b_stride, wa, wb, width, eps, scale));
  return (int)hipGetLastError();
}

extern "C" int mx_sigmoid_gate(void* out, int out_bf16, const float* o, const void* g, int g_bf16, long g_stride,
                               long rows, int n, hipStream_t s) {
  if (rows * n <= 0) return 0;
  const dim3 grid(ew_grid(rows * n)), block(256);
  if (g_bf16 && out_bf16)
    hipLaunchKernelGGL((sigmoid_gate_kernel<bf16_t, bf16_t>), grid, block, 0, s, (bf16_t*)out, o, (const bf16_t*)g,
                       g_stride, rows, n);
  else if (!g_bf16 && !out_bf16)
    hipLaunchKernelGGL((sigmoid_gate_kernel<float, float>), grid, block, 0, s, (float*)out, o, (const float*)g,
                       g_stride, rows, n);
  else
    return -1;
  return (int)hipGetLastError();
}

template <typename TY, typename TO>
static void launch_shift(float* x_out, const float* x_in, const void* y, long ys, const float* wb, const float* w,
                         const float* shift, void* out, float* state, int num_slots, const int* start,
                         const int* pos0, const int* slot, int num_segs, int max_rows, int rows, int width, float eps,
                         hipStream_t s) {
  const int vec = width % 4 == 0 && (y == nullptr || (ys % 4 == 0 && ((uintptr_t)y) % (4 * sizeof(TY)) == 0)) &&
                  ((uintptr_t)x_in | (uintptr_t)x_out | (uintptr_t)w | (uintptr_t)wb | (uintptr_t)shift |
                   (uintptr_t)state) % 16 == 0 && ((uintptr_t)out) % (4 * sizeof(TO)) == 0;
  row_chunks(width, vec, [&](auto c, auto v4) {
    constexpr int C = decltype(c)::value;
    hipLaunchKernelGGL((add_norm_shift_kernel<RowsOf<TY>, TO, decltype(v4)::value, kRowThreads, C>), dim3(rows), dim3(kRowThreads), 0, s, x_out,
                       x_in, RowsOf<TY>{(const TY*)y, ys}, wb, w, shift, (TO*)out, state, num_slots, start, pos0, slot,
                       num_segs, width, eps);
    if (max_rows > 1)
      hipLaunchKernelGGL((shift_state_kernel<decltype(v4)::value, kRowThreads, C>), dim3(num_segs), dim3(kRowThreads), 0, s, state,
                         num_slots, x_out, w, start, slot, width, eps);
  });
}

extern "C" int mx_row_max_width() { return kRowMaxWidth; }

extern "C" int mx_add_norm_shift(float* x_out, const float* x_in, const void* y, int y_bf16, long y_stride,
                                 const float* wb, const float* w, const float* shift, void* out, int out_bf16,
                                 float* state, int num_slots, const int* start, const int* pos0, const int* slot,
                                 int num_segs, int max_rows, int rows, int width, float eps, hipStream_t s) {
  if (rows <= 0 || num_segs <= 0) return 0;
  if (width < 1 || width > kRowMaxWidth || (y != nullptr && max_rows > 1 && x_out == x_in)) return -1;
#define MX_SHIFT(TY, TO)                                                                                       \
  launch_shift<TY, TO>(x_out, x_in, y, y_stride, wb, w, shift, out, state, num_slots, start, pos0, slot,       \
                       num_segs, max_rows, rows, width, eps, s)
  if (y_bf16 && out_bf16) MX_SHIFT(bf16_t, bf16_t);
  else if (y_bf16) MX_SHIFT(bf16_t, float);
  else if (out_bf16) MX_SHIFT(float, bf16_t);
  else MX_SHIFT(float, float);
#undef MX_SHIFT
  return (int)hipGetLastError();
}

// Tiles of 32 rows of the latent cache ([c (512) | rotated key (64)], bf16) in LDS, shared by the latent
// attention kernels (latent_prefill.hip, latent_decode.hip).  They arrive by global_load_lds_dwordx4; the same
// image is read as keys (ds_read_b128) and, transposed, as values (ds_read_b64_tr_b16).
// LDS image of a tile: 16-byte piece p of key k at ((p / 8 * 4 + k / 8) * 8 + k % 8) * 8 + (p % 8 ^ lp_swap(k)):
// eight neighbouring lanes of a load read 128 neighbouring bytes of a cache row (with a key per lane the load
// unit, one line at a time, took 5% more), and neither way of reading has bank conflicts within 16 lanes (those
// counted are a tenth of the cycles).
#pragma once
#include "mx_common.h"
#include "ft_lds.h"

namespace mx {

typedef __bf16 lp_bf16x8 __attribute__((ext_vector_type(8)));
typedef float lp_f32x4 __attribute__((ext_vector_type(4)));
typedef short lp_i16x4 __attribute__((ext_vector_type(4)));

constexpr int kLpRank = 512, kLpRot = 64, kLpWidth = kLpRank + kLpRot;
constexpr int kLpKeys = 32;
constexpr int kLpTile = kLpKeys * kLpWidth * 2;       // bytes
constexpr int kLpDma = kLpTile / 4096;                // 1 KiB loads of eight keys' 128 bytes each

__device__ __forceinline__ int lp_swap(int key) { return ((key >> 1) & 3) * 2 + ((key >> 3) & 1); }

__device__ __forceinline__ lp_f32x4 lp_mfma(const uint4& a, const uint4& b, lp_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(lp_bf16x8, a), __builtin_bit_cast(lp_bf16x8, b), c,
                                                 0, 0, 0);
}

typedef __attribute__((address_space(3))) lp_i16x4 lp_lds_i16x4;

// byte offsets in a tile for lane (g4, n).  As keys: piece 4 s + g4 of key n (odd s: 4 pieces on; keys 16 ..:
// 2048 on; steps 2 s: 4096 s on).  As values: key n / 4 of the group's four, columns 4 (n % 4) .. of a 16-column
// tile (column tile mod 4; four tiles: 4096 on)
__device__ __forceinline__ void lp_offsets(int n, int g4, int (&k_off)[2], int (&v_off)[4]) {
#pragma unroll
  for (int h = 0; h < 2; ++h) k_off[h] = n * 128 + ((4 * h + g4) ^ lp_swap(n)) * 16;
  const int vkey = 4 * g4 + (n >> 2);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    v_off[j] = vkey * 128 + ((2 * j + ((n >> 1) & 1)) ^ lp_swap(vkey)) * 16 + (n & 1) * 8;
}

// values of column tile u: keys 4 g4 .. + 3 and 16 + 4 g4 .. + 3 of column n
__device__ __forceinline__ uint4 lp_values(const uint8_t* tile, int u, const int (&v_off)[4]) {
  const uint8_t* at = tile + (u >> 2) * 4096 + v_off[u & 3];
  const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp_lds_i16x4*)at));
  const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp_lds_i16x4*)(at + 2048)));
  return make_uint4(lo.x, lo.y, hi.x, hi.y);
}

// eight keys' loads: `row` this lane's cache row (key lane / 8 of octet ko), dst the tile's LDS address
__device__ __forceinline__ void lp_issue(const bf16_t* row, int ko, int lane, uint32_t dst) {
  const bf16_t* src = row + ((lane & 7) ^ lp_swap(8 * ko + (lane >> 3))) * 8;
#pragma unroll
  for (int i = 0; i < kLpDma; ++i) ft::glds16(src + i * 64, dst + ko * 1024 + i * 4096);
}

}  // namespace mx

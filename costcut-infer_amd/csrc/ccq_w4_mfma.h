// Pieces shared by the AWQ int4 kernels: the scale/zero word layout, the
// 16-bit activation types, the MFMA wrappers and the in-register dequantization
// of packed weight dwords (layouts: ccq_w4.hip).
#pragma once

#include "ccq_common.h"

namespace ccq {

__host__ __device__ inline int64_t sz_words_per_column(int64_t K, int64_t G) {
  return ((K / 128 + 3) / 4) * 4 * (128 / G);
}

// ------------------------------------------------------------- MFMA pieces --
template <typename AT>
struct Act;
template <>
struct Act<__bf16> {
  using vec = bf16x8;
  static constexpr uint32_t kMagic2 = 0x43004300u;  // bf16 128.0 twice
  static constexpr float kMagic = 128.0f;
  static constexpr uint32_t kOne2 = 0x3F803F80u;
};
template <>
struct Act<_Float16> {
  using vec = f16x8;
  static constexpr uint32_t kMagic2 = 0x64006400u;  // fp16 1024.0 twice
  static constexpr float kMagic = 1024.0f;
  static constexpr uint32_t kOne2 = 0x3C003C00u;
};

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(f16x8 a, f16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
// 32x32x16: A lane l = row l & 31, B lane l = column l & 31, both with
// k = 8*(l >> 5) + e; D register i of lane l = (row 8*(i/4) + 4*(l >> 5) + i%4,
// column l & 31).
__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma32(f16x8 a, f16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

template <typename AT>
__device__ __forceinline__ typename Act<AT>::vec dq_b(uint32_t w) {
  u32x4 r;
  r[0] = (w & 0x000F000Fu) | Act<AT>::kMagic2;
  r[1] = ((w >> 4) & 0x000F000Fu) | Act<AT>::kMagic2;
  r[2] = ((w >> 8) & 0x000F000Fu) | Act<AT>::kMagic2;
  r[3] = ((w >> 12) & 0x000F000Fu) | Act<AT>::kMagic2;
  return __builtin_bit_cast(typename Act<AT>::vec, r);
}

// dq_b with one v_and_or_b32 per weight pair: the mask and the magic come in
// as run-time values (an SGPR and a VGPR), since a VOP3 op on gfx9 takes no
// literal and (w & literal) | literal would cost two ops.
template <typename AT>
__device__ __forceinline__ typename Act<AT>::vec dq_b3(uint32_t w, uint32_t mask_s, uint32_t magic_v) {
  u32x4 r;
  r[0] = (w & mask_s) | magic_v;
  r[1] = ((w >> 4) & mask_s) | magic_v;
  r[2] = ((w >> 8) & mask_s) | magic_v;
  r[3] = ((w >> 12) & mask_s) | magic_v;
  return __builtin_bit_cast(typename Act<AT>::vec, r);
}

__device__ __forceinline__ void store_val(void* y, int64_t i, float v, int dt) {
  if (dt == CCQ_F32)
    reinterpret_cast<float*>(y)[i] = v;
  else if (dt == CCQ_BF16)
    reinterpret_cast<uint16_t*>(y)[i] = (uint16_t)f32_to_bf16_bits(v);
  else
    reinterpret_cast<uint16_t*>(y)[i] = (uint16_t)f32_to_f16_bits(v);
}

template <typename ST>
__device__ __forceinline__ float sz_scale(uint32_t word);
template <>
__device__ __forceinline__ float sz_scale<__bf16>(uint32_t word) {
  return __uint_as_float(word << 16);
}
template <>
__device__ __forceinline__ float sz_scale<_Float16>(uint32_t word) {
  return f16_bits_to_f32(word & 0xFFFFu);
}

// Dense y[M, N] = x[M, K] @ W (ccq_w4_dense.hip), for M above the 16 rows of
// the decode kernel.
struct W4DenseP {
  const void* x;
  const uint32_t* w;   // tiled weights
  const uint32_t* sz;  // scale / zero words
  void* y;
  int x_bf16, s_bf16, y_dtype;
  int64_t M, K, N, G;
};
// Waves of the 16-row kernel's grid (w4_skinny_kernel): its weight passes times
// its workgroups of up to 8 waves on 64 (G = 32: 32) columns.  N / 16 that is no
// multiple of 4 has 32- or 16-column workgroups, up to four times as many; they
// count as 64 columns all the same, since more of them share a CU (counted one
// by one, M=65 K=3584 N=1040 would leave this kernel's 11.3 us for 15.6).
inline int64_t w4_skinny_waves(int64_t M, int64_t K, int64_t N, int64_t G) {
  return cdiv(M, 16) * cdiv(N, G == 32 ? 32 : 64) * imin64(8, cdiv(K / 128, 4));
}
// Shapes of the 128-row grouped kernel.
inline bool w4_grouped_shape(int64_t M, int64_t K, int64_t N, int64_t G) {
  return M > 64 && G == 128 && N % 128 == 0 && K >= 256;
}
// It takes them unless the 16-row kernel does them in two rounds of the 256
// CUs (8 waves each) or the slab kernel in one round of its 64 x 64 blocks:
// the grouped kernel's row sums, split-K sums and launches cost about 20 us
// by themselves (M=128 K=2048 N=2048 10.4 us against 22.0, M=65 K=2048 N=9216
// 15.1 against 24, both the 16-row kernel; M=256 K=4096 N=4096 33 against 17
// of the slab kernel; past those M=400 K=4096 N=4096 39 against 76 and M=128
// K=4096 N=14336 40 against 81 and 50).  A short K has few waves however many
// rows there are: past two rounds of 64 x 64 blocks the grouped kernel takes
// those too (K=512: M=1024 N=2048 13.7 us against 18.6, but M=1024 N=2176 21.6
// -> 14.1 and M=8192 N=512 31.3 -> 20.5; K=256 the same way, 11.4 against 14.8
// and 17.0 -> 11.5, 22.7 -> 16.2).
inline bool w4_grouped_takes(int64_t M, int64_t K, int64_t N, int64_t G) {
  const int64_t blocks = cdiv(M, 64) * cdiv(N, 64);
  return w4_grouped_shape(M, K, N, G) && blocks > 256 && (blocks > 512 || w4_skinny_waves(M, K, N, G) > 2 * 256 * 8);
}
bool w4_slab_takes(int64_t M, int64_t K, int64_t N, int64_t G);
size_t w4_slab_workspace(int64_t M, int64_t K, int64_t N);  // 0 when K is not split
// y = the sum of `splits` float32 partials of n values each, n % 4 == 0
int launch_w4_split_sum(const float* part, void* y, int y_dtype, int splits, int64_t n, hipStream_t st);
int launch_w4_slab(const W4DenseP& p, void* workspace, size_t workspace_bytes, hipStream_t st);

}  // namespace ccq

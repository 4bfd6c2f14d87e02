// Pieces shared by the decoded-weight MFMA linears (ccq_wmfma.hip up to 64
// rows, ccq_wtile.hip above): parameters, formats and the in-register decode.
#pragma once

#include "ccq_common.h"

namespace ccq {

struct WqP {
  const float* x;
  const uint8_t* w;
  const void* scale;  // float [N] (row formats), E8M0 bytes [N, K / G] (MX), or null (MXFP4 only)
  float* y;
  int64_t M, K, N;
  int G;
  float s2;
};

template <int FMT>
struct WqTraits {
  static constexpr int WB = FMT == WQ_MXFP4 ? 1 : 2;      // 16-byte weight pieces per lane and chunk
  static constexpr int KDIV = FMT == WQ_MXFP4 ? 2 : 1;    // k per weight byte
  static constexpr bool MX = FMT == WQ_MXFP8 || FMT == WQ_MXFP4;
};

__device__ __forceinline__ bf16x8 pack_bf16x8(const float (&v)[8]) {
  u32x4 r;
  r[0] = bf16x2_bits(v[0], v[1]);
  r[1] = bf16x2_bits(v[2], v[3]);
  r[2] = bf16x2_bits(v[4], v[5]);
  r[3] = bf16x2_bits(v[6], v[7]);
  return __builtin_bit_cast(bf16x8, r);
}

// Eight consecutive weights (8 bytes w0, w1; one word w0 of MXFP4 codes),
// times the group scale s for the MX formats, as bf16.
template <int FMT>
__device__ __forceinline__ bf16x8 wq_decode8(uint32_t w0, uint32_t w1, float s) {
  float v[8];
  if constexpr (FMT == WQ_MXFP4) {
    mx4_word(w0, v);
  } else if constexpr (FMT == WQ_INT8_ROW) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = (float)(int8_t)(w0 >> (8 * j));
      v[4 + j] = (float)(int8_t)(w1 >> (8 * j));
    }
  } else {
    const auto a = __builtin_amdgcn_cvt_pk_f32_fp8((int)w0, false);
    const auto b = __builtin_amdgcn_cvt_pk_f32_fp8((int)w0, true);
    const auto c = __builtin_amdgcn_cvt_pk_f32_fp8((int)w1, false);
    const auto d = __builtin_amdgcn_cvt_pk_f32_fp8((int)w1, true);
    v[0] = a[0], v[1] = a[1], v[2] = b[0], v[3] = b[1];
    v[4] = c[0], v[5] = c[1], v[6] = d[0], v[7] = d[1];
  }
  if constexpr (WqTraits<FMT>::MX) {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] *= s;
  }
  return pack_bf16x8(v);
}

// The lane's weight values 8i..8i+7 of the chunk as the MFMA's B fragment.
template <int FMT>
__device__ __forceinline__ bf16x8 wq_decode(const u32x4 (&wr)[WqTraits<FMT>::WB], int i, float s) {
  if constexpr (FMT == WQ_MXFP4)
    return wq_decode8<FMT>(wr[0][i], 0, s);
  else
    return wq_decode8<FMT>(wr[i >> 1][(i & 1) * 2], wr[i >> 1][(i & 1) * 2 + 1], s);
}

// The tiled form for many rows; -1 when it does not take the shape.
int wq_tile_linear(int fmt, const WqP& p, bool g16, hipStream_t st, const char* name);

}  // namespace ccq

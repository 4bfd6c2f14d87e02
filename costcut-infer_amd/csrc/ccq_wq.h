// Pieces shared by the decoded-weight MFMA linears (ccq_wrows.hip up to 16 rows,
// ccq_wmfma.hip up to 64 rows a workgroup, ccq_wtile.hip above): parameters, formats and the in-register decode.
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

// The bf16 values of the reference's 4-bit table times 2^(e - 127) (E8M0 byte
// e: 0 -> 0, 255 -> NaN), as byte tables for v_perm_b32: low bytes, high bytes
// of codes 0-3 and of codes 4-7 (the negated values).  Exact: 0.5, 1 and 1.5
// times a power of two, with 0.5 * 2^-126 the subnormal 0x0040.
struct Mx4Lut {
  uint32_t lo, hp, hn;
};
__device__ __forceinline__ Mx4Lut mx4_lut(uint32_t e) {
  const uint32_t l2 = (e & 1u) << 7, l1 = e == 1u ? 0x40u : (((e - 1u) & 1u) << 7);
  const uint32_t h2 = e >> 1, h1 = (e - 1u) >> 1;
  Mx4Lut t;
  t.lo = (l1 << 8) | (l2 << 16) | ((l2 | 0x40u) << 24);
  t.hp = (h1 << 8) | (h2 * 0x01010000u);
  if (e == 0u) t.lo = t.hp = 0u;
  if (e == 255u) {
    t.lo = 0xC0C0C0C0u;
    t.hp = 0x7F7F7F7Fu;
  }
  t.hn = t.hp | 0x80808080u;
  return t;
}
// Columns 8w..8w+7 of one word of codes (low nibble = even column): 15 integer
// operations, against 29 for the f16 table, float conversion and scaling.
__device__ __forceinline__ bf16x8 mx4_word_bf16(uint32_t w, const Mx4Lut& t) {
  const uint32_t se = w & 0x07070707u, so = (w >> 4) & 0x07070707u;
  const uint32_t el = __builtin_amdgcn_perm(t.lo, t.lo, se), eh = __builtin_amdgcn_perm(t.hn, t.hp, se);
  const uint32_t ol = __builtin_amdgcn_perm(t.lo, t.lo, so), oh = __builtin_amdgcn_perm(t.hn, t.hp, so);
  const uint32_t e01 = __builtin_amdgcn_perm(eh, el, 0x05010400u), e23 = __builtin_amdgcn_perm(eh, el, 0x07030602u);
  const uint32_t o01 = __builtin_amdgcn_perm(oh, ol, 0x05010400u), o23 = __builtin_amdgcn_perm(oh, ol, 0x07030602u);
  u32x4 r;
  r[0] = __builtin_amdgcn_perm(o01, e01, 0x05040100u);
  r[1] = __builtin_amdgcn_perm(o01, e01, 0x07060302u);
  r[2] = __builtin_amdgcn_perm(o23, e23, 0x05040100u);
  r[3] = __builtin_amdgcn_perm(o23, e23, 0x07060302u);
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

// The form for up to 16 rows: its 16-column tiles per workgroup, 0 for shapes it
// does not take (the launch: -1).
int wq_rows_route(int fmt, bool g16, int64_t M, int64_t K, int64_t N);
int wq_rows_linear(int fmt, const WqP& p, bool g16, hipStream_t st, const char* name);
// The tiled form for many rows: its tile, false for shapes it does not take
// (the launch: -1).
bool wq_tile_route(int fmt, int64_t M, int64_t K, int64_t N, int& bm, int& bn);
int wq_tile_linear(int fmt, const WqP& p, bool g16, hipStream_t st, const char* name);

}  // namespace ccq

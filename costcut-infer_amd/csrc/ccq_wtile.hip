// Decoded-weight MFMA linear for many rows: y[M, N] = x[M, K] @ W[N, K]^T in
// float32 on byte-coded weights (formats and arithmetic: ccq_wmfma.hip).
//
// The kernel for up to 64 rows reads and converts all activations once per 64
// columns and all weights once per 64 rows; here a workgroup owns a BM x BN
// tile (128 x 256 at most), converts its activations to bf16 parts and decodes
// its weights once into LDS, and 8 waves multiply 32x32x16 MFMA tiles from
// there.  K runs in chunks of 64, double-buffered: the next chunk's global
// loads are in flight during the MFMAs and are converted into the other
// buffer after them, one barrier per chunk.  LDS rows are 128 bytes, their
// 16-byte pieces XOR-swizzled by (row >> 1): 16 rows of an operand read, and
// the 16 pieces that two rows' worth of writers store, hit 16 different bank
// groups.
//
// What bounds it (fp8 M=512 K=4096 N=14336, 129 us = 0.93 PFLOP/s of bf16 MFMA
// work; 332 us before): 224 workgroups of 128 x 256 and, in each, the MFMAs of
// a chunk (about 0.9 of its 2 us) followed by its conversions.
//
// Activation parts: two (x = hi + lo, |x - hi - lo| <= 2^-17 |x|, as the
// 64-row kernel) where in_features % 256 == 0; three otherwise, since those
// shapes otherwise run on the float32 streaming kernels: truncations to 8 bits
// each, so that x = hi + mid + lo exactly down to |x| = 2^-110 (below, what is
// under bf16's smallest step 2^-133 is lost).
//
// Weights are exact in bf16 except MXFP8 codes under the E8M0 bytes 1 and 2
// (scales 2^-126 and 2^-125), which reach below bf16's smallest step 2^-133.
// With three parts (the float32 kernels took those shapes) a workgroup that
// meets such a byte starts over: once with bf16 weights that are zero only
// where the weight is, once with 2^64 times what those leave (wq_tiny8).  The
// others pay an OR per scale byte.
//
// Sums: the MFMAs add up 128 k, and these spans are added on the VALU: K / 16
// dependent roundings in one chain would cost more than the parts do (K=2176:
// 4.3e-7 relative against 64 bits in one chain, the streaming kernels 1.3e-7).
#include "ccq_wq.h"

#include <type_traits>

namespace ccq {

namespace {

constexpr int WT_KC = 64;

// 8 floats -> NSP bf16 pieces of 16 bytes (fin_only, three parts: Inf and NaN -> 0)
template <int NSP>
__device__ __forceinline__ void split8(const float (&v)[8], u32x4 (&o)[NSP], bool fin_only) {
  if constexpr (NSP == 2) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t h = bf16x2_bits(v[2 * j], v[2 * j + 1]);
      o[0][j] = h;
      o[1][j] = bf16x2_bits(v[2 * j] - __uint_as_float(h << 16), v[2 * j + 1] - __uint_as_float(h & 0xffff0000u));
    }
  } else {
    uint32_t p[3][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t u = __float_as_uint(v[e]);
      const bool fin = (u & 0x7f800000u) != 0x7f800000u;
      const float r = fin ? v[e] - __uint_as_float(u & 0xffff0000u) : 0.f;
      const uint32_t ur = __float_as_uint(r);
      // a NaN stays one when its low bits go
      p[0][e] = fin_only && !fin ? 0u : (!fin && (u & 0x007fffffu) ? u | 0x00400000u : u);
      p[1][e] = ur;
      p[2][e] = __float_as_uint(r - __uint_as_float(ur & 0xffff0000u));
    }
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j) o[q][j] = __builtin_amdgcn_perm(p[q][2 * j + 1], p[q][2 * j], 0x07060302u);
  }
}

// Eight MXFP8 weights under the scale byte 1 or 2: rounded to bf16, but never to
// zero (Inf times a weight that is not zero is no NaN), or (left) 2^64 times
// what that leaves, at most three steps of 2^-135: exact.
__device__ __forceinline__ bf16x8 wq_tiny8(uint32_t w0, uint32_t w1, uint32_t e, bool left) {
  const float s = e8m0_to_f32(e);
  float o[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float v = fp8_e4m3_to_f32(((j < 4 ? w0 : w1) >> (8 * (j & 3))) & 0xFFu) * s;
    uint32_t h = f32_to_bf16_bits(v);
    if (!(h & 0x7FFFu) && v != 0.f) h |= 1u;
    o[j] = left ? (v - bf16_bits_to_f32(h)) * 0x1p64f : bf16_bits_to_f32(h);
  }
  return pack_bf16x8(o);
}

// WM x WN waves, each RT x CT tiles of 32 x 32; NSP activation parts.
template <int FMT, bool G16, int WM, int WN, int RT, int CT, int NSP>
__global__ __launch_bounds__(512, 2) void wq_tile_kernel(const WqP p) {
  using Tr = WqTraits<FMT>;
  constexpr int BM = 32 * WM * RT, BN = 32 * WN * CT;
  constexpr int A_PART = BM * 128, A_BYTES = NSP * A_PART, BUF = A_BYTES + BN * 128;
  constexpr int XP = BM * 8 / 512;             // activation pieces (8 floats) per thread and chunk
  constexpr int WPT = BN * WT_KC / 512;        // weights per thread and chunk, consecutive k
  constexpr int WW = WPT / Tr::KDIV / 4;       // ... in 32-bit words
  constexpr int TPR = WT_KC / WPT;             // threads per weight row
  constexpr int NSC = Tr::MX ? (WPT > (G16 ? 16 : 32) ? 2 : 1) : 0;
  constexpr bool TINY = FMT == WQ_MXFP8 && NSP == 3;
  static_assert(WM * WN == 8 && XP >= 1 && (WPT == 16 || WPT == 32) && 2 * BUF <= 160 * 1024, "tile shape");
  __shared__ __align__(16) char smem[2 * BUF];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int c32 = lane & 31, h = lane >> 5;
  // the row tiles of a column block are neighbours on one XCD (shared weights)
  const int mtiles = (int)cdiv(p.M, BM);
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int64_t m0 = (int64_t)(id % mtiles) * BM, n0 = (int64_t)(id / mtiles) * BN;
  const int64_t K = p.K;
  const int nch = (int)(K / WT_KC);

  // ---- global side: rows past M and columns past N repeat the last one ----
  const float* xp[XP];
  uint32_t xd[XP];
#pragma unroll
  for (int i = 0; i < XP; ++i) {
    const int q = tid + 512 * i, row = q >> 3, piece = q & 7;
    xp[i] = p.x + imin64(m0 + row, p.M - 1) * K + 8 * piece;
    xd[i] = (uint32_t)(row * 128 + ((piece ^ ((row >> 1) & 7)) * 16));
  }
  const int wrow = tid / TPR, wk = (tid % TPR) * WPT;
  const int64_t wn_row = imin64(n0 + wrow, p.N - 1);
  const uint8_t* wp = p.w + wn_row * (K / Tr::KDIV) + wk / Tr::KDIV;
  const bool has_sc = Tr::MX && p.scale != nullptr;
  constexpr int G = G16 ? 16 : 32;
  const uint8_t* sp = has_sc ? reinterpret_cast<const uint8_t*>(p.scale) + wn_row * (K / G) + wk / G : nullptr;

  float4 xr[XP][2];
  uint32_t wr[WW], sr[NSC > 0 ? NSC : 1];
  auto load = [&](int c) {
#pragma unroll
    for (int i = 0; i < XP; ++i) {
      xr[i][0] = *reinterpret_cast<const float4*>(xp[i] + (int64_t)c * WT_KC);
      xr[i][1] = *reinterpret_cast<const float4*>(xp[i] + (int64_t)c * WT_KC + 4);
    }
    const uint8_t* w = wp + (int64_t)c * (WT_KC / Tr::KDIV);
    if constexpr (WW % 4 == 0) {
#pragma unroll
      for (int j = 0; j < WW / 4; ++j) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(w + 16 * j);
#pragma unroll
        for (int e = 0; e < 4; ++e) wr[4 * j + e] = v[e];
      }
    } else {
      const u32x2 v = *reinterpret_cast<const u32x2*>(w);
      wr[0] = v[0];
      wr[1] = v[1];
    }
    if constexpr (NSC > 0) {
#pragma unroll
      for (int j = 0; j < NSC; ++j) sr[j] = has_sc ? sp[(int64_t)c * (WT_KC / G) + j] : 127u;
    }
  };
  bool tiny = false;  // a scale byte 1 or 2 in this thread's weights
  auto store = [&](int buf, auto exact_c, bool left) {
    constexpr bool EXACT = decltype(exact_c)::value;
    char* S = smem + buf * BUF;
#pragma unroll
    for (int i = 0; i < XP; ++i) {
      const float v[8] = {xr[i][0].x, xr[i][0].y, xr[i][0].z, xr[i][0].w, xr[i][1].x, xr[i][1].y, xr[i][1].z, xr[i][1].w};
      u32x4 o[NSP];
      split8<NSP>(v, o, EXACT && left);
#pragma unroll
      for (int q = 0; q < NSP; ++q) *reinterpret_cast<u32x4*>(S + q * A_PART + xd[i]) = o[q];
    }
#pragma unroll
    for (int j = 0; j < WPT / 8; ++j) {
      bf16x8 b;
      const uint32_t e = Tr::MX ? sr[NSC == 2 ? j * 8 / G : 0] & 255u : 0u;
      if constexpr (FMT == WQ_MXFP4)
        b = mx4_word_bf16(wr[j], mx4_lut(e));
      else
        b = wq_decode8<FMT>(wr[2 * j], wr[2 * j + 1], Tr::MX ? e8m0_to_f32(e) : 1.f);
      if constexpr (EXACT) {
        if (e - 1u < 2u)
          b = wq_tiny8(wr[2 * j], wr[2 * j + 1], e, left);
        else if (left)
          b = bf16x8{};
      } else if constexpr (TINY) {
        tiny |= e - 1u < 2u;
      }
      const int piece = wk / 8 + j;
      *reinterpret_cast<bf16x8*>(S + A_BYTES + wrow * 128 + ((piece ^ ((wrow >> 1) & 7)) * 16)) = b;
    }
  };

  // acc: sums of whole 128-k spans; t: the span's products; small (three
  // parts): the products of mid and lo, whose roundings are 2^-8 of the others
  f32x16 acc[RT][CT], t[RT][CT], small[NSP == 3 ? RT : 1][NSP == 3 ? CT : 1];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      acc[r][c] = f32x16{};
      t[r][c] = f32x16{};
      if constexpr (NSP == 3) small[r][c] = f32x16{};
    }
  auto fold = [&](f32x16 (&a)[RT][CT], f32x16 (&v)[RT][CT], float f) {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < CT; ++c) {
#pragma unroll
        for (int i = 0; i < 16; ++i) a[r][c][i] += v[r][c][i] * f;
        v[r][c] = f32x16{};
      }
  };
  // operand piece 2s + h of row c32 of a tile (tiles start at multiples of 32
  // rows, which leave (row >> 1) & 7 as it is)
  auto frag = [&](const char* base, int row0, int s) {
    return *reinterpret_cast<const bf16x8*>(base + (row0 + c32) * 128 + (((2 * s + h) ^ ((c32 >> 1) & 7)) * 16));
  };
  auto multiply = [&](int buf) {
    const char* S = smem + buf * BUF;
#pragma unroll
    for (int s = 0; s < WT_KC / 16; ++s) {
      bf16x8 b[CT];
#pragma unroll
      for (int c = 0; c < CT; ++c) b[c] = frag(S + A_BYTES, 32 * (wn * CT + c), s);
#pragma unroll
      for (int q = 0; q < NSP; ++q)
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          const bf16x8 a = frag(S + q * A_PART, 32 * (wm * RT + r), s);
#pragma unroll
          for (int c = 0; c < CT; ++c) {
            if constexpr (NSP == 3) {
              if (q > 0) {
                small[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[c], small[r][c], 0, 0, 0);
                continue;
              }
            }
            t[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[c], t[r][c], 0, 0, 0);
          }
        }
    }
  };

  auto chunks = [&](auto exact_c, bool left, auto&& span_done) {
    load(0);
    store(0, exact_c, left);
    lds_barrier();
    for (int c = 0; c < nch; ++c) {
      if (c + 1 < nch) load(c + 1);
      multiply(c & 1);
      if ((c & 1) || c + 1 == nch) span_done();
      if (c + 1 < nch) store((c + 1) & 1, exact_c, left);  // last read in chunk c - 1, before the last barrier
      lds_barrier();
    }
  };
  chunks(std::false_type{}, false, [&] { fold(acc, t, 1.f); });

  if constexpr (NSP == 3) fold(acc, small, 1.f);
  if constexpr (TINY) {
    if (__syncthreads_or(tiny)) {
      for (int left = 0; left < 2; ++left) {
        if (!left) {
#pragma unroll
          for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int c = 0; c < CT; ++c) acc[r][c] = f32x16{};
        }
        chunks(std::true_type{}, left, [&] { fold(left ? small : acc, t, 1.f); });
        fold(acc, small, left ? 0x1p-64f : 1.f);
      }
    }
  }

  // register i of a tile: row 8 (i / 4) + 4 h + i % 4, column c32
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const int64_t n = n0 + 32 * (wn * CT + c) + c32;
    if (n >= p.N) continue;
    float f = 1.f;
    if constexpr (FMT == WQ_FP8_ROW || FMT == WQ_INT8_ROW) f = reinterpret_cast<const float*>(p.scale)[n];
    if constexpr (FMT == WQ_MXFP4) f = p.s2;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int64_t m = m0 + 32 * (wm * RT + r) + 8 * (i >> 2) + 4 * h + (i & 3);
        if (m < p.M) p.y[m * p.N + n] = FMT == WQ_MXFP8 ? acc[r][c][i] : acc[r][c][i] * f;
      }
  }
}

template <int FMT, bool G16>
void launch_tile(const WqP& p, int bm, int bn, hipStream_t st) {
  const dim3 grid((unsigned)(cdiv(p.M, bm) * cdiv(p.N, bn))), block(512);
  if (p.K % 256 == 0) {
    if (bn == 256)
      launch((wq_tile_kernel<FMT, G16, 2, 4, 2, 2, 2>), grid, block, 0, st, p);
    else if (bm == 128)
      launch((wq_tile_kernel<FMT, G16, 4, 2, 1, 2, 2>), grid, block, 0, st, p);
    else
      launch((wq_tile_kernel<FMT, G16, 2, 4, 1, 1, 2>), grid, block, 0, st, p);
  } else {
    if (bm == 128)
      launch((wq_tile_kernel<FMT, G16, 4, 2, 1, 2, 3>), grid, block, 0, st, p);
    else
      launch((wq_tile_kernel<FMT, G16, 2, 4, 1, 1, 3>), grid, block, 0, st, p);
  }
}

}  // namespace

bool wq_tile_route(int fmt, int64_t M, int64_t K, int64_t N, int& bm, int& bn) {
  if (K % WT_KC != 0) return false;
  if (K % 256 == 0) {
    // the 64-row kernel is as fast while its 64 x 64 blocks are one round of
    // the CUs (fp8 M=512 K=N=2048 26 us against 28; MXFP4 25 against 33); past
    // that fp8 K=4096 N=14336 M=65 79 -> 47 us, M=128 97 -> 49, M=512 332 -> 129
    if (M <= 64 || cdiv(M, 64) * cdiv(N, 64) <= 256) return false;
  } else {
    // a workgroup takes about 1 us per chunk however few there are, the
    // streaming kernels a time in proportion to M N (K=2176 N=4001 M=33: int8
    // 36.6 us against 37.6, MXFP4 62 against 44; K=4224 N=14336: int8 M=10 52
    // against 68, M=16 79 against 68, M=64 310 -> 70, M=512 2506 -> 241), and
    // with a longer K they do better (M=48 N=4096, M N = 3 << 16: int8 K=1600 33.3
    // -> 32.0, K=6208 90 against 113; M=32 N=4096, 1 << 17: MXFP8 K=1088 26.0 ->
    // 21.9, K=2176 35.4 against 40.6, K=4224 55.6 against 76.0)
    int64_t least = 3 << 16;  // M N from which the tiles are faster
    if (fmt == WQ_MXFP4) {
      least = 1 << 17;
    } else if (fmt == WQ_MXFP8) {
      least = K <= 1344 ? 1 << 17 : (K <= 2432 ? 9 << 14 : (3 << 16) + 1);
    } else if (K >= 2048) {
      least = fmt == WQ_INT8_ROW && K >= 4096 ? 7 << 15 : (3 << 16) + 1;
    }
    if (M <= 12 || M * N < least) return false;
  }
  // the largest tile that still gives most CUs one
  bm = 128;
  bn = K % 256 == 0 ? 256 : 128;
  if (cdiv(M, bm) * cdiv(N, bn) < 160) bn = 128;
  if (cdiv(M, bm) * cdiv(N, bn) < 160) bm = 64;
  return cdiv(M, bm) * cdiv(N, bn) <= 0x7fffffff;
}

int wq_tile_linear(int fmt, const WqP& p, bool g16, hipStream_t st, const char* name) {
  int bm, bn;
  if (!wq_tile_route(fmt, p.M, p.K, p.N, bm, bn)) return -1;
  switch (fmt) {
    case WQ_FP8_ROW: launch_tile<WQ_FP8_ROW, false>(p, bm, bn, st); break;
    case WQ_INT8_ROW: launch_tile<WQ_INT8_ROW, false>(p, bm, bn, st); break;
    case WQ_MXFP8:
      if (g16)
        launch_tile<WQ_MXFP8, true>(p, bm, bn, st);
      else
        launch_tile<WQ_MXFP8, false>(p, bm, bn, st);
      break;
    default:
      if (g16)
        launch_tile<WQ_MXFP4, true>(p, bm, bn, st);
      else
        launch_tile<WQ_MXFP4, false>(p, bm, bn, st);
      break;
  }
  return launch_status(name);
}

}  // namespace ccq

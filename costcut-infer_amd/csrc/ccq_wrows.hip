// Decoded-weight MFMA linear for up to 16 rows: y[M, N] = x[M, K] @ W[N, K]^T in
// float32 on byte-coded weights (formats and arithmetic: ccq_wmfma.hip).
//
// At these sizes the weights are the traffic, and the chunk loop of the 64-row
// kernel (stage, barrier, multiply) is bound by that sequence, not by bytes.
// Here nothing is shared in the loop: the 8 waves of a workgroup split K, each
// wave stages its own k-tiles of 128 (16 rows as bf16 hi and lo) in its own
// part of LDS, without a barrier, and multiplies them with 16 NB columns whose
// weights it loads two k-tiles ahead.  Activations are loaded as far ahead,
// since a wave's loads return in order.  The 8 partial sums are added in wave
// order at the end.
#include "ccq_wq.h"

namespace ccq {

namespace {

constexpr int WS_LD = 128 + 8;  // LDS row stride in bf16: rows 4 banks apart

// Lanes of one wave hand each other values through LDS: the hardware keeps a
// wave's LDS accesses in order, and the fences keep the compiler from moving
// them across (to a lane the other lanes' addresses are unrelated ones; the
// wave barrier alone only bounds the scheduling).  They emit no instruction.
__device__ __forceinline__ void lane_exchange() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int FMT, bool G16, int NB>
__global__ __launch_bounds__(512, 2) void wq_rows_kernel(const WqP p) {
  using Tr = WqTraits<FMT>;
  constexpr int NSC = Tr::MX ? (G16 ? 2 : 1) : 0;
  constexpr int G = G16 ? 16 : 32;
  __shared__ __align__(16) uint16_t xs[8][2][16][WS_LD];  // [wave][hi, lo][row][k]
  __shared__ __align__(16) f32x4 red[8][NB][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, q = lane >> 4;
  const int64_t K = p.K, N = p.N;
  const int M = (int)p.M, KT = (int)(K / 128);
  const int kt0 = KT * wave / 8, kt1 = KT * (wave + 1) / 8;

  // weights: column c16 of tile b, 32 consecutive k of quarter q (columns past
  // N repeat the last one, not stored).  Plain loads: a line of a row is read
  // in pieces by several lanes and loads, and non-temporal ones fetched it
  // more than once (fp8 M=16 K=4096 N=14336 on 64-column blocks, weights in the
  // Infinity Cache: 25.7 us against 17.9).
  const uint8_t* wp[NB];
  const uint8_t* sp[NB];
  const bool has_sc = Tr::MX && p.scale != nullptr;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int64_t n = imin64(((int64_t)blockIdx.x * NB + b) * 16 + c16, N - 1);
    wp[b] = p.w + n * (K / Tr::KDIV) + 32 * q / Tr::KDIV;
    sp[b] = has_sc ? reinterpret_cast<const uint8_t*>(p.scale) + n * (K / G) + 32 * q / G : nullptr;
  }
  // activations: piece j of a lane is float4 lane & 31 of row 2 j + (lane >> 5)
  // (rows past M repeat the last one, not stored)
  const float* xp[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) xp[j] = p.x + (int64_t)min(2 * j + (lane >> 5), M - 1) * K + 4 * (lane & 31);

  u32x4 wr[2][NB][Tr::WB];
  uint32_t sr[2][NB][NSC > 0 ? NSC : 1];
  float4 xr[2][8];
  auto load = [&](int kt, int d) {
    kt = min(kt, kt1 - 1);  // past the range: the last k-tile again, not multiplied
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const uint8_t* w = wp[b] + (int64_t)kt * (128 / Tr::KDIV);
#pragma unroll
      for (int i = 0; i < Tr::WB; ++i) wr[d][b][i] = *reinterpret_cast<const u32x4*>(w + 16 * i);
#pragma unroll
      for (int i = 0; i < NSC; ++i) sr[d][b][i] = has_sc ? sp[b][kt * (128 / G) + i] : 127u;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) xr[d][j] = *reinterpret_cast<const float4*>(xp[j] + (int64_t)kt * 128);
  };
  f32x4 acc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto multiply = [&](int d) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float4 v = xr[d][j];
      const uint32_t h01 = bf16x2_bits(v.x, v.y), h23 = bf16x2_bits(v.z, v.w);
      const uint32_t l01 = bf16x2_bits(v.x - __uint_as_float(h01 << 16), v.y - __uint_as_float(h01 & 0xffff0000u));
      const uint32_t l23 = bf16x2_bits(v.z - __uint_as_float(h23 << 16), v.w - __uint_as_float(h23 & 0xffff0000u));
      const int row = 2 * j + (lane >> 5), k = 4 * (lane & 31);
      *reinterpret_cast<u32x2*>(&xs[wave][0][row][k]) = u32x2{h01, h23};
      *reinterpret_cast<u32x2*>(&xs[wave][1][row][k]) = u32x2{l01, l23};
    }
    lane_exchange();
    bf16x8 ah[4], al[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ah[i] = *reinterpret_cast<const bf16x8*>(&xs[wave][0][c16][32 * q + 8 * i]);
      al[i] = *reinterpret_cast<const bf16x8*>(&xs[wave][1][c16][32 * q + 8 * i]);
    }
    lane_exchange();
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        bf16x8 w;
        const uint32_t e = Tr::MX ? sr[d][b][NSC == 2 ? i >> 1 : 0] & 255u : 0u;
        if constexpr (FMT == WQ_MXFP4)
          w = mx4_word_bf16(wr[d][b][0][i], mx4_lut(e));
        else
          w = wq_decode8<FMT>(wr[d][b][i >> 1][(i & 1) * 2], wr[d][b][i >> 1][(i & 1) * 2 + 1],
                              Tr::MX ? e8m0_to_f32(e) : 1.f);
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], w, acc[b], 0, 0, 0);
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], w, acc[b], 0, 0, 0);
      }
  };

  if (kt0 < kt1) {
    load(kt0, 0);
    load(kt0 + 1, 1);
    for (int kt = kt0; kt < kt1; kt += 2) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (kt + u < kt1) multiply(u);
        load(kt + u + 2, u);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) red[wave][b][lane] = acc[b];
  __syncthreads();
  if (wave >= NB) return;
  f32x4 v = red[0][wave][lane];
#pragma unroll
  for (int w = 1; w < 8; ++w) {
    const f32x4 o = red[w][wave][lane];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += o[i];
  }
  const int64_t n = ((int64_t)blockIdx.x * NB + wave) * 16 + c16;
  if (n >= N) return;
  float f = 1.f;
  if constexpr (FMT == WQ_FP8_ROW || FMT == WQ_INT8_ROW) f = reinterpret_cast<const float*>(p.scale)[n];
  if constexpr (FMT == WQ_MXFP4) f = p.s2;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 4 * q + i;
    if (row < M) p.y[(int64_t)row * N + n] = FMT == WQ_MXFP8 ? v[i] : v[i] * f;
  }
}

template <int FMT, bool G16>
void launch_rows(const WqP& p, int nb, hipStream_t st) {
  const dim3 grid((unsigned)cdiv(p.N, 16 * nb)), block(512);
  if constexpr (FMT == WQ_MXFP4) {
    if (nb == 4) {
      launch((wq_rows_kernel<FMT, G16, 4>), grid, block, 0, st, p);
      return;
    }
  }
  if (nb == 2)
    launch((wq_rows_kernel<FMT, G16, 2>), grid, block, 0, st, p);
  else
    launch((wq_rows_kernel<FMT, G16, 1>), grid, block, 0, st, p);
}

}  // namespace

int wq_rows_route(int fmt, bool g16, int64_t M, int64_t K, int64_t N) {
  if (M > 16 || K % 256 != 0 || cdiv(N, 64) > 256) return 0;
  // the fewest columns per workgroup whose workgroups are one round of the CUs
  const int nb = cdiv(N, 16) <= 256 ? 1 : (cdiv(N, 32) <= 256 ? 2 : 4);
  // With 64 columns the 64-row kernel keeps the one-byte formats: K=4096 N=14336
  // M=16, weights from HBM (12 sets in turn), fp8 20.7 us against 22.9 and MXFP8
  // 27.0 against 28.2 (from the Infinity Cache 20.0 against 18.0 and 26.1
  // against 23.8).  MXFP4: 19.7 -> 17.5 at M=1 and 22.1 -> 19.7 at M=16, but not
  // where each wave has three k-tiles, which its loop takes in pairs (K=3072
  // M=1 15.7 against 17.1), nor with 16-element groups unless the waves have
  // two or four k-tiles each, or more than that (K=2304 M=1 13.6 against 16.8,
  // K=4352 22.3 against 24.4; K=4096 M=16 23.4 -> 22.0, K=5120 31.2 -> 28.0).
  if (nb == 4) return fmt == WQ_MXFP4 && (g16 ? K % 2048 == 0 || K >= 5120 : K >= 2048 && K != 3072) ? nb : 0;
  // A short K, where a wave has no third k-tile to load ahead.  32 columns
  // (N=8192 M=16): fp8 K=1536 8.9 against 9.5, K=2048 10.7 -> 9.6; MXFP8 K=1280 9.1
  // against 10.0, 16-element groups K=512 5.8 against 7.1; MXFP4 K=256 3.9 against
  // 4.2, K=512 5.1 -> 4.9, 16-element groups K=512 5.8 against 6.4, K=768 7.1 ->
  // 7.0.  16 columns: the MX formats with K=256 (16-element groups, M=1 N=33 2.8
  // against 3.5).
  const int64_t shortest = fmt < WQ_MXFP8 ? (nb == 2 ? 2048 : 256)
                           : nb == 1      ? 512
                           : fmt == WQ_MXFP8 ? 1536
                                             : (g16 ? 768 : 512);
  if (K < shortest) return 0;
  return nb;
}

int wq_rows_linear(int fmt, const WqP& p, bool g16, hipStream_t st, const char* name) {
  const int nb = wq_rows_route(fmt, g16, p.M, p.K, p.N);
  if (nb == 0) return -1;
  switch (fmt) {
    case WQ_FP8_ROW: launch_rows<WQ_FP8_ROW, false>(p, nb, st); break;
    case WQ_INT8_ROW: launch_rows<WQ_INT8_ROW, false>(p, nb, st); break;
    case WQ_MXFP8:
      if (g16)
        launch_rows<WQ_MXFP8, true>(p, nb, st);
      else
        launch_rows<WQ_MXFP8, false>(p, nb, st);
      break;
    default:
      if (g16)
        launch_rows<WQ_MXFP4, true>(p, nb, st);
      else
        launch_rows<WQ_MXFP4, false>(p, nb, st);
      break;
  }
  return launch_status(name);
}

}  // namespace ccq

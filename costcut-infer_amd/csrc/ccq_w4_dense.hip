// AWQ int4 dense GEMM above the decode kernel's 16 rows: y[M, N] = x[M, K] @ W
// (weight and scale/zero layouts: ccq_w4.hip).
//
// w4_slab_kernel, 17 to 64 rows a workgroup.  Everything the loop reads goes from HBM
// straight into an LDS ring (global_load_lds): activations (pieces of 16 bytes
// XOR-swizzled by row), packed weight tiles and scale/zero words.  8 waves =
// CG column groups x KS k-tiles of a step; a wave multiplies all 16 MT rows by
// its 16 NB columns of its k-tile, and the KS partial sums are added through
// LDS at the end.  Each wave issues the same copies per step, so the waits are
// fixed counts on its in-order vmcnt, and one barrier per step publishes a
// stage and frees the one before.
//
// Dequantization: the identity of ccq_w4.hip.  Sx of a k-tile is needed by
// every column group, so the CG waves each compute a share of its row tiles
// (MFMAs against ones) and exchange them through LDS; the fold of a step's
// products waits for the next step's barrier.
//
// What bounds it (M=48 K=4096 N=14336, parts taken out of timing copies): the
// LDS reads of the activations, once per column group (all copies from one
// hot line and no products: 13 of 22 us), so 32 columns per wave and 4 k-tiles
// per step where the ring still holds two stages (M=37: 21.8 -> 19.6 us
// against 16 columns and 2 k-tiles), and the products (5 us).  Activations
// read straight from L2 by each wave (K split over the waves, no ring) took
// as long, their loads waiting behind the weights' in the wave's vmcnt.
#include "ccq_w4_mfma.h"

#include <type_traits>

namespace ccq {

namespace {

constexpr int WL_LDS = 158 * 1024;  // of a CU's 160 KiB

struct W4SlabP {
  const void* x;
  const uint32_t* w;
  const uint32_t* sz;
  void* y;        // output, or null: float32 partials to part
  float* part;    // [splits][M][N]
  int y_dtype, s_bf16;
  int M, N, K, KT, szw;
  int row_blocks, col_blocks, splits;
};

__device__ __forceinline__ float sz_scale_rt(uint32_t word, int bf16) {
  const float h = f16_bits_to_f32(word & 0xFFFFu), b = __uint_as_float(word << 16);
  return bf16 ? b : h;
}

// LDS plan of one instance.  Scale/zero words come in pieces of 16 bytes (4
// words of a column): one slot holds a step's pieces, or those of ZS steps
// when a step needs less than one piece per column.
template <int MT, int NB, int KS, int NG>
struct Slab {
  static constexpr int CG = 8 / KS, C = 16 * CG * NB;  // columns of a workgroup
  static constexpr int A = KS * MT * 4096, B = 8 * NB * 1024, STAGE = A + B;
  static constexpr int WS = KS * NG;                    // words per column and step
  static constexpr int ZS = WS < 4 ? 4 / WS : 1;        // steps per slot
  static constexpr int ZP = WS < 4 ? 1 : WS / 4;        // pieces per column and slot
  static constexpr int ZSLOT = ZP * C * 16, ZCOPIES = (ZP * C + 63) / 64;
  static constexpr int SX = KS * NG * MT * 64;          // Sx of one step
  static constexpr int zslots(int ns) { return (ns + ZS - 1) / ZS + 1; }
  static constexpr int lds(int ns) { return ns * STAGE + zslots(ns) * ZSLOT + 2 * SX; }
  static constexpr int fit() {
    int n = 2;
    while (n < 8 && lds(n + 1) <= WL_LDS) ++n;
    return n;
  }
  static constexpr int NS = fit(), NZ = zslots(NS);
  static constexpr int Z_OFF = NS * STAGE, SX_OFF = Z_OFF + NZ * ZSLOT;
  static constexpr int CA = KS * MT * 4 / 8;            // activation copies per wave and step
  static constexpr int COPIES = CA + NB;                // besides the scale/zero copies of some waves
  static_assert(lds(NS) <= WL_LDS && ZCOPIES <= 8 && (KS * MT) % 2 == 0 && KS * (8 / KS) == 8, "slab plan");
  static_assert(KS == 1 || KS * MT * NB * CG * 1024 <= Z_OFF, "the partial sums reuse the ring");
};

// Wait until at most min(n, N) steps of COPIES copies are in flight.
template <int N, int COPIES>
__device__ __forceinline__ void wait_steps(int n) {
  if constexpr (N > 0) {
    if (n >= N)
      wait_vmcnt<N * COPIES>();
    else
      wait_steps<N - 1, COPIES>(n);
  } else {
    wait_vmcnt<0>();
  }
}

// MT 16-row tiles, NB 16-column tiles per wave, KS k-tiles per step, NG
// quantization groups per 128-row k-tile.
template <typename AT, int MT, int NB, int KS, int NG>
__global__ __launch_bounds__(512, 2) void w4_slab_kernel(const W4SlabP p) {
  using V = typename Act<AT>::vec;
  using L = Slab<MT, NB, KS, NG>;
  constexpr int CG = L::CG, JS = 4 / NG;
  __shared__ __align__(16) char smem[L::lds(L::NS)];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cg = wave % CG, kg = wave / CG;
  const int r = lane & 15, kq = lane >> 4;
  // row blocks of one column block, then the column blocks of one slab of K,
  // are neighbours on one XCD: its L2 serves their weights / activations
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int rb = id % p.row_blocks, cs = id / p.row_blocks;
  const int cb = cs % p.col_blocks, sp = cs / p.col_blocks;
  const int row0 = rb * 16 * MT, rows = min(16 * MT, p.M - row0);
  // slabs start at a multiple of 4 k-tiles (16-byte pieces of scale/zero words)
  const int kt4 = (p.KT + 3) >> 2;
  const int kt0 = 4 * (int)((int64_t)kt4 * sp / p.splits), kt1 = min(p.KT, 4 * (int)((int64_t)kt4 * (sp + 1) / p.splits));
  const int S = (kt1 - kt0 + KS - 1) / KS;  // steps
  const int nt0 = cb * (L::C / 16), ntiles = p.N / 16;

  // ---- copies of one step by this wave ----
  // activations: copy c = wave * CA + i takes rows 4 (c mod 4 MT) .. + 3 of
  // k-tile c / (4 MT); a lane's piece (lane & 15) ^ (row & 15) lands at
  // position lane & 15.  Rows past M repeat the last one (not stored), k-tiles
  // past the slab its last one (not multiplied).
  uint32_t aoff[L::CA];
#pragma unroll
  for (int i = 0; i < L::CA; ++i) {
    const int row = 4 * ((wave * L::CA + i) % (4 * MT)) + kq;
    aoff[i] = (uint32_t)(min(row, rows - 1) * p.K * 2 + (r ^ (row & 15)) * 16);
  }
  const char* xb = reinterpret_cast<const char*>(p.x) + (int64_t)row0 * p.K * 2;
  // weight tiles of the wave (past N: the last one, not stored)
  const char* bsrc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
    bsrc[b] = reinterpret_cast<const char*>(p.w + (int64_t)min(nt0 + cg * NB + b, ntiles - 1) * p.KT * 256);
  // scale/zero pieces: waves 0 .. ZCOPIES - 1 copy 64 each, piece pc of column
  // col at (pc * C + col) * 16
  const int zq = min(wave * 64 + lane, L::ZP * L::C - 1), zpc = zq / L::C;
  const uint32_t zcol = (uint32_t)((int64_t)min(nt0 * 16 + zq % L::C, p.N - 1) * p.szw * 4);
  const int zlast = p.szw / 4 - 1;  // last piece of a column
  const uint32_t lds0 = lds_addr(smem);
  auto issue = [&](int i) {
    const uint32_t st = lds0 + (i % L::NS) * L::STAGE;
    if (i % L::ZS == 0 && wave < L::ZCOPIES) {
      const int pc = min((kt0 + i * KS) * NG / 4 + zpc, zlast);
      dma16(p.sz, zcol + pc * 16, lds0 + L::Z_OFF + (i / L::ZS % L::NZ) * L::ZSLOT + wave * 1024);
    }
    const int ktw = min(kt0 + i * KS + kg, kt1 - 1);
#pragma unroll
    for (int b = 0; b < NB; ++b) dma16_nt(bsrc[b] + (int64_t)ktw * 1024, lane * 16, st + L::A + (wave * NB + b) * 1024);
#pragma unroll
    for (int c = 0; c < L::CA; ++c) {
      const int q = wave * L::CA + c, kt = min(kt0 + i * KS + q / (4 * MT), kt1 - 1);
      dma16(xb + (int64_t)kt * 256, aoff[c], st + q * 1024);
    }
  };

  // Operands of one step in registers: read one step ahead, so that no LDS
  // latency stands between a step's barrier and its MFMAs, and the slot of a
  // step is free again when that step begins.
  struct Ops {
    V a[MT][4];
    u32x4 w[NB];
    uint32_t z[NB][NG];
  };
  constexpr int TB = NG == 1 ? 2 : 1;  // product buffers (two: the fold overlaps the next step's MFMAs)
  f32x4 acc[MT][NB], t[TB][NG][MT][NB];
  uint32_t zw[2][NB][NG];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[m][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const u32x4 ones_u = {Act<AT>::kOne2, Act<AT>::kOne2, Act<AT>::kOne2, Act<AT>::kOne2};
  const V ones = __builtin_bit_cast(V, ones_u);
  uint32_t mask_s = 0x000F000Fu, magic_v = Act<AT>::kMagic2;
  asm volatile("s_mov_b32 %0, %0" : "+s"(mask_s));
  asm volatile("v_mov_b32 %0, %0" : "+v"(magic_v));

  auto read = [&](int i, Ops& o) {
    const char* st = smem + (i % L::NS) * L::STAGE;
    const char* as = st + kg * MT * 4096;
    const char* zs = smem + L::Z_OFF + (i / L::ZS % L::NZ) * L::ZSLOT;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      o.w[b] = *reinterpret_cast<const u32x4*>(st + L::A + (wave * NB + b) * 1024 + lane * 16);
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const int w = (i % L::ZS) * L::WS + kg * NG + g;
        o.z[b][g] = *reinterpret_cast<const uint32_t*>(zs + (((w >> 2) * L::C + (cg * NB + b) * 16 + r) * 4 + (w & 3)) * 4);
      }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        o.a[m][j] = *reinterpret_cast<const V*>(as + (16 * m + r) * 256 + (((4 * j + kq) ^ r) * 16));
  };
  // Sx of k-tile kg, group g, row tile m of step i: 4 rows per lane quarter
  auto sx_at = [&](int i, int g, int m) {
    return reinterpret_cast<f32x4*>(smem + L::SX_OFF + (i & 1) * L::SX + (((kg * NG + g) * MT + m) * 4 + kq) * 16);
  };
  auto fold = [&](int i, const uint32_t (&z)[NB][NG], const f32x4 (&tt)[NG][MT][NB]) {
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const f32x4 sx = *sx_at(i, g, m);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const float s = sz_scale_rt(z[b][g], p.s_bf16), c = Act<AT>::kMagic + (float)(z[b][g] >> 16);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[m][b][e] = fmaf(s, fmaf(-c, sx[e], tt[g][m][b][e]), acc[m][b][e]);
        }
      }
  };
  auto multiply = [&](int i, const Ops& o, f32x4 (&tt)[NG][MT][NB]) {
    // this wave's share of the k-tile's Sx
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if (m % CG != cg) continue;
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        f32x4 sx = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < JS; ++j) sx = mfma16(o.a[m][g * JS + j], ones, sx);
        if (r == 0) *sx_at(i, g, m) = sx;
      }
    }
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int j = 0; j < JS; ++j)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const V bf = dq_b3<AT>(o.w[b][g * JS + j], mask_s, magic_v);
#pragma unroll
          for (int m = 0; m < MT; ++m)
            tt[g][m][b] = mfma16(o.a[m][g * JS + j], bf, j == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : tt[g][m][b]);
        }
  };

  Ops ops[2];
  const int pre = S < L::NS ? S : L::NS;
  for (int i = 0; i < pre; ++i) issue(i);
  wait_steps<L::NS - 1, L::COPIES>(S - 1);
  lds_barrier();
  read(0, ops[0]);
  bool live = false;  // the step before multiplied
  auto step = [&](int i, auto u_c) {
    constexpr int u = decltype(u_c)::value;
    wait_steps<L::NS - 2, L::COPIES>(S - 2 - i);  // the steps after i + 1 may stay in flight
    lds_barrier();
    if (i + L::NS < S) issue(i + L::NS);  // into the slot of step i
    if (i + 1 < S) read(i + 1, ops[u ^ 1]);
    const bool now = kt0 + i * KS + kg < kt1;
    if constexpr (TB == 1) {
      if (live) fold(i - 1, zw[u ^ 1], t[0]);
    }
    if (now) multiply(i, ops[u], t[TB == 1 ? 0 : u]);
    if constexpr (TB == 2) {
      if (live) fold(i - 1, zw[u ^ 1], t[u ^ 1]);
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int g = 0; g < NG; ++g) zw[u][b][g] = ops[u].z[b][g];
    live = now;
  };
  for (int i = 0; i < S; i += 2) {
    step(i, std::integral_constant<int, 0>{});
    if (i + 1 < S) step(i + 1, std::integral_constant<int, 1>{});
  }
  lds_barrier();
  if (live) {
    if ((S - 1) & 1)
      fold(S - 1, zw[1], t[TB - 1]);
    else
      fold(S - 1, zw[0], t[0]);
  }

  // the KS partial sums in k order, each wave a share of the tiles
  if constexpr (KS > 1) {
    f32x4* red = reinterpret_cast<f32x4*>(smem);
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int b = 0; b < NB; ++b) red[((kg * CG + cg) * MT * NB + m * NB + b) * 64 + lane] = acc[m][b];
    lds_barrier();
  }
  // register e of tile (m, b): row 16 m + 4 kq + e, column r of the tile
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      f32x4 v = acc[m][b];
      if constexpr (KS > 1) {
        if ((m * NB + b) % KS != kg) continue;
        const f32x4* red = reinterpret_cast<const f32x4*>(smem) + (cg * MT * NB + m * NB + b) * 64 + lane;
        v = red[0];
#pragma unroll
        for (int k = 1; k < KS; ++k) {
          const f32x4 o = red[k * CG * MT * NB * 64];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += o[e];
        }
      }
      const int nt = nt0 + cg * NB + b;
      if (nt >= ntiles) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 16 * m + 4 * kq + e;
        if (row >= rows) continue;
        const int64_t o = (int64_t)(row0 + row) * p.N + nt * 16 + r;
        if (p.y != nullptr)
          store_val(p.y, o, v[e], p.y_dtype);
        else
          p.part[(int64_t)sp * p.M * p.N + o] = v[e];
      }
    }
}

// y = sum of the splits' partials, in split order; 4 values per thread.
__global__ __launch_bounds__(256) void w4_split_sum_kernel(const float* __restrict__ part, void* __restrict__ y,
                                                           int y_dtype, int splits, int64_t n4) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  f32x4 v = reinterpret_cast<const f32x4*>(part)[i];
#pragma unroll 4
  for (int s = 1; s < splits; ++s) {
    const f32x4 o = reinterpret_cast<const f32x4*>(part)[s * n4 + i];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += o[e];
  }
  if (y_dtype == CCQ_F32)
    reinterpret_cast<f32x4*>(y)[i] = v;
  else if (y_dtype == CCQ_BF16)
    reinterpret_cast<u32x2*>(y)[i] = u32x2{f32_to_bf16_bits(v[0]) | (f32_to_bf16_bits(v[1]) << 16),
                                           f32_to_bf16_bits(v[2]) | (f32_to_bf16_bits(v[3]) << 16)};
  else
    reinterpret_cast<u32x2*>(y)[i] = u32x2{f32_to_f16_bits(v[0]) | (f32_to_f16_bits(v[1]) << 16),
                                           f32_to_f16_bits(v[2]) | (f32_to_f16_bits(v[3]) << 16)};
}

template <typename AT, int MT, int NB, int KS>
void launch_slab_ng(const W4SlabP& p, int ng, dim3 grid, hipStream_t st) {
  const dim3 block(512);
  if (ng == 1)
    launch((w4_slab_kernel<AT, MT, NB, KS, 1>), grid, block, 0, st, p);
  else if (ng == 2)
    launch((w4_slab_kernel<AT, MT, NB, KS, 2>), grid, block, 0, st, p);
  else
    launch((w4_slab_kernel<AT, MT, MT == 3 ? 1 : NB, MT == 3 ? 2 : KS, 4>), grid, block, 0, st, p);  // 48 x 32: spills
}

template <typename AT>
void launch_slab_mt(const W4SlabP& p, int mt, int ng, dim3 grid, hipStream_t st) {
  switch (mt) {
    case 2: launch_slab_ng<AT, 2, 2, 4>(p, ng, grid, st); break;
    case 3: launch_slab_ng<AT, 3, 2, 4>(p, ng, grid, st); break;
    default: launch_slab_ng<AT, 4, 1, 2>(p, ng, grid, st); break;
  }
}

// Rows per workgroup (in 16-row tiles) and K splits.
struct SlabPlan {
  int mt, row_blocks, col_blocks, splits;
};

SlabPlan plan_slab(int64_t M, int64_t K, int64_t N) {
  SlabPlan pl;
  const int64_t mt_all = cdiv(M, 16), KT = K / 128;
  pl.row_blocks = (int)cdiv(mt_all, 4);
  const int mt = (int)cdiv(mt_all, pl.row_blocks);
  pl.mt = mt <= 2 ? 2 : mt;
  pl.col_blocks = (int)cdiv(N, 64);
  const int64_t blocks = (int64_t)pl.row_blocks * pl.col_blocks;
  int64_t s = 256 / blocks;
  if (s > KT / 16) s = KT / 16;
  pl.splits = (int)(s < 1 ? 1 : s);
  return pl;
}

}  // namespace

// The 16-row kernel (w4_skinny_kernel) reads the weights again per 16 rows in
// workgroups of up to 8 waves on 64 (G = 32: 32) columns.  While all of those
// fit the 256 CUs at once (8 waves each) it is as fast or faster (M=64 K=4096
// N=4096 11.5 us against 15.6, K=2048 N=8192 10.5 against 14.0); past that it
// takes a second round and this kernel wins (M=33 K=4096 N=6144 17.9 against
// 12.9, M=17 N=14336 22.5 against 13.9, M=37 34.3 against 17.6, M=64 46.7
// against 24.1; G=32 M=64 67 against 32).
//
// Above 64 rows it takes, 64 rows at a time, what the 128-row grouped kernel
// does not (group 32 or 64, N not a multiple of 128): G=64 K=4096 N=14336
// M=128 86.9 -> 49.1 us, M=2048 1267 -> 671; G=32 M=2048 1963 -> 868.
// Of the grouped kernel's shapes it takes those of one round of its blocks
// (M=128 K=4096 N=4096 22.6 us of the 16-row kernel -> 16.4, M=130 K=7168
// N=2432 34.5 -> 18.4; two rounds: M=65 K=2048 N=9216 15.1 against 20.2).
//
// What the count of waves does not see, shapes where the 16-row kernel stays
// (us of it against this kernel; N % 32 != 0 is left out of most, its
// workgroups are narrower and slower there):
//  * a second round of 64 x 64 blocks that is nearly empty: up to 12 k-tiles for
//    groups 32 and 64 (G=32 M=128 K=1536 N=8256 26.9 against 28.4, M=96 21.7
//    against 23.5) and for up to 64 rows (G=128 M=64 K=1024 N=18432 15.2
//    against 16.8), and for 65 to 80 rows, which are 48-row blocks, also past
//    those (G=128 M=65 K=2048 N=8224 17.9 against 20.0, G=64 K=1664 16.7 against
//    21.4);
//  * groups 32 and 64 of one or two k-tiles (G=64 M=2048 K=256 N=4096 28.9 against
//    36.4; G=32 only for few rows, M=65 N=14336 7.9 against 10.0);
//  * group 64 with K of 768 and 1024, where two waves of the 16-row kernel share a
//    workgroup's columns and N % 128 == 0 keeps them on one XCD (M=2048 K=1024
//    N=4096 64.2 against 69.1; K=512, 896 and 1536 are this kernel's);
//  * groups 32 and 64 on few blocks whose K is not split (under 32 k-tiles) or
//    just split in two: one CU per block against up to three workgroups on each
//    (G=32 M=128 K=3072 N=2048 15.7 against 24.9, M=64 N=4096 16.0 against 25.0,
//    768 workgroups M=768 N=512 22.6 against 25.0, but M=121 K=2176 N=4096 23.6 ->
//    20.0; 48-row blocks take less, M=139 K=2816 N=2112 22.3 -> 19.1; G=64 M=512
//    K=3072 N=1024 18.7 against 20.1).
static bool w4_skinny_stays(int64_t M, int64_t K, int64_t N, int64_t G) {
  const int64_t KT = K / 128, blocks = cdiv(M, 64) * cdiv(N, 64);
  const bool wide = N % 32 == 0, second = blocks > 256 && blocks <= 320;
  if (wide && second && M > 64 && M <= 80 && (G == 64 || KT <= 16)) return true;
  if (wide && second && M > 32 && KT >= 6 && KT <= 12 && (G < 128 || M <= 64)) return true;
  if (G == 128) return false;
  if (wide && KT <= 2 && (G == 64 || M <= 80)) return true;
  if (G == 64) return N % 128 == 0 && (KT == 6 || KT == 8 || (blocks <= 128 && KT < 32 && M > 128));
  const int64_t wgs = cdiv(M, 16) * cdiv(N, 32), mt = cdiv(cdiv(M, 16), cdiv(M, 64));
  const int64_t most = KT <= 16 ? 18432 / KT : (KT < 28 ? 768 : (KT < 32 ? 680 : 512));  // workgroups of its rounds
  return blocks <= 128 && KT <= 32 && M > 32 && wgs <= (mt == 3 ? most * 7 / 10 : most);
}

bool w4_slab_takes(int64_t M, int64_t K, int64_t N, int64_t G) {
  const int64_t blocks = cdiv(M, 64) * cdiv(N, 64);
  return M > 16 && w4_skinny_waves(M, K, N, G) > 256 * 8 && (!w4_grouped_shape(M, K, N, G) || blocks <= 256) &&
         !w4_skinny_stays(M, K, N, G) &&
         64 * K * 2 < (1LL << 32) && N * sz_words_per_column(K, G) * 4 < (1LL << 32) && blocks <= 0x7fffffff;
}

size_t w4_slab_workspace(int64_t M, int64_t K, int64_t N) {
  const SlabPlan pl = plan_slab(M, K, N);
  return pl.splits > 1 ? (size_t)pl.splits * (size_t)M * (size_t)N * 4 : 0;
}

int launch_w4_slab(const W4DenseP& d, void* workspace, size_t workspace_bytes, hipStream_t st) {
  SlabPlan pl = plan_slab(d.M, d.K, d.N);
  // without the workspace (or with an output that takes no 16-byte stores) one
  // workgroup takes all of K
  if (workspace == nullptr || workspace_bytes < w4_slab_workspace(d.M, d.K, d.N) || !aligned(workspace, 16) ||
      !aligned(d.y, 16))
    pl.splits = 1;
  W4SlabP p = {};
  p.x = d.x;
  p.w = d.w;
  p.sz = d.sz;
  p.y = pl.splits > 1 ? nullptr : d.y;
  p.part = (float*)workspace;
  p.y_dtype = d.y_dtype;
  p.s_bf16 = d.s_bf16;
  p.M = (int)d.M;
  p.N = (int)d.N;
  p.K = (int)d.K;
  p.KT = (int)(d.K / 128);
  p.szw = (int)sz_words_per_column(d.K, d.G);
  p.row_blocks = pl.row_blocks;
  p.col_blocks = pl.col_blocks;
  p.splits = pl.splits;
  const dim3 grid((unsigned)((int64_t)pl.row_blocks * pl.col_blocks * pl.splits));
  const int ng = (int)(128 / d.G);
  if (d.x_bf16)
    launch_slab_mt<__bf16>(p, pl.mt, ng, grid, st);
  else
    launch_slab_mt<_Float16>(p, pl.mt, ng, grid, st);
  int rc = launch_status("w4 slab gemm");
  if (rc || pl.splits == 1) return rc;
  return launch_w4_split_sum((const float*)workspace, d.y, d.y_dtype, pl.splits, d.M * d.N, st);
}

int launch_w4_split_sum(const float* part, void* y, int y_dtype, int splits, int64_t n, hipStream_t st) {
  launch(w4_split_sum_kernel, dim3((unsigned)cdiv(n / 4, 256)), dim3(256), 0, st, part, y, y_dtype, splits, n / 4);
  return launch_status("w4 split sum");
}

}  // namespace ccq

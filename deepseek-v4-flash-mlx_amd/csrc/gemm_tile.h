// The K loop of the tiled bf16 product (gemm.hip): one workgroup's BM x BN tile of x . w^T, both
// operands K-contiguous, accumulated in fp32 by v_mfma_f32_32x32x16_bf16.
//
// Operands go HBM -> LDS by global_load_lds_dwordx4 into a ring of D stages of 64 k.  A copy
// instruction lands 64 x 16 bytes contiguously (8 rows of 128 bytes), so rows cannot be padded:
// chunk c of row r is stored in slot c ^ ((r / 2) mod 8), which keeps the fragment reads of 16
// consecutive rows in distinct banks (no conflicts counted).
//
// What bounds it is issue: a wave's MFMAs, fragment reads and copies share one in-order stream, so
// whatever is issued in a burst leaves the matrix core idle.  The fragments of the next 16 k are
// therefore read while the current ones are multiplied (two register sets), one read per MFMA; a
// step's copies are spread over two sub-steps, one every second MFMA; and the one barrier of a step
// stands before its last 16 k, whose fragments are in registers by then, so that the stage is free
// for the copies of step s + D.  sched_barrier pins that order.  [4096, 8192] x [4096, 8192]^T,
// 256 x 256 tiles of 8 waves: 1.39 PFLOP/s, against 1.13 for a loop that reads each sub-step's
// fragments right before its MFMAs and issues all copies behind the barrier (and 1.27 with the
// reads ahead but the copies in one burst).
#pragma once

#include "attn_common.h"
#include "smla_internal.h"

namespace smla_gemm {

using smla_attn::lds_barrier;
using smla_attn::lds_u32x4_t;
using smla_attn::lds_u8_t;
using smla_attn::wait_vm;

constexpr int kRow = 128;  // bytes of one tile row per K step (64 bf16)

template <int V>
struct Int {
  static constexpr int value = V;
};

// 16-byte HBM -> LDS copy for every lane (lane l lands at lds_dst + 16 l): 32-bit lane offsets from
// a wave-uniform base, so a K step advances scalars only
__device__ inline void dma16_s(const uint8_t* base, uint32_t off, uint32_t lds_dst) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_dst), "v"(off), "s"(base) : "memory", "m0");
}

// BM tokens x BN outputs by waves of WM x WN; D stages of 64 k in LDS
template <int BM, int BN, int WM, int WN, int D>
struct Tile {
  static constexpr int NW = (BM / WM) * (BN / WN);
  static constexpr int MB = WM / 32, NB = WN / 32;
  static constexpr int STAGE = (BM + BN) * kRow;
  static constexpr int CP = STAGE / 1024 / NW;  // 1 KB copies per wave per stage
  static constexpr int LDS = D * STAGE;
  static_assert(CP * NW * 1024 == STAGE, "whole copies per wave");
};

// acc[mb][nb] = rows 0 .. BM-1 of x (from xk, row stride ldx bytes; rows past tmax read row tmax)
// times rows 0 .. BN-1 of w (likewise), over nk >= D steps of 64 k.  Accumulator register r of block
// (mb, nb) is row WM wm + 32 mb + 8 (r / 4) + 4 (lane / 32) + r mod 4 of x, row WN wn + 32 nb +
// lane mod 32 of w, for wave wm + (BM / WM) wn.  BM ldx and BN ldw fit 31 bits.
// An output is one chain of fp32 accumulations over k = 0, 16, 32 .., whichever tile it is in: a token's sums
// do not depend on where it stands in the prompt.  landed(step, stage, Int<first>): run
// after a step's stage has landed and before it is read.
template <int BM, int BN, int WM, int WN, int D, class F>
__device__ __attribute__((always_inline)) inline void tile_loop(lds_u8_t* lds, const uint8_t* __restrict__ xk,
                                                                int64_t ldx, int tmax, const uint8_t* __restrict__ wk,
                                                                int64_t ldw, int nmax, int nk,
                                                                f32x16_t (&acc)[WM / 32][WN / 32], F&& landed) {
  using L = Tile<BM, BN, WM, WN, D>;
  constexpr int NM = L::MB * L::NB, NR = L::MB + L::NB, RPM = (NR + NM - 1) / NM;
  constexpr int Q3 = L::CP / 2;  // copies of a step issued behind its stage's barrier; the rest a sub-step later
  const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % (BM / WM), wn = wave / (BM / WM);
  // copy q = wave CP + i covers rows 8 (q mod BM/8) .. +7 of x (q < BM/8) or of w: lane l takes row
  // + l / 8, slot l mod 8 <- chunk (l mod 8) ^ ((row / 2) mod 8)
  uint32_t off[L::CP];
#pragma unroll
  for (int i = 0; i < L::CP; i++) {
    const int q = wave * L::CP + i;
    const bool isx = q < BM / 8;
    const int r = 8 * (isx ? q : q - BM / 8) + (lane >> 3);
    const int c = (lane & 7) ^ ((r >> 1) & 7);
    off[i] = (isx ? (uint32_t)min(r, tmax) * (uint32_t)ldx : (uint32_t)min(r, nmax) * (uint32_t)ldw) + 16 * c;
  }
  auto copy = [&](int ks, int i) __attribute__((always_inline)) {
    const int q = wave * L::CP + i;
    dma16_s((q < BM / 8 ? xk : wk) + (int64_t)ks * kRow, off[i], lds_base + (ks % D) * L::STAGE + q * 1024);
  };
  // fragments: row r, chunk 2 kk + lane / 32 at slot chunk ^ ((r / 2) mod 8); the blocks of 32 rows
  // share the swizzle
  const int r32 = lane & 31, kh = lane >> 5, sw = (r32 >> 1) & 7;
  const uint32_t xrow = (WM * wm + r32) * kRow, wrow = BM * kRow + (WN * wn + r32) * kRow;
  bf16x8_t a[2][L::MB], b[2][L::NB];
  auto read = [&](int ks, int kk, int buf, int i) __attribute__((always_inline)) {
    const lds_u8_t* st = lds + (ks % D) * L::STAGE + 16 * ((2 * kk + kh) ^ sw);
    if (i < L::NB) b[buf][i] = as_bf16x8(*(const lds_u32x4_t*)(st + wrow + 32 * kRow * i));
    else a[buf][i - L::NB] = as_bf16x8(*(const lds_u32x4_t*)(st + xrow + 32 * kRow * (i - L::NB)));
  };
  // the MFMAs of one sub-step, with the reads of sub-step (rs, RK) (RK < 0: none) and copies I0 ..
  // I1-1 of step `is` between them
  auto sub = [&](auto cur_, int rs, auto rk_, int is, auto i0_, auto i1_) __attribute__((always_inline)) {
    constexpr int cur = decltype(cur_)::value, rk = decltype(rk_)::value;
    constexpr int i0 = decltype(i0_)::value, nc = decltype(i1_)::value - i0;
#pragma unroll
    for (int j = 0; j < NM; j++) {
      if constexpr (rk >= 0) {
#pragma unroll
        for (int e = j * RPM; e < (j + 1) * RPM && e < NR; e++) read(rs, rk, cur ^ 1, e);
      }
      const int m = j / L::NB, n = j % L::NB;
      acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[cur][m], b[cur][n], acc[m][n], 0, 0, 0);
#pragma unroll
      for (int e = j * nc / NM; e < (j + 1) * nc / NM; e++) copy(is, i0 + e);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // step ks: MORE: the second part of step ks + D - 1's copies is still to be issued; FIRST: so is
  // the first part of step ks + D's; NEXT: a step follows.  Separate loops, not branches around
  // the MFMAs: a branch gives the accumulators two homes and copies between them.
  auto step = [&](int ks, auto more_, auto first_, auto next_) __attribute__((always_inline)) {
    constexpr int more = decltype(more_)::value, first = decltype(first_)::value, next = decltype(next_)::value;
    sub(Int<0>{}, ks, Int<1>{}, ks + D - 1, Int<Q3>{}, Int<more ? L::CP : Q3>{});
    sub(Int<1>{}, ks, Int<2>{}, 0, Int<0>{}, Int<0>{});
    sub(Int<0>{}, ks, Int<3>{}, 0, Int<0>{}, Int<0>{});
    if constexpr (next) {
      wait_vm(more ? (D - 2) * L::CP : 0);  // this wave's copies of step ks + 1
      lds_barrier();                         // everyone's; and step ks is in every wave's registers
      landed(ks + 1, lds + ((ks + 1) % D) * L::STAGE, Int<0>{});
      sub(Int<1>{}, ks + 1, Int<0>{}, ks + D, Int<0>{}, Int<first ? Q3 : 0>{});
    } else {
      sub(Int<1>{}, 0, Int<-1>{}, 0, Int<0>{}, Int<0>{});
    }
  };
#pragma unroll
  for (int m = 0; m < L::MB; m++)
#pragma unroll
    for (int n = 0; n < L::NB; n++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[m][n][r] = 0.f;
#pragma unroll
  for (int s = 0; s < D; s++)
#pragma unroll
    for (int i = 0; i < (s < D - 1 ? L::CP : Q3); i++) copy(s, i);
  wait_vm((D - 2) * L::CP + Q3);
  lds_barrier();
  landed(0, lds, Int<1>{});
#pragma unroll
  for (int i = 0; i < NR; i++) read(0, 0, 0, i);
  int ks = 0;
  for (; ks < nk - D; ks++) step(ks, Int<1>{}, Int<1>{}, Int<1>{});
  step(ks++, Int<1>{}, Int<0>{}, Int<1>{});
  for (; ks < nk - 1; ks++) step(ks, Int<0>{}, Int<0>{}, Int<1>{});
  step(ks, Int<0>{}, Int<0>{}, Int<0>{});
}

}  // namespace smla_gemm

// The K loop of the tiled fp32 product (gemm.hip): one workgroup's BM x BN tile of x . w^T, both
// operands K-contiguous fp32, on the bf16 matrix cores.
//
// An fp32 value, times 2^16, is the sum of three bf16 values, 2^16 x = h + m + l, each the nearest bf16 to
// what is left: exact for every x below 2^112 (the lowest bit of a subnormal, 2^-149, becomes a
// subnormal bf16's, 2^-133; without the factor a value below 2^-110 lost bits).  x w = hh + (hm + mh) +
// (hl + lh + mm) up to 2^-24 |x w|, of either sign: the products of bf16 values are exact in fp32 and
// v_mfma_f32_32x32x16_bf16 adds 16 k of one of them per accumulator rounding, against one rounding per k
// (or two) of a chain of fp32 fmas.  hh has an accumulator, the five small products share another, added
// once at the end: in one accumulator the 2^-16 of hl, lh and mm fall below half its last place once it
// holds some thousand products, always with the same sign (1.05e-5 for K = 4096 and operands of one
// sign).  Distance from float64 (relative, 2-norm), here / one chain of fp32 MFMAs:
//   K             64                1024              4096              8192
//   uniform 0..1  0.5 / 1.2e-7      0.7 / 4.3e-7      3.0 / 8.4e-7      4.2e-7 / 1.2e-6
//   normal        0.5 / 1.4e-7      1.1 / 5.7e-7      4.0e-7 / 1.2e-6   5.7e-7 / 1.6e-6
// An operand that the split cannot carry (infinite, NaN, from 2^112) or a sum from 2^96 is non-finite
// here, and every non-finite sum is taken from the fp32 MFMAs instead (block_f32), so infinities and
// NaN come out as fp32 arithmetic gives them.  The three-way split is that of G. Henry, P. Tang and
// A. Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for higher-precision
// computations" (2019).
//
// Six bf16 MFMAs carry 16 k in 192 cycles per 32 x 32 block where the fp32 MFMAs take 512.  [2046, 4096] x
// [2048, 4096]^T: 382 us with fp32 MFMAs and register staging, 197 us here (174 TFLOP/s; the fp32 MFMA
// peak is 157); [1, 8192] x [4096, 8192]^T 694 -> 50 us.
//
// What bounds it is the vector ALU work of the splits (13 instructions per pair of values, done by
// every wave that reads them) beside the MFMAs: either takes more than half of the cycles, and they
// overlap only in part (without the factor 2^16, 11 instructions: 184 us).  The splits of the next 16 k
// are therefore interleaved with the MFMAs of the current ones, and the raw values of the 16 k after
// those are read from LDS meanwhile (two register sets of each).
#pragma once

#include "gemm_tile.h"

namespace smla_gemm {

struct Split3 {
  bf16x8_t h, m, l;
};

// the high halves of a (low word) and b (high word)
__device__ inline uint32_t top_halves(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

// the parts of 2^16 x: its lowest bit is a bf16 (2^-149 of a subnormal comes to 2^-133)
__device__ inline Split3 split3(u32x4_t lo, u32x4_t hi) {
  u32x4_t h, m, l;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const float a = __uint_as_float(j < 2 ? lo[2 * j] : hi[2 * j - 4]) * 0x1p16f;
    const float b = __uint_as_float(j < 2 ? lo[2 * j + 1] : hi[2 * j - 3]) * 0x1p16f;
    h[j] = pack_bf16x2(a, b);
    const float a1 = a - __uint_as_float(h[j] << 16), b1 = b - __uint_as_float(h[j] & 0xffff0000u);
    m[j] = pack_bf16x2(a1, b1);
    const float a2 = a1 - __uint_as_float(m[j] << 16), b2 = b1 - __uint_as_float(m[j] & 0xffff0000u);
    l[j] = top_halves(a2, b2);
  }
  return {as_bf16x8(h), as_bf16x8(m), as_bf16x8(l)};
}

// acc[mb][nb] = rows 0 .. BM-1 of x times rows 0 .. BN-1 of w over nk >= D steps of 32 k; arguments and
// accumulator layout as tile_loop's.  Rows of 128 bytes (32 k) as there; the ring is one step further
// ahead: step s + 1 is read from LDS while step s is multiplied.
template <int BM, int BN, int WM, int WN, int D>
__device__ __attribute__((always_inline)) inline void tile_loop_f32(lds_u8_t* lds, const uint8_t* __restrict__ xk,
                                                                    int64_t ldx, int tmax,
                                                                    const uint8_t* __restrict__ wk, int64_t ldw,
                                                                    int nmax, int nk,
                                                                    f32x16_t (&acc)[WM / 32][WN / 32]) {
  using L = Tile<BM, BN, WM, WN, D>;
  constexpr int MB = L::MB, NB = L::NB, NR = MB + NB;
  const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % (BM / WM), wn = wave / (BM / WM);
  uint32_t off[L::CP];
#pragma unroll
  for (int i = 0; i < L::CP; i++) {
    const int q = wave * L::CP + i;
    const bool isx = q < BM / 8;
    const int r = 8 * (isx ? q : q - BM / 8) + (lane >> 3);
    const int c = (lane & 7) ^ ((r >> 1) & 7);
    off[i] = (isx ? (uint32_t)min(r, tmax) * (uint32_t)ldx : (uint32_t)min(r, nmax) * (uint32_t)ldw) + 16 * c;
  }
  auto copy = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < L::CP; i++) {
      const int q = wave * L::CP + i;
      dma16_s((q < BM / 8 ? xk : wk) + (int64_t)ks * kRow, off[i], lds_base + (ks % D) * L::STAGE + q * 1024);
    }
  };
  // a fragment is 8 k of a row, k 16 kk + 8 (lane / 32) ..: chunks 4 kk + 2 (lane / 32) and the next
  const int r32 = lane & 31, kh = lane >> 5, sw = (r32 >> 1) & 7;
  const uint32_t xrow = (WM * wm + r32) * kRow, wrow = BM * kRow + (WN * wn + r32) * kRow;
  u32x4_t raw[2][NR][2];
  Split3 sp[2][NR];
  auto read = [&](int ks, auto kk_) __attribute__((always_inline)) {
    constexpr int kk = decltype(kk_)::value;
    const lds_u8_t* st = lds + (ks % D) * L::STAGE;
#pragma unroll
    for (int i = 0; i < NR; i++)
#pragma unroll
      for (int e = 0; e < 2; e++)
        raw[kk][i][e] = *(const lds_u32x4_t*)(st + (i < MB ? xrow + 32 * kRow * i : wrow + 32 * kRow * (i - MB)) +
                                              16 * ((4 * kk + 2 * kh + e) ^ sw));
  };
  auto split = [&](auto kk_) __attribute__((always_inline)) {
    constexpr int kk = decltype(kk_)::value;
#pragma unroll
    for (int i = 0; i < NR; i++) sp[kk][i] = split3(raw[kk][i][0], raw[kk][i][1]);
  };
  // the MFMAs of sub-step kk: hh into acc, the others into low; the blocks alternate so that an
  // accumulator is not wanted again at once
  f32x16_t low[MB][NB];
  auto mul = [&](auto kk_) __attribute__((always_inline)) {
    constexpr int kk = decltype(kk_)::value;
#pragma unroll
    for (int p = 0; p < 6; p++)
#pragma unroll
      for (int j = 0; j < MB * NB; j++) {
        const Split3 &a = sp[kk][j / NB], &b = sp[kk][MB + j % NB];
        const bf16x8_t u = p == 0 ? a.m : p == 1 ? a.l : p == 3 ? a.m : a.h;
        const bf16x8_t v = p == 0 ? b.m : p == 2 ? b.l : p == 4 ? b.m : b.h;
        f32x16_t& c = p == 5 ? acc[j / NB][j % NB] : low[j / NB][j % NB];
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(u, v, c, 0, 0, 0);
      }
  };
  // 13 vector instructions per pair of values of the four, and some of the addresses' (with room for just
  // 52 the compiler takes 284 registers instead of 244, which is one wave per SIMD: 240 us instead of 197)
  auto pin = [&]() __attribute__((always_inline)) {
    constexpr int V = (NR * 56 + 6 * MB * NB - 1) / (6 * MB * NB);
#pragma unroll
    for (int j = 0; j < 6 * MB * NB; j++) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // MFMA
      __builtin_amdgcn_sched_group_barrier(0x2, V, 0);  // VALU
    }
  };
#pragma unroll
  for (int m = 0; m < MB; m++)
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[m][n][r] = low[m][n][r] = 0.f;
#pragma unroll
  for (int s = 0; s < D; s++) copy(s);
  wait_vm((D - 1) * L::CP);
  lds_barrier();
  read(0, Int<0>{});
  read(0, Int<1>{});
  split(Int<0>{});
  auto step = [&](int ks, auto more_, auto next_) __attribute__((always_inline)) {
    constexpr int more = decltype(more_)::value, next = decltype(next_)::value;
    if constexpr (next) {
      wait_vm(more ? (D - 2) * L::CP : 0);  // this wave's copies of step ks + 1
      lds_barrier();                         // everyone's; and step ks is in every wave's registers
      if constexpr (more) copy(ks + D);
      read(ks + 1, Int<0>{});
    }
    mul(Int<0>{});
    split(Int<1>{});
    pin();
    if constexpr (next) read(ks + 1, Int<1>{});
    mul(Int<1>{});
    if constexpr (next) split(Int<0>{});
    pin();
  };
  int ks = 0;
  for (; ks < nk - D; ks++) step(ks, Int<1>{}, Int<1>{});
  for (; ks < nk - 1; ks++) step(ks, Int<0>{}, Int<1>{});
  step(ks, Int<0>{}, Int<0>{});
#pragma unroll
  for (int m = 0; m < MB; m++)
#pragma unroll
    for (int n = 0; n < NB; n++) acc[m][n] = (acc[m][n] + low[m][n]) * 0x1p-32f;
}

// Block (mb, nb) of this wave's part of the tile by fp32 MFMAs, operands from memory; arguments and layout
// as tile_loop_f32's.  Lane half h takes k = 8 j + 4 h .. + 3 of its row of x and its row of w: one
// 16-byte load of each per four MFMAs.  Bound by the latency of those loads.  [1024, 8192] x [4096,
// 8192]^T with one infinite weight: 743 us (364 without it), against 21200 for one serial chain per output;
// with an infinity in every row of x 1338.
template <int BM, int BN, int WM, int WN>
__device__ __attribute__((always_inline)) inline f32x16_t block_f32(const uint8_t* __restrict__ xk, int64_t ldx, int tmax,
                                                       const uint8_t* __restrict__ wk, int64_t ldw, int nmax, int nk,
                                                       int mb, int nb) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave % (BM / WM), wn = wave / (BM / WM);
  const uint8_t* xr = xk + min(WM * wm + 32 * mb + (lane & 31), tmax) * ldx + 16 * (lane >> 5);
  const uint8_t* wr = wk + min(WN * wn + 32 * nb + (lane & 31), nmax) * ldw + 16 * (lane >> 5);
  f32x16_t c;
#pragma unroll
  for (int r = 0; r < 16; r++) c[r] = 0.f;
  for (int ks = 0; ks < nk; ks++) {
    f32x4_t a[4], b[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      a[j] = *(const f32x4_t*)(xr + (int64_t)ks * kRow + 32 * j);
      b[j] = *(const f32x4_t*)(wr + (int64_t)ks * kRow + 32 * j);
    }
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int i = 0; i < 4; i++) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j][i], b[j][i], c, 0, 0, 0);
  }
  return c;
}

}  // namespace smla_gemm

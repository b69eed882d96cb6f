// Tiled MFMA GEMM for the projections beyond the decode step's few rows (linear.hip):
//   y[t, g*N + n] = sum_k x[t, g*K + k] * w[g*N + n, k]      (v4mlx/mla.py:16-18, and the grouped
//   product of v4mlx/mla.py:49-53 for G > 1; ref_torch/compressor.py:28-29 with fp32 operands)
//
// Both operands are K-contiguous (x rows, w rows), which is the operand order of the gfx950 MFMA:
// a lane's A fragment is 8 consecutive k of one token row, its B fragment 8 consecutive k of one
// weight row.  Rows past T or N are loaded clamped (finite) and never stored.
//
// gemm_ring_kernel (bf16, K a multiple of 64): the K loop of gemm_tile.h in one of four tile forms.
// A product of a few hundred tokens has far fewer large tiles than the chip has CUs, and each tile's
// K range is a serial chain of steps, so the time is that chain's: the plan weighs smaller tiles (more
// workgroups, more operand bytes each) against splitting the K range over up to 8 workgroups per
// tile, whose fp32 partial sums gemm_reduce_kernel adds in split order.  Before and after, us:
//   [64, 8192] x [4096, 8192]^T 156 -> 16 (67 MB of weights at 4.2 TB/s), [300, 8192] x the same 184 ->
//   33, 8 groups of [300, 4096] x [1024, 4096]^T 100 -> 33, [1024, 4096] x [1024, 4096]^T 83 -> 17,
//   [4096, 8192] x [4096, 8192]^T 244 -> 210, [4096, 1024] x [32768, 1024]^T 291 -> 265.
//
// gemm_kernel (the K that the ring kernels do not take: bf16 below 128 or not a multiple of 64, fp32 below 64
// or not a multiple of 32, rows past 31-bit offsets): 4 waves computing a 128 x 128 tile, each wave a
// 64 x 64 quarter as 2 x 2 blocks of v_mfma_f32_32x32x16_bf16 (bf16 operands) or
// v_mfma_f32_32x32x2f32 (fp32 operands), accumulating in fp32.  K advances in steps of 128 bytes
// per row (64 bf16 / 32 fp32): the next step's tiles are loaded into registers while the current
// ones are multiplied out of LDS, two LDS stages, one barrier per step.  LDS rows are padded to
// 144 bytes so the 16-byte fragment reads of 32 consecutive rows spread over the banks.  K is a
// multiple of 16 bytes, and the 16-byte chunks of the last step that lie past K are zero.
//
// ROPE (bf16, the attention output projection of oracle/decode_engine.py:118-119): the K step that
// holds the last rd = 64 dims of a head has its (x0, x1) pairs rotated back to position 0 before it
// is read (inverse RoPE at pos[t], every product and sum rounded in float32, then bf16), the
// arithmetic of smla_rope.
#include "gemm_f32.h"
#include "gemm_tile.h"
#include "smla_internal.h"

namespace {

constexpr int kBM = 128, kBN = 128;   // tile: tokens x outputs
constexpr int kRowBytes = 128;        // bytes of one tile row per K step
constexpr int kLdsRow = 144;          // padded LDS row
constexpr int kTileLds = kBM * kLdsRow;
constexpr int kChunks = kBM * kRowBytes / 16 / 256;  // 16-byte chunks per thread per operand (4)

__device__ inline float mul_rn_g(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}
__device__ inline float add_rn_g(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}
__device__ inline float sub_rn_g(float a, float b) {
#pragma clang fp contract(off)
  return a - b;
}

// inverse RoPE of 4 (x0, x1) bf16 pairs held in one 16-byte chunk, pairs p0 .. p0+3 at one position
__device__ inline u32x4_t inv_rope4(u32x4_t v, f32x4_t c, f32x4_t s) {
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const float x0 = __uint_as_float(v[j] << 16), x1 = __uint_as_float(v[j] & 0xffff0000u);
    const float o0 = add_rn_g(mul_rn_g(x0, c[j]), mul_rn_g(x1, s[j]));
    const float o1 = sub_rn_g(mul_rn_g(x1, c[j]), mul_rn_g(x0, s[j]));
    v[j] = pack_bf16x2(o0, o1);
  }
  return v;
}

template <bool BF16, int YDT, bool ROPE>
__global__ __launch_bounds__(256) void gemm_kernel(const uint8_t* __restrict__ x, int64_t ldx,
                                                   const uint8_t* __restrict__ w, int T, int N, int K, int ntn,
                                                   const int32_t* __restrict__ pos, const float* __restrict__ cos_t,
                                                   const float* __restrict__ sin_t, int head_dim,
                                                   void* __restrict__ y, int64_t ldy) {
  constexpr int ES = BF16 ? 2 : 4;              // element bytes
  constexpr int KSTEP = kRowBytes / ES;         // K per step: 64 / 32
  __shared__ __align__(16) uint8_t lds[2][2][kTileLds];  // [stage][A, B]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = blockIdx.x / ntn;
  const int n0 = (blockIdx.x % ntn) * kBN;
  const int t0 = blockIdx.y * kBM;
  const int wm = wave & 1, wn = wave >> 1;

  // this thread's chunks: chunk c = tid + 256 i -> tile row c / 8, 16-byte column c % 8
  const uint8_t* ap[kChunks];
  const uint8_t* bp[kChunks];
  int lofs[kChunks];
  const float* csp[kChunks];
  const float* snp[kChunks];
#pragma unroll
  for (int i = 0; i < kChunks; i++) {
    const int c = tid + 256 * i, row = c >> 3, col = c & 7;
    const int t = min(t0 + row, T - 1);
    const int n = min(n0 + row, N - 1);
    ap[i] = x + ((int64_t)t * ldx + (int64_t)g * K) * ES + col * 16;
    bp[i] = w + ((int64_t)g * N + n) * K * ES + col * 16;
    lofs[i] = row * kLdsRow + col * 16;
    if constexpr (ROPE) {
      const int64_t p = pos[t];
      csp[i] = cos_t + p * 32 + 4 * col;   // rd / 2 = 32 pairs; this chunk holds pairs 4 col .. +3
      snp[i] = sin_t + p * 32 + 4 * col;
    }
  }
  u32x4_t ra[kChunks], rb[kChunks];
  const int kbytes = K * ES;
  const int ccol = (tid & 7) * 16;  // this thread's chunk column (the same for its kChunks chunks)
  auto load = [&](int ks) {
    const int64_t off = (int64_t)ks * kRowBytes;
    if (off + ccol < kbytes) {
#pragma unroll
      for (int i = 0; i < kChunks; i++) {
        ra[i] = *(const u32x4_t*)(ap[i] + off);
        rb[i] = *(const u32x4_t*)(bp[i] + off);
      }
    } else {
#pragma unroll
      for (int i = 0; i < kChunks; i++) ra[i] = rb[i] = u32x4_t{0u, 0u, 0u, 0u};
    }
  };
  auto store = [&](int stage, int ks) {
    if constexpr (ROPE) {
      if ((ks * KSTEP) % head_dim == head_dim - 64) {
#pragma unroll
        for (int i = 0; i < kChunks; i++) ra[i] = inv_rope4(ra[i], *(const f32x4_t*)csp[i], *(const f32x4_t*)snp[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < kChunks; i++) {
      *(u32x4_t*)&lds[stage][0][lofs[i]] = ra[i];
      *(u32x4_t*)&lds[stage][1][lofs[i]] = rb[i];
    }
  };

  f32x16_t acc[2][2];
#pragma unroll
  for (int mb = 0; mb < 2; mb++)
#pragma unroll
    for (int nb = 0; nb < 2; nb++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[mb][nb][r] = 0.f;

  const int nk = (kbytes + kRowBytes - 1) / kRowBytes;
  load(0);
  store(0, 0);
  __syncthreads();
  // fragment rows of this lane: A row 64 wm + 32 mb + lane % 32, B row 64 wn + 32 nb + lane % 32
  const int arow = (64 * wm + (lane & 31)) * kLdsRow, brow = (64 * wn + (lane & 31)) * kLdsRow;
  const int khalf = lane >> 5;
  for (int ks = 0; ks < nk; ks++) {
    const int st = ks & 1;
    if (ks + 1 < nk) load(ks + 1);
    const uint8_t* A = lds[st][0];
    const uint8_t* B = lds[st][1];
    if constexpr (BF16) {
#pragma unroll
      for (int kk = 0; kk < 4; kk++) {   // 16 k per MFMA: lane half h holds k = 16 kk + 8 h ..
        const int ko = kk * 32 + khalf * 16;
        bf16x8_t a[2], b[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
          a[j] = as_bf16x8(*(const u32x4_t*)&A[arow + 32 * j * kLdsRow + ko]);
          b[j] = as_bf16x8(*(const u32x4_t*)&B[brow + 32 * j * kLdsRow + ko]);
        }
#pragma unroll
        for (int mb = 0; mb < 2; mb++)
#pragma unroll
          for (int nb = 0; nb < 2; nb++)
            acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[mb], b[nb], acc[mb][nb], 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < 16; kk++) {  // 2 k per MFMA: lane half h holds k = 2 kk + h
        const int ko = (2 * kk + khalf) * 4;
        float a[2], b[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
          a[j] = *(const float*)&A[arow + 32 * j * kLdsRow + ko];
          b[j] = *(const float*)&B[brow + 32 * j * kLdsRow + ko];
        }
#pragma unroll
        for (int mb = 0; mb < 2; mb++)
#pragma unroll
          for (int nb = 0; nb < 2; nb++)
            acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[mb], b[nb], acc[mb][nb], 0, 0, 0);
      }
    }
    if (ks + 1 < nk) store(st ^ 1, ks + 1);
    __syncthreads();
  }

  // accumulator r of block (mb, nb): token 64 wm + 32 mb + 8 (r / 4) + 4 (lane / 32) + r % 4,
  // output 64 wn + 32 nb + lane % 32
#pragma unroll
  for (int mb = 0; mb < 2; mb++)
#pragma unroll
    for (int nb = 0; nb < 2; nb++) {
      const int n = n0 + 64 * wn + 32 * nb + (lane & 31);
      if (n >= N) continue;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int t = t0 + 64 * wm + 32 * mb + 8 * (r >> 2) + 4 * khalf + (r & 3);
        if (t < T) {
          const int64_t o = (int64_t)t * ldy + (int64_t)g * N + n;
          if constexpr (YDT == SMLA_BF16)
            __builtin_nontemporal_store((uint16_t)bf16_rne(acc[mb][nb][r]), (uint16_t*)y + o);
          else
            __builtin_nontemporal_store(acc[mb][nb][r], (float*)y + o);
        }
      }
    }
}

// ---- the ring kernel's tile forms (tokens x outputs, waves of .. x .., stages)
template <int FORM>
struct Form;
template <>
struct Form<0> {  // 4 waves, 64 KB: two workgroups per CU
  static constexpr int BM = 64, BN = 64, WM = 32, WN = 32, D = 4;
};
template <>
struct Form<1> {  // 4 waves, 128 KB
  static constexpr int BM = 128, BN = 128, WM = 64, WN = 64, D = 4;
};
template <>
struct Form<2> {  // 8 waves, 144 KB
  static constexpr int BM = 128, BN = 256, WM = 64, WN = 64, D = 3;
};
template <>
struct Form<3> {  // 8 waves, 128 KB
  static constexpr int BM = 256, BN = 256, WM = 128, WN = 64, D = 2;
};
constexpr int kForms = 4;
constexpr int kFormBM[kForms] = {64, 128, 128, 256}, kFormBN[kForms] = {64, 128, 256, 256};
constexpr int kFormD[kForms] = {Form<0>::D, Form<1>::D, Form<2>::D, Form<3>::D};  // least K steps of a workgroup
constexpr int kMaxSplits = 8;

struct RingArgs {
  const uint8_t* x;
  const uint8_t* w;
  const uint8_t* w2;  // the second group's weights (else group g's follow group g - 1's)
  int64_t ldx;        // bytes
  int64_t xg;         // bytes between the groups' slices of a row of x
  int T, N, K, G, nt, nn, splits;
  const int32_t* pos;
  const float* cos_t;
  const float* sin_t;
  uint32_t head_steps, head_magic;  // ROPE: K steps of 64 per head, ceil(2^32 / head_steps)
  uint8_t* y;
  int64_t ldy, split_stride;  // elements
  int vec;                    // rows and groups of y start at multiples of 16 bytes
  int pair;                   // 2: the tiles of two groups side by side, else 1
};

// The tile's outputs from the accumulators (layout of tile_loop) to rows t0 .., columns n0 .. of group g
// (of split sp's partial sums, with splits).
// Output rows leave through LDS (each wave its own region, MBP blocks of 32 rows at a time), so that
// a lane stores 16 bytes and a wave whole 128-byte lines: 16 stores per wave instead of 128 of two
// bytes per lane, few enough to stay in flight when the wave ends.  Chunk c of row r sits in slot
// c ^ swizzle(r), so that the two rows of a write (r and r + 4) and the rows of a read use distinct
// banks.  Nontemporal: the output is not read back by this launch.
template <class F, int YDT>
__device__ __attribute__((always_inline)) inline void store_tile(smla_attn::lds_u8_t* lds, const RingArgs& p, int sp,
                                                                 int g, int t0, int n0,
                                                                 const f32x16_t (&acc)[F::WM / 32][F::WN / 32]) {
  using namespace smla_gemm;
  constexpr int BM = F::BM, WM = F::WM, WN = F::WN;
  using L = Tile<F::BM, F::BN, F::WM, F::WN, F::D>;
  constexpr int ES = YDT == SMLA_BF16 ? 2 : 4, CH = WN * ES / 16, RPI = 64 / CH;  // chunks per row, rows per store
  constexpr int FIT = L::LDS / (L::NW * 32 * WN * ES), MBP = FIT < L::MB ? FIT : L::MB;
  static_assert(MBP >= 1 && L::MB % MBP == 0, "the waves' regions fit the ring's LDS");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave % (BM / WM), wn = wave / (BM / WM);
  const int64_t base = sp * p.split_stride + (int64_t)g * p.N;
  if (p.vec) {  // uniform
    lds_u8_t* reg = lds + wave * (MBP * 32 * WN * ES);
    auto slot = [](int r, int c) { return CH == 16 ? c ^ ((r << 1) & 8) : c ^ (r & (CH - 1)); };
    lds_barrier();  // every wave has read its last fragments
#pragma unroll
    for (int m0 = 0; m0 < L::MB; m0 += MBP) {
#pragma unroll
      for (int mb = 0; mb < MBP; mb++)
#pragma unroll
        for (int nb = 0; nb < L::NB; nb++)
#pragma unroll
          for (int r = 0; r < 16; r++) {
            const int row = 32 * mb + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3), col = (32 * nb + (lane & 31)) * ES;
            lds_u8_t* q = reg + row * (WN * ES) + 16 * slot(row, col >> 4) + (col & 15);
            if constexpr (YDT == SMLA_BF16) *(smla_attn::lds_u16_t*)q = bf16_rne(acc[m0 + mb][nb][r]);
            else *(smla_attn::lds_f32_t*)q = acc[m0 + mb][nb][r];
          }
      const int n = n0 + WN * wn + (lane % CH) * (16 / ES);
#pragma unroll
      for (int i = 0; i < MBP * 32 / RPI; i++) {
        const int row = RPI * i + lane / CH, t = t0 + WM * wm + 32 * m0 + row;
        const u32x4_t v = *(lds_u32x4_t*)(reg + row * (WN * ES) + 16 * slot(row, lane % CH));
        if (t < p.T && n < p.N)
          __builtin_nontemporal_store(v, (u32x4_t*)(p.y + (base + (int64_t)t * p.ldy + n) * ES));
      }
    }
    return;
  }
#pragma unroll
  for (int mb = 0; mb < L::MB; mb++)
#pragma unroll
    for (int nb = 0; nb < L::NB; nb++) {
      const int n = n0 + WN * wn + 32 * nb + (lane & 31);
      const int t1 = t0 + WM * wm + 32 * mb + 4 * (lane >> 5);
      if (n >= p.N) continue;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int t = t1 + 8 * (r >> 2) + (r & 3);
        if (t < p.T) {
          const int64_t o = base + (int64_t)t * p.ldy + n;
          if constexpr (YDT == SMLA_BF16) ((uint16_t*)p.y)[o] = bf16_rne(acc[mb][nb][r]);
          else ((float*)p.y)[o] = acc[mb][nb][r];
        }
      }
    }
}

// Workgroup order: the launch deals workgroups to the 8 XCDs round-robin; each XCD takes a
// contiguous run of tiles, ordered in groups of 4 token tiles over all output tiles, so that the
// tiles running together on an XCD share x and w rows in its L2.  Splits are outermost.  With pair, the 4
// token tiles of two groups take turns at every output tile: rows of x 64 KB apart fall in the same
// sets of an L2, which 8 token tiles of one group want at the same column, and two groups spread over
// twice the sets (8 groups of [4096, 4096] x [1024, 4096]^T 257 -> 225 us, [2000, 4096] 135 -> 120; four
// or eight groups, with as many times the weights, 247 and 255; tiles started 4 or 8 us apart 250 and 240).
struct TileId {
  int sp, g, tm, tn;  // split, group, token tile, output tile
};
__device__ inline TileId tile_id(const RingArgs& p) {
  const uint32_t tot = gridDim.x, per = tot / kXcds, rem = tot % kXcds, xcd = blockIdx.x % kXcds;
  uint32_t id = xcd * per + (xcd < rem ? xcd : rem) + blockIdx.x / kXcds;
  const uint32_t tiles = (uint32_t)p.nt * p.nn;
  uint32_t sg = id / (tiles * p.pair) * p.pair;  // split * G + group
  id -= sg * tiles;
  const uint32_t blk = 4u * p.nn * p.pair;
  const uint32_t grp = id / blk, gs = min(4u, (uint32_t)p.nt - 4 * grp), in = id - grp * blk;
  const uint32_t col = in / gs;  // output tile, of the pair's groups in turn
  sg += col % p.pair;
  TileId t;
  t.sp = sg / p.G;
  t.g = sg - t.sp * p.G;
  t.tm = 4 * grp + in % gs;
  t.tn = col / p.pair;
  return t;
}

__device__ inline const uint8_t* group_weights(const RingArgs& p, int g, int es) {
  return p.w2 && g > 0 ? p.w2 : p.w + (int64_t)g * p.N * (int64_t)p.K * es;
}

template <int FORM, int YDT, bool ROPE>
__global__ __launch_bounds__((Form<FORM>::BM / Form<FORM>::WM) * (Form<FORM>::BN / Form<FORM>::WN) * 64) void
gemm_ring_kernel(const RingArgs p) {
  using namespace smla_gemm;
  using F = Form<FORM>;
  constexpr int BM = F::BM, BN = F::BN, WM = F::WM, WN = F::WN, D = F::D;
  using L = Tile<BM, BN, WM, WN, D>;
  extern __shared__ __align__(16) uint8_t lds_g[];
  const TileId id = tile_id(p);
  const int sp = id.sp, g = id.g, t0 = id.tm * BM, n0 = id.tn * BN;
  const int nk = p.K / 64, k0 = nk * sp / p.splits, k1 = nk * (sp + 1) / p.splits;
  const uint8_t* xk = p.x + (int64_t)t0 * p.ldx + g * p.xg + (int64_t)k0 * kRow;
  const uint8_t* wk = group_weights(p, g, 2) + (int64_t)n0 * p.K * 2 + (int64_t)k0 * kRow;

  // ROPE: the chunks of x this thread rotates in a step that holds a head's last 64 dims: chunk tid + i
  // threads is row j / 8, slot j mod 8, 4 (x0, x1) pairs from pair 4 c, c = slot ^ ((row / 2) mod 8).  Their
  // rotations are the same in every such step: loaded once, waited for once (with the first stage),
  // because a wait for a load inside the loop drains the ring's copies with it (the output path of 300
  // tokens 83 -> 81 us)
  constexpr int NT = L::NW * 64, ACH = BM * 8 / NT;
  f32x4_t cs[ACH], sn[ACH];
  if constexpr (ROPE) {
#pragma unroll
    for (int i = 0; i < ACH; i++) {
      const int j = threadIdx.x + NT * i, c = (j & 7) ^ ((j >> 4) & 7);
      const int64_t at = (int64_t)p.pos[min(t0 + (j >> 3), p.T - 1)] * 32 + 4 * c;
      cs[i] = *(const f32x4_t*)(p.cos_t + at);
      sn[i] = *(const f32x4_t*)(p.sin_t + at);
    }
  }
  f32x16_t acc[L::MB][L::NB];
  tile_loop<BM, BN, WM, WN, D>((lds_u8_t*)lds_g, xk, p.ldx, p.T - 1 - t0, wk, (int64_t)p.K * 2, p.N - 1 - n0, k1 - k0,
                               acc, [&](int ks, lds_u8_t* stage, auto first) __attribute__((always_inline)) {
    if constexpr (ROPE) {
      if constexpr (decltype(first)::value) {
#pragma unroll
        for (int i = 0; i < ACH; i++) asm volatile("" : "+v"(cs[i]), "+v"(sn[i]));
      }
      // step k of the row holds dims 64 (k mod head_steps) .. of a head (k < 2^16: the product is exact)
      const uint32_t k = k0 + ks;
      if (p.head_steps == 1 || k - __umulhi(k, p.head_magic) * p.head_steps == p.head_steps - 1) {
#pragma unroll
        for (int i = 0; i < ACH; i++) {
          const int j = threadIdx.x + NT * i;
          lds_u32x4_t* pa = (lds_u32x4_t*)(stage + (j >> 3) * kRow + 16 * (j & 7));
          *pa = inv_rope4(*pa, cs[i], sn[i]);
        }
        lds_barrier();
      }
    }
  });

  store_tile<F, YDT>((smla_attn::lds_u8_t*)lds_g, p, sp, g, t0, n0, acc);
}

// fp32 operands with K a multiple of 32 (the K loop of gemm_f32.h); forms of 64 x 64 and 128 x 128
// outputs, two workgroups per CU.
template <int FORM>
struct FormF32;
template <>
struct FormF32<0> {
  static constexpr int BM = 64, BN = 64, WM = 32, WN = 32, D = 4;
};
template <>
struct FormF32<1> {
  static constexpr int BM = 128, BN = 128, WM = 64, WN = 64, D = 2;
};
constexpr int kFormsF32 = 2;
constexpr int kFormF32B[kFormsF32] = {64, 128}, kFormF32D[kFormsF32] = {FormF32<0>::D, FormF32<1>::D};

template <int FORM, int YDT>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const RingArgs p) {
  using namespace smla_gemm;
  using F = FormF32<FORM>;
  constexpr int BM = F::BM, BN = F::BN, WM = F::WM, WN = F::WN, D = F::D;
  using L = Tile<BM, BN, WM, WN, D>;
  static_assert(L::NW == 4 && L::MB * L::NB * 16 <= 64, "256 threads; a mask bit per accumulator");
  extern __shared__ __align__(16) uint8_t lds_g[];
  const TileId id = tile_id(p);
  const int t0 = id.tm * BM, n0 = id.tn * BN;
  const int nk = p.K / 32, k0 = nk * id.sp / p.splits, k1 = nk * (id.sp + 1) / p.splits;
  const uint8_t* xk = p.x + (int64_t)t0 * p.ldx + id.g * p.xg + (int64_t)k0 * kRow;
  const uint8_t* wk = group_weights(p, id.g, 4) + (int64_t)n0 * p.K * 4 + (int64_t)k0 * kRow;
  f32x16_t acc[L::MB][L::NB];
  tile_loop_f32<BM, BN, WM, WN, D>((lds_u8_t*)lds_g, xk, p.ldx, p.T - 1 - t0, wk, (int64_t)p.K * 4, p.N - 1 - n0, k1 - k0,
                                   acc);
  store_tile<F, YDT>((lds_u8_t*)lds_g, p, id.sp, id.g, t0, n0, acc);
  // a sum that is infinite or NaN may be so only because an operand has no split or the scaled sum no
  // room: it is taken from the fp32 MFMAs, a wave's block of 32 x 32 at a time, and stored again behind
  // the first store
  uint64_t bad = 0;
#pragma unroll
  for (int i = 0; i < L::MB * L::NB * 16; i++)
    bad |= (uint64_t)!(__builtin_fabsf(acc[i / 16 / L::NB][i / 16 % L::NB][i % 16]) < SMLA_INF) << i;
  if (__any(bad != 0)) {
    wait_vm(0);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave % (BM / WM), wn = wave / (BM / WM);
#pragma unroll 1
    for (int blk = 0; blk < L::MB * L::NB; blk++, bad >>= 16) {
      if (!__any((bad & 0xffffu) != 0)) continue;
      const f32x16_t f = block_f32<BM, BN, WM, WN>(xk, p.ldx, p.T - 1 - t0, wk, (int64_t)p.K * 4, p.N - 1 - n0, k1 - k0,
                                                   blk / L::NB, blk % L::NB);
      const int t = t0 + WM * wm + 32 * (blk / L::NB) + 4 * (lane >> 5), n = n0 + WN * wn + 32 * (blk % L::NB) + (lane & 31);
      const int64_t o = id.sp * p.split_stride + (int64_t)id.g * p.N + n;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int tr = t + 8 * (r >> 2) + (r & 3);
        if (!(bad >> r & 1) || tr >= p.T || n >= p.N) continue;
        if constexpr (YDT == SMLA_BF16) ((uint16_t*)p.y)[o + (int64_t)tr * p.ldy] = bf16_rne(f[r]);
        else ((float*)p.y)[o + (int64_t)tr * p.ldy] = f[r];
      }
    }
  }
}

// The q up projection of a prompt with its per-head epilogue (oracle/decode_engine.py:78-80): a tile is
// 128 tokens x one head of 512, so the head's RMS norm (weightless, v4mlx/mla.py:26-28) and the RoPE of
// its last 64 dims run on the accumulators and bf16 leaves.  As two launches the fp32 projection went
// out and came back (1.07 GB for 4096 tokens x 64 heads).  Two stages of (128 + 512) x 64 k fill the 160 KB
// of LDS.  4096 tokens, K 1024: 297-310 us repeated alone (the fp32 product 278-286 and the epilogue 276-280
// as two launches), about 350 in a layer, where the operands come from memory; 8 tiles per CU one after
// the other, each a K loop of 16 steps, then the norms, then 128 KB of rows, and nothing of one tile
// overlaps the next (the same product in 256 x 256 tiles with bf16 results takes 232-245).
struct HeadForm {
  static constexpr int BM = 128, BN = 512, WM = 64, WN = 128, D = 2;
};

__global__ __launch_bounds__(512) void gemm_heads_kernel(const RingArgs p, int64_t n_pos, float eps) {
  using namespace smla_gemm;
  using F = HeadForm;
  using L = Tile<F::BM, F::BN, F::WM, F::WN, F::D>;
  extern __shared__ __align__(16) uint8_t lds_g[];
  lds_u8_t* lds = (lds_u8_t*)lds_g;
  const TileId id = tile_id(p);
  const int t0 = id.tm * F::BM, n0 = id.tn * F::BN;
  f32x16_t acc[L::MB][L::NB];
  tile_loop<F::BM, F::BN, F::WM, F::WN, F::D>(lds, p.x + (int64_t)t0 * p.ldx, p.ldx, p.T - 1 - t0,
                                              p.w + (int64_t)n0 * p.K * 2, (int64_t)p.K * 2, F::BN - 1, p.K / 64, acc,
                                              [](int, lds_u8_t*, auto) {});
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave % 2, wn = wave / 2;
  // sums of squares: a row's 512 values sit in the 32 lanes of a half wave of four waves; the waves' sums
  // and then the rows' factors go through LDS past the region the stores use.  The epilogue is
  // row_epilogue_kernel's to the bit, so that a prompt's rows do not depend on its length: a thread there
  // holds channels 2t and 2t + 1 and a wave the 128 channels of a wave here, so pairs are summed first,
  // then threads 32, 16 (blocks of 32 channels), 8, 4, 2, 1 apart (16, 8, 4, 2 lanes here; row_ror:8 and :4
  // where the values repeat every 8 lanes), then the waves in order
  smla_attn::lds_f32_t* ss = (smla_attn::lds_f32_t*)(lds + 8 * F::WM * F::WN * 2);  // [4][128], then [128]
  static_assert(8 * F::WM * F::WN * 2 + 5 * 128 * 4 <= L::LDS, "the sums fit behind the staged rows");
  // the tile's rotations (128 rows of 32 cos and 32 sin) come in beside the sums, two 16-byte pieces of
  // each per thread, and are read from LDS (one wave gathering them itself: 443 against 369 us, profiled)
  f32x4_t rot[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int e = threadIdx.x + 512 * i;  // row e / 8, piece e mod 8
    int64_t ps = p.pos[min(t0 + (e >> 3), p.T - 1)];
    ps = ps < 0 ? 0 : ps >= n_pos ? n_pos - 1 : ps;
    rot[0][i] = *(const f32x4_t*)(p.cos_t + ps * 32 + 4 * (e & 7));
    rot[1][i] = *(const f32x4_t*)(p.sin_t + ps * 32 + 4 * (e & 7));
  }
  lds_barrier();  // every wave has read its last fragments
#pragma unroll
  for (int mb = 0; mb < L::MB; mb++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      float pr[4];
#pragma unroll
      for (int nb = 0; nb < L::NB; nb++) {
        const float v0 = dpp_f<0xA0>(acc[mb][nb][r]), v1 = dpp_f<0xF5>(acc[mb][nb][r]);
        pr[nb] = __builtin_fmaf(v0, v0, mul_rn_g(v1, v1));
      }
      float q = (pr[0] + pr[2]) + (pr[1] + pr[3]);
      const auto h = __builtin_amdgcn_permlane16_swap(__float_as_uint(q), __float_as_uint(q), false, false);
      q = __uint_as_float(h[0]) + __uint_as_float(h[1]);
      q += dpp_f<0x128>(q);
      q += dpp_f<0x124>(q);
      q += dpp_f<0x4E>(q);
      if ((lane & 31) == 0) ss[128 * wn + 64 * wm + 32 * mb + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)] = q;
    }
  smla_attn::lds_f32x4_t* cs = (smla_attn::lds_f32x4_t*)lds;  // cos then sin, [128][32]
#pragma unroll
  for (int i = 0; i < 2; i++) {
    cs[threadIdx.x + 512 * i] = rot[0][i];
    cs[1024 + threadIdx.x + 512 * i] = rot[1][i];
  }
  lds_barrier();
  if (threadIdx.x < 128) {
    const int i = threadIdx.x;
    ss[512 + i] = rsqrtf((((ss[i] + ss[128 + i]) + ss[256 + i]) + ss[384 + i]) / 512.f + eps);
  }
  lds_barrier();
#pragma unroll
  for (int mb = 0; mb < L::MB; mb++)
#pragma unroll
    for (int q4 = 0; q4 < 4; q4++) {
      const int row = 64 * wm + 32 * mb + 8 * q4 + 4 * (lane >> 5);
      const f32x4_t inv = *(smla_attn::lds_f32x4_t*)(ss + 512 + row);
#pragma unroll
      for (int j = 0; j < 4; j++) {
#pragma unroll
        for (int nb = 0; nb < L::NB; nb++) acc[mb][nb][4 * q4 + j] *= inv[j];
        if (wn == 3) {  // uniform: this wave holds dims 384 .. 511; pair i sits in lanes 2 i and 2 i + 1
          const smla_attn::lds_f32_t* cr = (const smla_attn::lds_f32_t*)lds + 32 * (row + j);
#pragma unroll
          for (int nb = 2; nb < 4; nb++) {
            const int i = 16 * (nb - 2) + ((lane & 31) >> 1);
            const float v = acc[mb][nb][4 * q4 + j], c = cr[i], s = cr[4096 + i];
            const float y0 = dpp_f<0xA0>(v), y1 = dpp_f<0xF5>(v);  // y0 c - y1 s, y0 s + y1 c
            acc[mb][nb][4 * q4 + j] = __builtin_fmaf(y0, lane & 1 ? s : c, mul_rn_g(y1, lane & 1 ? c : -s));
          }
        }
      }
    }
  store_tile<F, SMLA_BF16>(lds, p, 0, 0, t0, n0, acc);
}

// y[i] = part[0][i] + part[1][i] + ... in split order; V elements per thread
template <int YDT, int V>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const float* __restrict__ part, int splits, int64_t n,
                                                          void* __restrict__ y) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
  if (i >= n) return;
  typedef float vec_t __attribute__((ext_vector_type(V)));
  vec_t v[kMaxSplits];
#pragma unroll
  for (int s = 0; s < kMaxSplits; s++) v[s] = *(const vec_t*)(part + min(s, splits - 1) * n + i);
  vec_t sum = v[0];
#pragma unroll
  for (int s = 1; s < kMaxSplits; s++)
    if (s < splits) sum += v[s];
  if constexpr (YDT == SMLA_F32) {
    *(vec_t*)((float*)y + i) = sum;
  } else if constexpr (V == 4) {
    *(u32x2_t*)((uint16_t*)y + i) = (u32x2_t){pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3])};
  } else {
    ((uint16_t*)y)[i] = bf16_rne(sum[0]);
  }
}

// ---- the plan: tile form and splits for a bf16 product
struct RingPlan {
  int form, splits;
};

// whether the ring kernel takes the shape (else gemm_kernel): whole 64-k steps, enough of them for
// the shortest ring, and a tile's row offsets within 31 bits
bool ring_takes(int64_t ldx, int64_t K) {
  return K % 64 == 0 && K / 64 >= kFormD[3] && ldx % 8 == 0 && ldx * 2 * 256 < (1ll << 31) && K * 2 * 256 < (1ll << 31);
}

RingPlan ring_plan(int64_t T, int64_t G, int64_t N, int64_t K, bool may_split) {
  // A model of the launch in microseconds, its constants fitted to every (form, splits) of 154 products
  // (T 12 .. 4096 by the layer's weights, K 1024 .. 8192); the plan it picks is 1 % off the fastest on
  // average and 12 % at worst.  One 64-k step of a tile takes kIdle when few CUs run and kBusy when all
  // do (kPair for two co-resident 64 x 64 workgroups); the weights and tokens come in at 4.8 TB/s at
  // best; a split adds the reduce launch and its partial sums at 4.3 TB/s.
  constexpr double kIdle[kForms] = {0.24, 0.31, 0.57, 1.03}, kBusy[kForms] = {0.24, 0.53, 0.875, 1.47}, kPair = 0.36;
  constexpr double kEnds = 2.5, kReduce = 2.0, kHbm = 4.8e6, kPartial = 8 / 4.3e6;
  const int64_t cus = smla_num_cus(), nk = K / 64;
  const double in = 2.0 * K * G * (N + T) / kHbm;
  RingPlan best{3, 1};
  double bt = 1e30;
  for (int f = 0; f < kForms; f++) {
    const int64_t tiles = (T + kFormBM[f] - 1) / kFormBM[f] * G * ((N + kFormBN[f] - 1) / kFormBN[f]);
    const int64_t cap = f == 0 ? 2 * cus : cus;  // workgroups resident together
    for (int s = 1; s <= (may_split ? kMaxSplits : 1) && nk / s >= kFormD[f]; s++) {
      const int64_t rest = tiles * s % cap;
      double t = (double)(tiles * s / cap) * (f == 0 ? kPair : kBusy[f]);
      if (rest > cus) t += kPair;
      else if (rest > 0) t += kIdle[f] + (kBusy[f] - kIdle[f]) * (double)rest / (double)cus;
      t *= (double)((nk + s - 1) / s);
      t = kEnds + (t > in ? t : in);
      if (s > 1) t += kReduce + s * (double)T * G * N * kPartial;
      if (t < bt) bt = t, best = {f, s};
    }
  }
  return best;
}

// fp32 operands: the same with its own step times (32 k; the vector ALUs' splits and the MFMAs keep
// two co-resident workgroups of either form as long as one after the other)
bool f32_takes(int64_t ldx, int64_t K) {
  return K % 32 == 0 && K / 32 >= kFormF32D[1] && ldx * 4 * 128 < (1ll << 31) && K * 4 * 128 < (1ll << 31);
}

RingPlan f32_plan(int64_t T, int64_t G, int64_t N, int64_t K, bool may_split) {
  constexpr double kIdle[kFormsF32] = {0.5, 1.2}, kBusy[kFormsF32] = {0.6, 1.42};
  constexpr double kEnds = 2.5, kReduce = 2.0, kHbm = 4.8e6, kPartial = 8 / 4.3e6;
  const int64_t cus = smla_num_cus(), nk = K / 32;
  const double in = 4.0 * K * G * (N + T) / kHbm;
  RingPlan best{1, 1};
  double bt = 1e30;
  for (int f = 0; f < kFormsF32; f++) {
    const int64_t tiles = (T + kFormF32B[f] - 1) / kFormF32B[f] * G * ((N + kFormF32B[f] - 1) / kFormF32B[f]);
    for (int s = 1; s <= (may_split ? kMaxSplits : 1) && nk / s >= kFormF32D[f]; s++) {
      const int64_t rest = tiles * s % cus;
      double t = (double)(tiles * s / cus) * kBusy[f];
      if (rest > 0) t += kIdle[f] + (kBusy[f] - kIdle[f]) * (double)rest / (double)cus;
      t *= (double)((nk + s - 1) / s);
      t = kEnds + (t > in ? t : in);
      if (s > 1) t += kReduce + s * (double)T * G * N * kPartial;
      if (t < bt) bt = t, best = {f, s};
    }
  }
  return best;
}

template <int FORM>
int launch_ring(const RingArgs& a, int64_t wgs, bool rope, int y_dtype, hipStream_t st) {
  using F = Form<FORM>;
  using L = smla_gemm::Tile<F::BM, F::BN, F::WM, F::WN, F::D>;
  auto kern = rope ? (y_dtype == SMLA_BF16 ? gemm_ring_kernel<FORM, SMLA_BF16, true> : gemm_ring_kernel<FORM, SMLA_F32, true>)
                   : (y_dtype == SMLA_BF16 ? gemm_ring_kernel<FORM, SMLA_BF16, false> : gemm_ring_kernel<FORM, SMLA_F32, false>);
  // devices whose LDS limit is raised, one set per kernel (RoPE form x output type)
  static std::atomic<uint64_t> lds_attr[4] = {{0}, {0}, {0}, {0}};
  if (hipError_t e = smla_set_dynamic_lds((const void*)kern, L::LDS, lds_attr[(rope ? 2 : 0) + (y_dtype == SMLA_BF16 ? 1 : 0)]);
      e != hipSuccess)
    return (int)e;
  hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(L::NW * 64), L::LDS, st, a);
  SMLA_HIP_CHECK_LAUNCH();
  return SMLA_OK;
}

template <int FORM>
int launch_f32(const RingArgs& a, int64_t wgs, int y_dtype, hipStream_t st) {
  using F = FormF32<FORM>;
  using L = smla_gemm::Tile<F::BM, F::BN, F::WM, F::WN, F::D>;
  auto kern = y_dtype == SMLA_BF16 ? gemm_f32_kernel<FORM, SMLA_BF16> : gemm_f32_kernel<FORM, SMLA_F32>;
  static_assert(L::LDS <= 64 * 1024, "no raised LDS limit");
  hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(L::NW * 64), L::LDS, st, a);
  SMLA_HIP_CHECK_LAUNCH();
  return SMLA_OK;
}

}  // namespace

bool gemm_tiled_takes(int64_t G, int64_t K) { return ring_takes(G * K, K); }

int64_t gemm_tiled_workspace(int64_t T, int64_t G, int64_t N, int64_t K, bool f32_operands) {
  if (f32_operands ? !f32_takes(G * K, K) : !ring_takes(G * K, K)) return 0;
  const RingPlan p = f32_operands ? f32_plan(T, G, N, K, true) : ring_plan(T, G, N, K, true);
  return p.splits > 1 ? p.splits * T * G * N * (int64_t)sizeof(float) : 0;
}

// y [T, G*N] (row stride G*N) = grouped x [T, G*K] (row stride ldx elements) times w [G*N, K]^T.
// x and w both bf16 (f32_operands false) or both fp32; y bf16 or fp32.  With pos (bf16 only), inverse RoPE
// of the last 64 dims of every head_dim-wide head of x on load.  16-byte aligned rows (K % 8 for
// bf16, K % 4 for fp32).  ws: gemm_tiled_workspace bytes, 16-byte aligned, for the partial sums of a split
// K range, or less (null): the plan without splits.  With w2, G = 2 groups of weights w and w2 that both multiply
// the same x [T, K] (shapes the ring kernels take, else SMLA_E_UNSUPPORTED).  Returns SMLA_OK or a hipError_t.
int launch_gemm_tiled(const void* x, int64_t ldx, bool f32_operands, const void* w, int64_t T, int64_t G, int64_t N,
                      int64_t K, const int32_t* pos, const float* cos_t, const float* sin_t, int64_t head_dim,
                      void* y, int y_dtype, void* ws, size_t ws_bytes, hipStream_t st, const void* w2) {
  const int64_t ldy = G * N;
  if (f32_operands ? f32_takes(ldx, K) : ring_takes(ldx, K) && (!pos || head_dim % 64 == 0)) {
    const int64_t need = gemm_tiled_workspace(T, G, N, K, f32_operands);
    const bool split = need > 0 && usable_workspace(ws, ws_bytes, (size_t)need);
    const RingPlan p = f32_operands ? f32_plan(T, G, N, K, split) : ring_plan(T, G, N, K, split);
    const int bm = f32_operands ? kFormF32B[p.form] : kFormBM[p.form], bn = f32_operands ? bm : kFormBN[p.form];
    const int64_t nt = (T + bm - 1) / bm, nn = (N + bn - 1) / bn, wgs = nt * nn * G * p.splits;
    if (wgs > 0x7fffffff) return SMLA_E_UNSUPPORTED;
    const int64_t es = f32_operands ? 4 : 2;
    const uint32_t hs = pos ? (uint32_t)(head_dim / 64) : 1u;
    RingArgs a{(const uint8_t*)x, (const uint8_t*)w, (const uint8_t*)w2, ldx * es, w2 ? 0 : K * es, (int)T, (int)N, (int)K, (int)G, (int)nt,
               (int)nn, p.splits, pos, cos_t, sin_t, hs, hs > 1 ? (uint32_t)(((1ull << 32) + hs - 1) / hs) : 0u, (uint8_t*)(p.splits > 1 ? ws : y), ldy, T * ldy, 0, 1};
    const int odt = p.splits > 1 ? SMLA_F32 : y_dtype;
    if (!f32_operands && p.form == 3 && G % 2 == 0 && !w2 && a.ldx % 65536 == 0) a.pair = 2;
    a.vec = N % (odt == SMLA_BF16 ? 8 : 4) == 0 && ((uintptr_t)a.y & 15) == 0;
    const int rc = f32_operands  ? (p.form == 0 ? launch_f32<0>(a, wgs, odt, st) : launch_f32<1>(a, wgs, odt, st))
                   : p.form == 0 ? launch_ring<0>(a, wgs, pos != nullptr, odt, st)
                   : p.form == 1 ? launch_ring<1>(a, wgs, pos != nullptr, odt, st)
                   : p.form == 2 ? launch_ring<2>(a, wgs, pos != nullptr, odt, st)
                                 : launch_ring<3>(a, wgs, pos != nullptr, odt, st);
    if (rc != SMLA_OK || p.splits == 1) return rc;
    const int64_t n = T * ldy;
    const bool v4 = n % 4 == 0;
    const dim3 grid((unsigned)((n / (v4 ? 4 : 1) + 255) / 256));
    auto red = y_dtype == SMLA_BF16 ? (v4 ? gemm_reduce_kernel<SMLA_BF16, 4> : gemm_reduce_kernel<SMLA_BF16, 1>)
                                    : (v4 ? gemm_reduce_kernel<SMLA_F32, 4> : gemm_reduce_kernel<SMLA_F32, 1>);
    hipLaunchKernelGGL(red, grid, dim3(256), 0, st, (const float*)ws, p.splits, n, y);
    SMLA_HIP_CHECK_LAUNCH();
    return SMLA_OK;
  }
  if (w2) return SMLA_E_UNSUPPORTED;
  const int64_t ntn = (N + kBN - 1) / kBN;
  const dim3 grid((unsigned)(ntn * G), (unsigned)((T + kBM - 1) / kBM)), blk(256);
#define SMLA_GEMM(BF, YD, RP)                                                                                   \
  hipLaunchKernelGGL((gemm_kernel<BF, YD, RP>), grid, blk, 0, st, (const uint8_t*)x, ldx, (const uint8_t*)w,   \
                     (int)T, (int)N, (int)K, (int)ntn, pos, cos_t, sin_t, (int)head_dim, y, ldy)
  if (f32_operands) {
    if (y_dtype == SMLA_BF16) SMLA_GEMM(false, SMLA_BF16, false);
    else SMLA_GEMM(false, SMLA_F32, false);
  } else if (pos) {
    if (y_dtype == SMLA_BF16) SMLA_GEMM(true, SMLA_BF16, true);
    else SMLA_GEMM(true, SMLA_F32, true);
  } else {
    if (y_dtype == SMLA_BF16) SMLA_GEMM(true, SMLA_BF16, false);
    else SMLA_GEMM(true, SMLA_F32, false);
  }
#undef SMLA_GEMM
  SMLA_HIP_CHECK_LAUNCH();
  return SMLA_OK;
}

// out [T, heads, 512] bf16 = per-head RMS norm (eps) and RoPE of the last 64 dims (at pos) of x [T, K] times
// w [heads * 512, K]^T, bf16 operands.  K a multiple of 64 from 128.  Returns SMLA_OK or a hipError_t.
int launch_gemm_heads(const void* x, const void* w, int64_t T, int64_t heads, int64_t K, const int32_t* pos,
                      const float* cos_t, const float* sin_t, int64_t n_pos, float eps, void* out, hipStream_t st) {
  using F = HeadForm;
  using L = smla_gemm::Tile<F::BM, F::BN, F::WM, F::WN, F::D>;
  if (K % 64 != 0 || K / 64 < F::D || K * 2 * F::BN >= (1ll << 31) || heads * 512 > 0x7fffffff) return SMLA_E_UNSUPPORTED;
  const int64_t nt = (T + F::BM - 1) / F::BM, wgs = nt * heads;
  if (wgs > 0x7fffffff) return SMLA_E_UNSUPPORTED;
  RingArgs a{(const uint8_t*)x, (const uint8_t*)w, nullptr, K * 2, 0, (int)T, (int)(heads * 512), (int)K, 1, (int)nt,
             (int)heads, 1, pos, cos_t, sin_t, 8, 0, (uint8_t*)out, heads * 512, 0, 1, 1};
  static std::atomic<uint64_t> lds_attr{0};
  if (hipError_t e = smla_set_dynamic_lds((const void*)gemm_heads_kernel, L::LDS, lds_attr); e != hipSuccess) return (int)e;
  hipLaunchKernelGGL(gemm_heads_kernel, dim3((unsigned)wgs), dim3(L::NW * 64), L::LDS, st, a, n_pos, eps);
  SMLA_HIP_CHECK_LAUNCH();
  return SMLA_OK;
}

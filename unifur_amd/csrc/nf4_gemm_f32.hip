// nf4_gemm_f32.hip -- f32 GEMM over an NF4 weight dequantized exactly: the
// linear and its backward for f32 activations (and f32 dY) at batch sizes
// past the skinny kernel's, on the bf16 matrix cores.
//
// Forward: Y[M, N] = X[M, K] deq(W)[K, N] (+ bias) (+ scaling (X A) B), the
// reference's arithmetic for Nf4Linear::forward / QloraLinear::forward
// (src/qwennet.rs:238-241, :325-345): the weight value is
// NF4_LEVELS[c] * scale in f32 (src/quantize.rs:362, the reference's
// dequantized value bit for bit) and the sums are f32.  Backward (TRANS):
// dX[M, d_in] = dY[M, d_out] deq(W)^T (+ scaling (dY B^T) A^T), the autodiff
// of the same function with the base weight frozen (src/qwentrain.rs:421-470).
// No weight-sized scratch: each workgroup dequantizes the W tiles it needs.
//
// Products.  Each f32 operand is cut into three bf16 terms, each the nearest
// to what the ones before leave, v = hi + mid + lo exactly, and the product is
// six bf16 products (hi hi, hi mid, mid hi, mid mid, hi lo, lo hi),
// accumulated in f32 by v_mfma_f32_32x32x16_bf16.  mid is at most 2^-8 and lo
// 2^-17 of a value's power of two, so that what is left out is under 2^-24 of
// a product, 0.6e-8 rms, of either sign (terms cut by truncation leave 2^-21,
// always of the product's sign).  hi hi has an accumulator of its own, the
// other five share a second, and the two are added once at the end: added to
// the sum of hi hi, the small products would fall below half a unit of it once
// it is large and be lost, towards zero.  Six of these take 192 matrix-core
// cycles per 32 x 32 x 16 where v_mfma_f32_32x32x2f32 takes 512, and round the
// large accumulator once instead of eight times.  Relative 2-norm error
// against float64, 512 rows -> 8320 (one slab), of the f32 instruction and
// now, for N(0, 1) activations and for operands of one sign:
//   d_in 4      3.9e-8 2.6e-8   3.5e-8 2.6e-8
//   d_in 64     1.4e-7 4.3e-8   1.1e-7 4.5e-8
//   d_in 4096   1.1e-6 3.7e-7   8.9e-7 3.3e-7
//   d_in 11008  1.8e-6 6.5e-7   1.5e-6 5.4e-7
// (one product a sum: 2.53e-8 and 2.59e-8, at most 2^-24 and 2^-23.3).
// A value's terms are bf16 numbers down to the subnormals because X is cut
// at 2^24 times its size (kXScale).  Infinities and NaN, a scaled value or sum
// past the largest f32 and weights of the smallest scales have no such split:
// a wave with a sum that is not finite computes its tiles again with the f32
// instruction, from the same operands (exact_tile).  A bf16 X (XBF) is
// its own hi term, so its products with the weight's three terms are exact and
// there are three of them: the path of bf16 batches whose shape the bf16
// kernels do not take, where the weight stays the exact f32 one.
//
// What bounds it (counters in profiles/mfma_utilisation_prefill.txt): 2048 x
// 4096 -> 4096 in 370 us (601 with the f32 instruction) is 1.1 PFLOP/s of bf16
// products, what the library's large bf16 product reaches here, with the matrix
// cores busy 51 % of the cycles of a clock that falls to 2.1 GHz (its own: 50 %).
// 500 rows take 110 us (366 with the f32 instruction, whose 128 tiles left half
// the CUs idle; now four slabs of K): 0.9 PFLOP/s, busy 42 %; the slabs'
// partials, 33 MB written and read, take a 7 us reduction launch and part of the
// kernel's time, and the weight is decoded and cut once per 128 rows.  The
// second accumulator costs registers (134 -> 205 at 128 rows, two workgroups a
// CU) but no time: 2048 rows 380 us with one and 370 with two, 500 rows 112
// and 110, 1024 x 4096 -> 11008 606 and 577, 64 x 4096 -> 11008 52 and 51.
//
// Tiling.  A 256-thread workgroup owns 32 RT rows x 128 columns, K in steps
// of 32; each of its four waves owns 32 columns of all the rows, so that a
// weight value is dequantized and split once per workgroup, in the registers
// of the lane that feeds it to the MFMAs: a wave loads its 32 x 32 codes as 8
// bytes a lane and ds_read_b64_tr_b4 (four 16 x 16 nibble transposes) gives
// each lane 16 consecutive k of its column (TRANS: a lane's 8 bytes are
// already 16 consecutive k of its column).  X is split once per workgroup
// into three bf16 planes in LDS, two buffers, chunks swizzled so that eight
// lanes' 16-byte reads meet distinct banks; the next step's X and the codes
// two steps ahead are in flight during a step; one barrier per step.
#include "nf4_gemm_f32.hpp"

#include <algorithm>

#include "nf4_gemm.hpp"

namespace unifur {
namespace {

constexpr int kFN = 128, kFK = 32;
constexpr int kFThreads = 256;

// LDS of a workgroup of RT row tiles (byte offsets).
template <int RT>
struct FSmem {
  static constexpr int kPlane = RT * 32 * kFK * 2;  // one bf16 plane of the X tile
  static constexpr int kBuf = 3 * kPlane;
  static constexpr int kCodes = 2 * kBuf;           // 512 bytes a wave
  static constexpr int kLut = kCodes + 4 * 512;     // byte LUT: 256 x {level lo, level hi}
  static constexpr int kDq = kLut + 256 * 8;        // DQ scales: 256 x f32
  static constexpr int kBytes = kDq + 256 * 4;
};

// The terms of every f32 value have to be bf16 numbers.  A bf16 number has no
// bits below 2^-133, and an f32 value under 2^-110 has some, so X is
// multiplied by 2^24 before it is cut (exact; the sums are divided by it
// again, and one that overflows for it is not finite: exact_tile).  A weight
// value's scale under 2^-99, whose terms could be as small, is taken as NaN,
// which leads there too.
constexpr float kXScale = 16777216.0f;
constexpr uint32_t kTinyScale = (127u - 99u) << 23;

__device__ __forceinline__ uint32_t fbits(float v) { return __float_as_uint(v); }

__device__ __forceinline__ float dq_scale(int q, float scale_of_scales) { return ((float)q / 255.0f) * scale_of_scales; }

__device__ __forceinline__ float no_tiny_scale(float s) {
  return (fbits(s) & 0x7fffffffu) - 1u < kTinyScale - 1u ? __uint_as_float(0x7fc00000u) : s;
}

// Two values' bf16 terms, rounded to nearest, as one dword (a in the low
// half), and what is left of each (exact: at most half the term's last place).
// No contraction: fused with the product level * scale that a weight value
// comes from, the subtraction would leave the rest of the unrounded product,
// and the terms would not be those of the f32 value.
__device__ __forceinline__ uint32_t cut_pair(float& a, float& b) {
#pragma clang fp contract(off)
  const uint32_t pk = pack_bf16x2(a, b);
  a -= bf16_bits_to_f32(pk);
  b -= __uint_as_float(pk & 0xffff0000u);
  return pk;
}

// Eight values -> their hi, mid and lo planes, eight bf16 each (what is left
// after two terms has at most eight significant bits).
__device__ __forceinline__ void split8(float (&v)[8], u32x4 (&p)[3]) {
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int e = 0; e < 4; ++e) p[q][e] = cut_pair(v[2 * e], v[2 * e + 1]);
#pragma unroll
  for (int e = 0; e < 4; ++e) p[2][e] = perm_b32(fbits(v[2 * e + 1]), fbits(v[2 * e]), 0x07060302u);
}

// One step's codes of a lane: the 8 bytes it stages or uses, their block
// scale (f32 bits or the u8 DQ code; a row past K has scale zero).
struct FCodes {
  u32x2 code;
  uint32_t scale;
  bool live;
};

// Where a lane reads its codes.  Forward: row k = 32 s + 16 (l / 32) + l % 16
// of the wave's stripe l / 16 % 2 (the 16 columns from col).  TRANS: the 16
// columns 32 s + 16 (l / 32) of weight row n.
template <bool STRIPED, bool TRANS>
struct FLane {
  int row, col;  // forward: row within the step, first column; TRANS: weight row, column within the step
  __device__ __forceinline__ FLane(const F32GemmArgs& g, int n0, int lane) {
    if constexpr (TRANS) {
      row = min(n0 + (lane & 31), g.N - 1);
      col = 16 * (lane >> 5);
    } else {
      row = 16 * (lane >> 5) + (lane & 15);
      col = min(n0, g.N - 32) + 16 * ((lane >> 4) & 1);
    }
  }
};

template <bool DQ, bool STRIPED, bool TRANS>
__device__ __forceinline__ FCodes load_codes(const F32GemmArgs& g, const FLane<STRIPED, TRANS>& l, int k0) {
  FCodes c;
  const int wr = TRANS ? l.row : min(k0 + l.row, g.K - 1), wc = TRANS ? k0 + l.col : l.col;
  const int wrows = TRANS ? g.N : g.K, wcols = TRANS ? g.K : g.N;  // the stored weight's d_in, d_out
  c.live = TRANS || k0 + l.row < g.K;
  const size_t at = STRIPED ? ((size_t)(wc / 16) * wrows + wr) * 8 : (size_t)wr * (wcols / 2) + wc / 2;
  const size_t blk = STRIPED ? (size_t)(wc / kBlock) * wrows + wr : (size_t)wr * (wcols / kBlock) + wc / kBlock;
  c.code = *reinterpret_cast<const u32x2*>(g.packed + at);
  c.scale = DQ ? (uint32_t)g.scales.dq_codes[blk] : fbits(g.scales.absmax[blk]);
  return c;
}

// The X values of a step this thread stages: 4 RT consecutive k of one row.
// Past the end of the row its last ones again: they meet weights of zero.
template <int RT, bool XBF>
struct FX {
  f32x4 v[XBF ? RT / 2 : RT];  // XBF: eight bf16 each
};

template <int RT, bool XBF>
__device__ __forceinline__ FX<RT, XBF> load_x(const F32GemmArgs& g, int m0, int k0, int tid) {
  constexpr int kPerRow = 8 / RT, kRun = XBF ? 8 : 4;  // threads a row; k of a load (K is a multiple)
  FX<RT, XBF> x;
  const size_t at = (size_t)min(m0 + tid / kPerRow, g.M - 1) * g.K;
#pragma unroll
  for (int q = 0; q < 4 * RT / kRun; ++q) {
    const size_t i = at + min(k0 + 4 * RT * (tid % kPerRow) + kRun * q, g.K - kRun);
    x.v[q] = XBF ? *reinterpret_cast<const f32x4*>(static_cast<const uint16_t*>(g.x) + i)
                 : *reinterpret_cast<const f32x4*>(static_cast<const float*>(g.x) + i);
  }
  return x;
}

// 16-byte chunk c (8 k) of row r of a plane: rows are 64 bytes, the chunk is
// XORed with the row's group of four, so that eight consecutive rows (or four
// rows x two chunks) cover 128 bytes' worth of distinct banks.
__device__ __forceinline__ uint32_t x_at(int base, int r, int c) {
  return (uint32_t)(base + r * (kFK * 2) + ((c ^ ((r >> 2) & 3)) * 16));
}

template <int RT, bool XBF>
__device__ __forceinline__ void store_x(const FX<RT, XBF>& x, int buf, int tid) {
  constexpr int kPerRow = 8 / RT;
  const int r = tid / kPerRow, c0 = (RT / 2) * (tid % kPerRow);
  if constexpr (XBF) {
#pragma unroll
    for (int c = 0; c < RT / 2; ++c)
      *reinterpret_cast<lds_u32x4*>((size_t)x_at(buf * FSmem<RT>::kBuf, r, c0 + c)) =
          __builtin_bit_cast(u32x4, x.v[c]);
  } else {
#pragma unroll
    for (int c = 0; c < RT / 2; ++c) {
      float v[8] = {x.v[2 * c].x,     x.v[2 * c].y,     x.v[2 * c].z,     x.v[2 * c].w,
                    x.v[2 * c + 1].x, x.v[2 * c + 1].y, x.v[2 * c + 1].z, x.v[2 * c + 1].w};
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] *= kXScale;
      u32x4 p[3];
      split8(v, p);
#pragma unroll
      for (int q = 0; q < 3; ++q)
        *reinterpret_cast<lds_u32x4*>((size_t)x_at(buf * FSmem<RT>::kBuf + q * FSmem<RT>::kPlane, r, c0 + c)) = p[q];
    }
  }
}

// acc[i] (+)= the wave's tiles over [kb, ke) with the f32 instruction: the
// products of infinities and NaN, for a tile whose split sums are not finite.
template <int RT, bool DQ, bool STRIPED, bool TRANS, bool XBF>
__device__ void exact_tile(f32x16 (&acc)[RT], const F32GemmArgs& g, const unsigned char* smem, int m0, int n, int kb,
                           int ke, int lane) {
  const float* lut = reinterpret_cast<const float*>(smem + FSmem<RT>::kLut);  // lut[2 c] = level c, c < 16
  const float sos = DQ ? *g.scales.scale_of_scales : 0.0f;
#pragma unroll
  for (int i = 0; i < RT; ++i) acc[i] = f32x16{};
  const int nn = min(n, g.N - 1);
  const int wrows = TRANS ? g.N : g.K, wcols = TRANS ? g.K : g.N;
#pragma unroll 4
  for (int k0 = kb; k0 < ke; k0 += 2) {
    const int k = k0 + (lane >> 5), kc = min(k, g.K - 1);
    const bool in = k < ke;
    const int wr = TRANS ? nn : kc, wc = TRANS ? kc : nn;
    const size_t at =
        STRIPED ? ((size_t)(wc / 16) * wrows + wr) * 8 + (wc & 15) / 2 : (size_t)wr * (wcols / 2) + wc / 2;
    const size_t blk = STRIPED ? (size_t)(wc / kBlock) * wrows + wr : (size_t)wr * (wcols / kBlock) + wc / kBlock;
    const int code = (g.packed[at] >> (4 * (wc & 1))) & 15;
    const float s = DQ ? dq_scale(g.scales.dq_codes[blk], sos) : g.scales.absmax[blk];
    const float w = in ? lut[2 * code] * s : 0.0f;
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const size_t at_x = (size_t)min(m0 + 32 * i + (lane & 31), g.M - 1) * g.K + kc;
      const float v = XBF ? bf16_bits_to_f32(static_cast<const uint16_t*>(g.x)[at_x]) : static_cast<const float*>(g.x)[at_x];
      const float x = in ? v : 0.0f;
      acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, w, acc[i], 0, 0, 0);
    }
  }
}

// acc = the wave's sums over the slab [kb, ke), the adapter's term with them
// in the first slab.
template <int RT, bool DQ, bool STRIPED, bool TRANS, bool XBF>
__device__ __forceinline__ void slab_sums(f32x16 (&acc)[RT], const F32GemmArgs& g, const unsigned char* smem, int m0,
                                          int n0, int kb, int ke, int tid, int wave) {
  using S = FSmem<RT>;
  const int lane = tid & 63, h = lane >> 5, r32 = lane & 31;
  const float* dq_lut = reinterpret_cast<const float*>(smem + S::kDq);
  const FLane<STRIPED, TRANS> fl(g, n0, lane);
  const int last = (ke - 1) / kFK * kFK;  // code loads past the slab stay on its last step
  FX<RT, XBF> x = load_x<RT, XBF>(g, m0, kb, tid);
  FCodes c0 = load_codes<DQ, STRIPED, TRANS>(g, fl, kb);
  FCodes c1 = load_codes<DQ, STRIPED, TRANS>(g, fl, min(kb + kFK, last));
  store_x<RT, XBF>(x, 0, tid);
  __syncthreads();  // X of the first step, and the LUTs

  f32x16 low[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) acc[i] = low[i] = f32x16{};
  const uint32_t stage = (uint32_t)(S::kCodes + wave * 512 + lane * 8);
  int buf = 0;
  for (int k0 = kb; k0 < ke; k0 += kFK, buf ^= 1) {
    const bool more = k0 + kFK < ke;
    if (more) x = load_x<RT, XBF>(g, m0, k0 + kFK, tid);
    const FCodes c2 = load_codes<DQ, STRIPED, TRANS>(g, fl, min(k0 + 2 * kFK, last));

    // the step's weight: 16 codes of this lane's column, k = 16 h + 0 .. 15
    u32x2 nib = c0.code;
    if constexpr (!TRANS) {
      *reinterpret_cast<lds_u32x2*>((size_t)stage) = c0.code;
      nib = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr4_b64_v2i32(reinterpret_cast<lds_v2i32*>((size_t)stage)));
    }
    float s = DQ ? dq_lut[c0.scale & 0xffu] : __uint_as_float(c0.scale);
    if constexpr (!DQ) s = no_tiny_scale(s);
    s = c0.live ? s : 0.0f;
    float sc[16];
    if constexpr (!TRANS) row_lanes<0>(s, sc);  // row 16 h + j's scale sits in lane 16 (l / 16) + j
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      float w[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t byte = (nib[d] >> (8 * j)) & 0xffu;
        const f32x2 l = *reinterpret_cast<lds_f32x2_c*>((size_t)(S::kLut + byte * 8));
        w[2 * j] = l.x * (TRANS ? s : sc[8 * d + 2 * j]);
        w[2 * j + 1] = l.y * (TRANS ? s : sc[8 * d + 2 * j + 1]);
      }
      u32x4 wp[3];
      split8(w, wp);
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        u32x4 xp[3];
#pragma unroll
        for (int q = 0; q < (XBF ? 1 : 3); ++q)
          xp[q] = *reinterpret_cast<lds_u32x4*>((size_t)x_at(buf * S::kBuf + q * S::kPlane, 32 * i + r32, 2 * h + d));
        const auto mul = [&](f32x16& sum, int a, int c) {
          sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, xp[a]),
                                                        __builtin_bit_cast(bf16x8_t, wp[c]), sum, 0, 0, 0);
        };
        mul(acc[i], 0, 0);
        if constexpr (!XBF) mul(low[i], 2, 0);
        mul(low[i], 0, 2);
        if constexpr (!XBF) {
          mul(low[i], 1, 1);
          mul(low[i], 1, 0);
        }
        mul(low[i], 0, 1);
      }
    }
    c0 = c1;
    c1 = c2;
    if (more) store_x<RT, XBF>(x, buf ^ 1, tid);
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] += low[i][r];
  // a sum that is not finite: the wave's tiles again, with the f32
  // instruction (the wave as one: an MFMA reads every lane's operands)
  bool finite = true;
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) finite = finite && (fbits(acc[i][r]) & 0x7f800000u) != 0x7f800000u;
  if (__any(!finite)) {
    exact_tile<RT, DQ, STRIPED, TRANS, XBF>(acc, g, smem, m0, n0 + r32, kb, ke, lane);
  } else if constexpr (!XBF) {
#pragma unroll
    for (int i = 0; i < RT; ++i) acc[i] *= 1.0f / kXScale;
  }

  // the adapter, in the first slab's sums: acc += (xa scaling) B over the
  // rank; xa [M][lora_ld] f32 and B element (j, n) at lora_b[j sbj + n sbn].
  // Four steps' factors are loaded together, from clamped places and zeroed
  // past the rank: one step at a time waits out a latency every two ranks
  // (4096 -> 4096, rank 64, 70 / 500 rows 76 / 161 us so, 66 / 153 with four;
  // 120 -> 64, 300 rows 45 and 43)
  if (g.lora_xa && kb == 0) {
    const float* bcol = g.lora_b + (size_t)min(n0 + r32, g.N - 1) * g.lora_sbn;
    for (int j0 = 0; j0 < g.lora_rank; j0 += 8) {
      float av[4][RT], bv[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = min(j0 + 2 * q + h, g.lora_rank - 1);
        bv[q] = bcol[(size_t)j * g.lora_sbj];
#pragma unroll
        for (int i = 0; i < RT; ++i)
          av[q][i] = g.lora_xa[(size_t)min(m0 + 32 * i + r32, g.M - 1) * g.lora_ld + j];
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const bool in = j0 + 2 * q + h < g.lora_rank;
        const float bb = in ? bv[q] : 0.0f;
#pragma unroll
        for (int i = 0; i < RT; ++i)
          acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? av[q][i] * g.lora_scaling : 0.0f, bb, acc[i], 0, 0, 0);
      }
    }
  }
}

// One workgroup a (tile, slab), or with SERIAL one a tile that takes the
// slabs in turn and adds their sums in the order of the reduction: a call
// gives the same bits with and without room for the partials.  SERIAL has at
// most 256 workgroups (two slabs or more of kF32Grid), so one a CU is enough
// and its third set of sums stays in registers.
template <int RT, bool DQ, bool STRIPED, bool TRANS, bool XBF, bool SERIAL>
__global__ __launch_bounds__(kFThreads, SERIAL && RT == 4 ? 1 : 2) void gemm_f32_kernel(F32GemmArgs g) {
  using S = FSmem<RT>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // XCD-aware order: workgroup b runs on XCD b % 8; each XCD takes a
  // contiguous run of (slab, tile) in row-major (m, n) tile order (shared X rows)
  const int nb = gridDim.x, b = blockIdx.x;
  const int u = (nb % 8 == 0) ? (b % 8) * (nb / 8) + b / 8 : b;
  const int tiles_n = (g.N + kFN - 1) / kFN, tiles = SERIAL ? nb : nb / g.k_splits;
  const int slab = SERIAL ? 0 : u / tiles, t = SERIAL ? u : u % tiles;
  const int m0 = (t / tiles_n) * (32 * RT), n0 = (t % tiles_n) * kFN + 32 * wave;

  {
    float* lut = reinterpret_cast<float*>(smem + S::kLut);
    lut[2 * tid] = level(tid & 15);
    lut[2 * tid + 1] = level(tid >> 4);
    if constexpr (DQ)
      reinterpret_cast<float*>(smem + S::kDq)[tid] = no_tiny_scale(dq_scale(tid, *g.scales.scale_of_scales));
    __syncthreads();
  }
  f32x16 acc[RT];
  const int kb = slab * g.k_slab;
  slab_sums<RT, DQ, STRIPED, TRANS, XBF>(acc, g, smem, m0, n0, kb, min(g.K, kb + g.k_slab), tid, wave);
  if constexpr (SERIAL) {
    for (int k1 = g.k_slab; k1 < g.K; k1 += g.k_slab) {
      f32x16 part[RT];
      slab_sums<RT, DQ, STRIPED, TRANS, XBF>(part, g, smem, m0, n0, k1, min(g.K, k1 + g.k_slab), tid, wave);
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] += part[i][r];
    }
  }
  // acc[i][4 a + e] is C[row 32 i + 8 a + 4 (lane / 32) + e][col lane % 32]:
  // each store instruction writes 32 consecutive columns of two rows
  const int n = n0 + (lane & 31);
  if (n >= g.N) return;
  const bool parts = !SERIAL && g.k_splits > 1;
  const float bias = g.bias && !parts ? g.bias[n] : 0.0f;
  const size_t base = (size_t)slab * (size_t)g.M * (size_t)g.N;
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = m0 + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
      if (m >= g.M) continue;
      const size_t o = (size_t)m * g.N + n;
      const float y = g.bias && !parts ? acc[i][r] + bias : acc[i][r];
      if (parts)
        g.partials[base + o] = y;
      else if (g.y_bf16)
        reinterpret_cast<uint16_t*>(g.y)[o] = (uint16_t)(pack_bf16x2(y, 0.0f) & 0xffffu);
      else
        reinterpret_cast<float*>(g.y)[o] = y;
    }
}

// Row tiles of a workgroup: 128 rows, or 64 where a batch has no more (a
// 4096 / 11008 SwiGLU block at 64 rows: 170 us, against 269 at 128).
int row_tiles(int M) { return M <= 64 ? 2 : 4; }

template <int RT, bool DQ, bool STRIPED, bool TRANS, bool XBF>
hipError_t launch_f(const F32GemmArgs& g, hipStream_t stream) {
  const int tiles = ((g.M + 32 * RT - 1) / (32 * RT)) * ((g.N + kFN - 1) / kFN);
  static_assert(FSmem<RT>::kBytes <= 64 << 10, "more LDS needs the attribute");
  if (g.k_splits > 1 && !g.partials)
    gemm_f32_kernel<RT, DQ, STRIPED, TRANS, XBF, true><<<tiles, kFThreads, FSmem<RT>::kBytes, stream>>>(g);
  else
    gemm_f32_kernel<RT, DQ, STRIPED, TRANS, XBF, false><<<tiles * g.k_splits, kFThreads, FSmem<RT>::kBytes, stream>>>(g);
  return hipGetLastError();
}

}  // namespace

bool gemm_f32_mfma_supported(int M, int Kr, int N, int w_d_out, const void* x, bool x_bf16) {
  // the reduction dim a multiple of 4, or 8 for bf16 (whole 16-byte loads), the stored
  // weight's d_out of 64 (whole blocks along a row), 16-byte aligned X
  return M > 0 && Kr > 0 && N > 0 && Kr % (x_bf16 ? 8 : 4) == 0 && w_d_out % 64 == 0 &&
         (reinterpret_cast<uintptr_t>(x) & 15u) == 0 && (((uint64_t)M + 128) * (uint64_t)(Kr) < (1ull << 40));
}

// The slabs fill two workgroups a CU: 512 workgroups measured best, 4096 ->
// 4096 at 65 / 256 / 512 rows 41 / 66 / 109 us against 44 / 85 / 147 aiming
// for 256 and 41 / 81 / 131 for 768.
int gemm_f32_splits(int M, int Kr, int N) {
  if (N % 4 != 0) return 1;  // the reduction takes four columns at a time
  const int rows = 32 * row_tiles(M);
  const int64_t tiles = (int64_t)((M + rows - 1) / rows) * ((N + kFN - 1) / kFN);
  // a slab of at least eight steps, and partials no larger than three
  // quarters of the f32 weight this kernel does without
  const int64_t want = kF32Grid / tiles, most = Kr / (8 * kFK), room = 3 * (int64_t)Kr / (4 * (int64_t)M);
  return (int)std::max<int64_t>(1, std::min<int64_t>({want, most, room, 16}));
}

hipError_t launch_gemm_f32_mfma(F32GemmArgs g, bool dq, bool striped, bool trans, hipStream_t stream) {
  // the slabs are the shape's, whether or not there are partials for them
  const int steps = (g.K + kFK - 1) / kFK, want = gemm_f32_splits(g.M, g.K, g.N);
  g.k_slab = (steps + want - 1) / want * kFK;
  g.k_splits = (g.K + g.k_slab - 1) / g.k_slab;  // no empty slab
  if (g.k_splits > 1 && g.partials &&
      ((reinterpret_cast<uintptr_t>(g.y) & 15u) || (reinterpret_cast<uintptr_t>(g.bias) & 15u)))
    return hipErrorInvalidValue;
  hipError_t e = hipErrorInvalidValue;
  const int rt = row_tiles(g.M);
#define UNIFUR_F32_CASE(R, D, S, T, B) \
  if (rt == R && dq == D && striped == S && trans == T && (g.x_bf16 != 0) == B) e = launch_f<R, D, S, T, B>(g, stream);
#define UNIFUR_F32_CASES(R, T, B) \
  UNIFUR_F32_CASE(R, true, true, T, B) UNIFUR_F32_CASE(R, true, false, T, B) \
  UNIFUR_F32_CASE(R, false, true, T, B) UNIFUR_F32_CASE(R, false, false, T, B)
  UNIFUR_F32_CASES(2, false, false)
  UNIFUR_F32_CASES(4, false, false)
  UNIFUR_F32_CASES(2, false, true)
  UNIFUR_F32_CASES(4, false, true)
  UNIFUR_F32_CASES(2, true, false)
  UNIFUR_F32_CASES(4, true, false)
#undef UNIFUR_F32_CASES
#undef UNIFUR_F32_CASE
  if (e != hipSuccess || g.k_splits == 1 || !g.partials) return e;
  return launch_splitk_reduce(g.partials, g.k_splits, g.M, g.N, g.bias, g.y, g.y_bf16 != 0, stream);
}

}  // namespace unifur

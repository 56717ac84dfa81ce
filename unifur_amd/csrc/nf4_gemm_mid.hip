// nf4_gemm_mid.hip -- bf16 GEMM over a striped NF4 weight for batches just
// past the skinny kernel's: Y[M, N] = X[M, K] deq(W)[K, N] (+ bias)
// (+ scaling (X A) B) (Nf4Linear::forward and QloraLinear::forward,
// src/qwennet.rs:238-241, :325-345).
//
// The weight operand is bf16(NF4_LEVELS[c] * scale), the f32 product rounded
// once, as in the other bf16 kernels; products accumulate in f32
// (v_mfma_f32_32x32x16_bf16).  The adapter's term is f32 throughout.
//
// Tiling.  A 256-thread workgroup owns 96 or 128 rows x 128 columns, K in
// steps of 64; each of its four waves owns 32 columns of all the rows.  A wave
// dequantizes its own columns straight into the registers that feed the MFMAs
// -- no weight tile in LDS, no producer waves: it loads 32 x 32 codes as 8
// bytes a lane, ds_read_b64_tr_b4 (four 16 x 16 nibble transposes) gives each
// lane 16 consecutive k of its column, a byte of two codes is one lookup of
// two f32 levels (eight interleaved copies of the table, lane % 8 picks one),
// times the rows' scales by DPP broadcast.  X goes through LDS once per
// workgroup, two buffers of 128-byte rows whose 16-byte chunks are swizzled
// (x_swizzle).  d_in is split over workgroups so that the grid reaches about
// one a CU.
//
// What it is for: expanding a large weight to bf16 for a library product costs
// the same whatever the rows, 31 us in all over 4096 x 4096 and 52 over
// 11008 x 4096 at 100 rows; this kernel and its reduction take 18 and 24
// (gemm_mid_wanted has the rest).
//
// What bounds it: one wave a SIMD issues its VALU, LDS and MFMA work one after
// the other (counters at 128 x 4096 -> 32768, 54 us, in
// profiles/mfma_utilisation_prefill.txt: matrix cores busy 25 % of the cycles,
// VALU 28 %, LDS 16 %, waiting 25 %), 2050 cycles a step where the MFMAs need
// 512; deeper prefetch and LDS reads spread between the
// MFMAs measured the same, two workgroups a CU cost in partials what they
// gain.
#include "nf4_gemm_mid.hpp"

#include <algorithm>

#include "nf4_gemm.hpp"

namespace unifur {
namespace {

constexpr int kMN = 128, kMK = 64;
constexpr int kMThreads = 256;

constexpr int kCopies = 8;               // of the level-pair table
constexpr int kEntry = kCopies * 8;      // bytes from one byte value's pairs to the next
constexpr int kEntryShift = 2;           // (byte << 8 | lane part) >> this: byte * kEntry + copy * 8
static_assert((256 >> kEntryShift) == kEntry, "table stride");

template <int RT>
struct MSmem {
  static constexpr int kX = RT * 32 * kMK * 2;     // one X buffer
  static constexpr int kLut = 2 * kX;              // 256 x kCopies x {level lo, level hi}
  static constexpr int kCodes = kLut + 256 * kEntry;  // 512 bytes a wave and unit
  static constexpr int kDq = kCodes + 4 * 2 * 512;    // DQ scales, 256 x f32
  static constexpr int kBytes = kDq + 256 * 4;
};

struct MidArgs {
  const uint16_t* x;  // [M][K] bf16, 16-byte aligned
  int M, K, N;
  const uint8_t* packed;  // striped
  ScalesArg scales;
  const float* bias;     // [N] or null
  const float* lora_xa;  // [M][lora_rank] f32 x A, or null
  const float* lora_b;   // [lora_rank][N]
  int lora_rank;
  float lora_scaling;
  void* y;  // [M][N] f32 or bf16
  int y_bf16;
  int k_splits, k_slab;  // slabs of K, and the K of one
  float* partials;       // [k_splits][M][N], or null
};

// NF4_LEVELS[c] for a per-lane c from immediates (no memory access)
__device__ __forceinline__ float level_of(int c) {
  float v = level(0);
#pragma unroll
  for (int i = 1; i < 16; ++i) v = c == i ? level(i) : v;
  return v;
}

// The codes and block scales (f32 bits or u8 DQ codes) of one K step: two
// units of 32 rows, this lane's row of each.
struct MCodes {
  u32x2 code[2];
  uint32_t scale[2];
};

template <bool DQ>
__device__ __forceinline__ MCodes load_codes(const MidArgs& g, size_t code_at, size_t scale_at, int k0) {
  MCodes c;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    c.code[u] = *reinterpret_cast<const u32x2*>(g.packed + code_at + (size_t)(k0 + 32 * u) * 8);
    const size_t s = scale_at + k0 + 32 * u;
    c.scale[u] = DQ ? (uint32_t)g.scales.dq_codes[s] : __float_as_uint(g.scales.absmax[s]);
  }
  return c;
}

// A row's chunks are XORed with row % 8 and row / 8 % 4: sixteen consecutive
// rows' reads of one chunk then meet all 256 bytes of banks once (with
// row % 8 alone rows r and r + 8 met, and every X read took twice as long).
__device__ __forceinline__ int x_swizzle(int r) { return (r & 7) ^ ((r >> 3) & 3); }

template <int RT>
struct MX {
  u32x4 v[RT];
};

// X of one step: thread t copies chunk t % 8 of rows t / 8 + 32 q.
template <int RT>
__device__ __forceinline__ MX<RT> load_x(const MidArgs& g, int m0, int k0, int tid) {
  MX<RT> x;
#pragma unroll
  for (int q = 0; q < RT; ++q)
    x.v[q] = *reinterpret_cast<const u32x4*>(g.x + (size_t)min(m0 + tid / 8 + 32 * q, g.M - 1) * g.K + k0 +
                                             8 * (tid % 8));
  return x;
}

template <int RT>
__device__ __forceinline__ void store_x(const MX<RT>& x, int base, int tid) {
  const int r = tid / 8, c = tid % 8;
#pragma unroll
  for (int q = 0; q < RT; ++q)
    *reinterpret_cast<lds_u32x4*>((size_t)(base + (r + 32 * q) * (kMK * 2) + ((c ^ x_swizzle(r)) * 16))) = x.v[q];
}

// A step's codes with each lane's 16 consecutive k of its column (two 32-row
// units), and its row's scale of each unit.
struct MStep {
  u32x2 nib[2];
  float scale[2];
};

template <bool DQ>
__device__ __forceinline__ MStep transpose_codes(const MCodes& c, const unsigned char* dq, uint32_t stage) {
  MStep p;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const uint32_t at = stage + (uint32_t)u * 512u;
    *reinterpret_cast<lds_u32x2*>((size_t)at) = c.code[u];
    p.nib[u] =
        __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr4_b64_v2i32(reinterpret_cast<lds_v2i32*>((size_t)at)));
    p.scale[u] = DQ ? reinterpret_cast<const float*>(dq)[c.scale[u] & 0xffu] : __uint_as_float(c.scale[u]);
  }
  return p;
}

// What the MFMAs of one k16 phase read from LDS: the level pairs of the
// lane's eight codes and the X fragments.
template <int RT>
struct MPhase {
  f32x2 level[4];
  u32x4 x[RT];
};

template <int P, int RT>
__device__ __forceinline__ void issue_phase(MPhase<RT>& o, const MStep& p, uint32_t x_at, uint32_t x_chunk,
                                            uint32_t lane_off) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t at = perm_b32(p.nib[P >> 1][P & 1], lane_off, 0x0c0c0000u | (uint32_t)((4 + j) << 8)) >> kEntryShift;
    o.level[j] = *reinterpret_cast<lds_f32x2_c*>((size_t)(MSmem<RT>::kLut + at));
  }
  const uint32_t at = x_at + (x_chunk ^ (uint32_t)((4 * (P >> 1) + (P & 1)) * 16));
#pragma unroll
  for (int i = 0; i < RT; ++i) o.x[i] = *reinterpret_cast<lds_u32x4*>((size_t)(at + i * 32 * kMK * 2));
}

template <int P, int RT>
__device__ __forceinline__ void multiply_phase(f32x16 (&acc)[RT], const MPhase<RT>& o, const MStep& p) {
  u32x4 w;
  float sc[16];
  row_lanes<0>(p.scale[P >> 1], sc);  // row 16 h + j's scale sits in lane 16 (l / 16) + j
#pragma unroll
  for (int j = 0; j < 4; ++j)
    w[j] = pack_bf16x2(o.level[j].x * sc[8 * (P & 1) + 2 * j], o.level[j].y * sc[8 * (P & 1) + 2 * j + 1]);
#pragma unroll
  for (int i = 0; i < RT; ++i)
    acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, o.x[i]),
                                                     __builtin_bit_cast(bf16x8_t, w), acc[i], 0, 0, 0);
}

// acc = the wave's sums over the slab [kb, ke), and its share of the adapter's
// ranks.  `luts`: build the tables first (the first slab of a
// workgroup).
//
// Software pipeline: a phase's table lookups and X fragments are read during
// the phase before, a step's codes are transposed during the step before, X
// and the codes are loaded two steps before their use.  The step's one barrier
// stands before its last phase, which reads the next step's first: the buffer
// it frees is the step's own, whose last reads were issued a phase earlier.
template <int RT, bool DQ>
__device__ __forceinline__ void slab_sums(f32x16 (&acc)[RT], const MidArgs& g, unsigned char* smem,
                                          int m0, int n0, int kb, int ke, int tid, int wave, bool luts) {
  using S = MSmem<RT>;
  const int lane = tid & 63, h = lane >> 5, r32 = lane & 31;

  // this lane's row and stripe of a 32 x 32 unit; a wave past N reads its
  // last columns and stores nothing
  const int nc = min(n0, g.N - 32), row = 16 * h + (lane & 15);
  const size_t code_at = ((size_t)(nc / 16 + ((lane >> 4) & 1)) * g.K + row) * 8;
  const size_t scale_at = (size_t)(nc / kBlock) * g.K + row;
  const int last = ke - kMK;  // loads past the slab stay on its last step
  float sos = 0.0f;  // by a vector load ahead of the others
  if constexpr (DQ) {
    const float* at = g.scales.scale_of_scales;
    asm volatile("" : "+v"(at));
    if (luts) sos = *at;
  }
  MX<RT> x[2];  // of the next step and the one after
  x[0] = load_x<RT>(g, m0, kb, tid);
  x[1] = load_x<RT>(g, m0, min(kb + kMK, last), tid);
  MCodes c[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) c[q] = load_codes<DQ>(g, code_at, scale_at, min(kb + q * kMK, last));

  if (luts) {
    const f32x2 l = {level_of(tid & 15), level_of(tid >> 4)};
#pragma unroll
    for (int c = 0; c < kCopies; ++c)
      *reinterpret_cast<f32x2*>(smem + S::kLut + tid * kEntry + ((c + tid) & (kCopies - 1)) * 8) = l;
    if constexpr (DQ) reinterpret_cast<float*>(smem + S::kDq)[tid] = ((float)tid / 255.0f) * sos;
  }
#pragma unroll
  for (int i = 0; i < RT; ++i) acc[i] = f32x16{};
  // (xa scaling) B on the f32 instruction, while the first loads are in
  // flight; four steps' factors are loaded together, from clamped places
  // and zeroed past the rank.  Each eight ranks wait out a memory latency, so
  // the slabs take turns at them (4096 -> 4096, rank 64, 128 rows: 44 us with
  // all of them in the first slab, 36 with this)
  if (g.lora_xa) {
    const float* bcol = g.lora_b + nc + r32;
    for (int j0 = kb / g.k_slab * 8; j0 < g.lora_rank; j0 += 8 * g.k_splits) {
      float av[4][RT], bv[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = min(j0 + 2 * q + h, g.lora_rank - 1);
        bv[q] = bcol[(size_t)j * g.N];
#pragma unroll
        for (int i = 0; i < RT; ++i)
          av[q][i] = g.lora_xa[(size_t)min(m0 + 32 * i + r32, g.M - 1) * g.lora_rank + j];
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
  store_x<RT>(x[0], 0, tid);
  x[0] = load_x<RT>(g, m0, min(kb + 2 * kMK, last), tid);
  __syncthreads();

  const unsigned char* dq = smem + S::kDq;
  const uint32_t stage = (uint32_t)(S::kCodes + wave * 1024 + lane * 8);
  const uint32_t lane_off = (uint32_t)(lane & (kCopies - 1)) << (3 + kEntryShift);
  const uint32_t x_row = (uint32_t)(r32 * (kMK * 2)), x_chunk = (uint32_t)(((2 * h) ^ x_swizzle(r32)) * 16);
  MStep p = transpose_codes<DQ>(c[0], dq, stage);
  c[0] = load_codes<DQ>(g, code_at, scale_at, min(kb + 2 * kMK, last));
  MPhase<RT> fa, fb;
  issue_phase<0, RT>(fa, p, x_row, x_chunk, lane_off);
  // one step from X buffer `buf`; xn: the next step's X, cn: its codes, each
  // replaced by the one its ring's length later
  const auto step = [&](int k0, uint32_t buf, MX<RT>& xn, MCodes& cn) {
    store_x<RT>(xn, (int)(buf ^ S::kX), tid);
    xn = load_x<RT>(g, m0, min(k0 + 3 * kMK, last), tid);
    issue_phase<1, RT>(fb, p, buf + x_row, x_chunk, lane_off);
    __builtin_amdgcn_sched_barrier(0);
    multiply_phase<0, RT>(acc, fa, p);
    const MStep pn = transpose_codes<DQ>(cn, dq, stage);
    cn = load_codes<DQ>(g, code_at, scale_at, min(k0 + 3 * kMK, last));
    issue_phase<2, RT>(fa, p, buf + x_row, x_chunk, lane_off);
    __builtin_amdgcn_sched_barrier(0);
    multiply_phase<1, RT>(acc, fb, p);
    issue_phase<3, RT>(fb, p, buf + x_row, x_chunk, lane_off);
    __builtin_amdgcn_sched_barrier(0);
    multiply_phase<2, RT>(acc, fa, p);
    __syncthreads();
    issue_phase<0, RT>(fa, pn, (buf ^ S::kX) + x_row, x_chunk, lane_off);
    __builtin_amdgcn_sched_barrier(0);
    multiply_phase<3, RT>(acc, fb, p);
    p = pn;
  };
  for (int k0 = kb; k0 < ke; k0 += 2 * kMK) {
    step(k0, 0, x[1], c[1]);
    if (k0 + kMK < ke) step(k0 + kMK, S::kX, x[0], c[0]);
  }
  __syncthreads();  // the next slab writes the buffers
}

// One workgroup a (tile, slab), or with SERIAL one a tile that takes the
// slabs in turn and adds their sums in the order of the reduction: a call
// gives the same bits with and without room for the partials.
template <int RT, bool DQ, bool SERIAL>
__global__ __launch_bounds__(kMThreads, SERIAL && RT == 4 ? 1 : 2) void gemm_mid_kernel(MidArgs g) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // XCD-aware order: workgroup b runs on XCD b % 8; each XCD takes a
  // contiguous run of (slab, column tile, row tile), rows fastest: the row
  // tiles that share a weight tile meet it in one L2
  const int nb = gridDim.x, b = blockIdx.x;
  const int t = (nb % 8 == 0) ? (b % 8) * (nb / 8) + b / 8 : b;
  const int tiles_m = (g.M + 32 * RT - 1) / (32 * RT), tiles = SERIAL ? nb : nb / g.k_splits;
  const int slab = SERIAL ? 0 : t / tiles, tt = SERIAL ? t : t % tiles;
  const int m0 = (tt % tiles_m) * (32 * RT), n0 = (tt / tiles_m) * kMN + 32 * wave;

  f32x16 acc[RT];
  const int kb = slab * g.k_slab;
  slab_sums<RT, DQ>(acc, g, smem, m0, n0, kb, min(g.K, kb + g.k_slab), tid, wave, true);
  if constexpr (SERIAL) {
    for (int k1 = g.k_slab; k1 < g.K; k1 += g.k_slab) {
      f32x16 part[RT];
      slab_sums<RT, DQ>(part, g, smem, m0, n0, k1, min(g.K, k1 + g.k_slab), tid, wave, false);
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] += part[i][r];
    }
  }

  // The store, a 32 x 32 block at a time through the wave's part of the X
  // buffers (slab_sums ends with a barrier): four 16-byte stores of eight rows
  // a block.  acc[i][4 a + e] is C[row 32 i + 8 a + 4 (lane / 32) + e][col
  // lane % 32]; stored from there it is sixteen 4-byte stores a block, and
  // their unrolled code, which a short launch fetches once, cost it 4 us.
  if (n0 >= g.N) return;
  constexpr int kPitch = 40;  // floats a row: the half-waves' rows, four apart, meet other banks
  float* blk = reinterpret_cast<float*>(smem) + wave * (32 * kPitch);
  const bool parts = !SERIAL && g.k_splits > 1;
  const int er = lane >> 3, ec = 4 * (lane & 7);
  f32x4 bias = {};
  const bool add = g.bias && !parts;
  if (add) bias = f32x4{g.bias[n0 + ec], g.bias[n0 + ec + 1], g.bias[n0 + ec + 2], g.bias[n0 + ec + 3]};
  const bool wide = (reinterpret_cast<uintptr_t>(g.y) & 15u) == 0;
#pragma unroll
  for (int i = 0; i < RT; ++i) {
#pragma unroll
    for (int r = 0; r < 16; ++r)
      blk[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * kPitch + (lane & 31)] = acc[i][r];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f32x4 v = *reinterpret_cast<const f32x4*>(blk + (8 * q + er) * kPitch + ec);
      const int m = m0 + 32 * i + 8 * q + er;
      if (m >= g.M) continue;
      const size_t o = (size_t)m * g.N + n0 + ec;
      if (parts) {
        *reinterpret_cast<f32x4*>(g.partials + (size_t)slab * g.M * g.N + o) = v;
        continue;
      }
      if (add) v = f32x4{v.x + bias.x, v.y + bias.y, v.z + bias.z, v.w + bias.w};
      if (g.y_bf16) {
        uint16_t* y = reinterpret_cast<uint16_t*>(g.y) + o;
        const u32x2 p = {pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w)};
        if (wide) *reinterpret_cast<u32x2*>(y) = p;
        else for (int e = 0; e < 4; ++e) y[e] = (uint16_t)(p[e >> 1] >> (16 * (e & 1)));
      } else {
        float* y = reinterpret_cast<float*>(g.y) + o;
        if (wide) *reinterpret_cast<f32x4*>(y) = v;
        else for (int e = 0; e < 4; ++e) y[e] = v[e];
      }
    }
  }
}

// Row tiles of a workgroup: 96 or 128 rows, whichever pads the batch less
// (128 on a tie: a weight tile is dequantized once per row tile).
int row_tiles(int M) { return (M + 95) / 96 * 96 < (M + 127) / 128 * 128 ? 3 : 4; }

template <int RT, bool DQ>
hipError_t launch_m(const MidArgs& g, hipStream_t stream) {
  static_assert(MSmem<RT>::kBytes <= 64 << 10, "more LDS needs the attribute");
  const int tiles = ((g.M + 32 * RT - 1) / (32 * RT)) * ((g.N + kMN - 1) / kMN);
  if (g.k_splits > 1 && !g.partials)
    gemm_mid_kernel<RT, DQ, true><<<tiles, kMThreads, MSmem<RT>::kBytes, stream>>>(g);
  else
    gemm_mid_kernel<RT, DQ, false><<<tiles * g.k_splits, kMThreads, MSmem<RT>::kBytes, stream>>>(g);
  return hipGetLastError();
}

}  // namespace

bool gemm_mid_supported(int M, int K, int N, const void* x) {
  return M > 0 && K > 0 && N > 0 && K % kMK == 0 && N % 64 == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
}

// Measured against the expanded weight and the library product, us per call at
// 65 / 128 / 192 / 256 rows, without an adapter and with one of rank 16 and 64
// (whose x A is a launch of its own here and merged into the expansion there;
// both take one path, so that an adapter of zeros adds nothing to the bit):
//   4096 -> 4096       16.4 20.4 21.2       against 31.4 30.9 31.7
//            rank 16   21.3 25.8 27.3               30.8 31.1 31.1
//            rank 64   25.3 30.8 35.3               41.8 41.7 43.3
//   4096 -> 8192       19.2 25.6 29.8 32.2          35.0 36.3 39.1 41.2
//            rank 16   25.1 29.7 36.2 40.0          37.4 38.8 41.9 44.2
//            rank 64   28.9 34.2 44.0 50.1          62.7 64.7 68.3 72.3
//   8192 -> 2048       17.0 21.5 21.7               32.3 31.3 35.1
//            rank 16   25.7 30.1 30.1               32.3 31.3 34.9
//            rank 64   27.9 32.0 36.3               44.7 44.0 49.0
//   11008 -> 4096      21.9 25.6 33.0 37.7          49.8 52.1 55.5 58.5
//            rank 64   36.7 42.8 56.5 62.0          87.2 89.6 93.5 95.0
//   512 -> 32768       10.5 11.9 13.9               30.3 29.6 31.5
//            rank 64   22.7 32.2 40.7               38.1 37.9 40.5
//   16384 -> 1024      20.1 25.5 22.8               33.1 32.1 37.4
//            rank 16   30.4 32.9 34.4               33.0 32.1 38.3
// so from 2^24 weights up to 192 rows, from 2^25 up to 256: the line is where
// an adapted call still gains or breaks even.  (4096 -> 2048 without an
// adapter would gain too, 15 to 21 us against 23 to 26, but loses with one of
// rank 16, 24 to 27 against 23 to 26.)
bool gemm_mid_wanted(int M, int K, int N) {
  const int64_t weights = (int64_t)K * N;
  return weights >= (int64_t)1 << 24 && M <= (weights >= (int64_t)1 << 25 ? 256 : 192);
}

int gemm_mid_splits(int M, int K, int N, size_t max_floats) {
  const int rows = 32 * row_tiles(M);
  const int64_t tiles = (int64_t)((M + rows - 1) / rows) * ((N + kMN - 1) / kMN);
  const int64_t want = kMidGrid / tiles, most = K / (4 * kMK), room = (int64_t)(max_floats / ((size_t)M * N));
  return (int)std::max<int64_t>(1, std::min<int64_t>({want, most, room}));
}

hipError_t launch_gemm_mid(const uint16_t* x, const uint8_t* packed, const ScalesArg& scales, int M, int K, int N,
                           const float* bias, const float* lora_xa, const float* lora_b, int lora_rank,
                           float lora_scaling, void* y, bool y_bf16, hipStream_t stream, int k_splits,
                           float* partials) {
  if (!gemm_mid_supported(M, K, N, x) || k_splits < 1 ||
      (k_splits > 1 && partials && ((reinterpret_cast<uintptr_t>(y) & 15u) || (reinterpret_cast<uintptr_t>(bias) & 15u))))
    return hipErrorInvalidValue;
  MidArgs g{};
  g.x = x;
  g.M = M;
  g.K = K;
  g.N = N;
  g.packed = packed;
  g.scales = scales;
  g.bias = bias;
  g.lora_xa = lora_xa;
  g.lora_b = lora_b;
  g.lora_rank = lora_rank;
  g.lora_scaling = lora_scaling;
  g.y = y;
  g.y_bf16 = y_bf16;
  const int steps = K / kMK;
  g.k_slab = (steps + k_splits - 1) / k_splits * kMK;
  g.k_splits = (K + g.k_slab - 1) / g.k_slab;  // no empty slab
  g.partials = g.k_splits > 1 ? partials : nullptr;
  const bool dq = scales.kind == kScalesDQ;
  hipError_t e = hipSuccess;
  if (row_tiles(M) == 3) e = dq ? launch_m<3, true>(g, stream) : launch_m<3, false>(g, stream);
  else e = dq ? launch_m<4, true>(g, stream) : launch_m<4, false>(g, stream);
  if (e != hipSuccess || !g.partials) return e;
  return launch_splitk_reduce(partials, g.k_splits, M, N, bias, y, y_bf16, stream);
}

}  // namespace unifur

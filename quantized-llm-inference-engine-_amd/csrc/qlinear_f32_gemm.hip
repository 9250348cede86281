// fp32 activations on a bf16 MFMA GEMM without loss: QuantLinear.forward with compute_dtype float32
// (src/llmopt/quantization/quant_linear.py:93-113, the reference engine's own configuration,
// engine/llm_engine.py:258-264) for batches past the decode kernels.
//
//   y[m, n] = sum over groups g of s[n, g] * sum over k in g of (q[n, k] - z[n, g]) * x[m, k] + b[n]
//
// q - z is a small integer, exact in bf16, and an fp32 activation is exactly the sum of three bf16
// pieces, so each group's inner sum runs on v_mfma_f32_32x32x16_bf16 with exact operands and exact
// products (three MFMAs per 16 k instead of one); its fp32 result is folded into the output
// accumulator with one fp32 fma by the group's scale. Nothing is rounded below fp32 anywhere, and
// the weight is never rounded at all.
//
// What bounds it: three bf16 MFMAs per fp32 multiply-add, i.e. at most a third of the bf16 matrix
// rate (833 TFLOP/s), against 157 TFLOP/s for the fp32 vector and matrix units that a dense fp32
// product over the dequantized weight uses.
//
// Measured (MI355X, groups of 64; us against the dense fp32 product over the dequantized weight, or, at
// 24 tokens, two passes of the decode kernels): gate_up 24 tokens 51 / 69, 128 tokens 111 / 341, 2048
// tokens 1257 / 3294 (383 TFLOP/s, 1.15 PFLOP/s of bf16 products: 82 % of what a large bf16 library
// product reaches on the same card); down 2048 tokens 662 / 1643; o 128 tokens 35 / 58. Error against
// float64 (2-norm, K = 4096 / 14336): 1.7e-7 / 2.8e-7, against 1.1e-6 / 2.1e-6.
//
// Two kernels. split_tiles_kernel cuts x into its pieces once (truncation: each piece takes the
// next eight significand bits, so hi + mid + lo = x exactly, and an infinite or NaN x is carried by hi
// alone; rows of very large or small values are scaled first) and lays them out as the GEMM's LDS images: [32-token block][64-wide
// k stage][piece][token][16-byte chunk, XOR-swizzled], 12 KB per block and stage, so that a stage is
// copied to LDS by direct loads of consecutive kilobytes. f32_gemm_kernel: a workgroup of four waves
// owns 256 output features x 32 TT tokens; each wave takes 64 features and every token, so an LDS
// fragment read (the A operand, 32 tokens x 16 k) feeds two MFMAs and a weight fragment (the B operand,
// one 32-bit word of packed codes per lane) is dequantized by exactly one wave and feeds 3 TT. Two
// workgroups share a CU (72 KB of LDS and at most 229 registers each), which fills one's barriers, folds and
// dequantization with the other's MFMAs.
#include <algorithm>
#include <type_traits>

#include "qcommon.hpp"
#include "qkernels.hpp"

namespace llmopt {
namespace {

constexpr int kBN = 256;        // output features per workgroup (4 waves x 64)
constexpr int kBK = 64;         // K per stage
constexpr int kThreads = 256;
constexpr int kSplitThreads = 512;
constexpr int kBuffers = 3;     // LDS stage buffers
constexpr int kBlockBytes = 3 * 32 * kBK * 2;  // one 32-token block of one stage: three pieces
constexpr int kMaxSplits = 16;
constexpr int kGroupM = 8;      // token tiles per sweep over the feature tiles

typedef unsigned char uc4 __attribute__((ext_vector_type(4)));
typedef signed char sc4 __attribute__((ext_vector_type(4)));

// Byte offset of 16-byte chunk c of token row r in a [32][64] image of 16-bit values: 16 consecutive
// rows of one chunk fall on 16 distinct 4-bank groups.
__device__ __forceinline__ int swz(int r, int c) { return r * 128 + ((c ^ ((r >> 1) & 7)) << 4); }

__device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}

// ---- x -> pieces ------------------------------------------------------------------------------------
// A row's 8-wide chunks go to the threads in turn; with `parts` (a power of two) > 1 workgroups per row, each
// sees all of them and splits every parts-th round (small batches: few rows for many CUs). A row whose
// largest finite |x| lies outside 2^-64 .. 2^81 is split a second time, brought to that range by a power of
// two that is undone on the outputs: below it the pieces' last bits fall under bf16's subnormals, above it a
// group's unscaled sum, up to 255 |x| per product, overflows where the scaled result does not. Other rows
// are split as they are, and so exact down to 2^-110. With `sums`, also the fp32 sum of each (stage, token)
// -- read by the GEMM only for zero points that are not integers. Rows past M are left as they are: an
// MFMA's output row depends on its own row only, and theirs are not stored.
// Bound by latency at small batches: 3.0 us for 24 rows of 4096, 5.1 for 32 of 14336, against 2.7 and 5.1
// without the row's range; qkv at 24 tokens 22.7 -> 23.2 us, MLP at 32 77.9 -> 79.8. The usual row costs two
// ballots and one exchange beside the stores. One workgroup of 512 threads per row, whatever its length: 3.2
// and about 6.5 us; the row held and its exact maximum found first: 3.3 at 24 rows of 4096.
template <bool VEC>
__device__ __forceinline__ void load_chunk(const float* src, float* v) {
  if (VEC) {
    const f32x4 lo = *reinterpret_cast<const f32x4*>(src), hi = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = lo[j], v[4 + j] = hi[j];
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = src[j];
  }
}

__device__ __forceinline__ void split_chunk(const float* in, float factor, int64_t m, int64_t mpad, int ktiles, int c8,
                                            uint8_t* pieces, float* sums) {
  const int kt = c8 >> 3, c = c8 & 7;
  float v[8];
  uint32_t p[3][8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    v[j] = in[j] * factor;
    const uint32_t u = __float_as_uint(v[j]);
    const bool finite = (u & 0x7F800000u) != 0x7F800000u;
    // A NaN whose payload sits in the low half would truncate to infinity: keep it a NaN.
    const uint32_t h = (u & 0xFFFF0000u) | (finite || (u & 0x7FFFFFu) == 0u ? 0u : 0x00400000u);
    const float r1 = finite ? v[j] - __uint_as_float(h) : 0.0f;  // exact
    const uint32_t mid = __float_as_uint(r1) & 0xFFFF0000u;
    const float r2 = r1 - __uint_as_float(mid);  // exact, at most eight significant bits
    p[0][j] = h;
    p[1][j] = mid;
    p[2][j] = __float_as_uint(r2);
  }
  uint8_t* dst = pieces + ((m >> 5) * ktiles + kt) * kBlockBytes + swz(int(m & 31), c);
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    u32x4 w;
    w.x = (p[q][0] >> 16) | (p[q][1] & 0xFFFF0000u);
    w.y = (p[q][2] >> 16) | (p[q][3] & 0xFFFF0000u);
    w.z = (p[q][4] >> 16) | (p[q][5] & 0xFFFF0000u);
    w.w = (p[q][6] >> 16) | (p[q][7] & 0xFFFF0000u);
    *reinterpret_cast<u32x4*>(dst + q * (32 * kBK * 2)) = w;
  }
  if (sums) {  // the eight chunks of a stage are in eight neighbouring lanes
    float t = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    t += __shfl_xor(t, 1, 64);
    t += __shfl_xor(t, 2, 64);
    t += __shfl_xor(t, 4, 64);
    if (c == 0) sums[int64_t(kt) * mpad + m] = t;
  }
}

template <bool VEC>
__global__ void __launch_bounds__(kSplitThreads) split_tiles_kernel(const float* x, int64_t ldx, int64_t mpad, int ktiles,
                                                                    int parts, uint8_t* pieces, float* sums,
                                                                    float* undo) {
  constexpr int kHeld = 4;  // chunks in flight per thread
  __shared__ uint32_t seen[kSplitThreads / 64];
  const int64_t m = blockIdx.x;
  const int part = blockIdx.y;
  const int threads = int(blockDim.x), waves = threads / 64;
  const int chunks = ktiles * 8;  // a multiple of 16: the eight lanes of a stage stay together
  const float* row = x + m * ldx;
  float most = 0.0f;  // the largest |x| but NaN
  auto split_row = [&](float factor, auto find) {
    for (int c0 = int(threadIdx.x), round = 0; c0 < chunks; c0 += kHeld * threads, round += kHeld) {
      float v[kHeld][8];
#pragma unroll
      for (int i = 0; i < kHeld; ++i)
        if (c0 + i * threads < chunks) load_chunk<VEC>(row + int64_t(c0 + i * threads) * 8, v[i]);
#pragma unroll
      for (int i = 0; i < kHeld; ++i)
        if (c0 + i * threads < chunks) {
          if (decltype(find)::value) {
#pragma unroll
            for (int j = 0; j < 8; ++j) most = fmaxf(most, __builtin_fabsf(v[i][j]));
          }
          if (((round + i) & (parts - 1)) == part)
            split_chunk(v[i], factor, m, mpad, ktiles, c0 + i * threads, pieces, sums);
        }
    }
  };
  split_row(1.0f, std::true_type{});
  // What the row's waves saw: anything from 2^-64 on, and anything from 2^81 on.
  constexpr uint32_t kLow = 127 - 64, kHigh = 127 + 80;
  const bool some = __builtin_amdgcn_ballot_w64(most >= __uint_as_float(kLow << 23)) != 0;
  const bool large = __builtin_amdgcn_ballot_w64(most >= __uint_as_float((kHigh + 1) << 23)) != 0;
  if ((threadIdx.x & 63) == 0) seen[threadIdx.x >> 6] = (some ? 1u : 0u) | (large ? 2u : 0u);
  __syncthreads();
  uint32_t all = 0;
  for (int w = 0; w < waves; ++w) all |= seen[w];
  const bool first = threadIdx.x == 0 && part == 0;
  if (all == 1u) {  // the usual row
    if (first) undo[m] = 1.0f;
    return;
  }
  // The largest finite |x|, and whether there is anything else.
  uint32_t top = 0, others = 0;
  for (int c8 = int(threadIdx.x); c8 < chunks; c8 += threads) {
    float v[8];
    load_chunk<VEC>(row + int64_t(c8) * 8, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t u = __float_as_uint(v[j]) & 0x7FFFFFFFu;
      if (u >= 0x7F800000u)
        others = 0x80000000u;
      else if (u > top)
        top = u;
    }
  }
  top |= others;  // in the sign bit
#pragma unroll
  for (int d = 1; d < 64; d *= 2) {
    const uint32_t t = uint32_t(__shfl_xor(int(top), d, 64));
    top = max(top & 0x7FFFFFFFu, t & 0x7FFFFFFFu) | ((top | t) & 0x80000000u);
  }
  __syncthreads();  // the flags have been read
  if ((threadIdx.x & 63) == 0) seen[threadIdx.x >> 6] = top;
  __syncthreads();
  for (int w = 0; w < waves; ++w)
    top = max(top & 0x7FFFFFFFu, seen[w] & 0x7FFFFFFFu) | ((top | seen[w]) & 0x80000000u);
  const uint32_t e = (top & 0x7FFFFFFFu) >> 23;  // biased exponent
  const int shift = (top & 0x7FFFFFFFu) == 0 ? 0 : e < kLow ? int(kLow - e) : e > kHigh ? int(kHigh) - int(e) : 0;
  if (first) undo[m] = __uint_as_float((uint32_t(127 - shift) << 23) | (top & 0x80000000u));
  if (shift != 0) split_row(__uint_as_float(uint32_t(127 + shift) << 23), std::false_type{});
}

// ---- codes -> exact bf16 operands -----------------------------------------------------------------
// The integer part of a zero point, within the range whose differences stay exact in bf16
// (|q - zi| <= 256) and, for nibbles, in a byte; the rest of z, normally 0, is applied in the fold.
template <int FMT>
__device__ __forceinline__ float int_zero(float z) {
  const float r = __builtin_rintf(z);
  const float lo = FMT == kNibble ? -112.0f : 0.0f, hi = FMT == kNibble ? 127.0f : 255.0f;
  return r >= lo && r <= hi ? r : (FMT == kNibble ? 8.0f : 128.0f);  // also NaN
}

__device__ __forceinline__ uint32_t pack_exact(float lo, float hi) {  // both exact in bf16
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

// Eight nibble codes -> (q - zi) in bf16, natural order. `bias` holds 128 - zi in each byte: q + 128 -
// zi lies in [1, 255], so no carry crosses a byte, and flipping the top bit makes it the signed byte
// q - zi. 19 VALU operations for eight codes.
__device__ __forceinline__ u32x4 operand_nibbles(uint32_t word, uint32_t bias) {
  const sc4 lo = __builtin_bit_cast(sc4, ((word & 0x0F0F0F0Fu) + bias) ^ 0x80808080u);         // codes 0, 2, 4, 6
  const sc4 hi = __builtin_bit_cast(sc4, (((word >> 4) & 0x0F0F0F0Fu) + bias) ^ 0x80808080u);  // codes 1, 3, 5, 7
  return u32x4{pack_exact(float(lo.x), float(hi.x)), pack_exact(float(lo.y), float(hi.y)),
               pack_exact(float(lo.z), float(hi.z)), pack_exact(float(lo.w), float(hi.w))};
}

// Eight byte codes -> (q - zi); signed codes arrive with their sign bit flipped and 128 in zi.
__device__ __forceinline__ u32x4 operand_bytes(uint32_t w0, uint32_t w1, float zi) {
  const uc4 a = __builtin_bit_cast(uc4, w0), b = __builtin_bit_cast(uc4, w1);
  return u32x4{pack_exact(float(a.x) - zi, float(a.y) - zi), pack_exact(float(a.z) - zi, float(a.w) - zi),
               pack_exact(float(b.x) - zi, float(b.y) - zi), pack_exact(float(b.z) - zi, float(b.w) - zi)};
}

struct GemmArgs {
  const uint8_t* pieces;
  const float* sums;   // [ktiles][mpad], or null: no zero points in memory
  const float* undo;   // [mpad]: the power of two that undoes a token's scaling; negative: x holds infinities or NaN
  int64_t mpad;
  int tiles_m, tiles_n, splits;
  float* partials;     // splits > 1: [splits][M][N]
};

// PER: stages per fold (a group is a multiple of PER stages). Code words of stage kt sit in ring slot
// kt % 2. Loads per stage, in this order: at the top the 3 TT direct-to-LDS loads of stage kt + 2
// (whose buffer every wave left before the barrier), at the end the codes of stage kt + 2 and once per
// group the next group's scales and zeros. At the top of stage kt + 1 at least those 3 TT direct loads
// were issued after stage kt + 1's own, so vmcnt(3 TT) guarantees them.
template <int TT, int PER, int FMT, bool ASYM>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
    f32_gemm_kernel(const LinearArgs a, const GemmArgs g) {
  constexpr int kCB = FMT == kNibble ? 1 : 2;      // 16-byte code loads per row and stage
  constexpr int kStage = TT * kBlockBytes;         // bytes of one stage's image
  constexpr int kDirect = kStage / 1024 / 4;       // direct loads per wave and stage
  static_assert(kDirect == 3 * TT, "a stage is 12 TT kilobytes, dealt to four waves");
  __shared__ __attribute__((aligned(16))) uint8_t xs[kBuffers * kStage];

  // Tile order: an even split over the XCDs; K splits outermost, then kGroupM token tiles per sweep
  // over the feature tiles, so that workgroups that run together share operands in L2.
  int bid = blockIdx.x;
  const int nblk = gridDim.x;
  if (nblk % 8 == 0) bid = (bid % 8) * (nblk / 8) + bid / 8;
  const int ntiles = g.tiles_m * g.tiles_n;
  const int split = bid / ntiles;
  const int tile = bid - split * ntiles;
  const int per_group = kGroupM * g.tiles_n;
  const int first_m = (tile / per_group) * kGroupM;
  const int rows_in_group = min(g.tiles_m - first_m, kGroupM);
  const int tm = first_m + (tile % per_group) % rows_in_group;
  const int tn = (tile % per_group) / rows_in_group;
  const int64_t m0 = int64_t(tm) * 32 * TT;
  const int64_t n0 = int64_t(tn) * kBN;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = lane & 31, half = lane >> 5;

  const int ktotal = int(a.K / kBK);
  const int units = ktotal / 2;  // splits are cut at pairs of stages
  const int kt_base = int(int64_t(split) * units / g.splits) * 2;
  const int n_stages = int(int64_t(split + 1) * units / g.splits) * 2 - kt_base;

  // ---- weight rows n0 + 64 wave + 32 i + row: bytes 16 kCB half .. of each stage slice ----
  const auto wq = make_rsrc(a.qw, uint32_t(a.N * a.ldq));
  const uint32_t meta_bytes = uint32_t(a.N * a.G * 4);
  const auto ms = make_rsrc(a.scales, meta_bytes);
  const auto mz = make_rsrc(ASYM ? a.zeros : a.scales, meta_bytes);
  uint32_t wq_off[2], meta_off[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    int64_t n = n0 + 64 * wave + 32 * i + row;
    n = n < a.N ? n : a.N - 1;  // rows past N repeat row N-1; their outputs are never stored
    wq_off[i] = uint32_t(n * a.ldq + half * 16 * kCB);
    meta_off[i] = uint32_t(n * a.G * 4);
  }
  const bool flipped = FMT == kByte && a.signed_codes;
  const uint32_t flip = flipped ? 0x80808080u : 0u;
  const float z_add = flipped ? 128.0f : 0.0f;
  const int stages_per_group = int(a.group / kBK);

  u32x4 wring[2][2][kCB];
  auto load_codes = [&](int slot, int kt) {
    const int ktc = kt_base + (kt < n_stages ? kt : n_stages - 1);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int c = 0; c < kCB; ++c) wring[slot][i][c] = buf_load16(wq, wq_off[i] + 16 * c, uint32_t(ktc) * 32 * kCB);
  };
  float s_next[2], z_next[2];  // the next fold's scale and zero point, in flight
  auto load_meta = [&](int kt) {
    const int ktc = kt_base + (kt < n_stages ? kt : n_stages - 1);
    const uint32_t g4 = uint32_t(ktc / stages_per_group) * 4;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      s_next[i] = buf_load_f32(ms, meta_off[i], g4);
      if (ASYM) z_next[i] = buf_load_f32(mz, meta_off[i], g4);
    }
  };
  float s[2], zi[2], zr[2];
  uint32_t bias[2];
  auto take_meta = [&]() {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float z = (ASYM ? z_next[i] : a.zero_const) + z_add;
      s[i] = s_next[i];
      zi[i] = int_zero<FMT>(z);
      zr[i] = z - zi[i];
      if (FMT == kNibble) bias[i] = uint32_t(128 - int(zi[i])) * 0x01010101u;
    }
  };

  // ---- activations: wave w copies kilobytes w kDirect .. of the stage image ----
  const auto xr = make_rsrc(g.pieces, uint32_t(g.mpad / 32 * ktotal * kBlockBytes));
  auto load_x = [&](int kt) {
    const int ktc = kt_base + (kt < n_stages ? kt : n_stages - 1);
    uint8_t* dst = xs + (kt % kBuffers) * kStage;
#pragma unroll
    for (int d = 0; d < kDirect; ++d) {
      const int kb = wave * kDirect + d;           // kilobyte of the image
      const int blk = kb / (kBlockBytes / 1024);   // its 32-token block
      const uint32_t soff = uint32_t((int64_t(tm * TT + blk) * ktotal + ktc) * kBlockBytes) +
                            uint32_t(kb - blk * (kBlockBytes / 1024)) * 1024;
      load_lds16_cached(xr, dst + kb * 1024, 16 * lane, soff);
    }
  };

  f32x16 acc[2][TT], part[2][TT];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < TT; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
  const f32x16 zero16 = {};

  bool remainders = false;
  auto word = [](const u32x4& q, int w) { return w == 0 ? q.x : w == 1 ? q.y : w == 2 ? q.z : q.w; };
  auto stage = [&](const int u, const int kt, const bool first, const bool last) {
    wait_lgkmcnt0();       // this wave's fragment reads of stage kt - 1
    wait_vmcnt<kDirect>(); // this wave's share of stage kt's image
    __builtin_amdgcn_s_barrier();
    load_x(kt + 2);
    const uint8_t* cur = xs + (kt % kBuffers) * kStage;
#pragma unroll
    for (int ks = 0; ks < kBK / 16; ++ks) {
      u32x4 wf[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if constexpr (FMT == kNibble) {
          wf[i] = operand_nibbles(word(wring[u][i][0], ks), bias[i]);
        } else {
          const u32x4 q = wring[u][i][ks >> 1];
          wf[i] = operand_bytes(word(q, (2 * ks) & 3) ^ flip, word(q, (2 * ks + 1) & 3) ^ flip, zi[i]);
        }
      }
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int j = 0; j < TT; ++j) {
          const u32x4 xf = *reinterpret_cast<const u32x4*>(cur + j * kBlockBytes + p * (32 * kBK * 2) +
                                                           swz(row, 4 * half + ks));
#pragma unroll
          for (int i = 0; i < 2; ++i)
            part[i][j] = mfma(xf, wf[i], first && ks == 0 && p == 0 ? zero16 : part[i][j]);
        }
    }
    load_codes(u, kt + 2);
    if (last) {
      // Lane: output feature 32 i + row of the wave, tokens 8 (v / 4) + 4 half + v % 4 of block j.
#pragma unroll
      for (int j = 0; j < TT; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[i][j][v] = __builtin_fmaf(s[i], part[i][j][v], acc[i][j][v]);
      if (ASYM && __builtin_amdgcn_ballot_w64(zr[0] != 0.0f || zr[1] != 0.0f)) {
        // A zero point that is not an integer in range: its remainder times the group's sums of x.
        remainders = true;
#pragma unroll 1
        for (int t = 0; t < PER; ++t) {
          const float* sum = g.sums + int64_t(kt_base + kt - t) * g.mpad + m0 + 4 * half;
#pragma unroll
          for (int j = 0; j < TT; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
              const float x1 = sum[32 * j + 8 * (v / 4) + v % 4];
#pragma unroll
              for (int i = 0; i < 2; ++i) acc[i][j][v] = __builtin_fmaf(-(s[i] * zr[i]), x1, acc[i][j][v]);
            }
        }
      }
      take_meta();
      load_meta(kt + 1 + PER);
    }
  };

  // With a remainder r = z - zi, an infinite x enters a sum as (q - zi) x and as -r x, which may be NaN where
  // (q - z) x is infinite: such a token's sum is what its infinities and NaN alone give, term by term.
  auto redo_infinite = [&]() {
    bool any = false;
#pragma unroll
    for (int j = 0; j < TT; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t m = m0 + 32 * j + 8 * q + 4 * half;
        const f32x4 u = *reinterpret_cast<const f32x4*>(g.undo + m);  // rows past M hold anything
#pragma unroll
        for (int r = 0; r < 4; ++r) any |= m + r < a.M && u[r] < 0.0f;
      }
    if (!__builtin_amdgcn_ballot_w64(any)) return;
#pragma unroll 1
    for (int t = 0; t < 16 * TT; ++t) {
      const int64_t m = m0 + 32 * (t / 16) + 8 * (t % 16 / 4) + 4 * half + t % 4;
      const bool mine = m < a.M && g.undo[m] < 0.0f;
      float exact[2] = {0.0f, 0.0f};
      bool found = false;
      if (__builtin_amdgcn_ballot_w64(mine)) {
        const float* xm = static_cast<const float*>(a.x) + (mine ? m : 0) * a.ldx;
#pragma unroll 1
        for (int kt = kt_base; kt < kt_base + n_stages; ++kt) {
          const bool here = mine && !(__builtin_fabsf(g.sums[int64_t(kt) * g.mpad + m]) < __builtin_inff());
          if (!__builtin_amdgcn_ballot_w64(here && !(found && exact[0] != exact[0] && exact[1] != exact[1]))) continue;
#pragma unroll 1
          for (int k = kt * kBK; k < (kt + 1) * kBK; ++k) {
            const float v = xm[k];
            if (!here || __builtin_fabsf(v) < __builtin_inff()) continue;
            found = true;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
              const int64_t n = min(n0 + 64 * wave + 32 * i + row, a.N - 1), gi = n * a.G + k / a.group;
              const uint8_t* codes = a.qw + n * a.ldq;
              const float q = FMT == kNibble     ? float((codes[k >> 1] >> (4 * (k & 1))) & 15)
                              : a.signed_codes ? float(int8_t(codes[k]))
                                               : float(codes[k]);
              exact[i] += (q - a.zeros[gi]) * a.scales[gi] * v;
            }
          }
        }
      }
#pragma unroll
      for (int j = 0; j < TT; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          if (found && t == 16 * j + v) {
#pragma unroll
            for (int i = 0; i < 2; ++i) acc[i][j][v] = exact[i];
          }
    }
  };

  load_meta(0);
  load_codes(0, 0);
  load_codes(1, 1);
  take_meta();
  load_meta(PER);
  load_x(0);
  load_x(1);
  for (int kt = 0; kt < n_stages; kt += 2) {
    stage(0, kt, true, PER == 1);
    stage(1, kt + 1, PER == 1, true);
  }
  if (ASYM && remainders) redo_infinite();
  f32x4 undo[TT][4];
  if (g.splits == 1) {  // else the reduction does it
#pragma unroll
    for (int j = 0; j < TT; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        undo[j][q] = *reinterpret_cast<const f32x4*>(g.undo + m0 + 32 * j + 8 * q + 4 * half);
  }
  // Direct loads past the last stage are still in flight: they end before the LDS is released.
  wait_vmcnt<0>();
  if (g.splits == 1) {
#pragma unroll
    for (int j = 0; j < TT; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] *= __builtin_fabsf(undo[j][v / 4][v % 4]);
  }
  const float* b = static_cast<const float*>(a.bias);
  if (a.epilogue == kEpiSwiglu && g.splits == 1) {
    // Fused rows 8p .. 8p + 3 are gate features 4p .. and rows 8p + 4 .. the up features (N % 8 == 0): lane
    // l's partner is lane l ^ 4. Of two tokens v and v + 1 the gate lane finishes the first and the up lane
    // the second, so one exchange serves both. (MLP of 1536 tokens: 1546 -> 1449 us against the product in
    // memory and a combining pass.)
    const bool up = row & 4;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t n = n0 + 64 * wave + 32 * i + row;
      const float bn = b && n < a.N ? b[n] : 0.0f;
      float* dst = static_cast<float*>(a.y) + (n >> 3) * 4 + (n & 3);
#pragma unroll
      for (int j = 0; j < TT; ++j)
#pragma unroll
        for (int v = 0; v < 16; v += 2) {
          const float t0 = b ? acc[i][j][v] + bn : acc[i][j][v], t1 = b ? acc[i][j][v + 1] + bn : acc[i][j][v + 1];
          const float got = __uint_as_float(__builtin_amdgcn_ds_swizzle(__float_as_uint(up ? t0 : t1), 0x101F));
          const float h = up ? swiglu<ActF32>(got, t1) : swiglu<ActF32>(t0, got);
          const int64_t m = m0 + 32 * j + 8 * (v / 4) + 4 * half + v % 4 + (up ? 1 : 0);
          if (m < a.M && n < a.N) dst[m * a.ldy] = h;
        }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int64_t n = n0 + 64 * wave + 32 * i + row;
    if (n >= a.N) continue;
    const float bn = g.splits == 1 && b ? b[n] : 0.0f;
    float* dst = g.splits == 1 ? static_cast<float*>(a.y) + n : g.partials + size_t(split) * a.M * a.N + n;
    const int64_t ld = g.splits == 1 ? a.ldy : a.N;
#pragma unroll
    for (int j = 0; j < TT; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int64_t m = m0 + 32 * j + 8 * (v / 4) + 4 * half + v % 4;
        if (m < a.M) dst[m * ld] = b ? acc[i][j][v] + bn : acc[i][j][v];
      }
  }
}

// y = bias + the splits' partial sums, in split order; four columns per thread where they align.
template <int V>
__global__ void __launch_bounds__(64) f32_reduce_kernel(const LinearArgs a, const float* partials, const float* undo,
                                                        int splits) {
  const int64_t nv = (a.N + V - 1) / V;
  const int64_t e = int64_t(blockIdx.x) * 64 + threadIdx.x;
  if (e >= a.M * nv) return;
  const int64_t m = e / nv, n = (e - m * nv) * V;
  const size_t plane = size_t(a.M) * a.N;
  const float* p = partials + size_t(m) * a.N + n;
  const float back = __builtin_fabsf(undo[m]);
  typedef float vec __attribute__((ext_vector_type(V)));
  constexpr int kBatch = 8;  // planes in flight together
  vec t = {};
  for (int s0 = 0; s0 < splits; s0 += kBatch) {
    vec in[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i)
      if (s0 + i < splits) in[i] = *reinterpret_cast<const vec*>(p + size_t(s0 + i) * plane);
#pragma unroll
    for (int i = 0; i < kBatch; ++i)
      if (s0 + i < splits) t = s0 + i == 0 ? in[i] : t + in[i];
  }
  const float* b = static_cast<const float*>(a.bias);
  float* y = static_cast<float*>(a.y) + m * a.ldy + n;
  t *= back;
#pragma unroll
  for (int r = 0; r < V; ++r) y[r] = b ? t[r] + b[n + r] : t[r];
}

// The same for fused gate/up columns: eight of them, four outputs, per thread (N % 8 == 0).
__global__ void __launch_bounds__(64) f32_reduce_swiglu_kernel(const LinearArgs a, const float* partials,
                                                               const float* undo, int splits) {
  const int64_t nv = a.N / 8;
  const int64_t e = int64_t(blockIdx.x) * 64 + threadIdx.x;
  if (e >= a.M * nv) return;
  const int64_t m = e / nv, n = (e - m * nv) * 8;
  const size_t plane = size_t(a.M) * a.N;
  const float* p = partials + size_t(m) * a.N + n;
  const float back = __builtin_fabsf(undo[m]);
  f32x4 t = *reinterpret_cast<const f32x4*>(p), u = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll 4
  for (int s = 1; s < splits; ++s) {
    t += *reinterpret_cast<const f32x4*>(p + size_t(s) * plane);
    u += *reinterpret_cast<const f32x4*>(p + size_t(s) * plane + 4);
  }
  t *= back;
  u *= back;
  const float* b = static_cast<const float*>(a.bias);
  float* y = static_cast<float*>(a.y) + m * a.ldy + n / 2;
#pragma unroll
  for (int r = 0; r < 4; ++r) y[r] = swiglu<ActF32>(b ? t[r] + b[n + r] : t[r], b ? u[r] + b[n + 4 + r] : u[r]);
}

size_t align256(size_t b) { return (b + 255) / 256 * 256; }

struct Plan {
  int tt = 0;  // 0: not taken: a group or K of another size, or pieces beyond 32-bit offsets
  int splits = 1;
  int tiles_m = 0, tiles_n = 0;
  int64_t mpad = 0;
  size_t pieces = 0, sums = 0, undo = 0, partials = 0;
  size_t total() const { return pieces + sums + undo + partials; }
};

// Tile height and K splits from a small time model, its constants measured on MI355X (sweeps of both
// heights and 1 - 16 splits over 12 - 1024 tokens of 4096 - 28672 features): a stage of 64 (32) tokens
// takes 1.4 (0.95) us with one workgroup on a CU and 2.5 (1.6) us for both of two; a workgroup's start
// and end cost about three stages; a split writes and re-reads its fp32 partial sums at 3.7 TB/s and
// adds a launch.
Plan plan(int64_t M, int64_t N, int64_t K, int64_t group) {
  Plan best;
  if (M < 1 || N < 1 || K < 2 * kBK || group % kBK != 0 || K % (2 * kBK) != 0) return best;
  const int64_t units = K / kBK / 2;
  double best_t = 1e30;
  for (int tt : {2, 1}) {
    const int64_t tm = (M + 32 * tt - 1) / (32 * tt), tn = (N + kBN - 1) / kBN;
    if (tm * tn > (int64_t(1) << 24)) continue;
    for (int sp = 1; sp <= kMaxSplits && sp <= units; ++sp) {
      const int64_t wgs = tm * tn * sp;
      const double stages = double((units + sp - 1) / sp * 2);
      const double full = double(wgs / 512), rest = double(wgs % 512);
      const double one = tt == 2 ? 1.4 : 0.95, two = tt == 2 ? 2.5 : 1.6;
      const double rounds = full * two + (rest == 0 ? 0.0 : rest <= 256 ? one : two);
      const double red = sp > 1 ? 2.0 * sp * double(M) * double(N) * 4.0 / 3.7e6 + 4.0 : 0.0;
      const double t = rounds * (stages + 3) + red;
      if (t < best_t * 0.97) {
        best_t = t;
        best.tt = tt;
        best.splits = sp;
        best.tiles_m = int(tm);
        best.tiles_n = int(tn);
      }
    }
  }
  if (best.tt) {
    best.mpad = int64_t(best.tiles_m) * 32 * best.tt;
    best.pieces = align256(size_t(best.mpad) * K * 6);
    if (best.pieces >= size_t(1) << 31) return Plan{};
    best.sums = align256(size_t(best.mpad) * (K / kBK) * 4);
    best.undo = align256(size_t(best.mpad) * 4);
    best.partials = best.splits > 1 ? align256(size_t(best.splits) * M * N * 4) : 0;
  }
  return best;
}

template <int TT, int FMT>
void launch_tt(const LinearArgs& a, const GemmArgs& g, hipStream_t stream) {
  const dim3 grid(unsigned(g.tiles_m) * unsigned(g.tiles_n) * unsigned(g.splits)), block(kThreads);
  const bool pairs = a.group % (2 * kBK) == 0;
  if (a.symmetric) {
    if (pairs)
      hipLaunchKernelGGL((f32_gemm_kernel<TT, 2, FMT, false>), grid, block, 0, stream, a, g);
    else
      hipLaunchKernelGGL((f32_gemm_kernel<TT, 1, FMT, false>), grid, block, 0, stream, a, g);
  } else {
    if (pairs)
      hipLaunchKernelGGL((f32_gemm_kernel<TT, 2, FMT, true>), grid, block, 0, stream, a, g);
    else
      hipLaunchKernelGGL((f32_gemm_kernel<TT, 1, FMT, true>), grid, block, 0, stream, a, g);
  }
}

}  // namespace

// The decode kernels take the pieces of 16 tokens (groups of 64) or 21 in one pass over the weight;
// past that they need a second, and this GEMM is faster. Groups of 64, us on the decode kernels against
// here: 24 tokens qkv 29.6 / 23.7, o 26.3 / 22.3, gate_up 68.9 / 48.8, down 50.8 / 32.4; 12 tokens (one
// pass) 16.8 / 22.5, 14.9 / 20.5, 37.3 / 46.4, 26.8 / 30.7.
int64_t f32_gemm_min_tokens(int64_t group) { return f32_chunk_tokens(group) + 1; }

size_t f32_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K, int64_t group) {
  return plan(M, N, K, group).total();
}

hipError_t launch_linear_f32_gemm(const LinearArgs& a, hipStream_t stream, bool* fits) {
  *fits = false;
  if (a.act != kDtF32 || a.M < 1 || a.N < 1) return hipSuccess;
  if (a.epilogue != kEpiNone && (a.epilogue != kEpiSwiglu || a.N % 8 != 0)) return hipSuccess;
  // Pairs of 64-wide stages, each within one group; 16-byte aligned code rows; 32-bit buffer offsets.
  if (a.ldq % 16 != 0 || reinterpret_cast<uintptr_t>(a.qw) % 16 != 0) return hipSuccess;
  if (a.N * a.ldq >= (int64_t(1) << 31) || a.N * a.G * 4 >= (int64_t(1) << 31)) return hipSuccess;
  const Plan p = plan(a.M, a.N, a.K, a.group);
  if (p.tt == 0) return hipSuccess;
  if (!a.workspace || a.workspace_bytes < p.total() || reinterpret_cast<uintptr_t>(a.workspace) % 256 != 0)
    return hipSuccess;
  *fits = true;
  uint8_t* ws = static_cast<uint8_t*>(a.workspace);
  GemmArgs g;
  g.pieces = ws;
  float* sums = a.symmetric ? nullptr : reinterpret_cast<float*>(ws + p.pieces);
  g.sums = sums;
  g.mpad = p.mpad;
  g.tiles_m = p.tiles_m;
  g.tiles_n = p.tiles_n;
  g.splits = p.splits;
  float* undo = reinterpret_cast<float*>(ws + p.pieces + p.sums);
  g.undo = undo;
  g.partials = reinterpret_cast<float*>(ws + p.pieces + p.sums + p.undo);
  const float* x = static_cast<const float*>(a.x);
  // Up to 128 rows: several workgroups per row, of 256 threads where four rounds of them cover it.
  const int64_t chunks = a.K / 8;
  const int64_t threads = std::min<int64_t>(a.M <= 128 && chunks <= 1024 ? 256 : kSplitThreads, (chunks + 63) / 64 * 64);
  const int64_t rounds = (chunks + threads - 1) / threads;
  int parts = 1;
  while (a.M <= 128 && 2 * parts <= rounds) parts *= 2;
  const dim3 sgrid(unsigned(a.M), unsigned(parts)), sblock{unsigned(threads)};
  if (a.ldx % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0)
    hipLaunchKernelGGL(split_tiles_kernel<true>, sgrid, sblock, 0, stream, x, a.ldx, p.mpad,
                       int(a.K / kBK), parts, ws, sums, undo);
  else
    hipLaunchKernelGGL(split_tiles_kernel<false>, sgrid, sblock, 0, stream, x, a.ldx, p.mpad,
                       int(a.K / kBK), parts, ws, sums, undo);
  if (a.fmt == kNibble)
    p.tt == 2 ? launch_tt<2, kNibble>(a, g, stream) : launch_tt<1, kNibble>(a, g, stream);
  else
    p.tt == 2 ? launch_tt<2, kByte>(a, g, stream) : launch_tt<1, kByte>(a, g, stream);
  if (p.splits > 1 && a.epilogue == kEpiSwiglu) {
    hipLaunchKernelGGL(f32_reduce_swiglu_kernel, dim3(unsigned((a.M * (a.N / 8) + 63) / 64)), dim3(64), 0, stream, a,
                       g.partials, undo, p.splits);
  } else if (p.splits > 1) {
    const bool vec = a.N % 4 == 0;
    const int64_t threads = a.M * (vec ? a.N / 4 : a.N);
    const dim3 rgrid(unsigned((threads + 63) / 64));
    if (vec)
      hipLaunchKernelGGL(f32_reduce_kernel<4>, rgrid, dim3(64), 0, stream, a, g.partials, undo, p.splits);
    else
      hipLaunchKernelGGL(f32_reduce_kernel<1>, rgrid, dim3(64), 0, stream, a, g.partials, undo, p.splits);
  }
  return hipGetLastError();
}

}  // namespace llmopt

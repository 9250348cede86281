// Prefill attention straight from the block table: PagedAttention.forward with several query tokens
// per sequence (src/llmopt/attention/paged_attention.py:145-290, the causal mask of :207-216), which
// gathers K/V into a padded tensor, repeats each KV head for its query heads and runs matmul /
// softmax / matmul. Cache layout and key rules as in the decode attention: token t of sequence s
// is slot t % block_size of block block_ids[s, t / block_size], a key iff t < context_lens[s] and
// that block id names a block; query token j sits at position context_lens[s] - q_len + j and sees
// the keys up to its own position.
//
// A workgroup of four waves owns 128 query rows of one (sequence, KV head): 128 / GQ consecutive
// tokens x the GQ query heads that share the KV head, 32 rows per wave. It walks the keys in tiles
// of 64, whose K and V rows (whole 2 HD-byte rows, gathered by slot) come into LDS by direct loads
// one tile ahead and serve all 128 rows. Per tile and wave, all on v_mfma_f32_32x32x16:
//   * S^T = K Q^T (A: 32 keys x 16 dims from LDS, B: 16 dims x 32 rows, in registers): lane l holds
//     row l % 32 against 16 keys per block of 32 -- keys 8 q + 4 (l / 32) + r -- so a row's softmax
//     takes one exchange between the two lane halves;
//   * online softmax in fp32, in powers of two; the probabilities, rounded to the cache dtype as the
//     reference's softmax output is, are summed in fp32 as rounded (v_dot2_f32: the weights of a row add up
//     to one) and are the B operand of
//   * O^T += V^T P^T as they lie: the MFMA sums over k, so the operands only have to agree that slot
//     4 a + r of lane half h is key 8 a + 4 h + r of the slice. V^T comes from the row-major V tile by
//     transposing LDS reads (ds_read_b64_tr_b16: of 16 lanes, lane 4 r + c reads dims 4 c .. of key r
//     and lane i receives dim i of keys 0 .. 3).
// What bounds it: long walks by issue -- per tile a wave has 32 MFMAs (1024 cycles of the matrix pipe), 48 LDS
// reads and about 300 VALU operations with 32 exponentials among them (1700 cycles), and two waves per SIMD
// (231 registers, two workgroups of 64 KB of LDS per CU) overlap them; short prompts by the query's and
// output's bytes and a workgroup's start (table entry, then keys).
// Measured (MI355X, bf16, 32 heads / 8 KV heads of 128; us against 16-row blocks per wave that read
// their keys from L1 / L2): 32 prompts of 512 tokens 139 / 448 (494 TFLOP/s), 4 of 2048 178 / 410 (772),
// one of 512 18.9 / 55.4, 8 chunks of 100 after 512 cached 21.1 / 70.8, 64 of 5 after 295 18.7 / 25.1.
// The roundings: a probability is rounded least where it is near 1, so the maximum moves in steps of 16, 16 and
// 32 keys in the first tile, where most maxima are, and once per tile after it. 2-norm error against float64 in
// that order, here / one step per tile and the sum of unrounded probabilities / that other kernel (steps of 16,
// unrounded): 1.935 / 1.970 / 1.947, 1.994 / 2.022 / 2.002, 1.929 / 1.962 / 1.938, 2.181 / 2.191 / 2.179, 2.151 /
// 2.169 / 2.149 e-3. It costs 5 % of the first figure, 2 % of the second.
//
// K chunks are XOR-swizzled by the row's low bits (16 rows of one chunk fall on distinct banks), V
// chunks by the key's low bits in steps of 64 bytes (the four keys of a transposing read do).
#include "qcommon.hpp"
#include "qkernels.hpp"

namespace llmopt {
namespace {

constexpr int kThreads = 256;
constexpr int kRows = 128;  // query rows per workgroup
constexpr int kKeys = 64;   // keys per tile
constexpr float kLog2e = 1.44269504088896340736f;

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

template <class C>
struct Mfma;
template <>
struct Mfma<ActBf16> {
  __device__ static f32x16 run(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  }
  __device__ static uint32_t pack(float lo, float hi) {
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  }
  __device__ static float add_pair(uint32_t pair, float sum) {  // sum + both halves, in fp32
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), __builtin_bit_cast(bf16x2, 0x3F803F80u),
                                           sum, false);
  }
};
template <>
struct Mfma<ActF16> {
  __device__ static f32x16 run(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
  }
  __device__ static uint32_t pack(float lo, float hi) {
    return uint32_t(__builtin_bit_cast(uint16_t, _Float16(lo))) |
           (uint32_t(__builtin_bit_cast(uint16_t, _Float16(hi))) << 16);
  }
  __device__ static float add_pair(uint32_t pair, float sum) {
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, pair), __builtin_bit_cast(f16x2, 0x3C003C00u), sum, false);
  }
};

// Four 16-bit elements of one column: see the transposing reads above.
__device__ __forceinline__ u32x2 read_transposed(const uint8_t* p) {
  return __builtin_bit_cast(u32x2,
                            __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p));
}

// v of this lane and of the lane 32 away, in that order for the lower half.
__device__ __forceinline__ void halves(float v, float& lo, float& hi) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  lo = __uint_as_float(r[0]);
  hi = __uint_as_float(r[1]);
}

// Position of 16-byte chunk c within row r of a K or V tile.
template <int HD>
__device__ __forceinline__ int k_chunk(int r, int c) {
  return HD == 128 ? c ^ (r & 15) : c ^ ((r >> 1) & 7);
}
template <int HD>
__device__ __forceinline__ int v_chunk(int r, int c) {
  return HD == 128 ? c ^ ((r & 3) << 2) : c ^ ((r & 2) << 1);
}

template <class C, int HD, int GQ>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
    paged_prefill_kernel(const PagedDecodeArgs a) {
  constexpr int kTok = kRows / GQ;          // query tokens per workgroup
  constexpr int kCh = HD / 8;               // 16-byte chunks per row
  constexpr int kRowBytes = HD * 2;
  constexpr int kTile = kKeys * kRowBytes;  // one K (or V) tile
  constexpr int kRpl = 64 / kCh;            // rows per direct load (1 KB)
  constexpr int kLoads = 16 / kRpl;         // direct loads per wave and tile, of K and of V: 16 rows
  constexpr int kS = HD / 16;               // 16-dim slices of the scores
  constexpr int kD = HD / 32;               // 32-dim blocks of the output
  __shared__ __attribute__((aligned(16))) uint8_t kv[2][2 * kTile];  // double buffer: K, V

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, half = lane >> 5;
  // Workgroups in the order (KV head, query block, sequence), a sequence's last blocks (the longest walks)
  // first: those that run together walk the keys of a few sequences, which stay in L2. The KV heads vary
  // fastest, so with a multiple of eight of them a sequence's keys of one head are in one XCD's L2.
  const uint32_t kv_heads = uint32_t(a.kv_heads), seqs = uint32_t(a.num_seqs);
  const uint32_t blocks = gridDim.x / (kv_heads * seqs);
  const uint32_t rest = blockIdx.x / kv_heads;
  const int64_t kvh = blockIdx.x - rest * kv_heads, s = rest / blocks;
  const int j0 = int(blocks - 1 - rest % blocks) * kTok;
  const int q_len = int(a.q_len);
  const int ctx = int(a.context_lens[s]);
  const int base = ctx - q_len;  // position of query token 0
  const int tok = j0 + (32 * wave + col) / GQ;
  const bool row_ok = tok < q_len;
  const int q_pos = row_ok ? base + tok : -1;
  const int first_pos = base + j0 + 32 * wave / GQ;  // the wave's first and last positions
  const int wave_last = j0 + 32 * wave / GQ < q_len ? base + min(j0 + (32 * wave + 31) / GQ, q_len - 1) : -1;
  // The workgroup's keys: t < t_end, within the table (its width in tokens stays below 2^31).
  const int t_end = max(0, min(base + min(j0 + kTok, q_len), int(a.ldb * a.block_size)));
  const int n_tiles = (t_end + kKeys - 1) / kKeys;

  // ---- the wave's query rows: the B operand, dims 16 m + 8 half .. of row col ----
  // Rows of the cache dtype come in whole by direct loads into the second tile buffer (q_direct, checked on
  // the host: 16-byte aligned rows, a workgroup's rows within 2 GiB); other dtypes and alignments convert.
  u32x4 qf[kS];
  if (a.q_direct) {
    const auto qrs = make_rsrc(static_cast<const uint16_t*>(a.query) + s * a.q_seq_stride + j0 * a.q_tok_stride +
                                   kvh * GQ * a.q_head_stride, 0x7FFFFFFFu);
#pragma unroll
    for (int i = 0; i < 32 / kRpl; ++i) {
      const int r = kRpl * i + lane / kCh;  // of the wave's 32
      const int t = min(j0 + (32 * wave + r) / GQ, q_len - 1) - j0;  // rows past the chunk repeat its last token
      load_lds16_cached(qrs, kv[1] + (32 * wave + kRpl * i) * kRowBytes,
                        uint32_t((t * a.q_tok_stride + r % GQ * a.q_head_stride) * 2) +
                            16 * k_chunk<HD>(r, lane % kCh), 0);
    }
  } else {
    const int64_t q0 = s * a.q_seq_stride + int64_t(row_ok ? tok : 0) * a.q_tok_stride +
                       (kvh * GQ + col % GQ) * a.q_head_stride + 8 * half;
    float x[kS][8];
    if (a.q_dtype == kDtF32) {
      const float* q = static_cast<const float*>(a.query) + q0;
      if (a.q_vec) {
#pragma unroll
        for (int m = 0; m < kS; ++m) {
          const f32x4 v0 = *reinterpret_cast<const f32x4*>(q + 16 * m);
          const f32x4 v1 = *reinterpret_cast<const f32x4*>(q + 16 * m + 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) x[m][e] = v0[e], x[m][e + 4] = v1[e];
        }
      } else {
#pragma unroll
        for (int m = 0; m < kS; ++m)
#pragma unroll
          for (int e = 0; e < 8; ++e) x[m][e] = q[16 * m + e];
      }
    } else {
      const uint16_t* q = static_cast<const uint16_t*>(a.query) + q0;
      const bool f16 = a.q_dtype == kDtF16;
      auto cvt = [&](uint16_t h) { return f16 ? f16_to_f32(h) : bf16_to_f32(h); };
      if (a.q_vec) {
#pragma unroll
        for (int m = 0; m < kS; ++m) {
          const u32x4 w = *reinterpret_cast<const u32x4*>(q + 16 * m);
          const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) x[m][2 * e] = cvt(uint16_t(ws[e])), x[m][2 * e + 1] = cvt(uint16_t(ws[e] >> 16));
        }
      } else {
#pragma unroll
        for (int m = 0; m < kS; ++m)
#pragma unroll
          for (int e = 0; e < 8; ++e) x[m][e] = cvt(q[16 * m + e]);
      }
    }
#pragma unroll
    for (int m = 0; m < kS; ++m) {
      uint32_t w[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        w[e] = row_ok ? uint32_t(C::store(x[m][2 * e])) | (uint32_t(C::store(x[m][2 * e + 1])) << 16) : 0u;
      qf[m] = u32x4{w[0], w[1], w[2], w[3]};
    }
  }

  // ---- key tiles ----
  const uint32_t row_stride = uint32_t(a.kv_heads * HD * 2);  // bytes between two slots
  const uint32_t cache_bytes = uint32_t(a.num_blocks * a.block_size) * row_stride;
  const auto krs = make_rsrc(a.key_cache, cache_bytes);
  const auto vrs = make_rsrc(a.value_cache, cache_bytes);
  const auto trs = make_rsrc(a.block_ids + s * a.ldb, uint32_t(a.ldb * 4));
  const uint32_t head_off = uint32_t(kvh * HD * 2);
  const uint32_t bsz = uint32_t(a.block_size), ldb = uint32_t(a.ldb), nblk = uint32_t(a.num_blocks);
  // Block sizes are powers of two in practice: a shift then, else the division (uniform branch).
  const bool pow2 = (bsz & (bsz - 1)) == 0;
  const int sh = __builtin_ctz(bsz);
  auto block_of = [&](uint32_t t) -> uint32_t { return pow2 ? t >> sh : t / bsz; };
  uint32_t k_off[kLoads], v_off_load[kLoads];  // which chunk of its row a lane brings in, per load
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int r = wave * 16 + kRpl * i + lane / kCh;
    k_off[i] = 16 * k_chunk<HD>(r, lane % kCh);
    v_off_load[i] = 16 * v_chunk<HD>(r, lane % kCh);
  }
  // Lane l looks up key t0 + l: the table entry a tile ahead of the slot row it becomes.
  auto fetch_entry = [&](int t0) -> int32_t {
    const uint32_t bi = block_of(uint32_t(t0 + lane));
    return int32_t(__builtin_amdgcn_raw_buffer_load_b32(trs, int((bi < ldb ? bi : 0u) * 4u), 0, kLoadPolicy));
  };
  // Starts the loads of the tile at t0 into buffer b; returns its valid keys. Rows that are no keys
  // read slot row 0: their scores are dropped, and their V rows cleared before they are used.
  auto fetch_tile = [&](int t0, int32_t entry, int b) -> uint64_t {
    const uint32_t t = uint32_t(t0 + lane);
    const uint32_t bi = block_of(t);
    const bool ok = int(t) < t_end && bi < ldb && entry >= 0 && uint32_t(entry) < nblk;
    const uint32_t slot = (ok ? uint32_t(entry) * bsz + (t - bi * bsz) : 0u) * row_stride;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int r = wave * 16 + kRpl * i + lane / kCh;  // this lane's row of the load
      const uint32_t row = uint32_t(__shfl(int(slot), r, 64));
      uint8_t* dst = kv[b] + (wave * 16 + kRpl * i) * kRowBytes;
      load_lds16_cached(krs, dst, row + k_off[i], head_off);
      load_lds16_cached(vrs, dst + kTile, row + v_off_load[i], head_off);
    }
    return __builtin_amdgcn_ballot_w64(ok);
  };

  const float neg_inf = -__int_as_float(0x7F800000);
  // Probabilities are 2^(score c - m c), one fma and one exponential per score. c has to be positive for
  // the maximum of the scores to be that of the exponents: a negative scale moves into the query rows, a
  // zero one becomes too small to matter.
  const bool capped = a.softcap > 0.0f;
  const float magnitude = __builtin_fabsf(a.scale) * kLog2e;
  const float c2 = capped ? kLog2e : magnitude > 0.0f ? magnitude : 1e-30f;
  const uint32_t q_sign = !capped && a.scale < 0.0f ? 0x80008000u : 0u;
  // Per row: the running maximum m_run (mc = m_run c2, 0 without keys so far), and this lane's share of
  // the sum. (Letting the maximum lag by up to eight powers of two, so that most tiles skip the rescale, was
  // 2 - 10 % faster and 3 - 6 % less exact: the largest probabilities are then no longer near 1, which bf16
  // rounds least.)
  float m_run = neg_inf, mc = 0.0f, l_run = 0.0f;
  f32x16 o[kD];
#pragma unroll
  for (int d = 0; d < kD; ++d)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[d][v] = 0.0f;

  // Per-lane LDS addresses: K row col of a block; V key 4 half + (lane % 16) / 4, dims 16 ((lane / 16) %
  // 2) + 4 (lane % 4) of a block (chunk 2 ((lane / 16) % 2) + (lane % 4) / 2, its half lane % 2).
  const int vkey = 4 * half + ((lane & 15) >> 2);
  const int vc = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
  const int v_off = vkey * kRowBytes + 8 * (lane & 1);

  auto compute = [&](const uint8_t* kt, int t0, uint64_t mask) {
    const uint8_t* vt = kt + kTile;
    f32x16 sc[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int v = 0; v < 16; ++v) sc[kb][v] = 0.0f;
#pragma unroll
      for (int m = 0; m < kS; ++m) {
        const u32x4 kf = *reinterpret_cast<const u32x4*>(kt + (32 * kb + col) * kRowBytes +
                                                         16 * k_chunk<HD>(col, 2 * m + half));
        sc[kb] = Mfma<C>::run(kf, qf[m], sc[kb]);
      }
    }
    if (capped) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int v = 0; v < 16; ++v) sc[kb][v] = tanhf(sc[kb][v] * a.scale / a.softcap) * a.softcap;
    }
    if (mask != ~uint64_t(0) || t0 + kKeys - 1 > first_pos) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        // Bit 8 q + r: key 8 q + 4 half + r of the block is a key at or before this row's token.
        const int room = q_pos - t0 - 32 * kb - 4 * half;
        const uint32_t bits = (uint32_t(mask >> (32 * kb)) >> (4 * half)) &
                              (room >= 31 ? ~0u : room < 0 ? 0u : (2u << room) - 1u);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const uint32_t keep = uint32_t(int32_t(bits << (31 - (8 * (v / 4) + v % 4))) >> 31);
          sc[kb][v] = __uint_as_float((__float_as_uint(sc[kb][v]) & keep) | (__float_as_uint(neg_inf) & ~keep));
        }
      }
    }
    // Slices of 16 keys: slice i is v = 8 (i % 2) .. + 7 of block i / 2. The running maximum moves before a
    // tile's first slice, in the first tile also before its second and third.
    float top[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      top[i] = neg_inf;
#pragma unroll
      for (int v = 0; v < 8; ++v) top[i] = fmaxf(top[i], sc[i / 2][8 * (i % 2) + v]);
    }
    top[2] = fmaxf(top[2], top[3]);
    if (t0 > 0) top[0] = fmaxf(fmaxf(top[0], top[1]), top[2]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u32x4 vf[kD];
#pragma unroll
      for (int d = 0; d < kD; ++d) {
        // Keys 16 i + vkey and 8 further: both have vkey's low bits, so one swizzle.
        const uint8_t* p0 = vt + 16 * i * kRowBytes + v_off + 16 * v_chunk<HD>(vkey, 4 * d + vc);
        const u32x2 lo = read_transposed(p0), hi = read_transposed(p0 + 8 * kRowBytes);
        vf[d] = u32x4{lo.x, lo.y, hi.x, hi.y};
      }
      if (i == 0 || (t0 == 0 && i < 3)) {
        float t_lo, t_hi;
        halves(top[i], t_lo, t_hi);
        const float m_new = fmaxf(m_run, fmaxf(t_lo, t_hi));
        if (__builtin_amdgcn_ballot_w64(m_new > m_run)) {
          const float mc_new = m_new == neg_inf ? 0.0f : m_new * c2;
          const float alpha = m_run == neg_inf ? 0.0f : __builtin_amdgcn_exp2f(mc - mc_new);
          m_run = m_new;
          mc = mc_new;
          if (i > 0 || t0 > 0) {
            l_run *= alpha;
#pragma unroll
            for (int d = 0; d < kD; ++d)
#pragma unroll
              for (int v = 0; v < 16; ++v) o[d][v] *= alpha;
          }
        }
      }
      float p[8];
#pragma unroll
      for (int v = 0; v < 8; ++v)
        p[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[i / 2][8 * (i % 2) + v], c2, -mc));
      const u32x4 pf = {Mfma<C>::pack(p[0], p[1]), Mfma<C>::pack(p[2], p[3]), Mfma<C>::pack(p[4], p[5]),
                        Mfma<C>::pack(p[6], p[7])};
      l_run += Mfma<C>::add_pair(pf.w, Mfma<C>::add_pair(pf.z, Mfma<C>::add_pair(pf.y, Mfma<C>::add_pair(pf.x, 0.0f))));
#pragma unroll
      for (int d = 0; d < kD; ++d) o[d] = Mfma<C>::run(vf[d], pf, o[d]);
    }
  };

  if (n_tiles > 0) {
    uint64_t mask = fetch_tile(0, fetch_entry(0), 0);
    int32_t entry = fetch_entry(kKeys);
    if (a.q_direct) {
      wait_vmcnt<2 * kLoads + 1>();  // the query rows: this tile's loads and the entries came after them
#pragma unroll
      for (int m = 0; m < kS; ++m)
        qf[m] = *reinterpret_cast<const u32x4*>(kv[1] + (32 * wave + col) * kRowBytes +
                                                16 * k_chunk<HD>(col, 2 * m + half));
    }
#pragma unroll
    for (int m = 0; m < kS; ++m) qf[m] ^= q_sign;
    for (int i = 0; i < n_tiles; ++i) {
      const int t0 = i * kKeys, b = i & 1;
      wait_vmcnt<0>();  // this wave's rows of tile i, and the next entries
      if (mask != ~uint64_t(0)) {
#pragma unroll
        for (int l = 0; l < kLoads; ++l) {
          const int r = wave * 16 + kRpl * l + lane / kCh;
          if (!((mask >> r) & 1u))
            *reinterpret_cast<u32x4*>(kv[b] + kTile + r * kRowBytes + 16 * (lane % kCh)) = u32x4{0u, 0u, 0u, 0u};
        }
      }
      wait_lgkmcnt0();  // the clearing stores, and this wave's reads of the buffer that is refilled next
      __builtin_amdgcn_s_barrier();
      uint64_t next = 0;
      if (i + 1 < n_tiles) {
        const int32_t e = entry;
        entry = fetch_entry(t0 + 2 * kKeys);
        next = fetch_tile(t0 + kKeys, e, b ^ 1);
      }
      if (t0 <= wave_last) compute(kv[b], t0, mask);
      mask = next;
    }
  }

  if (n_tiles == 0) wait_vmcnt<0>();  // query rows nobody needs: they land before the LDS is used again

  // ---- output: row col, dims 32 d + 8 q + 4 half + r ----
  float l_lo, l_hi;
  halves(l_run, l_lo, l_hi);
  const float l = l_lo + l_hi;
  const bool any = l > 0.0f;  // false without keys, and for a NaN sum: zeros, as the reference's nan_to_num gives
  const float inv = 1.0f / l;
  auto value = [&](float v) { return any ? v * inv : 0.0f; };
  const int64_t out0 = s * a.out_seq_stride;
  const int64_t h0 = kvh * GQ;
  const bool vec = a.out_dtype != kDtF32 &&
                   ((a.out_seq_stride | a.out_tok_stride | a.out_head_stride) % 8 == 0) &&
                   reinterpret_cast<uintptr_t>(a.out) % 16 == 0;
  const bool f16 = a.out_dtype == kDtF16;
  auto narrow = [&](float v) -> uint32_t { return f16 ? f32_to_f16_rne(v) : f32_to_bf16_rne(v); };
  // Two outputs in one word: the hardware's pair conversion for the cache dtype, the usual case.
  const bool same = a.out_dtype == C::id;
  if (vec) {
    // Through LDS, 32 rows of the wave at a time, so that the stores are whole rows.
    wait_lgkmcnt0();
    __builtin_amdgcn_s_barrier();  // every wave is past its last tile
    uint8_t* tile = kv[0] + wave * 32 * kRowBytes;
    auto stage_rows = [&](auto pair) {
#pragma unroll
      for (int d = 0; d < kD; ++d)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const u32x2 w = {pair(value(o[d][4 * q]), value(o[d][4 * q + 1])),
                           pair(value(o[d][4 * q + 2]), value(o[d][4 * q + 3]))};
          *reinterpret_cast<u32x2*>(tile + col * kRowBytes + 16 * k_chunk<HD>(col, 4 * d + q) + 8 * half) = w;
        }
    };
    if (same)
      stage_rows([](float lo, float hi) { return Mfma<C>::pack(lo, hi); });
    else
      stage_rows([&](float lo, float hi) { return narrow(lo) | (narrow(hi) << 16); });
    wait_lgkmcnt0();  // the wave's own tile: no barrier
#pragma unroll
    for (int i = 0; i < 32 / kRpl; ++i) {
      const int r = kRpl * i + lane / kCh, c = lane % kCh;
      const int t = j0 + (32 * wave + r) / GQ;
      if (t >= q_len) continue;
      const u32x4 w = *reinterpret_cast<const u32x4*>(tile + r * kRowBytes + 16 * k_chunk<HD>(r, c));
      uint16_t* dst = static_cast<uint16_t*>(a.out) + out0 + int64_t(t) * a.out_tok_stride +
                      (h0 + r % GQ) * a.out_head_stride + 8 * c;
      *reinterpret_cast<u32x4*>(dst) = w;
    }
    return;
  }
  if (!row_ok) return;
  const int64_t at = out0 + int64_t(tok) * a.out_tok_stride + (h0 + col % GQ) * a.out_head_stride + 4 * half;
#pragma unroll
  for (int d = 0; d < kD; ++d)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int64_t i = at + 32 * d + 8 * (v / 4) + v % 4;
      const float val = value(o[d][v]);
      if (a.out_dtype == kDtF32)
        static_cast<float*>(a.out)[i] = val;
      else
        static_cast<uint16_t*>(a.out)[i] = uint16_t(narrow(val));
    }
}

template <class C, int HD, int GQ>
void launch_group(const PagedDecodeArgs& a, hipStream_t stream) {
  constexpr int kTok = kRows / GQ;
  const dim3 grid(unsigned(a.kv_heads * a.num_seqs * ((a.q_len + kTok - 1) / kTok)));
  hipLaunchKernelGGL((paged_prefill_kernel<C, HD, GQ>), grid, dim3(kThreads), 0, stream, a);
}

template <class C, int HD>
hipError_t launch_hd(const PagedDecodeArgs& a, hipStream_t stream) {
  switch (a.num_heads / a.kv_heads) {
    case 1: launch_group<C, HD, 1>(a, stream); break;
    case 2: launch_group<C, HD, 2>(a, stream); break;
    case 4: launch_group<C, HD, 4>(a, stream); break;
    case 8: launch_group<C, HD, 8>(a, stream); break;
    case 16: launch_group<C, HD, 16>(a, stream); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_paged_prefill(const PagedDecodeArgs& a, hipStream_t stream) {
  if (a.num_seqs == 0 || a.q_len == 0) return hipSuccess;
  if (a.cache_dtype == kDtBf16)
    return a.head_dim == 128 ? launch_hd<ActBf16, 128>(a, stream) : launch_hd<ActBf16, 64>(a, stream);
  return a.head_dim == 128 ? launch_hd<ActF16, 128>(a, stream) : launch_hd<ActF16, 64>(a, stream);
}

}  // namespace llmopt

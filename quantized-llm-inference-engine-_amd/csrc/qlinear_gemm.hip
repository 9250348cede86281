// The prefill GEMM's plan and launch, its bf16 instantiations (the kernel: qlinear_gemm.hpp), and the
// fixed-order reduction of K splits.
#include "qlinear_gemm.hpp"

namespace llmopt {
namespace {

// Threads per workgroup of the reduction kernel: small workgroups spread a few thousand threads
// over every CU.
constexpr int kReduceThreads = 64;
// Splits whose partial sums a thread loads before adding any of them: the loads of a batch are
// in flight together instead of one round trip per split (down at 16 tokens, 14 splits: 5.4 us
// for the reduction with one load at a time). Up to eight splits, which is all the GEMM has, a batch is
// eight: sixteen take registers that long batches miss (o at 900 tokens 58.6 us against 62.2, qkv at
// 640 58.4 / 61.5). More, only in 8-bit K slices of the decode kernel, sixteen: 8-bit down at 3 - 32 tokens, 14
// splits, 0.7 - 0.9 us less per call than two batches of eight.
constexpr int kReduceBatch = 8, kReduceBatchMany = 16;

// y[m, n] = bias[n] + sum over splits, in split order, of partials[split][m][n]: four columns
// per thread. Deterministic: the order of the additions never depends on timing.
template <class Act, int BATCH>
__global__ void __launch_bounds__(kReduceThreads) splitk_reduce_kernel(const LinearArgs a, const float* partials, int splits) {
  using Raw = typename Act::raw;
  if (a.epilogue == kEpiSwiglu) {
    // One thread per output feature group of four: fused columns 8p .. 8p+7 (N % 8 == 0).
    const int64_t p8 = a.N / 8;
    const int64_t e = int64_t(blockIdx.x) * kReduceThreads + threadIdx.x;
    if (e >= a.M * p8) return;
    const int64_t m = e / p8;
    const int64_t n = (e - m * p8) * 8;
    const size_t plane = size_t(a.M) * a.N;
    const float* p = partials + size_t(m) * a.N + n;
    float g[4], u[4];
    for (int s0 = 0; s0 < splits; s0 += BATCH) {
      f32x4 tg[BATCH], tu[BATCH];
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        if (s0 + i < splits) {
          tg[i] = *reinterpret_cast<const f32x4*>(p + size_t(s0 + i) * plane);
          tu[i] = *reinterpret_cast<const f32x4*>(p + size_t(s0 + i) * plane + 4);
        }
      }
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        if (s0 + i < splits) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            g[r] = s0 + i == 0 ? tg[i][r] : g[r] + tg[i][r];
            u[r] = s0 + i == 0 ? tu[i][r] : u[r] + tu[i][r];
          }
        }
      }
    }
    const Raw* bias = static_cast<const Raw*>(a.bias);
    Raw* y = static_cast<Raw*>(a.y) + m * a.ldy + n / 2;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float gb = bias ? g[r] + Act::load(bias[n + r]) : g[r];
      const float ub = bias ? u[r] + Act::load(bias[n + 4 + r]) : u[r];
      y[r] = Act::store(swiglu<Act>(gb, ub));
    }
    return;
  }
  const int64_t n4 = (a.N + 3) / 4;
  const int64_t e = int64_t(blockIdx.x) * kReduceThreads + threadIdx.x;
  if (e >= a.M * n4) return;
  const int64_t m = e / n4;
  const int64_t n = (e - m * n4) * 4;
  const size_t plane = size_t(a.M) * a.N;
  const Raw* bias = static_cast<const Raw*>(a.bias);
  const float* p = partials + size_t(m) * a.N + n;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  if (n + 3 < a.N && a.N % 4 == 0) {
    for (int s0 = 0; s0 < splits; s0 += BATCH) {
      f32x4 t[BATCH];
#pragma unroll
      for (int i = 0; i < BATCH; ++i)
        if (s0 + i < splits) t[i] = *reinterpret_cast<const f32x4*>(p + size_t(s0 + i) * plane);
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        if (s0 + i < splits) {
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = s0 + i == 0 ? t[i][r] : v[r] + t[i][r];
        }
      }
    }
  } else {
    for (int s = 0; s < splits; ++s)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < a.N) v[r] = s == 0 ? p[s * plane + r] : v[r] + p[s * plane + r];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (n + r >= a.N) break;
    float o = v[r];
    if (bias) o += Act::load(bias[n + r]);
    put_y<Act>(a, m * a.ldy + n + r, o);
  }
}

// ---- launch plan: token-tile height (32 * TT) and K splits ----------------------------------
//
// A 256 x 256 tile is the most efficient per MFMA, but a short or narrow GEMM gives too few of
// them for 256 CUs (one workgroup per CU). Smaller token tiles raise the workgroup count at a
// higher dequantization cost per MFMA; K splits raise it at the cost of storing and re-reading
// fp32 partial sums that a second kernel adds up. The plan minimizes a simple time model:
// rounds of 256 workgroups x stages per workgroup x time per stage, plus the partial-sum
// traffic of a split, with per-stage times measured on MI355X. The heights between 128 and 256 serve
// ragged batches over wide weights, which run in one round of fewer padded tokens (gate_up with SwiGLU, us
// against 128- and 256-token tiles alone: 300 tokens 126 -> 94, 350 127 -> 104, 600 231 -> 187, 700 233 ->
// 205); only the heights 64 and 128 split K, where a grid is small.
GemmPlan plan_gemm(int64_t M, int64_t N, int64_t K, int64_t group, int fmt) {
  GemmPlan best;
  if (M < 1 || N < 1 || K % kBK != 0 || group % 32 != 0) return best;
  const int gp = group % 128 == 0 ? 2 : 1;
  const int64_t units = K / kBK / gp;
  const double stage_us[9] = {0, 0, 0.95, 0, 1.35, 1.54, 1.73, 1.92, 2.1};
  double best_t = 1e30;
  for (int tt : {8, 7, 6, 5, 4, 2}) {
    if (fmt == kByte && tt > 4) continue;  // the byte-code ring does not fit beyond the 128-token tile
    const int64_t tm = (M + 32 * tt - 1) / (32 * tt);
    const int64_t tn = (N + kBN - 1) / kBN;
    if (tm * tn > 0x7FFFFFFF / 8) continue;
    for (int sp = 1; sp <= 8; ++sp) {
      if (sp > units || (sp > 1 && tt != 4 && tt != 2)) break;  // only two heights split
      const int64_t wgs = tm * tn * sp;
      const int64_t rounds = (wgs + 255) / 256;
      const double stages = double((units + sp - 1) / sp * gp);
      // Split: write and re-read sp fp32 planes of M x N at ~4 TB/s, plus one more launch.
      const double red = sp > 1 ? 2.0 * sp * double(M) * double(N) * 4.0 / 4e6 + 3.0 : 0.0;
      const double t = double(rounds) * stages * stage_us[tt] + red;
      if (t < best_t * 0.97) {
        best_t = t;
        best.tt = tt;
        best.splits = sp;
        best.tiles_m = tm;
        best.tiles_n = tn;
      }
    }
  }
  if (best.tt) {
    best.partial_bytes = size_t(best.splits) * size_t(M) * size_t(N) * 4;
  }
  return best;
}

}  // namespace

hipError_t launch_splitk_reduce(const LinearArgs& a, const float* partials, int splits, hipStream_t stream) {
  const int64_t threads = a.epilogue == kEpiSwiglu ? a.M * (a.N / 8) : a.M * ((a.N + 3) / 4);
  const dim3 grid(unsigned((threads + kReduceThreads - 1) / kReduceThreads)), block(kReduceThreads);
  const bool many = splits > kReduceBatch;
  if (a.act == kDtBf16) {
    if (many)
      hipLaunchKernelGGL((splitk_reduce_kernel<ActBf16, kReduceBatchMany>), grid, block, 0, stream, a, partials, splits);
    else
      hipLaunchKernelGGL((splitk_reduce_kernel<ActBf16, kReduceBatch>), grid, block, 0, stream, a, partials, splits);
  } else if (many) {
    hipLaunchKernelGGL((splitk_reduce_kernel<ActF16, kReduceBatchMany>), grid, block, 0, stream, a, partials, splits);
  } else {
    hipLaunchKernelGGL((splitk_reduce_kernel<ActF16, kReduceBatch>), grid, block, 0, stream, a, partials, splits);
  }
  return hipGetLastError();
}

size_t gemm_workspace_bytes(int64_t M, int64_t N, int64_t K, int64_t group, int fmt) {
  return plan_gemm(M, N, K, group, fmt).workspace();
}

hipError_t launch_linear_gemm(const LinearArgs& a, hipStream_t stream, bool* fits) {
  *fits = false;
  if (a.act != kDtBf16 && a.act != kDtF16) return hipSuccess;
  if (a.M < 1) return hipSuccess;
  // A lane's 32 codes of a stage lie in one group; 16-byte aligned rows and activations.
  if (a.K % kBK != 0 || a.K / kBK >= 65536 || a.group % 32 != 0) return hipSuccess;
  if (a.ldq % 16 != 0 || reinterpret_cast<uintptr_t>(a.qw) % 16 != 0) return hipSuccess;
  if (a.ldx % 8 != 0 || reinterpret_cast<uintptr_t>(a.x) % 16 != 0) return hipSuccess;
  if (a.N * a.ldq >= (int64_t(1) << 31) || a.N * a.G * 4 >= (int64_t(1) << 31)) return hipSuccess;
  if (a.M * a.ldx * 2 >= (int64_t(1) << 31)) return hipSuccess;
  if (a.epilogue == kEpiSwiglu && a.N % 8 != 0) return hipSuccess;
  const GemmPlan plan = plan_gemm(a.M, a.N, a.K, a.group, a.fmt);
  if (plan.tt == 0) return hipSuccess;
  // Without a large enough workspace the plan runs unsplit (same tiles, one workgroup per tile).
  int splits = plan.splits;
  if (splits > 1 && (a.workspace == nullptr || a.workspace_bytes < plan.workspace() ||
                     reinterpret_cast<uintptr_t>(a.workspace) % 16 != 0))
    splits = 1;
  const uint32_t g = uint32_t(a.group);
  const uint32_t magic =
      g == 1 ? 0u : uint32_t((uint64_t(1) << 32) / g + ((uint64_t(1) << 32) % g != 0));
  *fits = true;
  if (a.act == kDtBf16) return launch_act<ActBf16>(a, plan, splits, stream, magic);
  return launch_gemm_f16(a, plan.tt, plan.tiles_m, plan.tiles_n, splits, stream, magic);
}

}  // namespace llmopt

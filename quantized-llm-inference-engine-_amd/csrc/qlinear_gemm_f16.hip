// The prefill GEMM's fp16 instantiations (the kernel: qlinear_gemm.hpp).
#include "qlinear_gemm.hpp"

namespace llmopt {

hipError_t launch_gemm_f16(const LinearArgs& a, int tt, int64_t tiles_m, int64_t tiles_n, int splits,
                           hipStream_t stream, uint32_t magic) {
  GemmPlan plan;
  plan.tt = tt;
  plan.splits = splits;
  plan.tiles_m = tiles_m;
  plan.tiles_n = tiles_n;
  return launch_act<ActF16>(a, plan, splits, stream, magic);
}

}  // namespace llmopt

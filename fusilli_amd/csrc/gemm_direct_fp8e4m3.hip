// Direct matrix-product kernels for fp8e4m3 operands.
#include "gemm_direct_kernel.h"

int direct_launch_fp8e4m3(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch) {
  return direct_launch_kind<GK_FP8E4M3>(ctx, p, g, batch);
}

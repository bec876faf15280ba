// Direct matrix-product kernels for fp8e5m2 operands.
#include "gemm_direct_kernel.h"

int direct_launch_fp8e5m2(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch) {
  return direct_launch_kind<GK_FP8E5M2>(ctx, p, g, batch);
}

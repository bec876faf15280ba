// Direct matrix-product kernels for bf16 operands.
#include "gemm_direct_kernel.h"

int direct_launch_bf16(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch) {
  return direct_launch_kind<GK_BF16>(ctx, p, g, batch);
}

// Direct matrix-product kernels for i8 operands.
#include "gemm_direct_kernel.h"

int direct_launch_i8(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch) {
  return direct_launch_kind<GK_I8>(ctx, p, g, batch);
}

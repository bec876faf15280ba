// Direct matrix-product kernels for f32 operands.
#include "gemm_direct_kernel.h"

int direct_launch_f32(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch) {
  return direct_launch_kind<GK_F32>(ctx, p, g, batch);
}

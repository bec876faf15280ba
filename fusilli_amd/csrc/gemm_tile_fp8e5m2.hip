// Matrix products on register-staged LDS tiles, fp8e5m2 operands.
#include "gemm_tile_kernel.h"

int tile_launch_fp8e5m2(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch) {
  return tile_launch_kind<GK_FP8E5M2>(ctx, p, g, batch);
}

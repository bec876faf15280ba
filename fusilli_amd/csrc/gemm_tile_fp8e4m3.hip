// Matrix products on register-staged LDS tiles, fp8e4m3 operands.
#include "gemm_tile_kernel.h"

int tile_launch_fp8e4m3(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch) {
  return tile_launch_kind<GK_FP8E4M3>(ctx, p, g, batch);
}

// Matrix products on register-staged LDS tiles, i8 operands.
#include "gemm_tile_kernel.h"

int tile_launch_i8(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch) {
  return tile_launch_kind<GK_I8>(ctx, p, g, batch);
}

// Matrix products on register-staged LDS tiles, bf16 operands.
#include "gemm_tile_kernel.h"

int tile_launch_bf16(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch) {
  return tile_launch_kind<GK_BF16>(ctx, p, g, batch);
}

// Convolutions on register-staged LDS tiles, bf16 operands.
#include "conv_tile_kernel.h"

int conv_tile_launch_bf16(fhip_ctx *ctx, bool dgrad, const ConvTilePlan &p, const ConvTileArgs &g) {
  return conv_tile_kind<GK_BF16>(ctx, dgrad, p, g);
}

// Convolutions on register-staged LDS tiles, f16 operands.
#include "conv_tile_kernel.h"

int conv_tile_launch_f16(fhip_ctx *ctx, bool dgrad, const ConvTilePlan &p, const ConvTileArgs &g) {
  return conv_tile_kind<GK_F16>(ctx, dgrad, p, g);
}

// Forward convolution on gathered MFMA tiles (conv_gather.hip).
#ifndef FUSILLI_AMD_CSRC_CONV_GATHER_H
#define FUSILLI_AMD_CSRC_CONV_GATHER_H

#include "common.h"

struct ConvGatherArgs {
  const char *x, *w;
  void *out;
  float *part;      // reduction cut into parts: plain sums [part][M][N]; else null
  int64_t M;        // output pixels
  int32_t N, J;     // output channels, R * S * C
  int32_t H, W, C, P, Q, S;
  int32_t pad_h, pad_w, str_h, str_w, dil_h, dil_w;
  uint32_t x_bytes; // < 2^31
  int32_t tiles_n;
  int32_t steps;    // steps of 64 per part
  int32_t y_dt, o_dt;
  DevEpilogue epi;  // rank 3: strides {0, per pixel, per channel}
};

constexpr int kConvGatherTile = 64; // pixels and channels of a tile

struct ConvGatherPlan {
  int parts; // of the reduction; 0: not this kernel
};

ConvGatherPlan conv_gather_plan(int64_t M, int64_t N, int64_t J, bool may_split);
// Fills tiles_n and steps; x and w 16-byte aligned, C a multiple of 8.
int conv_gather_launch(fhip_ctx *ctx, bool bf16, const ConvGatherPlan &p, ConvGatherArgs &a);

#endif // FUSILLI_AMD_CSRC_CONV_GATHER_H

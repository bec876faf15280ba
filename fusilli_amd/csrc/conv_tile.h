// Forward convolution and data gradient on register-staged tiles (conv_tile.hip).
#ifndef FUSILLI_AMD_CSRC_CONV_TILE_H
#define FUSILLI_AMD_CSRC_CONV_TILE_H

#include "gemm_direct_kernel.h"

constexpr int kConvTileParts = 16; // most products that one launch covers

// A product: all output pixels (forward, unit strides), or those rows and columns of DX that
// leave one remainder.
struct ConvTilePart {
  int32_t M, P, Q;      // output pixels; rows and columns of an image
  int32_t J, S;         // taps * channels; taps along W (at least 1)
  int32_t off_h, off_w; // the first tap's place under output pixel (0, 0)
  int32_t h, w;         // gradient: the remainders
  int32_t w_first, w_row, w_tap; // gradient: bytes of the first tap, to the next row of taps, to the next tap
  uint32_t magic_p, magic_q, magic_s;
  int32_t adv_s, adv_r; // 64 values on: taps of a row, whole rows of taps (and adv_c channels)
};

// (What every workgroup reads first lies together: a kernel's arguments come from the host's
// memory, a cache line at a time.)
template <int PARTS> struct ConvTileArgsOf {
  int32_t parts;
  int32_t H, W, C;      // of the gathered tensor
  int32_t str_h, str_w, dil_h, dil_w;
  int32_t adv_c;
  uint32_t magic_c;
  uint32_t x_bytes, w_bytes; // < 2^31
  int32_t w_pitch;      // gradient: bytes between the filters of W
  int32_t out_h, out_w, step_h, step_w; // gradient: DX and the strides
  ConvTilePart part[PARTS];
  DirectArgs d;
};
using ConvTileArgs = ConvTileArgsOf<kConvTileParts>;

// Microseconds that a kernel of bm x bn tiles takes, `occ` workgroups to a compute unit: what a
// workgroup does once, its slices at a pace (alone, or `shared` by those on its compute unit), a
// round's fixed part, the parts' round trip of a split, the fused chain.
struct ConvTileTimes {
  int bm, bn, teams, occ;
  double once, alone, shared, round, sum, part, fused, fused_round;
};
double conv_tile_us(const ConvTileTimes &f, const ConvTileArgs &g, int split, bool fused);

struct ConvTilePlan {
  int bm = 0, bn = 0; // 0: no plan
  int teams = 1;      // that share K; 0: the kernel for short reductions
  int splits = 1;
  double us = 0;
};

// The shortest estimate over the tiles.  `room`: bytes that the parts of a split reduction may
// take, 0: no split.
ConvTilePlan conv_tile_plan(const ConvTileArgs &g, bool dgrad, bool fused, size_t room);
size_t conv_tile_scratch(const ConvTilePlan &p, const ConvTileArgs &g);
// Fills tiles and splits and launches; `partial`: conv_tile_scratch bytes.
int conv_tile_launch(fhip_ctx *ctx, bool bf16, bool dgrad, const ConvTilePlan &p, ConvTileArgs &g, void *partial);
// Sets lean and lean_op from the fused chain in g.epi (strides 0, per pixel, per channel).
void conv_tile_lean(const fhip_epilogue &e, ConvTileArgs &g);

int conv_tile_launch_bf16(fhip_ctx *ctx, bool dgrad, const ConvTilePlan &p, const ConvTileArgs &g);
int conv_tile_launch_f16(fhip_ctx *ctx, bool dgrad, const ConvTilePlan &p, const ConvTileArgs &g);

#endif // FUSILLI_AMD_CSRC_CONV_TILE_H

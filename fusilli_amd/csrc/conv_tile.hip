// Convolutions on register-staged tiles, host side: the choice of tile and split, launches.
#include "conv_tile.h"

#include <algorithm>

namespace {

struct TileLoad {
  int64_t tiles = 0, most = 0; // of all products, of the largest
  double slices = 0;           // of all tiles
  int longest = 0;             // reduction, in slices
  TileLoad(const ConvTileTimes &f, const ConvTileArgs &g) {
    const int64_t tn = (g.d.N + f.bn - 1) / f.bn;
    for (int i = 0; i < g.parts; ++i) {
      const int64_t t = (g.part[i].M + f.bm - 1) / f.bm * tn;
      const int run = (g.part[i].J + 63) / 64;
      tiles += t, slices += (double)t * run;
      most = t > most ? t : most;
      longest = run > longest ? run : longest;
    }
  }
};

double tile_us(const ConvTileTimes &f, const TileLoad &l, bool one, int split, bool fused) {
  auto up = [](double v) { return (double)(int64_t)(v + (1.0 - 1e-9)); };
  const double load = (double)(l.tiles * split) / 256.0;
  // (the fullest compute unit decides)
  const double even = load <= f.occ ? 0.2 * load + 0.8 * up(load) : 0.7 * load + 0.3 * f.occ * up(load / f.occ);
  const double pace = std::max(f.alone * std::max(1.0, load / f.occ), f.shared * std::max(1.0, even));
  const int run = (l.longest + split - 1) / split;
  const double chain = one ? run * pace : std::max(run * f.alone, l.slices / (double)l.tiles * pace);
  double us = f.once + chain / (f.teams > 1 ? f.teams : 1) + f.round * std::max(1.0, load);
  if (fused)
    us += f.fused + f.fused_round * std::max(1.0, load);
  if (split > 1)
    us += f.sum + f.part * split * (double)(l.tiles * f.bm * f.bn) * 4e-6;
  return us;
}

} // namespace

double conv_tile_us(const ConvTileTimes &f, const ConvTileArgs &g, int split, bool fused) {
  return tile_us(f, TileLoad(f, g), g.parts == 1, split, fused);
}

// Fitted to the times of every tile at up to seven splits on 300 random layers (8 to 64 images
// of 7 to 64 pixels a side, 32 to 512 channels, filters of 1, 3 and 5, strides 1 and 2; 3660
// forward and 2550 gradient times, 5 to 11 % rms on one chip), the wider tiles' raised by 5 %,
// for where they are chosen they are chosen for a low estimate; the choice loses 1 % against
// the best.
ConvTilePlan conv_tile_plan(const ConvTileArgs &g, bool dgrad, bool fused, size_t room) {
  static const ConvTileTimes kForward[] = {
      {64, 64, 0, 3, 3.854, 0.348, 0.245, 1.219, 1.743, 0.413, 1.579, 0.466},
      {64, 64, 2, 2, 0.944, 0.154, 0.489, 4.558, 1.887, 0.627, 0.226, 1.490},
      {64, 128, 1, 2, 4.688, 0.422, 0.354, 2.733, 0, 0.558, 0.568, 2.349},
      {128, 64, 1, 2, 4.363, 0.573, 0.396, 3.187, 0.070, 0.618, 0.762, 2.043},
      {128, 128, 1, 1, 5.704, 0.529, 0.771, 3.527, 0, 0.237, 0, 3.915}};
  static const ConvTileTimes kGradient[] = {
      {64, 64, 0, 3, 4.279, 0.381, 0.257, 0.901, 1.513, 0.529, 0, 0},
      {64, 64, 2, 2, 1.312, 0.568, 0.568, 4.618, 1.438, 0.745, 0, 0},
      {64, 128, 1, 2, 4.091, 0.540, 0.417, 2.946, 0.771, 0.648, 0, 0},
      {128, 64, 1, 2, 3.843, 0.619, 0.431, 2.948, 1.101, 0.608, 0, 0},
      {128, 128, 1, 2, 4.369, 0.880, 0.654, 3.878, 0, 0.613, 0, 0}};
  ConvTilePlan best;
  for (const ConvTileTimes &f : dgrad ? kGradient : kForward) {
    const TileLoad l(f, g);
    if (l.most >= (1ll << 23))
      continue;
    // (a split leaves the tiles' work as it is and adds to all else: nothing shorter comes
    // behind one whose work and rounds alone take longer than the best so far)
    const double load = (double)l.tiles / 256.0, teams = f.teams > 1 ? f.teams : 1;
    const double least = f.once + f.sum + l.longest * load * std::max(f.alone / f.occ, f.shared) / teams;
    const double each = f.round * load + f.part * (double)(l.tiles * f.bm * f.bn) * 4e-6;
    for (int split = 1; split <= 12; ++split) {
      if (split > 1 && (g.parts > 1 || l.longest / split < 2 || l.most * split > 1500 ||
                        (size_t)split * (size_t)(l.most * f.bm * f.bn) * sizeof(float) > room ||
                        least + split * each >= best.us))
        break;
      const double us = tile_us(f, l, g.parts == 1, split, fused);
      if (best.bm == 0 || us < best.us)
        best.bm = f.bm, best.bn = f.bn, best.teams = f.teams, best.splits = split, best.us = us;
    }
  }
  return best;
}

size_t conv_tile_scratch(const ConvTilePlan &p, const ConvTileArgs &g) {
  if (p.splits <= 1)
    return 0;
  const size_t tiles = (size_t)((g.part[0].M + p.bm - 1) / p.bm) * (size_t)((g.d.N + p.bn - 1) / p.bn);
  return (size_t)p.splits * tiles * (size_t)(p.bm * p.bn) * sizeof(float);
}

void conv_tile_lean(const fhip_epilogue &e, ConvTileArgs &g) {
  g.d.lean = fhip_epilogue_is_fast(e), g.d.lean_op = -1;
  for (int i = 0; i < g.d.epi.count; ++i) {
    const DevEpiOp &o = g.d.epi.op[i];
    if (o.kind == FHIP_OPERAND_TENSOR) {
      const bool typed = o.operand_dtype == FHIP_FLOAT || o.operand_dtype == FHIP_BFLOAT16 || o.operand_dtype == FHIP_HALF;
      if (o.stride[0] != 0 || o.stride[1] != 0 || !typed || g.d.lean_op >= 0)
        g.d.lean = 0;
      g.d.lean_op = i;
    }
  }
}

int conv_tile_launch(fhip_ctx *ctx, bool bf16, bool dgrad, const ConvTilePlan &p, ConvTileArgs &g, void *partial) {
  int64_t most = 0;
  const int taps = 64 / g.C;
  g.adv_c = 64 - taps * g.C, g.magic_c = conv_magic(g.C);
  for (int i = 0; i < g.parts; ++i) {
    ConvTilePart &q = g.part[i];
    most = q.M > most ? q.M : most;
    q.adv_r = taps / q.S, q.adv_s = taps - q.adv_r * q.S;
    q.magic_s = conv_magic(q.S);
    q.magic_p = conv_magic(q.P), q.magic_q = conv_magic(q.Q);
  }
  g.d.tiles_m = (int)((most + p.bm - 1) / p.bm);
  g.d.tiles_n = (g.d.N + p.bn - 1) / p.bn;
  g.d.splits = p.splits;
  g.d.partial = p.splits > 1 ? partial : nullptr;
  FHIP_REQUIRE(ctx, (int64_t)g.d.tiles_m * g.d.tiles_n < (1ll << 23), "conv: too many tiles");
  return bf16 ? conv_tile_launch_bf16(ctx, dgrad, p, g) : conv_tile_launch_f16(ctx, dgrad, p, g);
}

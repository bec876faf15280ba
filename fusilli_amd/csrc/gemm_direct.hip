// Host side of the direct matrix-product kernels (gemm_direct_kernel.h) and of the
// register-staged tiles (gemm_tile_kernel.h): which descriptors they take, tile, wavefronts
// and split of K, and the choice between them and the tiled GEMM.
#include "fast_paths.h"
#include "gemm_tile_kernel.h"

#include <cmath>

namespace {

// Products over a short K with many results are bound by their stores and by what a
// workgroup does once, and the general path's 64 x 64 f32 tiles (generic_ops.hip), one
// slice of 16 K at a time and whole rows stored, finish them sooner.  `p`: the plan for the
// direct kernel; `tiles`: 64 x 64 tiles of all batches.  Where the line lies was measured
// at 32 values of K, 17 shapes of 64 to 4096 tiles and 11 batched ones in all four
// orientations (3380 f32 products, 0.2 % of the better kernel's time left on average); it
// lies anew for every round of slices that a tile's wavefronts take, lower where K is whole
// slices, and for 16 bits (whose general path widens them) at 12 to 58.  us, f32 tiles /
// here: f32 1000 x 1000 K16 4.8 / 8.5, K88 8.7 / 9.0, K128 10.2 / 8.3; 2048 x 2048 K40 14.0
// / 18.6, K136 25.6 / 27.5, K160 27.5 / 24.4; both K-contiguous, 1600 x 1600 K128 20.7 /
// 15.8, K264 35.8 / 36.1; 200 batches of 64 x 64 K40 6.5 / 11.1; f16 2048 x 2048, neither,
// K24 13.2 / 20.7, K68 22.3 / 19.4; both, K16 10.8 / 14.0, K44 16.2 / 14.1.
bool short_k(const DirectPlan &p, const DirectArgs &g, int64_t M, int64_t N, int64_t K, int64_t batch) {
  if (p.kind != GK_F32 && p.kind != GK_BF16 && p.kind != GK_F16)
    return false; // (8-bit products have no such path)
  const int64_t tiles = (M + 63) / 64 * ((N + 63) / 64) * batch;
  if (p.mt == 1 || tiles < 64 || (tiles < 128 && K >= 128))
    return false;
  const bool whole = g.slices * 32 == K; // (f32: no slice is cut)
  // (smaller tiles that are no more than the rows or columns ask for)
  const bool halves = p.mt != 4 && 2 * (int64_t)g.tiles_m * g.tiles_n * batch > 3 * tiles;
  if (p.mt != 4 && p.b_kc) // (32 x 32 tiles keep up)
    return p.kind == GK_F32 && halves && tiles >= 110 && K < 17;
  const int rounds = (g.slices + p.waves - 1) / p.waves;
  if (p.kind == GK_F32) {
    if (tiles < 130)
      return !p.b_kc && K <= 40;
    if (p.mt != 4) { // (32 x 64)
      if (!halves)
        return K < (tiles <= 256 ? 20 : whole ? 65 : p.a_kc ? 113 : 60);
      if (tiles <= 256)
        return K < (p.a_kc && !whole ? 150 : 130);
      return K < (rounds == 1 ? 205 : 300);
    }
    if (whole)
      return K < (!p.b_kc ? (tiles > 256 && tiles <= 512 ? 97 : 65) : p.a_kc && tiles > 512 ? 65 : 33);
    if (rounds == 1)
      return K < (p.b_kc ? (tiles > 256 ? (p.a_kc ? 113 : 81) : p.a_kc ? 81 : 57)
                         : !p.a_kc ? 85 : tiles > 256 ? 113 : 89);
    return rounds == 2 && p.a_kc && K < (p.b_kc && tiles > 512 ? 153 : 145);
  }
  if (tiles < 130)
    return !p.a_kc && p.b_kc && K < 20;
  if (p.mt != 4)
    return p.a_kc && K < 40;
  if (p.a_kc)
    return K < (p.b_kc ? 34 : 24);
  return K < (tiles <= 256 ? (p.b_kc ? 20 : 12) : (p.b_kc ? 50 : 40) + (tiles >= 1024 ? 8 : 0));
}

bool direct_plan(const fhip_matmul_desc *d, DirectPlan *p, DirectArgs *g, int64_t *batch, double *us,
                 bool *too_short) {
  const int r = d->a.rank;
  if ((r != 2 && r != 3) || d->a.dtype != d->b.dtype)
    return false;
  switch (d->a.dtype) {
  case FHIP_BFLOAT16: p->kind = GK_BF16; break;
  case FHIP_HALF: p->kind = GK_F16; break;
  case FHIP_INT8: p->kind = GK_I8; break;
  case FHIP_FP8E4M3: p->kind = GK_FP8E4M3; break;
  case FHIP_FP8E5M2: p->kind = GK_FP8E5M2; break;
  case FHIP_FLOAT: p->kind = GK_F32; break;
  default: return false;
  }
  const int elem = fhip_dtype_size(d->a.dtype);
  auto f = [](int dt) { return dt == FHIP_FLOAT || dt == FHIP_BFLOAT16 || dt == FHIP_HALF; };
  if (p->kind == GK_I8
          ? d->c.dtype != FHIP_INT32 || d->out.dtype != FHIP_INT32 || d->epilogue.count != 0
          : !f(d->c.dtype) || !f(d->out.dtype))
    return false;
  const int64_t M = d->a.dim[r - 2], K = d->a.dim[r - 1], N = d->b.dim[r - 1];
  *batch = r == 3 ? d->c.dim[0] : 1;
  const int64_t a_sm = d->a.stride[r - 2], a_sk = d->a.stride[r - 1];
  const int64_t b_sk = d->b.stride[r - 2], b_sn = d->b.stride[r - 1];
  p->a_kc = a_sk == 1;
  p->b_kc = b_sk == 1;
  if ((!p->a_kc && a_sm != 1 && M != 1) || (!p->b_kc && b_sn != 1 && N != 1))
    return false;
  const int64_t a_ld = p->a_kc ? a_sm : a_sk, b_ld = p->b_kc ? b_sn : b_sk;
  // a 16-byte piece of K; 32-bit lane offsets over a tile's rows or a step's
  // K-rows (at most 128)
  if (K * elem < 16 || a_ld * elem >= (1 << 24) || b_ld * elem >= (1 << 24) || M >= (1ll << 31) ||
      N >= (1ll << 31) || K >= (1ll << 31) || *batch > 65535)
    return false;
  g->slices = (int)((K * elem + 127) / 128);
  // Tile, wavefronts and split of K: the shortest of an estimate in
  // microseconds.  A compute unit pulls some 50 KB of whole lines in one (half
  // of that in shorter runs), its matrix pipes do 256 (f32) to 8192 (8-bit)
  // operations a clock, and a split adds the second kernel and the partial
  // tiles' round trip.
  static const struct { int mt, nt_kc, nt, waves; } kShapes[] = {
      {1, 1, 4, 16}, {1, 2, 4, 8}, {2, 2, 4, 8}, {4, 4, 4, 4}};
  const double ops = p->kind == GK_F32 ? 5.6e5 : elem == 2 ? 4e6 : 8e6; // per us and compute unit
  double best = 0;
  for (const auto &c : kShapes) {
    const int mt = c.mt, nt = p->b_kc ? c.nt_kc : c.nt;
    // (a run of the interleaved rows lies inside the operand)
    if ((!p->b_kc && N < nt) || (!p->a_kc && M < mt) || (!p->b_kc && c.nt_kc == 2 && mt == 1))
      continue;
    const int most = p->b_kc || mt > 1 ? c.waves : 8;
    const int64_t tm = (M + 16 * mt - 1) / (16 * mt), tn = (N + 16 * nt - 1) / (16 * nt);
    const int64_t wgs = tm * tn * *batch;
    if (tm * tn >= (1ll << 31))
      continue;
    // (one thread for every four results, 64 x 64 tiles: sixteen)
    int waves = g->slices, least = mt * nt == 16 ? 4 : mt * nt;
    waves = waves > least ? waves : least;
    waves = waves < 1 ? 1 : waves < most ? waves : most;
    const double pull_a = 16.0 * mt * K * elem / (p->a_kc || mt * elem >= 8 ? 5e4 : 2.5e4);
    const double pull_b = 16.0 * nt * K * elem / (p->b_kc || nt * elem >= 8 ? 5e4 : 2.5e4);
    const double work = 512.0 * mt * nt * (double)K;
    for (int split = 1; split <= 32; split *= 2) {
      if (split > 1 && (g->slices < 2 * split * waves || wgs * split > 512))
        break;
      // (workgroups that share a compute unit: whole rounds matter below two)
      const double share = (double)(wgs * split) / 256.0;
      const double rounds = share <= 1.0 ? 1.0 : fmax(share, mt == 4 ? 1.5 : 1.2);
      const double us = 2.0 + rounds * fmax(pull_a + pull_b, work / ops) / split +
                        (split > 1 ? 3.0 + 2.0 * split * wgs * mt * nt * 1024.0 / 4e6 : 0.0);
      if (best == 0 || us < best) {
        best = us;
        p->mt = mt, p->nt = nt, p->waves = waves, g->splits = split;
        g->tiles_m = (int)tm, g->tiles_n = (int)tn;
      }
    }
  }
  if (best == 0)
    return false;
  *us = best;
  // (16-bit operands into f32: the f32 tiles would be further from the exact sums, f16 K24
  // 1.3 units of 2^-24 against 0.7)
  const bool f32_of_16 = p->kind != GK_F32 && d->c.dtype == FHIP_FLOAT && d->out.dtype == FHIP_FLOAT;
  *too_short = !f32_of_16 && short_k(*p, *g, M, N, K, *batch);
  if (*too_short)
    return false;
  g->M = (int)M, g->N = (int)N, g->K = (int)K;
  g->a_ldb = a_ld * elem, g->b_ldb = b_ld * elem;
  if (r == 3) {
    g->a_batch = d->a.dim[0] == 1 ? 0 : d->a.stride[0];
    g->b_batch = d->b.dim[0] == 1 ? 0 : d->b.stride[0];
    g->o_batch = d->out.dim[0] == 1 ? 0 : d->out.stride[0];
  }
  g->o_sm = d->out.stride[r - 2];
  g->o_sn = d->out.stride[r - 1];
  g->c_dt = d->c.dtype;
  g->o_dt = d->out.dtype;
  p->ok = true;
  return true;
}

// What the planners' estimates leave out, fitted to 400 random products (16 and 8 bits, M from
// 1 to 4096) that all three families ran: us = once + scale * estimate, more where operands'
// rows start off 16 bytes, lie along M or N, or the chain ends in GELU.  With them the family
// chosen is 1.5 % slower than the best one on average; over 400 others 12 % faster than the tiled
// GEMM where its contract held and the direct kernels elsewhere, up to 4 times.
struct ProductTimes {
  struct Line {
    double once, scale, gelu_once, loose, rows;
  };
  int loose, rows; // operands whose rows start off 16 bytes / lie along M or N
  bool gelu, wide; // 64 x 64 tiles
  bool few, byte;  // 16 rows; 8-bit operands
  ProductTimes(const DirectPlan &p, const DirectArgs &g, const fhip_matmul_desc *d, int elem, const void *a,
               const void *b)
      : loose(((g.a_ldb | (int64_t)(uintptr_t)a) % 16 != 0) + ((g.b_ldb | (int64_t)(uintptr_t)b) % 16 != 0)),
        rows(!p.a_kc + !p.b_kc), gelu(fhip_epilogue_is_transcendental(d->epilogue)), wide(p.mt == 4),
        few(p.mt == 1), byte(elem == 1) {}
  double of(const Line &l, double us) const {
    return us > 0 ? l.once + us * (l.scale + l.loose * loose + l.rows * rows) + (gelu ? l.gelu_once : 0.0) : 0.0;
  }
  double direct(double us, const DirectArgs &g, int64_t batch) const {
    static const Line k16[2] = {{2.55, 0.75, 1.12, 0.09, 0.11}, {2.29, 0.89, 1.37, 0.19, 0.11}};
    static const Line k8[2] = {{2.50, 0.61, 0.54, 0, -0.10}, {1.97, 0.99, 0.47, 0, -0.16}};
    if (!wide)
      return of((byte ? k8 : k16)[few ? 0 : 1], us);
    // 64 x 64 tiles (229 of them): a wavefront's slices at a pace, alone or with another
    // workgroup, as for the tiles below
    const double load = (double)((int64_t)g.tiles_m * g.tiles_n * batch * g.splits) / 256.0;
    const int run = (g.slices + 4 * g.splits - 1) / (4 * g.splits);
    const double alone = byte ? 0.87 : 1.27, shared = byte ? 2.03 : 2.19;
    const double pace = (load <= 1.0 ? alone : shared * (load <= 2.0 ? 1.0 : 0.25 * load + 0.5 * ceil(0.5 * load))) *
                        (byte ? 1.0 + 0.70 * rows : 1.0 + 0.12 * loose + 0.06 * rows);
    return (byte ? 4.55 : 2.94) + run * pace +
           fmax(1.0, load) * (byte ? 1.5 + 1.3 * gelu : 2.4 + 1.5 * gelu) +
           (g.splits > 1 ? 0.3 + (byte ? 0.67 : 0.85) * g.splits * (double)g.tiles_m * g.tiles_n * batch * 4096 * 4e-6
                         : 0.0);
  }
  double tile(double us) const {
    static const Line k16 = {-0.39, 1.01, 0.34, 0.07, 0.06}, k8 = {-0.91, 1.11, 0.98, 0, 0.06};
    return of(byte ? k8 : k16, us);
  }
};

// The shortest estimate of the LDS-tiled kernels (gemm_tile_kernel.h) for the product that `p`
// and `g` describe; us, 0: none applies.  A workgroup's time is its slices at a pace (alone on
// its compute unit, or two to one: they share its LDS) plus what it does once; with a split,
// the parts' round trip and the second kernel.  Fitted to 453 + 624 times (16 and 8 bits) of
// random products of 17 to 4096 rows, 256 to 8192 columns and K, in all orientations, on one
// chip, 10 to 13 % rms; the choice between these tiles loses 2 % against the best of them.
double tile_plan(const DirectPlan &dp, const DirectArgs &g, int elem, bool gelu, int64_t batch, DirectPlan *p, int *tiles_m,
                 int *tiles_n, int *splits) {
  struct Fit {
    int mt, nt, waves;
    double once, alone, shared, round, sum, part, gelu;
  };
  static const Fit k16[] = {{4, 4, 4, 4.33, 0.253, 0.483, 1.75, 1.77, 0.34, 0.81},
                             {4, 4, 8, 2.06, 0.444, 1.155, 3.42, 2.36, 0.40, 0.95},
                             {4, 8, 4, 5.54, 0.412, 0.700, 2.50, 0.00, 0.44, 1.65},
                             {8, 4, 4, 5.49, 0.402, 0.702, 2.53, 0.57, 0.41, 0.97},
                             {8, 8, 4, 3.69, 0.662, 1.080, 5.12, 0.00, 0.39, 1.78}};
  static const Fit k8[] = {{4, 4, 4, 3.76, 0.188, 0.497, 1.35, 1.90, 0.45, 1.00},
                             {4, 4, 8, 2.84, 0.334, 1.354, 2.05, 2.16, 0.55, 1.00},
                             {4, 8, 4, 4.24, 0.303, 0.680, 2.39, 0.97, 0.57, 1.00},
                             {8, 4, 4, 3.61, 0.297, 0.681, 2.45, 1.66, 0.48, 1.00},
                             {8, 8, 4, 2.11, 0.470, 1.002, 5.22, 0.81, 0.52, 1.00}};
  const int pe = 16 / elem;
  if ((!dp.a_kc && g.M < pe) || (!dp.b_kc && g.N < pe)) // (whole chunks of the other operand)
    return 0;
  double best = 0;
  for (const Fit &f : elem == 2 ? k16 : k8) {
    const int bm = 16 * f.mt, bn = 16 * f.nt;
    const int64_t tm = (g.M + bm - 1) / bm, tn = (g.N + bn - 1) / bn;
    if (tm * tn >= (1ll << 31))
      continue;
    for (int split = 1; split <= 16; ++split) {
      const int run = (g.slices + split - 1) / split;
      if (split > 1 && (run < 3 || tm * tn * batch * split > 2048))
        break;
      const double load = (double)(tm * tn * batch * split) / 256.0;
      const double pace = load <= 1.0 ? f.alone
                                      : f.shared * (load <= 2.0 ? 1.0 : 0.25 * load + 0.5 * ceil(0.5 * load));
      const int teams = f.waves / 4;
      double us = f.once + (double)((run + teams - 1) / teams) * pace + fmax(1.0, load) * (f.round + (gelu ? f.gelu : 0.0));
      if (split > 1)
        us += f.sum + f.part * split * (double)(tm * tn * batch * bm * bn) * 4e-6;
      if (best == 0 || us < best) {
        best = us;
        *p = dp;
        p->tile = true, p->mt = f.mt, p->nt = f.nt, p->waves = f.waves;
        *tiles_m = (int)tm, *tiles_n = (int)tn, *splits = split;
      }
    }
  }
  return best;
}

} // namespace

int fhip_direct_matmul(fhip_ctx *ctx, const fhip_matmul_desc *d, const void *a, const void *b,
                       const DevEpilogue &epi, void *out, double other_us, bool whole, bool *handled,
                       bool *short_k) {
  *handled = *short_k = false;
  DirectPlan p;
  DirectArgs g{};
  int64_t batch = 1;
  double us = 0;
  if (!direct_plan(d, &p, &g, &batch, &us, short_k))
    return 0;
  // operands at their own alignment
  const uintptr_t am = fhip_dtype_size(d->a.dtype) - 1;
  if ((((uintptr_t)a | (uintptr_t)b) & am) != 0)
    return 0;
  g.a = (const char *)a;
  g.b = (const char *)b;
  g.out = (char *)out;
  g.epi = epi;
  g.epi.rank = 3;
  const int r = d->a.rank;
  for (int i = 0; i < epi.count; ++i) {
    const DevEpiOp &s = epi.op[i];
    DevEpiOp &o = g.epi.op[i];
    o.stride[0] = r == 3 ? s.stride[0] : 0;
    o.stride[1] = s.stride[r - 2];
    o.stride[2] = s.stride[r - 1];
  }
  g.lean = fhip_epilogue_is_fast(d->epilogue), g.lean_op = -1;
  for (int i = 0; i < epi.count; ++i) {
    const DevEpiOp &o = g.epi.op[i];
    if (o.kind == FHIP_OPERAND_TENSOR) {
      const bool typed = o.operand_dtype == FHIP_FLOAT || o.operand_dtype == FHIP_BFLOAT16 || o.operand_dtype == FHIP_HALF;
      if (o.stride[0] != 0 || o.stride[1] != 0 || !typed || g.lean_op >= 0)
        g.lean = 0;
      g.lean_op = i;
    }
  }
  // f32 results of 16-bit or fp8 operands keep the kernel they had: the length of the chains
  // that the sums are taken in shows there.
  const bool f32_out = p.kind != GK_I8 && d->c.dtype == FHIP_FLOAT && d->out.dtype == FHIP_FLOAT;
  // Split products over a long K stay on the tiled GEMM, and so do those over one whole slice (bf16
  // 5696 x 5184 x 64 in four batches 59 us, here 416; 1536 x 448 x 64 5.7 / 9.5); those over less
  // than a slice stay here.
  if (whole && (f32_out || g.slices >= 128 || g.slices == 1))
    return 0;
  if (p.kind != GK_F32 && !f32_out && g.slices > 1) {
    DirectPlan t;
    int tm = 0, tn = 0, splits = 1;
    const int elem = fhip_dtype_size(d->a.dtype);
    const ProductTimes times(p, g, d, elem, a, b);
    // the kernel that took the product before there were tiles of every size, or the tiled
    // GEMM where K fills no slice; the tiles where they clearly outrun it
    const double direct_us = times.direct(us, g, batch);
    const bool other = other_us > 0 && (whole || other_us * 1.08 < direct_us);
    const double known_us = other ? other_us : direct_us;
    // (tiles that are at least half full; none takes less than 6 us)
    const bool fills = g.M > 32 && g.N > 32 && (int64_t)g.M * g.N >= 2048 && known_us > 6.0;
    const double tile_us =
        fills ? times.tile(tile_plan(p, g, elem, times.gelu, batch, &t, &tm, &tn, &splits)) : 0;
    if (tile_us > 0 && tile_us * (other ? 1.08 : 1.04) < known_us)
      p = t, g.tiles_m = tm, g.tiles_n = tn, g.splits = splits;
    else if (other)
      return 0;
  }
  *handled = true;
  if (g.splits > 1) {
    const size_t bytes = (size_t)g.splits * (size_t)batch * g.tiles_m * g.tiles_n * (p.mt * p.nt * 1024);
    if (!fhip_ctx_scratch_ready(ctx, bytes))
      g.splits = 1;
    else if (fhip_ctx_scratch(ctx, bytes, &g.partial) != 0)
      return 1;
  }
  if (p.tile) {
    static const char *const kKindName[] = {"bf16", "f16", "i8", "fp8e4m3", "fp8e5m2"};
    fhip_note_kernel(ctx, "gemm_mfma %s %dx%d waves=%d split=%d", kKindName[p.kind], 16 * p.mt, 16 * p.nt, p.waves, g.splits);
    switch (p.kind) {
    case GK_BF16: return tile_launch_bf16(ctx, p, g, batch);
    case GK_F16: return tile_launch_f16(ctx, p, g, batch);
    case GK_I8: return tile_launch_i8(ctx, p, g, batch);
    case GK_FP8E4M3: return tile_launch_fp8e4m3(ctx, p, g, batch);
    default: return tile_launch_fp8e5m2(ctx, p, g, batch);
    }
  }
  fhip_note_kernel(ctx, "gemm_direct %dx%d waves=%d split=%d", 16 * p.mt, 16 * p.nt, p.waves, g.splits);
  switch (p.kind) {
  case GK_BF16: return direct_launch_bf16(ctx, p, g, batch);
  case GK_F16: return direct_launch_f16(ctx, p, g, batch);
  case GK_I8: return direct_launch_i8(ctx, p, g, batch);
  case GK_FP8E4M3: return direct_launch_fp8e4m3(ctx, p, g, batch);
  case GK_FP8E5M2: return direct_launch_fp8e5m2(ctx, p, g, batch);
  default: return direct_launch_f32(ctx, p, g, batch);
  }
}

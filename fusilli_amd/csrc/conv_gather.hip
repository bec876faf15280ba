// Forward convolution of channels-last 16-bit tensors whose channel count is no multiple
// of a 128-byte slice (one group, C a multiple of 8), and of those whose output channels
// fill the other kernels' tiles badly.
//
//   OUT[m, n] = epilogue(sum over j = (r, s, c) of X[pixel of m shifted by (r, s), c] * W[n, j])
//
// Bound by LDS reads and MFMA about alike (two 16-byte reads of 64 lanes
// per 32 x 32 x 16 MFMA).  The reduction runs over the filter
// row as it lies, 64 values a step: a 16-byte run of X lies inside one tap, so a lane
// keeps its own tap and channel and fetches each of its pixels with one range-checked
// load (zeros outside the image); a filter row's end is not padded.  The MFMA GEMM
// gather needs whole 128-byte slices of a tap, hence copies of X and W with padded
// channels before it, and multiplies the padding.
// Stages of 64 values sit in LDS twice; loads run two steps ahead in registers.  The
// result goes through LDS so that a lane finishes and stores 8 channels of a pixel.
//
// N16 48 -> 48, 48 x 32, 3 x 3, f16: copy + product 16.9 us -> 9.  Long reductions and few
// tiles: conv_tile_kernel.h.
// (128 x 128, 256 x 64, 128 x 64 and 128 x 32 tiles of the same kernel are slower.)
//
// Reference semantics: aten.convolution (reference support/asm_emitter.h:690-701).
#include "conv_gather.h"

#include <type_traits>

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kCgThreads = 256;
constexpr int kCgRow = 128; // bytes of a stage row: 64 values
constexpr int kCgNone = -(1 << 20); // row of a pixel that does not exist

template <bool BF16>
__device__ __forceinline__ f32x16 cg_mfma(const u32x4 &a, const u32x4 &b, const f32x16 &c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t cg_rsrc(const char *base, uint32_t bytes) {
  const uint64_t b = (uint64_t)base;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
  return __builtin_amdgcn_make_buffer_rsrc((void *)(((uint64_t)hi << 32) | lo), 0,
                                           (int)__builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

// Byte of 16-byte run `chunk` of a stage row: the runs of a row are permuted by its
// number, so that 16 rows' reads of one run meet all banks once.
__device__ __forceinline__ int cg_place(int row, int chunk) {
  return row * kCgRow + ((chunk ^ ((row >> 1) & 7)) << 4);
}

// WM x WN wavefronts of MT x NT tiles of 32 pixels x 32 channels.
template <bool BF16>
__global__ __launch_bounds__(kCgThreads) __attribute__((amdgpu_waves_per_eu(2, 4))) void
conv_gather_kernel(ConvGatherArgs g) {
  constexpr int WM = 2, WN = 2, MT = 1, NT = 1;
  constexpr int TM = 32 * MT * WM, TN = 32 * NT * WN;
  static_assert(TM == kConvGatherTile && TN == kConvGatherTile, "the launch counts these tiles");
  constexpr int NA = TM / 32, NB = TN / 32; // loads per thread and step
  constexpr int kStage = (TM + TN) * kCgRow;
  constexpr int kPitch = NT * 32 + 4; // floats of a result row in LDS
  constexpr int kLds = 2 * kStage > 4 * 32 * kPitch * 4 ? 2 * kStage : 4 * 32 * kPitch * 4;
  __shared__ __attribute__((aligned(16))) char smem[kLds];
  const int tid = threadIdx.x, l = tid & 63, wave = tid >> 6;
  // (workgroups go to the eight L2 slices in turn: each slice gets a run of neighbouring
  // tiles, which read the same pixels)
  uint32_t id = blockIdx.x;
  {
    const uint32_t per = gridDim.x / 8, rest = gridDim.x % 8, slice = id % 8;
    id = slice * per + (slice < rest ? slice : rest) + id / 8;
  }
  const int64_t m0 = (int64_t)(id / (uint32_t)g.tiles_n) * TM;
  const int n0 = (int)(id % (uint32_t)g.tiles_n) * TN;
  // ---- what this thread brings in: 16-byte run tid % 8 of rows tid / 8 + 32 i
  const int chunk = tid & 7, row0 = tid >> 3;
  int at[NA], h0[NA], w0[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int64_t m = m0 + row0 + 32 * i;
    const uint32_t e = m < g.M ? (uint32_t)m : 0u;
    const uint32_t t = e / (uint32_t)g.Q, q = e - t * (uint32_t)g.Q;
    const uint32_t n = t / (uint32_t)g.P, p = t - n * (uint32_t)g.P;
    const int h = (int)p * g.str_h - g.pad_h;
    w0[i] = (int)q * g.str_w - g.pad_w;
    at[i] = (int)((n * (uint32_t)g.H + (uint32_t)h) * (uint32_t)g.W + (uint32_t)w0[i]) * g.C * 2;
    h0[i] = m < g.M ? h : kCgNone;
  }
  const int first = blockIdx.y * g.steps;
  const int total = (g.J + 63) / 64;
  const int last = first + g.steps < total ? first + g.steps : total;
  int j = first * 64 + chunk * 8; // first value of the run, its tap and channel
  int r, s, c;
  {
    const int tap = j / g.C;
    c = j - tap * g.C;
    r = tap / g.S, s = tap - r * g.S;
  }
  const __amdgpu_buffer_rsrc_t rx = cg_rsrc(g.x, g.x_bytes);
  const int rows_n = g.N - n0 < TN ? g.N - n0 : TN;
  const __amdgpu_buffer_rsrc_t rw =
      cg_rsrc(g.w + (int64_t)n0 * g.J * 2, (uint32_t)rows_n * (uint32_t)g.J * 2u);
  u32x4 va[2][NA], vb[2][NB];
  auto fetch = [&](auto set, int t) {
    constexpr int B = decltype(set)::value;
    if (t >= last)
      return;
    const bool in_row = j < g.J;
    const int dh = r * g.dil_h, dw = s * g.dil_w;
    const int tap = ((dh * g.W + dw) * g.C + c) * 2;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const bool in = in_row && (unsigned)(h0[i] + dh) < (unsigned)g.H &&
                      (unsigned)(w0[i] + dw) < (unsigned)g.W;
      va[B][i] = __builtin_amdgcn_raw_buffer_load_b128(rx, in ? at[i] + tap : (int)0x80000000, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) // (rows past N: out of range)
      vb[B][i] = __builtin_amdgcn_raw_buffer_load_b128(
          rw, in_row ? ((row0 + 32 * i) * g.J + j) * 2 : (int)0x80000000, 0, 0);
    j += 64, c += 64;
    while (c >= g.C) {
      c -= g.C;
      if (++s == g.S)
        s = 0, ++r;
    }
  };
  f32x16 acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        acc[a][b][i] = 0.f;
  const int wm = wave / WN, wn = wave % WN;
  auto step = [&](auto set, int t) {
    constexpr int B = decltype(set)::value;
    char *to = smem + B * kStage;
#pragma unroll
    for (int i = 0; i < NA; ++i)
      *(u32x4 *)(to + cg_place(row0 + 32 * i, chunk)) = va[B][i];
#pragma unroll
    for (int i = 0; i < NB; ++i)
      *(u32x4 *)(to + cg_place(TM + row0 + 32 * i, chunk)) = vb[B][i];
    fetch(set, t + 2);
    // (one barrier per step: a stage is written again two steps later, behind the
    // barrier that its readers reach after reading)
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      // lane l: row l % 32, values 8 (l / 32) .. + 7 of the 16
      u32x4 fa[MT], fb[NT];
#pragma unroll
      for (int a = 0; a < MT; ++a)
        fa[a] = *(const u32x4 *)(to + cg_place((wm * MT + a) * 32 + (l & 31), ks * 2 + (l >> 5)));
#pragma unroll
      for (int b = 0; b < NT; ++b)
        fb[b] = *(const u32x4 *)(to + cg_place(TM + (wn * NT + b) * 32 + (l & 31), ks * 2 + (l >> 5)));
#pragma unroll
      for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NT; ++b)
          acc[a][b] = cg_mfma<BF16>(fa[a], fb[b], acc[a][b]);
    }
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  fetch(S0{}, first);
  fetch(S1{}, first + 1);
  for (int t = first; t < last; t += 2) {
    step(S0{}, t);
    if (t + 1 < last)
      step(S1{}, t + 1);
  }
  // ---- results: value i of a lane is pixel 8 (i / 4) + 4 (l / 32) + i % 4 of the tile,
  // channel l % 32; a wavefront's own LDS turns them into runs of 8 channels
  __syncthreads();
  float *mine = (float *)smem + wave * 32 * kPitch;
#pragma unroll
  for (int a = 0; a < MT; ++a) {
#pragma unroll
    for (int b = 0; b < NT; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        mine[(8 * (i >> 2) + 4 * (l >> 5) + (i & 3)) * kPitch + b * 32 + (l & 31)] = acc[a][b][i];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma clang loop unroll(disable)
    for (int e = l; e < 32 * NT * 4; e += 64) {
      const int row = e / (NT * 4), col = e % (NT * 4) * 8;
      const int64_t m = m0 + (wm * MT + a) * 32 + row;
      const int n = n0 + wn * NT * 32 + col;
      if (m >= g.M || n >= g.N)
        continue;
      const f32x4 lo = *(const f32x4 *)(mine + row * kPitch + col);
      const f32x4 hi = *(const f32x4 *)(mine + row * kPitch + col + 4);
      float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      const int live = g.N - n < 8 ? g.N - n : 8;
      if (g.part) { // (N is a multiple of 4)
        float *to = g.part + ((int64_t)blockIdx.y * g.M + m) * g.N + n;
        *(f32x4 *)to = lo;
        if (live == 8)
          *(f32x4 *)(to + 4) = hi;
        continue;
      }
      fhip_round_fast_vec<8>(g.y_dt, v);
      if (g.epi.count > 0) {
        int64_t coord[FHIP_MAX_RANK] = {};
        coord[1] = m;
        int64_t cols[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
          cols[i] = n + (i < live ? i : 0);
        fhip_apply_epilogue_many<float, 8>(g.epi, v, coord, 2, cols);
      }
      const int64_t o = m * g.N + n;
      if (live == 8 && g.o_dt != FHIP_FLOAT) {
        typedef uint32_t loose __attribute__((ext_vector_type(4), aligned(2)));
        u32x4 t;
        if (g.o_dt == FHIP_BFLOAT16) {
          bf16x8 h;
#pragma unroll
          for (int i = 0; i < 8; ++i)
            h[i] = (__bf16)v[i];
          t = __builtin_bit_cast(u32x4, h);
        } else {
          f16x8 h;
#pragma unroll
          for (int i = 0; i < 8; ++i)
            h[i] = (_Float16)v[i];
          t = __builtin_bit_cast(u32x4, h);
        }
        *(loose *)((uint16_t *)g.out + o) = t;
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (i < live)
            fhip_store<float>(g.out, g.o_dt, o + i, v[i]);
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

} // namespace

ConvGatherPlan conv_gather_plan(int64_t M, int64_t N, int64_t J, bool may_split) {
  // 64 x 64 tiles, of which four workgroups share a compute unit and cover each other's
  // loads: the step's latency, not its product, is what larger tiles wait for (training
  // steps, 64 x 64 against 128 x 128, us: N16 48 -> 48, 48 x 32 49.3 / 58.1; N16 80 -> 40,
  // 56 x 56 65.9 / 80.0; N40 240 -> 240, 10 x 10 76.4 / 83.0; N32 112 -> 384, 26 x 26
  // 145.4 / 146.8).
  const int64_t steps = (J + 63) / 64;
  const int tile = kConvGatherTile;
  ConvGatherPlan best{1};
  // Few tiles: the reduction is cut where the shorter chain of steps (about 0.6 us each)
  // outweighs the parts' stores and the kernel that adds them.
  const double tiles = (double)((M + tile - 1) / tile) * (double)((N + tile - 1) / tile);
  double least = 0;
  for (int parts = 1; parts <= (may_split ? 8 : 1) && (parts == 1 || steps / parts >= 4); ++parts) {
    const double rounds = tiles * parts / 512.0;
    double us = (rounds > 1.0 ? rounds : 1.0) * 0.6 * (double)((steps + parts - 1) / parts);
    if (parts > 1)
      us += 4.0 + 2.0 * parts * (double)M * (double)N * 4.0 / 5.0e6;
    if (parts == 1 || us < least)
      least = us, best.parts = parts;
  }
  return best;
}

int conv_gather_launch(fhip_ctx *ctx, bool bf16, const ConvGatherPlan &p, ConvGatherArgs &a) {
  a.tiles_n = (a.N + kConvGatherTile - 1) / kConvGatherTile;
  const int steps = (a.J + 63) / 64;
  a.steps = (steps + p.parts - 1) / p.parts;
  const int64_t blocks = (a.M + kConvGatherTile - 1) / kConvGatherTile * a.tiles_n;
  FHIP_REQUIRE(ctx, blocks < (1ll << 23), "conv: too many tiles");
  const dim3 grid((unsigned)blocks, (unsigned)p.parts);
  auto go = [&](auto bf) {
    constexpr bool B = decltype(bf)::value;
    hipLaunchKernelGGL(conv_gather_kernel<B>, grid, dim3(kCgThreads), 0, ctx->stream, a);
  };
  if (bf16)
    go(std::true_type{});
  else
    go(std::false_type{});
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  return 0;
}

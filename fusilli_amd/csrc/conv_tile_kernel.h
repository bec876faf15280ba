// Convolutions and their data gradients on the register-staged tiles of gemm_tile_kernel.h.
//
//   forward   OUT[m, n] = epilogue(sum over j = (r, s, c) of X[pixel of m shifted by (r, s), c] W[n, j])
//   gradient  DX[m, c] = sum over j = (r, s, k) of DY[pixel of m shifted by (r, s), k] W[k, r, s, c]
//
// The reduction runs over the taps and channels as they lie, 64 values a slice: a 16-byte run
// lies inside one tap (channels are a multiple of 8), so a lane keeps its own tap and channel
// and steps them without a branch, and one range-checked load per run fetches zeros outside the
// image and behind the last tap.  The gradient reads the filter in place, channels along the
// tile's columns (transposing LDS reads): no mirrored copy.
//
// Strides above one: the rows (and columns) of DX that leave one remainder share their taps,
// so a gradient is stride_h * stride_w convolutions of DY at unit stride, each with its share of
// the filter, longest reduction first in one launch.  (Spread over a zero grid, DY took
// stride^2 times the products and two more launches.)
//
// Bound as gemm_tile_kernel.h is, by LDS and the latency of few tiles; the runs' addresses are
// 14 vector instructions a slice and operand.  us, before -> now: gradients N32 288 -> 176, 38 x 38,
// 5 x 5 at stride 2 264 -> 85 (350 TFLOP/s of the products it cannot do without), N35 64 -> 320,
// 21 x 21, 3 x 3 at stride 2 35 -> 14, N20 64 -> 384, 11 x 11, 5 x 5 70 -> 18; forward N31 192 ->
// 192, 11 x 11, 5 x 5 36 -> 24.5, N9 128 -> 128, 12 x 12, 5 x 5 23.4 -> 11.9; 600 random layers:
// gradients 0.75 of their time, forward 0.92.
#ifndef FUSILLI_AMD_CSRC_CONV_TILE_KERNEL_H
#define FUSILLI_AMD_CSRC_CONV_TILE_KERNEL_H

#include "conv_tile.h"
#include "gemm_tile_kernel.h"

__device__ __forceinline__ __amdgpu_buffer_rsrc_t conv_tile_rsrc(const char *base, uint32_t bytes) {
  const uint64_t b = (uint64_t)base;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
  return __builtin_amdgcn_make_buffer_rsrc((void *)(((uint64_t)hi << 32) | lo), 0,
                                           (int)__builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

constexpr int kConvTileNone = (int)0x80000000; // an offset behind every buffer

// Output pixel m of a part: image, row and column.
__device__ __forceinline__ void conv_tile_pixel(const ConvTilePart &p, int m, int &n, int &i, int &j) {
  const int t = conv_div(m, p.Q, p.magic_q);
  j = m - t * p.Q;
  n = conv_div(t, p.P, p.magic_p);
  i = t - n * p.P;
}

// Pixels of the tile: rows of the gathered operand.
template <int KIND, int ROWS, int T, int STEPS>
struct ConvPixels : TileOperand<KIND, true, ROWS, T, STEPS> {
  using Base = TileOperand<KIND, true, ROWS, T, STEPS>;
  using Raw = typename Base::Raw;
  static constexpr int LOADS = Base::LOADS;
  __amdgpu_buffer_rsrc_t x;
  int at[LOADS], h0[LOADS], w0[LOADS]; // under the first tap
  int j, c, s, dh, dw, off;            // this lane's run of the next slice, its tap's place
  int J, C, S, H, W;
  int adv_c, adv_s, adv_h, adv_w, adv_off; // to the next slice, ...
  int wrap_w, wrap_off, row_h, row_w, row_off; // ... past a tap, past a row of taps

  template <class Args>
  __device__ __forceinline__ void setup(const Args &g, const ConvTilePart &p, int m0, int t, int tile0, int step0,
                                        uint32_t lds, int first) {
    this->ragged = false, this->cut = 0, this->k0 = 0;
    this->place(t, tile0, step0, lds);
    J = p.J, C = g.C, S = p.S, H = g.H, W = g.W;
    x = conv_tile_rsrc(g.d.a, g.x_bytes);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int m = m0 + t / 8 + i * Base::STEP;
      int n, y, z;
      conv_tile_pixel(p, m < p.M ? m : 0, n, y, z);
      const int h = y * g.str_h + p.off_h;
      w0[i] = z * g.str_w + p.off_w;
      at[i] = (int)((((uint32_t)n * (uint32_t)H + (uint32_t)h) * (uint32_t)W + (uint32_t)w0[i]) * (uint32_t)C * 2u);
      h0[i] = m < p.M ? h : -(1 << 20);
    }
    j = first * 64 + t % 8 * 8;
    const int tap = conv_div(j, C, g.magic_c), r = conv_div(tap, S, p.magic_s);
    c = j - tap * C, s = tap - r * S;
    dh = r * g.dil_h, dw = s * g.dil_w;
    off = ((dh * W + dw) * C + c) * 2;
    adv_c = g.adv_c, adv_s = p.adv_s;
    adv_h = p.adv_r * g.dil_h, adv_w = adv_s * g.dil_w;
    adv_off = ((adv_h * W + adv_w) * C + adv_c) * 2;
    wrap_w = g.dil_w, wrap_off = (g.dil_w - 1) * C * 2;
    row_h = g.dil_h, row_w = S * g.dil_w, row_off = (g.dil_h * W - S * g.dil_w) * C * 2;
  }

  template <bool TAIL> __device__ __forceinline__ void fetch(int, int, Raw &raw) {
    const bool in_row = j < J;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const bool in = in_row && (unsigned)(h0[i] + dh) < (unsigned)H && (unsigned)(w0[i] + dw) < (unsigned)W;
      raw.v[i] = __builtin_amdgcn_raw_buffer_load_b128(x, in ? at[i] + off : kConvTileNone, 0, 0);
    }
    j += 64, c += adv_c, s += adv_s, dh += adv_h, dw += adv_w, off += adv_off;
    const bool tap = c >= C;
    c -= tap ? C : 0, s += tap ? 1 : 0, dw += tap ? wrap_w : 0, off += tap ? wrap_off : 0;
    const bool row = s >= S;
    s -= row ? S : 0, dh += row ? row_h : 0, dw -= row ? row_w : 0, off += row ? row_off : 0;
  }
};

// Filter rows of the forward convolution: J values as they lie.
template <int KIND, int ROWS, int T, int STEPS>
struct ConvFilterRows : TileOperand<KIND, true, ROWS, T, STEPS> {
  using Base = TileOperand<KIND, true, ROWS, T, STEPS>;
  using Raw = typename Base::Raw;
  static constexpr int LOADS = Base::LOADS;
  __amdgpu_buffer_rsrc_t w;
  int at[LOADS], j, J;

  template <class Args>
  __device__ __forceinline__ void setup(const Args &g, const ConvTilePart &p, int n0, int t, int tile0, int step0,
                                        uint32_t lds, int first) {
    this->ragged = false, this->cut = 0, this->k0 = 0;
    this->place(t, tile0, step0, lds);
    J = p.J;
    const int rows = g.d.N - n0 < ROWS ? g.d.N - n0 : ROWS;
    w = conv_tile_rsrc(g.d.b + (int64_t)n0 * J * 2, (uint32_t)rows * (uint32_t)J * 2u);
    j = first * 64 + t % 8 * 8;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) // (rows behind N lie behind the buffer)
      at[i] = ((t / 8 + i * Base::STEP) * J + j) * 2;
  }

  template <bool TAIL> __device__ __forceinline__ void fetch(int, int, Raw &raw) {
    const bool in = j < J;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      raw.v[i] = __builtin_amdgcn_raw_buffer_load_b128(w, in ? at[i] : kConvTileNone, 0, 0);
      at[i] += 128;
    }
    j += 64;
  }
};

// The filter under the data gradient: value (tap, k) of the reduction is a run of channels.
template <int KIND, int ROWS, int T, int STEPS>
struct ConvFilterTaps : TileOperand<KIND, false, ROWS, T, STEPS> {
  using Base = TileOperand<KIND, false, ROWS, T, STEPS>;
  using Raw = typename Base::Raw;
  static constexpr int LOADS = Base::LOADS;
  __amdgpu_buffer_rsrc_t w;
  int j, J, K, S;
  int k[LOADS], s[LOADS], at[LOADS];
  int adv_k, adv_s, adv_off, wrap_off, row_off;

  template <class Args>
  __device__ __forceinline__ void setup(const Args &g, const ConvTilePart &p, int n0, int t, int tile0, int step0,
                                        uint32_t lds, int first) {
    this->ragged = false, this->cut = 0;
    this->place(t, tile0, step0, lds);
    J = p.J, K = g.C, S = p.S;
    w = conv_tile_rsrc(g.d.b, g.w_bytes);
    const int n = n0 + t % Base::CPR * 8;
    j = first * 64 + t / Base::CPR;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int jj = j + i * Base::STEP, tap = conv_div(jj, K, g.magic_c), r = conv_div(tap, S, p.magic_s);
      k[i] = jj - tap * K, s[i] = tap - r * S;
      at[i] = p.w_first + r * p.w_row + s[i] * p.w_tap + k[i] * g.w_pitch + n * 2;
    }
    if (n >= g.d.N) // (N is a multiple of 8)
      J = 0;
    adv_k = g.adv_c, adv_s = p.adv_s;
    adv_off = adv_k * g.w_pitch + adv_s * p.w_tap + p.adv_r * p.w_row;
    wrap_off = p.w_tap - K * g.w_pitch;
    row_off = p.w_row - S * p.w_tap;
  }

  template <bool TAIL> __device__ __forceinline__ void fetch(int, int, Raw &raw) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      raw.v[i] = __builtin_amdgcn_raw_buffer_load_b128(w, j + i * Base::STEP < J ? at[i] : kConvTileNone, 0, 0);
      k[i] += adv_k, s[i] += adv_s, at[i] += adv_off;
      const bool tap = k[i] >= K;
      k[i] -= tap ? K : 0, s[i] += tap ? 1 : 0, at[i] += tap ? wrap_off : 0;
      const bool row = s[i] >= S;
      s[i] -= row ? S : 0, at[i] += row ? row_off : 0;
    }
    j += 64;
  }
};

template <int KIND, bool DGRAD, int PARTS, class S, int U>
__global__ __launch_bounds__(256 * S::TEAMS)
__attribute__((amdgpu_waves_per_eu(2, 8))) void conv_tile_kernel(ConvTileArgsOf<PARTS> g) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const ConvTilePart &p = g.part[PARTS > 1 ? blockIdx.z : 0];
  const uint32_t id = tile_id(); // (row after row: neighbours read the same pixels)
  const int tile_m = id / (uint32_t)g.d.tiles_n, tile_n = id % (uint32_t)g.d.tiles_n;
  const int m0 = tile_m * S::BM, n0 = tile_n * S::BN;
  if (m0 >= p.M) // (parts of fewer pixels)
    return;
  const TileWave<S> at;
  const int t = threadIdx.x & 255;
  const TilePart share((p.J + 63) / 64, 0, g.d.splits, S::TEAMS, at.team);
  using OA = ConvPixels<KIND, S::BM, S::TM, S::STEPS>;
  using OB = std::conditional_t<DGRAD, ConvFilterTaps<KIND, S::BN, S::TN, S::STEPS>,
                                ConvFilterRows<KIND, S::BN, S::TN, S::STEPS>>;
  const uint32_t lds = (uint32_t)(uintptr_t)smem + (uint32_t)(at.team * 2 * S::kStage);
  OA oa;
  OB ob;
  oa.setup(g, p, m0, t, at.wm * S::TM, at.wk * S::STEPS, lds, share.s0);
  ob.setup(g, p, n0, t, at.wn * S::TN, at.wk * S::STEPS, lds + OA::BYTES, share.s0);
  tile_run<KIND, S, U, false, DGRAD>(
      g.d, (uint32_t)(uintptr_t)smem, share, at, oa, ob, id, 0, m0, n0, [&](int m) -> int64_t {
        if (m >= p.M)
          return -1;
        if (PARTS == 1)
          return (int64_t)m * g.d.o_sm;
        int n, i, j;
        conv_tile_pixel(p, m, n, i, j);
        return (((int64_t)n * g.out_h + i * g.step_h + p.h) * g.out_w + j * g.step_w + p.w) * g.d.o_sm;
      });
}

template <int KIND, bool DGRAD, int PARTS, int U, int MT, int NT, int TEAMS, bool SHORT = false>
int conv_tile_go(fhip_ctx *ctx, const ConvTileArgsOf<PARTS> &g) {
  using S = TileShape<KIND, MT, NT, TEAMS, SHORT>;
  auto kernel = conv_tile_kernel<KIND, DGRAD, PARTS, S, U>;
  static FhipOncePerDevice configured;
  if (S::kLds > 64 * 1024 && !configured.done(ctx->device)) {
    FHIP_HIP_CHECK(ctx, hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, S::kLds));
    configured.mark(ctx->device);
  }
  const dim3 grid((unsigned)(g.d.tiles_m * g.d.tiles_n), (unsigned)g.d.splits, (unsigned)g.parts);
  hipLaunchKernelGGL(kernel, grid, dim3(256 * TEAMS), S::kLds, ctx->stream, g);
  if (PARTS == 1 && g.d.splits > 1)
    hipLaunchKernelGGL((gemm_tile_finish_kernel<float, S::BM, S::BN, true>), dim3(grid.x, S::BM * S::BN / 1024),
                       dim3(256), 0, ctx->stream, g.d);
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  return 0;
}

template <int KIND, bool DGRAD, int PARTS>
int conv_tile_shape(fhip_ctx *ctx, const ConvTilePlan &p, const ConvTileArgsOf<PARTS> &g) {
  if (p.bm == 128 && p.bn == 128)
    return conv_tile_go<KIND, DGRAD, PARTS, 2, 2, 2, 1>(ctx, g);
  if (p.bm == 128)
    return conv_tile_go<KIND, DGRAD, PARTS, 4, 2, 1, 1>(ctx, g);
  if (p.bn == 128)
    return conv_tile_go<KIND, DGRAD, PARTS, 4, 1, 2, 1>(ctx, g);
  if (p.teams == 2)
    return conv_tile_go<KIND, DGRAD, PARTS, 2, 1, 1, 2>(ctx, g);
  return conv_tile_go<KIND, DGRAD, PARTS, 2, 1, 1, 1, true>(ctx, g);
}

template <int KIND> int conv_tile_kind(fhip_ctx *ctx, bool dgrad, const ConvTilePlan &p, const ConvTileArgs &g) {
  if (g.parts > 1)
    return conv_tile_shape<KIND, true, kConvTileParts>(ctx, p, g);
  ConvTileArgsOf<1> one{1,         g.H,     g.W,       g.C,       g.str_h, g.str_w, g.dil_h,  g.dil_w,  g.adv_c,
                        g.magic_c, g.x_bytes, g.w_bytes, g.w_pitch, g.out_h, g.out_w, g.step_h, g.step_w, {g.part[0]},
                        g.d};
  return dgrad ? conv_tile_shape<KIND, true, 1>(ctx, p, one) : conv_tile_shape<KIND, false, 1>(ctx, p, one);
}

#endif // FUSILLI_AMD_CSRC_CONV_TILE_KERNEL_H

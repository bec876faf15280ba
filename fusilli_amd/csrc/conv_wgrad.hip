// Convolution weight gradient for channels-last 16-bit tensors, any filter, stride,
// padding and dilation (most 3 x 3 filters at unit stride have conv_wgrad_direct.hip).
//
//   DW[k, (r, s, c)] = sum over output pixels m of
//                      DY[m, k] * X[pixel of m shifted by (r, s), c]
//
// A matrix product of K rows and J = R * S * C columns whose long reduction runs along
// both tensors' slow dimension.  Bound by LDS reads (eight transposing reads per four
// 32 x 32 x 16 MFMAs of a wavefront's 64 x 64 block) and, with few outputs, by the
// partial sums.  No operand is copied or padded in memory: C is a multiple of 8, so
// every 16-byte run of a column block lies inside one tap, and a lane fetches it from
// the shifted pixel, the buffer descriptor's range check giving zeros outside the
// image, the pixel range and the channel counts.  Where a pixel lies is decided once
// per chunk of pixels and kept in LDS; loads run three steps of 32 pixels ahead.
// Workgroups take a tile of outputs and a run of pixels; a second kernel adds the
// runs' sums in a fixed order.
//
// Before, both operands were copied into zero-padded grids for a batched GEMM of 128
// columns at least: N62 256 -> 48, 39 x 39, 3 x 3, bf16: 248 us -> 48.7; N32 112 ->
// 384, 26 x 26: 138 -> 34.4; N16 48 -> 48, 48 x 32: 36.7 -> 15.5.
//
// Reference semantics: node/conv_node.h:255-426 (ConvWGradNode),
// aten.convolution_backward, weight gradient.
#include "common.h"
#include "fast_paths.h"

#include <type_traits>

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
#define WG_AS3 __attribute__((address_space(3)))

constexpr int kWgThreads = 256;
constexpr int kWgStep = 32;    // pixels per step
constexpr int kWgChunk = 2048; // pixels whose places are in LDS at once
constexpr int kWgGroup = 15;   // steps of a short chain (a multiple of the three fetches in flight)

struct WgArgs {
  const char *x, *dy;
  float *part; // [run][K][J]
  int32_t H, W, C, K, P, Q, S, J;
  int32_t pad_h, pad_w, str_h, str_w, dil_h, dil_w;
  int32_t jtiles, tiles;
  int64_t pixels, run; // all, per workgroup (a multiple of the step)
  int64_t image_bytes;
  uint32_t chunk_images; // images that a chunk may touch
};

template <bool BF16> __device__ __forceinline__ f32x16 wg_mfma(const s16x8 &a, const s16x8 &b, const f32x16 &c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Byte of 16-byte run `chunk` of pixel slot `px` in a stage with rows of ROW bytes.  The
// 64-byte groups of a row are permuted by the pixel, so that the 8 pixels of a
// transposing read (64 bytes each) meet every bank twice.
template <int ROW> __device__ __forceinline__ int wg_swizzle(int px, int group) {
  if constexpr (ROW >= 256)
    return group ^ (px & 3);
  else if constexpr (ROW == 128)
    return group ^ ((px >> 1) & 1);
  else
    return group;
}
template <int ROW> __device__ __forceinline__ int wg_place(int px, int chunk) {
  return px * ROW + (wg_swizzle<ROW>(px, chunk >> 2) << 6) + ((chunk & 3) << 4);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t wg_rsrc(const char *base, uint32_t bytes) {
  const uint64_t b = (uint64_t)base;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
  return __builtin_amdgcn_make_buffer_rsrc((void *)(((uint64_t)hi << 32) | lo), 0,
                                           (int)__builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

// WK x WJ wavefronts of MT x 2 tiles of 32 x 32 outputs.
// SHORT, for gradients that are stored in f32: the accumulators start from zero every
// kWgGroup steps (480 pixels, 30 additions) and are added to a second set.  In one chain over
// a run, which has ten thousand pixels and more where tiles are many and runs few, the
// gradient of N8 512 -> 512, 112 x 112, 3 x 3 was 19.7 units of 2^-24 from the exact one and
// that of N32 512 -> 512, 56 x 56 at stride 2 9.7; 3.5 and 2.5 so, at 0 to 3 % more time
// (256 x 64 tiles 8 %).  Rounded to 16 bits it does not show.
template <bool BF16, int WK, int WJ, int MT, bool SHORT>
__global__ __launch_bounds__(kWgThreads) __attribute__((amdgpu_waves_per_eu(2, 4))) void
conv_wgrad_gather_kernel(WgArgs g) {
  constexpr int TK = 32 * MT * WK, TJ = 64 * WJ;
  constexpr int ROWA = TK * 2, ROWB = TJ * 2;
  constexpr int CA = TK / 8, CB = TJ / 8; // 16-byte runs per pixel
  constexpr int NA = (kWgStep * CA + kWgThreads - 1) / kWgThreads, NB = kWgStep * CB / kWgThreads;
  constexpr int kStage = kWgStep * (ROWA + ROWB);
  __shared__ __attribute__((aligned(16))) char stage[2 * kStage];
  __shared__ int2 place[kWgChunk];
  const int tid = threadIdx.x, l = tid & 63, wave = tid >> 6;
  // (workgroups go to the eight L2 slices in turn: the tiles of a run of pixels share one)
  uint32_t id = blockIdx.x;
  {
    const uint32_t per = gridDim.x / 8, rest = gridDim.x % 8, slice = id % 8;
    id = slice * per + (slice < rest ? slice : rest) + id / 8;
  }
  const int tile = (int)(id % (uint32_t)g.tiles);
  const uint32_t which = id / (uint32_t)g.tiles; // run of pixels
  const int64_t m0 = (int64_t)which * g.run;
  const int64_t m1 = m0 + g.run < g.pixels ? m0 + g.run : g.pixels;
  const int k0 = tile / g.jtiles * TK, j0 = tile % g.jtiles * TJ;
  // this thread's run of columns: its tap's shift and bytes behind a pixel's place
  int shift_h, shift_w, jbytes;
  {
    const int j = j0 + tid % CB * 8;
    const int tap = j / g.C, c = j - tap * g.C;
    const int r = tap / g.S, s = tap - r * g.S;
    shift_h = j < g.J ? r * g.dil_h : 1 << 20; // (beyond every image)
    shift_w = s * g.dil_w;
    jbytes = ((r * g.dil_h * g.W + s * g.dil_w) * g.C + c) * 2;
  }
  const int ka = k0 + tid % CA * 8;
  const bool a_in = ka < g.K && tid / CA < kWgStep;
  f32x16 acc[MT][2], sum[MT][2];
  auto clear = [](f32x16 (&v)[MT][2]) {
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          v[a][b][i] = 0.f;
  };
  clear(acc);
  if constexpr (SHORT)
    clear(sum);
  // transposing reads: 16 lanes address 4 pixels x 16 channels, lane i receives
  // channel i of the 4 pixels; lanes 32 .. 63 hold the upper 8 pixels of a step of 16
  const int wk = wave / WJ, wj = wave % WJ;
  const int lpx = (l >> 5) * 8 + ((l & 15) >> 2), lin = ((l >> 4) & 1) * 32 + (l & 3) * 8;
  int ra[MT], rb[2];
#pragma unroll
  for (int a = 0; a < MT; ++a)
    ra[a] = lpx * ROWA + (wg_swizzle<ROWA>(lpx, wk * MT + a) << 6) + lin;
#pragma unroll
  for (int b = 0; b < 2; ++b)
    rb[b] = kWgStep * ROWA + lpx * ROWB + (wg_swizzle<ROWB>(lpx, wj * 2 + b) << 6) + lin;

  for (int64_t c0 = m0; c0 < m1; c0 += kWgChunk) {
    const int count = (int)(m1 - c0 < kWgChunk ? m1 - c0 : kWgChunk);
    const int steps = (count + kWgStep - 1) / kWgStep;
    const int pq = g.P * g.Q;
    const int64_t first_image = c0 / pq;
    const int in_image = (int)(c0 - first_image * pq);
    __syncthreads(); // the last chunk's places and stages have been read
    for (int i = tid; i < steps * kWgStep; i += kWgThreads) {
      const uint32_t e = (uint32_t)(in_image + i);
      const uint32_t n = e / (uint32_t)pq, rest = e - n * (uint32_t)pq;
      const int p = (int)(rest / (uint32_t)g.Q), q = (int)(rest - (uint32_t)p * (uint32_t)g.Q);
      const int h = p * g.str_h - g.pad_h, w = q * g.str_w - g.pad_w;
      int2 v;
      v.x = (int)(n * (uint32_t)g.image_bytes) + (h * g.W + w) * g.C * 2;
      v.y = i < count ? (int)((uint32_t)(h & 0xffff) | ((uint32_t)w << 16)) : 0x8000; // row -32768
      place[i] = v;
    }
    const int64_t left = (g.pixels + pq - 1) / pq - first_image;
    const int64_t images = left < g.chunk_images ? left : g.chunk_images;
    const __amdgpu_buffer_rsrc_t rx =
        wg_rsrc(g.x + first_image * g.image_bytes, (uint32_t)(images * g.image_bytes));
    const __amdgpu_buffer_rsrc_t ry = wg_rsrc(g.dy + c0 * g.K * 2, (uint32_t)(count * g.K * 2));
    __syncthreads();
    u32x4 va[3][NA], vb[3][NB];
    auto fetch = [&](auto set, int t) {
      constexpr int B = decltype(set)::value;
      if (t >= steps)
        return;
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        const int px = t * kWgStep + tid / CA + i * (kWgThreads / CA);
        va[B][i] = __builtin_amdgcn_raw_buffer_load_b128(ry, a_in ? (px * g.K + ka) * 2 : (int)0x80000000, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const int2 v = place[t * kWgStep + tid / CB + i * (kWgThreads / CB)];
        const int h = (int)(short)(v.y & 0xffff) + shift_h, w = (v.y >> 16) + shift_w;
        const bool in = (unsigned)h < (unsigned)g.H && (unsigned)w < (unsigned)g.W;
        vb[B][i] = __builtin_amdgcn_raw_buffer_load_b128(rx, in ? v.x + jbytes : (int)0x80000000, 0, 0);
      }
    };
    auto step = [&](auto set, int t) {
      constexpr int B = decltype(set)::value;
      char *to = stage + (t & 1) * kStage;
#pragma unroll
      for (int i = 0; i < NA; ++i)
        if (NA * kWgThreads == kWgStep * CA || tid < kWgStep * CA)
          *(u32x4 *)(to + wg_place<ROWA>(tid / CA + i * (kWgThreads / CA), tid % CA)) = va[B][i];
#pragma unroll
      for (int i = 0; i < NB; ++i)
        *(u32x4 *)(to + kWgStep * ROWA + wg_place<ROWB>(tid / CB + i * (kWgThreads / CB), tid % CB)) = vb[B][i];
      fetch(set, t + 3);
      // (one barrier per step: a stage is written again two steps later, behind the
      // barrier that its readers reach after reading)
      __syncthreads();
      const WG_AS3 char *from = (const WG_AS3 char *)to;
#pragma unroll
      for (int ks = 0; ks < kWgStep / 16; ++ks) {
        s16x8 fa[MT], fb[2];
        auto read = [&](int at, int row) {
          const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((WG_AS3 s16x4 *)(from + at + ks * 16 * row));
          const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((WG_AS3 s16x4 *)(from + at + (ks * 16 + 4) * row));
          return s16x8{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        };
#pragma unroll
        for (int a = 0; a < MT; ++a)
          fa[a] = read(ra[a], ROWA);
#pragma unroll
        for (int b = 0; b < 2; ++b)
          fb[b] = read(rb[b], ROWB);
#pragma unroll
        for (int a = 0; a < MT; ++a)
#pragma unroll
          for (int b = 0; b < 2; ++b)
            acc[a][b] = wg_mfma<BF16>(fa[a], fb[b], acc[a][b]);
      }
    };
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    using S2 = std::integral_constant<int, 2>;
    fetch(S0{}, 0);
    fetch(S1{}, 1);
    fetch(S2{}, 2);
    auto walk = [&](int from, int to) {
      for (int t = from; t < to; t += 3) {
        step(S0{}, t);
        if (t + 1 < to)
          step(S1{}, t + 1);
        if (t + 2 < to)
          step(S2{}, t + 2);
      }
    };
    if constexpr (SHORT) {
      for (int t = 0; t < steps; t += kWgGroup) {
        walk(t, t + kWgGroup < steps ? t + kWgGroup : steps);
#pragma unroll
        for (int a = 0; a < MT; ++a)
#pragma unroll
          for (int b = 0; b < 2; ++b)
            sum[a][b] += acc[a][b];
        clear(acc);
      }
    } else {
      walk(0, steps);
    }
  }
  auto &result = SHORT ? sum : acc;
  // value i of a lane: row 8 * (i / 4) + 4 * (l / 32) + i % 4, column l % 32 of its tile
  float *out = g.part + (int64_t)which * g.K * g.J;
#pragma unroll
  for (int a = 0; a < MT; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int j = j0 + (wj * 2 + b) * 32 + (l & 31);
      if (j >= g.J)
        continue;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int k = k0 + (wk * MT + a) * 32 + 8 * (i >> 2) + 4 * (l >> 5) + (i & 3);
        if (k < g.K)
          out[(int64_t)k * g.J + j] = result[a][b][i];
      }
    }
}

struct WgradSumArgs {
  int32_t runs, J, S, C;
  int64_t total;          // K * J
  int64_t sk, sc, sr, ss; // element strides of DW [K, C, R, S]
  int32_t dt;
};

// DW = sum of the runs: a workgroup adds SLICES shares of the runs of 1024 / SLICES
// consecutive values (J is a multiple of 8), the shares in order.
template <int SLICES>
__global__ __launch_bounds__(256) void conv_wgrad_sum_kernel(WgradSumArgs a, const float *part,
                                                             void *dw) {
  constexpr int kLanes = 256 / SLICES;
  __shared__ f32x4 meet[SLICES][kLanes];
  const int o = threadIdx.x % kLanes, z = threadIdx.x / kLanes;
  const int64_t e = ((int64_t)blockIdx.x * kLanes + o) * 4;
  f32x4 s{0, 0, 0, 0};
  if (e < a.total) {
    const auto run = [&](int r) { return *(const f32x4 *)(part + r * a.total + e); };
    if constexpr (kLanes < 64)
      fhip_for_parts<4>(z, SLICES, a.runs, run, [&](f32x4 v, bool in) { s = in ? s + v : s; });
    else
      fhip_for_uniform_parts<8>(__builtin_amdgcn_readfirstlane(z), SLICES, a.runs, run, [&](f32x4 v) { s += v; });
  }
  if constexpr (SLICES > 1) {
    meet[z][o] = s;
    __syncthreads();
    if (z != 0)
      return;
#pragma unroll
    for (int i = 1; i < SLICES; ++i)
      s += meet[i][o];
  }
  if (e >= a.total)
    return;
  const int64_t k = __builtin_expect(a.total >> 32 != 0, 0) ? e / a.J : (uint32_t)e / (uint32_t)a.J;
  const int j = (int)(e - k * a.J), tap = j / a.C, c = j - tap * a.C;
  const int r = tap / a.S;
  const int64_t at = k * a.sk + r * a.sr + (tap - r * a.S) * a.ss + c * a.sc;
  const float v[4] = {s[0], s[1], s[2], s[3]};
  fhip_store_float(dw, a.dt, at, a.sc, v);
}

bool wg_channels_last(const fhip_tensor_desc &t) {
  int64_t expect = 1;
  int order[FHIP_MAX_RANK], n = 0;
  order[n++] = 1;
  for (int i = t.rank - 1; i >= 2; --i)
    order[n++] = i;
  order[n++] = 0;
  for (int i = 0; i < n; ++i) {
    const int d = order[i];
    if (t.dim[d] != 1 && t.stride[d] != expect)
      return false;
    expect *= t.dim[d];
  }
  return true;
}

struct WgradPlan {
  bool ok = false;
  WgArgs a{};
  int tk = 0, tj = 0;
  int64_t runs = 0;
  size_t part_bytes = 0, contract = 0;
};

// The workspace that callers bring, 0 for descriptors that ask for none.  Saved plans hold
// its size and are taken only where they equal the plan of today byte for byte
// (Graph::loadFromArtifact), so it stays what it was when X and DY were copied into
// zero-padded grids (rows and columns padded, 64-pixel pitch, DY of 128 channels at
// least) in front of the sums of every image's share; the sums of the runs fit in it.
size_t wgrad_contract(const fhip_conv_desc *d) {
  const int64_t N = d->x.dim[0], C = d->x.dim[1], K = d->w.dim[0], R = d->w.dim[2], S = d->w.dim[3];
  const int64_t P = d->y.dim[2], Q = d->y.dim[3], str = d->stride[0];
  if (str != d->stride[1] || d->dilation[1] != 1 || S * C < 128)
    return 0;
  const int64_t rows = (d->x.dim[2] + 2 * d->padding[0] + str - 1) / str * str, rows_y = rows / str;
  const int64_t pitch = (d->x.dim[3] + 2 * d->padding[1] + 63) / 64 * 64;
  if (P > rows_y || (Q - 1) * str + S > pitch)
    return 0;
  const int64_t Kp = K < 128 ? 128 : K, slices = rows_y * pitch / 64;
  auto line = [](int64_t bytes) { return (size_t)(bytes + 255) / 256 * 256; };
  int64_t split = 1;
  for (int64_t f = 1; f <= slices; ++f)
    if (slices % f == 0 && slices / f >= 8 && N * f * ((S * C + 127) / 128) * ((K + 127) / 128) <= 1024)
      split = f;
  const size_t x = line((N * rows * pitch * C + (R - 1) * d->dilation[0] * pitch * C + S * C) * 2);
  const size_t dy = line(N * rows_y * pitch * Kp * 2);
  if (x >= (1ull << 32) || dy >= (1ull << 32) || N * split > 65535)
    return 0;
  return x + dy + line(R * N * split * Kp * S * C * 4);
}

WgradPlan make_wgrad_plan(const fhip_conv_desc *d) {
  WgradPlan p;
  if (d->spatial_rank != 2)
    return p;
  const int dt = d->x.dtype, wdt = d->w.dtype;
  if ((dt != FHIP_BFLOAT16 && dt != FHIP_HALF) || d->y.dtype != dt)
    return p;
  if (wdt != FHIP_BFLOAT16 && wdt != FHIP_HALF && wdt != FHIP_FLOAT)
    return p;
  if (d->w.dim[1] != d->x.dim[1]) // groups
    return p;
  if (!wg_channels_last(d->x) || !wg_channels_last(d->y))
    return p;
  const int64_t N = d->x.dim[0], C = d->x.dim[1], H = d->x.dim[2], W = d->x.dim[3];
  const int64_t K = d->w.dim[0], R = d->w.dim[2], S = d->w.dim[3];
  const int64_t P = d->y.dim[2], Q = d->y.dim[3];
  if (C % 8 != 0 || K % 8 != 0) // whole 16-byte runs of a pixel's channels
    return p;
  // places of pixels are 16-bit signed pairs, -32768 marks none
  for (int i = 0; i < 2; ++i)
    if (d->x.dim[2 + i] >= 32768 || d->padding[i] >= 16384 || d->stride[i] >= 16384 ||
        d->dilation[i] >= 16384 || d->dilation[i] * (d->w.dim[2 + i] - 1) >= 16384 ||
        (d->y.dim[2 + i] - 1) * d->stride[i] - d->padding[i] >= 32768)
      return p;
  const int64_t J = R * S * C, pixels = N * P * Q, image = H * W * C * 2;
  const int64_t chunk_images = (kWgChunk + P * Q - 2) / (P * Q) + 1;
  // 32-bit offsets inside a chunk, taps in the padding included (they wrap)
  if (P * Q >= (1ll << 30) || K >= (1 << 18) || J >= (1ll << 30) || pixels >= (1ll << 40) ||
      (chunk_images + 1) * image >= (1ll << 31))
    return p;
  WgArgs &a = p.a;
  a.H = (int32_t)H, a.W = (int32_t)W, a.C = (int32_t)C, a.K = (int32_t)K;
  a.P = (int32_t)P, a.Q = (int32_t)Q, a.S = (int32_t)S, a.J = (int32_t)J;
  a.pad_h = (int32_t)d->padding[0], a.pad_w = (int32_t)d->padding[1];
  a.str_h = (int32_t)d->stride[0], a.str_w = (int32_t)d->stride[1];
  a.dil_h = (int32_t)d->dilation[0], a.dil_w = (int32_t)d->dilation[1];
  a.pixels = pixels, a.image_bytes = image, a.chunk_images = (uint32_t)chunk_images;
  // the tile with the least padding; equal ones: the squarest (fewest bytes per product)
  static const int shapes[4][2] = {{128, 128}, {64, 256}, {256, 64}, {32, 256}};
  int64_t best = 0;
  for (const auto &s : shapes) {
    const int64_t area = ((K + s[0] - 1) / s[0]) * ((J + s[1] - 1) / s[1]) * s[0] * s[1];
    if (p.tk == 0 || area < best)
      best = area, p.tk = s[0], p.tj = s[1];
  }
  a.jtiles = (int32_t)((J + p.tj - 1) / p.tj);
  const int64_t tiles = ((K + p.tk - 1) / p.tk) * a.jtiles;
  if (tiles >= (1 << 20))
    return p;
  a.tiles = (int32_t)tiles;
  // runs of pixels: two workgroups per compute unit where each then has 16 steps, else
  // one, of 4 steps at least (planned for 256 units whatever the device: the workspace
  // size is answered without one)
  const int64_t steps = (pixels + kWgStep - 1) / kWgStep;
  int64_t runs = (steps * tiles >= 512 * 16 ? 512 : 256) / tiles;
  p.contract = wgrad_contract(d);
  if (p.contract && runs > (int64_t)p.contract / (K * J * 4))
    runs = (int64_t)p.contract / (K * J * 4);
  runs = runs < steps / 4 ? runs : steps / 4;
  runs = runs < 1 ? 1 : runs;
  a.run = (steps + runs - 1) / runs * kWgStep;
  p.runs = (pixels + a.run - 1) / a.run;
  p.part_bytes = (size_t)(p.runs * K * J) * sizeof(float);
  p.ok = p.runs * tiles < (1ll << 23);
  return p;
}

int wg_run(fhip_ctx *ctx, const fhip_conv_desc *d, const WgradPlan &p, const void *dy,
           const void *x, void *dw, void *part) {
  WgArgs a = p.a;
  a.x = (const char *)x, a.dy = (const char *)dy, a.part = (float *)part;
  auto go = [&](auto bf, auto sh) {
    constexpr bool B = decltype(bf)::value, S = decltype(sh)::value;
    auto kernel = p.tk == 32    ? conv_wgrad_gather_kernel<B, 1, 4, 1, S>
                  : p.tk == 64  ? conv_wgrad_gather_kernel<B, 1, 4, 2, S>
                  : p.tk == 128 ? conv_wgrad_gather_kernel<B, 2, 2, 2, S>
                                : conv_wgrad_gather_kernel<B, 4, 1, 2, S>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(p.runs * a.tiles)), dim3(kWgThreads), 0, ctx->stream, a);
  };
  // (a gradient rounded to 16 bits does not show the difference)
  const bool shorter = d->w.dtype == FHIP_FLOAT;
  if (d->x.dtype == FHIP_BFLOAT16)
    shorter ? go(std::true_type{}, std::true_type{}) : go(std::true_type{}, std::false_type{});
  else
    shorter ? go(std::false_type{}, std::true_type{}) : go(std::false_type{}, std::false_type{});
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  WgradSumArgs s;
  s.runs = (int32_t)p.runs, s.J = a.J, s.S = a.S, s.C = a.C;
  s.total = (int64_t)a.K * a.J;
  s.sk = d->w.dim[0] == 1 ? 0 : d->w.stride[0];
  s.sc = d->w.dim[1] == 1 ? 0 : d->w.stride[1];
  s.sr = d->w.dim[2] == 1 ? 0 : d->w.stride[2];
  s.ss = d->w.dim[3] == 1 ? 0 : d->w.stride[3];
  s.dt = d->w.dtype;
  auto sum = [&](auto zz) {
    constexpr int Z = decltype(zz)::value;
    const int64_t per = 1024 / Z;
    hipLaunchKernelGGL(conv_wgrad_sum_kernel<Z>, dim3((unsigned)((s.total + per - 1) / per)), dim3(256),
                       0, ctx->stream, s, (const float *)part, dw);
  };
  // (eight loads in flight per thread: more shares where there are more runs)
  if (s.runs > 32)
    sum(std::integral_constant<int, 16>{});
  else if (s.runs > 8)
    sum(std::integral_constant<int, 4>{});
  else
    sum(std::integral_constant<int, 1>{});
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  fhip_note_kernel(ctx, "conv_wgrad_gather %dx%d runs=%d", p.tk, p.tj, (int)p.runs);
  return 0;
}

} // namespace

// Descriptors whose partial sums go to the caller's workspace; the others that the
// kernel takes (fewer than 128 columns per filter row, unequal strides, dilation along
// W) keep them in the context's scratch.
bool fhip_fast_conv_wgrad_applicable(const fhip_conv_desc *d,
                                     size_t *workspace_bytes) {
  if (fhip_fast_conv_wgrad_direct_applicable(d, workspace_bytes))
    return true;
  const WgradPlan p = make_wgrad_plan(d);
  const bool ok = p.ok && p.contract != 0;
  if (workspace_bytes)
    *workspace_bytes = ok ? p.contract : 0;
  return ok;
}

int fhip_fast_conv_wgrad(fhip_ctx *ctx, const fhip_conv_desc *d, const void *dy,
                         const void *x, void *dw, void *workspace, size_t workspace_bytes) {
  {
    bool handled = false;
    const int rc = fhip_fast_conv_wgrad_direct(ctx, d, dy, x, dw, workspace, workspace_bytes, &handled);
    if (handled || rc != 0)
      return rc;
  }
  const WgradPlan p = make_wgrad_plan(d);
  FHIP_REQUIRE(ctx, p.ok, "conv wgrad: descriptor not supported by the MFMA path");
  FHIP_REQUIRE(ctx, ((uintptr_t)workspace & 255) == 0 && ((uintptr_t)x & 15) == 0 &&
                        ((uintptr_t)dy & 15) == 0,
               "conv wgrad: workspace must be 256-byte and tensors 16-byte aligned");
  return wg_run(ctx, d, p, dy, x, dw, workspace);
}

int fhip_gather_conv_wgrad(fhip_ctx *ctx, const fhip_conv_desc *d, const void *dy, const void *x,
                           void *dw, bool *handled) {
  *handled = false;
  const WgradPlan p = make_wgrad_plan(d);
  if (!p.ok || (((uintptr_t)x | (uintptr_t)dy) & 15) != 0)
    return 0;
  const int rc = fhip_fast_conv_wgrad_direct(ctx, d, dy, x, dw, nullptr, 0, handled);
  if (*handled || rc != 0)
    return rc;
  if (!fhip_ctx_scratch_ready(ctx, p.part_bytes))
    return 0;
  void *scratch = nullptr;
  if (fhip_ctx_scratch(ctx, p.part_bytes, &scratch) != 0)
    return 1;
  *handled = true;
  return wg_run(ctx, d, p, dy, x, dw, scratch);
}

// Batch normalisation forward for dense channels-last tensors.
//
// X [N, C, spatial...] with the channel as the fastest dim is a matrix of
// rows = N * spatial pixels by C channels, and the statistics are column
// sums.  A thread owns one 16-byte chunk of channels (8 of a 16-bit type, 4
// floats) -- the same chunk in every row it visits -- so loads are whole
// pixel vectors, the per-channel parameters stay in registers, and nothing is
// indexed per element:
//
//   training   pass 1  a workgroup walks a block of rows; its threads add
//                      (x - p) and (x - p)^2 per channel around a pivot p =
//                      the channel's value in row 0 (the variance does not
//                      cancel for channels far from 0), the row lanes of a
//                      chunk meet in LDS, and the workgroup's two sums per
//                      channel go to the context's scratch;
//              pass 2  every workgroup adds the sums of its channels (in a
//                      fixed order: the same mean and multiplier everywhere),
//                      then y = (x - mean) * a + b over its rows (X comes
//                      from the caches where it still is there);
//   inference  pass 2 with the running statistics.
//
// Workgroups take up to 64 channels (128 bytes of a row of 16-bit values), as
// many beside each other as the channels need, so that pass 2 reads few sums: a
// launch of its own for them, as large as its wait for a few workgroups' loads,
// took 3.3 to 12 us (16 x 48 x 48 x 32 f16 13.3 us in three launches, 9.7 in two;
// 16 x 256 x 14 x 14 12.9, 9.1; 16 x 2048 x 14 x 14 28.2, 13; 64 x 256 x 56 x 56 53.5, 51).
//
// Reference semantics: aten.native_batch_norm (reference
// support/asm_emitter.h:1066-1290, node/batchnorm_node.h:33-245): biased
// variance, saved statistics = (mean, 1 / sqrt(var + eps)).
#include "common.h"
#include "fast_paths.h"

namespace {

constexpr int kBnThreads = 256;
constexpr int kBnWidth = 64; // most channels of a workgroup

struct BnFastArgs {
  const void *x;
  void *y;
  const void *scale, *bias, *mean, *var; // per-channel vectors (may be null)
  void *saved_mean, *saved_inv;
  float *partial; // [workgroups][2][C], then pivot[C]
  int64_t rows;
  int32_t C, row_lanes, rows_per_wg, nwg;
  int32_t groups, chunks; // workgroups beside each other, the chunks of each
  int32_t scale_dt, bias_dt, running_dt, stats_dt;
  int32_t training;
  float eps;
};

template <typename T> struct BnVec;
template <> struct BnVec<float> {
  static constexpr int kN = 4;
  typedef float Raw __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ void load(const void *p, int64_t i, float (&v)[4]) {
    const float4 t = *(const float4 *)((const float *)p + i);
    v[0] = t.x, v[1] = t.y, v[2] = t.z, v[3] = t.w;
  }
  static __device__ __forceinline__ void store(void *p, int64_t i, const float (&v)[4]) {
    *(float4 *)((float *)p + i) = make_float4(v[0], v[1], v[2], v[3]);
  }
};
template <typename H> struct BnVec16 {
  static constexpr int kN = 8;
  typedef H hx8 __attribute__((ext_vector_type(8)));
  typedef hx8 Raw;
  static __device__ __forceinline__ void load(const void *p, int64_t i, float (&v)[8]) {
    const hx8 t = *(const hx8 *)((const H *)p + i);
#pragma unroll
    for (int k = 0; k < 8; ++k)
      v[k] = (float)t[k];
  }
  static __device__ __forceinline__ void store(void *p, int64_t i, const float (&v)[8]) {
    hx8 t;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      t[k] = (H)v[k];
    __builtin_nontemporal_store(t, (hx8 *)((H *)p + i));
  }
};
template <> struct BnVec<__bf16> : BnVec16<__bf16> {};
template <> struct BnVec<_Float16> : BnVec16<_Float16> {};

// pass 1: partial[wg][0][c] = sum (x - p), partial[wg][1][c] = sum (x - p)^2
template <typename T>
__global__ __launch_bounds__(kBnThreads) void bn_stats_kernel(BnFastArgs g) {
  using V = BnVec<T>;
  extern __shared__ __attribute__((aligned(16))) float red[]; // [row_lanes][2][width]
  const int chunk = threadIdx.x % g.chunks, lane = threadIdx.x / g.chunks;
  const int width = g.chunks * V::kN, base = (int)blockIdx.y * width; // this workgroup's channels
  const int c0 = base + chunk * V::kN;
  float s1[V::kN], s2[V::kN];
#pragma unroll
  for (int k = 0; k < V::kN; ++k)
    s1[k] = s2[k] = 0.f;
  if (lane < g.row_lanes && c0 < g.C) {
    float pv[V::kN];
    V::load(g.x, c0, pv); // row 0
    // (pass 2 may write over it: Y may be X)
    if (blockIdx.x == 0 && lane == 0)
#pragma unroll
      for (int k = 0; k < V::kN; k += 4)
        *(float4 *)&g.partial[(int64_t)g.nwg * 2 * g.C + c0 + k] = make_float4(pv[k], pv[k + 1], pv[k + 2], pv[k + 3]);
    const int64_t r0 = (int64_t)blockIdx.x * g.rows_per_wg;
    const int64_t r1 = r0 + g.rows_per_wg < g.rows ? r0 + g.rows_per_wg : g.rows;
    // eight rows in flight per lane (a workgroup has a dozen or so in all:
    // the loop is as long as its loads' latency, not its arithmetic); rows
    // past the end re-read the last one and count as zero
    constexpr int kFly = 8;
    for (int64_t r = r0 + lane; r < r1; r += (int64_t)kFly * g.row_lanes) {
      float v[kFly][V::kN];
#pragma unroll
      for (int u = 0; u < kFly; ++u) {
        const int64_t rr = r + (int64_t)u * g.row_lanes;
        V::load(g.x, (rr < r1 ? rr : r1 - 1) * g.C + c0, v[u]);
      }
      // (a round's sums from zero: chains of roundings as long as the rounds are many)
#pragma unroll
      for (int k = 0; k < V::kN; ++k) {
        float t1 = 0.f, t2 = 0.f;
#pragma unroll
        for (int u = 0; u < kFly; ++u) {
          const float d = r + (int64_t)u * g.row_lanes < r1 ? v[u][k] - pv[k] : 0.f;
          t1 += d;
          t2 = __builtin_fmaf(d, d, t2);
        }
        s1[k] += t1, s2[k] += t2;
      }
    }
    // (whole 16-byte stores: scalar ones would meet on the banks eight at a time)
#pragma unroll
    for (int k = 0; k < V::kN; k += 4) {
      *(float4 *)&red[(lane * 2 + 0) * width + c0 - base + k] =
          make_float4(s1[k], s1[k + 1], s1[k + 2], s1[k + 3]);
      *(float4 *)&red[(lane * 2 + 1) * width + c0 - base + k] =
          make_float4(s2[k], s2[k + 1], s2[k + 2], s2[k + 3]);
    }
  }
  __syncthreads();
  // the row lanes' sums, in a fixed order, by the first 2 * width threads (in turns)
  for (int o = threadIdx.x; o < 2 * width; o += kBnThreads) {
    const int which = o >= width, c = base + o - which * width;
    if (c >= g.C)
      continue;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    int l = 0;
#pragma unroll 2
    for (; l + 4 <= g.row_lanes; l += 4)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        acc[i] += red[(l + i) * 2 * width + o];
    for (; l < g.row_lanes; ++l)
      acc[0] += red[l * 2 * width + o];
    g.partial[((int64_t)blockIdx.x * 2 + which) * g.C + c] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  }
}

// (the other types' code out of the way)
__device__ __forceinline__ float bn_load(const void *p, int dt, int c) {
  return __builtin_expect(dt == FHIP_FLOAT, 1) ? ((const float *)p)[c] : fhip_load<float>(p, dt, c);
}
// pass 2: y = (x - mean) * (inv * scale) + bias
template <typename T>
__global__ __launch_bounds__(kBnThreads) void bn_apply_kernel(BnFastArgs g) {
  using V = BnVec<T>;
  typedef typename V::Raw Raw;
  constexpr int kFly = 4;
  __shared__ __attribute__((aligned(16))) float red[kBnThreads * 4]; // [slices][2][width]
  __shared__ float abm[3][kBnWidth];
  const int tid = threadIdx.x, chunk = tid % g.chunks, lane = tid / g.chunks;
  const int width = g.chunks * V::kN, base = (int)blockIdx.y * width;
  const int c0 = base + chunk * V::kN;
  const bool mine = lane < g.row_lanes && c0 < g.C;
  const int64_t step = (int64_t)gridDim.x * g.row_lanes;
  int64_t r = (int64_t)blockIdx.x * g.row_lanes + lane;
  // (the first rows and the channels' own values are requested ahead of the sums)
  Raw v[kFly];
  auto fetch = [&]() {
#pragma unroll
    for (int u = 0; u < kFly; ++u) {
      const int64_t rr = r + u * step;
      v[u] = *(const Raw *)((const T *)g.x + (mine && rr < g.rows ? rr * g.C + c0 : 0));
    }
  };
  fetch();
  const int c = base + tid;
  const bool owner = tid < width && c < g.C;
  float sc = 1.f, bi = 0.f, mean = 0.f, var = 0.f;
  if (owner) {
    if (g.scale)
      sc = bn_load(g.scale, g.scale_dt, c);
    if (g.bias)
      bi = bn_load(g.bias, g.bias_dt, c);
    if (g.training) {
      mean = g.partial[(int64_t)g.nwg * 2 * g.C + c]; // (the pivot)
    } else {
      mean = bn_load(g.mean, g.running_dt, c);
      var = bn_load(g.var, g.running_dt, c);
    }
  }
  if (g.training) {
    const int quads = width / 2, slices = kBnThreads / quads; // runs of four of 2 * width sums
    const int q = tid % quads, slice = tid / quads, which = q >= width / 4;
    const int qc = base + (q - which * (width / 4)) * 4;
    // (two chains in turn)
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f), other = s;
    if (slice < slices && qc < g.C) {
      const float *p = g.partial + (int64_t)which * g.C + qc;
      fhip_for_parts<8>(
          slice, slices, g.nwg, [&](int w) { return *(const float4 *)(p + (int64_t)w * 2 * g.C); },
          [&](float4 t, bool in) {
            const float4 was = s;
            s.x = in ? other.x + t.x : other.x, s.y = in ? other.y + t.y : other.y;
            s.z = in ? other.z + t.z : other.z, s.w = in ? other.w + t.w : other.w;
            other = was;
          });
      *(float4 *)&red[(slice * quads + q) * 4] =
          make_float4(s.x + other.x, s.y + other.y, s.z + other.z, s.w + other.w);
    }
    __syncthreads();
    if (owner) {
      // (eight or more slices, four chains; those behind the last count as zero)
      float u1[4] = {0.f, 0.f, 0.f, 0.f}, u2[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
      for (int i = 0; i < slices; i += 4)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const float *at = red + (i + k < slices ? i + k : 0) * 2 * width + tid;
          u1[k] += i + k < slices ? at[0] : 0.f;
          u2[k] += i + k < slices ? at[width] : 0.f;
        }
      const float s1 = (u1[0] + u1[1]) + (u1[2] + u1[3]), s2 = (u2[0] + u2[1]) + (u2[2] + u2[3]);
      const float n = (float)g.rows;
      const float m1 = s1 / n;
      mean += m1;
      var = s2 / n - m1 * m1;
      var = var > 0.f ? var : 0.f;
    }
  }
  if (owner) {
    const float inv = 1.0f / sqrtf(var + g.eps);
    if (g.training && blockIdx.x == 0) {
      if (__builtin_expect(g.stats_dt == FHIP_FLOAT, 1)) {
        ((float *)g.saved_mean)[c] = mean;
        ((float *)g.saved_inv)[c] = inv;
      } else {
#pragma clang loop unroll(disable)
        for (int i = 0; i < 2; ++i)
          fhip_store<float>(i ? g.saved_inv : g.saved_mean, g.stats_dt, c, i ? inv : mean);
      }
    }
    abm[0][tid] = inv * sc, abm[1][tid] = bi, abm[2][tid] = mean;
  }
  __syncthreads();
  if (!mine)
    return;
  float a[V::kN], m[V::kN], b[V::kN];
#pragma unroll
  for (int k = 0; k < V::kN; ++k) {
    a[k] = abm[0][c0 - base + k];
    b[k] = abm[1][c0 - base + k];
    m[k] = abm[2][c0 - base + k];
  }
  while (r < g.rows) {
#pragma unroll
    for (int u = 0; u < kFly; ++u) {
      const int64_t rr = r + u * step;
      if (rr >= g.rows)
        break;
      float o[V::kN];
#pragma unroll
      for (int k = 0; k < V::kN; ++k)
        o[k] = __builtin_fmaf((float)v[u][k] - m[k], a[k], b[k]);
      V::store(g.y, rr * g.C + c0, o);
    }
    r += kFly * step;
    if (r < g.rows)
      fetch();
  }
}

// dense channels-last strides of dims [N, C, spatial...]
bool bn_channels_last(const fhip_tensor_desc &t) {
  if (t.dim[1] != 1 && t.stride[1] != 1)
    return false;
  int64_t expect = t.dim[1];
  for (int i = t.rank - 1; i >= 2; --i) {
    if (t.dim[i] != 1 && t.stride[i] != expect)
      return false;
    expect *= t.dim[i];
  }
  return t.dim[0] == 1 || t.stride[0] == expect;
}

bool bn_plan(const fhip_batchnorm_desc *d, BnFastArgs &g) {
  if (d->x.rank < 2 || d->x.dtype != d->y.dtype)
    return false;
  const int dt = d->x.dtype;
  if (dt != FHIP_FLOAT && dt != FHIP_BFLOAT16 && dt != FHIP_HALF)
    return false;
  const int vec = dt == FHIP_FLOAT ? 4 : 8;
  const int64_t C = d->x.dim[1];
  if (C < vec || C % vec != 0 || C / vec > kBnThreads)
    return false;
  if (!bn_channels_last(d->x) || !bn_channels_last(d->y))
    return false;
  const int64_t total = fhip_desc_volume(d->x);
  if (total <= 0 || total >= (1ll << 40))
    return false;
  g.C = (int32_t)C;
  g.rows = total / C;
  g.chunks = (int32_t)(C / vec);
  g.training = d->training;
  g.scale_dt = d->scale_dtype, g.bias_dt = d->bias_dtype;
  g.running_dt = d->running_dtype, g.stats_dt = d->stats_dtype;
  g.eps = d->epsilon;
  g.groups = (g.chunks + kBnWidth / vec - 1) / (kBnWidth / vec);
  g.chunks = (g.chunks + g.groups - 1) / g.groups;
  g.row_lanes = kBnThreads / g.chunks;
  // Blocks of rows: as many as the row lanes have in flight at once (eight each), and no more than
  // 256 workgroups, whose sums all of pass 2 reads (16 x 48 x 48 x 32: 74 blocks 10.0 us, 37 11.0, 147 11.1).
  const int64_t lanes = (g.rows + g.row_lanes - 1) / g.row_lanes;
  int64_t nwg = 256 / g.groups;
  nwg = nwg < (lanes + 7) / 8 ? nwg : (lanes + 7) / 8;
  g.rows_per_wg = (int32_t)((g.rows + nwg - 1) / nwg);
  g.nwg = (int32_t)((g.rows + g.rows_per_wg - 1) / g.rows_per_wg);
  return true;
}

template <typename T> void bn_launch(fhip_ctx *ctx, const BnFastArgs &g) {
  const int64_t lanes = (g.rows + g.row_lanes - 1) / g.row_lanes;
  if (g.training)
    hipLaunchKernelGGL(bn_stats_kernel<T>, dim3((unsigned)g.nwg, (unsigned)g.groups), dim3(kBnThreads),
                       (size_t)g.row_lanes * 2 * g.chunks * BnVec<T>::kN * 4, ctx->stream, g);
  // (every workgroup adds its channels' sums before it walks: one per compute unit, two from eight
  // rows a lane on; 16 x 48 x 48 x 32 with 1024 10.0 us, 512 9.4, 256 9.2, 64 x 64 x 56 x 56 21.6, 20.7, 20.8)
  const int64_t most = (lanes * g.groups <= 2048 ? 256 : 512) / g.groups;
  hipLaunchKernelGGL(bn_apply_kernel<T>, dim3((unsigned)(lanes < most ? lanes : most), (unsigned)g.groups),
                     dim3(kBnThreads), 0, ctx->stream, g);
}

} // namespace

bool fhip_fast_batchnorm_applicable(const fhip_batchnorm_desc *d) {
  BnFastArgs g{};
  return bn_plan(d, g);
}

int fhip_fast_batchnorm(fhip_ctx *ctx, const fhip_batchnorm_desc *d, const void *x,
                        const void *scale, const void *bias, const void *running_mean,
                        const void *running_var, void *y, void *saved_mean,
                        void *saved_inv_variance) {
  BnFastArgs g{};
  FHIP_REQUIRE(ctx, bn_plan(d, g), "batchnorm: descriptor not supported by the channels-last kernels");
  FHIP_REQUIRE(ctx, (((uintptr_t)x | (uintptr_t)y) & 15) == 0,
               "batchnorm: X and Y must be 16-byte aligned");
  void *scratch = nullptr;
  if (g.training && fhip_ctx_scratch(ctx, ((size_t)g.nwg * 2 + 1) * (size_t)g.C * sizeof(float), &scratch) != 0)
    return 1;
  g.x = x, g.y = y;
  g.scale = scale, g.bias = bias, g.mean = running_mean, g.var = running_var;
  g.saved_mean = saved_mean, g.saved_inv = saved_inv_variance;
  g.partial = (float *)scratch;
  if (d->x.dtype == FHIP_FLOAT)
    bn_launch<float>(ctx, g);
  else if (d->x.dtype == FHIP_BFLOAT16)
    bn_launch<__bf16>(ctx, g);
  else
    bn_launch<_Float16>(ctx, g);
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  fhip_note_kernel(ctx, "batchnorm_channels_last training=%d workgroups=%d", (int)d->training,
                   g.nwg);
  return 0;
}

// RMSNorm / LayerNorm forward for the dense rows that neither the
// register-resident nor the long-row kernels take: lengths and row strides that
// are no multiple of a 16-byte vector, long rows with a fused pointwise chain.
//
// Bound by memory (long rows) or by the latency of one launch (short ones); the
// generic kernel they ran on moves one element per thread with 64-bit index
// arithmetic, one workgroup per row whatever the row count.  Here a row's storage
// is walked linearly with 16-byte loads at element alignment (a misaligned vector
// costs one more cache line per wavefront, not one per lane) and the statistics are
// taken as before: the mean first, then the second moment around it.
//   * short rows: one wavefront each (four rows per workgroup), longer ones a
//     workgroup each; the second and third walk hit the caches;
//   * few long rows: segments of a row on workgroups of their own, sums through
//     the context's scratch, added in a fixed order (one launch per walk).
//
// bf16 RMSNorm + MUL 2 x 239616: 2465 us -> 8.6; f32 9 x 97280: 997 -> 8.7; bf16
// 16000 x 1003: 207 -> 20.3 (3.2 TB/s); f16 LayerNorm 9000 x 3001: 442 -> 49 (2.2 TB/s).
// (Unrolling the walk four times is slower: 49 -> 55.6.)
//
// Reference semantics: aten.rms_norm / aten.layer_norm over all dims except
// dim 0 (reference support/asm_emitter.h:1592-1626, 1427-1503;
// node/norm_utils.h:27-99).
#include "common.h"
#include "fast_paths.h"
#include "rownorm_kernel.h"

namespace {

constexpr int kRwThreads = 256;

struct RowWalkArgs {
  RowNormArgs n;
  double *partial; // [2][rows][splits]: sums of x, centred second moments
  double inv;      // 1 / elements per row
  int64_t seg;     // elements per segment, a multiple of the vector width
  int32_t splits;
};

template <typename T> struct RwVec {
  static constexpr int kN = 16 / sizeof(T);
  typedef T loose __attribute__((ext_vector_type(kN), aligned(sizeof(T))));
  static __device__ __forceinline__ void load(const T *p, float (&v)[kN]) {
    const loose t = *(const loose *)p;
#pragma unroll
    for (int k = 0; k < kN; ++k)
      v[k] = (float)t[k];
  }
  // the first `live` elements, zeros behind them
  static __device__ __forceinline__ void load_some(const T *p, int live, float (&v)[kN]) {
#pragma unroll
    for (int k = 0; k < kN; ++k)
      v[k] = k < live ? (float)p[k] : 0.f;
  }
  static __device__ __forceinline__ void store(T *p, const float (&v)[kN]) {
    loose t;
#pragma unroll
    for (int k = 0; k < kN; ++k)
      t[k] = (T)v[k];
    *(loose *)p = t;
  }
  static __device__ __forceinline__ void store_some(T *p, int live, const float (&v)[kN]) {
#pragma unroll
    for (int k = 0; k < kN; ++k)
      if (k < live)
        p[k] = (T)v[k];
  }
  // an operand of the row's type or f32
  static __device__ __forceinline__ void load_as(const void *p, int dt, int64_t at, int live,
                                                 float (&v)[kN]) {
    if (dt == DtypeOf<T>::value) {
      if (live == kN)
        load((const T *)p + at, v);
      else
        load_some((const T *)p + at, live, v);
    } else {
#pragma unroll
      for (int k = 0; k < kN; ++k)
        v[k] = k < live ? ((const float *)p)[at + k] : 0.f;
    }
  }
};

// Sums are f64 from a vector's pairs on, and the statistics are rounded once: a tree of
// f32 additions over lanes, wavefronts and segments left the means of 9000 x 3001 f16
// values 6.2e-8 off and those of 40 x 16385 9.5e-8 (generic kernel 6.0e-8 and 6.6e-8),
// 2.8e-8 so.

// Sum over a wavefront, the same in every lane: 16 lanes by data movement inside the
// vector unit, their four sums through scalar registers.
__device__ __forceinline__ double rw_wave_sum(double v) {
  auto add = [](double x, auto ctrl) {
    constexpr int kCtrl = decltype(ctrl)::value;
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, kCtrl, 0xF, 0xF, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), kCtrl, 0xF, 0xF, false);
    return x + __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
  };
  v = add(v, std::integral_constant<int, 0xB1>{});  // quad_perm [1,0,3,2]
  v = add(v, std::integral_constant<int, 0x4E>{});  // quad_perm [2,3,0,1]
  v = add(v, std::integral_constant<int, 0x124>{}); // row_ror 4
  v = add(v, std::integral_constant<int, 0x128>{}); // row_ror 8
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  double s[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, 16 * i);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), 16 * i);
    s[i] = __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
  }
  return (s[0] + s[1]) + (s[2] + s[3]);
}

// Sum over the WAVES wavefronts that share a row, the same in every lane.
template <int WAVES> __device__ __forceinline__ double rw_sum(double v, double *lds) {
  v = rw_wave_sum(v);
  if constexpr (WAVES > 1) {
    __syncthreads();
    if ((threadIdx.x & 63) == 0)
      lds[threadIdx.x >> 6] = v;
    __syncthreads();
    v = 0.;
#pragma unroll
    for (int i = 0; i < WAVES; ++i)
      v += lds[i];
  }
  return v;
}

// This lane's part of sum x (MOMENT 1) or sum (x - mean)^2 (MOMENT 2) of [lo, hi).
template <typename T, int MOMENT>
__device__ __forceinline__ double rw_walk(const T *xr, float mean, int64_t lo, int64_t hi, int lane,
                                          int lanes) {
  using V = RwVec<T>;
  double s = 0.;
  auto add = [&](const float (&v)[V::kN], int live) {
    float t[V::kN];
#pragma unroll
    for (int k = 0; k < V::kN; ++k) {
      const float d = v[k] - mean;
      t[k] = k < live ? (MOMENT == 1 ? v[k] : d * d) : 0.f;
    }
#pragma unroll
    for (int n = V::kN / 2; n > 0; n >>= 1)
#pragma unroll
      for (int k = 0; k < n; ++k)
        t[k] += t[k + n];
    s += (double)t[0];
  };
  int64_t i = lo + (int64_t)lane * V::kN;
  for (; i + V::kN <= hi; i += (int64_t)lanes * V::kN) {
    float v[V::kN];
    V::load(xr + i, v);
    add(v, V::kN);
  }
  if (i < hi) {
    float v[V::kN];
    V::load_some(xr + i, (int)(hi - i), v);
    add(v, (int)(hi - i));
  }
  return s;
}

template <typename T>
__device__ __forceinline__ void rw_apply(const RowNormArgs &g, int64_t row, float mean, float rstd,
                                         int64_t lo, int64_t hi, int lane, int lanes) {
  using V = RwVec<T>;
  constexpr int N = V::kN;
  const T *xr = (const T *)g.x + row * g.x_row_stride;
  T *orow = (T *)g.out + row * g.out_row_stride;
  for (int64_t i = lo + (int64_t)lane * N; i < hi; i += (int64_t)lanes * N) {
    const int live = hi - i < N ? (int)(hi - i) : N;
    float y[N], t[N];
    V::load_as(xr, DtypeOf<T>::value, i, live, y);
#pragma unroll
    for (int k = 0; k < N; ++k)
      y[k] = (y[k] - mean) * rstd;
    if (g.scale) {
      V::load_as(g.scale, g.scale_dt, i, live, t);
#pragma unroll
      for (int k = 0; k < N; ++k)
        y[k] *= t[k];
    }
    if (g.bias) {
      V::load_as(g.bias, g.bias_dt, i, live, t);
#pragma unroll
      for (int k = 0; k < N; ++k)
        y[k] += t[k];
    }
    fhip_round_fast_vec<N>(g.y_dt, y);
    for (int e = 0; e < g.epi_count; ++e) {
      const FastEpiOp &o = g.epi[e];
      if (o.kind == FHIP_OPERAND_NONE) {
        fhip_pw_fast_unary_vec<false, N>(o.mode, y, o.params.swish_beta);
      } else {
        if (o.kind == FHIP_OPERAND_TENSOR && o.col_unit) {
          V::load_as(o.ptr, o.operand_dtype, row * o.row_stride + i, live, t);
        } else {
          const float s = o.kind == FHIP_OPERAND_SCALAR ? o.scalar
                          : o.operand_dtype == DtypeOf<T>::value
                              ? (float)((const T *)o.ptr)[row * o.row_stride]
                              : ((const float *)o.ptr)[row * o.row_stride];
#pragma unroll
          for (int k = 0; k < N; ++k)
            t[k] = s;
        }
        fhip_pw_fast_binary_vec<N>(o.mode, o.acc_is_in1 != 0, y, t);
      }
      fhip_round_fast_vec<N>(o.result_dtype, y);
    }
    if (live == N)
      V::store(orow + i, y);
    else
      V::store_some(orow + i, live, y);
  }
}

__device__ __forceinline__ void rw_stats(const RowNormArgs &g, int64_t row, float mean, float rstd) {
  fhip_store<float>(g.mean, g.stats_dt, row, mean);
  fhip_store<float>(g.rstd, g.stats_dt, row, rstd);
}

// A row per WAVES wavefronts.
template <typename T, int WAVES>
__global__ __launch_bounds__(kRwThreads) void rownorm_walk_kernel(RowNormArgs g, double inv) {
  __shared__ double lds[WAVES];
  constexpr int kLanes = WAVES * 64;
  const int lane = threadIdx.x % kLanes;
  const int64_t row = (int64_t)blockIdx.x * (kRwThreads / kLanes) + threadIdx.x / kLanes;
  if (row >= g.rows) // (whole wavefronts; with WAVES > 1 the grid is exact)
    return;
  const T *xr = (const T *)g.x + row * g.x_row_stride;
  const float mean =
      g.is_layernorm ? (float)(rw_sum<WAVES>(rw_walk<T, 1>(xr, 0.f, 0, g.inner, lane, kLanes), lds) * inv) : 0.f;
  const float var = (float)(rw_sum<WAVES>(rw_walk<T, 2>(xr, mean, 0, g.inner, lane, kLanes), lds) * inv);
  const float rstd = 1.0f / sqrtf(var + g.eps);
  if (g.emit_stats && lane == 0)
    rw_stats(g, row, mean, rstd);
  rw_apply<T>(g, row, mean, rstd, 0, g.inner, lane, kLanes);
}

// The sum of a row's parts (at most one per thread).
__device__ __forceinline__ double rw_parts(const RowWalkArgs &g, int moment, int64_t row, double *lds) {
  const double *p = g.partial + ((moment - 1) * g.n.rows + row) * g.splits;
  return rw_sum<kRwThreads / 64>((int)threadIdx.x < g.splits ? p[threadIdx.x] : 0., lds);
}

template <typename T, int MOMENT>
__global__ __launch_bounds__(kRwThreads) void rownorm_walk_sums_kernel(RowWalkArgs g) {
  __shared__ double lds[kRwThreads / 64];
  const int64_t row = blockIdx.y, lo = blockIdx.x * g.seg;
  const int64_t hi = lo + g.seg < g.n.inner ? lo + g.seg : g.n.inner;
  float mean = 0.f;
  if (MOMENT == 2 && g.n.is_layernorm)
    mean = (float)(rw_parts(g, 1, row, lds) * g.inv);
  const T *xr = (const T *)g.n.x + row * g.n.x_row_stride;
  const double s = rw_sum<kRwThreads / 64>(rw_walk<T, MOMENT>(xr, mean, lo, hi, threadIdx.x, kRwThreads), lds);
  if (threadIdx.x == 0)
    g.partial[((MOMENT - 1) * g.n.rows + row) * g.splits + blockIdx.x] = s;
}

template <typename T>
__global__ __launch_bounds__(kRwThreads) void rownorm_walk_apply_kernel(RowWalkArgs g) {
  __shared__ double lds[kRwThreads / 64];
  const int64_t row = blockIdx.y, lo = blockIdx.x * g.seg;
  const int64_t hi = lo + g.seg < g.n.inner ? lo + g.seg : g.n.inner;
  const float mean = g.n.is_layernorm ? (float)(rw_parts(g, 1, row, lds) * g.inv) : 0.f;
  const float rstd = 1.0f / sqrtf((float)(rw_parts(g, 2, row, lds) * g.inv) + g.n.eps);
  if (g.n.emit_stats && blockIdx.x == 0 && threadIdx.x == 0)
    rw_stats(g.n, row, mean, rstd);
  rw_apply<T>(g.n, row, mean, rstd, lo, hi, threadIdx.x, kRwThreads);
}

template <typename T> void rw_launch_split(hipStream_t stream, const RowWalkArgs &g) {
  const dim3 grid((unsigned)g.splits, (unsigned)g.n.rows), wg(kRwThreads);
  if (g.n.is_layernorm)
    hipLaunchKernelGGL((rownorm_walk_sums_kernel<T, 1>), grid, wg, 0, stream, g);
  hipLaunchKernelGGL((rownorm_walk_sums_kernel<T, 2>), grid, wg, 0, stream, g);
  hipLaunchKernelGGL(rownorm_walk_apply_kernel<T>, grid, wg, 0, stream, g);
}

template <typename T> void rw_launch_rows(hipStream_t stream, const RowNormArgs &g, int waves) {
  const dim3 grid((unsigned)(waves == 1 ? (g.rows + 3) / 4 : g.rows)), wg(kRwThreads);
  if (waves == 1)
    hipLaunchKernelGGL((rownorm_walk_kernel<T, 1>), grid, wg, 0, stream, g, 1.0 / (double)g.inner);
  else
    hipLaunchKernelGGL((rownorm_walk_kernel<T, 4>), grid, wg, 0, stream, g, 1.0 / (double)g.inner);
}

} // namespace

// The caller (rownorm.hip) has checked that rows are dense and that X, OUT, scale,
// bias and the fused operands walk a row alike.
int fhip_norm_walk(fhip_ctx *ctx, int dtype, const RowNormArgs &n) {
  // A wavefront per row up to four vectors per lane, where the rows then still
  // fill half of the chip's wavefront slots or are shorter than two vectors per lane.
  const int64_t vec = 16 / (int64_t)fhip_dtype_size(dtype);
  const int waves = n.inner <= 128 * vec || (n.inner <= 256 * vec && n.rows >= 4096) ? 1 : 4;
  // Rows of more than four vectors per thread of a workgroup are cut where there are
  // fewer of them than two per compute unit, into about eight workgroups per unit and
  // segments of two vectors per thread at least (one launch more than whole rows).
  const int64_t cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  const int64_t min_seg = kRwThreads * vec * 2;
  int64_t splits = (8 * cus + n.rows - 1) / n.rows;
  const int64_t most = (n.inner + min_seg - 1) / min_seg;
  splits = splits < most ? splits : most;
  splits = splits < kRwThreads ? splits : kRwThreads;
  RowWalkArgs g{};
  const size_t sums = (size_t)(2 * n.rows * (splits > 0 ? splits : 0)) * sizeof(double);
  const bool cut = n.inner > 4 * kRwThreads * vec && n.rows < 2 * cus && splits > 1 &&
                   fhip_ctx_scratch_ready(ctx, sums);
  if (cut) {
    g.seg = ((n.inner + splits - 1) / splits + vec - 1) / vec * vec;
    g.splits = (int32_t)((n.inner + g.seg - 1) / g.seg);
    void *scratch = nullptr;
    if (fhip_ctx_scratch(ctx, sums, &scratch) != 0)
      return 1;
    g.partial = (double *)scratch;
    g.inv = 1.0 / (double)n.inner;
    g.n = n;
    fhip_note_kernel(ctx, "rownorm_walk segments=%d", g.splits);
  } else {
    fhip_note_kernel(ctx, "rownorm_walk waves_per_row=%d", waves);
  }
  auto go = [&](auto t) {
    typedef decltype(t) T;
    cut ? rw_launch_split<T>(ctx->stream, g) : rw_launch_rows<T>(ctx->stream, n, waves);
  };
  if (dtype == FHIP_BFLOAT16)
    go(__bf16{});
  else if (dtype == FHIP_HALF)
    go(_Float16{});
  else
    go(float{});
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  return 0;
}

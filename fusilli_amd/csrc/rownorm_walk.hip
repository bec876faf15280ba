// RMSNorm / LayerNorm forward for the dense rows that the register-resident kernels do not
// take or leave: lengths and row strides that are no multiple of a 16-byte vector, rows too
// long for registers, few long ones.
//
// Bound by memory (long rows) or by the latency of the launches (short ones); the
// generic kernel moves one element per thread with 64-bit index arithmetic, one
// workgroup per row whatever the row count.  Here a row's storage
// is walked linearly with 16-byte loads at element alignment (a misaligned vector
// costs one more cache line per wavefront, not one per lane) and the second moment is
// taken around a mean.
//   * short rows: one wavefront each (four rows per workgroup), longer ones a
//     workgroup each; the second and third walk hit the caches;
//   * few long rows: segments of a row on workgroups of their own, in two launches,
//     sums through the context's scratch, added in a fixed order.
//
// bf16 16000 x 1003 RMSNorm + MUL: 207 us (generic) -> 20.3 (3.2 TB/s); f16 LayerNorm 9000 x
// 3001: 442 -> 49 (2.2 TB/s).  (Unrolling the walk four times is slower: 49 -> 55.6.)
// Segments (recorded into a graph): bf16 LayerNorm 16 x 262144 9.8 -> 9.1 us, of which two launches
// that do next to nothing take 7; 600 x 300000 330 -> 246 (segments of eight vectors per thread),
// 204 x 9335 12.9 -> 9.0.
//
// Reference semantics: aten.rms_norm / aten.layer_norm over all dims except
// dim 0 (reference support/asm_emitter.h:1592-1626, 1427-1503;
// node/norm_utils.h:27-99).
#include "common.h"
#include "fast_paths.h"
#include "rownorm_kernel.h"

namespace {

constexpr int kRwThreads = 256;
constexpr int kRwWaves = kRwThreads / 64;
constexpr int64_t kRwResident = 16384; // vectors of the longest rows that rownorm_kernel.h holds

struct RowWalkArgs {
  RowNormArgs n;
  double *partial; // [rows][splits][2]: sums of x, second moments around the segment's mean
  double inv;      // 1 / elements per row,
  double inv_seg, inv_last; // per segment, of the last one
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
  // the same, kept in the row's type
  static __device__ __forceinline__ loose load_raw(const T *p, int live) {
    loose t;
    if (live == kN) {
      t = *(const loose *)p;
    } else {
#pragma unroll
      for (int k = 0; k < kN; ++k)
        t[k] = k < live ? p[k] : (T)0.f;
    }
    return t;
  }
  static __device__ __forceinline__ void widen(const loose &t, float (&v)[kN]) {
#pragma unroll
    for (int k = 0; k < kN; ++k)
      v[k] = (float)t[k];
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

// Sum of the first `live` x (MOMENT 1) or (x - mean)^2 (MOMENT 2) of a vector.
template <typename T, int MOMENT>
__device__ __forceinline__ double rw_tree(const float (&v)[RwVec<T>::kN], float mean, int live) {
  constexpr int N = RwVec<T>::kN;
  float t[N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const float d = v[k] - mean;
    t[k] = k < live ? (MOMENT == 1 ? v[k] : d * d) : 0.f;
  }
#pragma unroll
  for (int n = N / 2; n > 0; n >>= 1)
#pragma unroll
    for (int k = 0; k < n; ++k)
      t[k] += t[k + n];
  return (double)t[0];
}

// This lane's part of sum x (MOMENT 1) or sum (x - mean)^2 (MOMENT 2) of [lo, hi).
template <typename T, int MOMENT>
__device__ __forceinline__ double rw_walk(const T *xr, float mean, int64_t lo, int64_t hi, int lane,
                                          int lanes) {
  using V = RwVec<T>;
  double s = 0.;
  int64_t i = lo + (int64_t)lane * V::kN;
  for (; i + V::kN <= hi; i += (int64_t)lanes * V::kN) {
    float v[V::kN];
    V::load(xr + i, v);
    s += rw_tree<T, MOMENT>(v, mean, V::kN);
  }
  if (i < hi) {
    float v[V::kN];
    V::load_some(xr + i, (int)(hi - i), v);
    s += rw_tree<T, MOMENT>(v, mean, (int)(hi - i));
  }
  return s;
}

// Normalises, finishes and stores the `live` elements from `i` of a row, whose X, scale and
// bias (where there are any) are in x, sc and bi.
template <typename T>
__device__ __forceinline__ void rw_finish(const RowNormArgs &g, int64_t row, float mean, float rstd,
                                          int64_t i, int live, const float (&x)[RwVec<T>::kN],
                                          const float (&sc)[RwVec<T>::kN], const float (&bi)[RwVec<T>::kN]) {
  using V = RwVec<T>;
  constexpr int N = V::kN;
  float y[N], t[N];
#pragma unroll
  for (int k = 0; k < N; ++k)
    y[k] = (x[k] - mean) * rstd;
  if (g.scale) {
#pragma unroll
    for (int k = 0; k < N; ++k)
      y[k] *= sc[k];
  }
  if (g.bias) {
#pragma unroll
    for (int k = 0; k < N; ++k)
      y[k] += bi[k];
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
  T *orow = (T *)g.out + row * g.out_row_stride;
  if (live == N)
    V::store(orow + i, y);
  else
    V::store_some(orow + i, live, y);
}

template <typename T>
__device__ __forceinline__ void rw_apply(const RowNormArgs &g, int64_t row, float mean, float rstd,
                                         int64_t lo, int64_t hi, int lane, int lanes) {
  using V = RwVec<T>;
  constexpr int N = V::kN;
  const T *xr = (const T *)g.x + row * g.x_row_stride;
  for (int64_t i = lo + (int64_t)lane * N; i < hi; i += (int64_t)lanes * N) {
    const int live = hi - i < N ? (int)(hi - i) : N;
    float x[N], sc[N], bi[N];
    V::load_as(xr, DtypeOf<T>::value, i, live, x);
    if (g.scale)
      V::load_as(g.scale, g.scale_dt, i, live, sc);
    if (g.bias)
      V::load_as(g.bias, g.bias_dt, i, live, bi);
    rw_finish<T>(g, row, mean, rstd, i, live, x, sc, bi);
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

// Few long rows: a segment of a row per workgroup, two launches.  The first leaves every
// segment's sum and its second moment around the segment's own mean (RMSNorm: around zero);
// the second adds a row's pairs up, moved to the first segment's mean, and applies.
// (A segment per wavefront, no barrier in the first launch, but four times the pairs: bf16
// 4 x 65544 7.5 -> 7.9 us, f32 32 x 524288 34.8 -> 40.6.)
typedef double rw_pair __attribute__((ext_vector_type(2)));

// The mean of segment `i`, rounded: both launches have the same from a segment's sum.
__device__ __forceinline__ double rw_centre(const RowWalkArgs &g, int i, double sum) {
  return (double)(float)(sum * (i + 1 < g.splits ? g.inv_seg : g.inv_last));
}

// A segment is read once and reduced once.  A vector's deviations are taken in f32 from the
// vector's own mean (as f32 has it: their sum makes up for the difference) and moved in f64
// to `pivot`, an element of the segment, so that the second moment there is at most `elements`
// times the one around the segment's mean, to which it goes last: no digit that f32 holds is lost.
// (Sums first, then moments, of vectors kept or walked again: 0.2 to 0.6 us more.)
template <typename T>
__device__ __forceinline__ void rw_moments(const float (&v)[RwVec<T>::kN], int live, double pivot, double &s1,
                                           double &s2) {
  constexpr int N = RwVec<T>::kN;
  const float sum = (float)rw_tree<T, 1>(v, 0.f, live), mean = live == N ? sum * (1.f / N) : sum / (float)live;
  float d[N];
#pragma unroll
  for (int k = 0; k < N; ++k)
    d[k] = v[k] - mean;
  const double e = (double)mean - pivot, n = (double)live, rest = rw_tree<T, 1>(d, 0.f, live);
  // (around an infinite mean `rest` is NaN, where the row's mean is that infinity)
  s1 += __builtin_isfinite(sum) ? n * (double)mean + rest : (double)sum;
  s2 += rw_tree<T, 2>(d, 0.f, live) + e * (n * e + 2. * rest);
}

template <typename T, bool LAYER>
__global__ __launch_bounds__(kRwThreads) void rownorm_walk_sums_kernel(RowWalkArgs g) {
  using V = RwVec<T>;
  constexpr int N = V::kN, kStep = kRwThreads * N;
  __shared__ rw_pair lds[kRwWaves];
  const int64_t row = blockIdx.y, lo = blockIdx.x * g.seg;
  const int64_t hi = lo + g.seg < g.n.inner ? lo + g.seg : g.n.inner;
  const T *xr = (const T *)g.n.x + row * g.n.x_row_stride;
  double s1 = 0., s2 = 0.;
  if constexpr (LAYER) {
    const double pivot = (double)(float)xr[lo];
    auto add = [&](const typename V::loose &raw, int live) {
      float v[N];
      V::widen(raw, v);
      rw_moments<T>(v, live, pivot, s1, s2);
    };
    int64_t i = lo + (int64_t)threadIdx.x * N;
    for (; i + kStep + N <= hi; i += 2 * kStep) { // (two loads in flight)
      const typename V::loose a = V::load_raw(xr + i, N), b = V::load_raw(xr + i + kStep, N);
      add(a, N);
      add(b, N);
    }
    for (; i < hi; i += kStep) {
      const int live = hi - i < N ? (int)(hi - i) : N;
      add(V::load_raw(xr + i, live), live);
    }
  } else {
    s2 = rw_walk<T, 2>(xr, 0.f, lo, hi, threadIdx.x, kRwThreads);
  }
  s1 = LAYER ? rw_wave_sum(s1) : 0.;
  s2 = rw_wave_sum(s2);
  if ((threadIdx.x & 63) == 0)
    lds[threadIdx.x >> 6] = rw_pair{s1, s2};
  __syncthreads();
  if (threadIdx.x == 0) {
    s1 = s2 = 0.;
#pragma unroll
    for (int w = 0; w < kRwWaves; ++w) {
      s1 += lds[w].x;
      s2 += lds[w].y;
    }
    if constexpr (LAYER) {
      const double pivot = (double)(float)xr[lo], n = (double)(hi - lo);
      const double d = rw_centre(g, (int)blockIdx.x, s1) - pivot;
      s2 += d * (n * d - 2. * (s1 - n * pivot));
    }
    ((rw_pair *)g.partial)[row * g.splits + blockIdx.x] = rw_pair{s1, s2};
  }
}

// NV > 0 (LayerNorm): a thread's NV vectors of X come with their scale and bias while the pairs are
// on their way; 0: segments of any length are walked.
template <typename T, int NV>
__global__ __launch_bounds__(kRwThreads) void rownorm_walk_apply_kernel(RowWalkArgs g) {
  using V = RwVec<T>;
  constexpr int N = V::kN;
  __shared__ rw_pair lds[kRwWaves];
  const int64_t row = blockIdx.y, lo = blockIdx.x * g.seg;
  const int64_t hi = lo + g.seg < g.n.inner ? lo + g.seg : g.n.inner;
  // the pairs first: loads return in order
  const rw_pair *p = (const rw_pair *)g.partial + row * g.splits;
  const double first = p[0].x;
  const bool in = threadIdx.x < (unsigned)g.splits; // (at most one per thread)
  const rw_pair mine = p[in ? threadIdx.x : 0];
  typename V::loose rx[NV > 0 ? NV : 1], rs[NV > 0 ? NV : 1], rb[NV > 0 ? NV : 1];
  const bool own_s = g.n.scale && g.n.scale_dt == DtypeOf<T>::value;
  const bool own_b = g.n.bias && g.n.bias_dt == DtypeOf<T>::value;
  if constexpr (NV > 0) {
    const T *xr = (const T *)g.n.x + row * g.n.x_row_stride;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int64_t i = lo + (int64_t)(threadIdx.x + j * kRwThreads) * N;
      const int live = hi - i >= N ? N : hi > i ? (int)(hi - i) : 0;
      rx[j] = V::load_raw(xr + i, live);
      if (own_s)
        rs[j] = V::load_raw((const T *)g.n.scale + i, live);
      if (own_b)
        rb[j] = V::load_raw((const T *)g.n.bias + i, live);
    }
  }
  // sum (x - c0)^2 = sum (x - c)^2 + 2 d (sum x - n c) + n d^2 of a segment whose second
  // moment lies around c, d = c - c0 (RMSNorm: all zero)
  double c0 = 0., s = 0., q = in ? mine.y : 0.;
  const bool layer = NV > 0 || g.n.is_layernorm != 0;
  if (layer) {
    c0 = rw_centre(g, 0, first);
    const int64_t left = g.n.inner - (in ? threadIdx.x : 0) * g.seg;
    const double n = (double)(left < g.seg ? left : g.seg);
    const double c = rw_centre(g, in ? (int)threadIdx.x : 0, mine.x), d = c - c0;
    s = rw_wave_sum(in ? mine.x : 0.);
    q = in ? mine.y + 2. * d * (mine.x - n * c) + n * d * d : 0.;
  }
  q = rw_wave_sum(q);
  if ((threadIdx.x & 63) == 0)
    lds[threadIdx.x >> 6] = rw_pair{s, q};
  __syncthreads();
  s = q = 0.;
#pragma unroll
  for (int i = 0; i < kRwWaves; ++i) {
    s += lds[i].x;
    q += lds[i].y;
  }
  s *= g.inv;
  q *= g.inv;
  const float mean = (float)s;
  const double e = (double)mean - c0, around = q - 2. * e * (s - c0) + e * e;
  const float var = layer ? (around < 0. ? 0.f : (float)around) : (float)q;
  const float rstd = 1.0f / sqrtf(var + g.n.eps);
  if (g.n.emit_stats && blockIdx.x == 0 && threadIdx.x == 0)
    rw_stats(g.n, row, mean, rstd);
  if constexpr (NV > 0) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int64_t i = lo + (int64_t)(threadIdx.x + j * kRwThreads) * N;
      if (i >= hi)
        break;
      const int live = hi - i < N ? (int)(hi - i) : N;
      float v[N], sc[N], bi[N];
      V::widen(rx[j], v);
      if (own_s)
        V::widen(rs[j], sc);
      else if (g.n.scale)
        V::load_as(g.n.scale, g.n.scale_dt, i, live, sc);
      if (own_b)
        V::widen(rb[j], bi);
      else if (g.n.bias)
        V::load_as(g.n.bias, g.n.bias_dt, i, live, bi);
      rw_finish<T>(g.n, row, mean, rstd, i, live, v, sc, bi);
    }
  } else {
    rw_apply<T>(g.n, row, mean, rstd, lo, hi, threadIdx.x, kRwThreads);
  }
}

template <typename T> void rw_launch_split(hipStream_t stream, const RowWalkArgs &g, int64_t cus) {
  const dim3 grid((unsigned)g.splits, (unsigned)g.n.rows), wg(kRwThreads);
  if (g.n.is_layernorm)
    hipLaunchKernelGGL((rownorm_walk_sums_kernel<T, true>), grid, wg, 0, stream, g);
  else
    hipLaunchKernelGGL((rownorm_walk_sums_kernel<T, false>), grid, wg, 0, stream, g);
  // (RMSNorm has no bias to fetch ahead: walked segments are 2 to 8 % faster there, f16 28 x 229376
  // 12.4 us against 13.0, f32 22 x 195584 14.1 / 14.7; so are those of LayerNorm beyond four workgroups
  // per compute unit, which cover each other's waits: bf16 18 x 412672 13.9 / 15.8, 30 x 140288 10.4 / 11.1,
  // but f32 32 x 524288 35.4 / 34.3)
  if (g.seg <= 2 * kRwThreads * RwVec<T>::kN && g.n.is_layernorm && g.n.rows * g.splits <= 4 * cus)
    hipLaunchKernelGGL((rownorm_walk_apply_kernel<T, 2>), grid, wg, 0, stream, g);
  else
    hipLaunchKernelGGL((rownorm_walk_apply_kernel<T, 0>), grid, wg, 0, stream, g);
}

template <typename T> void rw_launch_rows(hipStream_t stream, const RowNormArgs &g, int waves) {
  const dim3 grid((unsigned)(waves == 1 ? (g.rows + 3) / 4 : g.rows)), wg(kRwThreads);
  if (waves == 1)
    hipLaunchKernelGGL((rownorm_walk_kernel<T, 1>), grid, wg, 0, stream, g, 1.0 / (double)g.inner);
  else
    hipLaunchKernelGGL((rownorm_walk_kernel<T, 4>), grid, wg, 0, stream, g, 1.0 / (double)g.inner);
}

} // namespace

// Segments that a row is cut into, 1: none.  Rows of more than four vectors per thread of a
// workgroup are cut into segments of two vectors per thread, 256 at most (a pair per thread of
// the second launch), unless whole ones, which take one launch and read X from memory once,
// keep up (us, whole / cut):
//   * more than sixteen rows (RMSNorm, which walks a row twice and not three times: four) per
//     compute unit: bf16 8000 x 16387 LayerNorm 196 / 204; RMSNorm bf16 3000 x 20001 63 / 65, f32
//     1200 x 30001 74 / 71, where many more walk as fast cut;
//   * LayerNorm in three segments, from 1.4 rows per unit on: f16 387 x 8818 10.6 / 11.7, bf16
//     1428 x 9324 19.1 / 24.7, f32 801 x 4463 9.9 / 13.4 (16 bits, 330 x 8510 11.5 / 10.2); in four, as
//     long as all rows run at once, eight workgroups to a unit: bf16 463 x 15564 15.7 / 14.8, 608 x 14156
//     16.3 / 17.3, 1381 x 12394 24.4 / 29.1, f32 1122 x 6187 17.7 / 21.2, 2234 x 6733 40.6 / 37.2; in five
//     854 x 17783 29.9 / 26.7;
//   * RMSNorm with more rows than two thirds of a unit's per segment: f32 671 x 4578 9.7 / 11.1, bf16
//     979 x 11162 15.9 / 17.6, 789 x 12434 16.3 / 17.4; but 543 x 13412 14.8 / 14.2, 713 x 19630 22.7 / 20.6.
// Segments' sums need the context's scratch.
int fhip_norm_walk_splits(fhip_ctx *ctx, int dtype, int64_t rows, int64_t inner, bool many_pay) {
  const int64_t vec = 16 / (int64_t)fhip_dtype_size(dtype);
  const int64_t cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  const int64_t unit = 2 * kRwThreads * vec;
  int64_t splits = (inner + unit - 1) / unit;
  splits = splits < kRwThreads ? splits : kRwThreads;
  const bool many = rows >= (many_pay ? 16 : 4) * cus && inner <= kRwResident * vec;
  const bool few = many_pay ? (splits == 3 && 10 * rows >= 14 * cus) ||
                                  (splits == 4 && 10 * rows >= 21 * cus && rows <= 8 * cus)
                            : 3 * rows >= 2 * cus * splits;
  if (inner <= 2 * unit || many || few || rows > 65535 ||
      !fhip_ctx_scratch_ready(ctx, (size_t)(2 * rows * splits) * sizeof(double)))
    return 1;
  return (int)splits;
}

// The caller (rownorm.hip) has checked that rows are dense and that X, OUT, scale,
// bias and the fused operands walk a row alike.
int fhip_norm_walk(fhip_ctx *ctx, int dtype, const RowNormArgs &n, bool cut_pays) {
  // A wavefront per row up to four vectors per lane, where the rows then still
  // fill half of the chip's wavefront slots or are shorter than two vectors per lane.
  const int64_t vec = 16 / (int64_t)fhip_dtype_size(dtype);
  const int waves = n.inner <= 128 * vec || (n.inner <= 256 * vec && n.rows >= 4096) ? 1 : 4;
  const int64_t splits = fhip_norm_walk_splits(ctx, dtype, n.rows, n.inner, cut_pays || n.is_layernorm);
  const bool cut = splits > 1;
  RowWalkArgs g{};
  if (cut) {
    g.seg = ((n.inner + splits - 1) / splits + vec - 1) / vec * vec;
    g.splits = (int32_t)((n.inner + g.seg - 1) / g.seg);
    void *scratch = nullptr;
    if (fhip_ctx_scratch(ctx, (size_t)(2 * n.rows * splits) * sizeof(double), &scratch) != 0)
      return 1;
    g.partial = (double *)scratch;
    g.inv = 1.0 / (double)n.inner;
    g.inv_seg = 1.0 / (double)g.seg;
    g.inv_last = 1.0 / (double)(n.inner - (g.splits - 1) * g.seg);
    g.n = n;
    fhip_note_kernel(ctx, "rownorm_walk segments=%d", g.splits);
  } else {
    fhip_note_kernel(ctx, "rownorm_walk waves_per_row=%d", waves);
  }
  auto go = [&](auto t) {
    typedef decltype(t) T;
    cut ? rw_launch_split<T>(ctx->stream, g, ctx->num_cus > 0 ? ctx->num_cus : 256) : rw_launch_rows<T>(ctx->stream, n, waves);
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

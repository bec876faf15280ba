// Bandwidth-bound keep-dim reductions of a dense tensor.  Over the trailing dims
// in memory order: X viewed as [rows, cols] -> Y[rows] (reduce_rows_kernel); with
// reduced dims in front of kept ones: ReduceMidArgs below.
//
// TPR lanes share a row (16, 64 or 256 by row length), each streaming 16-byte
// non-temporal loads into an f32 accumulator; the map (abs / square / zero->1)
// and the combine (add / mul / min / max) are compile-time, so the inner loop
// has no mode dispatch; lanes are combined with wavefront shuffles (+ one LDS
// hop for 256-lane rows).
//
// Reference semantics: node/reduction_node.h:47-56 (a dim is reduced where
// Y == 1 < X), support/asm_emitter.h:2165-2322 (SUM/ADD, MUL, MIN, MAX, AMAX,
// AVG, NORM1, NORM2, MUL_NO_ZEROS).
#include "common.h"
#include "fast_paths.h"

#include <type_traits>

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#define RF_AS1 __attribute__((address_space(1)))

enum { M_NONE = 0, M_ABS, M_SQUARE, M_ZERO_TO_ONE };
enum { C_ADD = 0, C_MUL, C_MIN, C_MAX };
enum { P_NONE = 0, P_MEAN, P_SQRT };

template <int MAP> __device__ __forceinline__ float rf_map(float v) {
  if constexpr (MAP == M_ABS)
    return fabsf(v);
  else if constexpr (MAP == M_SQUARE)
    return v * v;
  else if constexpr (MAP == M_ZERO_TO_ONE)
    return v == 0.f ? 1.f : v;
  else
    return v;
}

// min / max here ignore NaN (one instruction); NaN propagation (aten.amin /
// amax, and the generic kernel) is restored from `Acc::mag`, the largest
// |x| bit pattern seen: any NaN's pattern exceeds infinity's.
template <int COMB> __device__ __forceinline__ float rf_comb(float a, float b) {
  if constexpr (COMB == C_MUL)
    return a * b;
  else if constexpr (COMB == C_MIN)
    return fminf(a, b);
  else if constexpr (COMB == C_MAX)
    return fmaxf(a, b);
  else
    return a + b;
}

struct Acc {
  float v;      // running combine
  uint32_t mag; // min / max modes: largest magnitude bit pattern (f32 bits, or
                // two 16-bit patterns for the packed AMAX of 16-bit inputs)
};

template <int COMB> __device__ __forceinline__ float rf_identity() {
  if constexpr (COMB == C_MUL)
    return 1.f;
  else if constexpr (COMB == C_MIN)
    return INFINITY;
  else if constexpr (COMB == C_MAX)
    return -INFINITY;
  else
    return 0.f;
}

template <int MAP, int COMB> constexpr bool rf_is_amax() {
  return MAP == M_ABS && COMB == C_MAX;
}
template <int COMB> constexpr bool rf_tracks_nan() {
  return COMB == C_MIN || COMB == C_MAX;
}

template <typename T, int MAP, int COMB>
__device__ __forceinline__ void rf_chunk(const u32x4 v, Acc &a) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  if constexpr (rf_is_amax<MAP, COMB>()) {
    // max |x| on the bit patterns: unsigned compare orders magnitudes and
    // puts NaN above everything; 16-bit inputs two per instruction
    if constexpr (std::is_same<T, float>::value) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t m = w[i] & 0x7fffffffu;
        a.mag = a.mag > m ? a.mag : m;
      }
    } else {
      typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const u16x2 m = __builtin_bit_cast(u16x2, w[i] & 0x7fff7fffu);
        const u16x2 c = __builtin_bit_cast(u16x2, a.mag);
        a.mag = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(c, m));
      }
    }
  } else if constexpr (std::is_same<T, float>::value) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a.v = rf_comb<COMB>(a.v, rf_map<MAP>(__builtin_bit_cast(float, w[i])));
      if constexpr (rf_tracks_nan<COMB>()) {
        const uint32_t m = w[i] & 0x7fffffffu;
        a.mag = a.mag > m ? a.mag : m;
      }
    }
  } else {
    typedef T tx8 __attribute__((ext_vector_type(8)));
    const tx8 e = __builtin_bit_cast(tx8, v);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      a.v = rf_comb<COMB>(a.v, rf_map<MAP>((float)e[i]));
    if constexpr (rf_tracks_nan<COMB>()) {
      typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const u16x2 m = __builtin_bit_cast(u16x2, w[i] & 0x7fff7fffu);
        const u16x2 c = __builtin_bit_cast(u16x2, a.mag);
        a.mag = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(c, m));
      }
    }
  }
}

// Folds the two accumulators of a lane / two lanes; `mag` as 16-bit pairs for
// 16-bit inputs, as one f32 pattern otherwise.
template <typename T, int COMB>
__device__ __forceinline__ Acc rf_merge(const Acc &a, const Acc &b) {
  Acc r;
  r.v = rf_comb<COMB>(a.v, b.v);
  if constexpr (std::is_same<T, float>::value) {
    r.mag = a.mag > b.mag ? a.mag : b.mag;
  } else {
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    r.mag = __builtin_bit_cast(
        uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a.mag),
                                            __builtin_bit_cast(u16x2, b.mag)));
  }
  return r;
}

// Final value of a row from the merged accumulator.
template <typename T, int MAP, int COMB>
__device__ __forceinline__ float rf_finish(const Acc &a) {
  if constexpr (!rf_tracks_nan<COMB>()) {
    return a.v;
  } else {
    uint32_t mag; // as f32 bits
    if constexpr (std::is_same<T, float>::value) {
      mag = a.mag;
    } else {
      const uint32_t lo = a.mag & 0xffffu, hi = a.mag >> 16;
      const uint32_t m16 = lo > hi ? lo : hi;
      if constexpr (std::is_same<T, __bf16>::value) {
        mag = m16 << 16;
      } else {
        typedef _Float16 h1 __attribute__((ext_vector_type(1)));
        const unsigned short hs = (unsigned short)m16;
        mag = __builtin_bit_cast(uint32_t, (float)__builtin_bit_cast(_Float16, hs));
      }
    }
    const float magf = __builtin_bit_cast(float, mag);
    if (magf != magf)
      return magf; // a NaN was seen
    return rf_is_amax<MAP, COMB>() ? magf : a.v;
  }
}

struct ReduceRowsArgs {
  const char *x;
  void *y;
  int64_t rows;
  int64_t chunks; // 16-byte chunks per row
  int32_t y_dt, post;
  double inv_count; // mean: a product in 64 bits, exact for equal values (a division is longer code)
};

template <typename T, int MAP, int COMB, int TPR>
__global__ __launch_bounds__(256) void reduce_rows_kernel(ReduceRowsArgs g) {
  constexpr int RPW = 256 / TPR; // rows per workgroup
  const int lane = threadIdx.x % TPR;
  const int64_t row = (int64_t)blockIdx.x * RPW + threadIdx.x / TPR;
  const bool live = row < g.rows;
  const RF_AS1 u32x4 *src =
      (const RF_AS1 u32x4 *)(g.x) + (live ? row : 0) * g.chunks;
  // two accumulators: two independent loads in flight per lane
  Acc a0{rf_identity<COMB>(), 0u}, a1{rf_identity<COMB>(), 0u};
  int64_t c = lane;
  if (live) {
    for (; c + TPR < g.chunks; c += 2 * TPR) {
      const u32x4 v0 = __builtin_nontemporal_load(src + c);
      const u32x4 v1 = __builtin_nontemporal_load(src + c + TPR);
      rf_chunk<T, MAP, COMB>(v0, a0);
      rf_chunk<T, MAP, COMB>(v1, a1);
    }
    if (c < g.chunks)
      rf_chunk<T, MAP, COMB>(__builtin_nontemporal_load(src + c), a0);
  }
  Acc a = rf_merge<T, COMB>(a0, a1);
  // combine the lanes of a row (rows never straddle a wavefront for TPR <= 64)
  constexpr int WIDTH = TPR < 64 ? TPR : 64;
#pragma unroll
  for (int s = WIDTH / 2; s > 0; s >>= 1) {
    Acc o;
    o.v = __shfl_xor(a.v, s, 64);
    o.mag = (uint32_t)__shfl_xor((int)a.mag, s, 64);
    a = rf_merge<T, COMB>(a, o);
  }
  if constexpr (TPR == 256) {
    __shared__ float part_v[4];
    __shared__ uint32_t part_m[4];
    if ((threadIdx.x & 63) == 0) {
      part_v[threadIdx.x >> 6] = a.v;
      part_m[threadIdx.x >> 6] = a.mag;
    }
    __syncthreads();
    a = rf_merge<T, COMB>(
        rf_merge<T, COMB>(Acc{part_v[0], part_m[0]}, Acc{part_v[1], part_m[1]}),
        rf_merge<T, COMB>(Acc{part_v[2], part_m[2]}, Acc{part_v[3], part_m[3]}));
  }
  float acc = rf_finish<T, MAP, COMB>(a);
  if (lane == 0 && live) {
    if (g.post == P_MEAN)
      acc = (float)((double)acc * g.inv_count);
    else if (g.post == P_SQRT)
      acc = sqrtf(acc);
    if (g.y_dt == FHIP_FLOAT)
      ((RF_AS1 float *)g.y)[row] = acc;
    else if (g.y_dt == FHIP_BFLOAT16)
      ((RF_AS1 __bf16 *)g.y)[row] = (__bf16)acc;
    else
      ((RF_AS1 _Float16 *)g.y)[row] = (_Float16)acc;
  }
}

// Reductions that leave dims behind the reduced ones, X[r1][k][r2] -> Y[k]: the
// bias gradient of a convolution (channels-last: r2 = 1, otherwise r2 = H * W),
// column sums of a matrix.  The range of r1 (of r1 * r2 where r2 > 1) is cut into
// slices on workgroups of their own (partial[slice][k], f32), which a second kernel combines in slice
// order: no atomics.  Bound by reading X once.  N32 56 x 56 K128 bf16 in
// channels-last (25.7 MB): 104 us on the strided kernel (one workgroup per
// channel and slice reading one 2-byte element per pixel line) -> 8.4 -> 7.0 us
// (both launches); N100 K32 30 x 30 f32 channels-first (11.5 MB) 31 -> 10.2 us (5.5 +
// 4.6).
struct ReduceMidArgs {
  const char *x;
  void *y;
  float *partial; // null: one slice, the result goes to y
  int64_t r1, per_slice; // of a slice: rows (r2 == 1), vectors of the r1 * r2 range otherwise
  int32_t k, r2;         // r2: in vectors of the kernel's width
  uint32_t magic_r2;
  int32_t slices;
  int32_t y_dt, post;
  double inv_count; // mean: a product in 64 bits, exact for equal values (a division is longer code)
};

// NaN-propagating combine of two values (sums and products propagate by
// themselves; the others are one instruction each: bf16 [8, 7, 7] x 512 channels-last
// maxima 10.9 us with compares and selects)
template <int COMB> __device__ __forceinline__ float rf_comb_nan(float a, float b) {
  if constexpr (COMB == C_MIN)
    return __builtin_elementwise_minimum(a, b);
  else if constexpr (COMB == C_MAX)
    return __builtin_elementwise_maximum(a, b);
  else
    return rf_comb<COMB>(a, b);
}

// Running sums are held in f64, added to once per four f32 values: a thread's
// chain of f32 additions (hundreds of terms) was up to one and a half times as
// far from the exact sum as the strided kernel's 2048-element slices (bias gradient
// N32 K128 56 x 56 bf16: 8.0e-8 against 6.9e-8; N18 K32 39 x 39 f32 7.5e-8 there,
// 3.2e-8 now).  It costs no time: 8.5 us as before.
template <int COMB> struct RfRun {
  typedef float type;
};
template <> struct RfRun<C_ADD> {
  typedef double type;
};
template <int COMB, typename A> __device__ __forceinline__ A rf_run_comb(A a, A b) {
  if constexpr (COMB == C_ADD)
    return a + b;
  else
    return rf_comb_nan<COMB>(a, b);
}

__device__ __forceinline__ void rf_store(const ReduceMidArgs &g, int64_t i, float v) {
  if (g.post == P_MEAN)
    v = (float)((double)v * g.inv_count);
  else if (g.post == P_SQRT)
    v = sqrtf(v);
  if (g.y_dt == FHIP_FLOAT)
    ((RF_AS1 float *)g.y)[i] = v;
  else if (g.y_dt == FHIP_BFLOAT16)
    ((RF_AS1 __bf16 *)g.y)[i] = (__bf16)v;
  else
    ((RF_AS1 _Float16 *)g.y)[i] = (_Float16)v;
}

template <typename T, int VEC> struct RfVec {
  typedef T type __attribute__((ext_vector_type(VEC)));
};
template <typename T> struct RfVec<T, 1> {
  typedef T type;
};
template <typename T, int VEC>
__device__ __forceinline__ void rf_values(typename RfVec<T, VEC>::type v, float (&f)[VEC]) {
  if constexpr (VEC == 1) {
    f[0] = (float)v;
  } else {
#pragma unroll
    for (int i = 0; i < VEC; ++i)
      f[i] = (float)v[i];
  }
}

// r2 == 1: TX threads side by side on the columns (VEC each), 256 / TX rows at
// a time, for sums eight rows of loads in flight per thread: a workgroup per compute unit is
// bound by their latency (N32 56 x 56 K128 bf16, four rows 8.2 us, eight 6.9; more slices
// cost the combining launch what they save here: 512 of them 1.3 us more in all).
template <typename T, int MAP, int COMB, int VEC>
__global__ __launch_bounds__(256) void reduce_cols_kernel(ReduceMidArgs g, int tx_log2) {
  typedef typename RfVec<T, VEC>::type V;
  typedef typename RfRun<COMB>::type A;
  __shared__ A lds[256][VEC + 1];
  const int tx = 1 << tx_log2, ty = 256 >> tx_log2;
  const int c = blockIdx.x * tx + (threadIdx.x & (tx - 1)); // column vector
  const int row0 = threadIdx.x >> tx_log2;
  const int cols = g.k / VEC;
  const bool live = c < cols;
  const int64_t first = (int64_t)blockIdx.y * g.per_slice;
  const int64_t last = first + g.per_slice < g.r1 ? first + g.per_slice : g.r1;
  const RF_AS1 V *src = (const RF_AS1 V *)g.x + (live ? c : 0);
  A acc[VEC];
#pragma unroll
  for (int i = 0; i < VEC; ++i)
    acc[i] = rf_identity<COMB>();
  auto add = [&](V v) {
    float f[VEC];
    rf_values<T, VEC>(v, f);
#pragma unroll
    for (int i = 0; i < VEC; ++i)
      acc[i] = rf_run_comb<COMB, A>(acc[i], rf_map<MAP>(f[i]));
  };
  auto add4 = [&](V v0, V v1, V v2, V v3) {
    float f[4][VEC];
    rf_values<T, VEC>(v0, f[0]), rf_values<T, VEC>(v1, f[1]);
    rf_values<T, VEC>(v2, f[2]), rf_values<T, VEC>(v3, f[3]);
#pragma unroll
    for (int i = 0; i < VEC; ++i)
      acc[i] = rf_run_comb<COMB, A>(
          acc[i], rf_comb_nan<COMB>(rf_comb_nan<COMB>(rf_map<MAP>(f[0][i]), rf_map<MAP>(f[1][i])),
                                    rf_comb_nan<COMB>(rf_map<MAP>(f[2][i]), rf_map<MAP>(f[3][i]))));
  };
  int64_t r = first + row0;
  if constexpr (COMB == C_ADD)
    for (; r + 7 * ty < last; r += 8 * ty) {
      V v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        v[i] = src[(r + i * ty) * cols];
      add4(v[0], v[1], v[2], v[3]);
      add4(v[4], v[5], v[6], v[7]);
    }
  for (; r + 3 * ty < last; r += 4 * ty) {
    const V v0 = src[r * cols], v1 = src[(r + ty) * cols];
    const V v2 = src[(r + 2 * ty) * cols], v3 = src[(r + 3 * ty) * cols];
    if constexpr (COMB == C_ADD) {
      add4(v0, v1, v2, v3);
    } else {
      add(v0);
      add(v1);
      add(v2);
      add(v3);
    }
  }
  for (; r < last; r += ty)
    add(src[r * cols]);
#pragma unroll
  for (int i = 0; i < VEC; ++i)
    lds[threadIdx.x][i] = acc[i];
  for (int s = 128; s >= tx; s >>= 1) {
    __syncthreads();
    if ((int)threadIdx.x < s) {
#pragma unroll
      for (int i = 0; i < VEC; ++i)
        lds[threadIdx.x][i] = rf_run_comb<COMB, A>(lds[threadIdx.x][i], lds[threadIdx.x + s][i]);
    }
  }
  if ((int)threadIdx.x < tx && live) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      const float v = (float)lds[threadIdx.x][i];
      if (g.partial)
        g.partial[(int64_t)blockIdx.y * g.k + (int64_t)c * VEC + i] = v;
      else
        rf_store(g, (int64_t)c * VEC + i, v);
    }
  }
}

// r2 > 1: one k and one slice of the r1 * r2 range per workgroup, the range's runs of r2
// as one index.  (Without SLICED the range is whole: a million rows of 3 values are
// bound by what a workgroup does before its loop, 556 us against 616.)
template <typename T, int MAP, int COMB, int VEC, bool SLICED>
__global__ __launch_bounds__(256) void reduce_mid_kernel(ReduceMidArgs g) {
  typedef typename RfVec<T, VEC>::type V;
  typedef typename RfRun<COMB>::type A;
  __shared__ A part[4];
  uint32_t count = (uint32_t)g.per_slice, begin = 0; // < 2^31, < 2^24
  const RF_AS1 V *src = (const RF_AS1 V *)g.x + blockIdx.x * (int64_t)g.r2;
  if constexpr (SLICED) {
    const int64_t total = g.r1 * g.r2, first = (int64_t)blockIdx.y * g.per_slice;
    count = (uint32_t)(first + g.per_slice < total ? g.per_slice : total - first);
    const int64_t run0 = first / g.r2;
    begin = (uint32_t)(first - run0 * g.r2);
    src += run0 * g.k * g.r2;
  }
  const int64_t pitch = (int64_t)g.k * g.r2;
  A acc = rf_identity<COMB>();
  auto at = [&](uint32_t i) {
    if constexpr (SLICED)
      i += begin;
    uint32_t q = __umulhi(i, g.magic_r2); // (floor estimate: at most one too small)
    uint32_t rem = i - q * (uint32_t)g.r2;
    if (rem >= (uint32_t)g.r2)
      rem -= (uint32_t)g.r2, ++q;
    return src[(int64_t)q * pitch + rem];
  };
  auto add = [&](V v) {
    float f[VEC];
    rf_values<T, VEC>(v, f);
    if constexpr (COMB == C_ADD) { // a vector in pairs, then into the running sum
#pragma unroll
      for (int i = 0; i < VEC; ++i)
        f[i] = rf_map<MAP>(f[i]);
#pragma unroll
      for (int n = VEC / 2; n > 0; n >>= 1)
#pragma unroll
        for (int i = 0; i < n; ++i)
          f[i] += f[i + n];
      acc += f[0];
    } else {
#pragma unroll
      for (int i = 0; i < VEC; ++i)
        acc = rf_comb_nan<COMB>(acc, rf_map<MAP>(f[i]));
    }
  };
  constexpr uint32_t U = SLICED && VEC == 1 ? 8 : 4; // loads in flight per thread
  uint32_t i = threadIdx.x;
  for (; i + (U - 1) * 256 < count; i += U * 256) {
    V v[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u)
      v[u] = at(i + u * 256);
#pragma unroll
    for (uint32_t u = 0; u < U; ++u)
      add(v[u]);
  }
  for (; i < count; i += 256)
    add(at(i));
#pragma unroll
  for (int s = 32; s > 0; s >>= 1)
    acc = rf_run_comb<COMB, A>(acc, __shfl_xor(acc, s, 64));
  if ((threadIdx.x & 63) == 0)
    part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    const float v = (float)rf_run_comb<COMB, A>(rf_run_comb<COMB, A>(part[0], part[1]),
                                                rf_run_comb<COMB, A>(part[2], part[3]));
    if constexpr (SLICED)
      g.partial[(int64_t)blockIdx.y * g.k + blockIdx.x] = v;
    else
      rf_store(g, blockIdx.x, v);
  }
}

// Combines the slices: 2^cols_log2 columns per workgroup, the other threads of a column
// over its slices.
template <int COMB>
__global__ __launch_bounds__(256) void reduce_mid_finish_kernel(ReduceMidArgs g, int cols_log2) {
  typedef typename RfRun<COMB>::type A;
  __shared__ A lds[4][16];
  const int cols = 1 << cols_log2, per = 256 >> cols_log2; // (16 columns at most)
  const int cl = threadIdx.x & (cols - 1), sl = threadIdx.x >> cols_log2;
  const int64_t c = (int64_t)blockIdx.x * cols + cl;
  A acc = rf_identity<COMB>();
  if (c < g.k) {
    const RF_AS1 float *p = (const RF_AS1 float *)g.partial + c;
    fhip_for_parts<4>(
        sl, per, g.slices, [&](int s) { return p[(int64_t)s * g.k]; },
        [&](float v, bool in) { acc = in ? rf_run_comb<COMB, A>(acc, v) : acc; });
  }
  // (inside the wavefronts first: a barrier for every halving was 0.4 us slower)
  for (int s = 32; s >= cols; s >>= 1)
    acc = rf_run_comb<COMB, A>(acc, __shfl_xor(acc, s));
  if ((int)(threadIdx.x & 63) < cols)
    lds[threadIdx.x >> 6][cl] = acc;
  __syncthreads();
  if (sl == 0 && c < g.k)
    rf_store(g, c, (float)rf_run_comb<COMB, A>(rf_run_comb<COMB, A>(lds[0][cl], lds[1][cl]),
                                               rf_run_comb<COMB, A>(lds[2][cl], lds[3][cl])));
}

struct ReducePlan {
  bool ok = false;  // the row kernel takes it
  bool mid = false; // reduced dims in front of kept ones: the column kernels do
  int64_t rows = 0, cols = 0;
  int64_t r1 = 1, k = 1, r2 = 1;
  int map = M_NONE, comb = C_ADD, post = P_NONE;
};

ReducePlan make_plan(const fhip_reduce_desc *d) {
  ReducePlan p;
  const int xdt = d->x.dtype, ydt = d->y.dtype;
  auto f = [](int dt) {
    return dt == FHIP_FLOAT || dt == FHIP_BFLOAT16 || dt == FHIP_HALF;
  };
  if (!f(xdt) || !f(ydt))
    return p;
  // X's dims in memory order, outermost first (unit dims may sit anywhere);
  // both tensors dense in that order
  int order[FHIP_MAX_RANK], n = 0;
  for (int i = 0; i < d->x.rank; ++i)
    if (d->x.dim[i] != 1)
      order[n++] = i;
  for (int a = 1; a < n; ++a)
    for (int b = a; b > 0 && d->x.stride[order[b]] > d->x.stride[order[b - 1]]; --b) {
      const int t = order[b];
      order[b] = order[b - 1], order[b - 1] = t;
    }
  int64_t xs = 1, ys = 1;
  for (int a = n - 1; a >= 0; --a) {
    const int i = order[a];
    if (d->x.stride[i] != xs)
      return p;
    xs *= d->x.dim[i];
    if (d->y.dim[i] != 1) {
      if (d->y.stride[i] != ys)
        return p;
      ys *= d->y.dim[i];
    }
  }
  // runs of reduced (r1), kept (k) and reduced (r2) dims
  int stage = 0;
  for (int a = 0; a < n; ++a) {
    const int64_t dim = d->x.dim[order[a]];
    const bool reduced = d->y.dim[order[a]] == 1;
    if (reduced)
      stage == 0 ? p.r1 *= dim : p.r2 *= dim;
    else if (p.r2 != 1)
      return p;
    else
      p.k *= dim;
    if (!reduced)
      stage = 1;
  }
  if (stage == 0) // everything is reduced: one row
    p.r2 = p.r1, p.r1 = 1;
  switch (d->mode) {
  case FHIP_RED_ADD:
  case FHIP_RED_SUM:
    break;
  case FHIP_RED_MUL:
    p.comb = C_MUL;
    break;
  case FHIP_RED_MUL_NO_ZEROS:
    p.comb = C_MUL;
    p.map = M_ZERO_TO_ONE;
    break;
  case FHIP_RED_MIN:
    p.comb = C_MIN;
    break;
  case FHIP_RED_MAX:
    p.comb = C_MAX;
    break;
  case FHIP_RED_AMAX:
    p.comb = C_MAX;
    p.map = M_ABS;
    break;
  case FHIP_RED_AVG:
    p.post = P_MEAN;
    break;
  case FHIP_RED_NORM1:
    p.map = M_ABS;
    break;
  case FHIP_RED_NORM2:
    p.map = M_SQUARE;
    p.post = P_SQRT;
    break;
  default:
    return p;
  }
  p.rows = p.k;
  p.cols = p.r2;
  p.ok = p.r1 == 1 && p.cols >= 2 && (p.cols * fhip_dtype_size(xdt)) % 16 == 0 &&
         p.rows < (1ll << 31) * 16;
  p.mid = !p.ok && p.r1 * p.r2 >= 2 && p.k <= (1 << 24) && p.r2 < (1 << 24);
  return p;
}

// Slices of the reduced range and launches of the column kernels (see ReduceMidArgs):
// about four workgroups per compute unit over all columns, at least 2048 elements or
// eight rounds of rows (r2 == 1) each, at most 1024 (256 of more than 16 results: the
// combining kernel reads slices * k values).
//
// Slices of r1 alone left [2, 3, 1024, 1024] f32 -> 3 sums to six workgroups (59.5 us on
// the strided kernel, 74 so) and a sum of 10 000 001 values to one (88 -> 3670 us).
template <typename T, int MAP, int COMB>
int launch_mid(fhip_ctx *ctx, const ReducePlan &p, ReduceMidArgs g) {
  constexpr int VEC = 16 / (int)sizeof(T);
  const bool cols = p.r2 == 1;
  const bool vec = ((uintptr_t)g.x & 15) == 0 && (cols ? p.k % VEC == 0 : p.r2 % VEC == 0);
  int tx_log2 = 0;
  int64_t groups = p.k, most, range = p.r1;
  if (cols) {
    const int64_t cv = vec ? p.k / VEC : p.k;
    while ((1ll << tx_log2) < cv && tx_log2 < 8)
      ++tx_log2;
    most = p.r1 / ((256 >> tx_log2) * 8);
    // Few rows: one slice, and one launch, on narrow workgroups (eight vectors at least,
    // four rows per thread) unless there are 512 wide ones ([64, 2048] bf16 maxima: strided
    // 6.7 us, eight slices 8.4; [8, 7, 7] x 512 sums 6.7, so 4.4).  Beyond 512 rows the few
    // workgroups wait for memory where X is not in a cache: 1024 x 80 in a training step
    // that takes 31.0 us with slices, 33.2 in one; 950 x 256, 55.7 and 57.2.
    if (p.r1 <= 512) {
      while (tx_log2 > 3 && (cv >> tx_log2) < 512 && (512 >> tx_log2) * 4 <= p.r1)
        --tx_log2;
      most = 1;
    }
    groups = (cv + (1ll << tx_log2) - 1) >> tx_log2;
  } else {
    g.r2 = (int32_t)(vec ? p.r2 / VEC : p.r2);
    g.magic_r2 = g.r2 == 1 ? 0xffffffffu : (uint32_t)((1ull << 32) / (uint32_t)g.r2);
    most = p.r1 * p.r2 / 2048;
    range = p.r1 * g.r2;
  }
  int64_t slices = 4 * (int64_t)(ctx->num_cus > 0 ? ctx->num_cus : 256) / groups;
  slices = slices < most ? slices : most;
  const int64_t cap = p.k <= 16 ? 1024 : 256;
  slices = slices < cap ? slices : cap;
  // (a slice's flat index is 32-bit)
  const int64_t least = range / (1ll << 30) + 1;
  slices = slices > least ? slices : least;
  if (slices > 1 && !fhip_ctx_scratch_ready(ctx, (size_t)(slices * p.k) * sizeof(float)))
    slices = least; // (usually one: no scratch)
  g.per_slice = (range + slices - 1) / slices;
  slices = (range + g.per_slice - 1) / g.per_slice;
  if (slices > 65535 || g.per_slice >= (1ll << 31))
    return -1; // (the strided kernel's)
  g.slices = (int32_t)slices;
  if (slices > 1) {
    const size_t bytes = (size_t)(slices * p.k) * sizeof(float);
    void *sp = nullptr;
    if (!fhip_ctx_scratch_ready(ctx, bytes))
      return -1;
    if (fhip_ctx_scratch(ctx, bytes, &sp) != 0)
      return 1;
    g.partial = (float *)sp;
  }
  fhip_note_kernel(ctx, cols ? "reduce_cols slices=%d" : "reduce_mid slices=%d", (int)slices);
  const dim3 grid((unsigned)groups, (unsigned)slices);
  if (cols && vec)
    hipLaunchKernelGGL((reduce_cols_kernel<T, MAP, COMB, VEC>), grid, dim3(256), 0, ctx->stream, g, tx_log2);
  else if (cols)
    hipLaunchKernelGGL((reduce_cols_kernel<T, MAP, COMB, 1>), grid, dim3(256), 0, ctx->stream, g, tx_log2);
  else {
    auto kernel = slices > 1 ? (vec ? reduce_mid_kernel<T, MAP, COMB, VEC, true>
                                    : reduce_mid_kernel<T, MAP, COMB, 1, true>)
                             : (vec ? reduce_mid_kernel<T, MAP, COMB, VEC, false>
                                    : reduce_mid_kernel<T, MAP, COMB, 1, false>);
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, ctx->stream, g);
  }
  if (slices > 1) {
    int cols_log2 = 0;
    while ((1 << cols_log2) < p.k && cols_log2 < 4)
      ++cols_log2;
    hipLaunchKernelGGL(reduce_mid_finish_kernel<COMB>,
                       dim3((unsigned)((p.k + (1ll << cols_log2) - 1) >> cols_log2)), dim3(256), 0,
                       ctx->stream, g, cols_log2);
  }
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  return 0;
}

template <typename T, int MAP, int COMB>
int launch_tpr(fhip_ctx *ctx, const ReduceRowsArgs &g) {
  const int64_t row_bytes = g.chunks * 16;
  if (row_bytes >= 4096) {
    hipLaunchKernelGGL((reduce_rows_kernel<T, MAP, COMB, 256>),
                       dim3((unsigned)g.rows), dim3(256), 0, ctx->stream, g);
  } else if (row_bytes >= 512) {
    hipLaunchKernelGGL((reduce_rows_kernel<T, MAP, COMB, 64>),
                       dim3((unsigned)((g.rows + 3) / 4)), dim3(256), 0,
                       ctx->stream, g);
  } else {
    hipLaunchKernelGGL((reduce_rows_kernel<T, MAP, COMB, 16>),
                       dim3((unsigned)((g.rows + 15) / 16)), dim3(256), 0,
                       ctx->stream, g);
  }
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  return 0;
}

// The amax of |x| starts from 0, the others from their combine's identity;
// only these (map, combine) pairs occur.
template <typename F> int for_mode(const ReducePlan &p, F &&run) {
  using std::integral_constant;
  auto go = [&](auto map, auto comb) { return run(map, comb); };
  if (p.comb == C_ADD && p.map == M_NONE)
    return go(integral_constant<int, M_NONE>{}, integral_constant<int, C_ADD>{});
  if (p.comb == C_ADD && p.map == M_ABS)
    return go(integral_constant<int, M_ABS>{}, integral_constant<int, C_ADD>{});
  if (p.comb == C_ADD && p.map == M_SQUARE)
    return go(integral_constant<int, M_SQUARE>{}, integral_constant<int, C_ADD>{});
  if (p.comb == C_MUL && p.map == M_NONE)
    return go(integral_constant<int, M_NONE>{}, integral_constant<int, C_MUL>{});
  if (p.comb == C_MUL && p.map == M_ZERO_TO_ONE)
    return go(integral_constant<int, M_ZERO_TO_ONE>{}, integral_constant<int, C_MUL>{});
  if (p.comb == C_MIN)
    return go(integral_constant<int, M_NONE>{}, integral_constant<int, C_MIN>{});
  if (p.comb == C_MAX && p.map == M_ABS)
    return go(integral_constant<int, M_ABS>{}, integral_constant<int, C_MAX>{});
  return go(integral_constant<int, M_NONE>{}, integral_constant<int, C_MAX>{});
}

template <typename T>
int launch_mode(fhip_ctx *ctx, const ReducePlan &p, const ReduceRowsArgs &g) {
  return for_mode(p, [&](auto map, auto comb) {
    return launch_tpr<T, decltype(map)::value, decltype(comb)::value>(ctx, g);
  });
}

template <typename T>
int launch_mid_mode(fhip_ctx *ctx, const ReducePlan &p, const ReduceMidArgs &g) {
  return for_mode(p, [&](auto map, auto comb) {
    return launch_mid<T, decltype(map)::value, decltype(comb)::value>(ctx, p, g);
  });
}

} // namespace

bool fhip_fast_reduce_applicable(const fhip_reduce_desc *d) {
  return make_plan(d).ok;
}

int fhip_mid_reduce(fhip_ctx *ctx, const fhip_reduce_desc *d, const void *x, void *y,
                    bool *handled) {
  *handled = false;
  const ReducePlan p = make_plan(d);
  if (!p.mid)
    return 0;
  ReduceMidArgs g{};
  g.x = (const char *)x;
  g.y = y;
  g.r1 = p.r1;
  g.k = (int32_t)p.k;
  g.r2 = (int32_t)p.r2;
  g.y_dt = d->y.dtype;
  g.post = p.post;
  g.inv_count = 1.0 / (double)(p.r1 * p.r2);
  const int rc = d->x.dtype == FHIP_FLOAT      ? launch_mid_mode<float>(ctx, p, g)
                 : d->x.dtype == FHIP_BFLOAT16 ? launch_mid_mode<__bf16>(ctx, p, g)
                                               : launch_mid_mode<_Float16>(ctx, p, g);
  if (rc < 0)
    return 0;
  *handled = true;
  return rc;
}

int fhip_fast_reduce(fhip_ctx *ctx, const fhip_reduce_desc *d, const void *x,
                     void *y) {
  const ReducePlan p = make_plan(d);
  FHIP_REQUIRE(ctx, p.ok, "reduce: descriptor not supported by the row kernel");
  FHIP_REQUIRE(ctx, ((uintptr_t)x & 15) == 0, "reduce: X must be 16-byte aligned");
  ReduceRowsArgs g{};
  g.x = (const char *)x;
  g.y = y;
  g.rows = p.rows;
  g.chunks = p.cols * fhip_dtype_size(d->x.dtype) / 16;
  g.y_dt = d->y.dtype;
  g.post = p.post;
  g.inv_count = 1.0 / (double)p.cols;
  fhip_note_kernel(ctx, "reduce_rows");
  switch (d->x.dtype) {
  case FHIP_FLOAT:
    return launch_mode<float>(ctx, p, g);
  case FHIP_BFLOAT16:
    return launch_mode<__bf16>(ctx, p, g);
  default:
    return launch_mode<_Float16>(ctx, p, g);
  }
}

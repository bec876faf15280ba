// Convolutions over few input channels (the first layer of a network): one group,
// two spatial dims, channels-first tensors, at most 112 (channel, tap) pairs.
//
// Bound by reading and writing the many-channel tensor once; the direct kernels
// (conv_direct.hip) kept one pixel per thread and fetched every X or DY value from
// the caches once per tap and channel block.  All sums are f32; 16-bit tensors are widened when
// they are staged, but in the products of the data gradient, where the MFMA does that.
//   * forward: X of 256 output pixels, padded with zeros, and the filter sit in LDS;
//     pixels x output channels on 16 x 16 x 4 f32 MFMAs over the (channel, tap) pairs.
//     A wavefront's four tiles interleave their pixels so that a lane ends up with 16
//     consecutive pixels of one channel (16-bit OUT) or four runs that its neighbours continue;
//   * weight gradient: output channels x pairs on the same MFMAs over the pixels, DY
//     straight from memory (four consecutive pixels per lane), X from LDS; a
//     workgroup keeps its sums over many bands of rows, the workgroups' sums meet in
//     the context's scratch and are added in a fixed order;
//   * data gradient: products first (pairs x pixels of DY on the MFMAs, summed over the
//     output channels), then the taps of a DX pixel are added in LDS.  Where that takes
//     several passes over the input channels and does not pay, a lane computes 4 x 2 pixels x
//     all channels with vector instructions, the wavefronts of a workgroup each over a
//     share of the output channels, whose DY rows they stage for themselves; the shares are
//     added through LDS.
//
// One training step (us):
//   N100 3 -> 32, 32 x 32, 3 x 3, f32: fprop 26.2 -> 13.6 -> 12.0, dgrad 60.5 -> 15.0 -> 11.1, wgrad 46.1 -> 13.0
//   N122 1 -> 64, 57 x 57, 5 x 5, bf16: 136 -> 52.6, 701 -> 78.6 -> 33.0, 495 -> 45.7
// With elements found by steps, and quotients of uniform values in scalar multiplications, 36 random
// layers (sums of traced us): fprop 420.8 -> 398.4, dgrad 294.8 -> 287.2, wgrad 314.0 -> 296.
//
// Reference semantics: aten.convolution / aten.convolution_backward
// (reference support/asm_emitter.h:690-701, 868-873, 1030-1035).
#include "common.h"
#include "fast_paths.h"

#include <type_traits>

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kCfThreads = 256;
constexpr int kCfLds = 64 * 1024;
constexpr int kCfDgradLds = 160 * 1024;
constexpr int kCfMaxPairs = 112;

struct CfArgs {
  int32_t N, C, H, W, K, P, Q, R, S, J; // J = C * R * S
  int32_t pad_h, pad_w, str_h, str_w, dil_h, dil_w;
  int64_t xs[4], ws[4], ys[4]; // element strides; ys: Y (gradients) or OUT (forward)
  int32_t y_dt, o_dt;          // forward: rounding of the sum, type of OUT
  int32_t lw;                  // columns of the staged X
  uint32_t lw_magic, rows_magic, q_magic, rs_magic, s_magic;
  int32_t xrows;               // most rows of X staged at once
  int32_t col_step, row_step, c_step; // kCfThreads elements of the staged X
  int32_t tiles;               // forward: workgroups per image; gradients: bands
  int32_t band;                // output (data gradient: input) rows per band
  int32_t quads;               // data gradient: runs of 4 pixels per row,
  int32_t wt;                  // products: columns per band,
  int32_t cb, wpitch, gat, gpitch; // channels per pass, pitch of the filter, where G starts, pitch of a row in G
  int32_t packed;              // the filter of an output channel without gaps, in this order
  uint32_t w_magic, quads_magic, tiles_whole, q_whole;
  DevEpilogue epi;
};

// e / d for e, d < 2^16 with magic = 2^32 / d + 1 (0 stands for d = 1)
uint32_t cf_magic(int d) { return d == 1 ? 0u : (uint32_t)((1ull << 32) / (uint32_t)d + 1); }
__device__ __forceinline__ int cf_div(int e, uint32_t magic) {
  return (int)__umulhi((uint32_t)e, magic) + (magic == 0 ? e : 0);
}

// e / d of uniform values, any e >= 0, whole = (2^32 - 1) / d: a quotient at most one too small, in
// scalar multiplications (a division is some 30 dependent vector operations)
__device__ __forceinline__ int cf_div_uniform(int e, int d, uint32_t whole, int *rest) {
  int q = (int)__umulhi((uint32_t)e, whole);
  int r = e - q * d;
  if (r >= d)
    ++q, r -= d;
  *rest = r;
  return q;
}

// X rows [row0, row0 + rows) of all channels of an image, zeros outside it, as f32, in batches:
// request() issues a batch's loads, put() waits for them.  A thread steps from element to element:
// the first loads wait for what it takes to find them (multiplications of 32 bits are four times as
// long as additions).  TRIM: no loads behind the last element; in the loop over the bands of a weight
// gradient with much else in it the branches cost more (f32 N119 3 -> 64, 58 x 58 33.7 us without, 35.5
// with, one band each N38 3 -> 64, 24 x 24 6.4 and 6.1).
template <typename T, bool TRIM = true> struct CfStageX {
  static constexpr int kBatch = 8; // loads in flight per thread
  T v[kBatch];
  // where in an image a load goes, less its first row, and its row there, two to a register, 2^16 - 1
  // where it is in no column of the image
  uint32_t at[kBatch];
  uint32_t row[kBatch / 2];
  uint32_t live;
  // elements e0 + threadIdx.x + i * kCfThreads
  __device__ __forceinline__ void find(const CfArgs &g, int e0) {
    const int total = g.C * g.xrows * g.lw, e = e0 + (int)threadIdx.x;
    const int cr = cf_div(e, g.lw_magic);
    int c = cf_div(cr, g.rows_magic), r = cr - c * g.xrows, w = e - cr * g.lw - g.pad_w;
    const uint32_t sc = (uint32_t)g.xs[1], sr = (uint32_t)g.xs[2];
    uint32_t p = (uint32_t)c * sc + (uint32_t)r * sr + (uint32_t)w;
    const uint32_t step = (uint32_t)g.c_step * sc + (uint32_t)g.row_step * sr + (uint32_t)g.col_step;
    const uint32_t next_row = sr - (uint32_t)g.lw, next_c = sc - (uint32_t)g.xrows * sr;
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      if (TRIM && e0 + i * kCfThreads >= total) // (uniform)
        break;
      at[i] = p;
      const uint32_t mine = c < g.C && (unsigned)w < (unsigned)g.W ? (uint32_t)r : 0xffffu;
      row[i / 2] = i & 1 ? row[i / 2] | mine << 16 : mine;
      w += g.col_step, r += g.row_step, c += g.c_step, p += step;
      if (w >= g.lw - g.pad_w)
        w -= g.lw, ++r, p += next_row;
      if (r >= g.xrows)
        r -= g.xrows, ++c, p += next_c;
    }
  }
  __device__ __forceinline__ void request(const CfArgs &g, const T *x, int row0, int rows, int e0) {
    const int total = g.C * g.xrows * g.lw;
    const int r0 = row0 < 0 ? -row0 : 0, r1 = g.H - row0 < rows ? g.H - row0 : rows; // rows of the image
    const uint32_t add = (uint32_t)row0 * (uint32_t)g.xs[2];
    live = 0;
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      if (TRIM && e0 + i * kCfThreads >= total)
        break;
      const int r = (int)(i & 1 ? row[i / 2] >> 16 : row[i / 2] & 0xffffu);
      const bool in = r >= r0 && r < r1;
      // (the load is issued either way: a branch would wait for every value)
      v[i] = x[in ? at[i] + add : 0u];
      live |= (uint32_t)in << i;
    }
  }
  __device__ __forceinline__ void put(const CfArgs &g, int e0, float *xl) const {
    const int total = g.C * g.xrows * g.lw;
    float *to = xl + e0 + threadIdx.x;
#pragma unroll
    for (int i = 0; i < kBatch; ++i)
      if (e0 + i * kCfThreads + (int)threadIdx.x < total)
        to[i * kCfThreads] = (live >> i) & 1 ? (float)v[i] : 0.f;
  }
  // all batches from `e0` on
  static __device__ __forceinline__ void stage(const CfArgs &g, const T *x, int row0, int rows, int e0, float *xl) {
    for (; e0 < g.C * g.xrows * g.lw; e0 += kBatch * kCfThreads) {
      CfStageX b;
      b.find(g, e0);
      b.request(g, x, row0, rows, e0);
      b.put(g, e0, xl);
    }
  }
};

// where pair j = (channel, tap) lies in the staged X / in the filter
__device__ __forceinline__ int cf_pair(const CfArgs &g, int j, int *filter) {
  const int c = cf_div(j, g.rs_magic), t = j - c * g.R * g.S;
  const int r = cf_div(t, g.s_magic), s = t - r * g.S;
  *filter = c * (int)g.ws[1] + r * (int)g.ws[2] + s * (int)g.ws[3];
  return (c * g.xrows + r * g.dil_h) * g.lw + s * g.dil_w;
}

// ---- forward -------------------------------------------------------------------
// 16 values, four at a time TS elements apart
template <typename O, int TS>
__device__ __forceinline__ void cf_store16(void *out, int64_t at, const float (&v)[16]) {
  constexpr int N = 16 / sizeof(O);
  typedef O vec __attribute__((ext_vector_type(N), aligned(sizeof(O))));
#pragma unroll
  for (int i = 0; i < 16; i += N) {
    vec t;
#pragma unroll
    for (int k = 0; k < N; ++k)
      t[k] = (O)v[i + k];
    *(vec *)((O *)out + at + (i >> 2) * TS) = t;
  }
}

template <typename T, int KT>
__global__ __launch_bounds__(kCfThreads) void conv_few_fprop_kernel(CfArgs g, const T *x,
                                                                    const T *w, void *out) {
  constexpr int KP = KT * 16 + (KT % 2 ? 0 : 16); // (two rows of pairs in different banks)
  constexpr int K16 = KT * 16;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int j4 = (g.J + 3) & ~3;
  float *wl = smem;                            // [pair][output channel]
  float *ops = wl + j4 * KP;                   // [fused operation][output channel]
  int *tab = (int *)(ops + FHIP_MAX_EPILOGUE * K16); // where a pair's X lies
  float *xl = (float *)(tab + j4);
  const int tid = threadIdx.x, l = tid & 63, wave = tid >> 6;
  const int k0 = blockIdx.z * K16, n = blockIdx.y, t0 = blockIdx.x * kCfThreads;
  const int pq = g.P * g.Q;
  const int t1 = t0 + kCfThreads < pq ? t0 + kCfThreads : pq;
  int q0; // (column of the first pixel)
  const int p0 = cf_div_uniform(t0, g.Q, g.q_whole, &q0), p1 = p0 + cf_div(q0 + t1 - 1 - t0, g.q_magic);
  // Everything a workgroup reads is requested before the first wait: X, the filter, then the
  // fused operations' values per channel.  Nothing looks at a loaded value before that, not
  // even a select (f32 N22 1 -> 16, 28 x 28, 3 x 3 7.3 -> 6.8 us, bf16 N71 1 -> 32, 17 x 17, 5 x 5 9.1 -> 8.3).
  const int row0 = p0 * g.str_h - g.pad_h, xrows = (p1 - p0) * g.str_h + (g.R - 1) * g.dil_h + 1;
  CfStageX<T> xv0;
  xv0.find(g, 0);
  xv0.request(g, x + n * g.xs[0], row0, xrows, 0);
  constexpr int kBatch = 8;
  const int kk = tid % K16, jt = tid / K16; // this thread's channel, its first pair
  const bool k_in = k0 + kk < g.K;
  const T *wk = w + (k_in ? k0 + kk : k0) * g.ws[0];
  // (as many loads as there are pairs, up to a batch; those behind the last pair read the first)
  auto weights = [&](int j0, T (&v)[kBatch]) {
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      if (j0 - jt + i * (kCfThreads / K16) >= j4) // (uniform)
        break;
      int j = j0 + i * (kCfThreads / K16);
      j = j < g.J ? j : 0;
      if (!g.packed)
        cf_pair(g, j, &j);
      v[i] = wk[j];
    }
  };
  auto put_weights = [&](int j0, const T (&v)[kBatch]) {
#pragma unroll
    for (int i = 0; i < kBatch; ++i) {
      const int j = j0 + i * (kCfThreads / K16);
      if (j < j4)
        wl[j * KP + kk] = j < g.J && k_in ? (float)v[i] : 0.f;
    }
  };
  T wv0[kBatch];
  float op[FHIP_MAX_EPILOGUE];
  weights(jt, wv0);
#pragma unroll
  for (int e = 0; e < FHIP_MAX_EPILOGUE; ++e) {
    op[e] = 0.f;
    if (e < g.epi.count && g.epi.op[e].kind != FHIP_OPERAND_NONE) { // (uniform)
      const DevEpiOp &o = g.epi.op[e];
      op[e] = o.kind == FHIP_OPERAND_SCALAR
                  ? o.scalar
                  : fhip_load<float>(o.ptr, o.operand_dtype,
                                     n * o.stride[0] + (k_in ? k0 + kk : g.K - 1) * o.stride[1]);
    }
  }
  for (int j = tid; j < j4; j += kCfThreads) {
    int f;
    tab[j] = j < g.J ? cf_pair(g, j, &f) : 0;
  }
  xv0.put(g, 0, xl);
  CfStageX<T>::stage(g, x + n * g.xs[0], row0, xrows, CfStageX<T>::kBatch * kCfThreads, xl);
  put_weights(jt, wv0);
  for (int j0 = jt + kBatch * (kCfThreads / K16); j0 < j4; j0 += kBatch * (kCfThreads / K16)) {
    T v[kBatch];
    weights(j0, v);
    put_weights(j0, v);
  }
  if (tid < K16)
#pragma unroll
    for (int e = 0; e < FHIP_MAX_EPILOGUE; ++e)
      ops[e * K16 + tid] = op[e];
  __syncthreads();
  const int first = t0 + wave * 64;
  if (first >= t1)
    return;
  // Pixels of the four tiles: a lane ends up with 16 in a row where OUT has 16-bit elements
  // (two whole stores), else with runs of 4 that its neighbours continue (64 bytes a channel
  // and store, not 16 bytes each on 32 cache lines: N67 4 -> 32, 62 x 62, 3 x 3 27.2 -> 23.0 us, N60 1 -> 64, 40 x 40
  // 15.8 -> 13.1).
  const int ts = g.o_dt == FHIP_FLOAT ? 16 : 4, gs = 20 - ts;
  int base[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int m = l & 15;
    int px = first + (m >> 2) * gs + t * ts + (m & 3);
    // (row p and column i - p * Q behind p0's start)
    const int i = (px < t1 ? px : t1 - 1) - t0 + q0;
    base[t] = __mul24(i, g.str_w) + __mul24(cf_div(i, g.q_magic), g.str_h * g.lw - g.Q * g.str_w);
  }
  f32x4 acc[4][KT];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int u = 0; u < KT; ++u)
      acc[t][u] = f32x4{0, 0, 0, 0};
  int next = tab[l >> 4];
  for (int j = l >> 4; j < j4; j += 4) {
    const int off = next;
    next = tab[j + 4 < j4 ? j + 4 : j];
    float xv[4], wv[KT];
#pragma unroll
    for (int u = 0; u < KT; ++u)
      wv[u] = wl[j * KP + u * 16 + (l & 15)];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      xv[t] = xl[base[t] + off];
      xv[t] = j < g.J ? xv[t] : 0.f; // (0 x infinity)
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int u = 0; u < KT; ++u)
        acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[t], wv[u], acc[t][u], 0, 0, 0);
  }
  // value r of tile t: pixel first + (l / 16) * gs + t * ts + r of channel l % 16
  const int px = first + (l >> 4) * gs;
  if (px >= t1)
    return;
  // (one copy of the chain for all KT tiles: the next tile's sums move to the front)
#pragma clang loop unroll(disable)
  for (int u = 0; u < KT; ++u) {
    const int k = k0 + u * 16 + (l & 15);
    float v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i)
      v[i] = acc[i >> 2][0][i & 3];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i + 1 < KT; ++i)
        acc[t][i] = acc[t][i + 1];
    if (k >= g.K)
      continue;
    fhip_round_fast_vec<16>(g.y_dt, v);
    for (int e = 0; e < g.epi.count; ++e) {
      const DevEpiOp &o = g.epi.op[e];
      if (o.kind == FHIP_OPERAND_NONE) {
        fhip_pw_fast_unary_vec<true, 16>(o.mode, v, o.params.swish_beta,
                                         o.result_dtype != FHIP_FLOAT);
      } else {
        const float s = ops[e * K16 + u * 16 + (l & 15)];
        float other[16];
#pragma unroll
        for (int i = 0; i < 16; ++i)
          other[i] = s;
        fhip_pw_fast_binary_vec<16>(o.mode, o.acc_is_in1 != 0, v, other);
      }
      fhip_round_fast_vec<16>(o.result_dtype, v);
    }
    const int64_t at = n * g.ys[0] + k * g.ys[1] + px;
    if (px + 3 * ts + 4 <= t1) {
      if (g.o_dt == FHIP_FLOAT)
        cf_store16<float, 16>(out, at, v);
      else if (g.o_dt == FHIP_BFLOAT16)
        cf_store16<__bf16, 4>(out, at, v);
      else
        cf_store16<_Float16, 4>(out, at, v);
    } else if (g.o_dt == FHIP_FLOAT) {
      typedef float Four __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
      for (int i = 0; i < 16; i += 4) {
        float *to = (float *)out + at + 4 * i;
        const int left = t1 - (px + 4 * i);
        if (left >= 4) {
          *(Four *)to = Four{v[i], v[i + 1], v[i + 2], v[i + 3]};
        } else {
#pragma unroll
          for (int j = 0; j < 3; ++j)
            if (j < left)
              to[j] = v[i + j];
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (px + i < t1)
          fhip_store<float>(out, g.o_dt, at + i, v[i]);
    }
  }
}

// ---- weight gradient -----------------------------------------------------------
template <typename T, int KT>
__device__ __forceinline__ void cf_load_dy(const T *const (&dy)[KT], int px, int np,
                                           float (&a)[KT][4]) {
  typedef T vec __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  if (px + 4 <= np) {
#pragma unroll
    for (int u = 0; u < KT; ++u) {
      const vec v = *(const vec *)(dy[u] + px);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        a[u][i] = (float)v[i];
    }
  } else {
#pragma unroll
    for (int u = 0; u < KT; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float t = (float)dy[u][px + i < np ? px + i : 0];
        a[u][i] = px + i < np ? t : 0.f;
      }
  }
}

// partial[run][k block][KT * JT tiles][4][64]: the fragments as they lie
template <typename T, int KT, int JT>
__global__ __launch_bounds__(kCfThreads) void conv_few_wgrad_kernel(CfArgs g, const T *dy,
                                                                    const T *x, float *partial) {
  constexpr int kFrag = KT * JT * 256;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  int *pixtab = (int *)smem; // where a band's pixel lies in the staged X
  const int slots = (g.band * g.Q + 15) & ~15;
  float *xl = smem + slots;
  const int tid = threadIdx.x, l = tid & 63, wave = tid >> 6;
  const int k0 = blockIdx.y * KT * 16;
  for (int i = tid; i < slots; i += kCfThreads) {
    const int p = cf_div(i, g.q_magic), q = i - p * g.Q;
    pixtab[i] = i < g.band * g.Q ? p * g.str_h * g.lw + q * g.str_w : 0;
  }
  int joff[JT];
#pragma unroll
  for (int u = 0; u < JT; ++u) {
    const int j = u * 16 + (l & 15);
    int f;
    joff[u] = j < g.J ? cf_pair(g, j, &f) : 0;
  }
  f32x4 acc[KT][JT];
#pragma unroll
  for (int u = 0; u < KT; ++u)
#pragma unroll
    for (int v = 0; v < JT; ++v)
      acc[u][v] = f32x4{0, 0, 0, 0};
  CfStageX<T, (KT <= 2 && JT <= 3)> xs; // (the same elements of every band)
  xs.find(g, 0);
  const int items = g.N * g.tiles;
  for (int item = blockIdx.x; item < items; item += gridDim.x) {
    int p0;
    const int n = cf_div_uniform(item, g.tiles, g.tiles_whole, &p0);
    p0 *= g.band;
    const int rows = g.P - p0 < g.band ? g.P - p0 : g.band;
    const int np = rows * g.Q;
    const T *src[KT];
#pragma unroll
    for (int u = 0; u < KT; ++u) {
      const int k = k0 + u * 16 + (l & 15);
      src[u] = dy + n * g.ys[0] + (k < g.K ? k : g.K - 1) * g.ys[1] + (int64_t)p0 * g.Q;
    }
    float a[2][KT][4];
    const int px0 = wave * 16 + (l >> 4) * 4;
    cf_load_dy<T, KT>(src, px0, np, a[0]);
    const int row0 = p0 * g.str_h - g.pad_h, xrows = (rows - 1) * g.str_h + (g.R - 1) * g.dil_h + 1;
    xs.request(g, x + n * g.xs[0], row0, xrows, 0);
    __syncthreads();
    xs.put(g, 0, xl);
    CfStageX<T>::stage(g, x + n * g.xs[0], row0, xrows, CfStageX<T>::kBatch * kCfThreads, xl);
    __syncthreads();
    auto spend = [&](const float (&b)[KT][4], int px) {
      const int4 at = *(const int4 *)(pixtab + px);
      const int off[4] = {at.x, at.y, at.z, at.w};
      float xv[JT][4];
#pragma unroll
      for (int v = 0; v < JT; ++v)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          xv[v][i] = xl[off[i] + joff[v]];
          xv[v][i] = px + i < np ? xv[v][i] : 0.f;
        }
      if constexpr (sizeof(T) == 4) {
        // The 16 products of a group from zero, then one addition to the running sum: a
        // chain of roundings as many groups long as this wavefront sees, not as many
        // pixels.  (In one chain N64 3 -> 32, 128 x 128, 3 x 3 was 4.1e-7 from the exact
        // gradient, 1.6e-7 so, the kernel of one pixel per thread 2.4e-7; 49.4 -> 51.3 us.
        // A gradient rounded to 16 bits does not show either.)
#pragma unroll
        for (int v = 0; v < JT; ++v) {
          f32x4 part[KT];
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int u = 0; u < KT; ++u)
              part[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                  b[u][i], xv[v][i], i == 0 ? f32x4{0, 0, 0, 0} : part[u], 0, 0, 0);
#pragma unroll
          for (int u = 0; u < KT; ++u)
            acc[u][v] += part[u];
        }
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int v = 0; v < JT; ++v)
#pragma unroll
            for (int u = 0; u < KT; ++u)
              acc[u][v] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[u][i], xv[v][i], acc[u][v], 0, 0, 0);
      }
    };
    // (groups of 16 pixels, the wavefronts in turn, the next group's DY in flight)
    for (int grp = wave * 16; grp < np; grp += 128) {
      const int px = grp + (l >> 4) * 4;
      cf_load_dy<T, KT>(src, px + 64, np, a[1]);
      spend(a[0], px);
      if (grp + 64 >= np)
        break;
      cf_load_dy<T, KT>(src, px + 128, np, a[0]);
      spend(a[1], px + 64);
    }
  }
  // the wavefronts' sums in a fixed order: 2 -> 0, 3 -> 1, 1 -> 0
  __syncthreads();
  auto put = [&](float *to) {
#pragma unroll
    for (int u = 0; u < KT; ++u)
#pragma unroll
      for (int v = 0; v < JT; ++v)
        *(f32x4 *)(to + ((u * JT + v) * 64 + l) * 4) = acc[u][v];
  };
  auto take = [&](const float *from) {
#pragma unroll
    for (int u = 0; u < KT; ++u)
#pragma unroll
      for (int v = 0; v < JT; ++v)
        acc[u][v] += *(const f32x4 *)(from + ((u * JT + v) * 64 + l) * 4);
  };
  if (wave >= 2)
    put(smem + (wave - 2) * kFrag);
  __syncthreads();
  if (wave < 2)
    take(smem + wave * kFrag);
  __syncthreads();
  if (wave == 1)
    put(smem);
  __syncthreads();
  if (wave == 0) {
    take(smem);
    put(partial + ((int64_t)blockIdx.x * gridDim.y + blockIdx.y) * kFrag);
  }
}

// DW = sum of the workgroups' fragments: 16 values per workgroup, 64 slices of the
// runs, added in a fixed order.
__global__ __launch_bounds__(256) void conv_few_wgrad_sum_kernel(CfArgs g, const float *partial,
                                                                 void *dw, int dw_dt, int kt, int jt,
                                                                 int64_t frags, int runs) {
  __shared__ float lds[4][16];
  const int tid = threadIdx.x;
  const int64_t e0 = (int64_t)blockIdx.x * 16;
  const float *src = partial + e0 + (tid & 3) * 4;
  f32x4 s{0, 0, 0, 0};
  fhip_for_parts<4>(
      tid >> 2, 64, runs, [&](int r) { return *(const f32x4 *)(src + r * frags); },
      [&](f32x4 v, bool in) { s = in ? s + v : s; });
#pragma unroll
  for (int i = 0; i < 4; ++i)
    for (int o = 4; o < 64; o <<= 1)
      s[i] += __shfl_xor(s[i], o, 64);
  if ((tid & 63) < 4)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      lds[tid >> 6][(tid & 3) * 4 + i] = s[i];
  __syncthreads();
  if (tid >= 16)
    return;
  // value r of lane l of tile (u, v): channel u * 16 + (l / 16) * 4 + r, pair v * 16 + l % 16
  const int64_t e = e0 + tid;
  const int r = (int)(e & 3), l = (int)(e >> 2) & 63;
  const int tile = (int)(e >> 8);
  const int v = tile % jt, u = tile / jt % kt, kb = tile / (jt * kt);
  const int k = (kb * kt + u) * 16 + (l >> 4) * 4 + r, j = v * 16 + (l & 15);
  if (k >= g.K || j >= g.J)
    return;
  int f;
  cf_pair(g, j, &f);
  const float sum[1] = {(lds[0][tid] + lds[1][tid]) + (lds[2][tid] + lds[3][tid])};
  fhip_store_float(dw, dw_dt, k * g.ws[0] + f, 0, sum);
}

// ---- data gradient (unit stride and dilation) -----------------------------------
constexpr int kCfStage = 16; // loads per lane of one channel's rows of DY
constexpr int kCfRows = 2;   // rows of DX per lane: every staged row feeds two of them

template <typename T, int C, int S>
__global__ __launch_bounds__(512) void conv_few_dgrad_kernel(CfArgs g, const T *dy, const T *w,
                                                             T *dx) {
  constexpr int WP = (S * C + 3) & ~3; // a filter row of all channels
  constexpr int SPAN = (S + 3 + 3) & ~3;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int tid = threadIdx.x, l = tid & 63, wave = tid >> 6;
  const int threads = blockDim.x, waves = threads >> 6;
  const int pitch = 4 * g.quads + SPAN - 4, rows = g.band + g.R - 1;
  float *wl = smem; // [k][r][S][C]
  float *tile = smem + g.K * g.R * WP + wave * rows * pitch;
  const int n = blockIdx.x / g.tiles, h0 = (blockIdx.x % g.tiles) * g.band;
  // the element of every staged row this lane brings in, -1: a zero
  int at[kCfStage];
#pragma unroll
  for (int i = 0; i < kCfStage; ++i) {
    const int e = l + 64 * i;
    const int row = cf_div(e, g.lw_magic), col = e - row * pitch;
    const int p = h0 + g.pad_h - (g.R - 1) + row, q = g.pad_w - (S - 1) + col;
    at[i] = row < rows && (unsigned)p < (unsigned)g.P && (unsigned)q < (unsigned)g.Q
                ? p * (int)g.ys[2] + q * (int)g.ys[3]
                : -1;
  }
  const int loads = (rows * pitch + 63) / 64;
  T ahead[kCfStage];
  auto fetch = [&](int k) {
    const T *src = dy + n * g.ys[0] + k * g.ys[1];
#pragma unroll
    for (int i = 0; i < kCfStage; ++i)
      if (i < loads)
        ahead[i] = src[at[i] >= 0 ? at[i] : 0];
  };
  if (wave < g.K)
    fetch(wave);
#pragma unroll 4
  for (int e = tid; e < g.K * g.R * WP; e += threads) {
    const int kr = e / WP, sc = e % WP < S * C ? e % WP : 0;
    const int k = kr / g.R, r = kr - k * g.R;
    wl[e] = (float)w[k * g.ws[0] + (sc % C) * g.ws[1] + r * g.ws[2] + (sc / C) * g.ws[3]];
  }
  // (lanes behind the band repeat its last rows)
  const int hl = l / g.quads * kCfRows, qd = l % g.quads;
  const float *mine = tile + (hl + kCfRows <= g.band ? hl : g.band - kCfRows) * pitch + qd * 4;
  float acc[kCfRows][C][4];
#pragma unroll
  for (int y = 0; y < kCfRows; ++y)
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        acc[y][c][i] = 0.f;
  __syncthreads();
  for (int k = wave; k < g.K; k += waves) {
    // (a wavefront's LDS operations complete in order: its tile needs no barrier)
#pragma unroll
    for (int i = 0; i < kCfStage; ++i)
      if (i < loads && l + 64 * i < rows * pitch)
        tile[l + 64 * i] = at[i] >= 0 ? (float)ahead[i] : 0.f;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (k + waves < g.K)
      fetch(k + waves);
    // staged row t is tap R - 1 - t of this lane's first row, tap R - t of its second
    float f[kCfRows][WP];
    for (int t = 0; t < g.R + kCfRows - 1; ++t) {
      float v[SPAN];
#pragma unroll
      for (int i = 0; i < SPAN; i += 4) {
        const f32x4 x = *(const f32x4 *)(mine + t * pitch + i);
        v[i] = x.x, v[i + 1] = x.y, v[i + 2] = x.z, v[i + 3] = x.w;
      }
#pragma unroll
      for (int i = 0; i < WP; ++i)
        f[1][i] = f[0][i];
      if (t < g.R) {
        const float *wr = wl + (k * g.R + g.R - 1 - t) * WP;
#pragma unroll
        for (int i = 0; i < WP; i += 4) {
          const f32x4 x = *(const f32x4 *)(wr + i);
          f[0][i] = x.x, f[0][i + 1] = x.y, f[0][i + 2] = x.z, f[0][i + 3] = x.w;
        }
      }
      auto add = [&](auto yy) {
        constexpr int Y = decltype(yy)::value;
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
          for (int c = 0; c < C; ++c)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              acc[Y][c][i] = __builtin_fmaf(v[i + S - 1 - s], f[Y][s * C + c], acc[Y][c][i]);
      };
      if (t < g.R)
        add(std::integral_constant<int, 0>{});
      if (t > 0)
        add(std::integral_constant<int, 1>{});
    }
    __builtin_amdgcn_wave_barrier();
  }
  // the wavefronts' sums, added in their order: [wave][row][channel][lane][pixel]
  __syncthreads();
#pragma unroll
  for (int y = 0; y < kCfRows; ++y)
#pragma unroll
    for (int c = 0; c < C; ++c)
      *(f32x4 *)(smem + (((wave * kCfRows + y) * C + c) * 64 + l) * 4) =
          f32x4{acc[y][c][0], acc[y][c][1], acc[y][c][2], acc[y][c][3]};
  __syncthreads();
  const int quad = (tid & 255) >> 2;
  const int row0 = quad / g.quads * kCfRows, col = (quad % g.quads) * 4 + (tid & 3);
  if (row0 + kCfRows > g.band || col >= g.W)
    return;
  for (int yc = tid >> 8; yc < kCfRows * C; yc += threads >> 8) {
    const int y = yc / C, c = yc % C;
    if (h0 + row0 + y >= g.H)
      continue;
    const float *s = smem + yc * 256 + (tid & 255);
    float sum = s[0];
    for (int i = 1; i < waves; ++i)
      sum += s[i * kCfRows * C * 256];
    dx[n * g.xs[0] + c * g.xs[1] + (h0 + row0 + y) * g.xs[2] + col * g.xs[3]] = (T)sum;
  }
}

// ---- data gradient, products first ----------------------------------------------
// G[pair][pixel of DY] = sum over the output channels on the matrix cores, into LDS; a DX
// pixel then adds the R * S values of G that fall on it.  Bound by latency: a wavefront requests
// its 64 pixels of all channels at once, straight from memory, 4 consecutive pixels of a channel
// per load, and the filter behind them.  f32 N100 3 -> 32, 32 x 32, 3 x 3 (medians): 2.2 us to the
// last request, 1.6 for the data, 2.1 products, 2.8 taps; the lanes that keep 4 x 2 pixels take 7.3
// us for their loop of dependent rounds.  Where three tiles of pairs do not hold all input channels,
// passes of `cb` channels follow each other on the same registers or, while that fits two workgroups
// per compute unit, lie side by side.
//
// us, before -> now: f32 N100 3 -> 32, 32 x 32, 3 x 3 12.9 -> 11.1, N110 1 -> 32, 20 x 20 9.6 -> 5.6, N67
// 4 -> 32, 62 x 62 28.5 -> 25.7; bf16 N122 1 -> 64, 57 x 57, 5 x 5 77.0 -> 33.0, N118 3 -> 64, 39 x 39,
// 3 x 3 36.8 -> 15.1, N49 4 -> 64, 24 x 24 23.1 -> 7.2.
template <typename T> struct CfDgrad {
  static constexpr bool WIDE = sizeof(T) == 4; // f32: 16 x 16 x 4 products, else 16 x 16 x 32
  static constexpr int STEP = WIDE ? 4 : 32;   // channels of a product
  static constexpr int ROWS = WIDE ? 1 : 8;    // of them in a lane
  typedef T Quad __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  typedef T Eight __attribute__((ext_vector_type(8)));
};

// (a 16-bit product of eight channels per lane; never called with f32)
template <typename T, typename V> __device__ __forceinline__ f32x4 cf_mfma(V a, V b, f32x4 c) {
  if constexpr (std::is_same<T, __bf16>::value)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// KB: output channels in registers at once; PT: tiles of 16 pairs.
template <typename T, int S, int PT, int KB>
__global__ __launch_bounds__(1024) void conv_few_dgrad_products_kernel(CfArgs g, const T *dy, const T *w,
                                                             T *dx) {
  typedef CfDgrad<T> D;
  typedef typename D::Quad Quad;
  constexpr int STEPS = KB / D::STEP;
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int tid = threadIdx.x, l = tid & 63, threads = blockDim.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = threads >> 6;
  int h0;
  const int n = cf_div_uniform(blockIdx.x, g.tiles, g.tiles_whole, &h0);
  h0 *= g.band;
  const int w0 = blockIdx.y * g.wt;
  const int rows = g.H - h0 < g.band ? g.H - h0 : g.band, cols = g.W - w0 < g.wt ? g.W - w0 : g.wt;
  // Rows and columns of DY that reach this band (whole rows unless bands are cut).  A row is
  // whole quads, in G followed by the zeros that the taps beside the image meet.
  int p0 = h0 + g.pad_h - (g.R - 1), p1 = h0 + rows - 1 + g.pad_h;
  p0 = p0 < 0 ? 0 : p0;
  p1 = p1 < g.P ? p1 : g.P - 1;
  const int np = p1 >= p0 ? p1 - p0 + 1 : 0;
  int q0 = 0, q1 = g.Q - 1;
  if (gridDim.y > 1) {
    q0 = w0 + g.pad_w - (S - 1), q1 = w0 + cols - 1 + g.pad_w;
    q0 = q0 < 0 ? 0 : q0 < g.Q ? q0 : g.Q - 1;
    q1 = q1 < q0 ? q0 : q1 < g.Q ? q1 : g.Q - 1;
  }
  const int nq = q1 - q0 + 1, per_row = (nq + 3) >> 2, pitch = g.gpitch;
  const int quads = np * per_row, units = (quads + 15) >> 4;
  // A row's last quad may reach behind it (its values are not used) wherever DY goes on there.
  const bool whole = (nq & 3) == 0 ||
                     (g.Q >= 4 && ((p1 + 1 < g.P && g.ys[2] >= 4) || (n + 1 < g.N && g.ys[0] >= 4)));
  // (then a row's address is a uniform one plus 32 bits per lane)
  const bool fast = whole && (D::WIDE || (g.K & 7) == 0) && g.ys[1] < (1 << 24) && g.ys[2] < (1 << 16);
  const T *src = dy + n * g.ys[0] + (int64_t)p0 * g.ys[2] + q0;
  auto quad_row = [&](int i) { return gridDim.y > 1 ? i / per_row : cf_div(i, g.quads_magic); };
  Quad raw[STEPS][D::ROWS];
  auto fetch = [&](int unit, int k0) {
    asm volatile("" : "+s"(k0)); // (row addresses are not kept from one call to the next)
    int i = unit * 16 + (l & 15);
    i = i < quads ? i : quads - 1;
    const int row = quad_row(i), col = (i - row * per_row) * 4;
    if (fast) {
      const uint32_t at = (uint32_t)(row * (int)g.ys[2] + col);
      const uint32_t part = (uint32_t)((l >> 4) * D::ROWS), ks = (uint32_t)g.ys[1];
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
        // (channels behind the last one stand for channels in front of it)
        const int k = k0 + s * D::STEP, left = g.K - k;
        const uint32_t last = left >= D::STEP ? D::STEP : left > 0 ? (uint32_t)left - D::ROWS : 0u;
        const uint32_t off = (at + (part < last ? part : last) * ks) * (uint32_t)sizeof(T);
#pragma unroll
        for (int r = 0; r < D::ROWS; ++r) {
          const T *base = src + (k + r < g.K ? k + r : g.K - 1) * g.ys[1];
          raw[s][r] = *(const Quad *)((const char *)base + off);
        }
      }
    } else {
#pragma unroll
      for (int s = 0; s < STEPS; ++s)
#pragma unroll
        for (int r = 0; r < D::ROWS; ++r) {
          int k = k0 + s * D::STEP + (l >> 4) * D::ROWS + r;
          k = k < g.K ? k : g.K - 1;
          const T *q = src + ((int64_t)row * g.ys[2] + k * g.ys[1]);
#pragma unroll
          for (int j = 0; j < 4; ++j)
            raw[s][r][j] = q[col + j < nq ? col + j : nq - 1];
          __builtin_amdgcn_sched_barrier(0);
        }
    }
  };
  // the filter: f32 [channel][pair], else [pair][channel], zeros behind the last channel
  T *wl = (T *)smem;
  const int kpad = (g.K + D::STEP - 1) / D::STEP * D::STEP;
  auto stage = [&](auto packed) {
    constexpr int kBatch = 8; // (loads in flight; in branches of their own they would wait for each other)
    const int total = g.K * g.J;
    for (int e0 = tid; e0 < total; e0 += kBatch * threads) {
      T v[kBatch];
      int to[kBatch];
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        int e = e0 + i * threads;
        e = e < total ? e : total - 1;
        const int k = cf_div(e, g.q_magic), j = e - k * g.J;
        to[i] = D::WIDE ? k * g.wpitch + j : j * g.wpitch + k;
        if constexpr (decltype(packed)::value) {
          v[i] = w[e];
        } else {
          const int c = cf_div(j, g.rs_magic), t = j - c * g.R * S, r = cf_div(t, g.s_magic);
          v[i] = w[k * g.ws[0] + c * (int)g.ws[1] + r * (int)g.ws[2] + (t - r * S) * (int)g.ws[3]];
        }
      }
      // (the last one may be written several times)
#pragma unroll
      for (int i = 0; i < kBatch; ++i)
        wl[to[i]] = v[i];
    }
    for (int e = tid; e < (kpad - g.K) * g.J; e += threads) {
      const int k = cf_div(e, g.q_magic), j = e - k * g.J;
      wl[D::WIDE ? (g.K + k) * g.wpitch + j : j * g.wpitch + g.K + k] = (T)0.f;
    }
  };
  float *gl = smem + g.gat + 4; // G, [pair][row][column], zeros in front of it
  const int gp = np * pitch, rs = g.R * S;
  const bool held = units <= waves && g.K <= KB;
  bool first = true;
  for (int c0 = blockIdx.z * g.cb; c0 < g.C; c0 += gridDim.z * g.cb) {
    const int cs = g.C - c0 < g.cb ? g.C - c0 : g.cb, pairs = cs * rs;
    // (every wavefront takes part in every round: the first one holds a barrier)
    for (int unit = wave; unit - wave < units; unit += waves) {
      f32x4 acc[PT][4];
#pragma unroll
      for (int u = 0; u < PT; ++u)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          acc[u][t] = f32x4{0, 0, 0, 0};
      for (int k0 = 0; k0 < g.K; k0 += KB) {
        if (first || !held)
          fetch(unit, k0);
        if (first) {
          if (g.packed && g.ws[0] == g.J)
            stage(std::true_type{});
          else
            stage(std::false_type{});
          if (tid < 4)
            gl[tid - 4] = 0.f;
          if (pitch > 4 * per_row)
            for (int i = tid; i < g.cb * rs * np; i += threads)
              for (int j = 4 * per_row; j < pitch; j += 4)
                *(f32x4 *)(gl + i * pitch + j) = f32x4{0, 0, 0, 0};
          __syncthreads();
          first = false;
        }
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
          const int k = k0 + s * D::STEP;
          if (k >= g.K)
            continue;
          if (k + D::STEP > g.K) // (0 x infinity)
#pragma unroll
            for (int r = 0; r < D::ROWS; ++r)
              if (k + (l >> 4) * D::ROWS + r >= g.K)
                raw[s][r] = Quad{};
          if constexpr (D::WIDE) {
            const float *wr = (const float *)wl + (k + (l >> 4)) * g.wpitch + c0 * rs + (l & 15);
#pragma unroll
            for (int u = 0; u < PT; ++u) {
              const float a = wr[u * 16];
#pragma unroll
              for (int t = 0; t < 4; ++t)
                acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, (float)raw[s][0][t], acc[u][t], 0, 0, 0);
            }
          } else {
            typename D::Eight b[4];
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
              for (int r = 0; r < 8; ++r)
                b[t][r] = raw[s][r % D::ROWS][t];
#pragma unroll
            for (int u = 0; u < PT; ++u) {
              const auto a = *(const typename D::Eight *)(wl + (c0 * rs + u * 16 + (l & 15)) * g.wpitch + k +
                                                          (l >> 4) * 8);
#pragma unroll
              for (int t = 0; t < 4; ++t)
                acc[u][t] = cf_mfma<T>(a, b[t], acc[u][t]);
            }
          }
        }
      }
      // value r of tile (u, t): pair u * 16 + (l / 16) * 4 + r, pixel t of quad l % 16
      const int i = unit * 16 + (l & 15);
      if (i < quads) {
        const int row = quad_row(i), col = (i - row * per_row) * 4;
        float *to = gl + (l >> 4) * 4 * gp + row * pitch + col;
        if (col + 4 > nq)
#pragma unroll
          for (int t = 1; t < 4; ++t)
            if (col + t >= nq)
#pragma unroll
              for (int u = 0; u < PT; ++u)
                acc[u][t] = f32x4{0, 0, 0, 0};
#pragma unroll
        for (int u = 0; u < PT; ++u)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (u * 16 + (l >> 4) * 4 + r < pairs)
              *(f32x4 *)(to + (u * 16 + r) * gp) = f32x4{acc[u][0][r], acc[u][1][r], acc[u][2][r], acc[u][3][r]};
      }
    }
    __syncthreads();
    // runs of four pixels of DX
    const int per = (cols + 3) >> 2, plane = rows * per;
    for (int e = tid; e < cs * plane; e += threads) {
      int c = 0, i = e;
      for (; i >= plane; i -= plane)
        ++c;
      const int hh = cols == g.wt ? cf_div(i, g.w_magic) : i / per, wc = (i - hh * per) * 4;
      // tap (r, s) of a pixel: row p - r, column q - s of DY
      const int p = h0 + hh + g.pad_h, q = w0 + wc + g.pad_w - q0;
      const float *from = gl + c * rs * gp;
      typedef float Four __attribute__((ext_vector_type(4), aligned(4)));
      f32x4 sum{0, 0, 0, 0};
#pragma unroll 3
      for (int r = 0; r < g.R; ++r) {
        const bool in = p - r >= p0 && p - r <= p1;
        const float *row = from + r * S * gp + (in ? (p - r - p0) * pitch + q : 0);
        f32x4 v[S];
#pragma unroll
        for (int s = 0; s < S; ++s)
          v[s] = *(const Four *)(row + s * gp - s);
#pragma unroll
        for (int s = 1; s < S; ++s)
          v[0] += v[s];
        sum += in ? v[0] : f32x4{0, 0, 0, 0};
      }
      T *to = dx + (n * g.xs[0] + (c0 + c) * g.xs[1] + (h0 + hh) * g.xs[2] + w0 + wc);
      if (wc + 4 <= cols) {
        Quad t;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          t[j] = (T)sum[j];
        *(Quad *)to = t;
      } else {
#pragma unroll
        for (int j = 0; j < 3; ++j)
          if (wc + j < cols)
            to[j] = (T)sum[j];
      }
    }
    if (c0 + (int)gridDim.z * g.cb < g.C)
      __syncthreads();
  }
}

// ---- host side -------------------------------------------------------------------
bool cf_type(int dt) { return dt == FHIP_FLOAT || dt == FHIP_BFLOAT16 || dt == FHIP_HALF; }

// Everything but the tiling; `y`: OUT (forward) or DY.
bool cf_args(const fhip_conv_desc *d, const fhip_tensor_desc &y, CfArgs &g) {
  if (d->spatial_rank != 2 || d->x.rank != 4 || d->w.rank != 4 || y.rank != 4)
    return false;
  if (d->w.dim[1] != d->x.dim[1] || d->x.dtype != d->w.dtype || !cf_type(d->x.dtype))
    return false;
  const int64_t lim = 1 << 16;
  for (int i = 0; i < 4; ++i)
    if (d->x.dim[i] >= lim || d->w.dim[i] >= lim || y.dim[i] >= lim)
      return false;
  for (int i = 0; i < 2; ++i)
    if (d->padding[i] >= lim || d->stride[i] >= lim || d->dilation[i] >= lim)
      return false;
  const int64_t J = d->w.dim[1] * d->w.dim[2] * d->w.dim[3];
  // (fewer output channels than half a tile stay on the kernel of one pixel per thread)
  if (J > kCfMaxPairs || d->w.dim[0] < 8)
    return false;
  g.N = (int32_t)d->x.dim[0], g.C = (int32_t)d->x.dim[1];
  g.H = (int32_t)d->x.dim[2], g.W = (int32_t)d->x.dim[3];
  g.K = (int32_t)d->w.dim[0], g.R = (int32_t)d->w.dim[2], g.S = (int32_t)d->w.dim[3];
  g.P = (int32_t)y.dim[2], g.Q = (int32_t)y.dim[3];
  g.J = (int32_t)J;
  g.rs_magic = cf_magic(g.R * g.S), g.s_magic = cf_magic(g.S);
  g.q_magic = cf_magic(g.Q), g.q_whole = 0xffffffffu / (uint32_t)g.Q;
  g.pad_h = (int32_t)d->padding[0], g.pad_w = (int32_t)d->padding[1];
  g.str_h = (int32_t)d->stride[0], g.str_w = (int32_t)d->stride[1];
  g.dil_h = (int32_t)d->dilation[0], g.dil_w = (int32_t)d->dilation[1];
  auto strides = [](const fhip_tensor_desc &t, int64_t (&s)[4]) {
    int64_t image = 0;
    for (int i = 0; i < 4; ++i) {
      s[i] = t.dim[i] == 1 ? 0 : t.stride[i];
      if (s[i] >= (1ll << 31))
        return false;
      image += i ? (t.dim[i] - 1) * s[i] : 0;
    }
    return image < (1ll << 31); // offsets inside one image are 32-bit
  };
  if (!strides(d->x, g.xs) || !strides(d->w, g.ws) || !strides(y, g.ys))
    return false;
  g.packed = (g.S == 1 || g.ws[3] == 1) && (g.R == 1 || g.ws[2] == g.S) && (g.C == 1 || g.ws[1] == g.R * g.S);
  // X walked along its rows (channels-last tensors have kernels of their own)
  return g.W == 1 || g.xs[3] == 1;
}

// pixels of a plane of OUT / DY consecutive
bool cf_planes(const CfArgs &g) {
  return (g.Q == 1 || g.ys[3] == 1) && (g.P == 1 || g.ys[2] == g.Q);
}

// staged X of `span` rows of output; false where LDS does not hold it beside `other` floats
bool cf_stage(CfArgs &g, int span, int64_t other, size_t *bytes) {
  const int64_t lw = (int64_t)(g.Q - 1) * g.str_w + (int64_t)(g.S - 1) * g.dil_w + 1;
  const int64_t rows = (int64_t)(span - 1) * g.str_h + (int64_t)(g.R - 1) * g.dil_h + 1;
  const int64_t total = lw * rows * g.C;
  if (lw >= (1 << 16) || rows >= (1 << 16) || total >= (1 << 16) || (total + other) * 4 > kCfLds)
    return false;
  g.lw = (int32_t)lw, g.lw_magic = cf_magic(g.lw);
  g.xrows = (int32_t)rows, g.rows_magic = cf_magic(g.xrows);
  g.col_step = kCfThreads % g.lw;
  g.row_step = kCfThreads / g.lw % g.xrows, g.c_step = kCfThreads / g.lw / g.xrows;
  *bytes = (size_t)(total + other) * 4;
  return true;
}

template <typename F> void cf_by_type(int dt, F &&f) {
  if (dt == FHIP_FLOAT)
    f(float{});
  else if (dt == FHIP_BFLOAT16)
    f(__bf16{});
  else
    f(_Float16{});
}

} // namespace

int fhip_few_conv_fprop(fhip_ctx *ctx, const fhip_conv_desc *d, const void *x, const void *w,
                        const DevEpilogue &epi, void *out, bool *handled) {
  *handled = false;
  CfArgs g{};
  if (!cf_args(d, d->out, g) || !cf_planes(g) || !cf_type(d->y.dtype) || !cf_type(d->out.dtype) ||
      !fhip_epilogue_is_fast(d->epilogue))
    return 0;
  for (int i = 0; i < epi.count; ++i)
    if (epi.op[i].kind == FHIP_OPERAND_TENSOR &&
        ((g.P > 1 && epi.op[i].stride[2] != 0) || (g.Q > 1 && epi.op[i].stride[3] != 0)))
      return 0; // (operands per channel only)
  g.tiles = (int32_t)(((int64_t)g.P * g.Q + kCfThreads - 1) / kCfThreads);
  const int64_t blocks = (int64_t)g.N * g.tiles;
  if ((int64_t)g.P * g.Q >= (1ll << 30) || blocks >= (1ll << 23))
    return 0;
  const int j4 = (g.J + 3) / 4 * 4;
  const int span = (kCfThreads - 1 + g.Q - 1) / g.Q + 1;
  size_t lds = 0;
  int kt = g.K > 32 ? 4 : g.K > 16 ? 2 : 1;
  auto fits = [&]() {
    const int kp = kt * 16 + (kt % 2 ? 0 : 16);
    return cf_stage(g, span < g.P ? span : g.P, (int64_t)j4 * (kp + 1) + FHIP_MAX_EPILOGUE * kt * 16, &lds);
  };
  if (!fits())
    return 0;
  const int64_t cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  // (few tiles: a workgroup of 64 channels is a long chain of its own, mostly scalar loads
  // of the fused operations, so fewer channels each until there are two workgroups per
  // compute unit: N16 3 -> 64, 20 x 20, 3 x 3 f32 64 channels 14.9 us, 16 of them 8.8, the
  // kernel of one pixel per thread 11.2; shorter ones until there are 1.6: bf16 N71 4 -> 32,
  // 40 x 40, 497 tiles 10.5, with 16 channels each 11.5)
  const int64_t enough = g.K > 32 ? 2 * cus : 8 * cus / 5;
  while (kt > 1 && blocks * ((g.K + kt * 16 - 1) / (kt * 16)) < enough)
    kt /= 2;
  if (!fits())
    return 0;
  g.y_dt = d->y.dtype, g.o_dt = d->out.dtype;
  g.epi = epi;
  *handled = true;
  fhip_note_kernel(ctx, "conv_few fprop channels=%d", kt * 16);
  const dim3 grid((unsigned)g.tiles, (unsigned)g.N, (unsigned)((g.K + kt * 16 - 1) / (kt * 16)));
  cf_by_type(d->x.dtype, [&](auto t) {
    typedef decltype(t) T;
    auto kernel = kt == 4   ? conv_few_fprop_kernel<T, 4>
                  : kt == 2 ? conv_few_fprop_kernel<T, 2>
                            : conv_few_fprop_kernel<T, 1>;
    hipLaunchKernelGGL(kernel, grid, dim3(kCfThreads), lds, ctx->stream, g, (const T *)x,
                       (const T *)w, out);
  });
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  return 0;
}

int fhip_few_conv_wgrad(fhip_ctx *ctx, const fhip_conv_desc *d, const void *dy, const void *x,
                        void *dw, bool *handled) {
  *handled = false;
  CfArgs g{};
  if (!cf_args(d, d->y, g) || !cf_planes(g) || d->y.dtype != d->x.dtype)
    return 0;
  int kt = g.K > 32 ? 4 : g.K > 16 ? 2 : 1;
  const int tiles_j = (g.J + 15) / 16;
  const int jt = tiles_j <= 2 ? 2 : tiles_j <= 3 ? 3 : tiles_j <= 5 ? 5 : 7;
  // bands of about 256 pixels, of equal height
  int band = 256 / g.Q;
  band = band < 1 ? 1 : band < g.P ? band : g.P;
  g.tiles = (g.P + band - 1) / band;
  g.band = (g.P + g.tiles - 1) / g.tiles;
  g.tiles = (g.P + g.band - 1) / g.band;
  g.tiles_whole = 0xffffffffu / (uint32_t)g.tiles;
  size_t lds = 0;
  const int64_t slots = ((int64_t)g.band * g.Q + 15) / 16 * 16;
  if (slots >= (1 << 14) || !cf_stage(g, g.band, slots, &lds))
    return 0;
  const int64_t items = (int64_t)g.N * g.tiles;
  const int64_t cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  // (few bands: their products are a workgroup's longest part, so fewer output channels
  // each; N4 12 -> 64, 16 x 16, 3 x 3 f32: 20.8 us with 64)
  while (kt > 1 && items * ((g.K + kt * 16 - 1) / (kt * 16)) < cus)
    kt /= 2;
  const size_t meet = (size_t)2 * kt * jt * 256 * sizeof(float);
  lds = lds < meet ? meet : lds;
  const int kblocks = (g.K + kt * 16 - 1) / (kt * 16);
  const int64_t frags = (int64_t)kblocks * kt * jt * 256;
  if (items >= (1ll << 31) || kblocks > 65535)
    return 0;
  // Two workgroups per compute unit with 64 channels each, as their registers allow, else three (f32
  // N89 1 -> 32, 57 x 57, 3 x 3 17.9 us with two, 15.9 with three, 17.3 with four; N124 4 -> 16, 37 x 37 11.4, 9.3
  // and 10.0; N119 3 -> 64, 58 x 58 36.2 with two, 41.1 with three), no more than 8 MB of partial sums.
  int64_t runs = (kt == 4 ? 2 : 3) * cus / kblocks, most = (8ll << 20) / (frags * 4);
  runs = runs < most ? runs : most;
  runs = runs < items ? runs : items;
  runs = runs < 1 ? 1 : runs;
  const size_t bytes = (size_t)(runs * frags) * sizeof(float);
  void *scratch = nullptr;
  if (!fhip_ctx_scratch_ready(ctx, bytes))
    return 0;
  if (fhip_ctx_scratch(ctx, bytes, &scratch) != 0)
    return 1;
  *handled = true;
  fhip_note_kernel(ctx, "conv_few wgrad tiles=%dx%d", kt, jt);
  const dim3 grid((unsigned)runs, (unsigned)kblocks);
  cf_by_type(d->x.dtype, [&](auto t) {
    typedef decltype(t) T;
    auto with = [&](auto kk) {
      constexpr int KT = decltype(kk)::value;
      auto kernel = jt == 2   ? conv_few_wgrad_kernel<T, KT, 2>
                    : jt == 3 ? conv_few_wgrad_kernel<T, KT, 3>
                    : jt == 5 ? conv_few_wgrad_kernel<T, KT, 5>
                              : conv_few_wgrad_kernel<T, KT, 7>;
      hipLaunchKernelGGL(kernel, grid, dim3(kCfThreads), lds, ctx->stream, g, (const T *)dy,
                         (const T *)x, (float *)scratch);
    };
    if (kt == 4)
      with(std::integral_constant<int, 4>{});
    else if (kt == 2)
      with(std::integral_constant<int, 2>{});
    else
      with(std::integral_constant<int, 1>{});
  });
  hipLaunchKernelGGL(conv_few_wgrad_sum_kernel, dim3((unsigned)(frags / 16)), dim3(256), 0,
                     ctx->stream, g, (const float *)scratch, dw, (int)d->w.dtype, kt, jt, frags,
                     (int)runs);
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  return 0;
}

static int cf_allow_lds(fhip_ctx *ctx, const void *kernel, FhipOncePerDevice &configured) {
  if (configured.done(ctx->device))
    return 0;
  FHIP_HIP_CHECK(ctx, hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kCfDgradLds));
  configured.mark(ctx->device);
  return 0;
}

// conv_few_dgrad_kernel: bands of DX rows (a multiple of the rows per lane, of equal height) in `g`,
// workgroups, their wavefronts and LDS; `ok` false where it does not take the problem.
struct CfLanes {
  bool ok = false;
  int64_t blocks = 0, floats = 0;
  int waves = 0, pitch = 0;
};
static CfLanes cf_dgrad_lanes(fhip_ctx *ctx, CfArgs &g) {
  CfLanes p;
  g.quads = (g.W + 3) / 4;
  const int pairs = (g.H + kCfRows - 1) / kCfRows, most = 64 / g.quads;
  g.tiles = (pairs + most - 1) / most;
  g.band = (pairs + g.tiles - 1) / g.tiles * kCfRows;
  const int span = (g.S + 6) & ~3, rows = g.band + g.R - 1;
  p.pitch = 4 * g.quads + span - 4;
  const int64_t filter = (int64_t)g.K * g.R * ((g.S * g.C + 3) & ~3);
  p.blocks = (int64_t)g.N * g.tiles;
  // a quarter of the output channels per wavefront, an eighth where that leaves
  // fewer than two wavefronts per SIMD
  const int64_t cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  p.waves = p.blocks * 4 < 8 * cus ? 8 : 4;
  p.floats = filter + (int64_t)p.waves * rows * p.pitch;
  const int64_t meet = (int64_t)p.waves * kCfRows * 256 * g.C;
  p.floats = p.floats < meet ? meet : p.floats;
  p.ok = (int64_t)rows * p.pitch <= 64 * kCfStage && p.floats * 4 <= kCfLds && p.blocks < (1ll << 23);
  return p;
}

static int cf_dgrad_products(fhip_ctx *ctx, const fhip_conv_desc *d, CfArgs g, const void *dy, const void *w,
                             void *dx, bool *handled) {
  const int rs = g.R * g.S;
  if (rs > 48)
    return 0;
  // (three tiles of pairs at most)
  const int most = 48 / rs < g.C ? 48 / rs : g.C, passes = (g.C + most - 1) / most;
  g.cb = (g.C + passes - 1) / passes;
  const int pt = (g.cb * rs + 15) / 16;
  // The filter in LDS: f32 [channel][pair], the four rows of a product in different banks;
  // 16 bits [pair][channel], whole 16-byte runs.  Tiles read behind the last pair.
  const bool wide = d->x.dtype == FHIP_FLOAT;
  const int seen = (passes - 1) * g.cb * rs + pt * 16;
  const int64_t kpad = wide ? (g.K + 3) / 4 * 4 : (g.K + 31) / 32 * 32;
  g.wpitch = wide ? (seen + 15) / 32 * 32 + 16 : (int32_t)kpad + 8;
  const int64_t filter = (wide ? kpad * g.wpitch : (int64_t)seen * g.wpitch / 2 + 1) + 16;
  if (kpad * g.J >= (1 << 16))
    return 0;
  g.gat = (int32_t)((filter + 3) / 4 * 4);
  g.q_magic = cf_magic(g.J);
  const int64_t tiles_w = (g.W + 127) / 128;
  g.wt = (int32_t)((g.W + tiles_w - 1) / tiles_w);
  g.w_magic = cf_magic((g.wt + 3) / 4), g.quads_magic = cf_magic((g.Q + 3) / 4);
  const int64_t nq = tiles_w == 1 || g.wt + g.S - 1 > g.Q ? g.Q : g.wt + g.S - 1;
  const int beside = g.S - 1 > g.pad_w ? g.S - 1 - g.pad_w : 0; // columns that taps reach beside DY
  const int64_t row = (nq + beside + 3) / 4 * 4;
  g.gpitch = (int32_t)row;
  auto rows_dy = [&](int64_t band) { return band + g.R - 1 < g.P ? band + g.R - 1 : (int64_t)g.P; };
  auto units_of = [&](int64_t band) { return (rows_dy(band) * ((nq + 3) / 4) + 15) / 16; };
  // Rows of DX per band: G in `lds` bytes, a wavefront's 64 pixels once.
  auto band_of = [&](int64_t lds, int64_t waves) {
    int64_t fit = (lds / 4 - g.gat - 16) / (g.cb * rs * row), unit = waves * 16 / ((nq + 3) / 4);
    fit = fit < unit ? fit : unit;
    const int64_t band = fit >= g.P ? (int64_t)g.H : fit - (g.R - 1);
    return band < g.H ? band : (int64_t)g.H;
  };
  int64_t band = band_of(kCfDgradLds / 2, 8), alone = band_of(kCfDgradLds, 16);
  // (rows read per row written: f32 N128 4 -> 64, 64 x 64, 5 x 5 in half of LDS 304 us, in all of it
  // 174; N113 3 -> 16, 47 x 47, 3 x 3, where the difference is a tenth, 15.6 and 17.2)
  auto halo = [&](int64_t b) { return b < 1 ? 1e9 : b == g.H ? 1.0 : (double)(b + g.R - 1) / (double)b; };
  if (halo(alone) < 0.75 * halo(band))
    band = alone;
  if (band < 1)
    return 0;
  band = band * g.wt < (1 << 16) ? band : ((1 << 16) - 1) / g.wt;
  // Lower bands where that spreads the pixels better: rounds of workgroups over the compute units,
  // each a start and its wavefronts' products.  (f32 N100 3 -> 32, 32 x 32, 3 x 3: 300 workgroups
  // 13.5 us, 400 11.1; bf16 N22 1 -> 64, 54 x 54, 5 x 5: 308 8.9, 242 6.9.)
  const int64_t cus = ctx->num_cus > 0 ? ctx->num_cus : 256;
  double best = 1e30;
  for (int64_t t = (g.H + band - 1) / band; t <= g.H; ++t) {
    const int64_t b = (g.H + t - 1) / t, wgs = (int64_t)g.N * ((g.H + b - 1) / b) * tiles_w;
    const double cost = (double)((wgs + cus - 1) / cus) * ((double)units_of(b) + 2.0);
    if (cost < best)
      best = cost, g.band = (int32_t)b;
    if (wgs > 4 * cus || b < g.R)
      break;
  }
  g.tiles = (g.H + g.band - 1) / g.band;
  g.tiles_whole = 0xffffffffu / (uint32_t)g.tiles;
  const int64_t blocks = (int64_t)g.N * g.tiles;
  if (blocks >= (1ll << 23))
    return 0;
  const size_t lds = (size_t)(g.gat + 16 + rows_dy(g.band) * row * g.cb * rs) * 4;
  const int64_t units = units_of(g.band);
  const int waves = (int)(units < 2 ? 2 : units < 16 ? units : 16);
  const unsigned parts = passes > 1 && blocks * tiles_w * passes <= 2 * cus ? (unsigned)passes : 1u;
  // Passes on one workgroup pay where the taps' multiplications of conv_few_dgrad_kernel are many:
  // 16-bit tensors from 32 output channels on (us there / here, 5 x 5: bf16 N64 4 -> 64, 36 x 36 36.9 /
  // 16.6, 4 -> 32 21.8 / 14.9, 4 -> 16 13.3 / 15.5), f32 where the pixels are few besides (N64 3 -> 32,
  // 20 x 20 17.2 / 13.5, 36 x 36 18.1 / 18.1, N120, 50 x 50 46.7 / 53.2).
  if (passes > 1 && parts == 1 &&
      (g.K < 32 || (wide && (int64_t)g.N * g.H * g.W > 110 * cus)))
    return 0;
  // In f32 conv_few_dgrad_kernel takes over where a compute unit has much work here (rounds of
  // workgroups times wavefronts of each): its bands do not overlap, and up to two workgroups of eight
  // wavefronts to a unit it takes one round.  us, there / here, 5 x 5 over one channel: N22, 24 x 24 -> 16
  // 7.6 / 6.2, N69, 33 x 33 8.2 / 10.1, N101, 62 x 62 16.9 / 28.5; N67, 48 x 48 -> 32 without pad 15.9 / 12.8,
  // N120, 39 x 39 16.5 / 19.6; N50, 33 x 33 -> 64 18.4 / 15.8, N78, 45 x 45 25.8 / 31.1, N68, 55 x 55 27.8 /
  // 42.8.  3 x 3: N62 3 -> 64, 62 x 62 29.4 / 44.3, N62 4 -> 16, 60 x 60 13.8 / 17.8, N106 3 -> 16, 61 x 61 18.8 /
  // 24.3, N113 3 -> 64, 60 x 60 51.8 / 61.2, but N104 4 -> 16, 38 x 38 13.7 / 13.4, N120 3 -> 32, 49 x 49 29.9 / 24.5.
  // (16 bits: 3 x 3 always faster here, 5 x 5 from 32 channels on 1.4 to 3.9 times, -> 16 as often up to a
  // fifth slower as faster.)
  if (wide && passes == 1) {
    const int64_t work = (blocks * tiles_w + cus - 1) / cus * units;
    CfArgs other = g;
    const CfLanes lanes = cf_dgrad_lanes(ctx, other);
    const bool lead = g.K > 16 && g.K <= 32; // (32 channels are one block of registers here)
    const int64_t most = g.S == 5 ? (lead ? 16 : 8) : lanes.waves == 8 ? 16 : lead ? 36 : 24;
    if (lanes.ok && work > most)
      return 0;
  }
  *handled = true;
  fhip_note_kernel(ctx, "conv_few dgrad products channels=%d", g.C);
  int status = 0;
  cf_by_type(d->x.dtype, [&](auto t) {
    typedef decltype(t) T;
    auto with = [&](auto ss, auto tiles, auto block) {
      constexpr int S = decltype(ss)::value, PT = decltype(tiles)::value, KB = decltype(block)::value;
      constexpr bool held = sizeof(T) == 2 || PT < 3; // (see channels)
      auto kernel = conv_few_dgrad_products_kernel<T, S, PT, held ? KB : 32>;
      static FhipOncePerDevice configured;
      status = cf_allow_lds(ctx, reinterpret_cast<const void *>(kernel), configured);
      if (status == 0)
        hipLaunchKernelGGL(kernel, dim3((unsigned)blocks, (unsigned)tiles_w, parts), dim3(waves * 64), lds, ctx->stream, g,
                           (const T *)dy, (const T *)w, (T *)dx);
    };
    auto pairs = [&](auto ss, auto block) {
      if (pt == 1)
        with(ss, std::integral_constant<int, 1>{}, block);
      else if (pt == 2)
        with(ss, std::integral_constant<int, 2>{}, block);
      else
        with(ss, std::integral_constant<int, 3>{}, block);
    };
    auto channels = [&](auto ss) {
      // (128 registers: f32 channels beside three tiles of pairs in two blocks)
      if (g.K <= 32 || (wide && pt == 3))
        pairs(ss, std::integral_constant<int, 32>{});
      else
        pairs(ss, std::integral_constant<int, 64>{});
    };
    if (g.S == 3)
      channels(std::integral_constant<int, 3>{});
    else
      channels(std::integral_constant<int, 5>{});
  });
  if (status != 0)
    return status;
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  return 0;
}

int fhip_few_conv_dgrad(fhip_ctx *ctx, const fhip_conv_desc *d, const void *dy, const void *w,
                        void *dx, bool *handled) {
  *handled = false;
  CfArgs g{};
  if (!cf_args(d, d->y, g) || d->y.dtype != d->x.dtype)
    return 0;
  if (g.C > 4 || (g.S != 3 && g.S != 5) || g.str_h != 1 || g.str_w != 1 || g.dil_h != 1 ||
      g.dil_w != 1 || (g.Q > 1 && g.ys[3] != 1) || g.W > 256)
    return 0;
  const int status = cf_dgrad_products(ctx, d, g, dy, w, dx, handled);
  if (status != 0 || *handled)
    return status;
  const CfLanes lanes = cf_dgrad_lanes(ctx, g);
  if (!lanes.ok)
    return 0;
  g.lw_magic = cf_magic(lanes.pitch);
  *handled = true;
  fhip_note_kernel(ctx, "conv_few dgrad channels=%d", g.C);
  cf_by_type(d->x.dtype, [&](auto t) {
    typedef decltype(t) T;
    auto with = [&](auto cc) {
      constexpr int C = decltype(cc)::value;
      auto kernel = g.S == 3 ? conv_few_dgrad_kernel<T, C, 3> : conv_few_dgrad_kernel<T, C, 5>;
      hipLaunchKernelGGL(kernel, dim3((unsigned)lanes.blocks), dim3(lanes.waves * 64), (size_t)lanes.floats * 4,
                         ctx->stream, g, (const T *)dy, (const T *)w, (T *)dx);
    };
    if (g.C == 1)
      with(std::integral_constant<int, 1>{});
    else if (g.C == 2)
      with(std::integral_constant<int, 2>{});
    else if (g.C == 3)
      with(std::integral_constant<int, 3>{});
    else
      with(std::integral_constant<int, 4>{});
  });
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  return 0;
}

// Convolution weight gradient for 3 x 3 filters, straight from X and DY.
//
//   DW[k, r, s, c] = sum over n, p, q of DY[n, p, q, k] * X[n, p + r - pad, q + s - pad, c]
//
// (channels-last 16-bit tensors, one group, unit strides and dilations,
// padding up to 2 on all sides, DY of up to 56 columns, C and K multiples of 8).  As a GEMM
// this is skinny: 9 * C * K outputs, reduced over every pixel of the batch, and
// the reduction runs along the tensors' slow dimension.  The kernel therefore
//
//  * gives a workgroup one 32 x 32 block of (k, c) for all nine taps -- 144
//    accumulator registers per lane -- and an equal share of the batch's rows,
//    of which its eight wavefronts reduce equal shares; their results are summed
//    through LDS at the end, so a workgroup leaves 36 KB of partial sums, not 288 KB;
//  * streams image rows through small per-wavefront LDS rings by LDS-DMA (a
//    pixel's 32 channels of this block are 64 contiguous bytes) and takes the
//    MFMA operands out of them with transposing reads: 16 consecutive pixels of
//    a row are the K extent of one 32 x 32 x 16 MFMA, and a row takes as many
//    as it has (NKS), not the four of the widest;
//  * walks the rows of X: row rho pairs with the DY rows rho + pad, rho + pad - 1, rho + pad - 2
//    (filter rows 0, 1, 2), whose fragments stay in registers for the three
//    visits, and the three column taps are the same LDS row read one pixel
//    apart -- six fragment reads feed nine MFMAs;
//  * runs from one image into the next: the loads of a step are always the same
//    number (rows that do not exist are fetched from nowhere), kD steps ahead of it, so the
//    waits count and nothing drains between images;
//  * needs no barrier in the main loop: a wavefront only waits for its own DMA;
//  * multiplies X with existing DY only: products with rows that do not exist are branched
//    around and X is blanked past a row's end, so that an infinite X value shows in the taps
//    that meet it and in no other (58 layers 1.5 % slower in the mean for it, rows of one step 2 to 4).
//    An infinite DY value in the first and last columns meets the zeros of X's padding, as in
//    the gathered tiles; in the first and last rows it meets X alone.
//
// A second, small kernel sums the workgroups' partial results in a fixed
// order (the result does not depend on scheduling) and writes DW in its dtype
// and strides.
//
// Reference semantics: node/conv_node.h:255-426 (ConvWGradNode),
// aten.convolution_backward, weight gradient.
#include "common.h"
#include "fast_paths.h"
#include "gemm_kernel.h"

namespace {

constexpr int kWdWaves = 8;
constexpr int kWdThreads = kWdWaves * 64;
constexpr int kWdWaveLds = 20480;
constexpr int kWdLds = kWdWaves * kWdWaveLds; // 160 KB

// Rows of up to 16 NKS pixels (56 for NKS 4): LDS-DMA instructions of 16 pixels (1 KB) per row of
// X (one pixel of padding on each side) and of DY, and the steps that loads run ahead: as
// many as a wavefront's 20 KB hold (kD rows of DY, kD + 1 of X).
template <int NKS> struct WdRows {
  static constexpr int kX = NKS < 4 ? NKS + 1 : 4, kY = NKS;
  static constexpr int kD = NKS == 1 ? 6 : NKS == 2 ? 3 : 2;
  static constexpr uint32_t kXBytes = kX * 1024, kYBytes = kY * 1024, kYBase = (kD + 1) * kXBytes;
  static_assert(kYBase + kD * kYBytes <= kWdWaveLds && (kD - 1) * (kX + kY) < 64, "LDS, vmcnt");
};
constexpr int kWdMaxW = 56;
constexpr int kWdBlock = 9 * 16 * 64; // partial sums of one workgroup (floats)

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct WgDirectArgs {
  const char *x, *dy;
  float *part;
  int32_t H, W, C, K, P, Q;
  int32_t pad;
  int32_t rows;   // of X: N * H
  int32_t nparts; // workgroups per (k, c) block
  int32_t types, ctypes; // blocks, C / 32 rounded up
  int32_t total, per_xcd; // types * nparts, an eighth of it rounded up
  uint32_t magic_types, magic_ctypes, magic_h;
  uint32_t x_bytes, dy_bytes;
};

// rows [first, last) of share `i` of `n`
__device__ __forceinline__ int wd_share(int rows, int i, int n) { return (int)((int64_t)rows * i / n); }

template <int KIND>
__device__ __forceinline__ f32x16 wd_mfma(const u32x2 &a0, const u32x2 &a1,
                                          const u32x2 &b0, const u32x2 &b1,
                                          const f32x16 &c) {
  const u32x4 a = {a0.x, a0.y, a1.x, a1.y};
  const u32x4 b = {b0.x, b0.y, b1.x, b1.y};
  if constexpr (KIND == GK_BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(
        __builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(
        __builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Transposing LDS read: the 16 lanes of a group address a 4-pixel x 16-channel
// block (lane i: pixel i / 4, channels 4 * (i % 4) ..+3) and lane i receives
// channel i of the four pixels.  Written as asm so that the compiler does not
// tie it to the LDS-DMA loads in flight; wd_wait_lgkm says when the registers
// may be used.
template <int OFFSET>
__device__ __forceinline__ void wd_read_tr(u32x2 &dst, uint32_t addr) {
  static_assert(OFFSET >= 0 && OFFSET < 65536, "16-bit offset field");
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2"
               : "=v"(dst)
               : "v"(addr), "n"(OFFSET));
}

template <int N> __device__ __forceinline__ void wd_wait_lgkm() {
  static_assert(N >= 0 && N <= 15, "lgkmcnt is a 4-bit field");
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ void wd_pin(u32x2 &a) { asm volatile("" : "+v"(a)); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t wd_rsrc(const void *base,
                                                          uint32_t bytes) {
  const uint64_t b64 = (uint64_t)base;
  const uint32_t blo = __builtin_amdgcn_readfirstlane((uint32_t)b64);
  const uint32_t bhi = __builtin_amdgcn_readfirstlane((uint32_t)(b64 >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(
      (void *)(((uint64_t)bhi << 32) | blo), 0,
      (int)__builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}

template <int KIND, int NKS, bool PAD0>
__global__ __launch_bounds__(kWdThreads)
__attribute__((amdgpu_waves_per_eu(2, 2))) void
conv_wgrad_direct_kernel(WgDirectArgs g) {
  using R = WdRows<NKS>;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int l = threadIdx.x & 63;
  const int a_H = g.H, a_W = g.W;

  // Workgroup -> (part, block): a die's workgroups (every eighth) take the blocks of a part one
  // after another, which read the same rows of X and DY.
  const int lin = (int)(blockIdx.x & 7) * g.per_xcd + (int)(blockIdx.x >> 3);
  if (lin >= g.total)
    return;
  const int part = conv_div(lin, g.types, g.magic_types), type = lin - part * g.types;
  const int kb = conv_div(type, g.ctypes, g.magic_ctypes), cb = type - kb * g.ctypes;
  const int row0 = wd_share(g.rows, part, g.nparts), row1 = wd_share(g.rows, part + 1, g.nparts);
  const int first = row0 + (((row1 - row0) * wave) >> 3);
  const int last = row0 + (((row1 - row0) * (wave + 1)) >> 3);

  // A walk over rows [first, last) of X, cut into the images' runs.  Step t of a run
  // that starts at row p0 of its image brings DY row p0 + pad - 2 + t into registers and, from
  // t = 2 on, multiplies X row p0 + t - 2 with the three DY rows held: the newest is
  // filter row 0, the oldest filter row 2.
  struct Walk {
    int row, n, t; // the run's first row in X, its rows, the step
    int y, yrow;   // DY row of step 0 in its image and in the batch
  };
  const int img0 = conv_div(first, a_H, g.magic_h);
  auto begin = [&](int row, int p0, int img) __attribute__((always_inline)) {
    const int in_image = a_H - p0, left = last - row, y = p0 + g.pad - 2;
    return Walk{row, left < in_image ? left : in_image, 0, y, img * g.P + y};
  };
  auto next = [&](const Walk &w) __attribute__((always_inline)) {
    return begin(w.row + w.n, 0, conv_div(w.row, a_H, g.magic_h) + 1);
  };

  // ---- LDS-DMA lane offsets (relative to a row's first byte) --------------------
  // instruction j fills pixel slots 16 j .. 16 j + 15 of a row slice: lane d
  // carries 16 bytes (8 channels) d % 4 of slot 16 j + d / 4.  X slot t holds
  // image column t - pad (the slots outside the image are the zero
  // padding), DY slot t holds column t (zeros past the image); channels past C or K are zeros.
  uint32_t xrel[R::kX], yrel[R::kY];
#pragma unroll
  for (int j = 0; j < R::kX; ++j) {
    const int slot = 16 * j + (l >> 2);
    const int q = slot - g.pad;
    xrel[j] = (unsigned)q < (unsigned)a_W && cb * 32 + (l & 3) * 8 < g.C
                  ? (uint32_t)(q * g.C * 2 + cb * 64 + (l & 3) * 16)
                  : 0x80000000u;
    if (j < R::kY)
      yrel[j < R::kY ? j : 0] = slot < g.Q && kb * 32 + (l & 3) * 8 < g.K
                                    ? (uint32_t)(slot * g.K * 2 + kb * 64 + (l & 3) * 16)
                                    : 0x80000000u;
  }
  const __amdgpu_buffer_rsrc_t rx = wd_rsrc(g.x, g.x_bytes);
  const __amdgpu_buffer_rsrc_t ry = wd_rsrc(g.dy, g.dy_bytes);
  const __amdgpu_buffer_rsrc_t rnone = wd_rsrc(g.x, 0); // every lane reads zero
  const int x_pitch = a_W * g.C * 2, y_pitch = g.Q * g.K * 2;

  const uint32_t wbase = lds0 + (uint32_t)wave * kWdWaveLds;
  // fragment read address inside a row slice: lane l is MFMA row / column
  // l % 32 and K half l / 32 (pixels 8 h .. 8 h + 7 of the K-step)
  const uint32_t tbase = (uint32_t)(((l >> 5) * 8 + ((l & 15) >> 2)) * 64 +
                                    ((l >> 4) & 1) * 32 + (l & 3) * 8);
  // which of this lane's pixels of a row's last step exist (two to a register of X's fragments)
  uint32_t inside[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int q = 16 * (NKS - 1) + 8 * (l >> 5) + 2 * i;
    inside[i] = (q < g.Q ? 0xffffu : 0u) | (q + 1 < g.Q ? 0xffff0000u : 0u);
  }

  f32x16 acc[9];
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i)
      acc[t][i] = 0.f;

  if (first < last) {
    Walk ahead = begin(first, first - img0 * a_H, img0), now = ahead;
    // ring slots of the next loads and the next reads
    uint32_t put_x = 0, put_y = R::kYBase, get_x = 0, get_y = R::kYBase;
    auto turn = [](uint32_t &at, uint32_t by, uint32_t from, uint32_t to) __attribute__((always_inline)) {
      at = at + by == to ? from : at + by;
    };
    // the loads of a step, always kX + kY of them; rows outside the image, and all past the walk's
    // end, come from nowhere (DY rows of the neighbouring shares are real: they are this
    // share's halo)
    auto issue = [&]() __attribute__((always_inline)) {
      const bool live = ahead.n > 0;
      const bool y_ok = live && (unsigned)(ahead.y + ahead.t) < (unsigned)g.P, x_ok = live && ahead.t >= 2;
      const __amdgpu_buffer_rsrc_t ys = y_ok ? ry : rnone, xs = x_ok ? rx : rnone;
      const int y_off = y_ok ? (ahead.yrow + ahead.t) * y_pitch : 0;
      const int x_off = x_ok ? (ahead.row + ahead.t - 2) * x_pitch : 0;
#pragma unroll
      for (int j = 0; j < R::kX; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            xs, (GEMM_AS3 char *)__builtin_amdgcn_readfirstlane(wbase + put_x + j * 1024u), 16, (int)xrel[j], x_off,
            0, 0);
#pragma unroll
      for (int j = 0; j < R::kY; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            ys, (GEMM_AS3 char *)__builtin_amdgcn_readfirstlane(wbase + put_y + j * 1024u), 16, (int)yrel[j], y_off,
            0, 0);
      turn(put_x, R::kXBytes, 0, R::kYBase);
      turn(put_y, R::kYBytes, R::kYBase, R::kYBase + R::kD * R::kYBytes);
      if (live && ++ahead.t == ahead.n + 2)
        ahead = next(ahead);
    };
#pragma unroll
    for (int i = 0; i < R::kD; ++i)
      issue();

    // DY fragments of three rows: dyf[j] holds the row of a run's steps that are j modulo 3
    u32x2 dyf[3][NKS][2];
    auto read_y = [&](auto jc) __attribute__((always_inline)) {
      constexpr int J = decltype(jc)::value;
      const uint32_t ya = wbase + get_y + tbase;
      gemm_static_for<NKS>([&](auto kc) {
        constexpr int ks = decltype(kc)::value;
        wd_read_tr<ks * 1024>(dyf[J][ks][0], ya);
        wd_read_tr<ks * 1024 + 256>(dyf[J][ks][1], ya);
      });
    };
    // A step: its loads have landed when only those of the kD - 1 steps issued after it are
    // out.  Its DY row's slot, and the X slot of the step before, are free once the DY row
    // is in registers.
    auto light = [&](auto jc) __attribute__((always_inline)) {
      __builtin_amdgcn_s_waitcnt(gemm_wait_imm((R::kD - 1) * (R::kX + R::kY)));
      read_y(jc);
      turn(get_x, R::kXBytes, 0, R::kYBase);
      turn(get_y, R::kYBytes, R::kYBase, R::kYBase + R::kD * R::kYBytes);
      wd_wait_lgkm<0>();
      issue();
    };
    // `y`: the newest DY row in its image.  Filter rows whose DY row does not exist are left out, and so are
    // pixels past a row's end: an infinite X value would meet the zeros in their place (0 x inf).
    auto full = [&](auto jc, int y) __attribute__((always_inline)) {
      constexpr int J = decltype(jc)::value, J1 = (J + 2) % 3, J2 = (J + 1) % 3;
      __builtin_amdgcn_s_waitcnt(gemm_wait_imm((R::kD - 1) * (R::kX + R::kY)));
      read_y(jc);
      const uint32_t xa = wbase + get_x + tbase;
      turn(get_x, R::kXBytes, 0, R::kYBase);
      turn(get_y, R::kYBytes, R::kYBase, R::kYBase + R::kD * R::kYBytes);
      u32x2 xf[2][3][2];
      auto read_x = [&](auto kc) __attribute__((always_inline)) {
        constexpr int ks = decltype(kc)::value;
        gemm_static_for<3>([&](auto sc) {
          constexpr int s = decltype(sc)::value;
          wd_read_tr<ks * 1024 + s * 64>(xf[ks & 1][s][0], xa);
          wd_read_tr<ks * 1024 + s * 64 + 256>(xf[ks & 1][s][1], xa);
        });
      };
      read_x(std::integral_constant<int, 0>{});
      wd_wait_lgkm<6>();
      issue();
      // bit r: the DY row of filter row r, y - r, exists
      uint32_t rows = (y < 2 ? (2u << y) - 1 : 7u) & ~(y < g.P ? 0u : (2u << (y - g.P)) - 1);
      gemm_static_for<NKS>([&](auto kc) {
        constexpr int ks = decltype(kc)::value;
        if constexpr (ks + 1 < NKS) {
          read_x(std::integral_constant<int, ks + 1>{});
          wd_wait_lgkm<6>();
        } else {
          wd_wait_lgkm<0>();
        }
        u32x2(&xk)[3][2] = xf[ks & 1];
#pragma unroll
        for (int s = 0; s < 3; ++s) {
          wd_pin(xk[s][0]);
          wd_pin(xk[s][1]);
        }
        wd_pin(dyf[J][ks][0]);
        wd_pin(dyf[J][ks][1]);
        asm volatile("" : "+s"(rows)); // (a branch per filter row, not one path through all steps per combination)
        auto product = [&](int r, int s) __attribute__((always_inline)) {
          u32x2(&yk)[2] = dyf[r == 0 ? J : r == 1 ? J1 : J2][ks];
          acc[3 * r + s] = wd_mfma<KIND>(yk[0], yk[1], xk[s][0], xk[s][1], acc[3 * r + s]);
        };
        // Pixels past the row's end meet a column of X in the first tap (without padding in the second too); with
        // four steps the last two meet what lies behind X's slice in the other taps.
        auto blank = [&](int s, int from) __attribute__((always_inline)) {
          if constexpr (ks + 1 == NKS)
#pragma unroll
            for (int i = from; i < 4; ++i)
              xk[s][i >> 1][i & 1] &= inside[i];
        };
        blank(2, NKS == 4 ? 3 : 4);
        blank(1, PAD0 ? 0 : NKS == 4 ? 3 : 4);
        if constexpr (PAD0) {
          blank(0, 0);
          if (__builtin_expect(rows & 2u, 2u))
#pragma unroll
            for (int s = 0; s < 3; ++s)
              product(1, s);
        } else {
          // (the middle row's exists; the first tap is blanked in the shadow of the others' products)
          product(1, 2);
          product(1, 1);
          __builtin_amdgcn_sched_barrier(0);
          blank(0, 0);
          product(1, 0);
        }
#pragma unroll
        for (int r = 0; r < 3; r += 2)
          if (__builtin_expect(rows & (1u << r), 1u << r))
#pragma unroll
            for (int s = 0; s < 3; ++s)
              product(r, s);
      });
    };

    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    // (run by run, the products in a loop of their own: under a branch of one loop over all steps
    // the compiler copies the accumulators about and spills 440 to 880 registers)
    for (; now.n > 0; now = next(now)) {
      light(I0{});
      light(I1{});
      for (int left = now.n, y = now.y + 2;;) {
        full(I2{}, y++);
        if (--left == 0)
          break;
        full(I0{}, y++);
        if (--left == 0)
          break;
        full(I1{}, y++);
        if (--left == 0)
          break;
      }
    }
  }

  // ---- sum of the eight wavefronts through LDS, half of the block at a time ---
  // (the loads still in flight land before their slots hold sums)
  __builtin_amdgcn_s_waitcnt(gemm_wait_imm(0));
  __syncthreads();
  f32x4 *dst4 = (f32x4 *)(g.part + ((size_t)type * g.nparts + part) * kWdBlock);
  // entry e = 4 * tap + j is registers 4 j .. 4 j + 3 of a tap's accumulator:
  // one 16-byte LDS access per lane
  f32x4 *scr4 = (f32x4 *)smem; // [wavefront][18 entries][64 lanes]
  constexpr int kHalf = 18 * 64;
  gemm_static_for<2>([&](auto hc) {
    constexpr int h = decltype(hc)::value;
    gemm_static_for<18>([&](auto kc) {
      constexpr int k = decltype(kc)::value;
      constexpr int e = 18 * h + k, tap = e / 4, j = e % 4;
      const f32x4 v = {acc[tap][4 * j], acc[tap][4 * j + 1], acc[tap][4 * j + 2],
                       acc[tap][4 * j + 3]};
      scr4[(wave * 18 + k) * 64 + l] = v;
    });
    __syncthreads();
    for (int f = (int)threadIdx.x; f < kHalf; f += kWdThreads) {
      f32x4 sum = scr4[f];
#pragma unroll
      for (int v = 1; v < kWdWaves; ++v) {
        const f32x4 o = scr4[v * kHalf + f];
        sum[0] += o[0], sum[1] += o[1], sum[2] += o[2], sum[3] += o[3];
      }
      dst4[h * kHalf + f] = sum;
    }
    __syncthreads();
  });
}

struct WgDirectSumArgs {
  int32_t nparts, ctypes, C, K;
  int64_t sk, sc, sr, ss; // element strides of DW [K, C, R, S]
  int32_t dt;
};

// DW[k][c][r][s] = sum of the partial results of a (k, c) block's workgroups.
// 64 outputs per workgroup of 256 threads: thread (o, j) adds the partials
// j, j + 4, ... (all loads independent), the four sums are added in order.
// A partial block is [entry e = 4 * tap + i / 4][lane][i % 4].
__global__ __launch_bounds__(256) void
conv_wgrad_direct_sum_kernel(WgDirectSumArgs a, const float *part, void *dw) {
  // A workgroup adds 256 results: thread (o, j) the parts j, j + 4, ... of
  // four consecutive ones (16-byte loads; a wavefront reads 1 KB runs), then
  // the four j of a group meet in LDS, always in the same order.
  __shared__ f32x4 red[4][64];
  const int o = threadIdx.x & 63, j = threadIdx.x >> 6;
  const int64_t lin = ((int64_t)blockIdx.x * 64 + o) * 4;
  const int type = (int)(lin / kWdBlock);
  const int within = (int)(lin - (int64_t)type * kWdBlock);
  const float *src = part + (int64_t)type * a.nparts * kWdBlock + within;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  fhip_for_uniform_parts<8>(
      __builtin_amdgcn_readfirstlane(j), 4, a.nparts,
      [&](int p) { return *(const f32x4 *)(src + (int64_t)p * kWdBlock); }, [&](f32x4 v) { acc += v; });
  red[j][o] = acc;
  __syncthreads();
  if (j != 0)
    return;
  acc = ((red[0][o] + red[1][o]) + red[2][o]) + red[3][o];
  // within = [entry e = 4 * tap + i / 4][lane][i % 4]: the four values are i % 4 = 0 .. 3
  const int lane = (within >> 2) & 63, e = within >> 8;
  const int tap = e >> 2;
  const int kb = type / a.ctypes, cb = type - kb * a.ctypes;
  const int64_t c = cb * 32 + (lane & 31);
  const int r = tap / 3, sx = tap - r * 3;
  if (c >= a.C || kb * 32 + 8 * (e & 3) + 4 * (lane >> 5) >= a.K)
    return;
  const int64_t k = kb * 32 + 8 * (e & 3) + 4 * (lane >> 5);
  const float v[4] = {acc[0], acc[1], acc[2], acc[3]};
  fhip_store_float(dw, a.dt, k * a.sk + c * a.sc + r * a.sr + sx * a.ss, a.sk, v);
}

struct WgDirectPlan {
  bool ok = false;
  int kind = GK_BF16, nks = 4;
  WgDirectArgs a{};
  size_t contract = 0; // bytes of the caller's workspace
};

bool wd_channels_last(const fhip_tensor_desc &t) {
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

// `contract` is 0 for the problems that conv_wgrad.hip reports its workspace for.
WgDirectPlan make_wd_plan(const fhip_conv_desc *d) {
  WgDirectPlan p;
  const FhipKnobs &knobs = fhip_knobs();
  if (knobs.wgrad_direct == 0)
    return p;
  if (d->spatial_rank != 2)
    return p;
  const int dt = d->x.dtype;
  if (dt == FHIP_BFLOAT16)
    p.kind = GK_BF16;
  else if (dt == FHIP_HALF)
    p.kind = GK_F16;
  else
    return p;
  if (d->y.dtype != dt)
    return p;
  const int wdt = d->w.dtype;
  if (wdt != FHIP_BFLOAT16 && wdt != FHIP_HALF && wdt != FHIP_FLOAT)
    return p;
  const int64_t N = d->x.dim[0], C = d->x.dim[1], H = d->x.dim[2], W = d->x.dim[3];
  const int64_t K = d->w.dim[0], P = d->y.dim[2], Q = d->y.dim[3];
  if (d->w.dim[1] != C || d->w.dim[2] != 3 || d->w.dim[3] != 3)
    return p;
  for (int i = 0; i < 2; ++i)
    if (d->stride[i] != 1 || d->dilation[i] != 1 || d->padding[i] != d->padding[0] || d->padding[i] < 0 ||
        d->padding[i] > 2)
      return p;
  if (P != H + 2 * d->padding[0] - 2 || Q != W + 2 * d->padding[1] - 2 || d->y.dim[0] != N || d->y.dim[1] != K)
    return p;
  if (C % 8 != 0 || K % 8 != 0 || Q > kWdMaxW || Q < 1 || P < 1 || N < 1)
    return p;
  if (!wd_channels_last(d->x) || !wd_channels_last(d->y))
    return p;
  const int64_t x_bytes = N * H * W * C * 2, dy_bytes = N * P * Q * K * 2;
  if (x_bytes >= (1ll << 31) || dy_bytes >= (1ll << 31))
    return p;
  const int64_t types = ((C + 31) / 32) * ((K + 31) / 32);
  if (types > 4096)
    return p;
  WgDirectArgs &a = p.a;
  a.H = (int32_t)H, a.W = (int32_t)W, a.C = (int32_t)C, a.K = (int32_t)K;
  a.P = (int32_t)P, a.Q = (int32_t)Q;
  a.pad = (int32_t)d->padding[0];
  a.rows = (int32_t)(N * H);
  a.types = (int32_t)types, a.ctypes = (int32_t)((C + 31) / 32);
  a.magic_types = conv_magic(a.types), a.magic_ctypes = conv_magic(a.ctypes), a.magic_h = conv_magic(a.H);
  a.x_bytes = (uint32_t)x_bytes, a.dy_bytes = (uint32_t)dy_bytes;
  p.nks = (int)((Q + 15) / 16);
  p.ok = true;
  if (C % 32 != 0 || K % 32 != 0 || P != H || Q != W)
    return p;
  const int64_t cus = 256;
  // The caller's workspace: the partial sums of workgroups that take whole images, or row chunks
  // of one, a round of them and no fewer.  Saved plans hold its size and are taken only where they equal
  // the plan of today byte for byte (Graph::loadFromArtifact).
  int64_t chunks = 1, ipw = 1;
  if (types * N < cus) {
    chunks = (cus + types * N - 1) / (types * N);
    const int64_t most = (H + kWdWaves - 1) / kWdWaves;
    chunks = chunks < most ? chunks : most;
  } else {
    ipw = types * N / cus;
    ipw = ipw < 1 ? 1 : ipw;
  }
  const int64_t rpw = (H + 4 * chunks - 1) / (4 * chunks);
  chunks = (H + 4 * rpw - 1) / (4 * rpw);
  const int64_t igroups = (N + ipw - 1) / ipw;
  const int64_t whole = igroups * chunks;
  if (types * whole >= (1ll << 31) / kWdBlock || chunks > 65535 || igroups > 65535)
    return WgDirectPlan{};
  p.contract = (size_t)(types * whole) * kWdBlock * sizeof(float);
  return p;
}

// Workgroups per (k, c) block, `most` at most.  A compute unit holds one workgroup, so what
// counts is rounds times a round: 7.5 us of start and sums, 0.4 to 0.9 per row of a
// wavefront, and 15 ns a partial result (36 KB written and read).  Fitted to 17 layers with 2 to
// 1280 parts: 14 images of 24 x 24, 320 -> 480 (150 blocks) 43.9 us in one part, 41.4 in three,
// 54.0 in six; 14 x 14 x 14, 64 -> 192 (12) 11.6 in ten, 13.6 in 21, 21.8 in 42; 56 x 56 x 32, 64 -> 128
// (8) 28.1 in 16, 25.0 in 32, 35.0 in 64.  Shares of whole images took a round and a little
// more wherever the blocks do not divide 256 (those layers: 86.8, 22.3 and 24.9).
int wd_parts(const WgDirectArgs &a, int nks, int64_t most) {
  constexpr int64_t kCus = 256;
  const double row = nks == 1 ? 0.4 : nks == 2 ? 0.75 : nks == 3 ? 0.85 : 0.9;
  int64_t best = 1;
  double least = 0;
  for (const int quarters : {1, 2, 3, 4, 8, 12}) {
    int64_t parts = quarters * kCus / (4 * a.types);
    const int64_t useful = (a.rows + kWdWaves - 1) / kWdWaves;
    parts = parts < useful ? parts : useful;
    parts = parts < most ? parts : most;
    parts = parts < 1 ? 1 : parts;
    const int64_t deep = (a.rows + kWdWaves * parts - 1) / (kWdWaves * parts);
    const double us = (double)((parts * a.types + kCus - 1) / kCus) * (7.5 + row * (double)deep) +
                      0.015 * (double)(parts * a.types);
    if (quarters == 1 || us < least)
      least = us, best = parts;
  }
  return (int)best;
}

// Whether it replaces the gathered tiles of conv_wgrad.hip, which take these problems too.  On 58
// random layers of 8 to 64 images, 7 to 64 rows and 32 to 512 channels it is 1.2 to 1.4 times as fast, twice where their
// runs fall badly (N24 128 -> 144, 54 x 54 74.8 us, here 34.8; N37 448 -> 208, 8 x 31 55.4 / 28.0), but for small ones
// (N17 64 -> 80, 10 x 10 9.3 / 10.6; N30 176 -> 48, 7 x 7 10.9 / 11.9).  Gradients stored in f32 stay
// there: their chains of additions are shorter.
bool wd_pays(const WgDirectPlan &p, int w_dtype) {
  const WgDirectArgs &a = p.a;
  return w_dtype != FHIP_FLOAT && (double)a.C * a.K * ((double)a.rows / a.H * a.P * a.Q) >= 1.4e7;
}

template <int KIND, int NKS, bool PAD0> int wd_launch(fhip_ctx *ctx, const WgDirectArgs &a) {
  auto kernel = conv_wgrad_direct_kernel<KIND, NKS, PAD0>;
  static FhipOncePerDevice configured;
  if (!configured.done(ctx->device)) {
    FHIP_HIP_CHECK(ctx, hipFuncSetAttribute(
                            reinterpret_cast<const void *>(kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, kWdLds));
    configured.mark(ctx->device);
  }
  hipLaunchKernelGGL(kernel, dim3((unsigned)a.per_xcd * 8), dim3(kWdThreads), kWdLds, ctx->stream, a);
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  return 0;
}

template <int KIND, bool PAD0> int wd_launch(fhip_ctx *ctx, const WgDirectPlan &p) {
  return p.nks == 1   ? wd_launch<KIND, 1, PAD0>(ctx, p.a)
         : p.nks == 2 ? wd_launch<KIND, 2, PAD0>(ctx, p.a)
         : p.nks == 3 ? wd_launch<KIND, 3, PAD0>(ctx, p.a)
                      : wd_launch<KIND, 4, PAD0>(ctx, p.a);
}

} // namespace

bool fhip_fast_conv_wgrad_direct_applicable(const fhip_conv_desc *d,
                                            size_t *workspace_bytes) {
  const WgDirectPlan p = make_wd_plan(d);
  if (workspace_bytes)
    *workspace_bytes = p.contract;
  return p.ok && p.contract != 0;
}

int fhip_fast_conv_wgrad_direct(fhip_ctx *ctx, const fhip_conv_desc *d,
                                const void *dy, const void *x, void *dw,
                                void *workspace, size_t workspace_bytes, bool *handled) {
  // planned for 256 compute units whatever the device: the workspace size was
  // answered without one
  WgDirectPlan p = make_wd_plan(d);
  const bool ours = p.ok && p.contract != 0;
  *handled = false;
  if (!p.ok || (!ours && !wd_pays(p, d->w.dtype)))
    return 0;
  FHIP_REQUIRE(ctx, ((uintptr_t)workspace & 255) == 0 && ((uintptr_t)x & 15) == 0 &&
                        ((uintptr_t)dy & 15) == 0,
               "conv wgrad: workspace must be 256-byte and tensors 16-byte aligned");
  // As many parts as the descriptor's workspace holds at most (wd_parts would take more for 249 of 20 000
  // layers that this file reports the workspace for, at best 31 % faster by its estimate, and for 123 of 20 451 of
  // the gathered tiles', 9 %): graphs with workspaces of their own may run side by side, and nothing
  // depends on what the context has run before.  Without one, the context's scratch.
  constexpr size_t kBytes = kWdBlock * sizeof(float);
  const int64_t most = (1ll << 31) / kWdBlock / p.a.types, held = (int64_t)(workspace_bytes / kBytes) / p.a.types;
  if (workspace && held < 1)
    return 0;
  // Gradients stored in f32 show how long a wavefront's chain of additions is: all parts that the workspace has
  // (error against 64 bits, time: N14 320 -> 480, 24 x 24 in two parts 1.36e-7, 50.8 us, in one 1.87e-7, 44.4; N11
  // 288 -> 480, 29 x 29 in three 1.26e-7, 41.8, in one 2.05e-7, 41.3; N14 64 -> 192, 14 x 14 in 28 8.2e-8,
  // 19.5, in five 8.4e-8, 11.3).
  p.a.nparts = d->w.dtype == FHIP_FLOAT ? (int32_t)held : wd_parts(p.a, p.nks, workspace && held < most ? held : most);
  void *part = workspace;
  if (!workspace) {
    const size_t bytes = (size_t)p.a.types * p.a.nparts * kBytes;
    if (!fhip_ctx_scratch_ready(ctx, bytes))
      return 0;
    if (fhip_ctx_scratch(ctx, bytes, &part) != 0)
      return 1;
  }
  *handled = true;
  p.a.total = p.a.types * p.a.nparts;
  p.a.per_xcd = (p.a.total + 7) / 8;
  p.a.x = (const char *)x;
  p.a.dy = (const char *)dy;
  p.a.part = (float *)part;
  const bool pad0 = p.a.pad == 0, bf16 = p.kind == GK_BF16;
  if ((pad0 ? bf16 ? wd_launch<GK_BF16, true>(ctx, p) : wd_launch<GK_F16, true>(ctx, p)
       : bf16 ? wd_launch<GK_BF16, false>(ctx, p) : wd_launch<GK_F16, false>(ctx, p)) != 0)
    return 1;
  WgDirectSumArgs s;
  s.nparts = p.a.nparts, s.ctypes = p.a.ctypes, s.C = p.a.C, s.K = p.a.K;
  s.sk = d->w.dim[0] == 1 ? 0 : d->w.stride[0];
  s.sc = d->w.dim[1] == 1 ? 0 : d->w.stride[1];
  s.sr = d->w.dim[2] == 1 ? 0 : d->w.stride[2];
  s.ss = d->w.dim[3] == 1 ? 0 : d->w.stride[3];
  s.dt = d->w.dtype;
  const int64_t total = (int64_t)p.a.types * kWdBlock;
  hipLaunchKernelGGL(conv_wgrad_direct_sum_kernel, dim3((unsigned)(total / 256)),
                     dim3(256), 0, ctx->stream, s, (const float *)p.a.part, dw);
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  fhip_note_kernel(ctx, "conv_wgrad_direct steps=%d parts=%d", p.nks, p.a.nparts);
  return 0;
}

// Matrix products that the tiled GEMM (gemm_kernel.h) does not fit: few rows or
// columns, K that fills no 128-byte slice, rows that start on any element.
//
// What bounds them is the load path, not the matrix pipe: a compute unit takes one
// cache line of a load instruction per clock, whatever part of it is used, so the
// loads are made of whole 128-byte lines, and the wavefronts of a workgroup split K
// instead of sharing tiles: no barrier until their accumulators meet in LDS.  A
// workgroup owns a tile of 16 MT x 16 NT outputs; a wavefront walks its slices of K
// (128 bytes of a K-contiguous row) with the next U slices' loads in flight.
//
//   K-contiguous operand: eight rows x 128 bytes per load instruction (16 bytes a
//   lane, at element alignment), through a wavefront-private LDS region into the
//   fragment layout, with the row order and the chunk permutation of the tiled GEMM
//   that keep the 16-byte reads free of bank conflicts.  (Loading the fragments
//   straight from memory takes 16 half-used lines per instruction; N4096 K4096
//   bf16: M16 11.6 us against 10.7, M64 33.8 against 12.9.)  Rows past the edge
//   repeat the last one; in the last slice a chunk ends at K and is shifted down,
//   so zeros stand where K is over.
//   Other operand (K is the slow dim): lane l % 16 owns T neighbouring rows of the
//   operand (T tiles, interleaved), loads them for the K values of its block in
//   runs of T elements -- four K-rows of 16 T elements per instruction -- and
//   transposes the block in registers.
//
// Measured against the f32-MFMA tiles (16-bit, f32) and the one-thread-per-output
// kernel (8-bit) that took these products before: bf16 M16 N4096 K4096 273 -> 10.8
// us (B 33.5 MB: 3.1 TB/s), M1 217 -> 9.2, f16 M777 N1400 K1000 with bias and GELU
// 162 -> 18.8, fp8 M16 N4096 K4096 2266 -> 7.6, int8 M500 N2048 K1040 1148 -> 10.8,
// f32 256 x 256 x 512 11.3 -> 6.2.
//
// Where the tiles are few and K is long, K is also cut across workgroups: f32 (or
// int32) partial tiles in the context's scratch, added in a fixed order by
// gemm_direct_finish_kernel.
#ifndef FUSILLI_AMD_CSRC_GEMM_DIRECT_KERNEL_H
#define FUSILLI_AMD_CSRC_GEMM_DIRECT_KERNEL_H

#include "gemm_kernel.h"

enum { GK_F32 = 5 };

struct DirectArgs {
  const char *a, *b;
  char *out;
  void *partial; // [split][batch][tile][floats of a tile], or null
  int64_t a_ldb, b_ldb;     // bytes between rows (K-contiguous) or K-rows
  int64_t a_batch, b_batch; // elements
  int64_t o_sm, o_sn, o_batch;
  int32_t M, N, K;
  int32_t tiles_m, tiles_n;
  int32_t slices, splits; // of K; workgroups that share a tile's
  int32_t c_dt, o_dt;
  // fused chain of fast modes whose operands are scalars but for one at most (`lean_op`, -1:
  // none), which depends on the column alone
  int32_t lean, lean_op;
  DevEpilogue epi; // strides over (batch, m, n)
};

template <int KIND> struct DirectKind {
  static constexpr int ELEM = KIND == GK_F32 ? 4 : KIND == GK_BF16 || KIND == GK_F16 ? 2 : 1;
  static constexpr bool FP8 = KIND == GK_FP8E4M3 || KIND == GK_FP8E5M2;
  static constexpr int REGS = FP8 ? 8 : 4;     // of a fragment
  static constexpr int CE = REGS * 4 / ELEM;   // consecutive K elements of a lane
  static constexpr int KS = 4 * CE;            // K of a step (one MFMA, f32: four)
  static constexpr int SK = 128 / ELEM;        // K of a slice
  static constexpr int STEPS = SK / KS;        // steps of a slice: 2 (fp8: 1)
  using Acc = std::conditional_t<KIND == GK_I8, int, float>;
  typedef Acc Acc4 __attribute__((ext_vector_type(4)));
};

template <int KIND> struct DFrag {
  uint32_t r[DirectKind<KIND>::REGS];
};

template <int KIND>
__device__ __forceinline__ void direct_mfma(typename DirectKind<KIND>::Acc4 &c,
                                            const DFrag<KIND> &a, const DFrag<KIND> &b) {
  if constexpr (KIND == GK_F32) {
    // (K value e of every K block per instruction: both operands in the same order)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      c = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, a.r[e]),
                                               __builtin_bit_cast(float, b.r[e]), c, 0, 0, 0);
  } else {
    Frag<KIND> fa, fb;
#pragma unroll
    for (int i = 0; i < DirectKind<KIND>::REGS; ++i)
      fa.r[i] = a.r[i], fb.r[i] = b.r[i];
    mfma16<KIND>(c, fa, fb);
  }
}

// Unaligned global loads of 1 .. 16 bytes at a multiple of ALIGN.
template <int BYTES, int ALIGN> struct DirectLoad;
#define DIRECT_LOADS(ALIGN)                                                    \
  template <> struct DirectLoad<16, ALIGN> {                                   \
    typedef uint32_t type __attribute__((ext_vector_type(4), aligned(ALIGN))); \
  };                                                                           \
  template <> struct DirectLoad<8, ALIGN> {                                    \
    typedef uint32_t type __attribute__((ext_vector_type(2), aligned(ALIGN))); \
  };                                                                           \
  template <> struct DirectLoad<4, ALIGN> {                                    \
    typedef uint32_t type __attribute__((aligned(ALIGN)));                     \
  };
DIRECT_LOADS(4)
DIRECT_LOADS(2)
DIRECT_LOADS(1)
#undef DIRECT_LOADS
template <> struct DirectLoad<2, 2> {
  typedef uint16_t type;
};
template <> struct DirectLoad<2, 1> {
  typedef uint16_t type __attribute__((aligned(1)));
};
template <> struct DirectLoad<1, 1> {
  typedef uint8_t type;
};

// `n` bytes off the low end of 16, zeros from above (n >= 16: all zeros)
__device__ __forceinline__ u32x4 direct_shift16(u32x4 v, int n) {
  const uint64_t lo = (uint64_t)v.y << 32 | v.x, hi = (uint64_t)v.w << 32 | v.z;
  const int s = n * 8;
  uint64_t l, h;
  if (s < 64) {
    l = s == 0 ? lo : lo >> s | hi << (64 - s);
    h = hi >> s;
  } else {
    l = s < 128 ? hi >> (s - 64) : 0;
    h = 0;
  }
  return u32x4{(uint32_t)l, (uint32_t)(l >> 32), (uint32_t)h, (uint32_t)(h >> 32)};
}

// One operand of a workgroup's tile: T tiles of 16 rows.
template <int KIND, bool KC, int T> struct DirectOperand {
  using D = DirectKind<KIND>;
  static constexpr int ELEM = D::ELEM, CE = D::CE;
  static constexpr int PE = 16 / ELEM; // elements of a 16-byte chunk
  static constexpr int RUN = T * ELEM, RW = (RUN + 3) / 4; // other operand: bytes and registers of a run
  // registers of a slice on its way
  static constexpr int RAW = KC ? 8 * T : D::STEPS * CE * RW;
  static constexpr int LDS = KC ? 2048 * T : 0; // bytes per wavefront
  struct Raw {
    uint32_t r[RAW];
  };
  const char *base;    // uniform: the tile's first row at this wavefront's K
  int64_t slice_bytes; // per slice of K
  uint32_t off[KC ? 2 * T : 1];
  uint32_t ldb;        // K-rows: bytes between them
  int cut;             // K-rows: elements that a ragged edge's run starts early
  bool ragged;         // uniform
  uint32_t wr[KC ? 2 : 1], rd[KC ? D::REGS / 4 * D::STEPS : 1]; // LDS addresses

  __device__ __forceinline__ void setup(const char *p, int64_t ld_bytes, int row0, int rows,
                                        int64_t k0, uint32_t lds) {
    const int l = threadIdx.x & 63;
    ldb = (uint32_t)ld_bytes;
    if constexpr (KC) {
      base = p + (int64_t)row0 * ld_bytes + k0 * ELEM;
      slice_bytes = 128;
#pragma unroll
      for (int t = 0; t < 2 * T; ++t) {
        int r = row0 + t * 8 + (l >> 3);
        r = (r < rows ? r : rows - 1) - row0;
        off[t] = (uint32_t)r * ldb + (uint32_t)((l & 7) * 16);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) // the two halves of a 16-row tile
        wr[h] = lds + (uint32_t)((h * 8 + (l >> 3)) * 128 + (((l & 7) ^ kc_swz(h * 8 + (l >> 3))) << 4));
      const int r16 = Frag16Geom<GK_BF16>::row16(l & 15);
#pragma unroll
      for (int q = 0; q < D::REGS / 4 * D::STEPS; ++q) {
        // step q / (REGS / 4), piece q % (REGS / 4) of the lane's K block
        constexpr int P = D::REGS / 4;
        const int c = q / P * 4 * P + (l >> 4) * P + q % P;
        rd[q] = lds + (uint32_t)(r16 * 128 + ((c ^ kc_swz(r16)) << 4));
      }
    } else {
      // (a ragged tile's last run may start up to T - 1 rows in front of the tile:
      // offsets are unsigned, so they count from T rows in front of it)
      const int first = row0 < T ? 0 : row0 - T;
      base = p + (int64_t)first * ELEM + k0 * ld_bytes;
      slice_bytes = (int64_t)D::SK * ld_bytes;
      const int r = row0 + (l & 15) * T;
      const int rr = r + T <= rows ? r : rows - T; // (rows >= T)
      cut = r - rr;
      ragged = row0 + 16 * T > rows;
      off[0] = (uint32_t)(rr - first) * ELEM + (uint32_t)((l >> 4) * CE) * ldb;
    }
  }

  // Requests slice `s` (from this wavefront's first); TAIL: krem = K values left
  // from its start, less than a whole slice.
  template <bool TAIL> __device__ __forceinline__ void fetch(int s, int krem, Raw &raw) const {
    const char *p = base + s * slice_bytes;
    const int l = threadIdx.x & 63;
    if constexpr (KC) {
      typedef typename DirectLoad<16, ELEM>::type V;
#pragma unroll
      for (int t = 0; t < 2 * T; ++t) {
        u32x4 v;
        if constexpr (TAIL) {
          const int k = (l & 7) * PE;
          const int kk = k < krem - PE ? k : krem - PE; // (K >= PE)
          const V x = *(const GEMM_AS1 V *)(p + (int64_t)off[t] + (kk - k) * ELEM);
          v = direct_shift16(u32x4{x.x, x.y, x.z, x.w}, (k - kk) * ELEM);
        } else {
          const V x = *(const GEMM_AS1 V *)(p + off[t]);
          v = u32x4{x.x, x.y, x.z, x.w};
        }
        raw.r[4 * t] = v.x, raw.r[4 * t + 1] = v.y, raw.r[4 * t + 2] = v.z, raw.r[4 * t + 3] = v.w;
      }
    } else {
      typedef typename DirectLoad<RUN, ELEM>::type V;
#pragma unroll
      for (int u = 0; u < D::STEPS; ++u)
#pragma unroll
        for (int i = 0; i < CE; ++i) {
          const int kl = u * D::KS + i, k = (l >> 4) * CE + kl;
          const int kk = TAIL ? (k < krem ? k : krem - 1) - (l >> 4) * CE : kl;
          const V x = *(const GEMM_AS1 V *)(p + (int64_t)(off[0] + (uint32_t)kk * ldb));
          uint32_t *row = &raw.r[(u * CE + i) * RW];
          if constexpr (RW == 4)
            row[0] = x.x, row[1] = x.y, row[2] = x.z, row[3] = x.w;
          else if constexpr (RW == 2)
            row[0] = x.x, row[1] = x.y;
          else
            row[0] = x;
          if constexpr (TAIL) {
#pragma unroll
            for (int w = 0; w < RW; ++w)
              row[w] = k < krem ? row[w] : 0;
          }
        }
    }
  }

  // A fetched slice into LDS (K-contiguous), or a ragged edge's runs in place.
  __device__ __forceinline__ void stage(Raw &raw) const {
    if constexpr (KC) {
#pragma unroll
      for (int t = 0; t < 2 * T; ++t)
        *(GEMM_AS3 u32x4 *)(wr[t & 1] + (uint32_t)(t >> 1) * 2048u) =
            u32x4{raw.r[4 * t], raw.r[4 * t + 1], raw.r[4 * t + 2], raw.r[4 * t + 3]};
    } else if (ragged) {
      // the run ends at the last row: bring the wanted ones down
      const int n = cut * ELEM * 8;
#pragma unroll
      for (int i = 0; i < D::STEPS * CE; ++i) {
        uint32_t *row = &raw.r[i * RW];
        if constexpr (RW == 4) {
          const u32x4 v = direct_shift16(u32x4{row[0], row[1], row[2], row[3]}, cut * ELEM);
          row[0] = v.x, row[1] = v.y, row[2] = v.z, row[3] = v.w;
        } else if constexpr (RW == 2) {
          const uint64_t v = n < 64 ? ((uint64_t)row[1] << 32 | row[0]) >> n : 0;
          row[0] = (uint32_t)v, row[1] = (uint32_t)(v >> 32);
        } else {
          row[0] = n < 32 ? row[0] >> n : 0;
        }
      }
    }
  }

  // Fragments of step U of the staged slice.
  template <int U> __device__ __forceinline__ void get(const Raw &raw, DFrag<KIND> (&f)[T]) const {
    if constexpr (KC) {
      constexpr int P = D::REGS / 4;
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int q = 0; q < P; ++q) {
          const u32x4 v = *(const GEMM_AS3 u32x4 *)(rd[U * P + q] + (uint32_t)t * 2048u);
          f[t].r[4 * q] = v.x, f[t].r[4 * q + 1] = v.y;
          f[t].r[4 * q + 2] = v.z, f[t].r[4 * q + 3] = v.w;
        }
    } else {
      const uint32_t *row = &raw.r[U * CE * RW];
#pragma unroll
      for (int t = 0; t < T; ++t)
#pragma unroll
        for (int q = 0; q < D::REGS; ++q) {
          if constexpr (ELEM == 4) {
            f[t].r[q] = row[q * RW + t];
          } else if constexpr (ELEM == 2) {
            f[t].r[q] = __builtin_amdgcn_perm(row[(2 * q + 1) * RW + t / 2], row[2 * q * RW + t / 2],
                                              t & 1 ? 0x07060302u : 0x05040100u);
          } else {
            constexpr uint32_t kPair[4] = {0x0c0c0400u, 0x0c0c0501u, 0x0c0c0602u, 0x0c0c0703u};
            const uint32_t lo = __builtin_amdgcn_perm(row[(4 * q + 1) * RW], row[4 * q * RW], kPair[t & 3]);
            const uint32_t hi = __builtin_amdgcn_perm(row[(4 * q + 3) * RW], row[(4 * q + 2) * RW], kPair[t & 3]);
            f[t].r[q] = lo | hi << 16;
          }
        }
    }
  }
};

// Output coordinates of the four values of a lane's accumulator quad `q` (tile
// q / 64, lane q % 64): rows *m + r * (*dm), column *n.
template <bool A_KC, bool B_KC, int MT, int NT>
__device__ __forceinline__ void direct_coord(int q, int *m, int *dm, int *n) {
  const int l = q & 63, i = (q >> 6) / NT, j = (q >> 6) % NT;
  // (K-contiguous operands: lane i of a fragment holds tile row row16(i))
  const int g = l >> 4;
  *m = A_KC ? i * 16 + (g ^ (g >> 1)) * 4 : g * 4 * MT + i;
  *dm = A_KC ? 1 : MT;
  *n = B_KC ? j * 16 + Frag16Geom<GK_BF16>::row16(l & 15) : (l & 15) * NT + j;
}

// Finishes and stores N values of column n, value i at row rows[i] (all values of
// a thread together: a fused operand's loads are then one round trip, not one per
// four values -- a bias on 64 x 64 tiles cost 6 us).
template <typename Acc, int N>
__device__ __forceinline__ void direct_store(const DirectArgs &g, int64_t batch, const int (&row)[N], int n,
                                             const Acc (&acc)[N]) {
  if (n >= g.N)
    return;
  int64_t at[N], rows[N];
  uint32_t live = 0;
#pragma unroll
  for (int r = 0; r < N; ++r) {
    rows[r] = row[r] < g.M ? row[r] : g.M - 1;
    at[r] = batch * g.o_batch + (int64_t)n * g.o_sn + rows[r] * g.o_sm;
    live |= (uint32_t)(row[r] < g.M) << r;
  }
  if constexpr (std::is_same<Acc, int>::value) {
#pragma unroll
    for (int r = 0; r < N; ++r)
      if ((live >> r) & 1)
        ((GEMM_AS1 int32_t *)g.out)[at[r]] = acc[r];
  } else {
    float v[N];
#pragma unroll
    for (int r = 0; r < N; ++r)
      v[r] = acc[r];
    fhip_round_fast_vec<N>(g.c_dt, v);
    if (g.epi.count > 0) {
      const int64_t coord[3] = {batch, 0, n};
      fhip_apply_epilogue_many<float, N>(g.epi, v, coord, 1, rows);
    }
    if (g.o_dt == FHIP_FLOAT) {
#pragma unroll
      for (int r = 0; r < N; ++r)
        if ((live >> r) & 1)
          ((GEMM_AS1 float *)g.out)[at[r]] = v[r];
    } else if (g.o_dt == FHIP_BFLOAT16) {
#pragma unroll
      for (int r = 0; r < N; ++r)
        if ((live >> r) & 1)
          ((GEMM_AS1 __bf16 *)g.out)[at[r]] = (__bf16)v[r];
    } else {
#pragma unroll
      for (int r = 0; r < N; ++r)
        if ((live >> r) & 1)
          ((GEMM_AS1 _Float16 *)g.out)[at[r]] = (_Float16)v[r];
    }
  }
}

// (64 x 64 tiles leave two workgroups to a compute unit where 256 registers hold
// them without spills: M777 N1400 K1000 f16 33.6 -> 23.3 us)
template <int KIND, bool A_KC, bool B_KC, int MT, int NT, int U, int MAXW>
__global__ __launch_bounds__(MAXW * 64)
__attribute__((amdgpu_waves_per_eu(
    MAXW == 16 ? 4 : MAXW == 8 || (A_KC && (B_KC || DirectKind<KIND>::ELEM > 1)) ? 2 : 1, 8))) void gemm_direct_kernel(DirectArgs g) {
  using D = DirectKind<KIND>;
  using Acc = typename D::Acc;
  constexpr int F = MT * NT * 256; // values of a tile
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int waves = blockDim.x >> 6;
  const int l = threadIdx.x & 63;
  // column-major: workgroups that run side by side share the rows' operand
  const int tile_m = blockIdx.x % g.tiles_m, tile_n = blockIdx.x / g.tiles_m;
  const int64_t batch = blockIdx.z;
  const int m0 = tile_m * 16 * MT, n0 = tile_n * 16 * NT;
  // this wavefront's slices
  const int part = blockIdx.y * waves + wave, parts = g.splits * waves;
  const int s0 = (int)((int64_t)g.slices * part / parts);
  const int s1 = (int)((int64_t)g.slices * (part + 1) / parts);
  const bool tail = s1 == g.slices && s1 > s0 && g.K % D::SK != 0;
  using OA = DirectOperand<KIND, A_KC, MT>;
  using OB = DirectOperand<KIND, B_KC, NT>;
  // a wavefront's LDS: its operands' staging, then its accumulators
  constexpr int PRIVATE = OA::LDS + OB::LDS > F * 4 ? OA::LDS + OB::LDS : F * 4;
  const uint32_t lds0 = (uint32_t)(uintptr_t)smem + (uint32_t)wave * PRIVATE;
  OA oa;
  OB ob;
  oa.setup(g.a + batch * g.a_batch * D::ELEM, g.a_ldb, m0, g.M, (int64_t)s0 * D::SK, lds0);
  ob.setup(g.b + batch * g.b_batch * D::ELEM, g.b_ldb, n0, g.N, (int64_t)s0 * D::SK, lds0 + OA::LDS);
  typename D::Acc4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
      acc[i][j] = typename D::Acc4{0, 0, 0, 0};
  // One slice: to LDS / through the registers, `more` requests what replaces it,
  // then its products.  (The compiler keeps a wavefront's LDS accesses in order
  // across the empty asm; the hardware does so by itself.)
  auto spend = [&](typename OA::Raw &ra, typename OB::Raw &rb, auto &&more) {
    oa.stage(ra);
    ob.stage(rb);
    asm volatile("" ::: "memory");
    DFrag<KIND> fa[D::STEPS][MT], fb[D::STEPS][NT];
    gemm_static_for<D::STEPS>([&](auto uc) {
      constexpr int u = decltype(uc)::value;
      if constexpr (!A_KC)
        oa.template get<u>(ra, fa[u]);
      if constexpr (!B_KC)
        ob.template get<u>(rb, fb[u]);
    });
    more();
    __builtin_amdgcn_sched_barrier(0);
    gemm_static_for<D::STEPS>([&](auto uc) {
      constexpr int u = decltype(uc)::value;
      if constexpr (A_KC)
        oa.template get<u>(ra, fa[u]);
      if constexpr (B_KC)
        ob.template get<u>(rb, fb[u]);
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          direct_mfma<KIND>(acc[i][j], fa[u][i], fb[u][j]);
    });
    asm volatile("" ::: "memory");
  };
  const int full = s1 - s0 - (tail ? 1 : 0);
  // U slices requested ahead
  typename OA::Raw ra[U];
  typename OB::Raw rb[U];
  gemm_static_for<U>([&](auto uc) {
    constexpr int u = decltype(uc)::value;
    if (u < full) {
      ob.template fetch<false>(u, 0, rb[u]);
      oa.template fetch<false>(u, 0, ra[u]);
    }
  });
  __builtin_amdgcn_sched_barrier(0);
  for (int s = 0; s < full; s += U) {
    gemm_static_for<U>([&](auto uc) {
      constexpr int u = decltype(uc)::value;
      if (s + u < full)
        spend(ra[u], rb[u], [&] {
          if (s + u + U < full) {
            ob.template fetch<false>(s + u + U, 0, rb[u]);
            oa.template fetch<false>(s + u + U, 0, ra[u]);
          }
        });
    });
  }
  if (tail) {
    const int krem = g.K - (s1 - 1) * D::SK;
    ob.template fetch<true>(full, krem, rb[0]);
    oa.template fetch<true>(full, krem, ra[0]);
    spend(ra[0], rb[0], [] {});
  }
  // the wavefronts' accumulators meet in LDS
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
      *(GEMM_AS3 typename D::Acc4 *)(lds0 + (uint32_t)(((i * NT + j) * 64 + l) * 16)) = acc[i][j];
  __syncthreads();
  const GEMM_AS3 typename D::Acc4 *lds = (const GEMM_AS3 typename D::Acc4 *)(uint32_t)(uintptr_t)smem;
  // a thread's quads: one, or the four of a tile column (64 x 64 on 256 threads)
  constexpr int PER = MT * NT == 16 ? 4 : 1;
  static_assert(PER == 1 || NT == 4, "quads of a thread in one column");
  const int q0 = threadIdx.x;
  if (q0 >= F / 4 / PER)
    return;
  int row[PER * 4], n = 0;
  Acc vals[PER * 4];
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    const int q = q0 + e * 256;
    typename D::Acc4 v = lds[q];
    for (int w = 1; w < waves; ++w)
      v += lds[w * (PRIVATE / 16) + q];
    if (g.partial)
      ((GEMM_AS1 typename D::Acc4 *)g.partial)[(((int64_t)blockIdx.y * gridDim.z + batch) * gridDim.x + blockIdx.x) *
                                                   (F / 4) +
                                               q] = v;
    int m, dm;
    direct_coord<A_KC, B_KC, MT, NT>(q, &m, &dm, &n);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      row[e * 4 + r] = m0 + m + r * dm, vals[e * 4 + r] = v[r];
  }
  if (!g.partial)
    direct_store<Acc, PER * 4>(g, batch, row, n0 + n, vals);
}

// Adds the split parts of every tile in order and finishes as above.
template <typename Acc, bool A_KC, bool B_KC, int MT, int NT>
__global__ __launch_bounds__(64) void gemm_direct_finish_kernel(DirectArgs g) {
  typedef Acc Acc4 __attribute__((ext_vector_type(4)));
  constexpr int Q = MT * NT * 64;
  const int tile_m = blockIdx.x % g.tiles_m, tile_n = blockIdx.x / g.tiles_m;
  const int64_t batch = blockIdx.z;
  const int q = blockIdx.y * 64 + threadIdx.x;
  const GEMM_AS1 Acc4 *p = (const GEMM_AS1 Acc4 *)g.partial + (batch * gridDim.x + blockIdx.x) * Q + q;
  const int64_t stride = (int64_t)gridDim.z * gridDim.x * Q;
  Acc4 v = p[0];
  fhip_for_uniform_parts<4>(1, 1, g.splits, [&](int s) { return p[s * stride]; }, [&](Acc4 x) { v += x; });
  int m, dm, n;
  direct_coord<A_KC, B_KC, MT, NT>(q, &m, &dm, &n);
  m += tile_m * 16 * MT;
  const int row[4] = {m, m + dm, m + 2 * dm, m + 3 * dm};
  const Acc vals[4] = {v.x, v.y, v.z, v.w};
  direct_store<Acc, 4>(g, batch, row, tile_n * 16 * NT + n, vals);
}

// What the host decided about one call.
struct DirectPlan {
  bool ok = false;
  int kind = 0;
  bool a_kc = true, b_kc = true;
  int mt = 1, nt = 1, waves = 1;
  bool tile = false; // gemm_tile_kernel.h
};

template <int KIND, bool A_KC, bool B_KC, int MT, int NT, int U, int MAXW>
int direct_launch(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch) {
  using Acc = typename DirectKind<KIND>::Acc;
  constexpr int STAGE = DirectOperand<KIND, A_KC, MT>::LDS + DirectOperand<KIND, B_KC, NT>::LDS;
  constexpr int PRIVATE = STAGE > MT * NT * 1024 ? STAGE : MT * NT * 1024;
  static_assert(MAXW * PRIVATE <= 64 * 1024, "LDS without a raised limit");
  const dim3 grid((unsigned)(g.tiles_m * g.tiles_n), (unsigned)g.splits, (unsigned)batch);
  hipLaunchKernelGGL((gemm_direct_kernel<KIND, A_KC, B_KC, MT, NT, U, MAXW>), grid, dim3(p.waves * 64),
                     p.waves * PRIVATE, ctx->stream, g);
  if (g.splits > 1)
    hipLaunchKernelGGL((gemm_direct_finish_kernel<Acc, A_KC, B_KC, MT, NT>),
                       dim3(grid.x, MT * NT, grid.z), dim3(64), 0, ctx->stream, g);
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  return 0;
}

template <int KIND, bool A_KC, bool B_KC>
int direct_launch_shape(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch) {
  // Slices requested ahead: one tile of either operand leaves registers for more.
  constexpr bool KC2 = A_KC && B_KC;
  if (p.mt == 4)
    return direct_launch<KIND, A_KC, B_KC, 4, 4, 1, 4>(ctx, p, g, batch);
  if (p.mt == 2)
    return direct_launch<KIND, A_KC, B_KC, 2, B_KC ? 2 : 4, 1, 8>(ctx, p, g, batch);
  if constexpr (B_KC) {
    if (p.nt == 1)
      return direct_launch<KIND, A_KC, B_KC, 1, 1, KC2 ? 4 : 1, 16>(ctx, p, g, batch);
    return direct_launch<KIND, A_KC, B_KC, 1, 2, KC2 ? 2 : 1, 8>(ctx, p, g, batch);
  } else {
    return direct_launch<KIND, A_KC, B_KC, 1, 4, 1, 8>(ctx, p, g, batch);
  }
}

template <int KIND>
int direct_launch_kind(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch) {
  if (p.a_kc && p.b_kc)
    return direct_launch_shape<KIND, true, true>(ctx, p, g, batch);
  if (p.a_kc)
    return direct_launch_shape<KIND, true, false>(ctx, p, g, batch);
  if (p.b_kc)
    return direct_launch_shape<KIND, false, true>(ctx, p, g, batch);
  return direct_launch_shape<KIND, false, false>(ctx, p, g, batch);
}

int direct_launch_bf16(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch);
int direct_launch_f16(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch);
int direct_launch_i8(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch);
int direct_launch_fp8e4m3(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch);
int direct_launch_fp8e5m2(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch);
int direct_launch_f32(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch);

#endif // FUSILLI_AMD_CSRC_GEMM_DIRECT_KERNEL_H

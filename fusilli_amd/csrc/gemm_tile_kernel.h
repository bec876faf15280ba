// Matrix products on LDS tiles staged through registers: operands of any alignment, K
// that fills no 128-byte slice, tiles that are too few for the kernels of gemm_kernel.h.
//
// A workgroup owns a tile of 64 MT x 64 NT outputs.  TEAMS teams of four wavefronts share K: a
// team walks its slices of 128 bytes of K through two LDS stages of its own, the loads of the
// next U slices in registers, one barrier per slice; inside a team the wavefronts own 64 x 64
// outputs each and share a slice's K-steps.  The accumulators of all shares meet in LDS.
//
// What bounds a tile: a slice of 64 x 64 outputs alone on its compute unit takes 500 clocks,
// LDS writes (16 KB at 64 bytes a clock) and reads (16 KB at 128) and the barrier; deeper
// prefetch (U = 8) changes nothing.  Hence every byte is read from LDS as few times as a tile's
// shape allows (with 32 x 32 outputs a wavefront, each byte twice: 700 clocks), the next
// fragments' reads are issued before the products and everything else between them, and loads
// stand outside branches, where waits by count are exact (in one, 0.3 us a slice).  Where tiles
// are few, K is cut over teams first, which costs no memory traffic, then over workgroups.
// Registers, not LDS-DMA, bring the slices in: rows may start on any element, and what lies
// behind K, M or N is masked there.  (Fragments straight from memory, no LDS, every wavefront
// with slices of its own, are no faster on aligned rows and 3 to 10 times slower on odd ones.)
//
// us, before -> now: bf16 1024^3 11.8 -> 8.0 (tiled GEMM), with bias and GELU 18.8 -> 9.8; f16 777
// x 1400 x 1000 with both 18.9 -> 16.2 (direct kernel); bf16 132 x 2632 x 3392 35.8 -> 14.6; odd
// rows, bf16 4095 x 8191 x 2001 344 -> 228 (128 x 128 tiles, 589 TFLOP/s), 1177 x 2223 x 2160
// 44.2 -> 35.1, with B along K 55.1 -> 33.7.
//
//   K-contiguous operand: rows of 128 bytes, 16 bytes a lane, chunks permuted as in
//   gemm_kernel.h.  In the last slice a chunk ends at K and is shifted down, so zeros
//   stand where K is over.  Rows past the edge repeat the last one.
//   Other operand: K-rows of 64 MT (NT) elements, read back by the transposing LDS
//   reads.  In the last slice K-rows behind K are zeros; at a ragged edge a chunk ends at
//   the last row (column) and is shifted down.
#ifndef FUSILLI_AMD_CSRC_GEMM_TILE_KERNEL_H
#define FUSILLI_AMD_CSRC_GEMM_TILE_KERNEL_H

#include "gemm_direct_kernel.h"

// Chunk permutation of a 64-wide M/N-contiguous slice (the wider ones: nkc_pos): the
// K-rows whose banks coincide are two (16-bit) or four (8-bit) apart.
template <int ELEM, int RB> __device__ __forceinline__ int tile_pos(int k, int c) {
  if constexpr (ELEM == 2 && RB == 128)
    return c ^ ((k & 2) << 1);
  else if constexpr (ELEM == 1 && RB == 64)
    return c ^ ((k & 4) >> 1);
  else
    return nkc_pos<ELEM, RB, 0>(k, c);
}

// One operand of a workgroup's tile: ROWS rows, of which a wavefront's fragments take T
// tiles of 32, of STEPS of a slice's K-steps.
template <int KIND, bool KC, int ROWS, int T, int STEPS> struct TileOperand {
  using D = DirectKind<KIND>;
  static constexpr int ELEM = D::ELEM, PE = 16 / ELEM;
  static constexpr int BYTES = ROWS * 128;       // of a slice
  static constexpr int LOADS = BYTES / 16 / 256; // 16-byte chunks per thread
  static constexpr int RB = ROWS * ELEM;         // other operand: bytes per K-row
  static constexpr int CPR = KC ? 8 : RB / 16;   // chunks per LDS row
  static constexpr int STEP = 256 / CPR;         // LDS rows between a thread's chunks
  static constexpr int STEPB = KindTraits<KIND>::kStepBytes;
  static constexpr int KSTEPS = 128 / STEPB;
  static constexpr int CH = STEPB / 16, CHH = CH / 2;
  static constexpr int NADDR = KC ? STEPS * CHH : T;
  static constexpr int READS = T * CHH * (KC ? 1 : 2); // LDS reads of a step
  struct Raw {
    u32x4 v[LOADS];
  };
  const char *base;      // uniform: the tile's first row at K = 0
  int64_t slice_bytes;
  uint32_t off[KC ? LOADS : 1]; // of this thread's chunks
  uint32_t ldb;          // other operand: bytes between K-rows
  int k0, cut;           // first K-row of this thread; elements that a ragged edge's chunk starts early
  bool ragged;           // uniform
  uint32_t wr, rd[NADDR];

  // `t`: thread of the team; `lds`: the team's first stage of this operand.
  __device__ __forceinline__ void setup(const char *p, int64_t ld_bytes, int row0, int rows, int t, int tile0, int step0,
                                        uint32_t lds) {
    ldb = (uint32_t)ld_bytes;
    const int r = t / CPR, c = t % CPR;
    if constexpr (KC) {
      base = p + (int64_t)row0 * ld_bytes;
      slice_bytes = 128;
      k0 = c * PE, cut = 0, ragged = false;
#pragma unroll
      for (int j = 0; j < LOADS; ++j) {
        int row = row0 + r + j * STEP;
        row = (row < rows ? row : rows - 1) - row0;
        off[j] = (uint32_t)row * ldb + (uint32_t)(c * 16);
      }
    } else {
      // (rows >= PE; a chunk that starts early may start in front of the tile)
      const int first = row0 < PE ? 0 : row0 - PE;
      base = p + (int64_t)first * ELEM;
      slice_bytes = (int64_t)D::SK * ld_bytes;
      const int e = row0 + c * PE, ee = e + PE <= rows ? e : rows - PE;
      cut = e - ee;
      ragged = row0 + ROWS > rows;
      k0 = r;
      off[0] = (uint32_t)(ee - first) * ELEM + (uint32_t)r * ldb;
    }
    place(t, tile0, step0, lds);
  }

  // Where this thread's chunks go in LDS and its fragments come from.
  __device__ __forceinline__ void place(int t, int tile0, int step0, uint32_t lds) {
    const int l = t & 63;
    const int r = t / CPR, c = t % CPR;
    if constexpr (KC) {
      // (STEP is a multiple of 16: the permutation is the same in every load)
      static_assert(!KC || STEP % 16 == 0, "rows between a thread's chunks");
      wr = lds + (uint32_t)(r * 128 + ((c ^ kc_swz(r)) << 4));
      const int fr = tile0 * 32 + (l & 31), sw = kc_swz(l & 31);
#pragma unroll
      for (int s = 0; s < STEPS; ++s)
#pragma unroll
        for (int i = 0; i < CHH; ++i)
          rd[s * CHH + i] = lds + (uint32_t)(fr * 128 + ((((step0 + s) * CH + (l >> 5) * CHH + i) ^ sw) << 4));
    } else {
      static_assert(KC || STEP % 8 == 0, "the permutation is the same in every load");
      wr = lds + (uint32_t)(r * RB + tile_pos<ELEM, RB>(r, c) * 16);
      const int L = l & 15, h = (l >> 4) & 1;
      constexpr int KPL = STEPB / 2 / ELEM; // (a step is a multiple of the permutation's period)
      const int k = (l >> 5) * KPL + (ELEM == 2 ? L >> 2 : L >> 1);
#pragma unroll
      for (int i = 0; i < T; ++i) {
        const int cc = ELEM == 2 ? (tile0 + i) * 4 + h * 2 + ((L & 3) >> 1) : (tile0 + i) * 2 + h;
        rd[i] = lds + (uint32_t)((step0 * (STEPB / ELEM) + k) * RB + tile_pos<ELEM, RB>(k, cc) * 16 + (L & 1) * 8);
      }
    }
  }

  // Requests slice `s`; TAIL: `krem` values of K are left from its
  // start, fewer than a slice.
  template <bool TAIL> __device__ __forceinline__ void fetch(int s, int krem, Raw &raw) const {
    typedef typename DirectLoad<16, ELEM>::type V;
    const char *p = base + s * slice_bytes;
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      if constexpr (KC) {
        if constexpr (TAIL) {
          const int kk = k0 < krem - PE ? k0 : krem - PE; // (K >= PE: may lie in the slice before)
          const V x = *(const GEMM_AS1 V *)(p + ((int64_t)off[j] + (kk - k0) * ELEM));
          raw.v[j] = u32x4{x.x, x.y, x.z, x.w};
        } else {
          const V x = *(const GEMM_AS1 V *)(p + off[j]);
          raw.v[j] = u32x4{x.x, x.y, x.z, x.w};
        }
      } else {
        const int k = k0 + j * STEP;
        const int dk = TAIL ? (k < krem ? k : krem - 1) - k0 : j * STEP;
        const V x = *(const GEMM_AS1 V *)(p + ((int64_t)off[0] + (int64_t)dk * ldb));
        raw.v[j] = u32x4{x.x, x.y, x.z, x.w};
      }
    }
  }

  // A fetched slice into the stage `at` bytes behind the first, zeros behind K.
  template <bool TAIL = false> __device__ __forceinline__ void put(const Raw &raw, uint32_t at, int krem = 0) const {
#pragma unroll
    for (int j = 0; j < LOADS; ++j) {
      u32x4 v = raw.v[j];
      if constexpr (TAIL && KC)
        v = direct_shift16(v, (k0 - (k0 < krem - PE ? k0 : krem - PE)) * ELEM);
      if constexpr (TAIL && !KC)
        v = k0 + j * STEP < krem ? v : u32x4{0, 0, 0, 0};
      if constexpr (!KC)
        if (ragged)
          v = direct_shift16(v, cut * ELEM);
      *(GEMM_AS3 u32x4 *)(uintptr_t)(wr + at + (uint32_t)(j * STEP * (KC ? 128 : RB))) = v;
    }
  }

  // Fragments of the wavefront's step S.
  template <int S> __device__ __forceinline__ void get(uint32_t at, Frag<KIND> (&f)[T]) const {
#pragma unroll
    for (int i = 0; i < T; ++i) {
      if constexpr (KC) {
#pragma unroll
        for (int q = 0; q < CHH; ++q) {
          const u32x4 v = *(const GEMM_AS3 u32x4 *)(uintptr_t)(rd[S * CHH + q] + at + (uint32_t)(i * 32 * 128));
          f[i].r[4 * q] = v.x, f[i].r[4 * q + 1] = v.y, f[i].r[4 * q + 2] = v.z, f[i].r[4 * q + 3] = v.w;
        }
      } else {
        constexpr int KPL = STEPB / 2 / ELEM, RPK = ELEM == 2 ? 4 : 8;
        gemm_static_for<KPL / RPK>([&](auto rc) {
          constexpr int r = decltype(rc)::value;
          constexpr int OFF = (S * (STEPB / ELEM) + RPK * r) * RB;
          u32x2 w;
          if constexpr (ELEM == 2)
            w = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                              (GEMM_AS3 s16x4 *)(uintptr_t)(rd[i] + at + OFF)));
          else
            w = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                                              (GEMM_AS3 i32x2 *)(uintptr_t)(rd[i] + at + OFF)));
          f[i].r[2 * r] = w.x;
          f[i].r[2 * r + 1] = w.y;
        });
      }
    }
  }
};

// Order of a slice's last step: the next fragments' reads, then NM products with the NV LDS
// writes and NV loads of later slices between them.
template <int NM, int NR, int NV> __device__ __forceinline__ void tile_interleave() {
  __builtin_amdgcn_sched_group_barrier(0x100, NR, 0); // DS read
  gemm_static_for<NM>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); // MFMA
    constexpr int lo = 2 * NV * m / NM, hi = 2 * NV * (m + 1) / NM;
    constexpr int w = (hi < NV ? hi : NV) - (lo < NV ? lo : NV), v = hi - lo - w;
    if constexpr (w > 0)
      __builtin_amdgcn_sched_group_barrier(0x200, w, 0); // DS write
    if constexpr (v > 0)
      __builtin_amdgcn_sched_group_barrier(0x020, v, 0); // VMEM read
  });
}

// The operand of V columns of a fused chain whose one tensor operand depends on the column
// alone (`lean_op`): requested while the last slices are multiplied, widened when it is used.
template <int V> struct TileColumns {
  uint32_t raw[V];
  __device__ __forceinline__ void request(const DirectArgs &g, int n) {
    const DevEpiOp &o = g.epi.op[g.lean_op];
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const int64_t at = (int64_t)(n + i < g.N ? n + i : g.N - 1) * o.stride[2];
      if (o.operand_dtype == FHIP_FLOAT)
        raw[i] = ((const GEMM_AS1 uint32_t *)o.ptr)[at];
      else
        raw[i] = ((const GEMM_AS1 uint16_t *)o.ptr)[at];
    }
  }
  __device__ __forceinline__ void widen(int dt, float (&v)[V]) const {
#pragma unroll
    for (int i = 0; i < V; ++i)
      v[i] = dt == FHIP_FLOAT      ? __builtin_bit_cast(float, raw[i])
             : dt == FHIP_BFLOAT16 ? __builtin_bit_cast(float, raw[i] << 16)
                                   : (float)__builtin_bit_cast(_Float16, (uint16_t)raw[i]);
  }
};

// Finishes and stores the V values of columns n .. of row m, which starts at element `row` of
// OUT (-1: there is no such row).
template <typename Acc, int V, bool PLAIN = false>
__device__ __forceinline__ void tile_store(const DirectArgs &g, int64_t batch, int m, int64_t row, int n,
                                           const Acc (&acc)[V], const TileColumns<V> *lean = nullptr) {
  if (row < 0 || n >= g.N)
    return;
  const int live = g.N - n < V ? g.N - n : V;
  const int64_t at = row + (int64_t)n * g.o_sn;
  if constexpr (std::is_same<Acc, int>::value) {
    typedef int loose __attribute__((ext_vector_type(4), aligned(4)));
    GEMM_AS1 int32_t *out = (GEMM_AS1 int32_t *)g.out + at;
#pragma unroll
    for (int i = 0; i < V; i += 4) {
      if (live >= i + 4 && g.o_sn == 1) {
        *(GEMM_AS1 loose *)(out + i) = loose{acc[i], acc[i + 1], acc[i + 2], acc[i + 3]};
      } else {
#pragma unroll
        for (int k = i; k < i + 4; ++k)
          if (k < live)
            out[k * g.o_sn] = acc[k];
      }
    }
  } else {
    float v[V];
#pragma unroll
    for (int i = 0; i < V; ++i)
      v[i] = acc[i];
    fhip_round_fast_vec<V>(g.c_dt, v);
    if (PLAIN) { // (no fused chain)
    } else if (lean && g.lean) {
      for (int i = 0; i < g.epi.count; ++i) {
        const DevEpiOp &o = g.epi.op[i];
        if (o.kind == FHIP_OPERAND_NONE) {
          fhip_pw_fast_unary_vec<true, V>(o.mode, v, o.params.swish_beta, o.result_dtype != FHIP_FLOAT);
        } else {
          float w[V];
          if (i == g.lean_op) {
            lean->widen(o.operand_dtype, w);
          } else {
#pragma unroll
            for (int c = 0; c < V; ++c)
              w[c] = o.scalar;
          }
          fhip_pw_fast_binary_vec<V>(o.mode, o.acc_is_in1 != 0, v, w);
        }
        fhip_round_fast_vec<V>(o.result_dtype, v);
      }
    } else if (g.epi.count > 0) {
      const int64_t coord[3] = {batch, m, 0};
      int64_t cols[V];
#pragma unroll
      for (int i = 0; i < V; ++i)
        cols[i] = n + (i < live ? i : 0);
      fhip_apply_epilogue_many<float, V>(g.epi, v, coord, 2, cols);
    }
    // (whole runs of 16 bytes, or of the V columns, single values where the last one ends)
    if (g.o_dt == FHIP_FLOAT) {
      typedef float loose __attribute__((ext_vector_type(4), aligned(4)));
      GEMM_AS1 float *out = (GEMM_AS1 float *)g.out + at;
#pragma unroll
      for (int i = 0; i < V; i += 4) {
        if (live >= i + 4 && g.o_sn == 1) {
          *(GEMM_AS1 loose *)(out + i) = loose{v[i], v[i + 1], v[i + 2], v[i + 3]};
        } else {
#pragma unroll
          for (int k = i; k < i + 4; ++k)
            if (k < live)
              out[k * g.o_sn] = v[k];
        }
      }
    } else {
      constexpr int H = V < 8 ? V : 8;
      typedef uint16_t loose __attribute__((ext_vector_type(H), aligned(2)));
      GEMM_AS1 uint16_t *out = (GEMM_AS1 uint16_t *)g.out + at;
#pragma unroll
      for (int i = 0; i < V; i += H) {
        loose h;
#pragma unroll
        for (int k = 0; k < H; ++k)
          h[k] = g.o_dt == FHIP_BFLOAT16 ? __builtin_bit_cast(uint16_t, (__bf16)v[i + k])
                                         : __builtin_bit_cast(uint16_t, (_Float16)v[i + k]);
        if (live >= i + H && g.o_sn == 1) {
          *(GEMM_AS1 loose *)(out + i) = h;
        } else {
#pragma unroll
          for (int k = 0; k < H; ++k)
            if (i + k < live)
              out[(i + k) * g.o_sn] = h[k];
        }
      }
    }
  }
}

// Adds a tile's SUMS shares of K in LDS, finishes and stores it.
template <typename Acc, int V, int BM, int BN, int SUMS, int PITCH, int SUM, int THREADS, bool PLAIN, class Row>
__device__ __forceinline__ void tile_finish(const DirectArgs &g, uint32_t lds, uint32_t id, int64_t batch, int m0, int n0,
                                            const TileColumns<V> &columns, const Row &at_row) {
  typedef Acc Acc4 __attribute__((ext_vector_type(4)));
  constexpr int RUNS = BN / V; // runs of V columns in a row
#pragma clang loop unroll(disable)
  for (int e = threadIdx.x; e < BM * RUNS; e += THREADS) {
    const int row = e / RUNS, col = e % RUNS * V;
    Acc v[V];
#pragma unroll
    for (int q = 0; q < V; q += 4) {
      const GEMM_AS3 Acc4 *p = (const GEMM_AS3 Acc4 *)(uintptr_t)(lds + (uint32_t)((row * PITCH + col + q) * 4));
      Acc4 x = *p;
#pragma unroll
      for (int h = 1; h < SUMS; ++h)
        x += p[h * (SUM / 16)];
      v[q] = x.x, v[q + 1] = x.y, v[q + 2] = x.z, v[q + 3] = x.w;
    }
    tile_store<Acc, V, PLAIN>(g, batch, m0 + row, at_row(m0 + row), n0 + col, v, &columns);
  }
}

// The plain sums of a split product's tile: 16 bytes a lane, side by side (in runs of eight columns
// f16 605 x 296 x 3456 in five parts 10.8 us, so 10.4; of sixteen 11.3).
template <typename Acc, int BM, int BN, int SUMS, int PITCH, int SUM, int THREADS>
__device__ __forceinline__ void tile_part(const DirectArgs &g, uint32_t lds, uint32_t id, int64_t batch) {
  typedef Acc Acc4 __attribute__((ext_vector_type(4)));
  GEMM_AS1 Acc4 *to = (GEMM_AS1 Acc4 *)g.partial +
                      (((int64_t)blockIdx.y * gridDim.z + batch) * gridDim.x + id) * (BM * BN / 4);
#pragma unroll 4
  for (int e = threadIdx.x; e < BM * BN / 4; e += THREADS) {
    const GEMM_AS3 Acc4 *p =
        (const GEMM_AS3 Acc4 *)(uintptr_t)(lds + (uint32_t)((e / (BN / 4) * PITCH + e % (BN / 4) * 4) * 4));
    Acc4 x = *p;
#pragma unroll
    for (int h = 1; h < SUMS; ++h)
      x += p[h * (SUM / 16)];
    to[e] = x;
  }
}

// Wavefronts of a team own 64 x 64 outputs each and share the slice's K-steps where the tile
// is smaller than four of those, so that few bytes of a stage are read twice (fp8 has two
// K-steps only: 64 x 64 tiles, 64 x 32 outputs each).
// SHORT (64 x 64 tiles): a quarter of the tile each, every byte read twice, for reductions that
// are over before it shows: no shares to add, and half the registers.
template <int KIND, int MT, int NT, int TEAMS_, bool SHORT = false> struct TileShape {
  static constexpr int BM = 64 * MT, BN = 64 * NT, TEAMS = TEAMS_;
  static constexpr int WK = SHORT ? 1 : KindTraits<KIND>::kStepBytes == 64 && MT * NT == 1 ? 2 : 4 / (MT * NT);
  static constexpr int WM = SHORT ? 2 : MT, WN = 4 / WK / WM;
  static constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  static constexpr int STEPS = 128 / KindTraits<KIND>::kStepBytes / WK;
  static constexpr int kStage = (BM + BN) * 128;    // a slice of both operands
  static constexpr int kPitch = BN + 4;             // values of a result row in LDS
  static constexpr int kSum = BM * kPitch * 4;      // the accumulators of wavefronts with one share of K
  static constexpr int kSums = WK * TEAMS;
  static constexpr int kLds = TEAMS * 2 * kStage > kSums * kSum ? TEAMS * 2 * kStage : kSums * kSum;
  // Columns of a row that a thread finishes at once: the chain's loads and branches take a
  // wavefront on its own 0.8 us a run, 0.15 more a column (bias and GELU on 64 x 64 tiles of four
  // wavefronts: four runs of four 5.4 us, two of eight 3.9), so one run of sixteen where there are
  // as many: bf16 3050 x 512 x 384 11.1 -> 10.2 us, fp8 1536 x 2560 x 6192 41.1 -> 39.2.
  // Whole numbers have no chain, and 16 of them are 64 bytes a lane: i8 896 x 1792 x 1408 on 128 x 64
  // tiles 10.4 us, with eight 9.2, with four 9.35; 128 x 7552 x 1280 on 64 x 64 ones with eight 8.05, with four 7.75.
  static constexpr int V = KIND == GK_I8 ? (BM * BN / (256 * TEAMS) >= 32 ? 8 : 4)
                           : BM * BN / (256 * TEAMS) >= 16 ? 16
                           : BM * BN / (256 * TEAMS) >= 8  ? 8
                                                           : 4;
};

// The share of K of a team: its whole slices, and how many the longest team of the workgroup
// has; where K ends inside a slice, the last team of the last part takes that one first.
struct TilePart {
  int whole, krem, s0, count, longest;
  bool cut, cut_mine; // (`cut`: uniform over the workgroup)
  __device__ __forceinline__ TilePart(int whole_, int krem_, int splits, int teams, int team) : whole(whole_), krem(krem_) {
    const int parts = splits * teams, part = blockIdx.y * teams + team;
    s0 = (int)((int64_t)whole * part / parts);
    count = (int)((int64_t)whole * (part + 1) / parts) - s0;
    longest = (whole + parts - 1) / parts;
    cut = krem > 0 && (int)blockIdx.y == splits - 1;
    cut_mine = cut && team == teams - 1;
  }
};

// A team's wavefront: which share of a slice's K-steps, rows and columns it has.
template <class S> struct TileWave {
  int team, wk, wn, wm;
  __device__ __forceinline__ TileWave() {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), w = wave & 3;
    team = wave >> 2;
    wk = w % S::WK, wn = w / S::WK % S::WN, wm = w / (S::WK * S::WN);
  }
};

// (workgroups go to the eight L2 slices in turn: each slice gets a run of neighbouring tiles)
__device__ __forceinline__ uint32_t tile_id() {
  const uint32_t id = blockIdx.x, per = gridDim.x / 8, rest = gridDim.x % 8, slice = id % 8;
  return slice * per + (slice < rest ? slice : rest) + id / 8;
}

// The tile at (m0, n0) whose operands are set up; `at_row(m)`: where row m of OUT starts, -1
// behind the last.  PLAIN: no fused chain.
template <int KIND, class S, int U, bool CUT, bool PLAIN, class OA, class OB, class Row>
__device__ __forceinline__ void tile_run(const DirectArgs &g, uint32_t smem, const TilePart &p, const TileWave<S> &at, OA &oa,
                                         OB &ob, uint32_t id, int64_t batch, int m0, int n0, const Row &at_row) {
  using Acc = typename DirectKind<KIND>::Acc;
  constexpr int BM = S::BM, BN = S::BN, TM = S::TM, TN = S::TN, TEAMS = S::TEAMS;
  const int team = at.team, wk = at.wk, wn = at.wn, wm = at.wm, l = threadIdx.x & 63;
  const int s0 = p.s0, count = p.count, longest = p.longest;
  typename KindTraits<KIND>::AccVec acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        acc[i][j][r] = 0;
  static_assert(U % 2 == 0, "slices alternate between two stages");
  typename OA::Raw ra[U];
  typename OB::Raw rb[U];
  Frag<KIND> fa[2][TM], fb[2][TN]; // of two steps in a row
  auto read = [&](auto kc, uint32_t at, auto set) {
    constexpr int ks = decltype(kc)::value, f = decltype(set)::value;
    oa.template get<ks>(at, fa[f]);
    ob.template get<ks>(at, fb[f]);
  };
  auto product = [&](auto set) {
    constexpr int f = decltype(set)::value;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
        mfma32<KIND>(acc[i][j], fa[f][i], fb[f][j]);
  };
  auto meet = [&] {
    __builtin_amdgcn_s_waitcnt(gemm_wait_imm(63));
    gemm_barrier();
  };
  typename OA::Raw ca;
  typename OB::Raw cb;
  if constexpr (CUT) {
    if (p.cut_mine) {
      oa.template fetch<true>(p.whole, p.krem, ca);
      ob.template fetch<true>(p.whole, p.krem, cb);
    }
  }
  // Loads of whole slices stand outside every branch: where control flow joins, the compiler
  // can only wait for all loads in flight, and the slices ahead would be waited for with the
  // one that is due.  Behind a team's last slice (and for a team without any) they repeat one.
  auto fetch = [&](int s, typename OA::Raw &va, typename OB::Raw &vb) {
    const int last = s0 + (count > 0 ? count - 1 : 0);
    int at = s0 + s;
    at = at < last ? at : last;
    at = at < p.whole ? at : p.whole - 1;
    oa.template fetch<false>(at, 0, va);
    ob.template fetch<false>(at, 0, vb);
  };
  if (longest > 0)
    gemm_static_for<U>([&](auto uc) {
      constexpr int u = decltype(uc)::value;
      fetch(u, ra[u], rb[u]);
      __builtin_amdgcn_sched_barrier(0); // (in order: so are the waits)
    });
  using C0 = std::integral_constant<int, 0>;
  if (longest > 0) {
    oa.put(ra[0], 0);
    ob.put(rb[0], 0);
    fetch(U, ra[0], rb[0]);
  }
  if constexpr (CUT) {
    if (p.cut_mine) {
      oa.template put<true>(ca, S::kStage, p.krem);
      ob.template put<true>(cb, S::kStage, p.krem);
    }
  }
  meet();
  if constexpr (CUT) {
    if (p.cut) {
      if (p.cut_mine)
        gemm_static_for<S::STEPS>([&](auto kc) {
          read(kc, S::kStage, C0{});
          product(C0{});
        });
      meet(); // (the second stage is free again)
    }
  }
  // One barrier per slice.  In front of it the last fragments of slice s are read and the
  // products but the last step's are under way; behind it the first fragments of slice s + 1
  // are read, slice s + 2 goes to the stage of slice s, and the last products cover both.
  if (longest > 0) {
    read(C0{}, 0, C0{});
    oa.put(ra[1], S::kStage);
    ob.put(rb[1], S::kStage);
    fetch(1 + U, ra[1], rb[1]);
  }
  auto steps = [&](auto uc) { // of slice s + u, but the last one
    constexpr int u = decltype(uc)::value;
    gemm_static_for<S::STEPS - 1>([&](auto kc) {
      constexpr int ks = decltype(kc)::value, f = (u * S::STEPS + ks) & 1;
      read(std::integral_constant<int, ks + 1>{}, (u & 1) * S::kStage, std::integral_constant<int, f ^ 1>{});
      product(std::integral_constant<int, f>{});
    });
  };
  int s = 0;
  for (; s + U < longest; s += U) { // (shorter teams end at `longest` - 1)
    gemm_static_for<U>([&](auto uc) {
      constexpr int u = decltype(uc)::value, n = (u + 2) % U;
      constexpr int last = ((u + 1) * S::STEPS - 1) & 1;
      steps(uc);
      meet();
      read(C0{}, ((u + 1) & 1) * S::kStage, std::integral_constant<int, last ^ 1>{});
      oa.put(ra[n], (u & 1) * S::kStage);
      ob.put(rb[n], (u & 1) * S::kStage);
      fetch(s + u + 2 + U, ra[n], rb[n]);
      product(std::integral_constant<int, last>{});
      // (reads first: the next products wait for them; writes and requests between the products)
      tile_interleave<TM * TN, OA::READS + OB::READS, OA::LOADS + OB::LOADS>();
    });
  }
  // (a thread finishes the same columns of several rows)
  static_assert(256 * TEAMS % (BN / S::V) == 0, "columns of a thread");
  TileColumns<S::V> columns;
  if (!PLAIN && g.lean && g.lean_op >= 0 && !g.partial)
    columns.request(g, n0 + (int)(threadIdx.x % (BN / S::V)) * S::V);
  gemm_static_for<U>([&](auto uc) {
    constexpr int u = decltype(uc)::value, n = (u + 2) % U;
    constexpr int last = ((u + 1) * S::STEPS - 1) & 1;
    if (s + u < longest) { // (uniform over the workgroup)
      if (s + u < count)
        steps(uc);
      meet();
      if (s + u + 1 < longest)
        read(C0{}, ((u + 1) & 1) * S::kStage, std::integral_constant<int, last ^ 1>{});
      if (s + u + 2 < longest) {
        oa.put(ra[n], (u & 1) * S::kStage);
        ob.put(rb[n], (u & 1) * S::kStage);
      }
      if (s + u < count)
        product(std::integral_constant<int, last>{});
    }
  });
  // ---- the accumulators of all shares of K meet in LDS: value r of a lane is row 8 (r / 4) +
  // 4 (l / 32) + r % 4 of its 32 x 32 tile, column l % 32
  __syncthreads();
  {
    GEMM_AS3 Acc *mine = (GEMM_AS3 Acc *)(uintptr_t)(smem + (uint32_t)((team * S::WK + wk) * S::kSum));
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          mine[((wm * TM + i) * 32 + 8 * (r >> 2) + 4 * (l >> 5) + (r & 3)) * S::kPitch + (wn * TN + j) * 32 +
               (l & 31)] = acc[i][j][r];
  }
  __syncthreads();
  if (g.partial) {
    tile_part<Acc, BM, BN, S::kSums, S::kPitch, S::kSum, 256 * TEAMS>(g, smem, id, batch);
    return;
  }
  tile_finish<Acc, S::V, BM, BN, S::kSums, S::kPitch, S::kSum, 256 * TEAMS, PLAIN>(g, smem, id, batch, m0, n0, columns,
                                                                                  at_row);
}

template <int KIND, bool A_KC, bool B_KC, int MT, int NT, int TEAMS, int U>
__global__ __launch_bounds__(256 * TEAMS)
__attribute__((amdgpu_waves_per_eu(2, 8))) void gemm_tile_kernel(DirectArgs g) {
  using D = DirectKind<KIND>;
  using S = TileShape<KIND, MT, NT, TEAMS>;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const TileWave<S> at;
  const int t = threadIdx.x & 255;
  const uint32_t id = tile_id(); // (column after column)
  const int tile_m = id % (uint32_t)g.tiles_m, tile_n = id / (uint32_t)g.tiles_m;
  const int64_t batch = blockIdx.z;
  const int m0 = tile_m * S::BM, n0 = tile_n * S::BN;
  const int whole = g.K / D::SK;
  const TilePart p(whole, g.K - whole * D::SK, g.splits, TEAMS, at.team);
  using OA = TileOperand<KIND, A_KC, S::BM, S::TM, S::STEPS>;
  using OB = TileOperand<KIND, B_KC, S::BN, S::TN, S::STEPS>;
  const uint32_t lds = (uint32_t)(uintptr_t)smem + (uint32_t)(at.team * 2 * S::kStage);
  OA oa;
  OB ob;
  oa.setup(g.a + batch * g.a_batch * D::ELEM, g.a_ldb, m0, g.M, t, at.wm * S::TM, at.wk * S::STEPS, lds);
  ob.setup(g.b + batch * g.b_batch * D::ELEM, g.b_ldb, n0, g.N, t, at.wn * S::TN, at.wk * S::STEPS, lds + OA::BYTES);
  tile_run<KIND, S, U, true, false>(
      g, (uint32_t)(uintptr_t)smem, p, at, oa, ob, id, batch, m0, n0,
      [&](int m) { return m < g.M ? batch * g.o_batch + (int64_t)m * g.o_sm : (int64_t)-1; });
}

// Adds the split parts of every tile in order and finishes as above: four columns a thread.
template <typename Acc, int BM, int BN, bool BY_ROWS = false>
__global__ __launch_bounds__(256) void gemm_tile_finish_kernel(DirectArgs g) {
  typedef Acc Acc4 __attribute__((ext_vector_type(4)));
  const uint32_t run = (uint32_t)(BY_ROWS ? g.tiles_n : g.tiles_m); // tiles one after another, row by row or down a column
  const int along = blockIdx.x % run, over = blockIdx.x / run;
  const int tile_m = BY_ROWS ? over : along, tile_n = BY_ROWS ? along : over;
  const int64_t batch = blockIdx.z;
  const int q = blockIdx.y * 256 + threadIdx.x;
  TileColumns<4> columns;
  if (g.lean && g.lean_op >= 0)
    columns.request(g, tile_n * BN + q % (BN / 4) * 4);
  const GEMM_AS1 Acc4 *p = (const GEMM_AS1 Acc4 *)g.partial + (batch * gridDim.x + blockIdx.x) * (BM * BN / 4) + q;
  const int64_t stride = (int64_t)gridDim.z * gridDim.x * (BM * BN / 4);
  Acc4 x = p[0];
  fhip_for_uniform_parts<4>(1, 1, g.splits, [&](int s) { return p[s * stride]; }, [&](Acc4 v) { x += v; });
  const Acc v[4] = {x.x, x.y, x.z, x.w};
  const int m = tile_m * BM + q / (BN / 4);
  tile_store<Acc, 4>(g, batch, m, m < g.M ? batch * g.o_batch + (int64_t)m * g.o_sm : -1, tile_n * BN + q % (BN / 4) * 4, v,
                   &columns);
}

template <int KIND, bool A_KC, bool B_KC, int MT, int NT, int TEAMS, int U>
int tile_launch(fhip_ctx *ctx, const DirectArgs &g, int64_t batch) {
  using S = TileShape<KIND, MT, NT, TEAMS>;
  auto kernel = gemm_tile_kernel<KIND, A_KC, B_KC, MT, NT, TEAMS, U>;
  static FhipOncePerDevice configured;
  if (S::kLds > 64 * 1024 && !configured.done(ctx->device)) {
    FHIP_HIP_CHECK(ctx, hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, S::kLds));
    configured.mark(ctx->device);
  }
  const dim3 grid((unsigned)(g.tiles_m * g.tiles_n), (unsigned)g.splits, (unsigned)batch);
  hipLaunchKernelGGL(kernel, grid, dim3(256 * TEAMS), S::kLds, ctx->stream, g);
  if (g.splits > 1)
    hipLaunchKernelGGL((gemm_tile_finish_kernel<typename DirectKind<KIND>::Acc, S::BM, S::BN>),
                       dim3(grid.x, S::BM * S::BN / 1024, grid.z), dim3(256), 0, ctx->stream, g);
  FHIP_HIP_CHECK(ctx, hipGetLastError());
  return 0;
}

// Tiles of 16 `mt` x 16 `nt`, of 64 or 128; `waves` / 4 teams.
template <int KIND, bool A_KC, bool B_KC>
int tile_launch_shape(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch) {
  if (p.mt == 8 && p.nt == 8)
    return tile_launch<KIND, A_KC, B_KC, 2, 2, 1, 2>(ctx, g, batch);
  if (p.mt == 8)
    return tile_launch<KIND, A_KC, B_KC, 2, 1, 1, 4>(ctx, g, batch);
  if (p.nt == 8)
    return tile_launch<KIND, A_KC, B_KC, 1, 2, 1, 4>(ctx, g, batch);
  if (p.waves == 8)
    return tile_launch<KIND, A_KC, B_KC, 1, 1, 2, 2>(ctx, g, batch);
  return tile_launch<KIND, A_KC, B_KC, 1, 1, 1, 4>(ctx, g, batch);
}

template <int KIND>
int tile_launch_kind(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch) {
  if (p.a_kc && p.b_kc)
    return tile_launch_shape<KIND, true, true>(ctx, p, g, batch);
  if (p.a_kc)
    return tile_launch_shape<KIND, true, false>(ctx, p, g, batch);
  if (p.b_kc)
    return tile_launch_shape<KIND, false, true>(ctx, p, g, batch);
  return tile_launch_shape<KIND, false, false>(ctx, p, g, batch);
}

int tile_launch_bf16(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch);
int tile_launch_f16(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch);
int tile_launch_i8(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch);
int tile_launch_fp8e4m3(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch);
int tile_launch_fp8e5m2(fhip_ctx *ctx, const DirectPlan &p, const DirectArgs &g, int64_t batch);

#endif // FUSILLI_AMD_CSRC_GEMM_TILE_KERNEL_H

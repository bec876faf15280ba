// Attention forward for few query rows per key / value head (decode, short query
// blocks): the keys are split over workgroups and wavefronts.
//
// Bound by reading K and V once.  The tiled kernel (sdpa_fwd.hip) gives a workgroup
// 256 query rows and all keys of a head: with one row it multiplies 255 rows of
// padding, reads K and V once per query head, and fills one workgroup per head.
// Here the query rows that share a key / value head -- grouped heads times
// positions -- are packed into tiles of 16 rows; a wavefront walks chunks of 32
// keys with the next chunk's K and V in flight and keeps everything of a query row
// in the lanes l % 16:
//   * S^T = K Q^T on 16 x 16 x 32 MFMAs, K fragments straight from memory; a lane
//     ends up with 8 keys of one query;
//   * online softmax in those lanes (two exchanges over the four 16-lane groups);
//     the probabilities, rounded to the input type, are the operand of the next
//     product as they lie, with the chunk's keys in the order the lanes hold them;
//   * O^T += V^T P^T, where a lane loads T = HD / 16 neighbouring columns of the 8
//     V rows that match its keys and transposes the block in registers.
// The wavefronts' sums meet in LDS, the workgroups' (m, l, O) parts in the
// context's scratch, combined in a fixed order by a second kernel.
//
// B8, 32 query heads on 8 key / value heads, 4000 keys, D128 bf16 (131 MB): 110 us
// on the tiled kernel -> 30.4 (4.3 TB/s); B1 11.7 us of 81.6; one query block of 1024
// under a causal mask, 8 heads, D128: 37.3 -> 21.3.
//
// Reference semantics as in sdpa_fwd.hip.
#include "common.h"
#include "fast_paths.h"

#include <cmath>
#include <type_traits>

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
#define SD_AS1 __attribute__((address_space(1)))

constexpr int kWaves = 4;
constexpr int kChunk = 32; // keys of a step
constexpr float kNegBig = -1.0e30f;

struct DecodeArgs {
  const char *q, *k, *v;
  char *o;
  int64_t q_sb, q_sh, q_ss, k_sb, k_sh, k_ss, v_sb, v_sh, v_ss, o_sb, o_sh, o_ss; // elements
  float *part;       // [split][tile][16][HD] sums, then [split][tile][16] (m, l); null: one split
  float *part_ml;
  int32_t Sq, Skv, group, Hkv;
  int32_t heads;     // B * Hkv
  int32_t pitch;     // packed rows per query head: Sq, or Sq rounded up to whole tiles
  int32_t magic;     // 65536 / pitch + 1, where pitch < 16
  int32_t qtiles;    // tiles of 16 rows per key / value head
  int32_t splits, chunks, causal;
  float scale_log2e;
};

template <bool BF16>
__device__ __forceinline__ f32x4 dec_mfma(const uint32_t (&a)[4], const uint32_t (&b)[4], f32x4 c) {
  if constexpr (BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

template <bool BF16> __device__ __forceinline__ uint32_t dec_pack(float a, float b) {
  if constexpr (BF16) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, b2{(__bf16)a, (__bf16)b});
  } else {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, h2{(_Float16)a, (_Float16)b});
  }
}

template <bool BF16> __device__ __forceinline__ void dec_store(char *o, int64_t at, float v) {
  if constexpr (BF16)
    ((SD_AS1 __bf16 *)o)[at] = (__bf16)v;
  else
    ((SD_AS1 _Float16 *)o)[at] = (_Float16)v;
}

// A packed row's grouped head and position (at Sq and beyond it none).
struct DecRow {
  int hg, p;
};

// Row `i` < 16 behind row `first`.  (A division per row: 0.15 us of a small problem's 5.)
__device__ __forceinline__ DecRow dec_row(const DecodeArgs &g, const DecRow &first, int i) {
  const int x = first.p + i; // < pitch + 15
  const int n = g.pitch >= 16 ? (int)(x >= g.pitch) : x * g.magic >> 16;
  return DecRow{first.hg + n, x - n * g.pitch};
}

// Its offset in Q or O; positions past the last stand for it.
__device__ __forceinline__ int64_t dec_offset(const DecodeArgs &g, int b, int hk, const DecRow &r, int64_t sb,
                                              int64_t sh, int64_t ss) {
  return b * sb + (int64_t)(hk * g.group + r.hg) * sh + (int64_t)(r.p < g.Sq ? r.p : g.Sq - 1) * ss;
}

template <bool BF16, int HD>
__global__ __launch_bounds__(kWaves * 64)
__attribute__((amdgpu_waves_per_eu(2, 8))) void sdpa_decode_kernel(DecodeArgs g) {
  constexpr int T = HD / 16;       // columns of V per lane, 16-column tiles of O
  constexpr int KD = HD / 32;      // MFMA steps of a score tile
  constexpr int PITCH = 17;        // floats per column of O in LDS
  __shared__ float sums[kWaves][HD * PITCH];
  __shared__ float ml[kWaves][2][16];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, lq = l & 15, lg = l >> 4;
  // (tiles of one head land on one XCD where the head count allows: they read
  // the same K and V)
  const int per = g.heads * g.splits;
  const int qt = blockIdx.x / per, rest = blockIdx.x % per;
  const int head = rest / g.splits, split = rest % g.splits;
  const int b = head / g.Hkv, hk = head % g.Hkv;
  const int rows = g.group * g.pitch;
  const int left = rows - qt * 16; // of the packed rows from this tile's first
  const int hg0 = qt * 16 / g.pitch;
  const DecRow first{hg0, qt * 16 - hg0 * g.pitch};
  const DecRow mine = dec_row(g, first, lq < left ? lq : left - 1);
  const int pos = mine.p; // query position, for the causal mask

  uint32_t qf[KD][4];
  {
    const char *src = g.q + (dec_offset(g, b, hk, mine, g.q_sb, g.q_sh, g.q_ss) + lg * 8) * 2;
#pragma unroll
    for (int u = 0; u < KD; ++u) {
      const u32x4 x = *(const SD_AS1 u32x4 *)(src + u * 64);
      qf[u][0] = x.x, qf[u][1] = x.y, qf[u][2] = x.z, qf[u][3] = x.w;
    }
  }
  const char *kp = g.k + (b * g.k_sb + hk * g.k_sh) * 2 + lg * 16;
  const char *vp = g.v + (b * g.v_sb + hk * g.v_sh) * 2 + lq * T * 2;
  const uint32_t k_rowb = (uint32_t)(g.k_ss * 2), v_rowb = (uint32_t)(g.v_ss * 2);
  // this workgroup's chunks; the wavefronts take them in turn (under a causal
  // mask up to the last position of the tile's rows)
  int chunks = g.chunks;
  if (g.causal) {
    const DecRow last = dec_row(g, first, left < 16 ? left - 1 : 15);
    const int top = last.hg == first.hg && last.p < g.Sq ? last.p : g.Sq - 1;
    const int need = top / kChunk + 1;
    chunks = need < chunks ? need : chunks;
  }
  const int c0 = (int)((int64_t)chunks * split / g.splits);
  const int c1 = (int)((int64_t)chunks * (split + 1) / g.splits);

  typedef std::conditional_t<T == 8, u32x4, u32x2> VRow;
  u32x4 kf[2][2][KD]; // [buffer][16-key tile][step]
  VRow vf[2][8];
  auto fetch = [&](auto buf, int c) {
    constexpr int B = decltype(buf)::value;
    const int key0 = c * kChunk;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      int key = key0 + t * 16 + lq;
      key = key < g.Skv ? key : g.Skv - 1;
      const char *p = kp + (uint64_t)((uint32_t)key * k_rowb);
#pragma unroll
      for (int u = 0; u < KD; ++u)
        kf[B][t][u] = *(const SD_AS1 u32x4 *)(p + u * 64);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      int key = key0 + (i >> 2) * 16 + lg * 4 + (i & 3);
      key = key < g.Skv ? key : g.Skv - 1;
      vf[B][i] = *(const SD_AS1 VRow *)(vp + (uint64_t)((uint32_t)key * v_rowb));
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x4 o[T];
#pragma unroll
  for (int j = 0; j < T; ++j)
    o[j] = f32x4{0, 0, 0, 0};
  float m = kNegBig, sum = 0.f; // of query lq: max over all lanes, sum over this lane's keys
  auto spend = [&](auto buf, int c) {
    constexpr int B = decltype(buf)::value;
    // (keys past the last are copies of it with probability 0; its values may be infinite)
    if ((c + 1) * kChunk > g.Skv)
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (c * kChunk + (i >> 2) * 16 + lg * 4 + (i & 3) >= g.Skv)
          vf[B][i] = VRow{};
    float s[8];
    uint32_t live = 0;
    float top = kNegBig;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f32x4 a{0, 0, 0, 0};
#pragma unroll
      for (int u = 0; u < KD; ++u) {
        const u32x4 x = kf[B][t][u];
        const uint32_t f[4] = {x.x, x.y, x.z, x.w};
        a = dec_mfma<BF16>(f, qf[u], a);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = c * kChunk + t * 16 + lg * 4 + r;
        const bool in = key < g.Skv && (!g.causal || key <= pos);
        live |= (uint32_t)in << (t * 4 + r);
        s[t * 4 + r] = a[r] * g.scale_log2e;
        top = fmaxf(top, in ? s[t * 4 + r] : kNegBig);
      }
    }
    top = fmaxf(top, __shfl_xor(top, 16, 64));
    top = fmaxf(top, __shfl_xor(top, 32, 64));
    const float mn = fmaxf(m, top);
    if (__builtin_amdgcn_ballot_w64(mn > m)) {
      const float alpha = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      sum *= alpha;
#pragma unroll
      for (int j = 0; j < T; ++j)
        o[j] *= alpha;
    }
    float p[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      p[i] = (live >> i) & 1 ? __builtin_amdgcn_exp2f(s[i] - m) : 0.f;
      sum += p[i];
    }
    const uint32_t pf[4] = {dec_pack<BF16>(p[0], p[1]), dec_pack<BF16>(p[2], p[3]),
                            dec_pack<BF16>(p[4], p[5]), dec_pack<BF16>(p[6], p[7])};
#pragma unroll
    for (int j = 0; j < T; ++j) {
      uint32_t f[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        f[e] = __builtin_amdgcn_perm(vf[B][2 * e + 1][j / 2], vf[B][2 * e][j / 2],
                                     j & 1 ? 0x07060302u : 0x05040100u);
      o[j] = dec_mfma<BF16>(f, pf, o[j]);
    }
  };
  using Buf0 = std::integral_constant<int, 0>;
  using Buf1 = std::integral_constant<int, 1>;
  int c = c0 + wave;
  if (c < c1)
    fetch(Buf0{}, c);
  while (c < c1) {
    if (c + kWaves < c1)
      fetch(Buf1{}, c + kWaves);
    spend(Buf0{}, c);
    c += kWaves;
    if (c >= c1)
      break;
    if (c + kWaves < c1)
      fetch(Buf0{}, c + kWaves);
    spend(Buf1{}, c);
    c += kWaves;
  }
  // ---- the wavefronts' parts meet: O^T value r of tile j is column
  // (lg * 4 + r) * T + j of query lq
  sum += __shfl_xor(sum, 16, 64);
  sum += __shfl_xor(sum, 32, 64);
#pragma unroll
  for (int j = 0; j < T; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      sums[wave][((lg * 4 + r) * T + j) * PITCH + lq] = o[j][r];
  if (l < 16)
    ml[wave][0][l] = m, ml[wave][1][l] = sum;
  __syncthreads();
  const int tile = head * g.qtiles + qt;
  const int64_t tiles = (int64_t)g.heads * g.qtiles;
  const int d = threadIdx.x % HD;
  for (int q = threadIdx.x / HD; q < 16 && q < left; q += kWaves * 64 / HD) {
    const DecRow r = dec_row(g, first, q);
    if (r.p >= g.Sq)
      continue;
    float top = ml[0][0][q];
#pragma unroll
    for (int w = 1; w < kWaves; ++w)
      top = fmaxf(top, ml[w][0][q]);
    float acc = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float f = __builtin_amdgcn_exp2f(ml[w][0][q] - top);
      acc += sums[w][d * PITCH + q] * f;
      den += ml[w][1][q] * f;
    }
    if (g.part) {
      const int64_t at = (split * tiles + tile) * 16 + q;
      ((SD_AS1 float *)g.part)[at * HD + d] = acc;
      if (d == 0)
        ((SD_AS1 float *)g.part_ml)[at * 2] = top, ((SD_AS1 float *)g.part_ml)[at * 2 + 1] = den;
    } else {
      dec_store<BF16>(g.o, dec_offset(g, b, hk, r, g.o_sb, g.o_sh, g.o_ss) + d, acc / den);
    }
  }
}

// Combines the splits of one packed query row per HD threads.
template <bool BF16, int HD>
__global__ __launch_bounds__(256) void sdpa_decode_combine_kernel(DecodeArgs g) {
  const uint32_t rows = (uint32_t)(g.group * g.pitch);
  const uint32_t lin = blockIdx.x * (256 / HD) + threadIdx.x / HD; // (head, row; their parts fit the device)
  const int d = threadIdx.x % HD;
  if (lin >= (uint32_t)g.heads * rows)
    return;
  const int head = (int)(lin / rows), row = (int)(lin % rows);
  const int hg = row / g.pitch;
  const DecRow r{hg, row - hg * g.pitch};
  if (r.p >= g.Sq)
    return;
  const int64_t tiles = (int64_t)g.heads * g.qtiles;
  const int64_t at = (int64_t)(head * g.qtiles + row / 16) * 16 + row % 16;
  const SD_AS1 float *ml = (const SD_AS1 float *)g.part_ml;
  const SD_AS1 float *p = (const SD_AS1 float *)g.part;
  struct Part {
    float m, l, o;
  };
  const auto load = [&](int s) {
    const int64_t i = s * tiles * 16 + at;
    return Part{ml[i * 2], ml[i * 2 + 1], p[i * HD + d]};
  };
  // the first parts whole, so that up to eight splits cost one round of loads
  constexpr int U = 8;
  Part v[U];
#pragma unroll
  for (int s = 0; s < U; ++s)
    if (s < g.splits)
      v[s] = load(s);
  __builtin_amdgcn_sched_barrier(0);
  float top = kNegBig, acc = 0.f, den = 0.f;
#pragma unroll
  for (int s = 0; s < U; ++s)
    if (s < g.splits)
      top = fmaxf(top, v[s].m);
  fhip_for_uniform_parts<U>(
      U, 1, g.splits, [&](int s) { return ml[(s * tiles * 16 + at) * 2]; }, [&](float m) { top = fmaxf(top, m); });
  const auto add = [&](const Part &x) {
    const float f = __builtin_amdgcn_exp2f(x.m - top);
    den += x.l * f;
    acc += x.o * f;
  };
#pragma unroll
  for (int s = 0; s < U; ++s)
    if (s < g.splits)
      add(v[s]);
  fhip_for_uniform_parts<U>(U, 1, g.splits, load, add);
  dec_store<BF16>(g.o, dec_offset(g, head / g.Hkv, head % g.Hkv, r, g.o_sb, g.o_sh, g.o_ss) + d, acc / den);
}

} // namespace

int fhip_decode_sdpa(fhip_ctx *ctx, const fhip_sdpa_desc *d, const void *q, const void *k,
                     const void *v, void *o, bool *handled) {
  *handled = false;
  const int forced = fhip_knobs().sdpa_decode;
  if (d->mask.rank != 0 || forced == 0)
    return 0;
  DecodeArgs g{};
  const int64_t B = d->q.dim[0], Hq = d->q.dim[1], Hkv = d->k.dim[1], HD = d->q.dim[3];
  g.Sq = (int32_t)d->q.dim[2];
  g.Skv = (int32_t)d->k.dim[2];
  g.group = (int32_t)(Hq / Hkv);
  g.Hkv = (int32_t)Hkv;
  if (B * Hkv >= (1 << 24) || (int64_t)g.group * (g.Sq + 15) >= (1 << 24))
    return 0;
  g.heads = (int32_t)(B * Hkv);
  // Under a causal mask a tile walks the keys up to its last position.  With the end of
  // one head's positions and the start of the next in one tile, the first positions would
  // be multiplied (by zero) with values up to the last key, infinite or NaN ones included,
  // where the tiled kernel stops at their own 64 keys: there a head starts a tile.
  g.pitch = d->is_causal && g.Sq > 64 ? (g.Sq + 15) / 16 * 16 : g.Sq;
  g.magic = g.pitch < 16 ? 65536 / g.pitch + 1 : 0;
  const int rows = g.group * g.pitch;
  g.qtiles = (rows + 15) / 16;
  int kv = g.Skv; // keys that any row sees
  if (d->is_causal && g.Sq < kv)
    kv = g.Sq;
  g.chunks = (kv + kChunk - 1) / kChunk;
  const int64_t tiles = (int64_t)g.heads * g.qtiles;
  // two workgroups per compute unit, two chunks per wavefront at least
  int64_t splits = 512 / tiles, deep = g.chunks / (2 * kWaves);
  splits = splits < deep ? splits : deep;
  g.splits = (int32_t)(splits < 1 ? 1 : splits < 64 ? splits : 64);
  // Estimates in microseconds, fitted to both kernels' times on 1098 problems (1 to 1500
  // queries, 32 to 4096 keys, 1 to 64 heads, batches to 32), of which the slower kernel costs
  // 0.6 % on average.  Here: a wavefront's rounds of 32 keys, half of them under a causal
  // mask; the tiles' reads of K and V at 14.7 TB/s from the caches; a tile's rows; the second
  // launch.  The tiled kernel: 1.45 (D 64: 1.06) per 64 keys and round of 256 workgroups of
  // 256 rows, a long and a short tile per workgroup under a causal mask.  (Tiled / here: B21,
  // 64 heads on 8, 68 x 68 causal, D128, 5880 tiles 48.5 / 62.2; B4, 8 heads on 1, 320 x 3456,
  // D64 56.3 / 60.1; B2, 32 heads, 65 x 65 causal, D128 8.6 / 6.2; B7, 32 heads, 1 x 175, D128
  // 9.1 / 5.9.)
  const double half = d->is_causal && g.Sq > 16 ? 0.5 + 8.0 / g.Sq : 1.0;
  const double iters = ceil(g.chunks * half / (kWaves * g.splits)), keys = ceil(kv * half / kChunk) * kChunk;
  const double valid = fmin(1.0, (double)g.group * g.Sq / (16.0 * g.qtiles));
  const double here = (HD == 128 ? 4.2 + 0.99 * iters : 3.4 + 0.81 * iters) + (double)tiles * keys * HD * 4.0 * 0.068e-6 +
                      (double)tiles * HD * 1e-5 * fmax(0.0, 7.8 * valid - 2.7) + (g.splits > 1 ? 4.8 : 0.0);
  const int64_t big = (g.Sq + 255) / 256, kvt = (kv + 63) / 64;
  const bool pairs = d->is_causal && big > 1;
  const double per = HD == 128 ? 1.45 : 1.063, first = pairs ? 7.9 : HD == 128 ? 4.32 : 3.34;
  double there = (d->is_causal ? 1.36 : 0.16) +
                 ceil((double)(B * Hq * (pairs ? (big + 1) / 2 : big)) / 256.0) *
                     (first + per * (pairs ? (double)(kvt * (big + 1)) / (double)big : (double)kvt));
  // grouped heads folded, keys split between teams (never below 6)
  const double cut = here > 6.0 && here < there ? fhip_flash_sdpa_us(d) : -1;
  if (cut > 0 && cut < there)
    there = cut;
  if (here >= there && forced != 1)
    return 0;
  if (tiles * g.splits >= (1ll << 31))
    return 0;
  const size_t rows16 = (size_t)g.splits * (size_t)tiles * 16;
  const size_t part_bytes = rows16 * (size_t)(HD + 2) * sizeof(float);
  if (g.splits > 1 && !fhip_ctx_scratch_ready(ctx, part_bytes))
    g.splits = 1;
  *handled = true;
  g.q = (const char *)q, g.k = (const char *)k, g.v = (const char *)v, g.o = (char *)o;
  auto st = [](const fhip_tensor_desc &t, int i) { return t.dim[i] > 1 ? t.stride[i] : 0; };
  g.q_sb = st(d->q, 0), g.q_sh = st(d->q, 1), g.q_ss = st(d->q, 2);
  g.k_sb = st(d->k, 0), g.k_sh = st(d->k, 1), g.k_ss = st(d->k, 2);
  g.v_sb = st(d->v, 0), g.v_sh = st(d->v, 1), g.v_ss = st(d->v, 2);
  g.o_sb = st(d->o, 0), g.o_sh = st(d->o, 1), g.o_ss = st(d->o, 2);
  g.causal = d->is_causal != 0;
  const float scale = d->has_scale ? d->scale : 1.0f / sqrtf((float)HD);
  g.scale_log2e = scale * 1.4426950408889634f;
  if (g.splits > 1) {
    void *sp = nullptr;
    if (fhip_ctx_scratch(ctx, part_bytes, &sp) != 0)
      return 1;
    g.part = (float *)sp;
    g.part_ml = g.part + rows16 * HD;
  }
  fhip_note_kernel(ctx, "sdpa_decode d=%d tiles=%d splits=%d", (int)HD, (int)g.qtiles, g.splits);
  auto go = [&](auto bf, auto hd) {
    constexpr bool BF = decltype(bf)::value;
    constexpr int D = decltype(hd)::value;
    hipLaunchKernelGGL((sdpa_decode_kernel<BF, D>), dim3((unsigned)(tiles * g.splits)),
                       dim3(kWaves * 64), 0, ctx->stream, g);
    if (g.splits > 1)
      hipLaunchKernelGGL((sdpa_decode_combine_kernel<BF, D>),
                         dim3((unsigned)(((int64_t)g.heads * rows + 256 / D - 1) / (256 / D))), dim3(256),
                         0, ctx->stream, g);
    FHIP_HIP_CHECK(ctx, hipGetLastError());
    return 0;
  };
  using std::integral_constant;
  const bool bf = d->q.dtype == FHIP_BFLOAT16;
  if (HD == 128)
    return bf ? go(std::true_type{}, integral_constant<int, 128>{})
              : go(std::false_type{}, integral_constant<int, 128>{});
  return bf ? go(std::true_type{}, integral_constant<int, 64>{})
            : go(std::false_type{}, integral_constant<int, 64>{});
}

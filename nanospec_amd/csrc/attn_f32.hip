// Soft-max attention over the paged cache in 32-bit on the matrix cores (v_mfma_f32_16x16x4_f32: 32-bit products and sums),
// for keys and values of one size, a multiple of 16 up to 128, in pages of a power of two of at least 4 tokens.  What it
// computes, with which options, and the cache's layout: see attn_generic.hip, which keeps every other size.
//
// Everything is kept transposed, S^T = K Q^T and O^T = V^T P^T, in steps of 16 channels or keys: lane l holds row l % 16 of
// an operand and its channels (keys) 4 (l / 16) .. + 3, one 16-byte read for four instructions.  A lane's scores are then those
// of token l % 16 with keys 4 (l / 16) + i, which is the operand that the second product wants: weights never leave their
// lane, and a token's running maximum, sum and rescaling are its lanes' own.
//
//   attn_f32_kernel: prompt portions.  A workgroup is 32 tokens by two heads of a key/value head, a wave 16 tokens of a head; blocks
//     of 64 keys (counted from key 0) go through LDS, two buffers, the next block's loads in registers beside the arithmetic.
//     Bound by the matrix unit, 64 instructions of 32 cycles for each of the two products a wave and block of 64 keys at
//     head size 64.  LDS rows are 8 floats longer than their data, so that the lanes of a 16-byte read that are served together
//     touch all banks once.  777 tokens, 32 heads of 64 over 8: 1,617 (one workgroup a row and head) -> 63 us.
//   attn_f32_rows_kernel: single tokens.  All heads of a group are a wave's columns, keys and values go from the cache straight into
//     operand registers, four waves take a range's tiles of 16 keys in turn; ranges are added by attn_f32_join_kernel.  Bound
//     by the cache's bytes and the latency of a wave's loads.  5 rows at 900 keys, 32 heads of 64 over 8: 201 -> 16 us with the joining.
// A row's result depends on its own keys only, whatever stands beside it in the batch and however many workgroups share the work: keys go in
// ranges that lie at fixed places (256 keys of a portion, 128 of a single token, counted from key 0), every range is summed from nothing
// and the ranges are added in order by the same operations, in the registers of a workgroup that walks all of them or by
// attn_f32_join_kernel.  A row with more than 32 (64) of them has ranges of twice as many keys, four times, ...: a portion's tile and a single
// token choose by their own keys.  A block or range without a key that a token sees changes nothing of it.  (As a single token and as one
// of a portion a token's sums are ordered differently, and so they are for the tokens of a tile across 8,192, 16,384, ... keys when another cut
// of the prompt moves the tile.)
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
#define AF_KEYS 64
#define AF_TOKENS 32
#define AF_ROWS_TILES 4  // waves of a workgroup of the kernel for single tokens
#define AF_RANGE 4       // blocks of a range of a portion's keys
#define AF_RANGES 32     // the most ranges of a portion's keys
#define AF_ROWS_RANGES 64  // and of a single token's

struct AttnF32Params {
  float* out;        // [rows][heads * HD]
  float* part_o;     // [column][splits][HD], unnormalised, and
  float* part_ml;    // [column][splits][2] if splits > 1; column = (tile * tokens of a tile + token) * heads + head
  const float* q;
  const float* k_cache;
  const float* v_cache;
  const int* tiles;  // [n_tiles][8]: request, first token, row of the request's first token, tokens, keys
  const int* block_table;
  const float* sink_logit;
  int q_stride, table_stride, heads, kv_heads, page_shift, splits, range_tiles, window, chunk, sink, n_tiles;  // range_tiles: of 16 keys (single tokens)
  int rows;
  float scale, cap, slope_exp;
};

__device__ __forceinline__ int first_key(const AttnF32Params& p, int pos) {
  int lo = p.window > 0 ? max(0, pos - p.window + 1) : 0;
  if (p.chunk > 0) lo = max(lo, pos / p.chunk * p.chunk);
  return lo;
}

// Scores of keys key0 .. key0 + 3 as the soft-max meets them; -inf where the token does not see the key.
__device__ __forceinline__ f32x4 finish_scores(const AttnF32Params& p, f32x4 s, int key0, int lo, int pos, float slope) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float v = s[i];
    if (p.cap > 0.f) v = p.cap * tanhf(v / p.cap);
    if (p.slope_exp > 0.f) v -= slope * (float)(pos - key0 - i);
    s[i] = key0 + i >= lo && key0 + i <= pos ? v : -INFINITY;
  }
  return s;
}

// The ranges of blocks (of tiles of 16 keys for a single token) lo .. hi: ``length`` of them each, or twice as many, four times, ... until there
// are no more than ``most`` ranges; first: the one that holds lo, counted from key 0.
struct KeyRanges {
  unsigned length, first;
};
__device__ __forceinline__ KeyRanges key_ranges(unsigned lo, unsigned hi, unsigned length, unsigned most) {
  unsigned first = lo / length;
  for (; hi >= (first + most) * length; length *= 2) first /= 2;
  return {length, first};
}

// How a portion's tile is cut.  (The workspace may have room for fewer ranges than AF_RANGES; it then has room for all that a tile needs.)
__device__ __forceinline__ KeyRanges portion_ranges(const AttnF32Params& p, int tile_lo, int hi) {
  return key_ranges(tile_lo / AF_KEYS, hi / AF_KEYS, AF_RANGE, p.splits > 1 ? p.splits : AF_RANGES);
}
__device__ __forceinline__ unsigned range_count(const KeyRanges& r, int hi) { return (hi / AF_KEYS >> (31 - __clz(r.length))) - r.first + 1; }

// What a range with maximum m does to the sums of the ranges before it, whose maximum is top: sum = sum * old + range * now, the product
// with ``old`` rounded first.  The same operations wherever it is done.
struct RangeWeights {
  float old, now;
};
__device__ __forceinline__ RangeWeights range_weights(float top, float m) {
  const float both = fmaxf(top, m), ref = both == -INFINITY ? 0.f : both;
  return {top == -INFINITY ? 0.f : expf(top - ref), m == -INFINITY ? 0.f : expf(m - ref)};
}

__device__ __forceinline__ float over_groups_max(float v) {
  v = fmaxf(v, __shfl_xor(v, 16, 64));
  return fmaxf(v, __shfl_xor(v, 32, 64));
}
__device__ __forceinline__ float over_groups_sum(float v) {
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}

// The soft-max's term that has no value, in the units of the running maximum m.
__device__ __forceinline__ float sink_term(const AttnF32Params& p, int head, float m) {
  return p.sink_logit ? expf(p.sink_logit[head] - m) : (p.sink ? expf(-m) : 0.f);
}

template <int HD>
__global__ __launch_bounds__(256) void attn_f32_kernel(AttnF32Params p) {
  constexpr int C = HD / 16, KROW = HD + 8, VROW = AF_KEYS + 8, PER = HD / 16, KSIZE = AF_KEYS * KROW, BUF = KSIZE + HD * VROW;
  __shared__ __attribute__((aligned(16))) float lds[2 * BUF];
  __shared__ int odd_values[2][4];  // per buffer and wave: a value among those it brought is infinite or no number
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = lane & 15, g = lane >> 4;
  const int group = p.heads / p.kv_heads, pairs = (group + 1) / 2;
  // the key/value head is the fast index (workgroups go round the eight XCDs in launch order, and each has an L2 of its own); the
  // tiles behind, which have the most keys, start first
  const int kvh = blockIdx.x % p.kv_heads, pair = blockIdx.x / p.kv_heads % pairs, tile = p.n_tiles - 1 - blockIdx.x / (p.kv_heads * pairs);
  const int* info = p.tiles + 8 * tile;
  const int t0 = info[1], n_tok = min(AF_TOKENS, info[3] - t0);
  if (n_tok <= 0) return;  // a tile of a fixed shape that the batch does not fill
  const int* table = p.block_table + (size_t)info[0] * p.table_stride;
  const int base = info[4] - info[3] + t0;  // position of the tile's first token
  const int hi = base + n_tok - 1, tile_lo = first_key(p, base);
  const int in_group = 2 * pair + (wave >> 1), head = kvh * group + min(in_group, group - 1);
  const int tok = min(16 * (wave & 1) + col, n_tok - 1), pos = base + tok, lo = first_key(p, pos);
  const bool works = in_group < group && 16 * (wave & 1) < n_tok;
  const int wave_lo = first_key(p, base + min(16 * (wave & 1), n_tok - 1)), wave_hi = base + min(16 * (wave & 1) + 15, n_tok - 1);
  // full: every token of the wave sees every key of the block
  const int full_lo = first_key(p, wave_hi), full_hi = base + min(16 * (wave & 1), n_tok - 1);
  const float slope = p.slope_exp > 0.f ? exp2f(-p.slope_exp * (float)(head + 1) / (float)p.heads) : 0.f;
  const size_t row = (size_t)info[2] + t0 + tok;

  f32x4 q[C];
#pragma unroll
  for (int c = 0; c < C; ++c) q[c] = *reinterpret_cast<const f32x4*>(p.q + row * p.q_stride + head * HD + 16 * c + 4 * g) * p.scale;

  // this workgroup's ranges, a like share for each of the launch's workgroups in y
  const KeyRanges ranges = portion_ranges(p, tile_lo, hi);
  const int count = range_count(ranges, hi), share = gridDim.y == 1 ? count : (count + gridDim.y - 1) / gridDim.y, range0 = ranges.first + blockIdx.y * share;
  const int b0 = max(tile_lo / AF_KEYS, range0 * (int)ranges.length), b1 = min(hi / AF_KEYS + 1, (range0 + share) * (int)ranges.length);

  // a block of 64 keys: keys in pieces of four channels, values in pieces of four keys, PER of each a thread.  Keys outside of what the tile
  // sees are read as the nearest one it does (their pages may be gone) and their values taken as zero.
  const int mask = (1 << p.page_shift) - 1, vq = 4 * (tid & 15);
  int kid[PER], vid;
  f32x4 kreg[PER], vreg[PER];
  auto key_of = [&](int b, int i) { return min(max(b * AF_KEYS + (i * 256 + tid) / (HD / 4), tile_lo), hi); };
  auto value_of = [&](int b) { return min(max(b * AF_KEYS + vq, tile_lo & ~3), hi & ~3); };
  auto pages = [&](int b) {
#pragma unroll
    for (int i = 0; i < PER; ++i) kid[i] = table[key_of(b, i) >> p.page_shift];
    vid = table[value_of(b) >> p.page_shift];
  };
  auto fetch = [&](int b) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const size_t at = (((size_t)kid[i] * p.kv_heads + kvh) << p.page_shift) + (key_of(b, i) & mask);
      kreg[i] = *reinterpret_cast<const f32x4*>(p.k_cache + at * HD + 4 * ((i * 256 + tid) % (HD / 4)));
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const size_t at = ((size_t)vid * p.kv_heads + kvh) * HD + i * 16 + (tid >> 4);
      vreg[i] = *reinterpret_cast<const f32x4*>(p.v_cache + (at << p.page_shift) + (value_of(b) & mask));
    }
  };
  auto park = [&](int b, int buf) {
    float* to = lds + buf * BUF;
#pragma unroll
    for (int i = 0; i < PER; ++i) *reinterpret_cast<f32x4*>(to + (i * 256 + tid) / (HD / 4) * KROW + 4 * ((i * 256 + tid) % (HD / 4))) = kreg[i];
    bool odd = false;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int key = b * AF_KEYS + vq + e;
        if (key < tile_lo || key > hi) vreg[i][e] = 0.f;
        odd |= !(fabsf(vreg[i][e]) < INFINITY);
      }
      *reinterpret_cast<f32x4*>(to + KSIZE + (i * 16 + (tid >> 4)) * VROW + vq) = vreg[i];
    }
    const bool any = __any(odd);
    if (lane == 0) odd_values[buf][wave] = any;
  };

  float m = -INFINITY, l = 0.f;  // of the range so far; l: this lane's keys of every block
  float top = -INFINITY, sum = 0.f;  // of the ranges before
  f32x4 acc[C], all[C];
#pragma unroll
  for (int c = 0; c < C; ++c) acc[c] = all[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (b0 < b1) {
    pages(b0);
    fetch(b0);
    pages(b0 + 1);
    park(b0, 0);
  }
  const bool mine = works && 16 * (wave & 1) + col < n_tok;
  size_t at = (((size_t)tile * AF_TOKENS + tok) * p.heads + head) * p.splits + blockIdx.y * share;  // place of the range in the workspace
  auto end_range = [&]() {
    l = over_groups_sum(l);
    if (p.splits > 1) {
      if (mine) {
#pragma unroll
        for (int c = 0; c < C; ++c) *reinterpret_cast<f32x4*>(p.part_o + at * HD + 16 * c + 4 * g) = acc[c];
        if (g == 0) p.part_ml[2 * at] = m, p.part_ml[2 * at + 1] = l;
      }
      ++at;
    } else if (count == 1) {  // (what the sums below come to)
      top = m, sum = l;
#pragma unroll
      for (int c = 0; c < C; ++c) all[c] = acc[c];
    } else {
      const RangeWeights w = range_weights(top, m);
      top = fmaxf(top, m), sum = fmaf(l, w.now, sum * w.old);
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) all[c][i] = fmaf(acc[c][i], w.now, all[c][i] * w.old);
    }
    m = -INFINITY, l = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  for (int b = b0; b < b1; ++b) {
    const int buf = (b - b0) & 1;
    __syncthreads();
    if (b + 1 < b1) fetch(b + 1);
    pages(b + 2);
    const int k0 = b * AF_KEYS;
    if (works && k0 <= wave_hi && k0 + AF_KEYS > wave_lo) {
      const float* ks = lds + buf * BUF + col * KROW + 4 * g;
      const float* vs = lds + buf * BUF + KSIZE + col * VROW + 4 * g;
      f32x4 s[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < C; ++c) {
        f32x4 k[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) k[t] = *reinterpret_cast<const f32x4*>(ks + t * 16 * KROW + 16 * c);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int t = 0; t < 4; ++t) s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[t][e], q[c][e], s[t], 0, 0, 0);
      }
      const bool full = k0 >= full_lo && k0 + AF_KEYS - 1 <= full_hi;
      if (!full || p.cap > 0.f || p.slope_exp > 0.f) {
#pragma unroll
        for (int t = 0; t < 4; ++t) s[t] = finish_scores(p, s[t], k0 + 16 * t + 4 * g, lo, pos, slope);
      }
      float highest = s[0][0];
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) highest = fmaxf(highest, s[t][i]);
      const float m_new = fmaxf(m, over_groups_max(highest));
      const float ref = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = m == -INFINITY ? 0.f : expf(m - ref);
      float weights = 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[t][i] = expf(s[t][i] - ref);
          weights += s[t][i];
        }
      l = l * alpha + weights;
      m = m_new;
#pragma unroll
      for (int c = 0; c < C; ++c) acc[c] *= alpha;
      const int odd = odd_values[buf][0] | odd_values[buf][1] | odd_values[buf][2] | odd_values[buf][3];
      if (full || !odd) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          f32x4 v[C];
#pragma unroll
          for (int c = 0; c < C; ++c) v[c] = *reinterpret_cast<const f32x4*>(vs + c * 16 * VROW + 16 * t);
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int c = 0; c < C; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[c][e], s[t][e], acc[c], 0, 0, 0);
        }
      } else {
        // an infinite value or one that is no number, which some token of the wave may not see: a weight of zero would make it that
        // token's too, so each token adds the keys it sees only
        const float* at = lds + buf * BUF + KSIZE + 4 * g * VROW;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            for (int gg = 0; gg < 4; ++gg) {
              const int key = 16 * t + 4 * gg + i;
              const float w = __shfl(s[t][i], 16 * gg + col, 64);
              if (k0 + key >= lo && k0 + key <= pos) {
#pragma unroll
                for (int c = 0; c < C; ++c)
#pragma unroll
                  for (int j = 0; j < 4; ++j) acc[c][j] = fmaf(w, at[(16 * c + j) * VROW + key], acc[c][j]);
              }
            }
      }
    }
    if (b + 1 < b1) park(b + 1, buf ^ 1);
    if (b + 1 == b1 || !((b + 1) & (ranges.length - 1))) end_range();  // (a power of two)
  }
  if (!mine || p.splits > 1) return;
  sum += sink_term(p, head, top);
#pragma unroll
  for (int c = 0; c < C; ++c) *reinterpret_cast<f32x4*>(p.out + (row * p.heads + head) * HD + 16 * c + 4 * g) = all[c] / sum;
}

template <int HD>
__global__ __launch_bounds__(256) void attn_f32_rows_kernel(AttnF32Params p) {
  constexpr int C = HD / 16;
  __shared__ __attribute__((aligned(16))) float join_o[AF_ROWS_TILES][16][HD + 4];
  __shared__ float join_ml[AF_ROWS_TILES][16][2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, col = lane & 15, g = lane >> 4;
  const int group = p.heads / p.kv_heads, sets = (group + 15) / 16;
  const int kvh = blockIdx.x % p.kv_heads, set = blockIdx.x / p.kv_heads % sets, tile = blockIdx.x / (p.kv_heads * sets);
  const int* info = p.tiles + 8 * tile;
  if (info[3] <= 0) return;
  const int* table = p.block_table + (size_t)info[0] * p.table_stride;
  const int pos = info[4] - info[3] + info[1], lo = first_key(p, pos);
  const int in_group = 16 * set + col, head = kvh * group + min(in_group, group - 1);
  const float slope = p.slope_exp > 0.f ? exp2f(-p.slope_exp * (float)(head + 1) / (float)p.heads) : 0.f;
  const size_t row = (size_t)info[2] + info[1];
  f32x4 q[C];
#pragma unroll
  for (int c = 0; c < C; ++c) q[c] = *reinterpret_cast<const f32x4*>(p.q + row * p.q_stride + head * HD + 16 * c + 4 * g) * p.scale;

  const KeyRanges ranges = key_ranges(lo / 16, pos / 16, p.range_tiles, AF_ROWS_RANGES);
  const int range = ranges.first + blockIdx.y;
  const int first = range * (int)ranges.length + wave, end = min(pos / 16 + 1, (range + 1) * (int)ranges.length);
  const int mask = (1 << p.page_shift) - 1;
  int kid, vid;
  f32x4 k[2][C], v[2][C];
  auto key_of = [&](int t) { return min(max(16 * t + col, lo), pos); };
  auto value_of = [&](int t) { return min(max(16 * t + 4 * g, lo & ~3), pos & ~3); };
  auto pages = [&](int t) {
    kid = table[key_of(t) >> p.page_shift];
    vid = table[value_of(t) >> p.page_shift];
  };
  auto fetch = [&](int t, f32x4* kk, f32x4* vv) {
    const size_t ka = ((((size_t)kid * p.kv_heads + kvh) << p.page_shift) + (key_of(t) & mask)) * HD + 4 * g;
    const size_t va = ((size_t)vid * p.kv_heads + kvh) * HD + col;
#pragma unroll
    for (int c = 0; c < C; ++c) kk[c] = *reinterpret_cast<const f32x4*>(p.k_cache + ka + 16 * c);
#pragma unroll
    for (int c = 0; c < C; ++c) vv[c] = *reinterpret_cast<const f32x4*>(p.v_cache + ((va + 16 * c) << p.page_shift) + (value_of(t) & mask));
  };
  float m = -INFINITY, l = 0.f;
  f32x4 acc[C];
#pragma unroll
  for (int c = 0; c < C; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int t, const f32x4* kk, const f32x4* vv) {
    f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[c][e], q[c][e], s, 0, 0, 0);
    const int key0 = 16 * t + 4 * g;
    s = finish_scores(p, s, key0, lo, pos, slope);
    const float m_new = fmaxf(m, over_groups_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))));
    const float ref = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = m == -INFINITY ? 0.f : expf(m - ref);
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = expf(s[i] - ref);
    l = l * alpha + ((s[0] + s[1]) + (s[2] + s[3]));
    m = m_new;
    const bool edge = 16 * t < lo || 16 * t + 15 > pos;  // uniform: what lies outside may hold anything and counts as zero
#pragma unroll
    for (int c = 0; c < C; ++c) {
      f32x4 a = vv[c];
      if (edge) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (4 * g + 16 * t + e < lo || 4 * g + 16 * t + e > pos) a[e] = 0.f;
      }
      acc[c] *= alpha;
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], s[e], acc[c], 0, 0, 0);
    }
  };
  if (first < end) {
    pages(first);
    fetch(first, k[0], v[0]);
    pages(first + AF_ROWS_TILES);
    for (int t = first; t < end; t += 2 * AF_ROWS_TILES) {
      if (t + AF_ROWS_TILES < end) fetch(t + AF_ROWS_TILES, k[1], v[1]);
      pages(t + 2 * AF_ROWS_TILES);
      step(t, k[0], v[0]);
      if (t + AF_ROWS_TILES >= end) break;
      if (t + 2 * AF_ROWS_TILES < end) fetch(t + 2 * AF_ROWS_TILES, k[0], v[0]);
      pages(t + 3 * AF_ROWS_TILES);
      step(t + AF_ROWS_TILES, k[1], v[1]);
    }
  }
  l = over_groups_sum(l);
  // the four waves' results, in their order
#pragma unroll
  for (int c = 0; c < C; ++c) *reinterpret_cast<f32x4*>(&join_o[wave][col][16 * c + 4 * g]) = acc[c];
  if (g == 0) join_ml[wave][col][0] = m, join_ml[wave][col][1] = l;
  __syncthreads();
  for (int e = tid; e < 16 * HD; e += 256) {
    const int c = e / HD, d = e % HD;
    if (16 * set + c >= group) break;
    float top = -INFINITY, sum = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < AF_ROWS_TILES; ++w) top = fmaxf(top, join_ml[w][c][0]);
    const float ref = top == -INFINITY ? 0.f : top;
#pragma unroll
    for (int w = 0; w < AF_ROWS_TILES; ++w) {
      if (join_ml[w][c][0] == -INFINITY && join_ml[w][c][1] == 0.f) continue;  // a wave without keys
      const float f = expf(join_ml[w][c][0] - ref);
      sum = fmaf(f, join_ml[w][c][1], sum);
      o = fmaf(f, join_o[w][c][d], o);
    }
    const int hd = kvh * group + 16 * set + c;
    if (p.splits > 1) {
      const size_t at = ((size_t)tile * p.heads + hd) * p.splits + blockIdx.y;
      if (sum != 0.f) p.part_o[at * HD + d] = o;  // (a range without keys is not read)
      if (d == 0) p.part_ml[2 * at] = top, p.part_ml[2 * at + 1] = sum;
    } else {
      p.out[(row * p.heads + hd) * HD + d] = o / (sum + sink_term(p, hd, top));
    }
  }
}

// Adds the ranges of a (tile, token of the tile, head): a wave each.  A portion's in their order, as the kernel above does; a single token's, at
// most 64, by their common maximum.
__global__ __launch_bounds__(256) void attn_f32_join_kernel(AttnF32Params p, int tokens, int hd) {
  const int lane = threadIdx.x & 63;
  const size_t column = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (column >= (size_t)p.n_tiles * tokens * p.heads) return;
  const int head = column % p.heads, tok = column / p.heads % tokens, tile = column / p.heads / tokens;
  const int* info = p.tiles + 8 * tile;
  if (info[1] + tok >= info[3]) return;  // the tile holds fewer tokens
  const size_t row = (size_t)info[2] + info[1] + tok;
  if (!p.rows) {
    const int base = info[4] - info[3] + info[1];
    const KeyRanges ranges = portion_ranges(p, first_key(p, base), base + min(AF_TOKENS, info[3] - info[1]) - 1);
    // lane s: range s, the maximum of the ranges before it and its weights
    const int count = range_count(ranges, base + min(AF_TOKENS, info[3] - info[1]) - 1);
    const bool has = lane < count;
    const float m = has ? p.part_ml[2 * (column * p.splits + lane)] : -INFINITY, l = has ? p.part_ml[2 * (column * p.splits + lane) + 1] : 0.f;
    float top = m;
    for (int d = 1; d < AF_ROWS_RANGES; d *= 2) {
      const float before = __shfl_up(top, d, 64);
      if (lane >= d) top = fmaxf(before, top);
    }
    const float before = __shfl_up(top, 1, 64);
    const RangeWeights w = range_weights(lane ? before : -INFINITY, m);
    float sum = 0.f, o[2] = {0.f, 0.f};  // (a head is at most 128 channels)
    for (int s0 = 0; s0 < count; s0 += 8) {  // eight ranges' loads at a time
      float part[8][2];
#pragma unroll
      for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          part[s][i] = s0 + s < count && 64 * i + lane < hd ? p.part_o[(column * p.splits + s0 + s) * hd + 64 * i + lane] : 0.f;
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        if (s0 + s >= count) break;
        const float old = __shfl(w.old, s0 + s, 64), now = __shfl(w.now, s0 + s, 64);
        sum = fmaf(__shfl(l, s0 + s, 64), now, sum * old);
#pragma unroll
        for (int i = 0; i < 2; ++i) o[i] = fmaf(part[s][i], now, o[i] * old);
      }
    }
    sum += sink_term(p, head, __shfl(top, 63, 64));
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if (64 * i + lane < hd) p.out[(row * p.heads + head) * hd + 64 * i + lane] = o[i] / sum;
    return;
  }
  const float m = lane < p.splits ? p.part_ml[2 * (column * p.splits + lane)] : -INFINITY;
  const float top = wave_max(m), f = m == -INFINITY ? 0.f : expf(m - top);
  const float l = wave_sum(lane < p.splits ? f * p.part_ml[2 * (column * p.splits + lane) + 1] : 0.f) + sink_term(p, head, top);
  for (int d0 = 0; d0 < hd; d0 += 64) {  // (every lane takes part in the exchange, whatever the head size)
    const int d = d0 + lane;
    float o = 0.f;
    for (int s = 0; s < p.splits; ++s) {
      const float w = __shfl(f, s, 64);
      if (w != 0.f && d < hd) o = fmaf(w, p.part_o[(column * p.splits + s) * hd + d], o);
    }
    if (d < hd) p.out[(row * p.heads + head) * hd + d] = o / l;
  }
}

template <int HD>
static void launch_attn_f32(const AttnF32Params& p, int groups, hipStream_t stream) {
  const int group = p.heads / p.kv_heads;
  if (p.rows)
    attn_f32_rows_kernel<HD><<<dim3(p.n_tiles * p.kv_heads * ((group + 15) / 16), p.splits), 256, 0, stream>>>(p);
  else
    attn_f32_kernel<HD><<<dim3(p.n_tiles * p.kv_heads * ((group + 1) / 2), groups), 256, 0, stream>>>(p);
  if (p.splits > 1) {
    const int tokens = p.rows ? 1 : AF_TOKENS;
    attn_f32_join_kernel<<<((size_t)p.n_tiles * tokens * p.heads + 3) / 4, 256, 0, stream>>>(p, tokens, HD);
  }
}

// ``rows`` != 0: the tiles are single tokens, whose keys go in ranges of 16 ``range_tiles`` keys (or twice as many, ... so that there are at most 64);
// the caller launches ``splits`` workgroups, as many as the row with the most ranges has, one each.  0: up to 32 tokens each, whose keys
// go in at most 32 ranges of 256 keys or more; ``splits`` = 1: each tile's ranges by one workgroup, or the number of ranges that the workspace
// has room for (fewer than 32 only if no tile has more), dealt to ``groups`` workgroups.  Workspace, when splits > 1 (at most 64): part_o holds
// n_tiles * (rows ? 1 : 32) * heads * splits * hd floats and part_ml twice as many as there are ranges.
extern "C" int ns_attn_f32(float* out, float* part_o, float* part_ml, const float* q, int q_stride, const float* k_cache, const float* v_cache,
                           const int* tiles, const int* block_table, int table_stride, int n_tiles, int heads, int kv_heads, int hd,
                           int page_size, int rows, int splits, int groups, int range_tiles, float scale, int window, int chunk, float cap, int sink,
                           const float* sink_logit, float slope_exp, hipStream_t stream) {
  if (n_tiles <= 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads || window < 0 || chunk < 0 || cap < 0.f || slope_exp < 0.f ||
      splits < 1 || splits > AF_ROWS_RANGES || groups < 1 || groups > splits || range_tiles < 1 || (splits > 1 && (!part_o || !part_ml)))
    return NS_ERR_BAD_ARG;
  if (hd % 16 || hd < 16 || hd > 128 || page_size < 4 || page_size & (page_size - 1) || q_stride % 4 ||
      (((uintptr_t)out | (uintptr_t)part_o | (uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15))
    return NS_ERR_UNSUPPORTED;
  if ((long)n_tiles * heads * AF_TOKENS > 0x7fffffffL) return NS_ERR_BAD_ARG;
  int shift = 0;
  while (1 << shift < page_size) ++shift;
  const AttnF32Params p{out, part_o, part_ml, q, k_cache, v_cache, tiles, block_table, sink_logit, q_stride, table_stride, heads, kv_heads,
                        shift, splits, range_tiles, window, chunk, sink, n_tiles, rows, scale, cap, slope_exp};
  switch (hd) {
    case 16: launch_attn_f32<16>(p, groups, stream); break;
    case 32: launch_attn_f32<32>(p, groups, stream); break;
    case 48: launch_attn_f32<48>(p, groups, stream); break;
    case 64: launch_attn_f32<64>(p, groups, stream); break;
    case 80: launch_attn_f32<80>(p, groups, stream); break;
    case 96: launch_attn_f32<96>(p, groups, stream); break;
    case 112: launch_attn_f32<112>(p, groups, stream); break;
    default: launch_attn_f32<128>(p, groups, stream); break;
  }
  return ns_launch_status();
}

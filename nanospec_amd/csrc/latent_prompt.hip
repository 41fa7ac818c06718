// Latent attention (see latent.hip) for prompt portions in bfloat16: keys and values are made from the latents, head by head, and
// ordinary attention runs over them.  The form that latent.hip serves reads the latents themselves as ONE wide key/value head: for a
// token alone that is the least traffic, but a (query, key) pair then costs 2 C + R products a head (1,056 at a latent of 512 with 32
// rotated channels) instead of D + R + E (160 with 64 + 32 and 64), and a portion of a hundred tokens and more has the keys and values
// made in less time than that.  Keys, values and the heads' outputs are each rounded to bfloat16 once, where the other form rounds
// absorbed queries, weighted latents and outputs.
//
//   latent_expand_kernel: k_h(j) = [Uk_h c(j) | r(j)] and v_h(j) = Uv_h c(j) for the keys that a portion sees, from the cache's pages
//     into scratch laid out as the attention reads it: [portion][block of 64 keys][head]{ keys [64][D + R] | values [E][64] }, a
//     channel's keys in the order in which the lanes hold weights (within 32 keys, key 16 t + 4 g + i at place 8 g + 4 t + i).  A wave takes 32
//     keys of a head through both matrices; a fragment of the latents serves both as either operand.  Bound by the matrices' and
//     latents' way from L2 (each wave reading the matrices itself: 42 us for 2,048 keys, 32 heads, latent 512; through LDS: 20 us, and 29
//     in a prompt, where the matrices come from memory).
//   latent_prompt_kernel: a workgroup is 64 tokens of a head, a wave 16; a block of 64 keys and values is contiguous in the
//     scratch and goes through LDS, two buffers, the next one on its way in registers.  S^T = K Q^T and O^T = V^T P^T on
//     v_mfma_f32_16x16x32_bf16, so a token's scores, maximum and sums are its own lanes'.  Queries are rotated as they are read; the
//     sink's term, the gate per head and the gate per channel are applied to the 32-bit result before it is rounded.  LDS rows are 32
//     bytes longer than their data (no bank conflicts).  Bound by the matrix and the vector unit in turn (the soft-max of a block takes
//     about as long as its products) and the longest tile's chain of blocks, hence 64 tokens and not 128.  What is not finite
//     reaches the tokens that see it and no others; blocks at a tile's edges have code of their own for that, and the others then do
//     without a mask.  2,048 tokens, 32 heads of 64 + 32, both kernels: 75 us (128 tokens a workgroup: 25 us more); the wide form takes
//     545 us and 120 us around it.
#include "common.h"
#include "rope.h"

#include <type_traits>

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
#define LP_KEYS 64
#define LP_TOKENS 64       // tokens of a workgroup: two tiles of the batch's tile list
#define LX_ROW (64 + 16)   // bfloat16 values between the rows of a matrix's piece in LDS

struct LatentPromptParams {
  const bf16_t* latents;  // K pages [page][token][C + R] of the cache: normed latent, rotated part
  const bf16_t* uk;       // [H * D][C]
  const bf16_t* uv;       // [H * E][C]
  bf16_t* scratch;        // [portions][blocks][H][64 (D + R) + 64 E]
  const bf16_t* q;        // rows q_stride apart: [H][D + R], not rotated
  bf16_t* out;            // [rows][H * E]
  const int* tiles;       // [n_tiles][8]: request, first token, row of the request's first token, tokens, keys, -, portion; the p-th tile's last int is the
                          // number of portion p's first tile (-1: there is no such portion)
  const int* block_table;
  const float* inv_freq;
  const float* gate;         // null, or [rows][H]
  const bf16_t* zgate;       // null, or rows z_stride apart: [H * E]
  const float* sink_logits;  // null, or [H]
  int q_stride, z_stride, table_stride, n_tiles, H, C, page_shift, blocks, window;
  float scale_log2;
  RopeForm form;
};

template <int D, int R, int E>
__global__ __launch_bounds__(256) void latent_expand_kernel(LatentPromptParams p) {
  constexpr int KD = D + R, JK = D / 16, JV = E / 16;
  const int first = p.tiles[8 * blockIdx.z + 7];
  if (first < 0) return;
  const int* info = p.tiles + 8 * first;
  const int kv = info[4], start = kv - info[3], h = blockIdx.y, key0 = blockIdx.x * 2 * LP_KEYS;
  const int lo = p.window > 0 ? max(0, start - p.window + 1) : 0;  // the first key that the portion's first token sees
  if (key0 >= kv || key0 + 2 * LP_KEYS <= lo) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  const int* table = p.block_table + (size_t)info[0] * p.table_stride;
  const int CR = p.C + R, mask = (1 << p.page_shift) - 1;
  const bf16_t* lat[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int key = min(max(key0 + 32 * wave + 16 * t + r, lo), kv - 1);  // (keys outside are masked where they are read)
    lat[t] = p.latents + (((size_t)table[key >> p.page_shift] << p.page_shift) + (key & mask)) * CR + 8 * g;
  }
  f32x4 ak[2][JK], av[2][JV];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int j = 0; j < JK; ++j) ak[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < JV; ++j) av[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // the matrices' rows go through LDS in pieces of 64 latent channels, which all four waves read (rows 32 bytes apart from their data:
  // no bank conflicts), the latents straight into operands; the next piece is on its way beside the current one's products
  __shared__ __attribute__((aligned(16))) bf16_t ws[2][(D + E) * LX_ROW];
  constexpr int PER = (D + E) * 8 / 256;
  bf16x8 rows[PER], x[2][2][2];
  auto fetch = [&](int c) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int row = (i * 256 + (int)threadIdx.x) / 8, at = c + threadIdx.x % 8 * 8;
      rows[i] = *reinterpret_cast<const bf16x8*>((row < D ? p.uk + ((size_t)h * D + row) * p.C : p.uv + ((size_t)h * E + row - D) * p.C) + at);
    }
  };
  auto fetch_latents = [&](int buf, int c) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t) x[buf][s][t] = *reinterpret_cast<const bf16x8*>(lat[t] + c + 32 * s);
  };
  auto park = [&](int buf) {
#pragma unroll
    for (int i = 0; i < PER; ++i) *reinterpret_cast<bf16x8*>(&ws[buf][(i * 256 + threadIdx.x) / 8 * LX_ROW + threadIdx.x % 8 * 8]) = rows[i];
  };
  auto multiply = [&](int buf) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      bf16x8 k[JK], v[JV];
#pragma unroll
      for (int j = 0; j < JK; ++j) k[j] = *reinterpret_cast<const bf16x8*>(&ws[buf][(16 * j + r) * LX_ROW + 32 * s + 8 * g]);
#pragma unroll
      for (int j = 0; j < JV; ++j) v[j] = *reinterpret_cast<const bf16x8*>(&ws[buf][(D + 16 * j + r) * LX_ROW + 32 * s + 8 * g]);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int j = 0; j < JK; ++j) ak[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[j], x[buf][s][t], ak[t][j], 0, 0, 0);  // [channel][key]
#pragma unroll
        for (int j = 0; j < JV; ++j) av[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[buf][s][t], v[j], av[t][j], 0, 0, 0);  // [key][channel]
      }
    }
  };
  fetch(0);
  fetch_latents(0, 0);
  park(0);
  for (int c = 0; c < p.C; c += 2 * 64) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (c + 64 * u >= p.C) break;
      __syncthreads();
      const bool more = c + 64 * (u + 1) < p.C;
      if (more) {
        fetch(c + 64 * (u + 1));
        fetch_latents(u ^ 1, c + 64 * (u + 1));
      }
      multiply(u);
      if (more) park(u ^ 1);
    }
  }
  const int block = (key0 + 32 * wave) / LP_KEYS, in_block = 32 * (wave & 1);
  bf16_t* to = p.scratch + (((size_t)blockIdx.z * p.blocks + block) * p.H + h) * LP_KEYS * (KD + E);
  auto narrow = [](f32x4 a) { return bf16x4{(bf16_t)a[0], (bf16_t)a[1], (bf16_t)a[2], (bf16_t)a[3]}; };
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    bf16_t* krow = to + (in_block + 16 * t + r) * KD;
#pragma unroll
    for (int j = 0; j < JK; ++j) *reinterpret_cast<bf16x4*>(krow + 16 * j + 4 * g) = narrow(ak[t][j]);
#pragma unroll
    for (int d = 0; d < R; d += 32) *reinterpret_cast<bf16x8*>(krow + D + d + 8 * g) = *reinterpret_cast<const bf16x8*>(lat[t] + p.C + d);
#pragma unroll
    for (int j = 0; j < JV; ++j) *reinterpret_cast<bf16x4*>(to + LP_KEYS * KD + (16 * j + r) * LP_KEYS + in_block + 8 * g + 4 * t) = narrow(av[t][j]);
  }
}

template <int D, int R, int E>
__global__ __launch_bounds__(256, D == 64 ? 3 : 1) void latent_prompt_kernel(LatentPromptParams p) {
  constexpr int KD = D + R, KS = KD / 32, VT = E / 16, KROW = KD + 16, VROW = LP_KEYS + 16;
  constexpr int BLOCK = LP_KEYS * (KD + E), BUF = LP_KEYS * KROW + E * VROW, PER = BLOCK / 8 / 256;
  static_assert(BLOCK % (8 * 256) == 0 && KD % 32 == 0 && R % 32 == 0 && E % 16 == 0, "pieces of 16 bytes, 256 threads");
  __shared__ __attribute__((aligned(16))) bf16_t lds[2 * BUF];
  const int h = blockIdx.x % p.H, tile = p.n_tiles - 1 - (int)blockIdx.x / p.H;  // the tiles behind have the most keys and start first
  const int* info = p.tiles + 8 * tile;
  const int t0 = info[1], n = info[3], kv = info[4];
  if (t0 >= n || t0 % LP_TOKENS) return;  // (the tiles of 32 tokens in between belong to the workgroup of the one in front)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, g = lane >> 4;
  const int base = kv - n + t0, n_tok = min(LP_TOKENS, n - t0), hi = base + n_tok - 1;
  auto first_key = [&](int pos) { return p.window > 0 ? max(0, pos - p.window + 1) : 0; };
  const int w0 = 16 * wave;  // the wave's first token of the tile
  const bool works = w0 < n_tok;
  const int wave_lo = first_key(base + w0), wave_hi = base + min(w0 + 16, n_tok) - 1;
  const int tok = min(w0 + c, n_tok - 1), pos = base + tok, lo = first_key(pos);
  const size_t row = (size_t)info[2] + t0 + tok;
  bf16x8 q[KS];
  {
    const bf16_t* qr = p.q + row * p.q_stride + (size_t)h * KD;
#pragma unroll
    for (int i = 0; i < D / 32; ++i) q[i] = *reinterpret_cast<const bf16x8*>(qr + 32 * i + 8 * g);
    // the rotated part: both channels of a pair are read, this lane's eight kept
#pragma unroll
    for (int i = 0; i < R / 32; ++i) {
      const int d0 = 32 * i + 8 * g, other = p.form.interleaved ? d0 : (d0 < R / 2 ? d0 + R / 2 : d0 - R / 2);
      const bf16x8 own = *reinterpret_cast<const bf16x8*>(qr + D + d0), far = *reinterpret_cast<const bf16x8*>(qr + D + other);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int pair = p.form.interleaved ? (d0 + e) / 2 : (d0 + e) % (R / 2);
        const bool second = p.form.interleaved ? e & 1 : d0 >= R / 2;
        const float mine = to_f(own[e]), partner = p.form.interleaved ? to_f(own[e ^ 1]) : to_f(far[e]);
        float cs, sn, a, b;
        rope_cos_sin(p.form, pos, p.inv_freq[pair], cs, sn);
        rope_turn(second ? partner : mine, second ? mine : partner, cs, sn, a, b);
        q[D / 32 + i][e] = from_f<bf16_t>(second ? b : a);
      }
    }
  }
  const int b0 = first_key(base) / LP_KEYS, b1 = hi / LP_KEYS + 1;
  const bf16_t* blocks = p.scratch + ((size_t)info[6] * p.blocks * p.H + h) * BLOCK;
  bf16x8 reg[PER];
  auto fetch = [&](int b) {
#pragma unroll
    for (int i = 0; i < PER; ++i) reg[i] = *reinterpret_cast<const bf16x8*>(blocks + (size_t)b * p.H * BLOCK + 8 * (i * 256 + tid));
  };
  auto park = [&](int buf) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int piece = i * 256 + tid, v = piece - LP_KEYS * KD / 8;
      const int at = v < 0 ? piece / (KD / 8) * KROW + piece % (KD / 8) * 8 : LP_KEYS * KROW + v / 8 * VROW + v % 8 * 8;
      *reinterpret_cast<bf16x8*>(&lds[buf * BUF + at]) = reg[i];
    }
  };
  f32x4 o[VT];
  float m = -INFINITY, l = 0.f;  // l: this lane's keys
#pragma unroll
  for (int t = 0; t < VT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  // a block's part of a wave's 16 tokens; EDGE: some token of the workgroup does not see all of its keys
  auto work = [&](auto edge, int k0, int buf) {
    constexpr bool EDGE = decltype(edge)::value;
    const bf16_t* ks = lds + buf * BUF + c * KROW + 8 * g;
    const bf16_t* vs = lds + buf * BUF + LP_KEYS * KROW + c * VROW + 8 * g;
    f32x4 s[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      bf16x8 k[KS];
#pragma unroll
      for (int i = 0; i < KS; ++i) k[i] = *reinterpret_cast<const bf16x8*>(ks + 16 * t * KROW + 32 * i);
      s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < KS; ++i) s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[i], q[i], s[t], 0, 0, 0);
    }
    bf16x8 w[2];
    float top = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = k0 + 16 * t + 4 * g + i;
        if (EDGE && (key < lo || key > pos)) s[t][i] = -INFINITY;
        top = fmaxf(top, s[t][i]);
      }
    top = fmaxf(top, __shfl_xor(top, 16, 64));
    top = fmaxf(top, __shfl_xor(top, 32, 64));
    const float m_new = fmaxf(m, top), ref = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f((m - ref) * p.scale_log2), shift = -ref * p.scale_log2;
    const bool moved = __any(m_new != m);
    m = m_new;
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = __builtin_amdgcn_exp2f(fmaf(s[t][i], p.scale_log2, shift));
        sum += e;
        w[t / 2][4 * (t % 2) + i] = (bf16_t)e;
      }
    if (moved) {
      l *= alpha;
#pragma unroll
      for (int t = 0; t < VT; ++t) o[t] *= alpha;
    }
    l += sum;
    unsigned odd = 0;
    if (EDGE) {  // an infinite value or one that is no number among those that some token does not see: all bits of its exponent are set
#pragma unroll
      for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const uint4 v = *reinterpret_cast<const uint4*>(vs + 16 * t * VROW + 32 * i);
          const unsigned pairs[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) odd |= (pairs[e] & 0x7f807f80u) + 0x00800080u;
        }
    }
    if (!EDGE || !__any(odd & 0x80008000u)) {
#pragma unroll
      for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(vs + 16 * t * VROW + 32 * i), w[i], o[t], 0, 0, 0);
    } else {  // a weight of zero would make it that token's too, so each token adds the keys it sees only
      const bf16_t* at = lds + buf * BUF + LP_KEYS * KROW + 4 * g * VROW;
#pragma unroll
      for (int x = 0; x < 16; ++x)  // the weight that lanes 16 gg + c hold in place x % 8 of w[x / 8] is of key 32 (x / 8) + 16 (x % 8 / 4) + 4 gg + x % 4
        for (int gg = 0; gg < 4; ++gg) {
          const int key = k0 + 32 * (x / 8) + 16 * (x % 8 / 4) + 4 * gg + x % 4;
          const float weight = __shfl(to_f(w[x / 8][x % 8]), 16 * gg + c, 64);
          if (key < lo || key > pos) continue;
#pragma unroll
          for (int t = 0; t < VT; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) o[t][j] = fmaf(weight, to_f(at[(16 * t + j) * VROW + 32 * (x / 8) + 8 * gg + x % 8]), o[t][j]);
        }
    }
  };
  fetch(b0);
  park(0);
  for (int b = b0; b < b1; ++b) {
    const int buf = (b - b0) & 1, k0 = b * LP_KEYS;
    __syncthreads();
    if (b + 1 < b1) fetch(b + 1);
    if (works && k0 <= wave_hi && k0 + LP_KEYS > wave_lo) {
      if (k0 >= first_key(hi) && k0 + LP_KEYS - 1 <= base)
        work(std::false_type{}, k0, buf);
      else
        work(std::true_type{}, k0, buf);
    }
    if (b + 1 < b1) park(buf ^ 1);
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (w0 + c >= n_tok) return;
  if (p.sink_logits) l += exp2f(p.sink_logits[h] * 1.4426950408889634f - m * p.scale_log2);
  const float f = (p.gate ? p.gate[row * p.H + h] : 1.f) / l;
#pragma unroll
  for (int t = 0; t < VT; ++t) {
    f32x4 v = o[t] * f;
    if (p.zgate) {
      const bf16x4 z = *reinterpret_cast<const bf16x4*>(p.zgate + row * p.z_stride + (size_t)h * E + 16 * t + 4 * g);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] /= 1.f + expf(-to_f(z[i]));
    }
    *reinterpret_cast<bf16x4*>(p.out + (row * p.H + h) * E + 16 * t + 4 * g) = bf16x4{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]};
  }
}

template <int D, int R, int E>
static void launch_latent_prompt(const LatentPromptParams& p, int portions, hipStream_t stream) {
  latent_expand_kernel<D, R, E><<<dim3((p.blocks + 1) / 2, p.H, portions), 256, 0, stream>>>(p);
  latent_prompt_kernel<D, R, E><<<p.n_tiles * p.H, 256, 0, stream>>>(p);
}

// Elements of scratch a block of 64 keys takes for all heads; 0: the sizes are not taken.
extern "C" long ns_latent_prompt_block(int H, int D, int R, int E) {
  return (D == 64 && R == 32 && E == 64) || (D == 128 && R == 64 && E == 128) ? (long)H * LP_KEYS * (D + R + E) : 0;
}

// ``scratch``: portions * blocks * ns_latent_prompt_block elements; ``blocks`` (even): blocks of 64 keys that the longest portion's keys take at most.
extern "C" int ns_latent_prompt(void* out, const void* q, int q_stride, const void* latents, const void* uk, const void* uv, void* scratch,
                                const int* tiles, const int* block_table, int table_stride, const float* inv_freq, const float* gate, const void* zgate,
                                int z_stride, const float* sink_logits, int n_tiles, int portions, int blocks, int H, int D, int R, int E, int C,
                                int page_size, int window, float scale, int interleaved, float factor, hipStream_t stream) {
  if (n_tiles <= 0 || portions <= 0 || portions > 65535 || blocks <= 0 || blocks % 2 || H <= 0 || H > 65535 || C <= 0 || window < 0 || !(scale > 0.f) ||
      (long)n_tiles * H > 0x7fffffffL)
    return NS_ERR_BAD_ARG;
  if (!ns_latent_prompt_block(H, D, R, E) || C % 64 || page_size < 1 || page_size & (page_size - 1) || q_stride % 8 || (zgate && z_stride % 4) ||
      (((uintptr_t)out | (uintptr_t)zgate) & 7) || (((uintptr_t)q | (uintptr_t)latents | (uintptr_t)uk | (uintptr_t)uv | (uintptr_t)scratch) & 15))
    return NS_ERR_UNSUPPORTED;
  int shift = 0;
  while (1 << shift < page_size) ++shift;
  const LatentPromptParams p{(const bf16_t*)latents, (const bf16_t*)uk, (const bf16_t*)uv, (bf16_t*)scratch, (const bf16_t*)q, (bf16_t*)out, tiles,
                             block_table, inv_freq, gate, (const bf16_t*)zgate, sink_logits, q_stride, z_stride, table_stride, n_tiles, H, C, shift, blocks,
                             window, scale * 1.4426950408889634f, RopeForm{R, interleaved, factor}};
  if (D == 64)
    launch_latent_prompt<64, 32, 64>(p, portions, stream);
  else
    launch_latent_prompt<128, 64, 128>(p, portions, stream);
  return ns_launch_status();
}

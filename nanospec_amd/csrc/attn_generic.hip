// Soft-max attention over the paged cache for any head size and either storage type, one query row
// and one head per workgroup.  It takes what the matrix cores' kernels do not: head or value sizes that are no multiples of
// theirs, odd pages, and in 32-bit the options that attn_f32.hip has not.  Keys are walked in
// fixed chunks of 256 counted from key 0, so a row's result does not depend on how the tokens were
// cut into steps or on what else is in the batch.
//
// Query row i of request b stands at position p = kv_len[b] - q_len[b] + i and sees the keys
// max(0, p - window + 1) .. p  (window == 0: 0 .. p).          (reference: model/attention.py:22-43)
// Options that the reference's attention does not have, each off at 0: ``chunk`` (a query also sees no key before the
// start of its own chunk, floor(p / chunk) * chunk, chunks counted from position 0), ``cap`` (a score s, after the
// scale, becomes cap * tanh(s / cap)), ``sink`` (the soft-max's denominator holds one more term of score 0 that has no
// value; with ``sink_logit`` [heads] the term is exp(sink_logit[h]) instead, a learned number that is not scaled), values of another size ``vd`` than the keys' ``hd``, and ``slope_exp`` (a bias by distance: head h of H loses
// 2^(-slope_exp (h + 1) / H) * (p - key) from its score, after the cap).
// Query head h reads key/value head h / (heads / kv_heads).    (reference: model/attention.py:33)
// K pages: [page][kv head][token][hd];  V pages: [page][kv head][vd][token].
#include "common.h"
#include "rope.h"

#define AG_THREADS 256
#define AG_MAX_VD 1024  // the largest value size (a thread holds up to four channels of the output)

template <typename T>
__global__ __launch_bounds__(AG_THREADS) void attn_generic_kernel(
    T* __restrict__ out, const T* __restrict__ q, int q_stride, const T* __restrict__ k_cache,
    const T* __restrict__ v_cache, const int* __restrict__ token_req, const int* __restrict__ positions,
    const int* __restrict__ block_table, int table_stride, int heads, int kv_heads, int hd, int vd, int page_size, float scale,
    int window, int chunk, float cap, int sink, const float* __restrict__ sink_logit, float slope_exp) {
  extern __shared__ float smem[];  // q_s[hd] | p_s[AG_THREADS] | scratch[16]
  float* q_s = smem;
  float* p_s = smem + hd;
  float* scratch = p_s + AG_THREADS;
  const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int kvh = h / (heads / kv_heads);
  const int pos = positions[t];
  const int* table = block_table + (size_t)token_req[t] * table_stride;
  const T* qrow = q + (size_t)t * q_stride + h * hd;
  for (int d = tid; d < hd; d += AG_THREADS) q_s[d] = to_f(qrow[d]) * scale;
  __syncthreads();
  int lo = window > 0 ? max(0, pos - window + 1) : 0;
  if (chunk > 0) lo = max(lo, pos / chunk * chunk);
  const float inv_cap = cap > 0.f ? 1.f / cap : 0.f;
  const float slope = slope_exp > 0.f ? exp2f(-slope_exp * (float)(h + 1) / (float)heads) : 0.f;
  float m = -INFINITY, l = 0.f;
  float acc[AG_MAX_VD / AG_THREADS] = {};  // channels tid, tid + 256, ... of the output
  for (int c0 = (lo / AG_THREADS) * AG_THREADS; c0 <= pos; c0 += AG_THREADS) {
    const int key = c0 + tid;
    const bool valid = key >= lo && key <= pos;
    float s = -INFINITY;
    if (valid) {
      const int page = table[key / page_size];
      const T* kr = k_cache + (((size_t)page * kv_heads + kvh) * page_size + key % page_size) * hd;
      float dot = 0.f;
      for (int d = 0; d < hd; ++d) dot = fmaf(q_s[d], to_f(kr[d]), dot);
      s = cap > 0.f ? cap * tanhf(dot * inv_cap) : dot;
      s -= slope * (float)(pos - key);
    }
    const float m_new = fmaxf(m, block_max(s, scratch));
    const float p = valid ? expf(s - m_new) : 0.f;
    p_s[tid] = p;
    const float csum = block_sum(p, scratch);  // its barriers also publish p_s
    const float alpha = m == -INFINITY ? 0.f : expf(m - m_new);
    l = l * alpha + csum;
    m = m_new;
#pragma unroll
    for (int ci = 0; ci < AG_MAX_VD / AG_THREADS; ++ci) {
      const int ch = tid + ci * AG_THREADS;
      if (ch < vd) {
        float a = acc[ci] * alpha;
        const int hi = min(AG_THREADS, pos - c0 + 1);
        for (int j = max(0, lo - c0); j < hi; ++j) {
          const int kj = c0 + j;
          const int page = table[kj / page_size];
          const T* vp = v_cache + (((size_t)page * kv_heads + kvh) * vd + ch) * page_size + kj % page_size;
          a = fmaf(p_s[j], to_f(*vp), a);
        }
        acc[ci] = a;
      }
    }
    __syncthreads();
  }
  if (sink_logit)
    l += expf(sink_logit[h] - m);  // the learned term, in the units of the running maximum
  else if (sink)
    l += expf(-m);  // the term of score 0
#pragma unroll
  for (int ci = 0; ci < AG_MAX_VD / AG_THREADS; ++ci)
    if (tid + ci * AG_THREADS < vd) out[((size_t)t * heads + h) * vd + tid + ci * AG_THREADS] = from_f<T>(acc[ci] / l);
}

extern "C" int ns_attn_generic(void* out, const void* q, int q_stride, const void* k_cache, const void* v_cache,
                               const int* token_req, const int* positions, const int* block_table, int table_stride,
                               int n_tokens, int heads, int kv_heads, int hd, int vd, int page_size, float scale, int window,
                               int chunk, float cap, int sink, const float* sink_logit, float slope_exp, int dtype, hipStream_t stream) {
  if (n_tokens <= 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads || hd <= 0 || hd > 1024 || vd <= 0 || vd > AG_MAX_VD || page_size <= 0 ||
      window < 0 || chunk < 0 || cap < 0.f || slope_exp < 0.f)
    return NS_ERR_BAD_ARG;
  if (heads > 65535) return NS_ERR_BAD_ARG;
  dim3 grid(n_tokens, heads);
  const size_t smem = (size_t)(hd + AG_THREADS + 16) * sizeof(float);
  if (dtype == NS_DTYPE_F32)
    attn_generic_kernel<float><<<grid, AG_THREADS, smem, stream>>>((float*)out, (const float*)q, q_stride, (const float*)k_cache,
        (const float*)v_cache, token_req, positions, block_table, table_stride, heads, kv_heads, hd, vd, page_size, scale, window, chunk, cap, sink, sink_logit, slope_exp);
  else if (dtype == NS_DTYPE_BF16)
    attn_generic_kernel<bf16_t><<<grid, AG_THREADS, smem, stream>>>((bf16_t*)out, (const bf16_t*)q, q_stride, (const bf16_t*)k_cache,
        (const bf16_t*)v_cache, token_req, positions, block_table, table_stride, heads, kv_heads, hd, vd, page_size, scale, window, chunk, cap, sink, sink_logit, slope_exp);
  else
    return NS_ERR_UNSUPPORTED;
  return ns_launch_status();
}

// ------------------------------------------------------------------------------------------------
// What stands between an attention layer's projections and its scores, in pieces of 8 bytes: biases, the RMS norm of a head or of a whole projection, the rotation, keys and values
// into their pages.  The three entry points below take these kernels where sizes and addresses allow (``kv_rows_take``) and the plain ones, an element a lane, elsewhere.
// A workgroup is a token.  L neighbouring lanes take a head's channels, two pieces of H each (``unit_of``): with the half-split pairing a piece and its partners, else one
// after the other.  The cosines and sines of a token are made once for all its heads (with them in every head a third of the time).  Of the tokens of a request that stand side by
// side in a run of whole 16 bytes of a value page the first writes the values of all, 16 bytes a store; an element a store they are 2 bytes in every line of 32.
// Bound by launches and the row's way from memory and back, us before (plain) and now, bfloat16, 2,048 tokens, 32 heads of 64 over 8: norm a head 26.8 / 21.8 -> 18.2 / 11.8 (alone / beside
// two others), with weights, biases and rotation, 1,531 tokens, 29.8 / 24.0 -> 17.1 / 10.9; norm of the projection with rotation, 512 tokens, 15.4 / 8.5 -> 10.5 / 5.6, 8 tokens 6.9 / 4.1 -> 4.7 / 3.2.
// ------------------------------------------------------------------------------------------------
template <typename T>
struct KvRows {
  T* qkv;
  const T *bias, *qw, *kw;  // (each may be null)
  const int *positions, *token_req, *block_table;
  const float* inv_freq;
  T *k_cache, *v_cache;
  int stride, table_stride, n_tokens, heads, kv_heads, hd, vd, page_size, lanes, shares;  // kv_heads 0: no keys and values of its own
  float eps;
  RopeForm form;
  int norm_q, norm_k, v_is_k;
  int first;  // head: the queries before it stay as they are
  const T *lambda, *v_other;  // values <- (1 - lambda) values + lambda v_other
  T* v_keep;
  int v_other_stride, v_keep_stride;
};

template <typename T>
struct KvPiece {
  static constexpr int H = 8 / sizeof(T);
  typedef T type __attribute__((ext_vector_type(H)));
};

// the first channels of a lane's two pieces
template <typename T>
__device__ __forceinline__ void unit_of(const KvRows<T>& p, int l, int& d1, int& d2) {
  constexpr int H = KvPiece<T>::H;
  const int turned = p.form.interleaved ? 0 : p.form.rot / 2 / H;  // lanes whose pieces are partners
  d1 = l < turned ? l * H : 2 * l * H;
  d2 = d1 + (l < turned ? p.form.rot / 2 : H);
}

template <typename T>
__device__ __forceinline__ void load_piece(const T* row, const T* bias, float* v) {
  constexpr int H = KvPiece<T>::H;
  const auto r = *reinterpret_cast<const typename KvPiece<T>::type*>(row);
#pragma unroll
  for (int e = 0; e < H; ++e) v[e] = to_f((T)r[e]);
  if (bias) {
    const auto b = *reinterpret_cast<const typename KvPiece<T>::type*>(bias);
#pragma unroll
    for (int e = 0; e < H; ++e) v[e] += to_f((T)b[e]);
  }
}
template <typename T>
__device__ __forceinline__ void store_piece(T* to, const float* v) {
  typename KvPiece<T>::type o;
#pragma unroll
  for (int e = 0; e < KvPiece<T>::H; ++e) o[e] = from_f<T>(v[e]);
  *reinterpret_cast<typename KvPiece<T>::type*>(to) = o;
}

// A unit's channels times ``f`` (if its part is normed) and the weights, rotated, and to where they belong.  ``w``: the head's weights or null.
template <typename T>
__device__ __forceinline__ void finish_unit(const KvRows<T>& p, T* row, int h, int d1, int d2, float* a, float* b, float f, bool normed, const T* w, const float* cs, int page,
                                            int slot) {
  constexpr int H = KvPiece<T>::H;
  if (normed) {
#pragma unroll
    for (int e = 0; e < H; ++e) a[e] *= f, b[e] *= f;
  }
  if (w) {
    float wa[H], wb[H];
    load_piece<T>(w + d1, nullptr, wa), load_piece<T>(w + d2, nullptr, wb);
#pragma unroll
    for (int e = 0; e < H; ++e) a[e] *= wa[e], b[e] *= wb[e];
  }
  const int half = p.form.rot / 2;
  if (p.form.interleaved) {
#pragma unroll
    for (int e = 0; e < H; e += 2) {
      if (d1 + e < p.form.rot) rope_turn(a[e], a[e + 1], cs[(d1 + e) / 2], cs[half + (d1 + e) / 2], a[e], a[e + 1]);
      if (d2 + e < p.form.rot) rope_turn(b[e], b[e + 1], cs[(d2 + e) / 2], cs[half + (d2 + e) / 2], b[e], b[e + 1]);
    }
  } else if (d1 < half) {
#pragma unroll
    for (int e = 0; e < H; ++e) rope_turn(a[e], b[e], cs[d1 + e], cs[half + d1 + e], a[e], b[e]);
  }
  T* to = h < p.heads ? row + (size_t)h * p.hd : p.k_cache + (((size_t)page * p.kv_heads + (h - p.heads)) * p.page_size + slot) * p.hd;
  store_piece(to + d1, a), store_piece(to + d2, b);
}

// The values of a token, or of a run of tokens by its first; part ``part`` of ``parts`` of them.
template <typename T>
__device__ __forceinline__ void write_values(const KvRows<T>& p, int t, int part, int parts) {
  constexpr int H = KvPiece<T>::H, V = 2 * H;
  typedef T run_t __attribute__((ext_vector_type(V)));
  const int lane = threadIdx.x % NS_WAVE, req = p.token_req[t], pos = p.positions[t], slot = pos % p.page_size, nq = p.heads * p.hd;
  const int page = p.block_table[(size_t)req * p.table_stride + pos / p.page_size];
  int count = 1;
  if (p.page_size % V == 0) {  // lane i asks whether token t - 1 + i goes on with this one's run (one after the other that is a trip to memory each)
    const int other = min(max(t - 1 + lane, 0), p.n_tokens - 1), place = pos - 1 + lane;
    const bool goes_on = lane <= V && other == t - 1 + lane && p.token_req[other] == req && p.positions[other] == place && place / V == pos / V;
    const unsigned long long with = __ballot(goes_on);
    if (with & 1) return;
    count = __ffsll((long long)~(with >> 1)) - 1;
  }
  const int at = p.v_is_k ? nq : nq + p.kv_heads * p.hd;  // of the values in a row
  const float lam = p.lambda && p.v_other ? to_f(p.lambda[0]) : 0.f;
  // (neighbouring lanes have neighbouring channels, whose runs in a page are neighbours: four channels a lane, whose stores lie 128 bytes apart, 19.9 / 13.1 us in the first line above)
  for (int c = part * blockDim.x + threadIdx.x; c < p.kv_heads * p.vd; c += parts * blockDim.x) {
    T* to = p.v_cache + ((size_t)page * p.kv_heads * p.vd + c) * p.page_size + slot;  // (a page's heads and their channels lie one behind the other)
    const T *from = p.qkv + (size_t)t * p.stride + at + c, *from_other = p.v_other ? p.v_other + (size_t)t * p.v_other_stride + c : nullptr;
    const float bias = p.bias ? to_f(p.bias[at + c]) : 0.f;
    auto value = [&](int i, T v, T other) {  // of token t + i, from its own and the other layer's
      float z = to_f(v) + bias;
      if (from_other) z = (1.f - lam) * z + lam * to_f(other);
      v = from_f<T>(z);
      if (p.v_keep) p.v_keep[(size_t)(t + i) * p.v_keep_stride + c] = v;
      return v;
    };
    if (count == V) {  // (all loads ahead of the first use)
      run_t v, other = {};
#pragma unroll
      for (int i = 0; i < V; ++i) v[i] = from[(size_t)i * p.stride];
      if (from_other) {
#pragma unroll
        for (int i = 0; i < V; ++i) other[i] = from_other[(size_t)i * p.v_other_stride];
      }
#pragma unroll
      for (int i = 0; i < V; ++i) v[i] = value(i, v[i], other[i]);
      *reinterpret_cast<run_t*>(to) = v;
    } else {
      for (int i = 0; i < count; ++i) to[i] = value(i, from[(size_t)i * p.stride], from_other ? from_other[(size_t)i * p.v_other_stride] : from_f<T>(0.f));
    }
  }
}

// Few tokens: ``shares`` workgroups for a token's heads and more for its values, a value a thread (8 tokens 6.7 -> 3.8 us, 64 tokens of 40 heads of 128 6.4 -> 5.5); many: one for all of it.
template <typename T>
__device__ __forceinline__ bool only_values(const KvRows<T>& p) { return (int)blockIdx.y >= p.shares; }
template <typename T>
__device__ __forceinline__ bool values_too(const KvRows<T>& p) { return p.kv_heads && gridDim.y == 1; }

// A norm over every head.
template <typename T>
__global__ __launch_bounds__(512) void head_rows_kernel(const KvRows<T> p) {
  constexpr int H = KvPiece<T>::H;
  extern __shared__ float cs[];  // cos[rot / 2] | sin[rot / 2]
  const int t = blockIdx.x;
  if (only_values(p)) return write_values(p, t, blockIdx.y - p.shares, gridDim.y - p.shares);
  const int pos = p.positions[t], half = p.form.rot / 2;
  T* row = p.qkv + (size_t)t * p.stride;
  const int page = p.kv_heads ? p.block_table[(size_t)p.token_req[t] * p.table_stride + pos / p.page_size] : 0, slot = pos % p.page_size;
  if (half) {
    for (int j = threadIdx.x; j < half; j += blockDim.x) rope_cos_sin(p.form, pos, p.inv_freq[j], cs[j], cs[half + j]);
    __syncthreads();
  }
  // (a head's lanes stand in one wave and go round together)
  for (int u = blockIdx.y * blockDim.x + threadIdx.x; u < (p.heads - p.first + p.kv_heads) * p.lanes; u += p.shares * blockDim.x) {
    const int h = p.first + u / p.lanes;
    const bool is_q = h < p.heads, normed = is_q ? p.norm_q : p.norm_k;
    int d1, d2;
    unit_of(p, u % p.lanes, d1, d2);
    float a[H], b[H];
    load_piece<T>(row + (size_t)h * p.hd + d1, p.bias ? p.bias + (size_t)h * p.hd + d1 : nullptr, a);
    load_piece<T>(row + (size_t)h * p.hd + d2, p.bias ? p.bias + (size_t)h * p.hd + d2 : nullptr, b);
    float ss = 0.f;
    if (normed) {
#pragma unroll
      for (int e = 0; e < H; ++e) ss = fmaf(a[e], a[e], ss);
#pragma unroll
      for (int e = 0; e < H; ++e) ss = fmaf(b[e], b[e], ss);
      for (int o = 1; o < p.lanes; o <<= 1) ss += __shfl_xor(ss, o, NS_WAVE);
    }
    finish_unit(p, row, h, d1, d2, a, b, 1.f / sqrtf(ss / (float)p.hd + p.eps), normed, is_q ? p.qw : p.kw, cs, page, slot);
  }
  if (values_too(p)) write_values(p, t, 0, 1);
}

// A norm over all heads of q and one over all of k; a thread keeps up to UNITS units between the sums and what follows them.
#define WHOLE_UNITS 2
template <typename T>
__global__ __launch_bounds__(1024) void whole_rows_kernel(const KvRows<T> p) {
  constexpr int H = KvPiece<T>::H;
  extern __shared__ float cs[];  // cos[rot / 2] | sin[rot / 2]
  __shared__ float sums[2][16];
  const int t = blockIdx.x;
  if (only_values(p)) return write_values(p, t, blockIdx.y - p.shares, gridDim.y - p.shares);
  const int pos = p.positions[t], half = p.form.rot / 2, units = (p.heads + p.kv_heads) * p.lanes;
  T* row = p.qkv + (size_t)t * p.stride;
  const int page = p.block_table[(size_t)p.token_req[t] * p.table_stride + pos / p.page_size], slot = pos % p.page_size;
  float a[WHOLE_UNITS][H], b[WHOLE_UNITS][H], sq = 0.f, sk = 0.f;
#pragma unroll
  for (int i = 0; i < WHOLE_UNITS; ++i) {
    const int u = threadIdx.x + i * blockDim.x, h = u / p.lanes;
    if (u >= units) continue;
    int d1, d2;
    unit_of(p, u % p.lanes, d1, d2);
    load_piece<T>(row + (size_t)h * p.hd + d1, p.bias ? p.bias + (size_t)h * p.hd + d1 : nullptr, a[i]);
    load_piece<T>(row + (size_t)h * p.hd + d2, p.bias ? p.bias + (size_t)h * p.hd + d2 : nullptr, b[i]);
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < H; ++e) ss = fmaf(a[i][e], a[i][e], ss);
#pragma unroll
    for (int e = 0; e < H; ++e) ss = fmaf(b[i][e], b[i][e], ss);
    (h < p.heads ? sq : sk) += ss;
  }
  for (int j = threadIdx.x; j < half; j += blockDim.x) rope_cos_sin(p.form, pos, p.inv_freq[j], cs[j], cs[half + j]);
  sq = wave_sum(sq), sk = wave_sum(sk);
  if (threadIdx.x % NS_WAVE == 0) sums[0][threadIdx.x / NS_WAVE] = sq, sums[1][threadIdx.x / NS_WAVE] = sk;
  __syncthreads();
  sq = sk = 0.f;
  for (int i = 0; i < (int)blockDim.x / NS_WAVE; ++i) sq += sums[0][i], sk += sums[1][i];
  const float fq = 1.f / sqrtf(sq / (float)(p.heads * p.hd) + p.eps), fk = 1.f / sqrtf(sk / (float)(p.kv_heads * p.hd) + p.eps);
#pragma unroll
  for (int i = 0; i < WHOLE_UNITS; ++i) {
    const int u = threadIdx.x + i * blockDim.x, h = u / p.lanes;
    if (u >= units) continue;
    const bool is_q = h < p.heads;
    int d1, d2;
    unit_of(p, u % p.lanes, d1, d2);
    const T* w = is_q ? p.qw : p.kw;
    finish_unit(p, row, h, d1, d2, a[i], b[i], is_q ? fq : fk, is_q ? p.norm_q : p.norm_k, w ? w + (size_t)(is_q ? h : h - p.heads) * p.hd : nullptr, cs, page, slot);
  }
  if (values_too(p)) write_values(p, t, 0, 1);
}

// Whether the kernels above take these sizes and addresses; sets ``lanes``.
template <typename T>
static bool kv_rows_take(KvRows<T>& p) {
  constexpr int H = KvPiece<T>::H;
  const int rot = p.form.rot;
  if (p.hd % (2 * H) || p.vd % H || p.stride % H || (p.v_other && p.v_other_stride % H) || (p.v_keep && p.v_keep_stride % H)) return false;
  p.lanes = p.hd / (2 * H);
  if (p.lanes > NS_WAVE || (p.lanes & (p.lanes - 1))) return false;
  if (rot && !p.form.interleaved && (rot / 2 % H || (p.hd - rot) % (2 * H))) return false;
  if (((uintptr_t)p.qkv | (uintptr_t)p.bias | (uintptr_t)p.qw | (uintptr_t)p.kw | (uintptr_t)p.k_cache | (uintptr_t)p.v_other | (uintptr_t)p.v_keep) & 7) return false;
  return p.kv_heads == 0 || ((uintptr_t)p.v_cache & 15) == 0;
}

// (a workgroup that writes a run's values behind its heads is the last to end while the units have few of them: us, values behind the heads and by workgroups of their own, bfloat16, a norm a head and a
// norm of the projection with rotation: 300 tokens of 32 heads of 128 over 8 9.8 and 6.2, 10.8 and 6.5; 700 11.7 and 9.8, 12.9 and 11.2; of 64 8.0 and 6.7, 10.0 and 6.7; 1,024 of 128 11.7 and 14.9, of 64 8.2
// and 8.9)
#define FEW_TOKENS 1024
template <typename T>
static dim3 kv_rows_grid(const KvRows<T>& p, int threads) {
  const int parts = p.n_tokens < FEW_TOKENS ? (p.kv_heads * p.vd + threads - 1) / threads : 0;  // (of a token's values; none of its own: none)
  return dim3(p.n_tokens, p.shares + parts);
}

template <typename T>
static void launch_head_rows(KvRows<T> p, hipStream_t stream) {
  const int units = (p.heads - p.first + p.kv_heads) * p.lanes;
  p.shares = p.n_tokens < FEW_TOKENS ? (units + 255) / 256 : 1;
  const int rounds = p.shares > 1 ? p.shares : (units + 511) / 512;  // (as even as whole waves allow)
  int threads = ((units + rounds - 1) / rounds + NS_WAVE - 1) / NS_WAVE * NS_WAVE;
  if (threads < 256 && p.kv_heads * p.vd > threads) threads = p.kv_heads * p.vd < 256 ? (p.kv_heads * p.vd + NS_WAVE - 1) / NS_WAVE * NS_WAVE : 256;
  head_rows_kernel<T><<<kv_rows_grid(p, threads), threads, p.form.rot * sizeof(float), stream>>>(p);
}

// ------------------------------------------------------------------------------------------------
// What an attention layer without rotation does between its projections and its scores: the queries and keys of every
// head are divided by their root mean square over the head (``eps`` >= 0; a negative eps leaves them as they are), the
// queries in place; keys and values go into the pages of their positions.  A row of ``qkv`` is q [heads][hd], then, if
// the layer has keys and values of its own (``own_kv``), k [kv_heads][hd] and v [kv_heads][vd].
// ------------------------------------------------------------------------------------------------
// grid (tokens, Y): a wave takes one head's vector; the blocks after those copy the values, 1,024 a block.
template <typename T>
__global__ void unit_kv_write_kernel(T* __restrict__ qkv, int stride, const int* __restrict__ positions, const int* __restrict__ token_req,
                                     const int* __restrict__ block_table, int table_stride, T* __restrict__ k_cache, T* __restrict__ v_cache,
                                     int heads, int kv_heads, int hd, int vd, int page_size, float eps, int own_kv, int vec_blocks) {
  const int t = blockIdx.x, lane = threadIdx.x & (NS_WAVE - 1), wave = threadIdx.x / NS_WAVE;
  T* row = qkv + (size_t)t * stride;
  const int pos = positions[t];
  const int page = own_kv ? block_table[(size_t)token_req[t] * table_stride + pos / page_size] : 0;
  const int slot = pos % page_size;
  if ((int)blockIdx.y < vec_blocks) {
    const int vec = blockIdx.y * 4 + wave;
    if (vec >= heads + (own_kv ? kv_heads : 0)) return;
    T* p = row + (size_t)vec * hd;
    float f = 1.f;
    if (eps >= 0.f) {
      float ss = 0.f;
      for (int d = lane; d < hd; d += NS_WAVE) ss = fmaf(to_f(p[d]), to_f(p[d]), ss);
      ss = wave_sum(ss);
      f = 1.f / sqrtf(ss / (float)hd + eps);
    }
    if (vec < heads) {
      if (eps >= 0.f)
        for (int d = lane; d < hd; d += NS_WAVE) p[d] = from_f<T>(to_f(p[d]) * f);
    } else {
      T* dst = k_cache + (((size_t)page * kv_heads + (vec - heads)) * page_size + slot) * hd;
      for (int d = lane; d < hd; d += NS_WAVE) dst[d] = from_f<T>(to_f(p[d]) * f);
    }
    return;
  }
  if (own_kv) {
    const T* v = row + (size_t)(heads + kv_heads) * hd;
    const int part = blockIdx.y - vec_blocks;
    for (int i = part * 1024 + threadIdx.x; i < min(kv_heads * vd, (part + 1) * 1024); i += blockDim.x)
      v_cache[(((size_t)page * kv_heads + i / vd) * vd + i % vd) * page_size + slot] = v[i];
  }
}

extern "C" int ns_unit_kv_write(void* qkv, int stride, const int* positions, const int* token_req, const int* block_table, int table_stride,
                                void* k_cache, void* v_cache, int n_tokens, int heads, int kv_heads, int hd, int vd, int page_size,
                                float eps, int own_kv, int dtype, hipStream_t stream) {
  if (n_tokens <= 0 || heads <= 0 || kv_heads <= 0 || hd <= 0 || vd <= 0 || page_size <= 0) return NS_ERR_BAD_ARG;
  auto in_pieces = [&](auto* rows, auto* k, auto* v) {
    KvRows<typename std::remove_pointer<decltype(rows)>::type> p{};
    p.qkv = rows, p.k_cache = k, p.v_cache = v, p.positions = positions, p.token_req = token_req, p.block_table = block_table;
    p.stride = stride, p.table_stride = table_stride, p.n_tokens = n_tokens, p.heads = heads, p.kv_heads = own_kv ? kv_heads : 0, p.hd = hd, p.vd = vd, p.page_size = page_size;
    p.eps = eps, p.norm_q = p.norm_k = eps >= 0.f, p.first = eps >= 0.f ? 0 : heads;
    if (!kv_rows_take(p)) return false;
    if (own_kv || eps >= 0.f) launch_head_rows(p, stream);
    return true;
  };
  if (dtype == NS_DTYPE_F32 ? in_pieces((float*)qkv, (float*)k_cache, (float*)v_cache) : dtype == NS_DTYPE_BF16 && in_pieces((bf16_t*)qkv, (bf16_t*)k_cache, (bf16_t*)v_cache))
    return ns_launch_status();
  const int vec_blocks = (heads + (own_kv ? kv_heads : 0) + 3) / 4, copy_blocks = own_kv ? (kv_heads * vd + 1023) / 1024 : 0;
  if (vec_blocks + copy_blocks > 65535) return NS_ERR_BAD_ARG;
  const dim3 grid(n_tokens, vec_blocks + copy_blocks);
  if (dtype == NS_DTYPE_F32)
    unit_kv_write_kernel<float><<<grid, 256, 0, stream>>>((float*)qkv, stride, positions, token_req, block_table, table_stride,
                                                               (float*)k_cache, (float*)v_cache, heads, kv_heads, hd, vd, page_size, eps, own_kv, vec_blocks);
  else if (dtype == NS_DTYPE_BF16)
    unit_kv_write_kernel<bf16_t><<<grid, 256, 0, stream>>>((bf16_t*)qkv, stride, positions, token_req, block_table, table_stride,
                                                                (bf16_t*)k_cache, (bf16_t*)v_cache, heads, kv_heads, hd, vd, page_size, eps, own_kv, vec_blocks);
  else
    return NS_ERR_UNSUPPORTED;
  return ns_launch_status();
}

// ------------------------------------------------------------------------------------------------
// The same place in a layer whose projections carry biases, whose queries and keys pass an RMS norm over the WHOLE
// projection (all heads at once) with a weight per channel, and whose values may be mixed with the values that an earlier
// layer made for the same token:
//   q <- (q + bq) / sqrt(mean((q + bq)^2 over heads*hd) + eps) * qw         (in place)
//   k <- likewise over kv_heads*hd with kw                                   (into the K pages)
//   v <- v + bv;  v <- (1 - lambda) v + lambda v_other  if v_other is given   (into the V pages; also to v_keep if given)
// With ``form.rot`` > 0 the first ``rot`` channels of every head of q and k are then rotated by the token's position
// (``inv_freq`` [rot / 2]); a thread owns both channels of a pair.
// ``bias`` [heads*hd + kv_heads*(hd + vd)], ``qw``, ``kw`` and ``lambda`` (one value) may each be null.  One workgroup a token.
// ------------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(1024) void whole_norm_kv_write_kernel(
    T* __restrict__ qkv, int stride, const T* __restrict__ bias, const T* __restrict__ qw, const T* __restrict__ kw,
    const T* __restrict__ lambda, const T* __restrict__ v_other, int v_other_stride, T* __restrict__ v_keep, int v_keep_stride,
    const int* __restrict__ positions, const int* __restrict__ token_req, const int* __restrict__ block_table, int table_stride,
    T* __restrict__ k_cache, T* __restrict__ v_cache, int heads, int kv_heads, int hd, int vd, int page_size, float eps,
    const float* __restrict__ inv_freq, RopeForm form) {
  __shared__ float scratch[16];
  const int t = blockIdx.x;
  T* row = qkv + (size_t)t * stride;
  const int nq = heads * hd, nk = kv_heads * hd, nv = kv_heads * vd;
  const int pos = positions[t];
  const int page = block_table[(size_t)token_req[t] * table_stride + pos / page_size];
  const int slot = pos % page_size;
  float fq = 1.f, fk = 1.f;
  if (qw) {
    float ss = 0.f;
    for (int i = threadIdx.x; i < nq; i += blockDim.x) {
      const float v = to_f(row[i]) + (bias ? to_f(bias[i]) : 0.f);
      ss = fmaf(v, v, ss);
    }
    fq = 1.f / sqrtf(block_sum(ss, scratch) / (float)nq + eps);
  }
  if (kw) {
    float ss = 0.f;
    for (int i = threadIdx.x; i < nk; i += blockDim.x) {
      const float v = to_f(row[nq + i]) + (bias ? to_f(bias[nq + i]) : 0.f);
      ss = fmaf(v, v, ss);
    }
    fk = 1.f / sqrtf(block_sum(ss, scratch) / (float)nk + eps);
  }
  if (form.rot > 0) {
    // the rotated pairs of q and of k: item = (head among q heads then k heads, pair)
    const int half = form.rot / 2;
    for (int i = threadIdx.x; i < (heads + kv_heads) * half; i += blockDim.x) {
      const int h = i / half, j = i % half;
      const bool is_q = h < heads;
      int d1, d2;
      rope_pair_channels(form, j, d1, d2);
      const int at = h * hd;  // q heads and k heads follow each other in the row
      const T* w = is_q ? qw : kw;
      const int wat = is_q ? at : at - nq;
      const float f = is_q ? fq : fk;
      float a = to_f(row[at + d1]) + (bias ? to_f(bias[at + d1]) : 0.f), b = to_f(row[at + d2]) + (bias ? to_f(bias[at + d2]) : 0.f);
      if (w) a = a * f * to_f(w[wat + d1]), b = b * f * to_f(w[wat + d2]);
      float c, sn;
      rope_cos_sin(form, pos, inv_freq[j], c, sn);
      rope_turn(a, b, c, sn, a, b);
      if (is_q) {
        row[at + d1] = from_f<T>(a);
        row[at + d2] = from_f<T>(b);
      } else {
        T* kd = k_cache + (((size_t)page * kv_heads + (h - heads)) * page_size + slot) * hd;
        kd[d1] = from_f<T>(a);
        kd[d2] = from_f<T>(b);
      }
    }
  }
  for (int i = threadIdx.x; i < nq; i += blockDim.x) {
    if (i % hd < form.rot) continue;
    const float v = to_f(row[i]) + (bias ? to_f(bias[i]) : 0.f);
    row[i] = from_f<T>(qw ? v * fq * to_f(qw[i]) : v);
  }
  for (int i = threadIdx.x; i < nk; i += blockDim.x) {
    if (i % hd < form.rot) continue;
    const float v = to_f(row[nq + i]) + (bias ? to_f(bias[nq + i]) : 0.f);
    k_cache[(((size_t)page * kv_heads + i / hd) * page_size + slot) * hd + i % hd] = from_f<T>(kw ? v * fk * to_f(kw[i]) : v);
  }
  const float lam = (lambda && v_other) ? to_f(lambda[0]) : 0.f;
  for (int i = threadIdx.x; i < nv; i += blockDim.x) {
    float v = to_f(row[nq + nk + i]) + (bias ? to_f(bias[nq + nk + i]) : 0.f);
    if (v_other) v = (1.f - lam) * v + lam * to_f(v_other[(size_t)t * v_other_stride + i]);
    const T vs = from_f<T>(v);
    if (v_keep) v_keep[(size_t)t * v_keep_stride + i] = vs;
    v_cache[(((size_t)page * kv_heads + i / vd) * vd + i % vd) * page_size + slot] = vs;
  }
}

extern "C" int ns_whole_norm_kv_write(void* qkv, int stride, const void* bias, const void* qw, const void* kw, const void* lambda,
                                      const void* v_other, int v_other_stride, void* v_keep, int v_keep_stride, const int* positions,
                                      const int* token_req, const int* block_table, int table_stride, void* k_cache, void* v_cache,
                                      int n_tokens, int heads, int kv_heads, int hd, int vd, int page_size, float eps, const float* inv_freq,
                                      int rot, int interleaved, float factor, int dtype, hipStream_t stream) {
  if (n_tokens <= 0 || heads <= 0 || kv_heads <= 0 || hd <= 0 || vd <= 0 || page_size <= 0) return NS_ERR_BAD_ARG;
  if (rot < 0 || rot > hd || rot % 2 || (rot > 0 && !inv_freq)) return NS_ERR_BAD_ARG;
  const RopeForm form{rot, interleaved, factor};
  auto in_pieces = [&](auto* rows) {
    typedef typename std::remove_pointer<decltype(rows)>::type T;
    KvRows<T> p{};
    p.qkv = rows, p.bias = (const T*)bias, p.qw = (const T*)qw, p.kw = (const T*)kw, p.positions = positions, p.token_req = token_req, p.block_table = block_table;
    p.inv_freq = inv_freq, p.k_cache = (T*)k_cache, p.v_cache = (T*)v_cache, p.stride = stride, p.table_stride = table_stride, p.n_tokens = n_tokens;
    p.heads = heads, p.kv_heads = kv_heads, p.hd = hd, p.vd = vd, p.page_size = page_size, p.eps = eps, p.form = form, p.norm_q = qw != nullptr, p.norm_k = kw != nullptr;
    p.lambda = (const T*)lambda, p.v_other = (const T*)v_other, p.v_keep = (T*)v_keep, p.v_other_stride = v_other_stride, p.v_keep_stride = v_keep_stride;
    if (!kv_rows_take(p)) return false;
    const int units = (heads + kv_heads) * p.lanes, each = (units + WHOLE_UNITS - 1) / WHOLE_UNITS;
    if (each > 1024) return false;
    // few tokens: a unit a thread, if there are threads
    const int wanted = n_tokens <= 64 && units <= 1024 ? units : each;
    p.shares = 1;
    const int threads = (wanted + NS_WAVE - 1) / NS_WAVE * NS_WAVE;
    whole_rows_kernel<T><<<kv_rows_grid(p, threads), threads, rot * sizeof(float), stream>>>(p);
    return true;
  };
  if (dtype == NS_DTYPE_F32 ? in_pieces((float*)qkv) : dtype == NS_DTYPE_BF16 && in_pieces((bf16_t*)qkv)) return ns_launch_status();
  const int threads = n_tokens <= 64 && heads * hd > 1024 ? 1024 : 256;  // few tokens: more threads for each
  if (dtype == NS_DTYPE_F32)
    whole_norm_kv_write_kernel<float><<<n_tokens, threads, 0, stream>>>((float*)qkv, stride, (const float*)bias, (const float*)qw, (const float*)kw,
        (const float*)lambda, (const float*)v_other, v_other_stride, (float*)v_keep, v_keep_stride, positions, token_req, block_table,
        table_stride, (float*)k_cache, (float*)v_cache, heads, kv_heads, hd, vd, page_size, eps, inv_freq, form);
  else if (dtype == NS_DTYPE_BF16)
    whole_norm_kv_write_kernel<bf16_t><<<n_tokens, threads, 0, stream>>>((bf16_t*)qkv, stride, (const bf16_t*)bias, (const bf16_t*)qw, (const bf16_t*)kw,
        (const bf16_t*)lambda, (const bf16_t*)v_other, v_other_stride, (bf16_t*)v_keep, v_keep_stride, positions, token_req, block_table,
        table_stride, (bf16_t*)k_cache, (bf16_t*)v_cache, heads, kv_heads, hd, vd, page_size, eps, inv_freq, form);
  else
    return NS_ERR_UNSUPPORTED;
  return ns_launch_status();
}

// ------------------------------------------------------------------------------------------------
// Queries and keys with biases, an RMS norm per head whose weight [hd] all heads share, and a rotation of the head's first
// ``rot`` channels; optionally the key projection's raw output (bias added, no norm, no rotation) is stored as the values.
// A workgroup a token (few tokens: several, each with its share of the heads), a wave a head in turn.  A row of ``qkv`` is [q heads | k heads | v heads] (no v part if
// ``v_is_k``); q is normed and rotated in place, k and v go into the token's slot of their pages.  All of it in 32-bit.
template <typename T>
__global__ __launch_bounds__(256) void head_norm_rope_kv_write_kernel(
    T* __restrict__ qkv, int stride, const T* __restrict__ bias, const T* __restrict__ qw, const T* __restrict__ kw,
    const int* __restrict__ positions, const int* __restrict__ token_req, const int* __restrict__ block_table, int table_stride,
    const float* __restrict__ inv_freq, T* __restrict__ k_cache, T* __restrict__ v_cache, int heads, int kv_heads, int hd, int vd,
    int page_size, float eps, RopeForm form, int v_is_k) {
  const int t = blockIdx.x, lane = threadIdx.x % NS_WAVE, wave = threadIdx.x / NS_WAVE, waves = blockDim.x / NS_WAVE;
  T* row = qkv + (size_t)t * stride;
  const int pos = positions[t];
  const int page = block_table[(size_t)token_req[t] * table_stride + pos / page_size];
  const int slot = pos % page_size;
  const int half = form.rot / 2;
  for (int h = blockIdx.y * waves + wave; h < heads + kv_heads; h += waves * gridDim.y) {
    const bool is_q = h < heads;
    const int at = h * hd;  // q heads and k heads follow each other in the row
    const T* w = is_q ? qw : kw;
    float ss = 0.f;
    for (int c = lane; c < hd; c += NS_WAVE) {
      const float v = to_f(row[at + c]) + (bias ? to_f(bias[at + c]) : 0.f);
      ss = fmaf(v, v, ss);
    }
    const float rinv = w ? 1.f / sqrtf(wave_sum(ss) / (float)hd + eps) : 1.f;
    T* kd = is_q ? nullptr : k_cache + (((size_t)page * kv_heads + (h - heads)) * page_size + slot) * hd;
    if (!is_q && v_is_k) {
      T* vdst = v_cache + (((size_t)page * kv_heads + (h - heads)) * vd) * page_size + slot;
      for (int c = lane; c < hd; c += NS_WAVE)
        vdst[(size_t)c * page_size] = from_f<T>(to_f(row[at + c]) + (bias ? to_f(bias[at + c]) : 0.f));
    }
    // the rotated pairs: a lane reads both channels of its pair and writes both
    for (int j = lane; j < half; j += NS_WAVE) {
      int d1, d2;
      rope_pair_channels(form, j, d1, d2);
      float a = (to_f(row[at + d1]) + (bias ? to_f(bias[at + d1]) : 0.f)) * rinv * (w ? to_f(w[d1]) : 1.f);
      float b = (to_f(row[at + d2]) + (bias ? to_f(bias[at + d2]) : 0.f)) * rinv * (w ? to_f(w[d2]) : 1.f);
      float c, s;
      rope_cos_sin(form, pos, inv_freq[j], c, s);
      rope_turn(a, b, c, s, a, b);
      if (is_q) {
        row[at + d1] = from_f<T>(a);
        row[at + d2] = from_f<T>(b);
      } else {
        kd[d1] = from_f<T>(a);
        kd[d2] = from_f<T>(b);
      }
    }
    for (int c = form.rot + lane; c < hd; c += NS_WAVE) {
      const float v = (to_f(row[at + c]) + (bias ? to_f(bias[at + c]) : 0.f)) * rinv * (w ? to_f(w[c]) : 1.f);
      if (is_q)
        row[at + c] = from_f<T>(v);
      else
        kd[c] = from_f<T>(v);
    }
  }
  if (!v_is_k && blockIdx.y == 0) {
    const int nq = heads * hd, nk = kv_heads * hd, nv = kv_heads * vd;
    for (int i = threadIdx.x; i < nv; i += blockDim.x) {
      const float v = to_f(row[nq + nk + i]) + (bias ? to_f(bias[nq + nk + i]) : 0.f);
      v_cache[(((size_t)page * kv_heads + i / vd) * vd + i % vd) * page_size + slot] = from_f<T>(v);
    }
  }
}

extern "C" int ns_head_norm_rope_kv_write(void* qkv, int stride, const void* bias, const void* qw, const void* kw, const int* positions,
                                          const int* token_req, const int* block_table, int table_stride, const float* inv_freq,
                                          void* k_cache, void* v_cache, int n_tokens, int heads, int kv_heads, int hd, int vd, int page_size,
                                          float eps, int rot, int interleaved, float factor, int v_is_k, int dtype, hipStream_t stream) {
  if (n_tokens <= 0 || heads <= 0 || kv_heads <= 0 || hd <= 0 || vd <= 0 || page_size <= 0 || rot < 0 || rot > hd || rot % 2) return NS_ERR_BAD_ARG;
  if (v_is_k && vd != hd) return NS_ERR_BAD_ARG;
  if (rot > 0 && !inv_freq) return NS_ERR_BAD_ARG;
  const RopeForm form{rot, interleaved, factor};
  auto in_pieces = [&](auto* rows) {
    typedef typename std::remove_pointer<decltype(rows)>::type T;
    KvRows<T> p{};
    p.qkv = rows, p.bias = (const T*)bias, p.qw = (const T*)qw, p.kw = (const T*)kw, p.positions = positions, p.token_req = token_req, p.block_table = block_table;
    p.inv_freq = inv_freq, p.k_cache = (T*)k_cache, p.v_cache = (T*)v_cache, p.stride = stride, p.table_stride = table_stride, p.n_tokens = n_tokens;
    p.heads = heads, p.kv_heads = kv_heads, p.hd = hd, p.vd = vd, p.page_size = page_size, p.eps = eps, p.form = form, p.norm_q = qw != nullptr, p.norm_k = kw != nullptr;
    p.v_is_k = v_is_k;
    if (!kv_rows_take(p)) return false;
    launch_head_rows(p, stream);
    return true;
  };
  if (dtype == NS_DTYPE_F32 ? in_pieces((float*)qkv) : dtype == NS_DTYPE_BF16 && in_pieces((bf16_t*)qkv)) return ns_launch_status();
  // few tokens: a wave a head at once, over several workgroups a token
  const int shares = n_tokens >= 256 ? 1 : (heads + kv_heads + 3) / 4;
  if (n_tokens > 65535 * 32768 || shares > 65535) return NS_ERR_BAD_ARG;
  dim3 grid(n_tokens, shares);
  if (dtype == NS_DTYPE_F32)
    head_norm_rope_kv_write_kernel<float><<<grid, 256, 0, stream>>>((float*)qkv, stride, (const float*)bias, (const float*)qw, (const float*)kw,
        positions, token_req, block_table, table_stride, inv_freq, (float*)k_cache, (float*)v_cache, heads, kv_heads, hd, vd, page_size, eps, form, v_is_k);
  else if (dtype == NS_DTYPE_BF16)
    head_norm_rope_kv_write_kernel<bf16_t><<<grid, 256, 0, stream>>>((bf16_t*)qkv, stride, (const bf16_t*)bias, (const bf16_t*)qw, (const bf16_t*)kw,
        positions, token_req, block_table, table_stride, inv_freq, (bf16_t*)k_cache, (bf16_t*)v_cache, heads, kv_heads, hd, vd, page_size, eps, form, v_is_k);
  else
    return NS_ERR_UNSUPPORTED;
  return ns_launch_status();
}

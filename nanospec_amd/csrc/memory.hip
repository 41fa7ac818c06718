// A matrix memory with exponential gates (the mLSTM recurrence), token by token in 32-bit.  Per head: a matrix S [D][E], a
// vector n [D] and a running maximum m (a new sequence starts with S = 0, n = 0, m = 0):
//   i = cap tanh((x_i + b_i) / cap)                        log of the input gate
//   f = logsigmoid(cap tanh((x_f + b_f) / cap))            log of the forget gate
//   m' = max(f + m, i);   a = exp(f + m - m');   b = exp(i - m')
//   S <- a S + b k v^T;   n <- a n + b k;   o = S^T q / (max(|n . q|, exp(-m')) + den_eps)
// q (times ``q_scale``), k [H][D], v [H][E] and the two gate inputs x_i, x_f [H] are columns of one row per token (the
// result of one stacked product), in the model's precision; everything from there on is 32-bit.
//
// A column of S never meets another column, so a wave owns 64 / TPC columns and the TPC lanes of a column hold 8 key
// channels each; their partial sums meet through the vector unit's lane permutations (``group_sum``).  n is one more column
// of S, the one whose value is 1 for every token: one more workgroup a head carries it, and what it writes per token is the
// denominator max(|n . q|, exp(-m')) + den_eps.  The kernel leaves S^T q and the denominators; whoever reads the read-out
// divides (``gated_rms`` does, as it reads a head).  A workgroup is four waves that share the staged operands: the next
// block of tokens is fetched into registers while the current block is worked through from LDS, and four tokens are
// worked through together: only m, S and n pass from token to token.
//
// What a request keeps between steps lies in its state slot: S as [H][E][D] (a column's key channels contiguous), then
// room for n per workgroup of a head, [H][B][D] (the last workgroup's is the one in use), then m per workgroup, [H][B],
// with B = ``ns_memory_blocks(D, E)`` the workgroups of a head: each reads and writes only its own copy of m, so none can
// read what another has already written for the next step.
#include "chunk16.h"

#define MM_KPT 8  // key channels a lane holds of its column
#define MM_WAVES 4
#define MM_THREADS (MM_WAVES * NS_WAVE)

template <typename T> struct Vec8;
template <> struct Vec8<float> {
  static __device__ __forceinline__ void load(const float* p, float* out) {
    const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
    out[0] = a.x, out[1] = a.y, out[2] = a.z, out[3] = a.w, out[4] = b.x, out[5] = b.y, out[6] = b.z, out[7] = b.w;
  }
};
template <> struct Vec8<bf16_t> {
  static __device__ __forceinline__ void load(const bf16_t* p, float* out) {
    typedef bf16_t v8 __attribute__((ext_vector_type(8)));
    const v8 a = *reinterpret_cast<const v8*>(p);
#pragma unroll
    for (int j = 0; j < 8; ++j) out[j] = (float)a[j];
  }
};

__device__ __forceinline__ float mm_log_sigmoid(float z) {
  // log(1 / (1 + exp(-z))) without overflow on either side
  return fminf(z, 0.f) - log1pf(expf(-fabsf(z)));
}

struct MemoryParams {
  const void* proj;  // [tokens][stride]
  int stride, q_off, k_off, v_off, i_off, f_off;
  const float* gate_bias_i;  // [H]
  const float* gate_bias_f;  // [H]
  float* state;              // [slots][state_stride]
  long long state_stride;
  const int* qo_indptr;
  const int* state_slots;
  float* out;  // [tokens][H * E]: S^T q, not yet divided
  float* den;  // [tokens][H]: max(|n . q|, exp(-m)) + den_eps
  int H, D, E;
  float cap, q_scale, den_eps;
  int vec_ok;  // 8 channels of q and k can be fetched with one aligned vector load
  int below;   // requests of at least that many tokens are the chunks'
};

template <typename T, int TPC>
__global__ __launch_bounds__(MM_THREADS) void memory_scan_kernel(const MemoryParams p) {
  constexpr int DP = MM_KPT * TPC;                           // key channels of a column as the lanes hold them (D padded)
  constexpr int CPW = NS_WAVE / TPC;                         // columns a wave owns
  constexpr int CPG = CPW * MM_WAVES;                        // columns a workgroup owns
  constexpr int TB = TPC <= 16 ? 16 : (TPC == 32 ? 8 : 4);   // tokens a block
  constexpr int SLICES = TB * 2 * TPC;                       // 8-channel pieces of q and k in a block
  constexpr int PER = (SLICES + MM_THREADS - 1) / MM_THREADS;  // pieces a thread fetches
  constexpr int VALS = TB * CPG;                             // values of v in a block
  constexpr int VPER = (VALS + MM_THREADS - 1) / MM_THREADS;
  __shared__ __attribute__((aligned(16))) float qk_s[TB * 2 * DP];  // per token: q [DP], k [DP]
  __shared__ float v_s[VALS];
  __shared__ float gate_s[TB * 2];

  const int tid = threadIdx.x, lane = tid % NS_WAVE, wave = tid / NS_WAVE, h = blockIdx.y, b = blockIdx.z;
  const int t0 = p.qo_indptr[b], t1 = p.qo_indptr[b + 1];
  if (t1 <= t0 || t1 - t0 >= p.below) return;
  const int H = p.H, D = p.D, E = p.E;
  const int s = lane % TPC, cw = wave * CPW + lane / TPC, col = blockIdx.x * CPG + cw, d0 = s * MM_KPT;
  // the last workgroup of a head carries n as one more column of S whose value is 1 for every token: its first column's
  // lanes hold n where the others hold a column of S, and what it writes is the denominator
  const bool nblock = blockIdx.x == gridDim.x - 1;
  const bool col_ok = !nblock && col < E, n_lane = nblock && cw == 0;
  const T* proj = (const T*)p.proj;
  float* st = p.state + (long long)p.state_slots[b] * p.state_stride;
  float* st_S = st + ((size_t)h * E + (col_ok ? col : 0)) * D;
  const int B = gridDim.x;
  float* st_n = st + (size_t)H * E * D + ((size_t)h * B + blockIdx.x) * D;
  float* st_m = st + (size_t)H * E * D + (size_t)H * B * D + (size_t)h * B + blockIdx.x;

  float S[MM_KPT];
#pragma unroll
  for (int j = 0; j < MM_KPT; ++j) {
    const bool ok = d0 + j < D;
    S[j] = (ok && col_ok) ? st_S[d0 + j] : ((ok && n_lane) ? st_n[d0 + j] : 0.f);
  }
  float m = *st_m;
  const float bias_i = p.gate_bias_i ? p.gate_bias_i[h] : 0.f, bias_f = p.gate_bias_f ? p.gate_bias_f[h] : 0.f;

  float pre[PER][MM_KPT], vpre[VPER], gpre = 0.f;

  // fetch the operands of tokens [t, t + TB) into registers
  auto fetch = [&](int t) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int idx = tid + i * MM_THREADS;  // (token, q or k, piece)
      const int tk = idx / (2 * TPC), which = (idx / TPC) % 2, piece = idx % TPC;
      const bool live = idx < SLICES && t + tk < t1;
      const T* src = proj + (size_t)(t + (live ? tk : 0)) * p.stride + (which ? p.k_off : p.q_off) + (size_t)h * D + piece * MM_KPT;
      if (live && p.vec_ok && piece * MM_KPT + MM_KPT <= D) {
        Vec8<T>::load(src, pre[i]);
      } else {
#pragma unroll
        for (int j = 0; j < MM_KPT; ++j) pre[i][j] = (live && piece * MM_KPT + j < D) ? to_f(src[j]) : 0.f;
      }
      if (!which) {
#pragma unroll
        for (int j = 0; j < MM_KPT; ++j) pre[i][j] *= p.q_scale;
      }
    }
#pragma unroll
    for (int i = 0; i < VPER; ++i) {
      const int idx = tid + i * MM_THREADS, tk = idx / CPG, c = blockIdx.x * CPG + idx % CPG;
      if (nblock)
        vpre[i] = idx % CPG == 0 ? 1.f : 0.f;
      else
        vpre[i] = (idx < VALS && t + tk < t1 && c < E) ? to_f(proj[(size_t)(t + tk) * p.stride + p.v_off + (size_t)h * E + c]) : 0.f;
    }
    if (tid < 2 * TB) {
      const int tk = tid / 2, which = tid % 2;
      if (t + tk < t1) {
        const float x = to_f(proj[(size_t)(t + tk) * p.stride + (which ? p.f_off : p.i_off) + h]) + (which ? bias_f : bias_i);
        const float capped = p.cap * tanhf(x / p.cap);
        gpre = which ? mm_log_sigmoid(capped) : capped;
      }
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int idx = tid + i * MM_THREADS;
      if (idx < SLICES) {
        float4* dst = reinterpret_cast<float4*>(qk_s + (size_t)idx * MM_KPT);
        dst[0] = make_float4(pre[i][0], pre[i][1], pre[i][2], pre[i][3]);
        dst[1] = make_float4(pre[i][4], pre[i][5], pre[i][6], pre[i][7]);
      }
    }
#pragma unroll
    for (int i = 0; i < VPER; ++i) {
      const int idx = tid + i * MM_THREADS;
      if (idx < VALS) v_s[idx] = vpre[i];
    }
    if (tid < 2 * TB) gate_s[tid] = gpre;
  };

  fetch(t0);
  stage();
  __syncthreads();
  constexpr int UN = 4;  // tokens worked through together: only m, S and n pass from token to token, the rest overlaps
  static_assert(TB % UN == 0, "a block of tokens is whole groups");
  for (int t = t0; t < t1; t += TB) {
    if (t + TB < t1) fetch(t + TB);
    const int nb = min(TB, t1 - t);
    for (int tk0 = 0; tk0 < nb; tk0 += UN) {
      float a[UN], bv[UN], em[UN], num[UN];
      // the gates' chain: additions and maxima only; the exponentials hang off it
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const bool on = tk0 + u < nb;
        const float gi = gate_s[2 * (tk0 + u)], gf = gate_s[2 * (tk0 + u) + 1];
        const float mn = fmaxf(gf + m, gi);
        a[u] = on ? expf(gf + m - mn) : 1.f;
        const float bb = on ? expf(gi - mn) : 0.f;
        m = on ? mn : m;
        em[u] = nblock ? expf(-m) : 0.f;
        bv[u] = bb * v_s[(tk0 + u) * CPG + cw];
      }
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const float4* qp = reinterpret_cast<const float4*>(qk_s + (size_t)((tk0 + u) * 2) * DP + d0);
        const float4* kp = reinterpret_cast<const float4*>(qk_s + (size_t)((tk0 + u) * 2 + 1) * DP + d0);
        const float4 q0 = qp[0], q1 = qp[1], k0 = kp[0], k1 = kp[1];
        const float q[MM_KPT] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
        const float k[MM_KPT] = {k0.x, k0.y, k0.z, k0.w, k1.x, k1.y, k1.z, k1.w};
        float p0 = 0.f, p1 = 0.f;  // two partial sums: shorter chains
#pragma unroll
        for (int j = 0; j < MM_KPT; j += 2) {
          S[j] = fmaf(a[u], S[j], k[j] * bv[u]);
          S[j + 1] = fmaf(a[u], S[j + 1], k[j + 1] * bv[u]);
          p0 = fmaf(S[j], q[j], p0);
          p1 = fmaf(S[j + 1], q[j + 1], p1);
        }
        num[u] = p0 + p1;
      }
#pragma unroll
      for (int u = 0; u < UN; ++u) num[u] = group_sum<TPC>(num[u]);
      if (s == 0 && (col_ok || n_lane)) {
#pragma unroll
        for (int u = 0; u < UN; ++u)
          if (tk0 + u < nb) {
            if (n_lane)
              p.den[(size_t)(t + tk0 + u) * H + h] = fmaxf(fabsf(num[u]), em[u]) + p.den_eps;
            else
              p.out[(size_t)(t + tk0 + u) * H * E + (size_t)h * E + col] = num[u];
          }
      }
    }
    __syncthreads();
    if (t + TB < t1) stage();
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < MM_KPT; ++j) {
    if (d0 + j < D) {
      if (col_ok) st_S[d0 + j] = S[j];
      if (n_lane) st_n[d0 + j] = S[j];
    }
  }
  if (tid == 0) *st_m = m;
}

template <typename T>
static int memory_scan_launch(const MemoryParams& p, int n_reqs, hipStream_t stream) {
  int tpc = 1;
  while (tpc * MM_KPT < p.D) tpc *= 2;
  if (tpc > NS_WAVE) return NS_ERR_UNSUPPORTED;
  const int cpg = MM_WAVES * NS_WAVE / tpc;
  dim3 grid((p.E + cpg - 1) / cpg + 1, p.H, n_reqs);  // one more workgroup a head: the one that carries n
  switch (tpc) {
    case 1: memory_scan_kernel<T, 1><<<grid, MM_THREADS, 0, stream>>>(p); break;
    case 2: memory_scan_kernel<T, 2><<<grid, MM_THREADS, 0, stream>>>(p); break;
    case 4: memory_scan_kernel<T, 4><<<grid, MM_THREADS, 0, stream>>>(p); break;
    case 8: memory_scan_kernel<T, 8><<<grid, MM_THREADS, 0, stream>>>(p); break;
    case 16: memory_scan_kernel<T, 16><<<grid, MM_THREADS, 0, stream>>>(p); break;
    case 32: memory_scan_kernel<T, 32><<<grid, MM_THREADS, 0, stream>>>(p); break;
    default: memory_scan_kernel<T, 64><<<grid, MM_THREADS, 0, stream>>>(p); break;
  }
  return ns_launch_status();
}

// workgroups of one head: those that share its columns and the one that carries n (each keeps a copy of m, and room for n, in the state)
extern "C" int ns_memory_blocks(int D, int E) {
  int tpc = 1;
  while (tpc * MM_KPT < D) tpc *= 2;
  if (tpc > NS_WAVE) return -1;
  const int cpg = MM_WAVES * NS_WAVE / tpc;
  return (E + cpg - 1) / cpg + 1;
}

extern "C" int ns_memory_scan(const void* proj, int stride, int q_off, int k_off, int v_off, int i_off, int f_off, const float* gate_bias_i,
                              const float* gate_bias_f, float* state, long long state_stride, const int* qo_indptr, const int* state_slots,
                              float* out, float* den, int n_reqs, int H, int D, int E, float cap, float q_scale, float den_eps, int below, int dtype, hipStream_t stream) {
  if (n_reqs <= 0 || n_reqs > 65535 || H <= 0 || H > 65535 || D <= 0 || E <= 0 || !(cap > 0.f)) return NS_ERR_BAD_ARG;
  const int blocks = ns_memory_blocks(D, E);
  if (blocks < 0) return NS_ERR_UNSUPPORTED;
  if (state_stride < (long long)H * E * D + (long long)H * blocks * (D + 1)) return NS_ERR_BAD_ARG;
  MemoryParams p{proj, stride, q_off, k_off, v_off, i_off, f_off, gate_bias_i, gate_bias_f, state, state_stride, qo_indptr, state_slots,
                 out, den, H, D, E, cap, q_scale, den_eps, 0, below};
  const size_t elem = dtype == NS_DTYPE_F32 ? 4 : 2;
  p.vec_ok = D % 8 == 0 && stride % 8 == 0 && q_off % 8 == 0 && k_off % 8 == 0 && ((uintptr_t)proj % (8 * elem)) == 0;
  if (dtype == NS_DTYPE_F32) return memory_scan_launch<float>(p, n_reqs, stream);
  if (dtype == NS_DTYPE_BF16) return memory_scan_launch<bf16_t>(p, n_reqs, stream);
  return NS_ERR_UNSUPPORTED;
}

// ------------------------------------------------------------------------------------------------
// The same recurrence for prompt portions, sixteen tokens at a time.  With F_t the sum of the forget gates' logs up to t and m_t as above,
// everything a token reads of its chunk is
//   o_t = exp(F_t + m_0 - m_t) S_0^T q_t + sum_{j <= t} P_tj v_j,   P_tj = (q_t . k_j) exp(F_t - F_j + i_j - m_t)
//   S <- exp(F_C + m_0 - m_C) S + sum_j exp(F_C - F_j + i_j - m_C) k_j v_j^T
// with exponents of at most zero (up to m's rounding); m_0 and S_0 stand before the chunk, C is its last token.  (F, m) of two pieces of a prompt join as (F1 + F2,
// max(m1 + F2, m2)), so ``memory_gates_kernel`` finds all of them in log time, F in 64 bits because differences of it are used.
// ``memory_chunk_kernel`` makes P and the scaled keys and queries of all chunks at once, in the order of the matrix instruction's lanes
// (sums in 64 bits), and ``memory_pass_kernel`` goes from chunk to chunk with 16 columns of S in the registers of four waves
// (v_mfma_f32_16x16x4_f32, 32-bit products and sums); a fifth wave adds up the four waves' shares of the output.  n is a column
// of S of its own, as above.  Bound by the chain of a chunk (17 matrix instructions of 32 cycles, a barrier) where the token form's is 0.36 us a
// token.  8 heads of 128 by 256: one prompt of 2,048 tokens 729 -> 122 us, prompts of 700, 500 and 331 tokens 263 -> 62 us (6 gates, 12 chunks,
// 42 pass).  Relative error (2-norm, against 64 bits) of S^T q 1.9e-7 token by token and 1.4e-7 so with forget gates around 0.95, 9.7e-8
// and 7.6e-8 around 0.1, of the denominators 1.7e-7 and 1.3e-7, of S 1.1e-7 and 1.1e-7.
// ------------------------------------------------------------------------------------------------
#define MG_THREADS 1024

struct MemoryChunks {
  MemoryParams p;
  float* scratch;  // a record for every chunk and head: Q | K (16 D each) | P (256) | exp(F_C + m_0 - m_C) and three unused | exp(-m_t) (16)
  double* F;       // [tokens][H]: sum of the forget gates' logs from the request's first token on
  float* gi;       // [tokens][H]: the input gate's log
  float* m;        // [tokens][H]
  float* m0;       // [requests][H]: m before the step
  int n_reqs, from, min_tokens, blocks;
};

template <int D>
__device__ __forceinline__ size_t memory_record(const MemoryChunks& a, int chunk, int h) {
  return ((size_t)(chunk - a.from) * a.p.H + h) * (2 * DC_T * D + DC_T * DC_T + 4 + DC_T);
}

template <typename T>
__global__ __launch_bounds__(MG_THREADS) void memory_gates_kernel(const MemoryChunks a) {
  __shared__ double fs[MG_THREADS / NS_WAVE], ms[MG_THREADS / NS_WAVE];
  const MemoryParams& p = a.p;
  const int h = blockIdx.x, b = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, H = p.H;
  const int t0 = p.qo_indptr[b], t1 = p.qo_indptr[b + 1];
  if (t1 - t0 < a.min_tokens) return;
  float* st_m = p.state + (long long)p.state_slots[b] * p.state_stride + (size_t)H * p.E * p.D + (size_t)H * a.blocks * p.D + (size_t)h * a.blocks;
  const float bias_i = p.gate_bias_i ? p.gate_bias_i[h] : 0.f, bias_f = p.gate_bias_f ? p.gate_bias_f[h] : 0.f;
  double f_in = 0., m_in = *st_m;  // before this round of tokens
  if (threadIdx.x == 0) a.m0[(size_t)b * H + h] = (float)m_in;
  __syncthreads();
  for (int first = t0; first < t1; first += MG_THREADS) {
    const int t = first + threadIdx.x;
    double F = 0., M = -INFINITY;
    if (t < t1) {
      const T* row = (const T*)p.proj + (size_t)t * p.stride;
      const float i = p.cap * tanhf((to_f(row[p.i_off + h]) + bias_i) / p.cap);
      F = mm_log_sigmoid(p.cap * tanhf((to_f(row[p.f_off + h]) + bias_f) / p.cap)), M = i;
      a.gi[(size_t)t * H + h] = i;
    }
    for (int o = 1; o < NS_WAVE; o <<= 1) {  // inclusive, within a wave
      const double F1 = __shfl_up(F, o, NS_WAVE), M1 = __shfl_up(M, o, NS_WAVE);
      if (lane >= o) M = fmax(M1 + F, M), F += F1;
    }
    if (lane == 63) fs[wave] = F, ms[wave] = M;
    __syncthreads();
    double Fp = f_in, Mp = m_in;  // up to this wave
    for (int w = 0; w < wave; ++w) Mp = fmax(Mp + fs[w], ms[w]), Fp += fs[w];
    if (t < t1) {
      a.F[(size_t)t * H + h] = Fp + F;
      a.m[(size_t)t * H + h] = (float)fmax(Mp + F, M);
    }
    for (int w = 0; w < MG_THREADS / NS_WAVE; ++w) m_in = fmax(m_in + fs[w], ms[w]), f_in += fs[w];
    __syncthreads();
  }
  // every workgroup of the token form keeps a copy of m
  const float last = (float)m_in;
  for (int i = threadIdx.x; i < a.blocks; i += MG_THREADS) st_m[i] = last;
}

template <typename T, int D>
__global__ __launch_bounds__(256) void memory_chunk_kernel(const MemoryChunks a) {
  constexpr int LD = D + 4;
  __shared__ __attribute__((aligned(16))) float qk[2][DC_T][LD];
  __shared__ float p_s[DC_T][DC_T + 1], i_s[DC_T], m_s[DC_T];
  __shared__ double f_s[DC_T];
  const MemoryParams& p = a.p;
  const int chunk = a.from + blockIdx.y, h = blockIdx.x, tid = threadIdx.x, H = p.H;
  const int b = chunk_request(p.qo_indptr, a.n_reqs, chunk);
  const int r0 = p.qo_indptr[b], r1 = p.qo_indptr[b + 1], row0 = r0 + (chunk - r0 / DC_T - b) * DC_T;
  if (row0 >= r1 || r1 - r0 < a.min_tokens) return;
  const int n = min(DC_T, r1 - row0);
  // of the chunk's start: the sum of the logs and m behind the token before
  const double F0 = row0 > r0 ? a.F[(size_t)(row0 - 1) * H + h] : 0.;
  const float m0 = row0 > r0 ? a.m[(size_t)(row0 - 1) * H + h] : a.m0[(size_t)b * H + h];
  for (int e = tid; e < 2 * DC_T * (D / 8); e += 256) {
    const int which = e / (DC_T * (D / 8)), i = e / (D / 8) % DC_T, d = 8 * (e % (D / 8));
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (i < n) Vec8<T>::load((const T*)p.proj + (size_t)(row0 + i) * p.stride + (which ? p.k_off : p.q_off) + (size_t)h * D + d, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) qk[which][i][d + j] = which ? v[j] : v[j] * p.q_scale;
  }
  if (tid < DC_T) {
    const size_t at = (size_t)(row0 + min(tid, n - 1)) * H + h;
    f_s[tid] = a.F[at], i_s[tid] = a.gi[at], m_s[tid] = a.m[at];
  }
  __syncthreads();
  {  // P: a thread a pair of tokens
    const int t = tid / 16, j = tid % 16;
    double s0 = 0., s1 = 0.;
    if (j <= t && t < n) {
      for (int d = 0; d < D; d += 4) {
        const f32x4 q = *reinterpret_cast<const f32x4*>(&qk[0][t][d]), k = *reinterpret_cast<const f32x4*>(&qk[1][j][d]);
        s0 = fma((double)q[0], (double)k[0], s0), s1 = fma((double)q[1], (double)k[1], s1);
        s0 = fma((double)q[2], (double)k[2], s0), s1 = fma((double)q[3], (double)k[3], s1);
      }
      p_s[t][j] = (float)((s0 + s1) * (double)expf((float)(f_s[t] - f_s[j] + (double)i_s[j] - (double)m_s[t])));
    } else {
      p_s[t][j] = 0.f;
    }
  }
  __syncthreads();
  float* rec = a.scratch + memory_record<D>(a, chunk, h);
  for (int e = tid; e < 2 * DC_T * (D / 4); e += 256) {
    const int which = e / (DC_T * (D / 4)), at = e % (DC_T * (D / 4)), tile = at / NS_WAVE, r = at % 16, gq = at % NS_WAVE / 16;
    f32x4 v;
    if (which == 0) {  // row: token, four channels of the tile
      const int t = chunk_token(r);
      v = *reinterpret_cast<const f32x4*>(&qk[0][t][16 * tile + 4 * gq]) * expf((float)(f_s[t] - F0 + (double)m0 - (double)m_s[t]));
    } else {  // row: channel of the tile, four tokens
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = chunk_token(4 * gq + i);
        v[i] = t < n ? qk[1][t][16 * tile + r] * expf((float)(f_s[n - 1] - f_s[t] + (double)i_s[t] - (double)m_s[n - 1])) : 0.f;
      }
    }
    *reinterpret_cast<f32x4*>(rec + 4 * (size_t)e) = v;
  }
  if (tid < NS_WAVE) {
    const int r = tid % 16, gq = tid / 16;
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = p_s[chunk_token(r)][chunk_token(4 * gq + i)];
    *reinterpret_cast<f32x4*>(rec + 2 * DC_T * D + 4 * tid) = v;
  } else if (tid < NS_WAVE + DC_T) {
    rec[2 * DC_T * D + DC_T * DC_T + 4 + tid - NS_WAVE] = expf(-m_s[tid - NS_WAVE]);
  } else if (tid == NS_WAVE + DC_T) {
    rec[2 * DC_T * D + DC_T * DC_T] = expf((float)(f_s[n - 1] - F0 + (double)m0 - (double)m_s[n - 1]));
  }
}

template <typename T, int D>
__global__ __launch_bounds__(5 * NS_WAVE) void memory_pass_kernel(const MemoryChunks a, int to) {
  constexpr int TILES = D / 64;  // tiles of 16 key channels a wave holds
  __shared__ f32x4 part[2][4][NS_WAVE];
  const MemoryParams& p = a.p;
  const int b = blockIdx.z, h = blockIdx.x, lane = threadIdx.x & 63, c = lane & 15, gq = lane >> 4, H = p.H;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r0 = p.qo_indptr[b], r1 = p.qo_indptr[b + 1], first = r0 / DC_T + b;
  if (r1 - r0 < a.min_tokens) return;
  const int begin = max(first, a.from), end = min(first + (r1 - r0 + DC_T - 1) / DC_T, to);
  if (begin >= end) return;
  const bool nblock = blockIdx.y == gridDim.y - 1;  // the columns' last workgroup carries n in its first column
  const int col = nblock ? 0 : blockIdx.y * 16 + c;
  auto last_of = [&](int chunk) { return min(DC_T, r1 - r0 - (chunk - first) * DC_T) - 1; };
  if (wave < 4) {
    struct Operands {
      f32x4 q[TILES], k[TILES], p, v;
      float decay;
    };
    float* st = p.state + (long long)p.state_slots[b] * p.state_stride;
    float* S = nblock ? st + (size_t)H * p.E * D + ((size_t)h * a.blocks + a.blocks - 1) * D : st + ((size_t)h * p.E + col) * D;
    S += wave * TILES * 16 + 4 * gq;
    const bool mine = !nblock || c == 0;
    const T* v_src = (const T*)p.proj + p.v_off + (size_t)h * p.E + (nblock ? 0 : blockIdx.y * 16);
    unsigned v_at[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v_at[i] = (4 * i + gq) * p.stride + (nblock ? 0 : c);
    f32x4 s[TILES];
#pragma unroll
    for (int x = 0; x < TILES; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[x][i] = mine ? S[x * 16 + i] : 0.f;
    auto fetch = [&](Operands& o, int chunk) {
      chunk = min(chunk, end - 1);
      const float* rec = a.scratch + memory_record<D>(a, chunk, h);
#pragma unroll
      for (int x = 0; x < TILES; ++x) {
        o.q[x] = *reinterpret_cast<const f32x4*>(rec + (wave * TILES + x) * 256 + 4 * lane);
        o.k[x] = *reinterpret_cast<const f32x4*>(rec + DC_T * D + (wave * TILES + x) * 256 + 4 * lane);
      }
      o.p = *reinterpret_cast<const f32x4*>(rec + 2 * DC_T * D + 4 * lane);
      o.decay = rec[2 * DC_T * D + DC_T * DC_T];
      const T* src = v_src + (size_t)(r0 + (chunk - first) * DC_T) * p.stride;
      const unsigned last = last_of(chunk) * p.stride + (nblock ? 0 : c);
#pragma unroll
      for (int i = 0; i < 4; ++i) o.v[i] = to_f(src[min(v_at[i], last)]);
    };
    auto work = [&](const Operands& o, int chunk) {
      const int last = last_of(chunk);
      f32x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = 4 * i + gq <= last ? (nblock ? (c == 0 ? 1.f : 0.f) : o.v[i]) : 0.f;
      f32x4 out[TILES];
#pragma unroll
      for (int x = 0; x < TILES; ++x) out[x] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int x = 0; x < TILES; ++x) out[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.q[x][i], s[x][i], out[x], 0, 0, 0);
#pragma unroll
      for (int x = 1; x < TILES; ++x) out[0] += out[x];
      if (__any(not_finite(v))) {
        if (wave == 0) out[0] += lower_product(a.scratch + memory_record<D>(a, chunk, h) + 2 * DC_T * D, v, lane);
      } else {  // a wave gives four tokens' part of P v
        const float pw = wave < 2 ? (wave == 0 ? o.p[0] : o.p[1]) : (wave == 2 ? o.p[2] : o.p[3]);
        const float vw = wave < 2 ? (wave == 0 ? v[0] : v[1]) : (wave == 2 ? v[2] : v[3]);
        out[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(pw, vw, out[0], 0, 0, 0);
      }
      part[chunk & 1][wave][lane] = out[0];
#pragma unroll
      for (int x = 0; x < TILES; ++x) s[x] *= o.decay;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int x = 0; x < TILES; ++x) s[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.k[x][i], v[i], s[x], 0, 0, 0);
      __syncthreads();
    };
    Operands o0, o1, o2;  // two chunks ahead
    fetch(o0, begin), fetch(o1, begin + 1);
    int chunk = begin;
    for (; chunk + 2 < end; chunk += 3) {
      fetch(o2, chunk + 2);
      work(o0, chunk);
      fetch(o0, chunk + 3);
      work(o1, chunk + 1);
      fetch(o1, chunk + 4);
      work(o2, chunk + 2);
    }
    if (chunk < end) work(o0, chunk);
    if (chunk + 1 < end) work(o1, chunk + 1);
#pragma unroll
    for (int x = 0; x < TILES; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (mine) S[x * 16 + i] = s[x][i];
  } else {
    for (int chunk = begin; chunk < end; ++chunk) {
      f32x4 floor4 = {0.f, 0.f, 0.f, 0.f};
      if (nblock) {
        const float* em = a.scratch + memory_record<D>(a, chunk, h) + 2 * DC_T * D + DC_T * DC_T + 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) floor4[i] = em[4 * i + gq];
      }
      __syncthreads();
      const f32x4 out = (part[chunk & 1][0][lane] + part[chunk & 1][1][lane]) + (part[chunk & 1][2][lane] + part[chunk & 1][3][lane]);
      const int last = last_of(chunk), row = r0 + (chunk - first) * DC_T + gq;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (4 * i + gq > last) continue;
        if (!nblock)
          p.out[((size_t)(row + 4 * i) * H + h) * p.E + col] = out[i];
        else if (c == 0)
          p.den[(size_t)(row + 4 * i) * H + h] = fmaxf(fabsf(out[i]), floor4[i]) + p.den_eps;
      }
    }
  }
}

template <typename T, int D>
static int memory_chunks(MemoryChunks a, int n_tokens, size_t scratch_floats, hipStream_t stream) {
  const int chunks = n_tokens / DC_T + a.n_reqs;
  const size_t fit = scratch_floats / ((size_t)a.p.H * (2 * DC_T * D + DC_T * DC_T + 4 + DC_T));
  if (fit < 1) return NS_ERR_BAD_ARG;
  memory_gates_kernel<T><<<dim3(a.p.H, a.n_reqs), MG_THREADS, 0, stream>>>(a);
  for (int from = 0; from < chunks;) {
    const int left = chunks - from < 65535 ? chunks - from : 65535, now = fit < (size_t)left ? (int)fit : left;
    a.from = from;
    memory_chunk_kernel<T, D><<<dim3(a.p.H, now), 256, 0, stream>>>(a);
    memory_pass_kernel<T, D><<<dim3(a.p.H, a.p.E / 16 + 1, a.n_reqs), 5 * NS_WAVE, 0, stream>>>(a, from + now);
    from += now;
  }
  return ns_launch_status();
}

// Requests of at least ``min_tokens`` tokens; the others are ``ns_memory_scan``'s (with ``below`` the same number).  ``gates``: room for 16
// bytes a token and head and 4 a request and head.
extern "C" int ns_memory_chunks(const void* proj, int stride, int q_off, int k_off, int v_off, int i_off, int f_off, const float* gate_bias_i,
                                const float* gate_bias_f, float* state, long long state_stride, const int* qo_indptr, const int* state_slots, float* out,
                                float* den, int n_tokens, int n_reqs, int H, int D, int E, float cap, float q_scale, float den_eps, int min_tokens,
                                void* gates, float* scratch, size_t scratch_floats, int dtype, hipStream_t stream) {
  if (n_tokens <= 0 || n_reqs <= 0 || n_reqs > 65535 || H <= 0 || D <= 0 || E <= 0 || E % 16 || E / 16 + 1 > 65535 || min_tokens < 1 || !(cap > 0.f))
    return NS_ERR_BAD_ARG;
  const int blocks = ns_memory_blocks(D, E);
  const size_t elem = dtype == NS_DTYPE_F32 ? 4 : 2;
  if (state_stride < (long long)H * E * D + (long long)H * blocks * (D + 1) || stride % 8 || q_off % 8 || k_off % 8 || (uintptr_t)proj % (8 * elem) ||
      (uintptr_t)scratch % 16 || (uintptr_t)gates % 8)
    return NS_ERR_BAD_ARG;
  MemoryChunks a;
  a.p = MemoryParams{proj, stride, q_off, k_off, v_off, i_off, f_off, gate_bias_i, gate_bias_f, state, state_stride, qo_indptr, state_slots,
                     out, den, H, D, E, cap, q_scale, den_eps, 1, 0};
  a.scratch = scratch, a.F = (double*)gates, a.gi = (float*)(a.F + (size_t)n_tokens * H), a.m = a.gi + (size_t)n_tokens * H,
  a.m0 = a.m + (size_t)n_tokens * H;
  a.n_reqs = n_reqs, a.from = 0, a.min_tokens = min_tokens, a.blocks = blocks;
  if (D == 64 && dtype == NS_DTYPE_F32) return memory_chunks<float, 64>(a, n_tokens, scratch_floats, stream);
  if (D == 64 && dtype == NS_DTYPE_BF16) return memory_chunks<bf16_t, 64>(a, n_tokens, scratch_floats, stream);
  if (D == 128 && dtype == NS_DTYPE_F32) return memory_chunks<float, 128>(a, n_tokens, scratch_floats, stream);
  if (D == 128 && dtype == NS_DTYPE_BF16) return memory_chunks<bf16_t, 128>(a, n_tokens, scratch_floats, stream);
  return NS_ERR_UNSUPPORTED;
}

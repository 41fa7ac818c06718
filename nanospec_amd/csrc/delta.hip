// The gated delta rule with one decay per head and key channel, and what surrounds it: the short causal convolution
// over time with its carried inputs, the unit vectors, decays and write strengths, the recurrence over a request's
// tokens with the state carried in its slot, and the gated RMS norm of the read-out.
//
// Per head, with S [D key channels][E value channels] (float, one per request and head):
//   S <- diag(g_t) S;   u = beta_t (v_t - S^T k_t);   S <- S + k_t u^T;   o_t = S^T q_t
// Column j of S only ever meets column j of v and o, so the columns of a head are independent chains: a thread owns 16
// key channels of one column in registers, the RG = D/16 threads of a column sit in neighbouring lanes and add their
// parts of the two dot products by lane exchange, and nothing waits at a barrier.  Everything here is 32-bit.
//
// A request's slot holds S [H][D][E] and behind it the last K - 1 inputs of the convolution [K - 1][C] (oldest first).
#include "chunk16.h"
#include <type_traits>

#define ND_MAX_TAPS 16
#define ND_ROWS 16  // key channels of a column that one thread owns

// ------------------------------------------------------------------------------------------------
// y[r][c] = silu(bias[c] + sum_j taps[c][j] * in(i - (K-1) + j)),  i the token's index among its request's tokens of this step;
// in(t) is this step's input for t >= 0 and the carried input K-1+t for t < 0.  ``bias`` may be null.  ``copy`` (or null)
// receives y in the type of the input as well, for a product that reads it.  ``carry``: a request that brings one token has its
// carried inputs shifted right here, by the thread that has just read them.
// ------------------------------------------------------------------------------------------------
template <typename T>
__global__ void conv_silu_kernel(float* __restrict__ out, T* __restrict__ copy, const T* __restrict__ x, int x_stride,
                                 const float* __restrict__ taps, const float* __restrict__ bias, float* __restrict__ state, size_t slot_stride, size_t conv_off, const int* __restrict__ token_req,
                                 const int* __restrict__ qo_indptr, const int* __restrict__ state_slots, int C, int K, int carry) {
  const int r = blockIdx.x, c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int b = token_req[r];
  const int i = r - qo_indptr[b];
  float* carried = state + (size_t)state_slots[b] * slot_stride + conv_off;
  float y = bias ? bias[c] : 0.f;
  for (int j = 0; j < K; ++j) {
    const int t = i - (K - 1) + j;
    const float v = t >= 0 ? to_f(x[(size_t)(r - (K - 1) + j) * x_stride + c]) : carried[(size_t)(K - 1 + t) * C + c];
    y = fmaf(taps[(size_t)c * K + j], v, y);
  }
  y = y / (1.f + expf(-y));
  out[(size_t)r * C + c] = y;
  if (copy) copy[(size_t)r * C + c] = from_f<T>(y);
  if (carry && K > 1 && qo_indptr[b + 1] - qo_indptr[b] == 1) {
    for (int j = 0; j + 2 < K; ++j) carried[(size_t)j * C + c] = carried[(size_t)(j + 1) * C + c];
    carried[(size_t)(K - 2) * C + c] = to_f(x[(size_t)r * x_stride + c]);
  }
}

// The same for four neighbouring channels a thread, with 16-byte accesses to taps, carried inputs and results, for the
// usual numbers of taps (so that the taps are registers) and channels that are a multiple of four.  A thread takes STRIP tokens one after the other: taps are
// 64 bytes a thread and an input is read by K tokens, for 8 bytes of new input and 16 of result.  The first ``units.vectors`` runs of 4 ``units.lanes`` channels (no more
// than C) then become unit vectors, as delta_prep_kernel makes them, while their sums of squares are at hand: a kernel of its own reads and writes them again.
// Bound by the results' bytes: 2,048 tokens of 6,144 channels, 4 taps, bfloat16, a token a thread 35.0 / 27.2 us (alone / beside two
// others) and the unit vectors and decays behind it 38.3 / 31.8, both in a row 69.1 / 57.4; so 30.6 / 19.8 and (decays alone) 18.7 / 14.3, 46.3 / 31.5.
template <int LANES>
__device__ __forceinline__ float unit_scale(const float* y, bool first_half) {
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) ss = fmaf(y[e], y[e], ss);
  return (first_half ? 1.f / sqrtf(4.f * LANES) : 1.f) / sqrtf(group_sum<LANES>(ss) + 1e-6f);
}

struct ConvUnits {
  int vectors, lanes;  // (lanes: of a vector, a power of two)
};

template <typename T, int K, int STRIP>
__global__ __launch_bounds__(256) void conv_silu_vec_kernel(float* __restrict__ out, T* __restrict__ copy, const T* __restrict__ x, int x_stride,
                                     const float* __restrict__ taps, const float* __restrict__ bias, float* __restrict__ state, size_t slot_stride, size_t conv_off, const int* __restrict__ token_req,
                                     const int* __restrict__ qo_indptr, const int* __restrict__ state_slots, int n, int C, int carry, ConvUnits units) {
  typedef T vec_t __attribute__((ext_vector_type(4)));
  const int r0 = blockIdx.x * STRIP, c = (blockIdx.y * blockDim.x + threadIdx.x) * 4;
  if (c >= C) return;
  // (all loads of the strip's inputs ahead of the first use; beyond the last token the last)
  vec_t in[STRIP];
#pragma unroll
  for (int s = 0; s < STRIP; ++s) in[s] = *reinterpret_cast<const vec_t*>(x + (size_t)min(r0 + s, n - 1) * x_stride + c);
  float tp[4 * K];  // taps of channel c + e / K, tap e % K
#pragma unroll
  for (int e = 0; e < K; ++e) {
    const float4 t = reinterpret_cast<const float4*>(taps + (size_t)c * K)[e];
    tp[4 * e] = t.x, tp[4 * e + 1] = t.y, tp[4 * e + 2] = t.z, tp[4 * e + 3] = t.w;
  }
  float4 bv = {0.f, 0.f, 0.f, 0.f};
  if (bias) bv = *reinterpret_cast<const float4*>(bias + c);
  float before[K - 1][4];  // the inputs before the token, oldest first
  int req = -1;
#pragma unroll
  for (int s = 0; s < STRIP; ++s) {
    const int r = r0 + s;
    if (r >= n) break;
    const int b = token_req[r];
    float* carried = state + (size_t)state_slots[b] * slot_stride + conv_off;
    if (b != req) {  // (the strip's first token, or a request's; the same for the whole workgroup)
      const int i = r - qo_indptr[b];
#pragma unroll
      for (int j = 0; j < K - 1; ++j) {
        const int t = i - (K - 1) + j;
        if (t >= 0) {
          const vec_t xv = *reinterpret_cast<const vec_t*>(x + (size_t)(r - (K - 1) + j) * x_stride + c);
#pragma unroll
          for (int e = 0; e < 4; ++e) before[j][e] = to_f((T)xv[e]);
        } else {
          const float4 cv = *reinterpret_cast<const float4*>(carried + (size_t)(K - 1 + t) * C + c);
          before[j][0] = cv.x, before[j][1] = cv.y, before[j][2] = cv.z, before[j][3] = cv.w;
        }
      }
      req = b;
    }
    float y[4] = {bv.x, bv.y, bv.z, bv.w}, now[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      now[e] = to_f((T)in[s][e]);
#pragma unroll
      for (int j = 0; j < K - 1; ++j) y[e] = fmaf(tp[e * K + j], before[j][e], y[e]);
      y[e] = fmaf(tp[e * K + K - 1], now[e], y[e]);
    }
    if (carry && qo_indptr[b + 1] - qo_indptr[b] == 1) {
#pragma unroll
      for (int j = 0; j + 1 < K; ++j) {
        const float* v = j + 2 < K ? before[j + 1 < K - 1 ? j + 1 : 0] : now;
        *reinterpret_cast<float4*>(carried + (size_t)j * C + c) = make_float4(v[0], v[1], v[2], v[3]);
      }
    }
#pragma unroll
    for (int j = 0; j + 2 < K; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) before[j][e] = before[j + 1][e];
#pragma unroll
    for (int e = 0; e < 4; ++e) before[K - 2][e] = now[e], y[e] = y[e] / (1.f + expf(-y[e]));
    const int vector = units.vectors ? c / (4 * units.lanes) : 0;
    if (vector < units.vectors) {
      const bool first = vector < units.vectors / 2;
      float f;
      switch (units.lanes) {
        case 2: f = unit_scale<2>(y, first); break;
        case 4: f = unit_scale<4>(y, first); break;
        case 8: f = unit_scale<8>(y, first); break;
        case 16: f = unit_scale<16>(y, first); break;
        case 32: f = unit_scale<32>(y, first); break;
        default: f = unit_scale<64>(y, first);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] *= f;
    }
    *reinterpret_cast<float4*>(out + (size_t)r * C + c) = make_float4(y[0], y[1], y[2], y[3]);
    if (copy) {
      const vec_t cv = {from_f<T>(y[0]), from_f<T>(y[1]), from_f<T>(y[2]), from_f<T>(y[3])};
      *reinterpret_cast<vec_t*>(copy + (size_t)r * C + c) = cv;
    }
  }
}

// After the convolution has read them: the carried inputs become the last K-1 inputs including this step's.
template <typename T>
__global__ void conv_carry_kernel(const T* __restrict__ x, int x_stride, float* __restrict__ state, size_t slot_stride, size_t conv_off,
                                  const int* __restrict__ qo_indptr, const int* __restrict__ state_slots, int C, int K) {
  const int b = blockIdx.y, c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int r0 = qo_indptr[b], L = qo_indptr[b + 1] - r0;
  if (L <= 0) return;
  float* carried = state + (size_t)state_slots[b] * slot_stride + conv_off;
  float old[ND_MAX_TAPS];
  for (int j = 0; j < K - 1; ++j) old[j] = carried[(size_t)j * C + c];
  for (int j = 0; j < K - 1; ++j) {
    const int t = L - (K - 1) + j;
    carried[(size_t)j * C + c] = t >= 0 ? to_f(x[(size_t)(r0 + t) * x_stride + c]) : old[K - 1 + t];
  }
}

#define CONV_STRIP 8     // tokens of a strip at most
// Workgroups that a step's strips come to at least, else they are shorter: two a compute unit.  us with the carry, strips of 1, 2, 4 and 8: 512 tokens of 2,048 channels 7.9, 7.5, 8.0, 9.8, of 2,304
// 8.2, 8.1, 8.6, 9.8, of 6,144 14.6, 13.4, 12.4, 13.6; 1,024 of 6,144 21.4, 18.6, 18.5, 18.2; 2,048 of 2,048 17.0, 15.2, 14.8, 14.2; of 6,144 33.5, 28.1, 26.0, 25.5.
#define CONV_GROUPS 512

// ``single``: every request brings one token (at most); one kernel then does both.  ``unit_vectors`` (an even number, or 0): so many first runs of ``unit_size`` channels become unit
// vectors, the first half of them times unit_size^(-1/2); unit_size a power of two from 8 to 256, and sizes and addresses as the kernel in pieces wants them (NS_ERR_UNSUPPORTED).
extern "C" int ns_conv_silu_carry(float* out, void* copy, const void* x, int x_stride, const float* taps, const float* bias, float* state, size_t slot_stride,
                                  size_t conv_off, const int* token_req, const int* qo_indptr, const int* state_slots, int n_tokens,
                                  int n_reqs, int C, int K, int single, int unit_vectors, int unit_size, int dtype, hipStream_t stream) {
  if (n_tokens <= 0 || n_reqs <= 0 || n_reqs > 65535 || C <= 0 || K < 1 || K > ND_MAX_TAPS || unit_vectors < 0 || unit_vectors % 2) return NS_ERR_BAD_ARG;
  if (unit_vectors && (unit_size <= 0 || (long long)unit_vectors * unit_size > C)) return NS_ERR_BAD_ARG;
  if (dtype != NS_DTYPE_F32 && dtype != NS_DTYPE_BF16) return NS_ERR_UNSUPPORTED;
  const int bx = (C + 255) / 256;
  if (bx > 65535) return NS_ERR_BAD_ARG;
  const size_t esize = dtype == NS_DTYPE_F32 ? 4 : 2;
  const bool vec = C % 4 == 0 && x_stride % 4 == 0 && ((uintptr_t)x % (4 * esize)) == 0 && ((uintptr_t)out % 16) == 0 && ((uintptr_t)taps % 16) == 0 &&
                   ((uintptr_t)bias % 16) == 0 && ((uintptr_t)copy % (4 * esize)) == 0 &&
                   ((uintptr_t)state % 16) == 0 && slot_stride % 4 == 0 && conv_off % 4 == 0 && K >= 2 && K <= 4;
  if (unit_vectors && !(vec && unit_size >= 8 && unit_size <= 256 && (unit_size & (unit_size - 1)) == 0)) return NS_ERR_UNSUPPORTED;
  if (vec) {
    const ConvUnits units{unit_vectors, unit_vectors ? unit_size / 4 : 1};
    const int across = (C / 4 + 255) / 256;
    int strip = single ? 1 : CONV_STRIP;
    while (strip > 1 && (long long)((n_tokens + strip - 1) / strip) * across < CONV_GROUPS) strip /= 2;
    const dim3 grid((n_tokens + strip - 1) / strip, across);
    auto launch = [&](auto* in, auto taps_of, auto strip) {
      typedef typename std::remove_const<typename std::remove_pointer<decltype(in)>::type>::type T;
      conv_silu_vec_kernel<T, decltype(taps_of)::value, decltype(strip)::value><<<grid, 256, 0, stream>>>(
          out, (T*)copy, in, x_stride, taps, bias, state, slot_stride, conv_off, token_req, qo_indptr, state_slots, n_tokens, C, single, units);
    };
    auto of_taps = [&](auto* in, auto strip) {
      if (K == 2)
        launch(in, std::integral_constant<int, 2>(), strip);
      else if (K == 3)
        launch(in, std::integral_constant<int, 3>(), strip);
      else
        launch(in, std::integral_constant<int, 4>(), strip);
    };
    auto of_strip = [&](auto* in) {
      switch (strip) {
        case 8: return of_taps(in, std::integral_constant<int, 8>());
        case 4: return of_taps(in, std::integral_constant<int, 4>());
        case 2: return of_taps(in, std::integral_constant<int, 2>());
        default: of_taps(in, std::integral_constant<int, 1>());
      }
    };
    if (dtype == NS_DTYPE_F32)
      of_strip((const float*)x);
    else
      of_strip((const bf16_t*)x);
  } else {
    dim3 grid(n_tokens, bx);
    if (dtype == NS_DTYPE_F32)
      conv_silu_kernel<float><<<grid, 256, 0, stream>>>(out, (float*)copy, (const float*)x, x_stride, taps, bias, state, slot_stride, conv_off, token_req,
                                                         qo_indptr, state_slots, C, K, single);
    else
      conv_silu_kernel<bf16_t><<<grid, 256, 0, stream>>>(out, (bf16_t*)copy, (const bf16_t*)x, x_stride, taps, bias, state, slot_stride, conv_off, token_req,
                                                          qo_indptr, state_slots, C, K, single);
  }
  if (K > 1 && !single) {
    dim3 grid(bx, n_reqs);
    if (dtype == NS_DTYPE_F32)
      conv_carry_kernel<float><<<grid, 256, 0, stream>>>((const float*)x, x_stride, state, slot_stride, conv_off, qo_indptr, state_slots, C, K);
    else
      conv_carry_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)x, x_stride, state, slot_stride, conv_off, qo_indptr, state_slots, C, K);
  }
  return ns_launch_status();
}

// ------------------------------------------------------------------------------------------------
// Per token: q and k of every key/value head become unit vectors, x / sqrt(sum(x^2) + 1e-6), q times D^(-1/2), in
// place in qkv [n][2 G D + H E]; g = exp(-exp(A_log[h]) softplus(a + dt_bias)) [n][H D]; beta = sigmoid(b) [n][H].
// ------------------------------------------------------------------------------------------------
// grid (tokens, Y): the first ceil(2 G / 4) blocks of a token take one vector a wave; the others 1,024 decays each (and
// the first of them the write strengths), so that no wave walks through a chain of dependent loads.
template <typename T>
__global__ void delta_prep_kernel(float* __restrict__ qkv, int C, float* __restrict__ g, float* __restrict__ beta, const T* __restrict__ a,
                                  int a_stride, const T* __restrict__ bp, int b_stride, const float* __restrict__ dt_bias,
                                  const float* __restrict__ a_log, int H, int G, int D, int norm_blocks) {
  const int r = blockIdx.x, lane = threadIdx.x & (NS_WAVE - 1), wave = threadIdx.x / NS_WAVE;
  if ((int)blockIdx.y < norm_blocks) {
    const int vec = blockIdx.y * 4 + wave;  // q heads, then k heads
    if (vec >= 2 * G) return;
    float* p = qkv + (size_t)r * C + (size_t)vec * D;
    float ss = 0.f;
    for (int d = lane; d < D; d += NS_WAVE) ss = fmaf(p[d], p[d], ss);
    ss = wave_sum(ss);
    const float f = (vec < G ? 1.f / sqrtf((float)D) : 1.f) / sqrtf(ss + 1e-6f);
    for (int d = lane; d < D; d += NS_WAVE) p[d] *= f;
    return;
  }
  const int part = blockIdx.y - norm_blocks;
  for (int i = part * 1024 + threadIdx.x; i < min(H * D, (part + 1) * 1024); i += blockDim.x) {
    const float z = to_f(a[(size_t)r * a_stride + i]) + dt_bias[i];
    g[(size_t)r * H * D + i] = expf(-expf(a_log[i / D]) * softplus_f(z));
  }
  if (part == 0)
    for (int h = threadIdx.x; h < H; h += blockDim.x) beta[(size_t)r * H + h] = 1.f / (1.f + expf(-to_f(bp[(size_t)r * b_stride + h])));
}

// The decays and write strengths alone, four decays a thread, where the unit vectors have been made already.  Sizes and strides multiples of four, whole pieces.
template <typename T>
__global__ __launch_bounds__(256) void delta_decay_kernel(float* __restrict__ g, float* __restrict__ beta, const T* __restrict__ a, int a_stride, const T* __restrict__ bp,
                                                          int b_stride, const float* __restrict__ dt_bias, const float* __restrict__ a_log, int H, int D) {
  typedef T vec_t __attribute__((ext_vector_type(4)));
  const int r = blockIdx.x, i = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (i < H * D) {
    const vec_t av = *reinterpret_cast<const vec_t*>(a + (size_t)r * a_stride + i);
    const float4 dv = *reinterpret_cast<const float4*>(dt_bias + i);
    const float rate = -expf(a_log[i / D]), dt[4] = {dv.x, dv.y, dv.z, dv.w};
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = expf(rate * softplus_f(to_f((T)av[e]) + dt[e]));
    *reinterpret_cast<float4*>(g + (size_t)r * H * D + i) = make_float4(v[0], v[1], v[2], v[3]);
  }
  if (blockIdx.y == 0)
    for (int h = threadIdx.x; h < H; h += 256) beta[(size_t)r * H + h] = 1.f / (1.f + expf(-to_f(bp[(size_t)r * b_stride + h])));
}

// ``units_made``: q and k are unit vectors already.
extern "C" int ns_delta_prep(float* qkv, int C, float* g, float* beta, const void* a, int a_stride, const void* bp, int b_stride,
                             const float* dt_bias, const float* a_log, int n_tokens, int H, int G, int D, int units_made, int dtype, hipStream_t stream) {
  if (n_tokens <= 0 || H <= 0 || G <= 0 || H % G || D <= 0 || C < 2 * G * D) return NS_ERR_BAD_ARG;
  const size_t piece = dtype == NS_DTYPE_F32 ? 16 : 8;
  if (units_made && D % 4 == 0 && a_stride % 4 == 0 && (uintptr_t)a % piece == 0 && (((uintptr_t)g | (uintptr_t)dt_bias) & 15) == 0 &&
      (dtype == NS_DTYPE_F32 || dtype == NS_DTYPE_BF16)) {
    const dim3 grid(n_tokens, (H * D / 4 + 255) / 256);
    if (grid.y > 65535) return NS_ERR_BAD_ARG;
    if (dtype == NS_DTYPE_F32)
      delta_decay_kernel<float><<<grid, 256, 0, stream>>>(g, beta, (const float*)a, a_stride, (const float*)bp, b_stride, dt_bias, a_log, H, D);
    else
      delta_decay_kernel<bf16_t><<<grid, 256, 0, stream>>>(g, beta, (const bf16_t*)a, a_stride, (const bf16_t*)bp, b_stride, dt_bias, a_log, H, D);
    return ns_launch_status();
  }
  const int norm_blocks = units_made ? 0 : (2 * G + 3) / 4, decay_blocks = (H * D + 1023) / 1024;
  if (norm_blocks + decay_blocks > 65535) return NS_ERR_BAD_ARG;
  const dim3 grid(n_tokens, norm_blocks + decay_blocks);
  if (dtype == NS_DTYPE_F32)
    delta_prep_kernel<float><<<grid, 256, 0, stream>>>(qkv, C, g, beta, (const float*)a, a_stride, (const float*)bp, b_stride, dt_bias,
                                                        a_log, H, G, D, norm_blocks);
  else if (dtype == NS_DTYPE_BF16)
    delta_prep_kernel<bf16_t><<<grid, 256, 0, stream>>>(qkv, C, g, beta, (const bf16_t*)a, a_stride, (const bf16_t*)bp, b_stride,
                                                         dt_bias, a_log, H, G, D, norm_blocks);
  else
    return NS_ERR_UNSUPPORTED;
  return ns_launch_status();
}

// ------------------------------------------------------------------------------------------------
// The recurrence.  grid (blocks of columns, heads, requests); a thread = (column jl of the block, row group rg), lane
// = jl * RG + rg, RG a power of two (at most 64) with 16 RG >= D.  Channels beyond D carry zeros.
//
// A token's step is a chain (decay, dot product, lane exchange, update, dot product, lane exchange) that cannot start
// before the token's operands are there, so the operands of the next ND_STAGE_FLOATS floats' worth of tokens are
// fetched by the whole workgroup at once (coalesced, all loads in flight together), parked in registers while the
// current stage's tokens are worked through from LDS, and then written to the other LDS buffer.  The arithmetic of a
// token is the same whatever the stage it falls into: results do not depend on how a prompt was cut.
// ------------------------------------------------------------------------------------------------
#define ND_PITCH (ND_ROWS + 4)                     // floats between two row groups' channels in LDS
#define ND_STAGE_FLOATS 6144                       // floats of one stage in LDS (two stages are held)
#define ND_STAGE_REGS (ND_STAGE_FLOATS / 1024)     // of which each of the 256 threads fetches this many groups of four

struct DeltaShape {
  int C, H, G, D, E, RG, Dl, cols, tok_stride, stage_tokens, vec4;
};

template <bool VEC, int RG, int ROWS>
__global__ __launch_bounds__(256) void delta_scan_kernel(float* __restrict__ o, const float* __restrict__ qkv,
                                                         const float* __restrict__ g, const float* __restrict__ beta,
                                                         float* __restrict__ state, size_t slot_stride, const int* __restrict__ qo_indptr,
                                                         const int* __restrict__ state_slots, DeltaShape p, int below) {
  __shared__ __attribute__((aligned(16))) float stage[2][ND_STAGE_FLOATS];
  // (the request is the slowest index of the launch: workgroups are dealt to the eight XCDs in turn, and with the request
  // as the fastest index all workgroups of the one long request among eight would land on one XCD)
  const int b = blockIdx.z, h = blockIdx.y;
  const int r0 = qo_indptr[b], r1 = qo_indptr[b + 1];
  if (r1 <= r0 || r1 - r0 >= below) return;
  const int D = p.D, E = p.E;
  constexpr int PITCH = ROWS + 4;  // floats between two row groups' channels in LDS
  constexpr int DL = RG * PITCH, COLS = 256 / RG;
  const int jl = threadIdx.x / RG, rg = threadIdx.x % RG;
  const int j0 = blockIdx.x * COLS, j = j0 + jl;
  const bool col_ok = j < E;
  const int d0 = rg * ROWS;
  const int kh = h / (p.H / p.G);
  float* S = state + (size_t)state_slots[b] * slot_stride + (size_t)h * D * E;
  float s[ROWS];
#pragma unroll
  for (int i = 0; i < ROWS; ++i) s[i] = (col_ok && d0 + i < D) ? S[(size_t)(d0 + i) * E + j] : 0.f;

  // what element e of a stage that starts at row `first` is: token e / tok_stride, then q [Dl] | k [Dl] | g [Dl] | v [cols] | beta;
  // in q, k and g the 16 channels of a row group are followed by four unused floats (PITCH), so that the row groups'
  // 16-byte reads fall into different banks
  const float* q_src = qkv + (size_t)kh * D;
  const float* k_src = qkv + (size_t)p.G * D + (size_t)kh * D;
  const float* v_src = qkv + (size_t)2 * p.G * D + (size_t)h * E + j0;
  const float* g_src = g + (size_t)h * D;
  const int stage_elems = p.stage_tokens * p.tok_stride;
  // A thread fetches groups of four floats; every part of a token's record starts at a multiple of four.  Which group of
  // which token's record a thread's i-th load is does not change from stage to stage, so source, row pitch and what is
  // kept of it are worked out once; a stage's loads then differ only in the row, and are issued without a branch around
  // any of them (a group that holds nothing reads the start of its source and is dropped when it is parked), so that
  // all of a stage's loads are in flight together and nothing waits for one before the stage's tokens are done.
  const float* src_of[ND_STAGE_REGS];
  int pitch_of[ND_STAGE_REGS], token_of[ND_STAGE_REGS];
  unsigned keep = 0, is_beta = 0;  // four bits a group: which of its floats are kept; one bit a group: its first float is beta
  {
    int tt = threadIdx.x * 4 / p.tok_stride, off = threadIdx.x * 4 - tt * p.tok_stride;  // of element e, kept up as e grows by 1024
#pragma unroll
    for (int i = 0; i < ND_STAGE_REGS; ++i) {
      const int e = (threadIdx.x + i * 256) * 4;
      const bool used = e < stage_elems;
      const int part = off < DL ? 0 : (off < 2 * DL ? 1 : (off < 3 * DL ? 2 : 3));
      const int within = off - part * DL, chunk = within / PITCH, w = within - chunk * PITCH;
      const int d = w < ROWS ? chunk * ROWS + w : 0x3fffffff;  // (the unused floats keep nothing)
      const int c = off - 3 * DL;
      const int at = part < 3 ? d : c;
      const int lim = !used ? 0 : (part < 3 ? D : min(COLS, E - j0));
      const float* src = part == 0 ? q_src : (part == 1 ? k_src : (part == 2 ? g_src : v_src));
      const unsigned bits = VEC ? (at < lim ? 0xfu : 0u)
                                : ((at < lim ? 1u : 0u) | (at + 1 < lim ? 2u : 0u) | (at + 2 < lim ? 4u : 0u) | (at + 3 < lim ? 8u : 0u));
      src_of[i] = src + (bits ? at : 0);
      pitch_of[i] = part == 2 ? p.H * D : p.C;
      token_of[i] = tt;
      keep |= bits << (4 * i);
      is_beta |= (used && part >= 3 && c == COLS ? 1u : 0u) << i;
      off += 1024;
      while (off >= p.tok_stride) off -= p.tok_stride, ++tt;
    }
  }
  struct Stage {
    float4 v[ND_STAGE_REGS];
    float bt[ND_STAGE_REGS];
    unsigned live;  // one bit a group: its token is one of the request's
  };
  auto fetch = [&](Stage& st, int first) {
    st.live = 0;
#pragma unroll
    for (int i = 0; i < ND_STAGE_REGS; ++i) {
      const int r = min(first + token_of[i], r1 - 1);
      st.live |= (first + token_of[i] < r1 ? 1u : 0u) << i;
      const float* src = src_of[i] + (size_t)r * pitch_of[i];
      if constexpr (VEC) {
        st.v[i] = *reinterpret_cast<const float4*>(src);
      } else {
        const unsigned k = keep >> (4 * i);
        st.v[i] = float4{src[0], src[k & 2u ? 1 : 0], src[k & 4u ? 2 : 0], src[k & 8u ? 3 : 0]};
      }
      st.bt[i] = beta[(size_t)r * p.H + h];
    }
  };
  auto park = [&](const Stage& st, float* buf) {
#pragma unroll
    for (int i = 0; i < ND_STAGE_REGS; ++i) {
      const int e = (threadIdx.x + i * 256) * 4;
      const bool live = (st.live >> i) & 1u;
      const unsigned k = live ? keep >> (4 * i) : 0u;
      float4 val = {k & 1u ? st.v[i].x : 0.f, k & 2u ? st.v[i].y : 0.f, k & 4u ? st.v[i].z : 0.f, k & 8u ? st.v[i].w : 0.f};
      if (live && ((is_beta >> i) & 1u)) val.x = st.bt[i];
      if (e < stage_elems) *reinterpret_cast<float4*>(buf + e) = val;
    }
  };

  // where this thread's output of the next token goes (the first lane of a column's group writes it)
  const bool writes = rg == 0 && col_ok;
  const size_t out_stride = (size_t)p.H * E;
  float* op = o + (size_t)r0 * out_stride + (size_t)h * E + (col_ok ? j : 0);
  Stage regs;
  fetch(regs, r0);
  park(regs, stage[0]);
  __syncthreads();
  int cur = 0;
  for (int first = r0; first < r1; first += p.stage_tokens) {
    const bool more = first + p.stage_tokens < r1;
    if (more) fetch(regs, first + p.stage_tokens);
    const float* buf = stage[cur];
    const int n = min(p.stage_tokens, r1 - first);
    // Two sets of operand registers take turns: the next token's operands are read from LDS into one while the chain of
    // the current token runs on the other (written out twice, so that no set is ever copied into the other).
    struct Operands {
      float4 q[ROWS / 4], k[ROWS / 4], g[ROWS / 4];
      float v, b;
    };
    auto read_token = [&](Operands& t, int tt) {
      const float* tok = buf + tt * p.tok_stride;
#pragma unroll
      for (int i = 0; i < ROWS / 4; ++i) {
        t.q[i] = reinterpret_cast<const float4*>(tok + rg * PITCH)[i];
        t.k[i] = reinterpret_cast<const float4*>(tok + DL + rg * PITCH)[i];
        t.g[i] = reinterpret_cast<const float4*>(tok + 2 * DL + rg * PITCH)[i];
      }
      t.v = tok[3 * DL + jl], t.b = tok[3 * DL + COLS];
    };
    auto chain = [&](const Operands& t) {
      float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < ROWS / 4; ++i) {
        s[4 * i] *= t.g[i].x, s[4 * i + 1] *= t.g[i].y, s[4 * i + 2] *= t.g[i].z, s[4 * i + 3] *= t.g[i].w;
        part[0] = fmaf(t.k[i].x, s[4 * i], part[0]);
        part[1] = fmaf(t.k[i].y, s[4 * i + 1], part[1]);
        part[2] = fmaf(t.k[i].z, s[4 * i + 2], part[2]);
        part[3] = fmaf(t.k[i].w, s[4 * i + 3], part[3]);
      }
      const float dot = group_sum<RG>((part[0] + part[1]) + (part[2] + part[3]));
      const float u = t.b * (t.v - dot);
      float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < ROWS / 4; ++i) {
        s[4 * i] = fmaf(t.k[i].x, u, s[4 * i]);
        s[4 * i + 1] = fmaf(t.k[i].y, u, s[4 * i + 1]);
        s[4 * i + 2] = fmaf(t.k[i].z, u, s[4 * i + 2]);
        s[4 * i + 3] = fmaf(t.k[i].w, u, s[4 * i + 3]);
        acc[0] = fmaf(t.q[i].x, s[4 * i], acc[0]);
        acc[1] = fmaf(t.q[i].y, s[4 * i + 1], acc[1]);
        acc[2] = fmaf(t.q[i].z, s[4 * i + 2], acc[2]);
        acc[3] = fmaf(t.q[i].w, s[4 * i + 3], acc[3]);
      }
      const float out = group_sum<RG>((acc[0] + acc[1]) + (acc[2] + acc[3]));
      if (writes) *op = out;
      op += out_stride;
    };
    Operands ta, tb;
    read_token(ta, 0);
    for (int tt = 0; tt < n; tt += 2) {
      if (tt + 1 < n) read_token(tb, tt + 1);
      chain(ta);
      if (tt + 1 < n) {
        if (tt + 2 < n) read_token(ta, tt + 2);
        chain(tb);
      }
    }
    if (more) park(regs, stage[cur ^ 1]);
    __syncthreads();
    cur ^= 1;
  }
#pragma unroll
  for (int i = 0; i < ROWS; ++i)
    if (col_ok && d0 + i < D) S[(size_t)(d0 + i) * E + j] = s[i];
}

extern "C" int ns_delta_scan(float* o, const float* qkv, int C, const float* g, const float* beta, float* state, size_t slot_stride,
                             const int* qo_indptr, const int* state_slots, int n_reqs, int H, int G, int D, int E, int below, hipStream_t stream) {
  if (n_reqs <= 0 || H <= 0 || G <= 0 || H % G || D <= 0 || D > ND_ROWS * NS_WAVE || E <= 0 || H > 65535) return NS_ERR_BAD_ARG;
  DeltaShape p;
  p.C = C, p.H = H, p.G = G, p.D = D, p.E = E;
  // A thread owns 8 key channels of a column where the key size allows it (more, shorter chains: a token's step is
  // latency, and a single request leaves most of the GPU idle anyway), 16 beyond 512 channels.
  const int rows = D <= 8 * NS_WAVE ? 8 : ND_ROWS;
  p.RG = 1;
  while (p.RG * rows < D) p.RG *= 2;
  p.Dl = p.RG * (rows + 4);
  p.cols = 256 / p.RG;
  p.tok_stride = 3 * p.Dl + ((p.cols + 1 + 3) / 4) * 4;
  p.stage_tokens = ND_STAGE_FLOATS / p.tok_stride;
  if (p.stage_tokens < 1) return NS_ERR_BAD_ARG;
  if (p.stage_tokens > 64) p.stage_tokens = 64;
  // 16-byte loads where every group of four that a thread fetches starts at a multiple of four floats
  p.vec4 = (D % 4 == 0 && E % 4 == 0 && C % 4 == 0 && ((uintptr_t)qkv % 16) == 0 && ((uintptr_t)g % 16) == 0) ? 1 : 0;
  const int zb = (E + p.cols - 1) / p.cols;
  if (n_reqs > 65535) return NS_ERR_BAD_ARG;
  const dim3 grid(zb, H, n_reqs);
#define ND_LAUNCH2(R, W)                                                                                                               \
  if (p.vec4) delta_scan_kernel<true, R, W><<<grid, 256, 0, stream>>>(o, qkv, g, beta, state, slot_stride, qo_indptr, state_slots, p, below); \
  else delta_scan_kernel<false, R, W><<<grid, 256, 0, stream>>>(o, qkv, g, beta, state, slot_stride, qo_indptr, state_slots, p, below)
#define ND_LAUNCH(R)                    \
  case R:                               \
    if (rows == 8) { ND_LAUNCH2(R, 8); } \
    else { ND_LAUNCH2(R, ND_ROWS); }    \
    break
  switch (p.RG) {
    ND_LAUNCH(1);
    ND_LAUNCH(2);
    ND_LAUNCH(4);
    ND_LAUNCH(8);
    ND_LAUNCH(16);
    ND_LAUNCH(32);
    default: ND_LAUNCH(64);
  }
#undef ND_LAUNCH2
#undef ND_LAUNCH
  return ns_launch_status();
}

// ------------------------------------------------------------------------------------------------
// The same recurrence for prompt portions, sixteen tokens at a time.  With G_i the product of the decays of the chunk's tokens up to
// i (by key channel) and S the state before the chunk, the tokens of a chunk are one small triangular system:
//   A_ij = sum_d k_i k_j prod_{j < t <= i} g_t  (j < i);   P_ij = the same with q_i (j <= i);   T = (1 + diag(beta) A)^-1 diag(beta)
//   U = T (V - (K G) S);   O = (Q G) S + P U;   S <- G_15 S + (K prod_{t > i} g_t)^T U
// All products of decays are formed by multiplication, so that they are at most one and a decay of zero is no special case.
//
// The token form above is a chain of some 340 ns a token, whatever the GPU could do beside it.  Here what does not depend on the state (A, P, T
// and the scaled keys and queries) is made for all chunks at once by ``delta_chunk_kernel``, as the matrix instruction's operands in the order
// of its lanes, and ``delta_pass_kernel`` goes from chunk to chunk: four waves hold 16 columns of S in the layout in which the instruction
// leaves its result and takes its second operand alike (v_mfma_f32_16x16x4_f32, 32-bit products and sums), so S never leaves the
// registers; their shares of (K G) S and (Q G) S + P U meet in LDS, one barrier a chunk; a fifth wave adds up and writes the output.
// Bound by the chain of a chunk (29 matrix instructions of 32 cycles, two of them waiting for LDS).  16 heads of 128 by 128, 2,048 tokens:
// 672 us token by token, 43 + 114 us so; 512 tokens 174 -> 46 us.  The workgroups of a head lie on one XCD, whose L2 then serves the
// records to all its columns.  Sums over channels, products of decays and T are formed in 64 bits, which costs 18 us of the 43:
// relative error (2-norm, against 64 bits throughout) of the output 8.8e-8 token by token and 6.5e-8 so with decays around 0.5,
// 2.0e-7 and 1.6e-7 with decays around 0.99, of the state 5.1e-8 and 5.1e-8, 1.9e-7 and 1.5e-7.
// A sum of a product with a zero beside an infinity would carry a token's infinity to the tokens before it; where a chunk's values are
// not finite its sums leave out what they may not see.
// ------------------------------------------------------------------------------------------------
struct DeltaChunks {
  const float *qkv, *g, *beta;
  float *o, *state, *scratch;  // scratch: a record for every chunk and head: K G | Q G | K rest (16 D each) | T | P (256 each) | G_15 (D)
  const int *qo_indptr, *state_slots;
  size_t slot_stride;
  int C, H, G, E, n_reqs, from, min_tokens;  // the records begin at chunk `from`
};

template <int D>
__device__ __forceinline__ size_t chunk_record(const DeltaChunks& p, int chunk, int h) {
  return ((size_t)(chunk - p.from) * p.H + h) * (3 * DC_T * D + 2 * DC_T * DC_T + D);
}

template <int D>
__global__ __launch_bounds__(256) void delta_chunk_kernel(const DeltaChunks p) {
  constexpr int LD = D + 4, CH = D / 16;  // channels of a thread in the sums over channels
  constexpr int TASKS = (2 * D + 255) / 256;
  __shared__ __attribute__((aligned(16))) float kqg[3][DC_T][LD];
  __shared__ double a_s[DC_T][DC_T + 1];
  __shared__ float p_s[DC_T][DC_T + 1], t_s[DC_T][DC_T + 1], beta_s[DC_T];
  const int chunk = p.from + blockIdx.y, h = blockIdx.x, tid = threadIdx.x;
  const int lo = chunk_request(p.qo_indptr, p.n_reqs, chunk);
  const int r0 = p.qo_indptr[lo], r1 = p.qo_indptr[lo + 1], row0 = r0 + (chunk - r0 / DC_T - lo) * DC_T;
  if (row0 >= r1 || r1 - r0 < p.min_tokens) return;
  const int n = min(DC_T, r1 - row0), kh = h / (p.H / p.G);
  // tokens beyond the request's last: no key, no query, a decay of one, a write strength of zero
  for (int e = tid; e < 3 * DC_T * (D / 4); e += 256) {
    const int which = e / (DC_T * (D / 4)), i = e / (D / 4) % DC_T, d = 4 * (e % (D / 4));
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (which == 2) v = f32x4{1.f, 1.f, 1.f, 1.f};
    if (i < n) {
      const size_t r = row0 + i;
      v = *reinterpret_cast<const f32x4*>(which == 0   ? p.qkv + r * p.C + (size_t)p.G * D + (size_t)kh * D + d
                                          : which == 1 ? p.qkv + r * p.C + (size_t)kh * D + d
                                                       : p.g + (r * p.H + h) * D + d);
    }
    *reinterpret_cast<f32x4*>(&kqg[which][i][d]) = v;
  }
  if (tid < DC_T) beta_s[tid] = tid < n ? p.beta[(size_t)(row0 + tid) * p.H + h] : 0.f;
  __syncthreads();
  {  // A and P: a thread has one token j and every 16th piece of four channels
    const int j = tid / 16, seg = tid % 16;
    double w[CH], v[2 * DC_T];
#pragma unroll
    for (int u = 0; u < CH; u += 4) {
      const f32x4 k = *reinterpret_cast<const f32x4*>(&kqg[0][j][4 * seg + 16 * u]);
#pragma unroll
      for (int c = 0; c < 4; ++c) w[u + c] = k[c];
    }
#pragma unroll
    for (int i = 0; i < DC_T; ++i) {
      double ka = 0., qa = 0.;
#pragma unroll
      for (int u = 0; u < CH; u += 4) {
        const f32x4 k = *reinterpret_cast<const f32x4*>(&kqg[0][i][4 * seg + 16 * u]), q = *reinterpret_cast<const f32x4*>(&kqg[1][i][4 * seg + 16 * u]);
        const f32x4 g = *reinterpret_cast<const f32x4*>(&kqg[2][i][4 * seg + 16 * u]);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          w[u + c] = i > j ? w[u + c] * g[c] : w[u + c];
          ka = fma((double)k[c], w[u + c], ka);
          qa = fma((double)q[c], w[u + c], qa);
        }
      }
      v[i] = ka, v[DC_T + i] = qa;
    }
    // 32 sums over 16 lanes: in four steps every lane gives away half of what it has; lane seg ends up with sums 2 seg and 2 seg + 1
#pragma unroll
    for (int o = 8; o; o >>= 1)
#pragma unroll
      for (int x = 0; x < 2 * o; ++x) {
        const bool up = seg & o;
        const double keep = up ? v[x + 2 * o] : v[x], give = up ? v[x] : v[x + 2 * o];
        v[x] = keep + __shfl_xor(give, o, NS_WAVE);
      }
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      const int i = (2 * seg + x) % DC_T;
      if (seg < 8) a_s[i][j] = i > j ? v[x] : 0.;
      else p_s[i][j] = i >= j ? (float)v[x] : 0.f;
    }
  }
  // products of decays along the tokens: a thread a channel, forwards for K G and Q G, backwards for the keys' way to the chunk's end
  float* rec = p.scratch + chunk_record<D>(p, chunk, h);
  float first[TASKS][DC_T], second[TASKS][DC_T];
#pragma unroll
  for (int x = 0; x < TASKS; ++x) {
    const int task = tid + 256 * x, d = task % D;
    if (task < D) {
      double all = 1.;
#pragma unroll
      for (int i = 0; i < DC_T; ++i) {
        all *= kqg[2][i][d];
        first[x][i] = (float)(kqg[0][i][d] * all), second[x][i] = (float)(kqg[1][i][d] * all);
      }
      rec[3 * DC_T * D + 2 * DC_T * DC_T + d] = (float)all;
    } else if (task < 2 * D) {
      double rest = 1.;
#pragma unroll
      for (int i = DC_T - 1; i >= 0; --i) {
        first[x][i] = (float)(kqg[0][i][d] * rest);
        rest *= kqg[2][i][d];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int x = 0; x < TASKS; ++x) {
    const int task = tid + 256 * x, d = task % D;
    if (task < D) {
#pragma unroll
      for (int i = 0; i < DC_T; ++i) kqg[0][i][d] = first[x][i], kqg[1][i][d] = second[x][i];
    } else if (task < 2 * D) {
#pragma unroll
      for (int i = 0; i < DC_T; ++i) kqg[2][i][d] = first[x][i];
    }
  }
  if (tid < DC_T) {  // T, a column a lane
    double x[DC_T];
#pragma unroll
    for (int i = 0; i < DC_T; ++i) {
      double s = 0.;
#pragma unroll
      for (int j = 0; j < i; ++j) s = fma(a_s[i][j], x[j], s);
      x[i] = i < tid ? 0. : (i == tid ? 1. : -beta_s[i] * s);
    }
#pragma unroll
    for (int i = 0; i < DC_T; ++i) t_s[i][tid] = i < tid ? 0.f : (float)(x[i] * beta_s[tid]);  // (beta may be no number: 0 beta is none either)
  }
  __syncthreads();
  for (int e = tid; e < 3 * DC_T * (D / 4); e += 256) {
    const int which = e / (DC_T * (D / 4)), at = e % (DC_T * (D / 4)), tile = at / NS_WAVE, r = at % 16, gq = at % NS_WAVE / 16;
    f32x4 v;
    if (which < 2) {  // row: token, four channels of the tile
      v = *reinterpret_cast<const f32x4*>(&kqg[which][chunk_token(r)][16 * tile + 4 * gq]);
    } else {  // row: channel of the tile, four tokens
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = kqg[2][chunk_token(4 * gq + i)][16 * tile + r];
    }
    *reinterpret_cast<f32x4*>(rec + 4 * (size_t)e) = v;
  }
  if (tid < 2 * NS_WAVE) {
    const int r = tid % 16, gq = tid % NS_WAVE / 16;
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (tid < NS_WAVE ? t_s : p_s)[chunk_token(r)][chunk_token(4 * gq + i)];
    *reinterpret_cast<f32x4*>(rec + 3 * DC_T * D + 4 * tid) = v;
  }
}

template <int D>
__global__ __launch_bounds__(5 * NS_WAVE) void delta_pass_kernel(const DeltaChunks p, int to) {
  constexpr int TILES = D / 64;  // tiles of 16 key channels a wave holds
  __shared__ f32x4 part[2][2][4][NS_WAVE];
  const int b = blockIdx.z, h = blockIdx.x, lane = threadIdx.x & 63, c = lane & 15, gq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r0 = p.qo_indptr[b], r1 = p.qo_indptr[b + 1], first = r0 / DC_T + b;
  if (r1 - r0 < p.min_tokens) return;
  const int begin = max(first, p.from), end = min(first + (r1 - r0 + DC_T - 1) / DC_T, to);
  if (begin >= end) return;
  // the token of a lane's row i of a chunk is 4 i + gq; the last one that the request has
  auto last_of = [&](int chunk) { return min(DC_T, r1 - r0 - (chunk - first) * DC_T) - 1; };
  struct Operands {
    f32x4 k[TILES], q[TILES], rest[TILES], all[TILES], t, v;
    float p;
  };
  auto joined = [&](int which, int buf) {
    return (part[buf][which][0][lane] + part[buf][which][1][lane]) + (part[buf][which][2][lane] + part[buf][which][3][lane]);
  };
  // the operands of the two chunks ahead are on their way while one is worked through; (Q G) S + P U of a chunk is made behind the
  // barrier, (Q G) S while (K G) S comes back from LDS, and so meets the fifth wave a barrier later
  auto every = [&](auto&& fetch, auto&& work) {
    Operands o0, o1, o2;
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
  };
  if (wave < 4) {
    float* S = p.state + (size_t)p.state_slots[b] * p.slot_stride + ((size_t)h * D + wave * TILES * 16 + 4 * gq) * p.E + blockIdx.y * 16 + c;
    const float* v_src = p.qkv + (size_t)2 * p.G * D + (size_t)h * p.E + blockIdx.y * 16;
    unsigned v_at[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v_at[i] = (4 * i + gq) * p.C + c;
    f32x4 s[TILES];
#pragma unroll
    for (int x = 0; x < TILES; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[x][i] = S[(size_t)(x * 16 + i) * p.E];
    every(
        [&](Operands& o, int chunk) {
          chunk = min(chunk, end - 1);
          const float* rec = p.scratch + chunk_record<D>(p, chunk, h);
#pragma unroll
          for (int x = 0; x < TILES; ++x) {
            const int tile = wave * TILES + x;
            o.k[x] = *reinterpret_cast<const f32x4*>(rec + tile * 256 + 4 * lane);
            o.q[x] = *reinterpret_cast<const f32x4*>(rec + DC_T * D + tile * 256 + 4 * lane);
            o.rest[x] = *reinterpret_cast<const f32x4*>(rec + 2 * DC_T * D + tile * 256 + 4 * lane);
            o.all[x] = *reinterpret_cast<const f32x4*>(rec + 3 * DC_T * D + 2 * DC_T * DC_T + tile * 16 + 4 * gq);
          }
          o.t = *reinterpret_cast<const f32x4*>(rec + 3 * DC_T * D + 4 * lane);
          o.p = rec[3 * DC_T * D + DC_T * DC_T + 4 * lane + wave];  // what this wave gives of P U: four tokens
          const float* from = v_src + (size_t)(r0 + (chunk - first) * DC_T) * p.C;
          const unsigned last = last_of(chunk) * p.C + c;
#pragma unroll
          for (int i = 0; i < 4; ++i) o.v[i] = from[min(v_at[i], last)];
        },
        [&](const Operands& o, int chunk) {
          f32x4 ak[TILES], aq[TILES];
#pragma unroll
          for (int x = 0; x < TILES; ++x) ak[x] = aq[x] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int x = 0; x < TILES; ++x) ak[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.k[x][i], s[x][i], ak[x], 0, 0, 0);
#pragma unroll
          for (int x = 1; x < TILES; ++x) ak[0] += ak[x];
          part[chunk & 1][0][wave][lane] = ak[0];
          __syncthreads();
          f32x4 w = o.v - joined(0, chunk & 1), u = {0.f, 0.f, 0.f, 0.f};
          const int last = last_of(chunk);
#pragma unroll
          for (int i = 0; i < 4; ++i) w[i] = 4 * i + gq <= last ? w[i] : 0.f;
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int x = 0; x < TILES; ++x) aq[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.q[x][i], s[x][i], aq[x], 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) u = __builtin_amdgcn_mfma_f32_16x16x4f32(o.t[i], w[i], u, 0, 0, 0);
#pragma unroll
          for (int x = 1; x < TILES; ++x) aq[0] += aq[x];
          if (__any(not_finite(w) || not_finite(u))) {
            const float* t = p.scratch + chunk_record<D>(p, chunk, h) + 3 * DC_T * D;
            u = lower_product(t, w, lane);
            if (wave == 0) aq[0] += lower_product(t + DC_T * DC_T, u, lane);
          } else {
            aq[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.p, wave < 2 ? (wave == 0 ? u[0] : u[1]) : (wave == 2 ? u[2] : u[3]), aq[0], 0, 0, 0);
          }
          part[chunk & 1][1][wave][lane] = aq[0];
#pragma unroll
          for (int x = 0; x < TILES; ++x) s[x] *= o.all[x];
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int x = 0; x < TILES; ++x) s[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.rest[x][i], u[i], s[x], 0, 0, 0);
        });
    __syncthreads();
#pragma unroll
    for (int x = 0; x < TILES; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[(size_t)(x * 16 + i) * p.E] = s[x][i];
  } else {
    float* to_o = p.o + (size_t)h * p.E + blockIdx.y * 16;
    const int o_stride = p.H * p.E;
    for (int chunk = begin; chunk <= end; ++chunk) {
      __syncthreads();
      if (chunk == begin) continue;
      const f32x4 out = joined(1, (chunk - 1) & 1);
      float* row = to_o + (size_t)(r0 + (chunk - 1 - first) * DC_T) * o_stride;
      const int last = last_of(chunk - 1);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (4 * i + gq <= last) row[(4 * i + gq) * o_stride + c] = out[i];
    }
  }
}

template <int D>
static int delta_chunks(DeltaChunks p, int n_tokens, size_t scratch_floats, hipStream_t stream) {
  const int chunks = n_tokens / DC_T + p.n_reqs;
  const size_t per = (size_t)p.H * (3 * DC_T * D + 2 * DC_T * DC_T + D);
  const size_t fit = scratch_floats / per;  // chunks whose records fit; a longer batch goes in several passes, the state in its slots between them
  if (fit < 1) return NS_ERR_BAD_ARG;
  for (int from = 0; from < chunks;) {
    const int left = chunks - from < 65535 ? chunks - from : 65535, now = fit < (size_t)left ? (int)fit : left;
    p.from = from;
    delta_chunk_kernel<D><<<dim3(p.H, now), 256, 0, stream>>>(p);
    delta_pass_kernel<D><<<dim3(p.H, p.E / 16, p.n_reqs), 5 * NS_WAVE, 0, stream>>>(p, from + now);
    from += now;
  }
  return ns_launch_status();
}

// Requests of at least ``min_tokens`` tokens; the others are ``ns_delta_scan``'s (with ``below`` the same number).
extern "C" int ns_delta_chunks(float* o, const float* qkv, int C, const float* g, const float* beta, float* state, size_t slot_stride, const int* qo_indptr,
                               const int* state_slots, int n_tokens, int n_reqs, int H, int G, int D, int E, int min_tokens, float* scratch,
                               size_t scratch_floats, hipStream_t stream) {
  if (n_tokens <= 0 || n_reqs <= 0 || n_reqs > 65535 || H <= 0 || H > 65535 || G <= 0 || H % G || E <= 0 || E % 16 || C % 4 || min_tokens < 1 ||
      (uintptr_t)qkv % 16 || (uintptr_t)g % 16 || (uintptr_t)scratch % 16)
    return NS_ERR_BAD_ARG;
  const DeltaChunks p{qkv, g, beta, o, state, scratch, qo_indptr, state_slots, slot_stride, C, H, G, E, n_reqs, 0, min_tokens};
  if (D == 64) return delta_chunks<64>(p, n_tokens, scratch_floats, stream);
  if (D == 128) return delta_chunks<128>(p, n_tokens, scratch_floats, stream);
  return NS_ERR_UNSUPPORTED;
}

// ------------------------------------------------------------------------------------------------
// out[r][h][:] = o / sqrt(mean(o^2) + eps) * w[:] * sigmoid(gate[r][h][:]),  o float, gate and out in the model's type.
// ``gate_first``: the gate stands in front of the norm, x = o * gate, out = x / sqrt(mean(x^2) + eps) * w[:].
// ------------------------------------------------------------------------------------------------
template <typename T>
__global__ void gated_rms_kernel(T* __restrict__ out, const float* __restrict__ o, const T* __restrict__ gate, int gate_stride,
                                 const float* __restrict__ w, int w_stride, const float* __restrict__ den, int H, int E, float eps, int silu,
                                 int gate_first) {
  __shared__ float scratch[16];
  const int r = blockIdx.x, h = blockIdx.y;
  if (w) w += (size_t)h * w_stride;  // 0: all heads share one weight; no weight at all: the factor is 1
  const float* p = o + ((size_t)r * H + h) * E;
  const float dinv = den ? 1.f / den[(size_t)r * H + h] : 1.f;  // a head's read-out that comes undivided
  // the gate: sigmoid(z), or with ``silu`` z sigmoid(z)
  auto gate_of = [&](int e) {
    const float z = to_f(gate[(size_t)r * gate_stride + (size_t)h * E + e]);
    return (silu ? z : 1.f) / (1.f + expf(-z));
  };
  float ss = 0.f;
  for (int e = threadIdx.x; e < E; e += blockDim.x) {
    const float v = p[e] * dinv * (gate_first ? gate_of(e) : 1.f);
    ss = fmaf(v, v, ss);
  }
  ss = blockDim.x > NS_WAVE ? block_sum(ss, scratch) : wave_sum(ss);
  const float rinv = 1.f / sqrtf(ss / (float)E + eps);
  for (int e = threadIdx.x; e < E; e += blockDim.x)
    out[((size_t)r * H + h) * E + e] = from_f<T>(p[e] * dinv * rinv * (w ? w[e] : 1.f) * gate_of(e));
}

extern "C" int ns_gated_rms(void* out, const float* o, const void* gate, int gate_stride, const float* w, int w_stride, const float* den,
                            int n_tokens, int H, int E, float eps, int silu, int gate_first, int dtype, hipStream_t stream) {
  if (n_tokens <= 0 || H <= 0 || H > 65535 || E <= 0) return NS_ERR_BAD_ARG;
  dim3 grid(n_tokens, H);
  // a wave a head, four for wide heads (all heads normed as one), sixteen where there are few rows of them
  const int threads = E <= 512 ? NS_WAVE : (E > 1024 && n_tokens <= 64 ? 1024 : 256);
  if (dtype == NS_DTYPE_F32)
    gated_rms_kernel<float><<<grid, threads, 0, stream>>>((float*)out, o, (const float*)gate, gate_stride, w, w_stride, den, H, E, eps, silu, gate_first);
  else if (dtype == NS_DTYPE_BF16)
    gated_rms_kernel<bf16_t><<<grid, threads, 0, stream>>>((bf16_t*)out, o, (const bf16_t*)gate, gate_stride, w, w_stride, den, H, E, eps, silu, gate_first);
  else
    return NS_ERR_UNSUPPORTED;
  return ns_launch_status();
}

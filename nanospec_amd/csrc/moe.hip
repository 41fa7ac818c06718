// A mixture of small feed-forward experts, and the per-layer token input of a decoder that has one.
//
// Router: z = W_r h + b in 32-bit; the ``top`` largest logits are chosen (the lower index wins a tie) and weighted by the
// soft-max over the chosen logits alone; or sigmoid scores with a correction on the choice and groups of experts (see
// ``moe_choose_kernel``).
// Expert (``clipped GLU``): g = min(W_gate h, limit); u = clamp(W_up h, -limit, limit); y = W_down (g sigmoid(alpha g) (u + shift));
// an infinite limit clips nothing, and with alpha = 1 and shift = 0 the expert is W_down (silu(W_gate h) * W_up h).
// Or, without gate matrices (``wg`` null): y = W_down act(W_up h) with one of the activations that common.h numbers.
// The experts' matrices are stacked: gate and up [experts][ff][W], down [experts][W][ff].
// More rows may stand below the experts' in the router's matrix (a shared expert's gate): their logits are formed and kept
// beside the experts' and have no part in the choice.
// The last outputs of a router may be identity experts, which have no matrices: what such a pair adds is its weight times the
// input row, formed where the pairs are added up (``moe_combine``); the experts' kernels leave these pairs out.
#include "common.h"
#include "tile_quarters.h"

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
#define MOE_MAX_EXPERTS 1024
#define MOE_MAX_TOP 32

// Two kernels.  Logits: a workgroup takes ROUTE_TOK tokens and four experts, a wave an expert: it reads the expert's row
// once (16 bytes a lane a load where the sizes allow) for all of its tokens.  Choice: a wave a token.
#define ROUTE_TOK 8
template <typename T>
__global__ __launch_bounds__(256) void moe_logits_kernel(const T* __restrict__ h, int h_stride, const float* __restrict__ wr,
                                                         const float* __restrict__ br, float* __restrict__ z, int n, int W, int experts, int vec) {
  const int t0 = blockIdx.x * ROUTE_TOK, lane = threadIdx.x % NS_WAVE, wave = threadIdx.x / NS_WAVE;
  const int e = blockIdx.y * (blockDim.x / NS_WAVE) + wave;
  if (e >= experts) return;
  const int nt = min(ROUTE_TOK, n - t0);
  const float* w = wr + (size_t)e * W;
  float acc[ROUTE_TOK];
#pragma unroll
  for (int i = 0; i < ROUTE_TOK; ++i) acc[i] = 0.f;
  if (vec) {
#pragma unroll 2
    for (int c = lane * 4; c < W; c += NS_WAVE * 4) {
      const float4 wc = *reinterpret_cast<const float4*>(w + c);
#pragma unroll
      for (int i = 0; i < ROUTE_TOK; ++i)
        if (i < nt) {
          const T* x = h + (size_t)(t0 + i) * h_stride + c;
          acc[i] = fmaf(to_f(x[0]), wc.x, acc[i]), acc[i] = fmaf(to_f(x[1]), wc.y, acc[i]);
          acc[i] = fmaf(to_f(x[2]), wc.z, acc[i]), acc[i] = fmaf(to_f(x[3]), wc.w, acc[i]);
        }
    }
  } else {
    for (int c = lane; c < W; c += NS_WAVE) {
      const float wc = w[c];
#pragma unroll
      for (int i = 0; i < ROUTE_TOK; ++i)
        if (i < nt) acc[i] = fmaf(to_f(h[(size_t)(t0 + i) * h_stride + c]), wc, acc[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < ROUTE_TOK; ++i) {
    const float v = wave_sum(acc[i]);
    if (lane == 0 && i < nt) z[(size_t)(t0 + i) * experts + e] = v + (br ? br[e] : 0.f);
  }
}

// The same logits for many tokens, on the 32-bit matrix instruction (v_mfma_f32_16x16x4_f32: 32-bit products and sums): a workgroup takes 16
// tokens and up to 32 rows of the router, its eight waves every eighth piece of 16 columns, and adds the waves' sums in a fixed order; a
// token's logits do not depend on the tokens beside it.  Lane l holds columns 4 (l / 16) .. + 3 of row (token) l % 16 of an operand, one
// load for four instructions, four pieces on their way.  The kernel above is bound by its reads of the tokens (every four experts read them
// anew) and by the exchange that adds 64 lanes' sums; this one by the latency of a wave's rounds.  33 rows of 2,048, with the choice behind:
// 2,048 tokens 37.5 -> 19.9 us, 508 tokens 18.7 -> 18.5 (four waves 22.7 and 21.7).
// The logits decide which experts run, so no 32-bit chain is longer than 8 columns (two instructions), and the chains are added in 64 bits.
// Relative error (2-norm, against 64 bits) at 2,048 columns 5.9e-8, of the kernel above 1.2e-7, with one chain a wave 4.0e-7; it is below
// the other's down to 64 columns, from where on the launch takes this kernel.  W a multiple of 16.
// SETS of 16 rows of the router a workgroup: its 64-bit sums take as long as its matrix instructions, so a single set is ahead while the compute units have no more than a
// workgroup each: with the choice behind, alone, two sets and one: 32 rows of 2,048, 508 tokens 24.2 and 20.3 us, 36 rows 23.8 and 20.6, 64 rows of 4,096 35.7 and 28.4; level or
// behind beyond (64 rows of 4,096, 2,048 tokens 36.4 and 42.3).  The sums are the same.
#define MOE_LOGIT_WAVES 8
#define MOE_UNITS 256  // compute units
template <typename T, int SETS>
__global__ __launch_bounds__(NS_WAVE * MOE_LOGIT_WAVES) void moe_logits_many_kernel(const T* __restrict__ h, int h_stride, const float* __restrict__ wr,
                                                              const float* __restrict__ br, float* __restrict__ z, int n, int W, int experts) {
  constexpr int STEP = 16 * MOE_LOGIT_WAVES;  // columns from one piece of a wave to the next
  __shared__ double part[MOE_LOGIT_WAVES][SETS][16][17];  // [wave][16 rows of the router][token][row]
  const int lane = threadIdx.x % NS_WAVE, wave = threadIdx.x / NS_WAVE, r = lane % 16, g = lane / 16;
  const int t0 = blockIdx.x * 16, e0 = blockIdx.y * 16 * SETS;
  const T* x = h + (size_t)min(t0 + r, n - 1) * h_stride + 4 * g;
  const float* w[SETS];
#pragma unroll
  for (int i = 0; i < SETS; ++i) w[i] = wr + (size_t)min(e0 + 16 * i + r, experts - 1) * W + 4 * g;
  typedef T t4 __attribute__((ext_vector_type(4)));
  double sum[SETS][4] = {};
  for (int c = 16 * wave; c < W; c += 4 * STEP) {
    t4 xv[4];
    f32x4 wv[4][SETS];
#pragma unroll
    for (int s = 0; s < 4; ++s) {  // (a piece beyond the row is read at its start and not used)
      const int at = c + STEP * s < W ? c + STEP * s : 0;
      xv[s] = *reinterpret_cast<const t4*>(x + at);
#pragma unroll
      for (int i = 0; i < SETS; ++i) wv[s][i] = *reinterpret_cast<const f32x4*>(w[i] + at);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if (c + STEP * s >= W) break;
      f32x4 acc[2][SETS];
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int i = 0; i < SETS; ++i)
          acc[k / 2][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[s][i][k], to_f((T)xv[s][k]), k % 2 ? acc[k / 2][i] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < SETS; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) sum[i][k] += (double)acc[0][i][k] + (double)acc[1][i][k];
    }
  }
#pragma unroll
  for (int i = 0; i < SETS; ++i)
#pragma unroll
    for (int k = 0; k < 4; ++k) part[wave][i][r][4 * g + k] = sum[i][k];
  __syncthreads();
  for (int i = threadIdx.x; i < 256 * SETS; i += NS_WAVE * MOE_LOGIT_WAVES) {
    const int t = i / (16 * SETS), e = i % (16 * SETS);
    if (t0 + t >= n || e0 + e >= experts) continue;
    double v = br ? (double)br[e0 + e] : 0.;
#pragma unroll
    for (int j = 0; j < MOE_LOGIT_WAVES; ++j) v += part[j][e / 16][t][e % 16];
    z[(size_t)(t0 + t) * experts + e0 + e] = (float)v;
  }
}

// The same logits for a step of few tokens (up to ROUTE_TOK): a workgroup an expert, its four waves a quarter of the row each
// (a wave alone walks a row of 2,048 columns in eight dependent rounds; four waves in two), their sums joined in LDS in a
// fixed order.  A token's logit does not depend on how many tokens the step holds.
template <typename T>
__global__ __launch_bounds__(256) void moe_logits_few_kernel(const T* __restrict__ h, int h_stride, const float* __restrict__ wr,
                                                             const float* __restrict__ br, float* __restrict__ z, int n, int W, int experts, int vec) {
  __shared__ float part[4][ROUTE_TOK];
  const int e = blockIdx.x, lane = threadIdx.x % NS_WAVE, wave = threadIdx.x / NS_WAVE;
  const float* w = wr + (size_t)e * W;
  float acc[ROUTE_TOK];
#pragma unroll
  for (int i = 0; i < ROUTE_TOK; ++i) acc[i] = 0.f;
  if (vec) {
    for (int c = threadIdx.x * 4; c < W; c += 256 * 4) {
      const float4 wc = *reinterpret_cast<const float4*>(w + c);
#pragma unroll
      for (int i = 0; i < ROUTE_TOK; ++i)
        if (i < n) {
          const T* x = h + (size_t)i * h_stride + c;
          acc[i] = fmaf(to_f(x[0]), wc.x, acc[i]), acc[i] = fmaf(to_f(x[1]), wc.y, acc[i]);
          acc[i] = fmaf(to_f(x[2]), wc.z, acc[i]), acc[i] = fmaf(to_f(x[3]), wc.w, acc[i]);
        }
    }
  } else {
    for (int c = threadIdx.x; c < W; c += 256) {
      const float wc = w[c];
#pragma unroll
      for (int i = 0; i < ROUTE_TOK; ++i)
        if (i < n) acc[i] = fmaf(to_f(h[(size_t)i * h_stride + c]), wc, acc[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < ROUTE_TOK; ++i) {
    const float v = wave_sum(acc[i]);
    if (lane == 0) part[wave][i] = v;
  }
  __syncthreads();
  if (threadIdx.x < n) {
    const int i = threadIdx.x;
    z[(size_t)i * experts + e] = ((part[0][i] + part[1][i]) + (part[2][i] + part[3][i])) + (br ? br[e] : 0.f);
  }
}

// A wave a token: the choice scores in LDS, every lane looks through its share for the largest one not yet taken, the lanes'
// candidates meet by lane exchange (the larger value wins, the lower index among equals; what is no number counts as
// minus infinity, so a row of anything still chooses ``top`` different experts).
// ``score`` = MOE_CHOSEN_SOFTMAX: the choice goes by the logits and the weights are the soft-max over the chosen logits.
// ``score`` = MOE_SIGMOID: scores s = sigmoid(z); the choice goes by s + correction[e] (``correction`` may be null) and the
// weights are the chosen experts' s, not renormalized.
// ``score`` = MOE_SOFTMAX: scores s = soft-max over all logits; the choice goes by s + correction[e], the weights are the chosen
// s over the sum of the chosen s (+ 1e-20).
// All weights are then multiplied by ``scale``.  ``groups`` > 1: the experts form that many equal groups of neighbours; a
// group's score is the sum of its ``group_best`` (1 or 2) largest choice scores (of its one, if it has one), and only the
// ``keep`` best groups' experts can be chosen: the others never enter the comparison, whatever their scores' sign.
#define MOE_CHOSEN_SOFTMAX 0
#define MOE_SIGMOID 1
#define MOE_SOFTMAX 2
__device__ __forceinline__ void wave_best(float& bv, int& best) {
#pragma unroll
  for (int o = NS_WAVE / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(bv, o, NS_WAVE);
    const int oi = __shfl_xor(best, o, NS_WAVE);
    if (oi >= 0 && (best < 0 || ov > bv || (ov == bv && oi < best))) best = oi, bv = ov;
  }
}

__global__ __launch_bounds__(64) void moe_choose_kernel(const float* __restrict__ z, int z_stride, int* __restrict__ sel, float* __restrict__ wt,
                                                        int n, int experts, int top, int score, const float* __restrict__ correction, int groups,
                                                        int keep, int group_best, float scale) {
  __shared__ float zs[MOE_MAX_EXPERTS];   // choice scores
  __shared__ float ws[MOE_MAX_EXPERTS];   // what the weights are made from: the logits, or the sigmoid scores
  __shared__ float gs[MOE_MAX_EXPERTS];   // group scores
  __shared__ unsigned char taken[MOE_MAX_EXPERTS];
  __shared__ unsigned char gkept[MOE_MAX_EXPERTS];
  const int t = blockIdx.x, lane = threadIdx.x;
  float zmax = -INFINITY, zsum = 0.f;  // of the soft-max over all logits
  if (score == MOE_SOFTMAX) {
    for (int e = lane; e < experts; e += NS_WAVE) zmax = fmaxf(zmax, z[(size_t)t * z_stride + e]);
    zmax = wave_max(zmax);
    for (int e = lane; e < experts; e += NS_WAVE) zsum += expf(z[(size_t)t * z_stride + e] - zmax);
    zsum = wave_sum(zsum);
  }
  for (int e = lane; e < experts; e += NS_WAVE) {
    float v = z[(size_t)t * z_stride + e];
    if (score == MOE_SIGMOID) v = 1.f / (1.f + expf(-v));
    else if (score == MOE_SOFTMAX) v = expf(v - zmax) / zsum;
    ws[e] = v;
    if (correction) v += correction[e];
    zs[e] = v == v ? v : -INFINITY;
    taken[e] = 0;
  }
  __syncthreads();
  if (groups > 1) {
    const int per = experts / groups;
    for (int g = lane; g < groups; g += NS_WAVE) {
      float a = -INFINITY, b = -INFINITY;  // the two largest of the group
      for (int e = g * per; e < (g + 1) * per; ++e) {
        const float v = zs[e];
        if (v > a) b = a, a = v;
        else if (v > b) b = v;
      }
      const float v = per > 1 && group_best > 1 ? a + b : a;
      gs[g] = v == v ? v : -INFINITY;  // (what is no number, an expert's score or a group's, counts as the lowest: it would stop the exchange below)
      gkept[g] = 0;
    }
    __syncthreads();
    for (int k = 0; k < keep; ++k) {
      int best = -1;
      float bv = -INFINITY;
      for (int g = lane; g < groups; g += NS_WAVE)
        if (!gkept[g] && (best < 0 || gs[g] > bv)) best = g, bv = gs[g];
      wave_best(bv, best);
      if (lane == 0) gkept[best] = 1;
      __syncthreads();
    }
    for (int e = lane; e < experts; e += NS_WAVE)
      if (!gkept[e / per]) taken[e] = 1;
    __syncthreads();
  }
  float largest = 0.f, sum = 0.f, mine = 0.f;  // lane k keeps the k-th chosen value
  int mine_idx = 0;
  for (int k = 0; k < top; ++k) {
    int best = -1;
    float bv = -INFINITY;
    for (int e = lane; e < experts; e += NS_WAVE)
      if (!taken[e] && (best < 0 || zs[e] > bv)) best = e, bv = zs[e];
    wave_best(bv, best);
    if (lane == 0) taken[best] = 1;
    float w;
    if (score != MOE_CHOSEN_SOFTMAX) {
      w = ws[best];
    } else {
      if (k == 0) largest = bv;
      w = expf(bv - largest);
    }
    sum += w;
    if (lane == k % NS_WAVE && k < NS_WAVE) mine = w, mine_idx = best;
    __syncthreads();
  }
  if (lane < top) {
    sel[(size_t)t * top + lane] = mine_idx;
    wt[(size_t)t * top + lane] = (score == MOE_SIGMOID ? mine : mine / (score == MOE_SOFTMAX ? sum + 1e-20f : sum)) * scale;
  }
}

// The same choice among up to 64 experts, a lane an expert and four tokens a workgroup: a lane's rank is the number of allowed lanes in front of it,
// counted in one walk over the lanes by scalar reads, so nothing is exchanged through LDS and no turn waits for the one before.
// Bound by the chain of exchanges in the kernel above (a turn an expert to choose, six exchanges each).  The weights are the same, bit by
// bit.  Logits and choice, width 2,048, four chosen of 32: 8 tokens in groups 14.1 -> 11.8 us, 2,048 tokens 18.8 -> 16.5; of 36 in groups, 508 tokens 20.7 -> 19.3.
__device__ __forceinline__ float lane_read(float v, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane)); }

struct MoeChoice {
  int experts, top, score;
  const float* correction;
  int groups, keep, group_best;
  float scale;
};

// a wave's choice for token t, whose logits its lanes hold (``w``)
__device__ __forceinline__ void moe_choose_lanes(float w, size_t t, int* __restrict__ sel, float* __restrict__ wt, const MoeChoice& p) {
  const int lane = threadIdx.x % NS_WAVE, experts = p.experts, top = p.top, score = p.score, groups = p.groups, keep = p.keep, group_best = p.group_best;
  const float* __restrict__ correction = p.correction;
  const float scale = p.scale;
  const bool mine = lane < experts;
  w = mine ? w : -INFINITY;  // what the weights are made from: the logits, or the scores
  if (score == MOE_SOFTMAX) {
    const float zmax = wave_max(fmaxf(-INFINITY, w));
    const float e = expf(w - zmax);
    w = e / wave_sum(mine ? e : 0.f);
  } else if (score == MOE_SIGMOID) {
    w = 1.f / (1.f + expf(-w));
  }
  float c = correction && mine ? w + correction[lane] : w;  // what the choice goes by
  c = c == c ? c : -INFINITY;
  unsigned long long allowed = __ballot(mine);
  if (groups > 1) {
    const int per = experts / groups, group = lane / per;
    float a = -INFINITY, b = -INFINITY;  // the two largest of this lane's group
    for (int j = 0; j < experts; ++j) {
      const float v = lane_read(c, j);
      if (j / per != group) continue;
      if (v > a) b = a, a = v;
      else if (v > b) b = v;
    }
    float gs = per > 1 && group_best > 1 ? a + b : a;
    gs = gs == gs ? gs : -INFINITY;
    int before = 0;
    for (int g = 0; g < groups; ++g) {
      const float v = lane_read(gs, g * per);
      before += v > gs || (v == gs && g < group);
    }
    allowed = __ballot(mine && before < keep);
  }
  int rank = 0;
  for (unsigned long long m = allowed; m; m &= m - 1) {
    const int j = __ffsll(m) - 1;
    const float v = lane_read(c, j);
    rank += v > c || (v == c && j < lane);
  }
  const bool in = (allowed >> lane) & 1;
  if (score == MOE_CHOSEN_SOFTMAX) w = expf(c - lane_read(c, __ffsll(__ballot(in && rank == 0)) - 1));
  float sum = 0.f;
  for (int k = 0; k < top; ++k) sum += lane_read(w, __ffsll(__ballot(in && rank == k)) - 1);
  if (in && rank < top) {
    sel[(size_t)t * top + rank] = lane;
    wt[(size_t)t * top + rank] = (score == MOE_SIGMOID ? w : w / (score == MOE_SOFTMAX ? sum + 1e-20f : sum)) * scale;
  }
}

__global__ __launch_bounds__(256) void moe_choose_lanes_kernel(const float* __restrict__ z, int z_stride, int* __restrict__ sel, float* __restrict__ wt,
                                                               int n, const MoeChoice p) {
  const int t = blockIdx.x * 4 + threadIdx.x / NS_WAVE, lane = threadIdx.x % NS_WAVE;
  if (t >= n) return;
  moe_choose_lanes(lane < p.experts ? z[(size_t)t * z_stride + lane] : 0.f, t, sel, wt, p);
}

// Logits and choice of a step of few tokens in one launch: a workgroup a token, its four teams of four waves every fourth row of the router, four rows at a time; the
// first wave chooses by lanes.  Every workgroup reads the whole router (from L2 but for the first), so it has to be small; what is saved is a launch and a trip of the
// logits through memory in a chain of dependent kernels.  A logit's sum is ordered as in moe_logits_few_kernel, whose results these are bit by bit.
// us in two launches and in one: 8 tokens, width 2,048, four of 32 8.5 and 7.0, in 8 groups of which 4 are kept 11.2 and 9.7; 2 tokens, 4,096, two of 16 6.9 and 5.7; a larger router
// is more than a compute unit reads in that time: 8 of 4,096, 32 experts 10.4 and 10.5; 36 of 2,048 11.1 and 11.5 (a third round); 64 of 2,048 10.1 and 12.8.
#define MOE_ROUTE_FEW_ROWS 32
#define MOE_ROUTE_FEW_BYTES (256 << 10)
template <typename T>
__global__ __launch_bounds__(1024) void moe_route_few_kernel(const T* __restrict__ h, int h_stride, const float* __restrict__ wr, const float* __restrict__ br,
                                                             float* __restrict__ z, int* __restrict__ sel, float* __restrict__ wt, int W, int rows,
                                                             const MoeChoice p) {
  constexpr int TEAMS = 4, AT_ONCE = 4;
  __shared__ float part[4][MOE_ROUTE_FEW_ROWS], zs[MOE_ROUTE_FEW_ROWS];
  const size_t t = blockIdx.x;
  const int team = threadIdx.x / 256, tid = threadIdx.x % 256, lane = threadIdx.x % NS_WAVE, wave = tid / NS_WAVE;
  const T* x = h + t * h_stride;
  typedef T t4 __attribute__((ext_vector_type(4)));
  for (int e0 = team; e0 < rows; e0 += TEAMS * AT_ONCE) {
    float acc[AT_ONCE];
#pragma unroll
    for (int k = 0; k < AT_ONCE; ++k) acc[k] = 0.f;
    for (int c = tid * 4; c < W; c += 256 * 4) {
      const t4 xc = *reinterpret_cast<const t4*>(x + c);
      float4 wc[AT_ONCE];
#pragma unroll
      for (int k = 0; k < AT_ONCE; ++k) wc[k] = *reinterpret_cast<const float4*>(wr + (size_t)min(e0 + TEAMS * k, rows - 1) * W + c);
#pragma unroll
      for (int k = 0; k < AT_ONCE; ++k) {
        acc[k] = fmaf(to_f((T)xc[0]), wc[k].x, acc[k]), acc[k] = fmaf(to_f((T)xc[1]), wc[k].y, acc[k]);
        acc[k] = fmaf(to_f((T)xc[2]), wc[k].z, acc[k]), acc[k] = fmaf(to_f((T)xc[3]), wc[k].w, acc[k]);
      }
    }
#pragma unroll
    for (int k = 0; k < AT_ONCE; ++k) {
      const float v = wave_sum(acc[k]);
      if (lane == 0 && e0 + TEAMS * k < rows) part[wave][e0 + TEAMS * k] = v;
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < rows) {
    const int e = threadIdx.x;
    const float v = ((part[0][e] + part[1][e]) + (part[2][e] + part[3][e])) + (br ? br[e] : 0.f);
    zs[e] = v, z[t * rows + e] = v;
  }
  __syncthreads();
  if (threadIdx.x < NS_WAVE) moe_choose_lanes(lane < rows ? zs[lane] : 0.f, t, sel, wt, p);
}

// Which of the two (the results are the same), by what each takes, in steps of a walk over the experts (35 ns a token's chain, 110 ns of 8,192 tokens):
// by lanes one walk, three where experts are chosen in groups; by turns 20 an expert to choose, 10 a group to keep and 2.5 an expert of a
// group; with the GPU full of tokens 27 and 18, and the turns' workgroups of one wave cost 28 to 32 more.  us by turns and by lanes, with the
// logits, 64 tokens: 64 experts, one chosen 15.6 and 17.1, 8 chosen 20.5 and 17.3; 32 experts, one chosen 15.6 and 15.9, two 0.4 less by lanes;
// 64 in 8 groups of which 4 are kept, two chosen 2.4 more by lanes, 8 chosen 1.6 less; 64 in 2 groups, one kept, 8 chosen 24.4 and 22.6; 32 in 8,
// 4 kept, 4 chosen 2.4 less.  8,192 tokens: 64 in 8 groups, 4 kept, 4 chosen 5.3 less by lanes, one chosen 3.8 more.
static bool moe_choose_by_lanes(int n, int experts, int top, int groups, int keep) {
  if (experts > NS_WAVE) return false;
  const bool full = n >= 4096;
  if (groups == 1) return experts - (full ? 28 : 4) <= (full ? 27 : 20) * top;
  return 3 * experts - (full ? 52 : 20) <= (full ? 27 : 20) * top + (full ? 18 : 10) * keep + 5 * (experts / groups) / 2;
}

// ``z``: float32 [n][experts + extra]; ``extra``: rows of ``wr`` (and ``br``) below the experts'
extern "C" int ns_moe_route(const void* h, int h_stride, const float* wr, const float* br, float* z, int* sel, float* wt, int n, int W, int experts,
                            int extra, int top, int score, const float* correction, int groups, int keep, int group_best, float scale, int dtype,
                            hipStream_t stream) {
  if (n <= 0 || W <= 0 || experts <= 0 || experts > MOE_MAX_EXPERTS || top <= 0 || top > MOE_MAX_TOP || top > experts) return NS_ERR_BAD_ARG;
  if (extra < 0 || score < MOE_CHOSEN_SOFTMAX || score > MOE_SOFTMAX || (correction && score == MOE_CHOSEN_SOFTMAX) || group_best < 1 || group_best > 2)
    return NS_ERR_BAD_ARG;
  const int rows = experts + extra;
  if (groups < 1 || experts % groups || keep < 1 || keep > groups || top > keep * (experts / groups)) return NS_ERR_BAD_ARG;
  dim3 grid((n + ROUTE_TOK - 1) / ROUTE_TOK, (rows + 3) / 4);
  if (grid.y > 65535) return NS_ERR_UNSUPPORTED;
  const size_t elem = dtype == NS_DTYPE_F32 ? 4 : 2;
  const int vec = W % 4 == 0 && h_stride % 4 == 0 && (uintptr_t)wr % 16 == 0 && (uintptr_t)h % (4 * elem) == 0;
  if (dtype != NS_DTYPE_F32 && dtype != NS_DTYPE_BF16) return NS_ERR_UNSUPPORTED;
  const bool by_lanes = moe_choose_by_lanes(n, experts, top, groups, keep);
  const MoeChoice choice{experts, top, score, correction, groups, keep, group_best, scale};
  if (n <= ROUTE_TOK && vec && by_lanes && rows <= MOE_ROUTE_FEW_ROWS && (size_t)rows * W * sizeof(float) <= MOE_ROUTE_FEW_BYTES) {
    if (dtype == NS_DTYPE_F32)
      moe_route_few_kernel<float><<<n, 1024, 0, stream>>>((const float*)h, h_stride, wr, br, z, sel, wt, W, rows, choice);
    else
      moe_route_few_kernel<bf16_t><<<n, 1024, 0, stream>>>((const bf16_t*)h, h_stride, wr, br, z, sel, wt, W, rows, choice);
    return ns_launch_status();
  }
  if (n <= ROUTE_TOK) {  // few tokens: a workgroup an expert
    if (dtype == NS_DTYPE_F32)
      moe_logits_few_kernel<float><<<rows, 256, 0, stream>>>((const float*)h, h_stride, wr, br, z, n, W, rows, vec);
    else
      moe_logits_few_kernel<bf16_t><<<rows, 256, 0, stream>>>((const bf16_t*)h, h_stride, wr, br, z, n, W, rows, vec);
  } else if (vec && W % 16 == 0 && W >= 64) {
    // (sets of 16 rows of the router a workgroup: one where a compute unit then still has no more than one workgroup, MOE_UNITS of them)
    const long one = (long)((n + 15) / 16) * ((rows + 15) / 16);
    const bool single = one <= MOE_UNITS;
    const dim3 many((n + 15) / 16, single ? (rows + 15) / 16 : (rows + 31) / 32);
    if (dtype == NS_DTYPE_F32) {
      if (single) moe_logits_many_kernel<float, 1><<<many, NS_WAVE * MOE_LOGIT_WAVES, 0, stream>>>((const float*)h, h_stride, wr, br, z, n, W, rows);
      else moe_logits_many_kernel<float, 2><<<many, NS_WAVE * MOE_LOGIT_WAVES, 0, stream>>>((const float*)h, h_stride, wr, br, z, n, W, rows);
    } else {
      if (single) moe_logits_many_kernel<bf16_t, 1><<<many, NS_WAVE * MOE_LOGIT_WAVES, 0, stream>>>((const bf16_t*)h, h_stride, wr, br, z, n, W, rows);
      else moe_logits_many_kernel<bf16_t, 2><<<many, NS_WAVE * MOE_LOGIT_WAVES, 0, stream>>>((const bf16_t*)h, h_stride, wr, br, z, n, W, rows);
    }
  } else if (dtype == NS_DTYPE_F32)
    moe_logits_kernel<float><<<grid, 256, 0, stream>>>((const float*)h, h_stride, wr, br, z, n, W, rows, vec);
  else
    moe_logits_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)h, h_stride, wr, br, z, n, W, rows, vec);
  if (by_lanes)
    moe_choose_lanes_kernel<<<(n + 3) / 4, 256, 0, stream>>>(z, rows, sel, wt, n, choice);
  else
    moe_choose_kernel<<<n, 64, 0, stream>>>(z, rows, sel, wt, n, experts, top, score, correction, groups, keep, group_best, scale);
  return ns_launch_status();
}

__device__ __forceinline__ float clipped_glu(float g, float u, float limit, float alpha, float shift) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g / (1.f + expf(-alpha * g)) * (u + shift);
}

// ------------------------------------------------------------------------------------------------ few rows
// Steps of few rows stream the chosen experts' matrices, each exactly once per (token, expert) that chose it, cut into
// slices so that the launch fills the chip:
//   first:  grid (slices of inner channels, top, tokens): the token's row in LDS, a wave an inner channel in turn (its gate row,
//           if the expert has one, and its up row together, 16 bytes a lane a load); act [tokens][top][ff] in 32-bit, rounded as a store in the
//           model's precision would round it
//   second: grid (slices of output channels, top, tokens): the activations in LDS, a wave an output channel in turn;
//           out [tokens][top][W] in 32-bit, already times the router's weight
template <typename T> struct Row8;
template <> struct Row8<float> {
  static __device__ __forceinline__ void load(const float* p, float* out) {
    const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
    out[0] = a.x, out[1] = a.y, out[2] = a.z, out[3] = a.w, out[4] = b.x, out[5] = b.y, out[6] = b.z, out[7] = b.w;
  }
};
template <> struct Row8<bf16_t> {
  static __device__ __forceinline__ void load(const bf16_t* p, float* out) {
    typedef bf16_t v8 __attribute__((ext_vector_type(8)));
    const v8 a = __builtin_nontemporal_load(reinterpret_cast<const v8*>(p));
#pragma unroll
    for (int j = 0; j < 8; ++j) out[j] = (float)a[j];
  }
};

// sum_c w[c] x[c] over a wave; ``vec``: K is a multiple of 8 and the row starts at a multiple of 8 elements of an aligned base
template <typename T>
__device__ __forceinline__ float row_dot(const T* __restrict__ w, const float* __restrict__ x, int K, int lane, bool vec) {
  float acc = 0.f;
  if (vec) {
    for (int c = lane * 8; c < K; c += NS_WAVE * 8) {
      float v[8];
      Row8<T>::load(w + c, v);
      const float4 x0 = *reinterpret_cast<const float4*>(x + c), x1 = *reinterpret_cast<const float4*>(x + c + 4);
      acc = fmaf(v[0], x0.x, acc), acc = fmaf(v[1], x0.y, acc), acc = fmaf(v[2], x0.z, acc), acc = fmaf(v[3], x0.w, acc);
      acc = fmaf(v[4], x1.x, acc), acc = fmaf(v[5], x1.y, acc), acc = fmaf(v[6], x1.z, acc), acc = fmaf(v[7], x1.w, acc);
    }
  } else {
    for (int c = lane; c < K; c += NS_WAVE) acc = fmaf(to_f(w[c]), x[c], acc);
  }
  return wave_sum(acc);
}

template <typename T>
__global__ __launch_bounds__(256) void moe_rows_up_kernel(const T* __restrict__ h, int h_stride, const T* __restrict__ wg, const T* __restrict__ wu,
                                                          const int* __restrict__ sel, float* __restrict__ act, int W, int ff, int experts, int top, int per,
                                                          float limit, float alpha, float shift, int act_kind, int vec) {
  extern __shared__ __attribute__((aligned(16))) float moe_lds[];  // [W]
  const int t = blockIdx.z, k = blockIdx.y, lane = threadIdx.x % NS_WAVE, wave = threadIdx.x / NS_WAVE, waves = blockDim.x / NS_WAVE;
  const int e = sel[(size_t)t * top + k];
  if (e >= experts) return;  // an identity expert
  for (int c = threadIdx.x; c < W; c += blockDim.x) moe_lds[c] = to_f(h[(size_t)t * h_stride + c]);
  __syncthreads();
  const int f0 = blockIdx.x * per, f1 = min(ff, f0 + per);
  for (int f = f0 + wave; f < f1; f += waves) {
    const size_t row = ((size_t)e * ff + f) * W;
    const float g = wg ? row_dot(wg + row, moe_lds, W, lane, vec) : 0.f, u = row_dot(wu + row, moe_lds, W, lane, vec);
    if (lane == 0)
      act[((size_t)t * top + k) * ff + f] =
          round_to<T>(wg ? clipped_glu(round_to<T>(g), round_to<T>(u), limit, alpha, shift) : activation_of(round_to<T>(u), act_kind));
  }
}

template <typename T>
__global__ __launch_bounds__(256) void moe_rows_down_kernel(const float* __restrict__ act, const T* __restrict__ wd, const int* __restrict__ sel,
                                                            const float* __restrict__ wt, float* __restrict__ out, int W, int ff, int experts, int top,
                                                            int per, int vec) {
  extern __shared__ __attribute__((aligned(16))) float moe_lds[];  // [ff]
  const int t = blockIdx.z, k = blockIdx.y, lane = threadIdx.x % NS_WAVE, wave = threadIdx.x / NS_WAVE, waves = blockDim.x / NS_WAVE;
  const int e = sel[(size_t)t * top + k];
  if (e >= experts) return;
  const float share = wt[(size_t)t * top + k];
  for (int f = threadIdx.x; f < ff; f += blockDim.x) moe_lds[f] = act[((size_t)t * top + k) * ff + f];
  __syncthreads();
  const int c0 = blockIdx.x * per, c1 = min(W, c0 + per);
  for (int c = c0 + wave; c < c1; c += waves) {
    const float y = row_dot(wd + ((size_t)e * W + c) * ff, moe_lds, ff, lane, vec);
    if (lane == 0) out[((size_t)t * top + k) * W + c] = share * y;
  }
}

// channels a workgroup takes so that the launch has about 2048 workgroups, a multiple of the four waves
static int moe_slice(int channels, int rows) {
  int per = (int)(((long long)channels * rows + 2047) / 2048);
  per = (per + 3) / 4 * 4;
  return per < 4 ? 4 : per;
}

extern "C" int ns_moe_expert_rows(const void* h, int h_stride, const void* wg, const void* wu, const void* wd, const int* sel, const float* wt,
                                  float* act, float* out, int n, int W, int ff, int top, int experts, float limit, float alpha, float shift,
                                  int act_kind, int dtype, hipStream_t stream) {
  if (!wg && (act_kind < 0 || act_kind >= NS_ACTIVATIONS)) return NS_ERR_BAD_ARG;
  if (n <= 0 || n > 65535 || W <= 0 || ff <= 0 || top <= 0 || top > 65535 || experts <= 0) return NS_ERR_BAD_ARG;
  if ((size_t)W * sizeof(float) > 64 * 1024 || (size_t)ff * sizeof(float) > 64 * 1024) return NS_ERR_UNSUPPORTED;
  const size_t elem = dtype == NS_DTYPE_F32 ? 4 : 2;
  const int vec_up = W % 8 == 0 && (uintptr_t)wg % (8 * elem) == 0 && (uintptr_t)wu % (8 * elem) == 0;
  const int vec_down = ff % 8 == 0 && (uintptr_t)wd % (8 * elem) == 0;
  const int per_f = moe_slice(ff, n * top), per_c = moe_slice(W, n * top);
  dim3 g1((ff + per_f - 1) / per_f, top, n), g2((W + per_c - 1) / per_c, top, n);
  if (dtype == NS_DTYPE_F32) {
    moe_rows_up_kernel<float><<<g1, 256, W * sizeof(float), stream>>>((const float*)h, h_stride, (const float*)wg, (const float*)wu, sel, act, W, ff,
                                                                       experts, top, per_f, limit, alpha, shift, act_kind, vec_up);
    moe_rows_down_kernel<float><<<g2, 256, ff * sizeof(float), stream>>>(act, (const float*)wd, sel, wt, out, W, ff, experts, top, per_c, vec_down);
  } else if (dtype == NS_DTYPE_BF16) {
    moe_rows_up_kernel<bf16_t><<<g1, 256, W * sizeof(float), stream>>>((const bf16_t*)h, h_stride, (const bf16_t*)wg, (const bf16_t*)wu, sel, act, W,
                                                                        ff, experts, top, per_f, limit, alpha, shift, act_kind, vec_up);
    moe_rows_down_kernel<bf16_t><<<g2, 256, ff * sizeof(float), stream>>>(act, (const bf16_t*)wd, sel, wt, out, W, ff, experts, top, per_c, vec_down);
  } else {
    return NS_ERR_UNSUPPORTED;
  }
  return ns_launch_status();
}

// ------------------------------------------------------------------------------------------------ many rows
// Steps of many rows (bfloat16): the (token, chosen expert) pairs are sorted by expert on the device, and every expert's
// pairs are cut into even tiles of at most 128 rows (16 where the experts see few; ``moe_tile_cap``), which are multiplied on the matrix
// cores (v_mfma_f32_16x16x32_bf16).  The host never learns which experts were chosen: the launch has as many tiles as any
// choice can need (pairs / cap + experts), and workgroups beyond the tiles in use return.
//   first:  rows gathered from h by the sorted pairs; gate (if there is one: DUAL) and up matrices in the same pass; act [pairs
//           sorted][ff] in bfloat16
//   second: act times the down matrix; out [tokens][top][W] in 32-bit, each row back at its pair and times its weight

#define MG_ROWS 128                                 // rows of a tile at most
// By 256 rows of the matrices: one workgroup a compute unit; and by 128: two, with more stages on their way where half of the rows are enough (the matrices come
// from memory then: 8 experts of 4,096, two a token, with gates, 8 tokens three stages instead of two 83 -> 77 us).
// TURN: the stage of K that a workgroup begins with, block by block of channels (see moe_tile_kernel).
struct MoeTile {
  static constexpr int BN = 256, HALF_STAGES = 2, TURN = 0;
  static constexpr bool W_ONCE = false;
};
struct MoeFewTile {
  static constexpr int BN = 128, HALF_STAGES = 3, TURN = 7;
  static constexpr bool W_ONCE = true;
};
#define MG_GROUP 4                                  // blocks of channels that an expert's tiles take together

// What a tile is, in three words, from which a workgroup works out any tile of the same expert without another trip to memory: ``tile_e`` the expert
// and which of its tiles this is (-1: no tile), ``tile_r0`` the expert's first sorted row, ``tile_rows`` the expert's rows.
#define MG_E_BITS 10
static_assert(MOE_MAX_EXPERTS <= 1 << MG_E_BITS, "2^24 pairs in tiles of 16: an expert has 2^20 tiles at most");
__device__ __forceinline__ int tile_expert(int word) { return word & ((1 << MG_E_BITS) - 1); }

// rows before tile ``i`` of ``t`` even tiles of ``c`` rows (whole blocks of 16; c itself for i = t)
__device__ __forceinline__ int rows_before_tile(int c, int t, int i) {
  if (t == 1) return i ? c : 0;
  const int blocks = (c + 15) / 16;
  return min(c, 16 * (i * (blocks / t) + min(i, blocks % t)));
}

// Pairs sorted by expert and every expert's pairs cut into the fewest tiles of at most ``cap`` rows, as even as whole blocks of
// 16 rows allow (an expert with a few rows more than ``cap`` makes two tiles of about half, not a full one and a sliver).  The counts
// are taken and the places dealt with LDS atomics by all threads; the experts' places come from a scan over the lanes.
__global__ __launch_bounds__(1024) void moe_sort_kernel(const int* __restrict__ sel, int pairs, int experts, int cap, int* __restrict__ perm,
                                                        int* __restrict__ tile_e, int* __restrict__ tile_r0, int* __restrict__ tile_rows,
                                                        int max_tiles) {
  __shared__ int cnt[MOE_MAX_EXPERTS], cur[MOE_MAX_EXPERTS], tiles_of[MOE_MAX_EXPERTS], used;
  for (int e = threadIdx.x; e < experts; e += blockDim.x) cnt[e] = 0;
  __syncthreads();
  for (int p = threadIdx.x; p < pairs; p += blockDim.x) {
    const int e = sel[p];
    if (e < experts) atomicAdd(&cnt[e], 1);  // (pairs of identity experts have no place)
  }
  __syncthreads();
  if (threadIdx.x < NS_WAVE) {  // first places and first tiles: a scan over 64 experts at a time
    int rows_before = 0, tiles_before = 0;
    for (int e0 = 0; e0 < experts; e0 += NS_WAVE) {
      const int e = e0 + threadIdx.x, c = e < experts ? cnt[e] : 0, t = (c + cap - 1) / cap;
      int rows = c, tiles = t;
#pragma unroll
      for (int o = 1; o < NS_WAVE; o <<= 1) {
        const int r = __shfl_up(rows, o, NS_WAVE), u = __shfl_up(tiles, o, NS_WAVE);
        if ((int)threadIdx.x >= o) rows += r, tiles += u;
      }
      if (e < experts) cur[e] = rows_before + rows - c, tiles_of[e] = tiles_before + tiles - t;
      rows_before += __shfl(rows, NS_WAVE - 1, NS_WAVE), tiles_before += __shfl(tiles, NS_WAVE - 1, NS_WAVE);
    }
    if (threadIdx.x == 0) used = tiles_before;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < experts; e += blockDim.x) {
    const int c = cnt[e], t = (c + cap - 1) / cap;
    for (int i = 0; i < t; ++i)
      tile_e[tiles_of[e] + i] = e | i << MG_E_BITS, tile_r0[tiles_of[e] + i] = cur[e], tile_rows[tiles_of[e] + i] = c;
  }
  // (max_tiles is at least one more than any choice uses: behind the last tile stands how many there are)
  for (int i = used + threadIdx.x; i < max_tiles; i += blockDim.x) tile_e[i] = -1, tile_r0[i] = used, tile_rows[i] = 0;
  __syncthreads();
  // (which pair of an expert gets which of its places depends on timing; a pair's result does not depend on its place)
  for (int p = threadIdx.x; p < pairs; p += blockDim.x) {
    const int e = sel[p];
    if (e < experts) perm[atomicAdd(&cur[e], 1)] = p;
  }
}

// Steps of few rows an expert (decoding): the work is reading the chosen experts' matrices once.  A workgroup takes a tile of up to
// 16 rows and 16 output channels (of gate and up both); its four waves take pieces of 128 along K in turn, weights and rows going straight
// from memory into the operands of v_mfma_f32_16x16x32_bf16 (a wave's four loads of a matrix are 256 contiguous bytes of 16 rows), the
// next piece on its way beside the current one's products, and the waves' sums meet in LDS in a fixed order.
// Bound by the matrices' bytes: 8 tokens, 32 pairs over 32 experts of 1,024 in a width of 2,048, sorting included: 93 -> 58 us (4.0 TB/s
// of the chosen experts' matrices), against a tiled kernel of 160 workgroups (``moe_tile_cap`` has the present ones).
template <bool FIRST, bool DUAL>
__global__ __launch_bounds__(256) void moe_stream_kernel(const bf16_t* __restrict__ A, int a_stride, const bf16_t* __restrict__ B0,
                                                         const bf16_t* __restrict__ B1, const int* __restrict__ perm,
                                                         const int* __restrict__ tile_e, const int* __restrict__ tile_r0,
                                                         const int* __restrict__ tile_rows, bf16_t* __restrict__ act_out, float* __restrict__ out,
                                                         const float* __restrict__ wt, int N, int K, int top, float limit, float alpha, float shift,
                                                         int act_kind) {
  constexpr int MATS = DUAL ? 2 : 1;
  __shared__ __attribute__((aligned(16))) float part[4][MATS][16][20];  // [wave][matrix][row][channel]
  const int tile = blockIdx.y, word = tile_e[tile], e_row0 = tile_r0[tile], e_rows = tile_rows[tile];  // (r0 and rows in one trip to memory)
  if (word < 0) return;
  const int e = tile_expert(word), row0 = 16 * (word >> MG_E_BITS);  // (tiles of 16 rows: every one but an expert's last is full)
  const int r0 = e_row0 + row0, rows = min(16, e_rows - row0), n0 = blockIdx.x * 16;
  const int tid = threadIdx.x, lane = tid % NS_WAVE, wave = tid / NS_WAVE, r = lane % 16, g = lane / 16;
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  const size_t wrow = ((size_t)e * N + min(n0 + r, N - 1)) * K + 8 * g;
  const int xslot = r0 + min(r, rows - 1);
  const bf16_t* xrow = A + (size_t)(FIRST ? perm[xslot] / top : xslot) * a_stride + 8 * g;
  bf16x8 w[2][MATS][4], x[2][4];
  auto fetch = [&](int buf, int k0) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = k0 + 32 * s;
      const bool ok = k + 8 * g < K;
      w[buf][0][s] = ok ? __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(B0 + wrow + k)) : zero;
      if (DUAL) w[buf][MATS - 1][s] = ok ? __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(B1 + wrow + k)) : zero;
      x[buf][s] = ok ? *reinterpret_cast<const bf16x8*>(xrow + k) : zero;
    }
  };
  f32x4 acc[MATS];
#pragma unroll
  for (int i = 0; i < MATS; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int buf) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < MATS; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[buf][i][s], x[buf][s], acc[i], 0, 0, 0);
  };
  // (a piece beyond K is zeros and adds nothing)
  fetch(0, 128 * wave);
  for (int k0 = 128 * wave; k0 < K; k0 += 2 * 512) {
    fetch(1, k0 + 512);
    multiply(0);
    fetch(0, k0 + 1024);
    multiply(1);
  }
#pragma unroll
  for (int i = 0; i < MATS; ++i) *reinterpret_cast<f32x4*>(&part[wave][i][r][4 * g]) = acc[i];
  __syncthreads();
  const int row = tid / 16, c = tid % 16, col = n0 + c;
  if (row >= rows || col >= N) return;
  float v[MATS];
#pragma unroll
  for (int i = 0; i < MATS; ++i) v[i] = (part[0][i][row][c] + part[1][i][row][c]) + (part[2][i][row][c] + part[3][i][row][c]);
  const int slot = r0 + row;
  if (DUAL)
    act_out[(size_t)slot * N + col] = from_f<bf16_t>(clipped_glu(round_to<bf16_t>(v[0]), round_to<bf16_t>(v[MATS - 1]), limit, alpha, shift));
  else if (FIRST)
    act_out[(size_t)slot * N + col] = from_f<bf16_t>(activation_of(round_to<bf16_t>(v[0]), act_kind));
  else
    out[(size_t)perm[slot] * N + col] = wt[perm[slot]] * v[0];
}

// Many rows an expert.  A workgroup takes a tile of the sorted rows and BN rows of the matrices (with gates BN / 2 channels of
// both, the lower half of the tile's rows of w from the gate and the upper the same channels of the up matrix) through LDS (tile_quarters.h); up to 64 rows in
// half a tile.  Bound by the matrices' bytes up to some hundred tokens, beyond by the way from L2 to LDS and by how unevenly the experts' tiles deal.  us a call, sorting
// included, before (tiles by eight waves a whole stage ahead, every tile whole) and now, width 2,048, four of 32 a token, chosen unevenly (as a model's router does): 1,024
// channels with gates, 508 tokens 119 and 98, 1,531 149 and 146, 2,048 198 and 195; evenly 77 and 75, 147 and 141, 162 and 150; 1,536 without gates,
// 2,048 tokens 193 and 185, evenly 174 and 162; six of 64 of 1,408 without gates, 300 tokens 155 and
// 138; two of 8 of 14,336 with gates, width 4,096, 2,000 tokens 1,719 and 1,653, evenly 1,502 and 1,330.
// Workgroups go to the eight XCDs in launch order: each XCD takes an eighth of the work in use, neighbours first, so that an expert's
// matrices and rows come into one L2.  Where an expert has several tiles, all of them take four blocks of
// channels before the next four: all blocks of one tile first bring matrices larger than an L2 from beyond it once a tile (8 experts, two a token,
// width 4,096, 14,336 channels with gates, 2,000 tokens, with the tiles before: 2,264 and 1,689).
// Every expert begins at a stage of K of its own, and in the smaller tiles every block of channels too:
// workgroups that all read the same columns of rows 4 KiB apart keep a few memory channels busy (begun alike: 2 to 10% slower; in the larger tiles by blocks too: 1 to 4%).
// Inner sizes of an odd number of stages (2,880, 704) have a form of their own: with 64-bit addresses and a choice for every load, as sizes of no whole stages have them, and read
// through the caches, width and channels 2,880, with gates, took (evenly and unevenly) 64 tokens 284 and 192 us and take 260 and 178, 300 300 and 306 and 281 and 289, 512 319
// and 345 and 300 and 332, 1,024 377 and 424 and 358 and 411, 2,048 545 and 642 and 513 and 580.
struct MoeTileParams {
  const bf16_t *A, *B0, *B1;
  const int *perm, *tile_e, *tile_r0, *tile_rows;
  bf16_t* act_out;
  float* out;
  const float* wt;
  int a_stride, tiles, N, K, top, act_kind;
  float limit, alpha, shift;
};

// What follows a tile's products.  The activation (ACT; of experts without gates) is chosen once for the tile: with a choice for every value a wave, alone on its
// SIMD, waits for each value's chain of instructions (the first product of 32 experts of 1,536, width 2,048, 2,048 tokens, four a token evenly: 109 us with the
// choice inside, 87 as it is; the square of the ReLU, the whole call 183 and 162, chosen unevenly 201 and 185, 1,024 tokens 121 and 109).
template <class T, bool FIRST, bool DUAL, int ACT>
__device__ __forceinline__ void moe_tile_results(const MoeTileParams& p, const T& t, int r0, int rows, int n0) {
  constexpr int NJ = DUAL ? T::NH : T::NJ;
  const int r = t.lane % 16, g = t.lane / 16;
#pragma unroll
  for (int i = 0; i < T::MI; ++i) {
    const int row = 16 * (2 * i + t.wm) + r;
    if (row >= rows) continue;
    const int slot = r0 + row;
    const int pair = FIRST ? 0 : p.perm[slot];
    const float share_of = FIRST ? 0.f : p.wt[pair];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int col = n0 + 16 * (2 * j + t.wn) + 4 * g;
      if (col >= p.N) continue;  // (N is a multiple of 8: four columns are all inside or all outside)
      if (FIRST) {
        typedef bf16_t bf16x4 __attribute__((ext_vector_type(4)));
        bf16x4 o;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float z = round_to<bf16_t>(t.acc[i][j][q]);
          o[q] = from_f<bf16_t>(DUAL ? clipped_glu(z, round_to<bf16_t>(t.acc[i][T::NH + j][q]), p.limit, p.alpha, p.shift) : activation_as<ACT>(z));
        }
        *reinterpret_cast<bf16x4*>(p.act_out + (size_t)slot * p.N + col) = o;
      } else {
        typedef float f32x4_anywhere __attribute__((ext_vector_type(4), aligned(4)));  // (``out`` is a float's address and no more)
        f32x4_anywhere o;
#pragma unroll
        for (int q = 0; q < 4; ++q) o[q] = share_of * t.acc[i][j][q];
        *reinterpret_cast<f32x4_anywhere*>(p.out + (size_t)pair * p.N + col) = o;
      }
    }
  }
}

// ``rows`` sorted rows from ``r0`` on times expert e's rows of the matrices from channel n0 on
template <class T, bool FIRST, bool DUAL>
__device__ __forceinline__ void moe_one_tile(const MoeTileParams& p, bf16_t* lds, int e, int r0, int rows, int n0, int turn) {
  constexpr int HALF = T::BN / 2;
  T t;
  t.init(lds, p.K, turn);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const bf16_t* w = (DUAL && h ? p.B1 : p.B0) + ((size_t)e * p.N + n0) * p.K;
    const bf16_t* x = FIRST ? p.A : p.A + (size_t)r0 * p.a_stride;
    t.x_from(h, x), t.w_from(h, w);
#pragma unroll
    for (int q = 0; q < T::LA; ++q) {
      const int row = min(h * (T::BM / 2) + t.row_of(q), rows - 1), at = FIRST ? p.perm[r0 + row] / p.top : row;
      if (T::ANY)
        t.x_row(h, q, x + (size_t)at * p.a_stride);
      else
        t.xo[h][q] = 2 * (at * p.a_stride + t.piece());
    }
#pragma unroll
    for (int q = 0; q < T::LB; ++q) {
      const int row = min((DUAL ? 0 : h * HALF) + t.row_of(q), p.N - 1 - n0);
      if (T::ANY)
        t.w_row(h, q, w + (size_t)row * p.K);
      else
        t.wo[h][q] = 2 * (row * p.K + t.piece());
    }
  }
  t.run();

  if (!FIRST || DUAL || p.act_kind == 2)
    moe_tile_results<T, FIRST, DUAL, 2>(p, t, r0, rows, n0);
  else if (p.act_kind == 1)
    moe_tile_results<T, FIRST, DUAL, 1>(p, t, r0, rows, n0);
  else
    moe_tile_results<T, FIRST, DUAL, 0>(p, t, r0, rows, n0);
}

template <class S, bool FIRST, bool DUAL, QuarterInner INNER, bool W_ONCE>
__device__ __forceinline__ void moe_half_or_whole(const MoeTileParams& p, bf16_t* lds, int e, int r0, int rows, int n0, int turn) {
  if (rows <= MG_ROWS / 2)
    moe_one_tile<QuarterTile<MG_ROWS / 2, S::BN, S::HALF_STAGES, W_ONCE, INNER>, FIRST, DUAL>(p, lds, e, r0, rows, n0, turn);
  else
    moe_one_tile<QuarterTile<MG_ROWS, S::BN, 2, W_ONCE, INNER>, FIRST, DUAL>(p, lds, e, r0, rows, n0, turn);
}

template <class S, bool FIRST, bool DUAL, QuarterInner INNER>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1))) void moe_tile_kernel(const MoeTileParams p) {
  constexpr int CH = DUAL ? S::BN / 2 : S::BN;  // output channels of a workgroup
  typedef QuarterTile<MG_ROWS, S::BN, 2> Whole;
  typedef QuarterTile<MG_ROWS / 2, S::BN, S::HALF_STAGES> Half;
  __shared__ __attribute__((aligned(16))) bf16_t moe_tiles[Whole::VALUES > Half::VALUES ? Whole::VALUES : Half::VALUES];
  const int blocks_n = (p.N + CH - 1) / CH;
  const long long used = (long long)p.tile_r0[p.tiles - 1] * blocks_n, share = (used + 7) / 8;
  const long long turn = (long long)blockIdx.y * (gridDim.x >> 3) + (blockIdx.x >> 3), item = (blockIdx.x & 7) * share + turn;
  if (turn >= share || item >= used) return;
  // the expert that this item falls to and its first tile; then four blocks at a time, tile by tile
  const int some = (int)(item / blocks_n), word = p.tile_e[some], c = p.tile_rows[some], e = tile_expert(word), of_e = (c + MG_ROWS - 1) / MG_ROWS;
  const long long at = item - (long long)(some - (word >> MG_E_BITS)) * blocks_n;
  int nth = 0, block = (int)at;
  if (of_e > 1) {
    const int group = (int)(at / (MG_GROUP * of_e)), in_group = (int)(at % (MG_GROUP * of_e));
    const int wide = min(MG_GROUP, blocks_n - MG_GROUP * group);
    nth = in_group / wide, block = MG_GROUP * group + in_group % wide;
  }
  const int row0 = rows_before_tile(c, of_e, nth), rows = rows_before_tile(c, of_e, nth + 1) - row0;
  const int n0 = block * CH, r0 = p.tile_r0[some] + row0;
  // Past the caches only what is read once.  (Inner sizes of an odd number of stages, experts of several tiles, with and without the hint: width and channels 2,880, with
  // gates, 512 tokens of four experts, unevenly, 375 and 332 us; experts of one tile, evenly, 307 and 328, 64 tokens 250 and 285.)
  const int first_stage = block * S::TURN + e * 11;
  if (S::W_ONCE && INNER == QUARTER_ODD && of_e > 1)
    moe_half_or_whole<S, FIRST, DUAL, INNER, false>(p, moe_tiles, e, r0, rows, n0, first_stage);
  else
    moe_half_or_whole<S, FIRST, DUAL, INNER, S::W_ONCE>(p, moe_tiles, e, r0, rows, n0, first_stage);
}

// Rows that a tile holds at most: 16 (the kernel that streams matrices) for the smallest steps, else 128 (the tiled ones).  The tiled kernels take some 28 us
// however little there is to do (two kernels, each the chain of a tile's stages), the streamed one as long as the chosen experts' matrices take at some 4 TB/s,
// and longer where an expert has more than 16 rows.  So tiles from 2^27 bytes of matrices on, if there are workgroups enough for them (experts
// times blocks of 128 of the width) or the rows are several an expert, and from four rows an expert on in any case.  us streamed and in tiles, sorting included,
// width 2,048, unevenly chosen, with gates and without: 32 experts of 1,024, four a token, 2 tokens 30 and 29, 22 and 30; 4 44 and 36, 33 and 34; 8 66 and 61, 42 and 40; 16
// 81 and 65, 62 and 48; 16 of 1,408, two a token, 2 27 and 33, 21 and 30; 4 37 and 35, 28 and 35; 8 55 and 51, 36 and 36; 8 of 4,096, two a token, 2 43 and 48, 39 and 47; 4 60 and
// 67, 50 and 53; 8 88 and 77, 60 and 55; 16 83 and 78, 70 and 58; 8 of 1,024, one a token, 32 tokens 31 and 32, 25 and 30, 64 36 and 31, 33 and 30; 256 of 512, eight a
// token, 2 36 and 30, 29 and 29; 32 218 and 187, 145 and 125.
static int moe_tile_cap(long long pairs, int experts, int W, int ff, int gated) {
  const long long chosen = pairs < experts ? pairs : experts, bytes = chosen * ff * W * (gated ? 6 : 4);
  const bool enough = chosen * ((W + 127) / 128) >= 192 || pairs >= 2LL * experts;
  return pairs > 4LL * experts || (bytes >= 1LL << 27 && enough) ? MG_ROWS : 16;
}
static int moe_tiles(long long pairs, int experts, int cap) { return (int)((pairs + cap - 1) / cap) + experts; }

// Which tiles: up to 96 rows an expert on average the smaller ones, whose loads of the matrices go past the caches (most experts have one
// tile); beyond, the larger ones, which read less.  Neither is far ahead of the other near the line, and it moves with more than rows: us smaller
// and larger, evenly and unevenly chosen: with gates, 32 experts of 1,024, width 2,048, four a token: 64 rows an expert 79 and 91, 102 and 121, 128 rows 98 and 105, 142 and
// 135, 192 rows 153 and 140, 158 and 144; 1,536 channels without gates 128 rows 112 and 121, 157 and 165, 256 rows 174 and 181, 217 and 199; 8 experts, width 4,096, two a
// token: 4,096 channels 96 rows 153 and 182, 162 and 181, 128 rows 164 and 185, 243 and 222; 14,336 channels 64 rows 479 and 584, 501 and 600 (most unevenly 654 and 617).
// Inner sizes of an odd number of stages, whose smaller tiles read the matrices past the caches only where an expert has one tile (see moe_tile_kernel): up to 128. 128 and 192
// rows, with gates, width 2,880, 2,880 channels: 358 and 343, 411 and 424; 499 and 480, 502 and 512; 1,440 channels 208 and 227, 246 and 262; width 2,048, 704 channels, 125
// rows 75 and 81, 114 and 120.  Of no whole stages: the smaller ones at any number, on whose address and choice a load there is less to wait: 2,056 channels,
// width 1,448, 256 rows 309 and 316, 329 and 338; 1,440 of 1,440 204 and 205, 219 and 228, without gates 512 rows 257 and 244, 274 and 290.
static bool moe_few_rows(long long pairs, int experts, QuarterInner inner) {
  return inner == QUARTER_ANY || pairs <= (inner == QUARTER_ODD ? 128LL : 96LL) * experts;
}

// tiles that any choice of experts can need, whichever kernel takes them
extern "C" int ns_moe_group_tiles(int pairs, int experts) { return moe_tiles(pairs, experts, 16); }

// The launch for so many items of a tile and a block of channels: the XCDs' eight workgroups of a turn side by side, and the turns in two dimensions,
// because one holds fewer than 2^32 threads.
static dim3 moe_tile_grid(long long items) {
  const long long turns = (items + 7) / 8, row = turns < 65536 ? turns : 65536;
  return dim3((unsigned)(8 * row), (unsigned)((turns + row - 1) / row));
}

extern "C" void ns_moe_tile_grid(long long items, unsigned* xy) {
  const dim3 grid = moe_tile_grid(items);
  xy[0] = grid.x, xy[1] = grid.y;
}

struct MoeLaunch {
  const bf16_t *h, *wg, *wu, *wd;
  bf16_t* act;
  float* out;
  const int *perm, *tile_e, *tile_r0, *tile_rows;
  const float* wt;
  int h_stride, W, ff, top, tiles, act_kind;
  float limit, alpha, shift;
  long long pairs, rows;  // (rows of h)
  int experts;
  hipStream_t stream;

  template <class S, bool FIRST, bool DUAL, QuarterInner INNER>
  void launch(const MoeTileParams& p) const {
    constexpr int CH = DUAL ? S::BN / 2 : S::BN;
    moe_tile_kernel<S, FIRST, DUAL, INNER><<<moe_tile_grid((long long)tiles * ((p.N + CH - 1) / CH)), 256, 0, stream>>>(p);
  }
  template <bool FIRST, bool DUAL, QuarterInner INNER>
  void sized(const MoeTileParams& p) const {
    if (moe_few_rows(pairs, experts, INNER))
      launch<MoeFewTile, FIRST, DUAL, INNER>(p);
    else if constexpr (INNER != QUARTER_ANY)
      launch<MoeTile, FIRST, DUAL, INNER>(p);
  }
  template <bool FIRST, bool DUAL>
  void tiled(const bf16_t* a, int a_stride, const bf16_t* b0, const bf16_t* b1, int n, int k) const {
    const MoeTileParams p{a, b0, b1, perm, tile_e, tile_r0, tile_rows, act, out, wt, a_stride, tiles, n, k, top, act_kind, limit, alpha, shift};
    // whole stages, and all rows within 31 bits of bytes of their first
    const bool plain = k % QUARTER_K == 0 && k >= (k / QUARTER_K % 2 ? 5 : 4) * QUARTER_K && k < 1 << 22 && a_stride < 1 << 22 && (!FIRST || rows * a_stride < 1LL << 30);
    if (!plain)
      sized<FIRST, DUAL, QUARTER_ANY>(p);
    else if (k % QUARTER_K_MULTIPLE)
      sized<FIRST, DUAL, QUARTER_ODD>(p);
    else
      sized<FIRST, DUAL, QUARTER_PAIRS>(p);
  }
  template <bool DUAL>
  void first(int cap) const {
    const bf16_t *b0 = DUAL ? wg : wu, *b1 = DUAL ? wu : nullptr;
    if (cap == 16)
      moe_stream_kernel<true, DUAL><<<dim3((ff + 15) / 16, tiles), 256, 0, stream>>>(h, h_stride, b0, b1, perm, tile_e, tile_r0, tile_rows, act, nullptr,
                                                                                    nullptr, ff, W, top, limit, alpha, shift, act_kind);
    else
      tiled<true, DUAL>(h, h_stride, b0, b1, ff, W);
  }
  void second(int cap) const {
    if (cap == 16)
      moe_stream_kernel<false, false><<<dim3((W + 15) / 16, tiles), 256, 0, stream>>>(act, ff, wd, nullptr, perm, tile_e, tile_r0, tile_rows, nullptr, out, wt,
                                                                                     W, ff, top, limit, alpha, shift, act_kind);
    else
      tiled<false, false>(act, ff, wd, nullptr, W, ff);
  }
};

// ``ints``: scratch of pairs + 3 * ns_moe_group_tiles(...) 32-bit words; ``act``: bfloat16 [pairs][ff]
extern "C" int ns_moe_expert_groups(const void* h, int h_stride, const void* wg, const void* wu, const void* wd, const int* sel, const float* wt,
                                    int* ints, void* act, float* out, int n, int W, int ff, int top, int experts, float limit, float alpha, float shift,
                                    int act_kind, hipStream_t stream) {
  if (!wg && (act_kind < 0 || act_kind >= NS_ACTIVATIONS)) return NS_ERR_BAD_ARG;
  if (n <= 0 || W <= 0 || ff <= 0 || top <= 0 || experts <= 0 || experts > MOE_MAX_EXPERTS) return NS_ERR_BAD_ARG;
  if (W % 8 || ff % 8 || h_stride % 8 || (uintptr_t)h % 16 || (uintptr_t)wg % 16 || (uintptr_t)wu % 16 || (uintptr_t)wd % 16 || (uintptr_t)act % 16)
    return NS_ERR_UNSUPPORTED;
  const long long pairs = (long long)n * top;
  if (pairs > (1 << 24)) return NS_ERR_UNSUPPORTED;
  const int cap = moe_tile_cap(pairs, experts, W, ff, wg != nullptr), tiles = moe_tiles(pairs, experts, cap);
  int* perm = ints;
  int* tile_e = ints + pairs;
  int* tile_r0 = tile_e + tiles;
  int* tile_rows = tile_r0 + tiles;
  if (tiles > 65535) return NS_ERR_UNSUPPORTED;
  moe_sort_kernel<<<1, 1024, 0, stream>>>(sel, (int)pairs, experts, cap, perm, tile_e, tile_r0, tile_rows, tiles);
  const MoeLaunch l{(const bf16_t*)h, (const bf16_t*)wg, (const bf16_t*)wu, (const bf16_t*)wd, (bf16_t*)act, out, perm, tile_e, tile_r0,
                    tile_rows, wt, h_stride, W, ff, top, tiles, act_kind, limit, alpha, shift, pairs, n, experts, stream};
  if (wg)
    l.first<true>(cap);
  else
    l.first<false>(cap);
  l.second(cap);
  return ns_launch_status();
}

// out[t][f] = clipped_glu(gu[t][f], gu[t][ff + f]) for the result of a product with the stacked [gate; up] matrix
template <typename T>
__global__ void clipped_glu_kernel(T* __restrict__ out, const T* __restrict__ gu, int gu_stride, int ff, size_t count, float limit, float alpha, float shift) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x) {
    const size_t t = i / ff, f = i % ff;
    out[i] = from_f<T>(clipped_glu(to_f(gu[t * gu_stride + f]), to_f(gu[t * gu_stride + ff + f]), limit, alpha, shift));
  }
}

// A workgroup of 256 for rows of so many pieces of 16 bytes: x along a row, y rows.  As many along a row as leave the fewest beyond its end, half a KiB of it at least where
// it has that: with 256 along every row most of the threads of a narrow one have nothing to do (65,536 rows of 64 bfloat16 values, sum of two
// and clipped gate: 256 along 29.9 and 30.8 us, value by value 6.2 and 10.1, as it is 3.5 and 5.9; 2,048 of 2,560 6.4 and 9.6, 8.7 and 12.7, 4.2 and 7.2).
static dim3 piece_block(int pieces) {
  const auto padded = [pieces](int x) { return (pieces + x - 1) / x * x; };
  int x = 256;
  while (x > 32 && padded(x / 2) < padded(x)) x /= 2;
  while (x >= 2 * pieces) x /= 2;
  return dim3(x, 256 / x);
}
static dim3 piece_grid(int pieces, int rows, dim3 block) {
  const unsigned y = (rows + block.y - 1) / block.y;
  return dim3((pieces + block.x - 1) / block.x, y < 65535 ? y : 65535);
}

// The same in pieces of 16 bytes (nothing is divided).  Bound by the bytes: 2,048 rows of 4,096, bfloat16, 19.8 -> 10.4 us.
template <typename T>
__global__ __launch_bounds__(256) void clipped_glu_vec_kernel(T* __restrict__ out, const T* __restrict__ gu, int gu_stride, int n, int ff, float limit, float alpha,
                                                             float shift) {
  constexpr int V = 16 / sizeof(T);
  typedef T vec_t __attribute__((ext_vector_type(V)));
  const int f = (blockIdx.x * blockDim.x + threadIdx.x) * V;
  if (f >= ff) return;
  for (size_t t = blockIdx.y * blockDim.y + threadIdx.y; t < (size_t)n; t += gridDim.y * blockDim.y) {
    const vec_t g = *reinterpret_cast<const vec_t*>(gu + t * gu_stride + f), u = *reinterpret_cast<const vec_t*>(gu + t * gu_stride + ff + f);
    vec_t o;
#pragma unroll
    for (int i = 0; i < V; ++i) o[i] = from_f<T>(clipped_glu(to_f((T)g[i]), to_f((T)u[i]), limit, alpha, shift));
    *reinterpret_cast<vec_t*>(out + t * ff + f) = o;
  }
}

extern "C" int ns_clipped_glu(void* out, const void* gu, int gu_stride, int n, int ff, float limit, float alpha, float shift, int dtype, hipStream_t stream) {
  if (n <= 0 || ff <= 0) return NS_ERR_BAD_ARG;
  const int v = dtype == NS_DTYPE_F32 ? 4 : 8;
  if ((dtype == NS_DTYPE_F32 || dtype == NS_DTYPE_BF16) && ff % v == 0 && gu_stride % v == 0 && !(((uintptr_t)out | (uintptr_t)gu) & 15)) {
    const dim3 block = piece_block(ff / v), grid = piece_grid(ff / v, n, block);
    if (dtype == NS_DTYPE_F32)
      clipped_glu_vec_kernel<float><<<grid, block, 0, stream>>>((float*)out, (const float*)gu, gu_stride, n, ff, limit, alpha, shift);
    else
      clipped_glu_vec_kernel<bf16_t><<<grid, block, 0, stream>>>((bf16_t*)out, (const bf16_t*)gu, gu_stride, n, ff, limit, alpha, shift);
    return ns_launch_status();
  }
  const size_t count = (size_t)n * ff;
  size_t blocks = (count + 255) / 256;
  if (blocks > 65535) blocks = 65535;
  if (dtype == NS_DTYPE_F32)
    clipped_glu_kernel<float><<<(int)blocks, 256, 0, stream>>>((float*)out, (const float*)gu, gu_stride, ff, count, limit, alpha, shift);
  else if (dtype == NS_DTYPE_BF16)
    clipped_glu_kernel<bf16_t><<<(int)blocks, 256, 0, stream>>>((bf16_t*)out, (const bf16_t*)gu, gu_stride, ff, count, limit, alpha, shift);
  else
    return NS_ERR_UNSUPPORTED;
  return ns_launch_status();
}

// What the outputs of a router beyond the experts do: a pair (t, k) with sel[t][k] >= experts adds its weight times the input row.
struct MoeIdentity {
  const int* sel;   // [tokens][top], or null: the router has no such outputs
  const float* wt;  // [tokens][top]
  const void* h;    // [tokens][W] rows h_stride apart, in the model's precision
  int h_stride, experts;
};

// out[t][c] = (base ? base[t][c] : 0) + sum_k parts[t][k][c], in a fixed order; with ``zgate`` (32-bit, z_stride words from
// token to token) the base is multiplied by sigmoid(zgate[t])
template <typename T>
__global__ void moe_combine_kernel(T* __restrict__ out, const T* __restrict__ base, const float* __restrict__ zgate, int z_stride,
                                   const float* __restrict__ parts, const MoeIdentity id, int top, int W, size_t count) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x) {
    const size_t t = i / W, c = i % W;
    float acc = 0.f;
    for (int k = 0; k < top; ++k) {
      if (id.sel && id.sel[t * top + k] >= id.experts)
        acc = fmaf(id.wt[t * top + k], to_f(((const T*)id.h)[t * id.h_stride + c]), acc);
      else
        acc += parts[(t * top + k) * W + c];
    }
    if (base) acc += to_f(base[i]) * (zgate ? 1.f / (1.f + expf(-zgate[t * z_stride])) : 1.f);
    out[i] = from_f<T>(acc);
  }
}

// The same for rows in whole pieces of four (a workgroup is a token's 1,024 columns: nothing is divided, every load 16 bytes of the parts and 8
// or 16 of the rest).  Bound by the bytes: 2,048 tokens of four parts of 2,048: 27 -> 13 us.
template <typename T>
__global__ __launch_bounds__(256) void moe_combine_vec_kernel(T* __restrict__ out, const T* __restrict__ base, const float* __restrict__ zgate, int z_stride,
                                                              const float* __restrict__ parts, const MoeIdentity id, int top, int W) {
  typedef T t4 __attribute__((ext_vector_type(4)));
  const size_t t = blockIdx.x;
  const int c = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (c >= W) return;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < top; ++k) {
    if (id.sel && id.sel[t * top + k] >= id.experts) {
      const float share = id.wt[t * top + k];
      const t4 x = *reinterpret_cast<const t4*>((const T*)id.h + t * id.h_stride + c);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = fmaf(share, to_f((T)x[i]), acc[i]);
    } else {
      acc += *reinterpret_cast<const f32x4*>(parts + (t * top + k) * W + c);
    }
  }
  if (base) {
    const t4 b = *reinterpret_cast<const t4*>(base + t * W + c);
    const float share = zgate ? 1.f / (1.f + expf(-zgate[t * z_stride])) : 1.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] += to_f((T)b[i]) * share;
  }
  t4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = from_f<T>(acc[i]);
  *reinterpret_cast<t4*>(out + t * W + c) = o;
}

extern "C" int ns_moe_combine(void* out, const void* base, const float* zgate, int z_stride, const float* parts, const int* sel, const float* wt,
                              const void* h, int h_stride, int experts, int n, int top, int W, int dtype, hipStream_t stream) {
  if (n <= 0 || top <= 0 || W <= 0 || (sel && (!wt || !h || experts <= 0))) return NS_ERR_BAD_ARG;
  const MoeIdentity id{sel, wt, h, h_stride, experts};
  const uintptr_t piece = dtype == NS_DTYPE_F32 ? 15 : 7;  // four values of T
  if ((dtype == NS_DTYPE_F32 || dtype == NS_DTYPE_BF16) && W % 4 == 0 && (!sel || h_stride % 4 == 0) && !((uintptr_t)parts & 15) &&
      !(((uintptr_t)out | (uintptr_t)base | (uintptr_t)h) & piece) && (W + 1023) / 1024 <= 65535) {
    const dim3 grid(n, (W + 1023) / 1024);
    if (dtype == NS_DTYPE_F32)
      moe_combine_vec_kernel<float><<<grid, 256, 0, stream>>>((float*)out, (const float*)base, zgate, z_stride, parts, id, top, W);
    else
      moe_combine_vec_kernel<bf16_t><<<grid, 256, 0, stream>>>((bf16_t*)out, (const bf16_t*)base, zgate, z_stride, parts, id, top, W);
    return ns_launch_status();
  }
  const size_t count = (size_t)n * W;
  size_t blocks = (count + 255) / 256;
  if (blocks > 65535) blocks = 65535;
  if (dtype == NS_DTYPE_F32)
    moe_combine_kernel<float><<<(int)blocks, 256, 0, stream>>>((float*)out, (const float*)base, zgate, z_stride, parts, id, top, W, count);
  else if (dtype == NS_DTYPE_BF16)
    moe_combine_kernel<bf16_t><<<(int)blocks, 256, 0, stream>>>((bf16_t*)out, (const bf16_t*)base, zgate, z_stride, parts, id, top, W, count);
  else
    return NS_ERR_UNSUPPORTED;
  return ns_launch_status();
}

// out = sa * (a + bias_a) + sb * (b + bias_b) in 32-bit: two mixers side by side, each with a weight (the biases: a mixer's
// last bias that it left to its caller; either may be null)
template <typename T>
__global__ void scaled_sum_kernel(T* __restrict__ out, const T* __restrict__ a, const T* __restrict__ b, const T* __restrict__ bias,
                                  const T* __restrict__ bias_b, float sa, float sb, int W, size_t count) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x) {
    const float av = to_f(a[i]) + (bias ? to_f(bias[i % W]) : 0.f);
    const float bv = to_f(b[i]) + (bias_b ? to_f(bias_b[i % W]) : 0.f);
    out[i] = from_f<T>(sa * av + sb * bv);
  }
}

// The same in pieces of 16 bytes (nothing is divided).  Bound by the bytes: 1,531 rows of 2,048, bfloat16, 5.2 -> 3.1 us, 2,048 of 4,096 15.0 -> 8.7.
template <typename T>
__global__ __launch_bounds__(256) void scaled_sum_vec_kernel(T* __restrict__ out, const T* __restrict__ a, const T* __restrict__ b, const T* __restrict__ bias,
                                                            const T* __restrict__ bias_b, float sa, float sb, int n, int W) {
  constexpr int V = 16 / sizeof(T);
  typedef T vec_t __attribute__((ext_vector_type(V)));
  const int c = (blockIdx.x * blockDim.x + threadIdx.x) * V;
  if (c >= W) return;
  vec_t ba = {}, bb = {};
  if (bias) ba = *reinterpret_cast<const vec_t*>(bias + c);
  if (bias_b) bb = *reinterpret_cast<const vec_t*>(bias_b + c);
  for (size_t t = blockIdx.y * blockDim.y + threadIdx.y; t < (size_t)n; t += gridDim.y * blockDim.y) {
    const vec_t av = *reinterpret_cast<const vec_t*>(a + t * W + c), bv = *reinterpret_cast<const vec_t*>(b + t * W + c);
    vec_t o;
#pragma unroll
    for (int i = 0; i < V; ++i) o[i] = from_f<T>(sa * (to_f((T)av[i]) + to_f((T)ba[i])) + sb * (to_f((T)bv[i]) + to_f((T)bb[i])));
    *reinterpret_cast<vec_t*>(out + t * W + c) = o;
  }
}

extern "C" int ns_scaled_sum(void* out, const void* a, const void* b, const void* bias, const void* bias_b, float sa, float sb, int n, int W,
                             int dtype, hipStream_t stream) {
  if (n <= 0 || W <= 0) return NS_ERR_BAD_ARG;
  const int v = dtype == NS_DTYPE_F32 ? 4 : 8;
  if ((dtype == NS_DTYPE_F32 || dtype == NS_DTYPE_BF16) && W % v == 0 &&
      !(((uintptr_t)out | (uintptr_t)a | (uintptr_t)b | (uintptr_t)bias | (uintptr_t)bias_b) & 15)) {
    const dim3 block = piece_block(W / v), grid = piece_grid(W / v, n, block);
    if (dtype == NS_DTYPE_F32)
      scaled_sum_vec_kernel<float><<<grid, block, 0, stream>>>((float*)out, (const float*)a, (const float*)b, (const float*)bias, (const float*)bias_b, sa, sb, n, W);
    else
      scaled_sum_vec_kernel<bf16_t><<<grid, block, 0, stream>>>((bf16_t*)out, (const bf16_t*)a, (const bf16_t*)b, (const bf16_t*)bias, (const bf16_t*)bias_b, sa, sb, n, W);
    return ns_launch_status();
  }
  const size_t count = (size_t)n * W;
  size_t blocks = (count + 255) / 256;
  if (blocks > 65535) blocks = 65535;
  if (dtype == NS_DTYPE_F32)
    scaled_sum_kernel<float><<<(int)blocks, 256, 0, stream>>>((float*)out, (const float*)a, (const float*)b, (const float*)bias, (const float*)bias_b, sa, sb, W, count);
  else if (dtype == NS_DTYPE_BF16)
    scaled_sum_kernel<bf16_t><<<(int)blocks, 256, 0, stream>>>((bf16_t*)out, (const bf16_t*)a, (const bf16_t*)b, (const bf16_t*)bias, (const bf16_t*)bias_b, sa, sb, W, count);
  else
    return NS_ERR_UNSUPPORTED;
  return ns_launch_status();
}

// The same with a norm behind each side: out = sa * rms(a + bias_a) * wa + sb * rms(b + bias_b) * wb, rms over the row, in 32-bit.
// One workgroup a row.
template <typename T>
__global__ __launch_bounds__(1024) void normed_sum_kernel(T* __restrict__ out, const T* __restrict__ a, const T* __restrict__ b,
                                                         const T* __restrict__ bias, const T* __restrict__ bias_b, const T* __restrict__ wa,
                                                         const T* __restrict__ wb, float sa, float sb, int W, float eps) {
  __shared__ float scratch[16];
  const size_t at = (size_t)blockIdx.x * W;
  float ssa = 0.f, ssb = 0.f;
  for (int c = threadIdx.x; c < W; c += blockDim.x) {
    const float av = to_f(a[at + c]) + (bias ? to_f(bias[c]) : 0.f), bv = to_f(b[at + c]) + (bias_b ? to_f(bias_b[c]) : 0.f);
    ssa = fmaf(av, av, ssa), ssb = fmaf(bv, bv, ssb);
  }
  const float fa = sa / sqrtf(block_sum(ssa, scratch) / (float)W + eps);
  const float fb = sb / sqrtf(block_sum(ssb, scratch) / (float)W + eps);
  for (int c = threadIdx.x; c < W; c += blockDim.x) {
    const float av = to_f(a[at + c]) + (bias ? to_f(bias[c]) : 0.f), bv = to_f(b[at + c]) + (bias_b ? to_f(bias_b[c]) : 0.f);
    out[at + c] = from_f<T>(av * fa * to_f(wa[c]) + bv * fb * to_f(wb[c]));
  }
}

extern "C" int ns_normed_sum(void* out, const void* a, const void* b, const void* bias, const void* bias_b, const void* wa, const void* wb, float sa,
                             float sb, int n, int W, float eps, int dtype, hipStream_t stream) {
  if (n <= 0 || W <= 0 || !wa || !wb) return NS_ERR_BAD_ARG;
  const int threads = W > 1024 && n <= 64 ? 1024 : 256;
  if (dtype == NS_DTYPE_F32)
    normed_sum_kernel<float><<<n, threads, 0, stream>>>((float*)out, (const float*)a, (const float*)b, (const float*)bias, (const float*)bias_b, (const float*)wa, (const float*)wb, sa, sb, W, eps);
  else if (dtype == NS_DTYPE_BF16)
    normed_sum_kernel<bf16_t><<<n, threads, 0, stream>>>((bf16_t*)out, (const bf16_t*)a, (const bf16_t*)b, (const bf16_t*)bias, (const bf16_t*)bias_b, (const bf16_t*)wa, (const bf16_t*)wb, sa, sb, W, eps);
  else
    return NS_ERR_UNSUPPORTED;
  return ns_launch_status();
}

// The per-layer token input: y = W_proj (gelu_tanh(W_gate x) * e) with e = table[token] (this layer's ``dim`` columns of a
// row).  The two products are the framework's; between them: out[t][j] = gelu_tanh(g[t][j]) * table[ids[t]][j].
template <typename T>
__global__ void gelu_gather_mul_kernel(T* __restrict__ out, const T* __restrict__ g, int g_stride, const int* __restrict__ ids,
                                       const T* __restrict__ table, int dim, size_t count) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x) {
    const size_t t = i / dim, j = i % dim;
    const float z = to_f(g[t * g_stride + j]);
    out[i] = from_f<T>(round_to<T>(gelu_tanh(z)) * to_f(table[(size_t)ids[t] * dim + j]));
  }
}

extern "C" int ns_gelu_gather_mul(void* out, const void* g, int g_stride, const int* ids, const void* table, int n, int dim, int dtype,
                                  hipStream_t stream) {
  if (n <= 0 || dim <= 0) return NS_ERR_BAD_ARG;
  const size_t count = (size_t)n * dim;
  size_t blocks = (count + 255) / 256;
  if (blocks > 65535) blocks = 65535;
  if (dtype == NS_DTYPE_F32)
    gelu_gather_mul_kernel<float><<<(int)blocks, 256, 0, stream>>>((float*)out, (const float*)g, g_stride, ids, (const float*)table, dim, count);
  else if (dtype == NS_DTYPE_BF16)
    gelu_gather_mul_kernel<bf16_t><<<(int)blocks, 256, 0, stream>>>((bf16_t*)out, (const bf16_t*)g, g_stride, ids, (const bf16_t*)table, dim, count);
  else
    return NS_ERR_UNSUPPORTED;
  return ns_launch_status();
}

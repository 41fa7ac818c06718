// Products of many 32-bit rows on the float16 matrix cores, out[m][n] = sum_k x[m][k] w[n][k], in less than half of the 32-bit ones' time and nearer to 64 bits.
// (reference: the nn.Linear calls of model/llama.py:175,184,195)
//
// A float times a power of two is the sum of two float16 values, a = a0 + a1, each the nearest to what is left: |a1| <= 2^-11 |a|, and 2^-23 |a| at most is lost, or 2^-25 where
// the largest is 2^14 to 2^15: small ones keep what counts beside it.  Powers of two are chosen for each 32 k of a row of x, and for each row of w.  Of the four products of two such
// sums three are taken, the smallest first: a1 b0, a0 b1, a0 b0; the one left out is 2^-22 of a b at most, and its sign is any.  A product of two float16 values is exact in 32 bits.
// The matrix instruction adds up blocks of 8 k and rounds each sum to nearest, so three of them over a stage of 32 k begin at zero and the vector unit adds what they give to the
// sums, times the power of two of x.
// Error against 64 bits (2-norm), this in one range of K and the 32-bit instruction's four chains (gemm_generic.hip): both operands normal, K 2,048 1.8e-7 and 4.1e-7, K 8,192 3.2e-7
// and 8.1e-7; all of one sign 1.3e-7 and 1.8e-7, 2.5e-7 and 3.5e-7; x spread over 24 powers of two 1.9e-7 and 3.9e-7, 3.3e-7 and 7.6e-7; one k of 512 10^5 times the others 1.9e-7 and
// 4.6e-7, 3.2e-7 and 8.4e-7.  (Three bfloat16 values for a float, six products: 1.6e-7 and 3.1e-7 for normal operands, and twice the work of the matrix unit.)
//
// Both operands are split ahead, w once for all (as many bytes again as it has), x a call.  w split in registers on its way by every tile of x instead: 211 us for the 177 below.
// x comes through LDS, where the four waves share it, and each wave's own columns of w straight into the registers of the matrix instruction, both two stages ahead (one: tiles that have a
// compute unit to themselves 1.2 times as long).  us, the 32-bit instruction and this with the splitting of x and the sum of ranges of K, alone / a call beside two others:
// 832 rows, N 16,384, K 2,048 536 / 511 and 206 / 177 (315 TFLOP/s of products of 32 bits), N 2,048, K 8,192 307 / 272 and 122 / 102, N 3,072, K 2,048 96 / 89 and 66 / 35;
// 2,048 rows of 28,672 x 4,096 3,649 / 3,727 and 1,300 / 1,561.
// Bound by the power of the matrix unit: at the last size it works for 69% of the cycles and the clock sinks to 1.4 GHz.
#include "common.h"
#include "lds_loads.h"

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((__vector_size__(4 * sizeof(float))));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

#define SPLIT_K 32       // k of a stage
#define SPLIT_BLOCK 512  // values of a block: 16 rows of a stage
#define SPLIT_COLUMNS 2  // blocks of 16 rows of w a wave: with four, 112 rows of x a tile and two workgroups a compute unit instead of three, 173 us for the 177 above and 49 for the 35
#define SPLIT_DOWN 0x1p-15f  // with the scale of x: sums are kept as if a row's largest of w were 1/2 to 1, so that they are in range where x and the results are
#define SPLIT_STAGES 3   // at hand: one that is multiplied and two on their way

union Operand {  // of the matrix instruction: eight values, made two at a time
  f16x8 v;
  f16x2 pair[4];
};

// The power of two that brings ``largest`` into [2^14, 2^15) (as far as its inverse is a normal number too; nothing, infinities and no numbers: any), and its inverse.
__device__ __forceinline__ float split_scale(float largest) {
  const int e = max((int)(__builtin_bit_cast(unsigned, largest) >> 23 & 255), 15);
  return __builtin_bit_cast(float, (unsigned)(268 - e) << 23);
}
__device__ __forceinline__ float inverse_scale(float scale) { return __builtin_bit_cast(float, (254u << 23) - __builtin_bit_cast(unsigned, scale)); }

// Eight floats times a power of two into their two parts.
__device__ __forceinline__ void split_eight(const f32x4& low, const f32x4& high, float scale, Operand* part) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const f32x4& of = e < 2 ? low : high;
    const f32x2 v = {of[e % 2 * 2], of[e % 2 * 2 + 1]};
    const f16x2 first = __builtin_convertvector((f32x2{v[0] * scale, v[1] * scale}), f16x2);
    part[0].pair[e] = first;
    part[1].pair[e] = __builtin_convertvector((f32x2{fmaf(v[0], scale, -(float)first[0]), fmaf(v[1], scale, -(float)first[1])}), f16x2);  // (exact before it is rounded)
  }
}

// x [M, K] as parts[block of 16 rows][block of 32 k][part][lane][8], where lane 16 g + r holds of row r the k 8 g .. 8 g + 7 of the block: an operand of the matrix
// instruction as it lies in registers, so that any two blocks are two contiguous KB.  Rows beyond the last are zeros.
// ``scales`` (of w): a power of two a row.  Without them (of x) one a row and block, their inverses over 2^15 behind all parts, [block of 16 rows][block of 32 k][16]
// (below the normal numbers for the smallest of x, and exact there too).
__global__ __launch_bounds__(256) void split_rows_kernel(_Float16* __restrict__ parts, const float* __restrict__ x, const float* __restrict__ scales, int M, int K, int x_stride) {
  const int k_blocks = K / SPLIT_K, lane = threadIdx.x % NS_WAVE, r = lane % 16, g = lane / 16;
  const int kb = blockIdx.x * 4 + threadIdx.x / NS_WAVE, mb = blockIdx.y, row = mb * 16 + r;
  if (kb >= k_blocks) return;
  f32x4 low = {0.f, 0.f, 0.f, 0.f}, high = low;
  if (row < M) {
    const float* at = x + (size_t)row * x_stride + kb * SPLIT_K + 8 * g;
    low = *reinterpret_cast<const f32x4*>(at), high = *reinterpret_cast<const f32x4*>(at + 4);
  }
  const size_t block = (size_t)mb * k_blocks + kb;
  float scale = 1.f;
  if (scales) {
    if (row < M) scale = scales[row];
  } else {
    float largest = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) largest = fmaxf(largest, fmaxf(fabsf(low[e]), fabsf(high[e])));
    largest = fmaxf(largest, __shfl_xor(largest, 16)), largest = fmaxf(largest, __shfl_xor(largest, 32));
    scale = split_scale(largest);
    if (g == 0) reinterpret_cast<float*>(parts + (size_t)gridDim.y * k_blocks * 2 * SPLIT_BLOCK)[block * 16 + r] = inverse_scale(scale) * SPLIT_DOWN;
  }
  Operand part[2];
  split_eight(low, high, scale, part);
  f16x8* to = reinterpret_cast<f16x8*>(parts + block * 2 * SPLIT_BLOCK) + lane;
#pragma unroll
  for (int p = 0; p < 2; ++p) to[p * NS_WAVE] = part[p].v;
}

// The scale of each row of w, a row a wave.
__global__ __launch_bounds__(256) void split_scales_kernel(float* __restrict__ scales, const float* __restrict__ w, int N, int K) {
  const int n = blockIdx.x * 4 + threadIdx.x / NS_WAVE, lane = threadIdx.x % NS_WAVE;
  if (n >= N) return;
  float largest = 0.f;
  for (int k = 4 * lane; k < K; k += 4 * NS_WAVE) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(w + (size_t)n * K + k);
#pragma unroll
    for (int e = 0; e < 4; ++e) largest = fmaxf(largest, fabsf(v[e]));
  }
#pragma unroll
  for (int d = 1; d < NS_WAVE; d *= 2) largest = fmaxf(largest, __shfl_xor(largest, d));
  if (lane == 0) scales[n] = split_scale(largest);
}

struct SplitParams {
  float* out;  // [M, N], or with ranges of K [ranges][M][N]
  const _Float16 *parts, *w_parts;
  const float *x, *w, *w_scales;
  int M, N, K, x_stride, out_stride, m_tiles, n_tiles, ranges;
};

// One output as one chain over k in 32 bits, until it is no number.
__device__ __attribute__((noinline)) float split_plain(const float* a, const float* b, int k) {
  float s = 0.f;
  for (int i = 0; i < k && s == s; i += 4) {
    const f32x4 u = *reinterpret_cast<const f32x4*>(a + i), v = *reinterpret_cast<const f32x4*>(b + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) s = fmaf(u[e], v[e], s);
  }
  return s;
}

// Four waves, 16 MI rows of x by 128 of w.  A stage's parts of x lie in LDS and those of w in the registers of the wave whose columns they are, and the next two are on their way.
template <int MI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void gemm_split_kernel(const SplitParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(3))) void* lds_ptr;
  constexpr int NJ = SPLIT_COLUMNS, TM = 16 * MI, TN = 64 * NJ, STAGE = 2 * MI * SPLIT_BLOCK + SPLIT_BLOCK;
  constexpr int XPARTS = (2 * MI + 3) / 4, LOADS = XPARTS + 1 + 2 * NJ;  // of a wave for a stage
  static_assert(4 * MI <= NS_WAVE, "the scales of a stage by one load");
  __shared__ __attribute__((aligned(16))) _Float16 lds[SPLIT_STAGES * STAGE];  // a stage: the parts, and behind them the inverse scales (64 bytes a block; room for a whole load)
  // an XCD (workgroups go to the eight in launch order) takes every eighth tile of w and all tiles of x against it one after the other
  const int xcd = blockIdx.x & 7, turn = blockIdx.x >> 3, range = blockIdx.y;
  const int nt = (turn / p.m_tiles) * 8 + xcd, mt = turn % p.m_tiles;
  if (nt >= p.n_tiles) return;
  const int m0 = mt * TM, n0 = nt * TN, k_blocks = p.K / SPLIT_K;
  const int from = __builtin_amdgcn_readfirstlane((unsigned)k_blocks * range / p.ranges);  // (fewer than 2^16 of either)
  const int to = __builtin_amdgcn_readfirstlane((unsigned)k_blocks * (range + 1) / p.ranges);
  const int lane = threadIdx.x % NS_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / NS_WAVE), r = lane % 16, g = lane / 16;
  // blocks of rows that there are; those beyond are the last, their sums are not written
  const int high = min(MI, (p.M + 15) / 16 - mt * MI), wide = min(4 * NJ, (p.N + 15) / 16 - nt * 4 * NJ);

  // (the scales of x lie behind the parts)
  const auto xr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.parts + (size_t)mt * MI * k_blocks * 2 * SPLIT_BLOCK), 0, 0xffffffff, 0x00020000);
  const auto ir = __builtin_amdgcn_make_buffer_rsrc((void*)(p.parts + (size_t)((p.M + 15) / 16) * k_blocks * 2 * SPLIT_BLOCK + (size_t)mt * MI * k_blocks * 32), 0, 0xffffffff, 0x00020000);
  const auto wr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.w_parts + (size_t)nt * 4 * NJ * k_blocks * 2 * SPLIT_BLOCK), 0, 0xffffffff, 0x00020000);
  int xo[XPARTS], wo[NJ];  // bytes to what this wave loads (of x block b / 2, part b % 2; a wave that has none left the last once more, so that all wait for as many)
#pragma unroll
  for (int q = 0; q < XPARTS; ++q) {
    const int b = min(q * 4 + wave, 2 * MI - 1);
    xo[q] = (min(b / 2, high - 1) * k_blocks * 2 + b % 2) * (2 * SPLIT_BLOCK);
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) wo[j] = min(wave * NJ + j, wide - 1) * k_blocks * (4 * SPLIT_BLOCK);
  const int io = min(lane / 4, high - 1) * k_blocks * 64 + lane % 4 * 16;

  f16x8 b[SPLIT_STAGES][NJ][2];
  auto load = [&](int at, int kb) {
#pragma unroll
    for (int q = 0; q < XPARTS; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_ptr)(lds + at * STAGE + min(q * 4 + wave, 2 * MI - 1) * SPLIT_BLOCK), 16, lane * 16, xo[q] + kb * (4 * SPLIT_BLOCK), 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(ir, (lds_ptr)(lds + at * STAGE + 2 * MI * SPLIT_BLOCK), 16, io, kb * 64, 0, 0);  // (the same from every wave)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int q = 0; q < 2; ++q)
        b[at][j][q] = __builtin_bit_cast(f16x8, __builtin_amdgcn_raw_buffer_load_b128(wr, lane * 16, wo[j] + kb * (4 * SPLIT_BLOCK) + q * (2 * SPLIT_BLOCK), 0));
  };

  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = zero;

  auto stage = [&](int at, int kb) {
    // this stage has come, and every wave is done with the one before it, whose place the next but one is given (behind the last stage: that once more, not used)
    TILE_WAIT_LOADS(LOADS);
    TILE_BARRIER();
    load((at + 2) % SPLIT_STAGES, min(kb + 2, to - 1));
    __builtin_amdgcn_sched_barrier(0);
    f16x8 a[2][2];
    float inverse[2];
    auto read_x = [&](int i) {
#pragma unroll
      for (int q = 0; q < 2; ++q) a[i % 2][q] = *reinterpret_cast<const f16x8*>(lds + at * STAGE + (i * 2 + q) * SPLIT_BLOCK + lane * 8);
      inverse[i % 2] = reinterpret_cast<const float*>(lds + at * STAGE + 2 * MI * SPLIT_BLOCK)[i * 16 + r];
    };
    read_x(0);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      if (i + 1 < MI) read_x(i + 1);  // (under the products of i)
      __builtin_amdgcn_sched_barrier(0);
      f32x4 sum[NJ];
      constexpr int OF_W[3] = {1, 0, 0}, OF_X[3] = {0, 1, 0};
#pragma unroll
      for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int j = 0; j < NJ; ++j) sum[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[at][j][OF_W[q]], a[i % 2][OF_X[q]], q ? sum[j] : zero, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][j][e] = fmaf(sum[j][e], inverse[i % 2], acc[i][j][e]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  load(0, from);
  load(1, min(from + 1, to - 1));
  int kb = from;
  for (; kb + 2 < to; kb += 3) stage(0, kb), stage(1, kb + 1), stage(2, kb + 2);
  if (kb < to) stage(0, kb);
  if (kb + 1 < to) stage(1, kb + 1);
  TILE_WAIT_LOADS(0);  // (what was fetched again behind the last stage must not come into another workgroup's LDS)

  // acc[i][j], lane 16 g + r: row 16 i + r of the tile, columns 16 j + 4 g .. + 3 of the wave's.  No number or an infinity, of the floats or of the sums on their way: the
  // parts do not stand for the floats there, and the sum is taken from these.
  float* out = p.out + (size_t)range * p.M * p.N;
  const bool whole = p.N % 4 == 0 && p.out_stride % 4 == 0 && ((uintptr_t)out & 15) == 0;
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int m = m0 + 16 * i + r;
    if (m >= p.M) continue;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int n = n0 + 16 * (wave * NJ + j) + 4 * g;
      if (n >= p.N) continue;
      f32x4 v = acc[i][j];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = ldexpf(v[e], 127 + 15 - (int)(__builtin_bit_cast(unsigned, p.w_scales[min(n + e, p.N - 1)]) >> 23));
        if (n + e < p.N && !(fabsf(v[e]) < INFINITY))
          v[e] = split_plain(p.x + (size_t)m * p.x_stride + from * SPLIT_K, p.w + (size_t)(n + e) * p.K + from * SPLIT_K, (to - from) * SPLIT_K);
      }
      float* at = out + (size_t)m * p.out_stride + n;
      if (whole)
        *reinterpret_cast<f32x4*>(at) = v;
      else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < p.N) at[e] = v[e];
      }
    }
  }
#endif
}

template <int MI>
static int launch_split(SplitParams p, hipStream_t stream) {
  p.m_tiles = (p.M + 16 * MI - 1) / (16 * MI), p.n_tiles = (p.N + 64 * SPLIT_COLUMNS - 1) / (64 * SPLIT_COLUMNS);
  const long blocks = (long)p.m_tiles * ((p.n_tiles + 7) / 8 * 8);
  if (blocks > (1 << 22)) return NS_ERR_UNSUPPORTED;
  gemm_split_kernel<MI><<<dim3((unsigned)blocks, p.ranges), 256, 0, stream>>>(p);
  return ns_launch_status();
}

// parts: float16, 2 K values for each of M rows rounded up to 16, and without ``scales`` (null) K / 16 more.  K a multiple of 32, x_stride of 4, both on 16 bytes.
extern "C" int ns_split_rows(void* parts, const void* x, const void* scales, int M, int K, int x_stride, hipStream_t stream) {
  if (M <= 0 || K <= 0 || x_stride < K) return NS_ERR_BAD_ARG;
  if (K % SPLIT_K || x_stride % 4 || (((uintptr_t)x | (uintptr_t)parts) & 15) || (M + 15) / 16 > 65535) return NS_ERR_UNSUPPORTED;
  split_rows_kernel<<<dim3((K / SPLIT_K + 3) / 4, (M + 15) / 16), 256, 0, stream>>>((_Float16*)parts, (const float*)x, (const float*)scales, M, K, x_stride);
  return ns_launch_status();
}

// scales: a float for each of N rows.  w [N, K] without gaps on 16 bytes, K a multiple of 4.
extern "C" int ns_split_scales(void* scales, const void* w, int N, int K, hipStream_t stream) {
  if (N <= 0 || K <= 0) return NS_ERR_BAD_ARG;
  if (K % 4 || ((uintptr_t)w & 15)) return NS_ERR_UNSUPPORTED;
  split_scales_kernel<<<(N + 3) / 4, 256, 0, stream>>>((float*)scales, (const float*)w, N, K);
  return ns_launch_status();
}

// ``parts``: of ``x`` by ns_split_rows without scales; ``w_parts``: of ``w`` by ns_split_rows with ``w_scales``, those by ns_split_scales.  ``rows``: of a tile,
// 64, 96, 112 or 128.  ``ranges`` of K above 1: out is [ranges][M][N] (out_stride N), the sums of each.
// K a multiple of 32 below 2^19 (a tile's parts within 31 bits of bytes), x_stride of 4; x, w and parts on 16 bytes.
extern "C" int ns_gemm_split(void* out, const void* parts, const void* w_parts, const void* x, const void* w, const void* w_scales, int M, int N, int K, int x_stride,
                             int out_stride, int rows, int ranges, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0 || x_stride < K || out_stride < N || ranges < 1 || (ranges > 1 && out_stride != N)) return NS_ERR_BAD_ARG;
  if (K % SPLIT_K || x_stride % 4 || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)parts | (uintptr_t)w_parts) & 15) || K >= 1 << 19 || ranges > K / SPLIT_K)
    return NS_ERR_UNSUPPORTED;
  const SplitParams p{(float*)out, (const _Float16*)parts, (const _Float16*)w_parts, (const float*)x, (const float*)w, (const float*)w_scales, M, N, K, x_stride, out_stride, 0, 0, ranges};
  switch (rows) {
    case 64: return launch_split<4>(p, stream);
    case 96: return launch_split<6>(p, stream);
    case 112: return launch_split<7>(p, stream);
    case 128: return launch_split<8>(p, stream);
  }
  return NS_ERR_BAD_ARG;
}

// Products of many 32-bit rows on the bfloat16 matrix cores, out[m][n] = sum_k x[m][k] w[n][k], in less than half of the 32-bit ones' time and nearer to 64 bits.
// (reference: the nn.Linear calls of model/llama.py:175,184,195)
//
// A float is the sum of three bfloat16 values, a = a0 + a1 + a2, each the nearest to what the ones before it leave: |a1| <= 2^-8 |a|, |a2| <= 2^-17 |a|.  Of the nine
// products of two such sums six are taken, the smallest first: a2 b0, a0 b2, a1 b1, a1 b0, a0 b1, a0 b0; those left out are 2^-24 of a b at most together, and a product of two
// bfloat16 values is exact in 32 bits.  The matrix instruction adds up blocks of 8 k and rounds each sum to nearest, so six of them over a stage of 32 k
// begin at zero and the vector unit adds what they give to the sums: over a whole K of 2,048 in one chain the error is 7.1e-7 instead.
// Error against 64 bits (2-norm, both operands normal): K 2,048 1.6e-7, K 8,192 3.1e-7, of the 32-bit instruction's four chains (gemm_generic.hip) 4.1e-7 and 8.1e-7; all of
// one sign, K 8,192: 1.6e-7 and 3.3e-7; x spread over twelve powers of two: 2.3e-7 and 8.0e-7.
//
// x is split ahead (it is read by every tile of w, and small), w in registers on its way (it would take half as much memory again and more time to read): each wave
// owns columns of its own over all rows of the tile, so a piece of w is split once a tile, and a part of x comes from LDS once a wave.  us, the 32-bit instruction
// and this with the splitting of x and the sum of ranges of K, alone and a call beside two others: 777 rows, N 16,384, K 2,048 446 / 423 and 275 / 239 (219 TFLOP/s of products of
// 32 bits, 1.3 PFLOP/s of the matrix unit), N 2,048, K 8,192 254 / 227 and 171 / 133, N 3,072, K 2,048 95 / 85 and 77 / 56; 2,048 rows of 28,672 x 4,096 3,605 / 3,585 and 2,087 / 2,132.
// Bound by the matrix unit for 60% of the time, the clock sinking to 2.0 GHz under it; the sums in the vector unit are 7% of the rest, the loads of x and w 8% each.
#include "common.h"
#include "lds_loads.h"

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((__vector_size__(4 * sizeof(float))));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;

#define SPLIT_K 32       // k of a stage
#define SPLIT_BLOCK 512  // values of a block: 16 rows of a stage
#define SPLIT_COLUMNS 2  // blocks of 16 rows of w a wave: with four, two workgroups a compute unit instead of three (252 us of the 239 above)

union Operand {  // of the matrix instruction: eight values, made two at a time
  bf16x8 v;
  bf16x2 pair[4];
};

// Eight floats into their three parts.
__device__ __forceinline__ void split_eight(const f32x4& low, const f32x4& high, Operand* part) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const f32x4& of = e < 2 ? low : high;
    f32x2 v = {of[e % 2 * 2], of[e % 2 * 2 + 1]};
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      part[p].pair[e] = __builtin_convertvector(v, bf16x2);
      const unsigned bits = __builtin_bit_cast(unsigned, part[p].pair[e]);
      v = f32x2{v[0] - __builtin_bit_cast(float, bits << 16), v[1] - __builtin_bit_cast(float, bits & 0xffff0000u)};  // (exact)
    }
  }
}

// x [M, K] as parts[block of 16 rows][block of 32 k][part][lane][8], where lane 16 g + r holds of row r the k 4 g .. 4 g + 3 and 16 + 4 g .. 16 + 4 g + 3 of the
// block: an operand of the matrix instruction as it lies in registers, so that any three blocks are three contiguous KB.  (A lane's two loads of w then lie beside
// those of the lanes of the same row, 64 bytes an instruction.)  Rows beyond the last are zeros.
__global__ __launch_bounds__(256) void split_rows_kernel(bf16_t* __restrict__ parts, const float* __restrict__ x, int M, int K, int x_stride) {
  const int k_blocks = K / SPLIT_K, lane = threadIdx.x % NS_WAVE, r = lane % 16, g = lane / 16;
  const int kb = blockIdx.x * 4 + threadIdx.x / NS_WAVE, mb = blockIdx.y, row = mb * 16 + r;
  if (kb >= k_blocks) return;
  f32x4 low = {0.f, 0.f, 0.f, 0.f}, high = low;
  if (row < M) {
    const float* at = x + (size_t)row * x_stride + kb * SPLIT_K + 4 * g;
    low = *reinterpret_cast<const f32x4*>(at), high = *reinterpret_cast<const f32x4*>(at + 16);
  }
  Operand part[3];
  split_eight(low, high, part);
  bf16x8* to = reinterpret_cast<bf16x8*>(parts + ((size_t)mb * k_blocks + kb) * 3 * SPLIT_BLOCK) + lane;
#pragma unroll
  for (int p = 0; p < 3; ++p) to[p * NS_WAVE] = part[p].v;
}

struct SplitParams {
  float* out;  // [M, N], or with ranges of K [ranges][M][N]
  const bf16_t* parts;
  const float *x, *w;
  int M, N, K, x_stride, out_stride, m_tiles, n_tiles, ranges;
};

// One output as one chain over k in 32 bits.
__device__ __attribute__((noinline)) float split_plain(const float* a, const float* b, int k) {
  float s = 0.f;
  for (int i = 0; i < k; i += 4) {
    const f32x4 u = *reinterpret_cast<const f32x4*>(a + i), v = *reinterpret_cast<const f32x4*>(b + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) s = fmaf(u[e], v[e], s);
  }
  return s;
}

// Four waves, 16 MI rows of x by 128 of w.  A stage of x's parts lies in LDS while the next is on its way, and w's next in registers.
template <int MI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void gemm_split_kernel(const SplitParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(3))) void* lds_ptr;
  constexpr int NJ = SPLIT_COLUMNS, TM = 16 * MI, TN = 64 * NJ, STAGE = 3 * MI * SPLIT_BLOCK;
  __shared__ __attribute__((aligned(16))) bf16_t lds[2 * STAGE];
  // an XCD (workgroups go to the eight in launch order) takes every eighth tile of w and all tiles of x against it one after the other
  const int xcd = blockIdx.x & 7, turn = blockIdx.x >> 3, range = blockIdx.y;
  const int nt = (turn / p.m_tiles) * 8 + xcd, mt = turn % p.m_tiles;
  if (nt >= p.n_tiles) return;
  const int m0 = mt * TM, n0 = nt * TN, k_blocks = p.K / SPLIT_K;
  const int from = (int)((long)k_blocks * range / p.ranges), to = (int)((long)k_blocks * (range + 1) / p.ranges);
  const int lane = threadIdx.x % NS_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / NS_WAVE), r = lane % 16, g = lane / 16;
  const int high = min(MI, (p.M + 15) / 16 - mt * MI);  // blocks of rows that there are; those beyond are the last, their sums are not written

  const bf16_t* xs = p.parts + (size_t)mt * MI * k_blocks * 3 * SPLIT_BLOCK + lane * 8;
  const auto wr = __builtin_amdgcn_make_buffer_rsrc((void*)(p.w + (size_t)n0 * p.K), 0, 0xffffffff, 0x00020000);
  int wo[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) wo[j] = 4 * (min((wave * NJ + j) * 16 + r, p.N - 1 - n0) * p.K + 4 * g);

  auto load_x = [&](int buf, int kb) {
#pragma unroll
    for (int q = 0; q < (3 * MI + 3) / 4; ++q) {
      const int b = q * 4 + wave;  // block b / 3, part b % 3
      if (b < 3 * MI)
        __builtin_amdgcn_global_load_lds(xs + (((size_t)min(b / 3, high - 1) * k_blocks + kb) * 3 + b % 3) * SPLIT_BLOCK,
                                         (lds_ptr)(lds + buf * STAGE + b * SPLIT_BLOCK), 16, 0, 0);
    }
  };
  f32x4 raw[NJ][2];
  auto load_w = [&](int kb) {
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        raw[j][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, wo[j], kb * (4 * SPLIT_K) + 64 * h, 0));
  };

  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = zero;

  load_x(0, from);
  load_w(from);
  for (int kb = from; kb < to; ++kb) {
    const int buf = (kb - from) & 1, next = min(kb + 1, to - 1);  // (behind the last stage: it once more, not used)
    // this stage has come, and every wave is done with the one before it, whose place the next is given
    TILE_WAIT_LOADS(0);
    TILE_BARRIER();
    Operand part[NJ][3];
#pragma unroll
    for (int j = 0; j < NJ; ++j) split_eight(raw[j][0], raw[j][1], part[j]);
    load_x(buf ^ 1, next);
    load_w(next);
    __builtin_amdgcn_sched_barrier(0);
    bf16x8 a[2][3];
    auto read_x = [&](int i) {
#pragma unroll
      for (int q = 0; q < 3; ++q) a[i % 2][q] = *reinterpret_cast<const bf16x8*>(lds + buf * STAGE + (i * 3 + q) * SPLIT_BLOCK + lane * 8);
    };
    read_x(0);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      if (i + 1 < MI) read_x(i + 1);  // (under the products of i: 239 us of the first line, read where they are wanted 253)
      __builtin_amdgcn_sched_barrier(0);
      f32x4 sum[NJ];
      constexpr int OF_W[6] = {2, 0, 1, 1, 0, 0}, OF_X[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int j = 0; j < NJ; ++j) sum[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(part[j][OF_W[q]].v, a[i % 2][OF_X[q]], q ? sum[j] : zero, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] += sum[j];
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  TILE_WAIT_LOADS(0);  // (what was fetched again behind the last stage must not come into another workgroup's LDS)

  // acc[i][j], lane 16 g + r: row 16 i + r of the tile, columns 16 j + 4 g .. + 3 of the wave's.  No number, an infinity, or so small that parts of the operands may lie
  // below what bfloat16 holds: there the parts do not stand for the floats, and the sum is taken from these.
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
        const float size = fabsf(v[e]);
        if (n + e < p.N && !(size < INFINITY && (size >= 0x1p-80f || size == 0.f)))
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

// parts: bfloat16, 3 K values for each of M rows rounded up to 16.  K a multiple of 32, x_stride of 4, both on 16 bytes.
extern "C" int ns_split_rows(void* parts, const void* x, int M, int K, int x_stride, hipStream_t stream) {
  if (M <= 0 || K <= 0 || x_stride < K) return NS_ERR_BAD_ARG;
  if (K % SPLIT_K || x_stride % 4 || (((uintptr_t)x | (uintptr_t)parts) & 15) || (M + 15) / 16 > 65535) return NS_ERR_UNSUPPORTED;
  split_rows_kernel<<<dim3((K / SPLIT_K + 3) / 4, (M + 15) / 16), 256, 0, stream>>>((bf16_t*)parts, (const float*)x, M, K, x_stride);
  return ns_launch_status();
}

// ``parts``: of ``x`` by ns_split_rows.  ``rows``: of a tile, 64, 96, 112 or 128.  ``ranges`` of K above 1: out is [ranges][M][N] (out_stride N), the sums of each.
// K a multiple of 32 below 2^21 (a tile's rows of w within 31 bits of bytes), x_stride of 4; x, w and parts on 16 bytes.
extern "C" int ns_gemm_split(void* out, const void* parts, const void* x, const void* w, int M, int N, int K, int x_stride, int out_stride, int rows,
                             int ranges, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0 || x_stride < K || out_stride < N || ranges < 1 || (ranges > 1 && out_stride != N)) return NS_ERR_BAD_ARG;
  if (K % SPLIT_K || x_stride % 4 || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)parts) & 15) || K >= 1 << 21 || ranges > K / SPLIT_K || ranges > 65535)
    return NS_ERR_UNSUPPORTED;
  const SplitParams p{(float*)out, (const bf16_t*)parts, (const float*)x, (const float*)w, M, N, K, x_stride, out_stride, 0, 0, ranges};
  switch (rows) {
    case 64: return launch_split<4>(p, stream);
    case 96: return launch_split<6>(p, stream);
    case 112: return launch_split<7>(p, stream);
    case 128: return launch_split<8>(p, stream);
  }
  return NS_ERR_BAD_ARG;
}

// Products of many 32-bit rows on the float16 matrix cores, out[m][n] = sum_k x[m][k] w[n][k], in less than half of the 32-bit ones' time and nearer to 64 bits.
// (reference: the nn.Linear calls of model/llama.py:175,184,195)
//
// A float times a power of two, its largest neighbour brought to 2^14 to 2^15, is a0 + 2^-11 a1 of two float16 values, each the nearest to what is left: 2^-23 |a| at most is lost.  (The second
// at 2^11 times its size has the float16 range to itself: a value keeps its bits down to 2^-28 of the largest; at its own size down to 2^-17.)  Powers of two are chosen for each 32 k
// of a row of x, and for each row of w.  Of the four products of two such sums three are taken, a1 b0 + a0 b1 in a sum of their own and a0 b0; the one left out is 2^-22 of a b at most, and its
// sign is any.  A product of two float16 values is exact in 32 bits.  The matrix instruction adds up blocks of 8 k and rounds each sum to nearest, so those of a stage of 32 k begin at
// zero and the vector unit adds what they give to the sums, times the power of two of x.
// What the parts do not hold is counted where a block is split: values too small beside the largest, which are all that counts where that meets zeros; infinities; blocks whose products could
// leave the range of 32 bits on their way.  A row of x or of w that has two such values, or one that is not even held to 2^-18, is given to the 32-bit instruction by a launch behind the
// product (``split_mend_kernel``).  A single one, 10^-8 of its block's largest or less, is one in 10^8 normal values, and every product of a few million would have a row that goes that way for
// it; two are one row of K 2,048 in 10^9.  (A row that has a value that is no number is none whatever is done with it.)
// K is cut into segments, four or one by the matrix's sizes, whose sums are added in order, by one workgroup or from one each: an output is the same whatever the tile and the rows beside it.
// Error against 64 bits (2-norm), the 32-bit instruction's four chains (gemm_generic.hip) and this in four segments and one, K 2,048, and the first two at K 8,192: both operands normal 4.1e-7, 1.3e-7,
// 1.7e-7, 8.1e-7, 1.8e-7; all of one sign 1.8e-7, 0.5e-7, 1.3e-7, 3.5e-7, 0.7e-7; x spread over 16 powers of two 4.1e-7, 1.4e-7, 1.8e-7, 8.1e-7, 2.2e-7; one k of 512 10^5 times the others 4.6e-7,
// 1.5e-7, 1.9e-7, 8.3e-7, 2.3e-7, and against zeros in w 4.1e-7, 1.3e-7, 1.7e-7, 8.1e-7, 2.0e-7.  Behind the 32-bit instruction only where a row is zeros but for one k of 32, 1.1e-7, 1.2e-7, 1.7e-7,
// 2.1e-7, 1.7e-7, or but for one, none and 0.5e-7.
// (Three bfloat16 values for a float, six products: 1.6e-7 and 3.1e-7 for normal operands, and twice the work of the matrix unit.)
//
// Both operands are split ahead, w once for all (as many bytes again as it has), x a call.  w split in registers on its way by every tile of x instead: 211 us for 177 in the first size below beside two others.
// x comes through LDS, where the four waves share it, and each wave's own columns of w straight into the registers of the matrix instruction, both two stages ahead (one: tiles that have a
// compute unit to themselves 1.2 times as long).  us, the 32-bit instruction and this with the splitting of x and the sum of ranges of K, alone / a call beside two others:
// 832 rows, N 16,384, K 2,048 536 / 511 and 217 / 175 (315 TFLOP/s of products of 32 bits), N 2,048, K 8,192 307 / 272 and 133 / 108, N 3,072, K 2,048 96 / 89 and 71 / 40;
// 2,048 rows of 28,672 x 4,096 3,649 / 3,727 and 1,340 / 1,402.  The lower products in a sum of their own are twice the work of the vector unit: 1,273 us alone before for the last, 1,330 now, 2,048 rows of
// 4,096 x 14,336, two tiles a compute unit, 662 and 750; taken to the sums under the products of the next block it is hidden in the smaller ones.
// Bound by the power of the matrix unit: at the last size it works for 69% of the cycles and the clock sinks to 1.4 GHz.
#include "common.h"
#include "lds_loads.h"
#include <type_traits>

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((__vector_size__(4 * sizeof(float))));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

#define SPLIT_K 32       // k of a stage
#define SPLIT_BLOCK 512  // values of a block: 16 rows of a stage
#define SPLIT_COLUMNS 2  // blocks of 16 rows of w a wave: with four, 112 rows of x a tile and two workgroups a compute unit instead of three, 173 us for 177 in the first size above beside two others and 49 for 35 in the third
// Sums are kept 2^40 times what they are with a row's largest of w brought to 1/2 to 1.  With the largest of a block from 2^-64 to 2^68 that is 2^127 at most for K below 2^19, and the product
// of the smallest values that parts hold, 2^-50 of their largest, is a normal number.
#define SPLIT_UP 25  // (2^40 over the 2^15 of w)
#define SPLIT_LEAST 0x1p-64f
#define SPLIT_MOST 0x1p68f
#define SPLIT_STAGES 3   // at hand: one that is multiplied and two on their way

#define SPLIT_LOST 2  // values of a row that the parts do not hold, from which on it goes to the 32-bit instruction
#define SPLIT_GROUP 4 // blocks of 32 k whose counts are one word, two bits for each of 16 rows

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

// Eight floats times a power of two into their two parts.  How many of them are not held to 2^-23 of themselves; two for one that is not held to 2^-18 or infinite.
__device__ __forceinline__ int split_eight(const f32x4& low, const f32x4& high, float scale, Operand* part) {
  int lost = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const f32x4& of = e < 2 ? low : high;
    const f32x2 v = {of[e % 2 * 2] * scale, of[e % 2 * 2 + 1] * scale};
    const f16x2 first = __builtin_convertvector(v, f16x2);
    const f32x2 left = {(v[0] - (float)first[0]) * 0x1p11f, (v[1] - (float)first[1]) * 0x1p11f};  // (exact)
    const f16x2 second = __builtin_convertvector(left, f16x2);
    part[0].pair[e] = first, part[1].pair[e] = second;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float raw = of[e % 2 * 2 + i], off = fabsf(left[i] - (float)second[i]), of_one = fabsf(v[i]);
      const bool far = !(off <= 0x1p-7f * of_one) || (of_one == 0.f && raw != 0.f);
      lost += raw != raw ? 0 : far ? 2 : off > 0x1p-12f * of_one;
    }
  }
  return lost;
}
// The same of a block of 32 k, by the four lanes that have it, no more than 2.
__device__ __forceinline__ int lost_in(int lost) {
  lost += __shfl_xor(lost, 16), lost += __shfl_xor(lost, 32);
  return min(lost, 2);
}
__device__ __forceinline__ bool out_of_range(float largest) { return largest != 0.f && !(largest >= SPLIT_LEAST && largest <= SPLIT_MOST); }

// x [M, K] as parts[block of 16 rows][block of 32 k][part][lane][8], where lane 16 g + r holds of row r the k 8 g .. 8 g + 7 of the block: an operand of the matrix
// instruction as it lies in registers, so that any two blocks are two contiguous KB.  Rows beyond the last are zeros.
// ``w_scales`` (of w): a power of two a row.  Without them (of x) one a row and block, their inverses times 2^25 behind all parts, [block of 16 rows][block of 32 k][16].  lost[block of 16 rows][group
// of 128 k]: of row r in bits 2 r and 2 r + 1 how many values the parts do not hold, 2 for more; behind them ``call``, a number of the caller's, if any does (what lies there before may be anything).
// ``read_rows`` (or null): of the whole, of which x is the rows from ``first`` on, only so many count; the others are zeros, whatever lies there.  (A captured step's padding holds what
// earlier kernels left: taken as it is, its rows go to the 32-bit instruction, 45 us a layer in a prompt of 777 tokens that runs in 832.)
__global__ __launch_bounds__(256) void split_rows_kernel(_Float16* __restrict__ parts, const float* __restrict__ x, const float* __restrict__ w_scales, unsigned* __restrict__ lost, unsigned call,
                                                         const int* __restrict__ read_rows, int first, int M, int K, int x_stride) {
  __shared__ unsigned counts[SPLIT_GROUP][16];
  const int k_blocks = K / SPLIT_K, lane = threadIdx.x % NS_WAVE, wave = threadIdx.x / NS_WAVE, r = lane % 16, g = lane / 16;
  const int kb = blockIdx.x * SPLIT_GROUP + wave, mb = blockIdx.y, row = mb * 16 + r;
  if (read_rows) M = min(M, *read_rows - first);  // (then none of this workgroup may be left: its parts are zeros all the same)
  int count = 0;
  if (kb < k_blocks) {
    f32x4 low = {0.f, 0.f, 0.f, 0.f}, high = low;
    if (row < M) {
      const float* at = x + (size_t)row * x_stride + kb * SPLIT_K + 8 * g;
      low = *reinterpret_cast<const f32x4*>(at), high = *reinterpret_cast<const f32x4*>(at + 4);
    }
    const size_t block = (size_t)mb * k_blocks + kb;
    float scale = 1.f;
    if (w_scales) {
      if (row < M) scale = w_scales[row];
    } else {
      float largest = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) largest = fmaxf(largest, fmaxf(fabsf(low[e]), fabsf(high[e])));
      largest = fmaxf(largest, __shfl_xor(largest, 16)), largest = fmaxf(largest, __shfl_xor(largest, 32));
      scale = split_scale(largest);
      count = out_of_range(largest) ? SPLIT_LOST : 0;
      if (g == 0) reinterpret_cast<float*>(parts + (size_t)gridDim.y * k_blocks * 2 * SPLIT_BLOCK)[block * 16 + r] = inverse_scale(scale) * (float)(1 << SPLIT_UP);
    }
    Operand part[2];
    count += split_eight(low, high, scale, part);
    count += __shfl_xor(count, 16), count += __shfl_xor(count, 32);
    f16x8* to = reinterpret_cast<f16x8*>(parts + block * 2 * SPLIT_BLOCK) + lane;
#pragma unroll
    for (int p = 0; p < 2; ++p) to[p * NS_WAVE] = part[p].v;
  }
  if (g == 0) counts[wave][r] = count;
  __syncthreads();
  if (wave == 0) {
    count = 0;
#pragma unroll
    for (int i = 0; i < SPLIT_GROUP; ++i) count += counts[i][r];
    unsigned word = (unsigned)min(count, SPLIT_LOST) << 2 * r;
#pragma unroll
    for (int d = 1; d < 16; d *= 2) word |= __shfl_xor(word, d);
    if (lane == 0) {
      lost[(size_t)mb * gridDim.x + blockIdx.x] = word;
      if (word) lost[(size_t)gridDim.y * gridDim.x] = call;
    }
  }
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

// The blocks of 16 rows that have a row to mend: list[0] how many, then for each its number and the rows as bits, from the counts of ``lost`` [blocks][groups].  By all threads of a workgroup (1,024 at most).
// In the order of the blocks: every workgroup of split_mend_kernel makes the list for itself and takes its items by their places there.
__device__ __forceinline__ void list_lost(int* list, const unsigned* lost, int blocks, int groups) {
  __shared__ int found[16];  // by each wave
  const int lane = threadIdx.x % NS_WAVE, wave = threadIdx.x / NS_WAVE;
  if (threadIdx.x == 0) list[0] = 0;
  unsigned any = 0;
  for (size_t i = threadIdx.x; i < (size_t)blocks * groups; i += blockDim.x) any |= lost[i];
  if (!__syncthreads_or(any)) return;  // (all of the workgroup)
  int count = 0;
  for (int from = 0; from < blocks; from += blockDim.x) {
    const int b = from + threadIdx.x;
    unsigned more = 0, once = 0;  // (bits 2 r: rows with two, rows with one so far)
    for (int i = 0; b < blocks && i < groups; ++i) {
      const unsigned word = lost[(size_t)b * groups + i], one = word & 0x55555555u, two = word >> 1 & 0x55555555u;
      more |= two | (once & one), once |= one;
    }
    const unsigned long long with = __ballot(more != 0);
    if (lane == 0) found[wave] = __popcll(with);
    __syncthreads();
    int at = count + __popcll(with & ((1ull << lane) - 1));
    for (int i = 0; i < (int)blockDim.x / NS_WAVE; ++i) at += i < wave ? found[i] : 0, count += found[i];
    if (more) {
      int rows = 0;
      for (int r = 0; r < 16; ++r) rows |= (int)(more >> 2 * r & 1) << r;
      list[1 + 2 * at] = b, list[2 + 2 * at] = rows;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) list[0] = count;
  __syncthreads();
}
__global__ __launch_bounds__(1024) void split_list_kernel(int* __restrict__ list, const unsigned* __restrict__ lost, int blocks, int groups) { list_lost(list, lost, blocks, groups); }

struct SplitParams {
  float* out;  // [M, N], or with ranges of K [ranges][M][N]
  const _Float16 *parts, *w_parts;
  const float* w_scales;
  int M, N, K, out_stride, m_tiles, n_tiles, segments, ranges;
};

// Four waves, 16 MI rows of x by 128 of w.  A stage's parts of x lie in LDS and those of w in the registers of the wave whose columns they are, and the next two are on their way.
// SUMMED: of all segments, one after the other; else of segment blockIdx.y.
template <int MI, bool SUMMED>
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
  f32x4 acc[MI][NJ], total[MI][NJ];
  int to = 0;
  // ``behind``: loads of the next stage, which are on their way behind this one's.  The last stage but one fetches its next but one for nothing, and the compiler drops what goes to registers of that: the last waits until
  // no more than the others are left.
  typedef std::integral_constant<int, LOADS> Whole;
  typedef std::integral_constant<int, XPARTS + 1> ToLds;
  auto stage = [&](int at, int kb, auto behind) {
    // this stage has come, and every wave is done with the one before it, whose place the next but one is given (behind the last stage: that once more, not used)
    TILE_WAIT_LOADS(decltype(behind)::value);
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
    f32x4 low[2][NJ], sum[2][NJ];
    float scale[2];
    auto join = [&](int i) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][j][e] = fmaf(fmaf(low[i % 2][j][e], 0x1p-11f, sum[i % 2][j][e]), scale[i % 2], acc[i][j][e]);
    };
    read_x(0);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      if (i + 1 < MI) read_x(i + 1);  // (under the products of i)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NJ; ++j) low[i % 2][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[at][j][1], a[i % 2][0], zero, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NJ; ++j) low[i % 2][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[at][j][0], a[i % 2][1], low[i % 2][j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NJ; ++j) sum[i % 2][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[at][j][0], a[i % 2][0], zero, 0, 0, 0);
      scale[i % 2] = inverse[i % 2];
      if (i > 0) join(i - 1);
      if (i > 0) {
#pragma unroll
        for (int q = 0; q < 3 * NJ; ++q) __builtin_amdgcn_sched_group_barrier(0x8, 1, 0), __builtin_amdgcn_sched_group_barrier(0x2, 4, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    join(MI - 1);
    __builtin_amdgcn_sched_barrier(0);
  };
  for (int s = 0; s < (SUMMED ? p.segments : 1); ++s) {
    const int segment = SUMMED ? s : range;
    int kb = __builtin_amdgcn_readfirstlane((unsigned)k_blocks * segment / p.segments);  // (fewer than 2^16 of either)
    to = __builtin_amdgcn_readfirstlane((unsigned)k_blocks * (segment + 1) / p.segments);
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = zero;
    if (s) TILE_BARRIER();  // (every wave is done with the segment before)
    load(0, kb);
    __builtin_amdgcn_sched_barrier(0);  // (in this order: the waits count loads)
    load(1, min(kb + 1, to - 1));
    __builtin_amdgcn_sched_barrier(0);
    for (; kb + 2 < to; kb += 3) stage(0, kb, Whole()), stage(1, kb + 1, Whole()), stage(2, kb + 2, Whole());
    if (kb < to) stage(0, kb, Whole());
    if (kb + 1 < to) stage(1, kb + 1, ToLds());
    TILE_WAIT_LOADS(0);  // (what was fetched again behind the last stage must not come into another stage's LDS, or another workgroup's)
    if (SUMMED) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) total[i][j] = s ? total[i][j] + acc[i][j] : acc[i][j];
    }
  }

  // acc[i][j], lane 16 g + r: row 16 i + r of the tile, columns 16 j + 4 g .. + 3 of the wave's
  float* out = p.out + (size_t)range * p.M * p.N;
  const bool whole = p.N % 4 == 0 && p.out_stride % 4 == 0 && ((uintptr_t)out & 15) == 0;
  int down[NJ][4];  // the power of two that sums are taken times
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) down[j][e] = 127 - SPLIT_UP - (int)(__builtin_bit_cast(unsigned, p.w_scales[min(n0 + 16 * (wave * NJ + j) + 4 * g + e, p.N - 1)]) >> 23);
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int m = m0 + 16 * i + r;
    if (m >= p.M) continue;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int n = n0 + 16 * (wave * NJ + j) + 4 * g;
      if (n >= p.N) continue;
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = ldexpf((SUMMED ? total : acc)[i][j][e], down[j][e]);
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
  if (p.ranges == 1 && p.segments > 1)
    gemm_split_kernel<MI, true><<<(unsigned)blocks, 256, 0, stream>>>(p);
  else
    gemm_split_kernel<MI, false><<<dim3((unsigned)blocks, p.ranges), 256, 0, stream>>>(p);
  return ns_launch_status();
}

// The outputs of the rows of x and of w that the parts do not hold, by the 32-bit instruction from the floats, in gemm_f32_kernel's four chains (gemm_generic.hip): wave c adds up the k 16 c .. 16 c + 15
// of every 64, and the four sums are added as there.  None, as good as always: then the launch is all that this costs.  A few blocks of 16 rows: a workgroup takes one against 16 rows of the other
// operand, bound by the way of those from memory, hence 16 pieces on their way; many: four against 32, so that what comes from L2 is used more often.  One row of 832, N 16,384, K 2,048 40 us (its 134 MB of floats are read), N 2,048, K 8,192 40, N = K = 2,048 13;
// all 832 640, 390 and 107, where the 32-bit product alone takes 427, 246 and 69.
#define MEND_BLOCKS 256  // of 16 rows of x
#define MEND_MANY 8      // blocks from which on they go four at a time
#define MEND_GROUPS 512  // workgroups, two a compute unit
struct MendParams {
  float* out;
  const float *x, *w;
  const unsigned* lost;
  const int* w_list;
  int M, N, K, x_stride, out_stride;
  unsigned call;
};
struct MendBlock {  // of 16 rows, and those of them whose outputs are written whatever the other operand's
  int block, rows;
};

template <int MB, int NB, int AHEAD>
__device__ __forceinline__ void mend_tile(const MendParams& p, const MendBlock* of_x, const MendBlock* of_w, f32x4* sums) {
  const int lane = threadIdx.x % NS_WAVE, wave = threadIdx.x / NS_WAVE, r = lane % 16, g = lane / 16;
  const int k0 = 16 * wave, pieces = (p.K - k0 + 63) / 64;  // (K a multiple of 32: pieces are whole, and waves 2 and 3 may have one less)
  const float *a[MB], *b[NB];
  f32x4 u[AHEAD][MB], v[AHEAD][NB], chain[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i) a[i] = p.x + (size_t)min(of_x[i].block * 16 + r, p.M - 1) * p.x_stride + 4 * g;
#pragma unroll
  for (int j = 0; j < NB; ++j) b[j] = p.w + (size_t)min(of_w[j].block * 16 + r, p.N - 1) * p.K + 4 * g;
  auto load = [&](int at, int piece) {  // (behind the last piece K's last 16 once more, not used)
    const int k = min(k0 + 64 * piece, p.K - 16);
#pragma unroll
    for (int i = 0; i < MB; ++i) u[at][i] = *reinterpret_cast<const f32x4*>(a[i] + k);
#pragma unroll
    for (int j = 0; j < NB; ++j) v[at][j] = *reinterpret_cast<const f32x4*>(b[j] + k);
  };
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) chain[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < AHEAD; ++c) load(c, c);
  for (int piece = 0; piece < pieces; piece += AHEAD) {
#pragma unroll
    for (int c = 0; c < AHEAD; ++c) {
      if (piece + c < pieces) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) chain[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[c][j][e], u[c][i][e], chain[i][j], 0, 0, 0);
      }
      load(c, piece + c + AHEAD);
    }
  }
#pragma unroll
  for (int i = 0; i < MB * NB; ++i) sums[(wave * MB * NB + i) * NS_WAVE + lane] = chain[i / NB][i % NB];
  __syncthreads();
  // row r of x, row 4 g + e of w: a wave writes one e
#pragma unroll
  for (int i = 0; i < MB * NB; ++i) {
    const MendBlock x = of_x[i / NB], w = of_w[i % NB];
    const int m = x.block * 16 + r, n = w.block * 16 + 4 * g + wave;
    const f32x4* one = sums + i * NS_WAVE + lane;
    const float sum = (one[0][wave] + one[MB * NB * NS_WAVE][wave]) + (one[2 * MB * NB * NS_WAVE][wave] + one[3 * MB * NB * NS_WAVE][wave]);
    if (m < p.M && n < p.N && ((x.rows >> r | w.rows >> n % 16) & 1)) p.out[(size_t)m * p.out_stride + n] = sum;
  }
  __syncthreads();
}

// ``of_x``: the list is of blocks of x.
template <bool OF_X, int LISTED, int OTHER, int AHEAD>
__device__ __forceinline__ void mend_list(const MendParams& p, const int* list, int others, f32x4* sums) {
  const int groups = (others + OTHER - 1) / OTHER;
  const long items = (long)((list[0] + LISTED - 1) / LISTED) * groups;
  for (long item = blockIdx.x; item < items; item += gridDim.x) {
    MendBlock listed[LISTED], other[OTHER];
#pragma unroll
    for (int i = 0; i < LISTED; ++i) {  // (behind the last that once more)
      const int at = min((int)(item / groups) * LISTED + i, list[0] - 1);
      listed[i] = MendBlock{list[1 + 2 * at], list[2 + 2 * at]};
    }
#pragma unroll
    for (int i = 0; i < OTHER; ++i) other[i] = MendBlock{min((int)(item % groups) * OTHER + i, others - 1), 0};
    if constexpr (OF_X)
      mend_tile<LISTED, OTHER, AHEAD>(p, listed, other, sums);
    else
      mend_tile<OTHER, LISTED, AHEAD>(p, other, listed, sums);
  }
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void split_mend_kernel(const MendParams p) {
#if defined(__HIP_DEVICE_COMPILE__)
  __shared__ int list[1 + 2 * MEND_BLOCKS];
  __shared__ f32x4 sums[4 * 8 * NS_WAVE];
  const int m_blocks = (p.M + 15) / 16, n_blocks = (p.N + 15) / 16, groups = (p.K / SPLIT_K + SPLIT_GROUP - 1) / SPLIT_GROUP;
  if (p.lost[m_blocks * groups] == p.call) {
    list_lost(list, p.lost, m_blocks, groups);
    if (list[0] >= MEND_MANY)
      mend_list<true, 4, 2, 4>(p, list, n_blocks, sums);
    else
      mend_list<true, 1, 1, 16>(p, list, n_blocks, sums);
  }
  if (p.w_list[0] >= MEND_MANY)
    mend_list<false, 4, 2, 4>(p, p.w_list, m_blocks, sums);
  else if (p.w_list[0])
    mend_list<false, 1, 1, 16>(p, p.w_list, m_blocks, sums);
#endif
}

static int split_groups(int K) { return (K / SPLIT_K + SPLIT_GROUP - 1) / SPLIT_GROUP; }

// parts: float16, 2 K values for each of M rows rounded up to 16, and without ``w_scales`` (null) K / 16 more.  lost: a word for each 16 rows and each 128 k or what is left of them.  K a multiple of
// 32, x_stride of 4, both on 16 bytes.  ``lost`` has one word more, for ``call``: a number that differs from one call to the next over the same scratch (in a replay it is the same, and a word that an
// earlier replay left there only makes ns_split_mend look).
extern "C" int ns_split_rows(void* parts, void* lost, unsigned call, const void* x, const void* w_scales, const void* read_rows, int first, int M, int K, int x_stride,
                             hipStream_t stream) {
  if (M <= 0 || K <= 0 || x_stride < K) return NS_ERR_BAD_ARG;
  if (K % SPLIT_K || x_stride % 4 || (((uintptr_t)x | (uintptr_t)parts) & 15) || (M + 15) / 16 > 65535) return NS_ERR_UNSUPPORTED;
  split_rows_kernel<<<dim3(split_groups(K), (M + 15) / 16), NS_WAVE * SPLIT_GROUP, 0, stream>>>((_Float16*)parts, (const float*)x, (const float*)w_scales, (unsigned*)lost, call,
                                                                                               (const int*)read_rows, first, M, K, x_stride);
  return ns_launch_status();
}

// scales: a float for each of N rows.  w [N, K] without gaps on 16 bytes, K a multiple of 4.
extern "C" int ns_split_scales(void* scales, const void* w, int N, int K, hipStream_t stream) {
  if (N <= 0 || K <= 0) return NS_ERR_BAD_ARG;
  if (K % 4 || ((uintptr_t)w & 15)) return NS_ERR_UNSUPPORTED;
  split_scales_kernel<<<(N + 3) / 4, 256, 0, stream>>>((float*)scales, (const float*)w, N, K);
  return ns_launch_status();
}

// list: 1 and two words for each 16 of M rows, from what ns_split_rows counted of them.
extern "C" int ns_split_list(void* list, const void* lost, int M, int K, hipStream_t stream) {
  if (M <= 0 || K <= 0 || K % SPLIT_K) return NS_ERR_BAD_ARG;
  split_list_kernel<<<1, 1024, 0, stream>>>((int*)list, (const unsigned*)lost, (M + 15) / 16, split_groups(K));
  return ns_launch_status();
}

// ``parts``: of x by ns_split_rows without scales; ``w_parts``: of w by ns_split_rows with ``w_scales``, those by ns_split_scales.  ``rows``: of a tile,
// 64, 96, 112 or 128.  ``segments`` of K, by one workgroup after the other (``ranges`` 1) or by one each (as many): then out is [ranges][M][N] (out_stride N), the sums of each, to be added in order.
// K a multiple of 32 below 2^19 (a tile's parts within 31 bits of bytes), parts on 16 bytes.  What the parts do not hold is to be put right by ns_split_mend, behind the sum of the ranges.
extern "C" int ns_gemm_split(void* out, const void* parts, const void* w_parts, const void* w_scales, int M, int N, int K, int out_stride, int rows, int segments, int ranges,
                             hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0 || out_stride < N || segments < 1 || (ranges != 1 && ranges != segments) || (ranges > 1 && out_stride != N)) return NS_ERR_BAD_ARG;
  if (K % SPLIT_K || (((uintptr_t)parts | (uintptr_t)w_parts) & 15) || K >= 1 << 19 || segments > K / SPLIT_K) return NS_ERR_UNSUPPORTED;
  const SplitParams p{(float*)out, (const _Float16*)parts, (const _Float16*)w_parts, (const float*)w_scales, M, N, K, out_stride, 0, 0, segments, ranges};
  switch (rows) {
    case 64: return launch_split<4>(p, stream);
    case 96: return launch_split<6>(p, stream);
    case 112: return launch_split<7>(p, stream);
    case 128: return launch_split<8>(p, stream);
  }
  return NS_ERR_BAD_ARG;
}

// ``lost``, ``call``: of x by ns_split_rows; ``w_list``: of w by ns_split_list.  M at most 4,096; K a multiple of 32, x_stride of 4, x and w on 16 bytes.
extern "C" int ns_split_mend(void* out, const void* x, const void* w, const void* lost, unsigned call, const void* w_list, int M, int N, int K, int x_stride, int out_stride, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0 || x_stride < K || out_stride < N) return NS_ERR_BAD_ARG;
  if (M > 16 * MEND_BLOCKS || K % SPLIT_K || x_stride % 4 || (((uintptr_t)x | (uintptr_t)w) & 15)) return NS_ERR_UNSUPPORTED;
  const MendParams p{(float*)out, (const float*)x, (const float*)w, (const unsigned*)lost, (const int*)w_list, M, N, K, x_stride, out_stride, call};
  split_mend_kernel<<<MEND_GROUPS, 256, 0, stream>>>(p);
  return ns_launch_status();
}

// out[M, N] = x[M, K] . w[N, K]^T  with 32-bit accumulation in a fixed order, for any M, N, K.
//
// The products of the true 32-bit path, and the fall-back for shapes the bfloat16 matrix-core kernels refuse.  A row's
// result does not depend on which other rows share the launch.  Three kernels: a plain tiled one for any size and either
// type, whose outputs are each one chain of fused multiply-adds over k = 0..K-1; for 32-bit operands on whole 16-byte
// pieces one that reads w as fast as memory gives it (up to 8 rows) and one on the 32-bit matrix instructions (more rows).
// Which of the two is taken depends on the number of rows alone; their sums are ordered differently, so a token's 32-bit
// result as one of few rows and as one of many differ by rounding.
// (reference: the nn.Linear calls of model/llama.py:175,184,195,286)
#include "common.h"

#define GT_M 64
#define GT_N 64
#define GT_K 16

template <typename T, typename OutT>
__global__ __launch_bounds__(256) void gemm_generic_kernel(OutT* __restrict__ out, const T* __restrict__ x,
                                                            const T* __restrict__ w, int M, int N, int K, int x_stride,
                                                            int out_stride) {
  __shared__ float xs[GT_K][GT_M + 4];
  __shared__ float ws[GT_K][GT_N + 4];
  const int m0 = blockIdx.y * GT_M, n0 = blockIdx.x * GT_N;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;  // 16 x 16 threads, 4 x 4 outputs each
  float acc[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += GT_K) {
    // 64 rows x 16 k = 1024 elements per operand, 4 per thread; k is the fast index of a thread's loads
    for (int e = threadIdx.x; e < GT_M * GT_K; e += 256) {
      const int r = e / GT_K, kk = e % GT_K;
      const int m = m0 + r, n = n0 + r, k = k0 + kk;
      xs[kk][r] = (m < M && k < K) ? to_f(x[(size_t)m * x_stride + k]) : 0.f;
      ws[kk][r] = (n < N && k < K) ? to_f(w[(size_t)n * K + k]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < GT_K; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = xs[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = ws[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n < N) out[(size_t)m * out_stride + n] = (OutT)acc[i][j];
    }
  }
}

// Few rows (decode) in 32-bit: the work is reading w once.  A workgroup of eight waves owns ROWS_N rows of w and deals their
// K to its 512 lanes in units of four (16-byte loads, a wave's load a contiguous KiB of a row); every lane sums its own k in
// order for each of up to ROWS_M rows of x, the 64 partial sums of an output are added by a fixed butterfly that halves the
// values a lane holds at each step, and the eight waves' sums in LDS.  An output's value depends on its own row of x and of w
// only.  For K and the row strides multiples of 4 and 16-byte aligned operands.
// Bound by the loads: the waves of a workgroup share its rows of w, so each piece of x is read once for eight rows (once for
// four by a wave alone, over the whole of K, was bound by x coming from L2), and N = 2,048 still fills 256 compute units;
// two workgroups a unit, hence at most 128 registers (132 and one workgroup: 308 us in the last line).  Five rows:
//   N 2,048 K 2,048: 20 -> 8 us; N 2,048 K 8,192: 64 -> 19 us (3.5 TB/s); N 16,384 K 2,048: 38 -> 30 us (4.5 TB/s); N 128,256: 207 us
//   either way (5.1 TB/s)
#define ROWS_M 8
#define ROWS_N 8
#define ROWS_WAVES 8

// Sums of VALS (a power of two up to 64) values over the 64 lanes; lane l ends up with value l / (64 / VALS).
template <int VALS, int O = 32>
__device__ __forceinline__ float sum_over_lanes(float* v, int lane) {
  if constexpr (VALS > 1) {
    const bool upper = lane & O;
#pragma unroll
    for (int i = 0; i < VALS / 2; ++i) {
      const float give = upper ? v[i] : v[VALS / 2 + i], keep = upper ? v[VALS / 2 + i] : v[i];
      v[i] = keep + __shfl_xor(give, O, 64);
    }
    return sum_over_lanes<VALS / 2, O / 2>(v, lane);
  } else {
    float r = v[0];
#pragma unroll
    for (int o = O; o > 0; o >>= 1) r += __shfl_xor(r, o, 64);
    return r;
  }
}

template <int MT>  // rows of x that are summed for (a power of two; M of them count)
__global__ __launch_bounds__(64 * ROWS_WAVES, 4) void gemm_rows_f32_kernel(float* __restrict__ out, const float* __restrict__ x,
                                                                        const float* __restrict__ w, int M, int N, int K, int x_stride,
                                                                        int out_stride) {
  constexpr int VALS = ROWS_N * MT;
  __shared__ float part[ROWS_WAVES][VALS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n0 = blockIdx.x * ROWS_N;
  float acc[VALS];
#pragma unroll
  for (int i = 0; i < VALS; ++i) acc[i] = 0.f;
  const float4* wr[ROWS_N];
#pragma unroll
  for (int j = 0; j < ROWS_N; ++j) wr[j] = reinterpret_cast<const float4*>(w + (size_t)min(n0 + j, N - 1) * K);
  const int k4 = K / 4;
  for (int i = threadIdx.x; i < k4; i += 64 * ROWS_WAVES) {
    float4 wv[ROWS_N];
#pragma unroll
    for (int j = 0; j < ROWS_N; ++j) wv[j] = wr[j][i];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const float4 xv = reinterpret_cast<const float4*>(x + (size_t)min(m, M - 1) * x_stride)[i];
#pragma unroll
      for (int j = 0; j < ROWS_N; ++j) {
        float a = acc[j * MT + m];
        a = fmaf(xv.x, wv[j].x, a);
        a = fmaf(xv.y, wv[j].y, a);
        a = fmaf(xv.z, wv[j].z, a);
        a = fmaf(xv.w, wv[j].w, a);
        acc[j * MT + m] = a;
      }
    }
  }
  const float r = sum_over_lanes<VALS>(acc, lane);
  if (lane % (64 / VALS) == 0) part[wave][lane / (64 / VALS)] = r;
  __syncthreads();
  if (threadIdx.x < VALS) {
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < ROWS_WAVES; ++i) v += part[i][threadIdx.x];
    const int n = n0 + threadIdx.x / MT, m = threadIdx.x % MT;
    if (n < N && m < M) out[(size_t)m * out_stride + n] = v;
  }
}

// Many rows in 32-bit on the matrix cores (v_mfma_f32_16x16x4_f32, 32-bit products and sums: 157 TFLOP/s at the boost clock,
// the vector unit's own rate, but 2,048 operations an instruction and far fewer operand reads).  Bound by the matrix unit for many
// rows, by the latency of a workgroup's loads for few.  Against the tiled kernel above: 777 rows, N 16,384 K 2,048: 903 -> 512 us
// (102 TFLOP/s), N 2,048 K 8,192: 1,049 -> 283 us (92); 64 rows: 320 -> 51 and 1,201 -> 41 us; 9 rows: 263 -> 30 and 978 -> 33 us.
// Relative error (2-norm, against 64 bits) 4.1e-7 instead of 8.1e-7 at K 2,048, 8.1e-7 instead of 1.6e-6 at K 8,192: four chains for one.
// A workgroup of four waves owns TM rows of x and TN rows of w.  A stage is 64 k of both in LDS; wave i multiplies the k
// 16 i .. 16 i + 15 of every stage for the whole tile (so that a fragment from LDS serves as many instructions as the tile has
// rows or columns of 16) and the four waves' sums are added in a fixed order at the end: an output is the same four chains
// over k whatever the tile, so a row's result depends neither on the rows beside it nor on how many there are.  The operand
// lane l of an instruction holds row l % 16 and k = 4 (l / 16) + i in the i-th of four instructions: one 16-byte LDS read each.
// LDS rows are 64 + 8 floats long: lanes 0-7 and 16-23, which a 16-byte read serves together, then touch all 64 banks once.
// Loads run DEPTH stages ahead in registers.  K and the row strides multiples of 4, 16-byte aligned operands.
typedef float f32x4 __attribute__((ext_vector_type(4)));
#define G32_K 64
#define G32_LD (G32_K + 8)
#define G32_MAX_BLOCKS 0xffffffL  // workgroups of 256 threads that one dimension of a launch holds

// ENDS: the loop is asked for its end at every stage, not every 2 DEPTH of them; same sums.
template <int TM, int TN, int DEPTH, bool ENDS>
__global__ __launch_bounds__(256) void gemm_f32_kernel(float* __restrict__ out, const float* __restrict__ x,
                                                                 const float* __restrict__ w, int M, int N, int K, int x_stride,
                                                                 int out_stride, int m_tiles, int n_tiles) {
  constexpr int ROWS = TM + TN, PER = ROWS / 16;  // 16-byte pieces of a stage per thread: a row's 16 pieces by 16 neighbouring threads
  constexpr int MI = TM / 16, NI = TN / 16;
  constexpr int STAGE = ROWS * G32_LD, JOIN = 4 * TM * (TN + 4);
  __shared__ __attribute__((aligned(16))) float lds[2 * STAGE > JOIN ? 2 * STAGE : JOIN];
  // workgroups are dealt to the eight XCDs in launch order: an XCD takes every eighth tile of w and runs all tiles of x against
  // it one after the other, so that w is read into one L2 only
  const int xcd = blockIdx.x & 7, turn = blockIdx.x >> 3;
  const int nt = (turn / m_tiles) * 8 + xcd, mt = turn % m_tiles;
  if (nt >= n_tiles) return;
  const int m0 = mt * TM, n0 = nt * TN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int piece = tid & 15;  // k of this thread's pieces: 4 piece .. 4 piece + 3 of the stage
  const float* src[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int r = p * 16 + (tid >> 4);
    src[p] = (r < TM ? x + (size_t)min(m0 + r, M - 1) * x_stride : w + (size_t)min(n0 + r - TM, N - 1) * K) + 4 * piece;
  }
  f32x4 reg[DEPTH][PER];
  const int stages = (K + G32_K - 1) / G32_K;
  auto fetch = [&](f32x4* to, int stage) {
    const int k = stage * G32_K + 4 * piece;
#pragma unroll
    for (int p = 0; p < PER; ++p) to[p] = k < K ? *reinterpret_cast<const f32x4*>(src[p] + stage * G32_K) : f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto park = [&](const f32x4* from, int buf) {
#pragma unroll
    for (int p = 0; p < PER; ++p) *reinterpret_cast<f32x4*>(&lds[buf * STAGE + (p * 16 + (tid >> 4)) * G32_LD + 4 * piece]) = from[p];
  };
  f32x4 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int frag = (lane & 15) * G32_LD + 16 * wave + 4 * (lane >> 4);
  auto multiply = [&](int buf) {
    const float* base = &lds[buf * STAGE + frag];
    f32x4 a[NI], b[MI];
#pragma unroll
    for (int i = 0; i < MI; ++i) b[i] = *reinterpret_cast<const f32x4*>(base + i * 16 * G32_LD);
#pragma unroll
    for (int j = 0; j < NI; ++j) a[j] = *reinterpret_cast<const f32x4*>(base + (TM + j * 16) * G32_LD);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j][e], b[i][e], acc[i][j], 0, 0, 0);
  };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) fetch(reg[d], d);  // (a stage beyond K is zeros)
  park(reg[0], 0);
  for (int s0 = 0; s0 < stages; s0 += 2 * DEPTH) {
#pragma unroll
    for (int u = 0; u < 2 * DEPTH; ++u) {  // (stages beyond K, at most 2 DEPTH - 1, add zeros, unless ENDS)
      const int s = s0 + u;
      if (ENDS && s >= stages) break;
      __syncthreads();
      fetch(reg[u % DEPTH], s + DEPTH);
      multiply(u & 1);
      park(reg[(u + 1) % DEPTH], (u + 1) & 1);
    }
  }
  __syncthreads();
  // the waves' sums: [wave][row of x][row of w], rows 16 bytes apart from a multiple of the banks
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
      *reinterpret_cast<f32x4*>(&lds[(wave * TM + i * 16 + (lane & 15)) * (TN + 4) + j * 16 + 4 * (lane >> 4)]) = acc[i][j];
  __syncthreads();
  for (int e = tid; e < TM * TN / 4; e += 256) {
    const int m = e / (TN / 4), n = 4 * (e % (TN / 4));
    f32x4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const f32x4*>(&lds[(i * TM + m) * (TN + 4) + n]);
    const f32x4 sum = (v[0] + v[1]) + (v[2] + v[3]);
    if (m0 + m < M) {
      float* o = out + (size_t)(m0 + m) * out_stride + n0 + n;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (n0 + n + c < N) o[c] = sum[c];
    }
  }
}

template <int TM, int TN, int DEPTH>
static int launch_gemm_f32(float* out, const float* x, const float* w, int M, int N, int K, int x_stride, int out_stride, hipStream_t stream) {
  const int m_tiles = (M + TM - 1) / TM, n_tiles = (N + TN - 1) / TN;
  const long blocks = (long)m_tiles * ((n_tiles + 7) / 8 * 8);
  if (blocks > G32_MAX_BLOCKS) return NS_ERR_BAD_ARG;
  // Asking at every stage costs a long K up to 15% (777 rows, N 2,048, K 8,192: 273 -> 325 us) and saves a short one the stages of zeros behind
  // its last (2,048 rows, N 2,048, K 64: 45 -> 18 us): it pays where they are more than a fifth of the others.
  const int stages = (K + G32_K - 1) / G32_K, zeros = (2 * DEPTH - stages % (2 * DEPTH)) % (2 * DEPTH);
  (5 * zeros > stages ? gemm_f32_kernel<TM, TN, DEPTH, true> : gemm_f32_kernel<TM, TN, DEPTH, false>)<<<(unsigned)blocks, 256, 0, stream>>>(
      out, x, w, M, N, K, x_stride, out_stride, m_tiles, n_tiles);
  return ns_launch_status();
}

// out_f32 != 0 writes 32-bit results whatever the input type (logits).
extern "C" int ns_gemm_generic(void* out, const void* x, const void* w, int M, int N, int K, int x_stride, int out_stride,
                               int out_f32, int dtype, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0 || x_stride < K || out_stride < N) return NS_ERR_BAD_ARG;
  dim3 grid((N + GT_N - 1) / GT_N, (M + GT_M - 1) / GT_M);
  if (grid.y > 65535) return NS_ERR_BAD_ARG;
  // (more tiles of 32 x 32, in groups of eight, or of eight rows of w than one dimension of a launch holds: the plain kernel, which has two)
  const long tiles = (long)((M + 31) / 32) * (((long)N + 255) / 256 * 8);
  if (dtype == NS_DTYPE_F32 && K % 4 == 0 && x_stride % 4 == 0 && (((uintptr_t)x | (uintptr_t)w) & 15) == 0 && tiles <= G32_MAX_BLOCKS &&
      N < (1 << 26)) {
    float* o = (float*)out;
    const float *xf = (const float*)x, *wf = (const float*)w;
    if (M <= ROWS_M) {
      const int blocks = (N + ROWS_N - 1) / ROWS_N;
      if (M == 1)
        gemm_rows_f32_kernel<1><<<blocks, 64 * ROWS_WAVES, 0, stream>>>(o, xf, wf, M, N, K, x_stride, out_stride);
      else if (M == 2)
        gemm_rows_f32_kernel<2><<<blocks, 64 * ROWS_WAVES, 0, stream>>>(o, xf, wf, M, N, K, x_stride, out_stride);
      else if (M <= 4)
        gemm_rows_f32_kernel<4><<<blocks, 64 * ROWS_WAVES, 0, stream>>>(o, xf, wf, M, N, K, x_stride, out_stride);
      else
        gemm_rows_f32_kernel<8><<<blocks, 64 * ROWS_WAVES, 0, stream>>>(o, xf, wf, M, N, K, x_stride, out_stride);
      return ns_launch_status();
    }
    // Tiles of 32 x 32 where they fill the GPU and are not half empty, of 16 x 16 otherwise (777 rows, N 16,384, K 2,048: 512
    // against 740 us; 16 rows there 41 against 30; 64 rows, N 2,048, K 8,192: 73 against 41).  Larger tiles deal less evenly and
    // leave fewer workgroups to hide each other's loads (64 x 64: 583 us in the first of these, 350 against 283 at N 2,048, K 8,192).
    if (M <= 16 || (long)((M + 31) / 32) * ((N + 31) / 32) < 256)
      return launch_gemm_f32<16, 16, 8>(o, xf, wf, M, N, K, x_stride, out_stride, stream);
    return launch_gemm_f32<32, 32, 4>(o, xf, wf, M, N, K, x_stride, out_stride, stream);
  }
  if (dtype == NS_DTYPE_F32)
    gemm_generic_kernel<float, float><<<grid, 256, 0, stream>>>((float*)out, (const float*)x, (const float*)w, M, N, K, x_stride, out_stride);
  else if (dtype == NS_DTYPE_BF16 && out_f32)
    gemm_generic_kernel<bf16_t, float><<<grid, 256, 0, stream>>>((float*)out, (const bf16_t*)x, (const bf16_t*)w, M, N, K, x_stride, out_stride);
  else if (dtype == NS_DTYPE_BF16)
    gemm_generic_kernel<bf16_t, bf16_t><<<grid, 256, 0, stream>>>((bf16_t*)out, (const bf16_t*)x, (const bf16_t*)w, M, N, K, x_stride, out_stride);
  else
    return NS_ERR_UNSUPPORTED;
  return ns_launch_status();
}

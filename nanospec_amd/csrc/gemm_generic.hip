// out[M, N] = x[M, K] . w[N, K]^T  with 32-bit accumulation in a fixed order, for any M, N, K.
//
// The products of the true 32-bit path (of many rows where gemm_split.hip does not take them), and the fall-back for shapes the bfloat16 matrix-core kernels refuse.  A row's
// result does not depend on which other rows share the launch.  Three kernels: a plain tiled one for any size and either
// type, whose outputs are each one chain of fused multiply-adds over k = 0..K-1; for 32-bit operands on whole 16-byte
// pieces one that reads w as fast as memory gives it (up to 8 rows) and one on the 32-bit matrix instructions (more rows).
// Which of the two is taken depends on the number of rows alone; their sums are ordered differently, so a token's 32-bit
// result as one of few rows and as one of many differ by rounding.
// (reference: the nn.Linear calls of model/llama.py:175,184,195,286)
#include "common.h"
#include "lds_loads.h"
#include <type_traits>

typedef float f32x4 __attribute__((ext_vector_type(4)));

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

// Few rows (decode) in 32-bit: the work is reading w once.  A workgroup of WAVES waves owns eight rows of w and deals their
// K to its lanes in units of four (16-byte loads, a wave's load a contiguous KiB of a row); every lane sums its own k in
// order for each of MT rows of x, the 64 partial sums of an output are added in a fixed order by the vector unit (what lanes exchange for a sum of two of a wave's
// halves or quarters at a time, then of neighbours), and the waves' sums in LDS.  An output's value depends on its own row of x and of w only.
// For K and the row strides multiples of 4 and 16-byte aligned operands.
// Bound by the loads of w, read past the caches; what stands beside them are x, which comes from L2 (all of it once a workgroup) and the products, so a number of rows has
// a kernel of its own, and the addresses, which the scalar unit holds but for the lane's (in vector registers they would not leave room for 8 rows).  us, alone and a call beside two
// others, with sums through LDS's crossbar and 1, 2, 4 or 8 rows of x, and now: five rows, N 16,384, K 2,048 32.5 / 27.0 and 24.9 / 20.8 (5.4 TB/s, 6.5); N 2,048, K 8,192 19.0 /
// 13.6 and 16.0 / 12.8; N 2,048, K 2,048 8.7 / 6.2 and 7.2 / 5.4; N 128,256, K 2,048 212 / 215 and 158 / 158 (6.7 TB/s); eight rows 215 / 218 and 173 / 176, one row 170 / 165 and 156 / 152.
// (Captured steps run 1, 2, 4 or 8 rows; the other numbers are those of steps outside graphs.)
#define ROWS_M 8
#define ROWS_N 8

// Lanes 0-31 (of every pair of rows of 16 lanes the lower one) get the sum of ``a`` over both halves (rows), the others that of ``b``.
__device__ __forceinline__ float sum_halves(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float sum_rows(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int MT, int WAVES>
__global__ __launch_bounds__(64 * WAVES, 4) void gemm_rows_f32_kernel(float* __restrict__ out, const float* __restrict__ x, const float* __restrict__ w, int N, int K,
                                                                      int x_stride, int out_stride) {
  __shared__ float part[WAVES][ROWS_N * MT];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n0 = blockIdx.x * ROWS_N;
  float acc[ROWS_N][MT];
#pragma unroll
  for (int j = 0; j < ROWS_N; ++j)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[j][m] = 0.f;
  const char *wr[ROWS_N], *xr[MT];
#pragma unroll
  for (int j = 0; j < ROWS_N; ++j) wr[j] = reinterpret_cast<const char*>(w + (size_t)min(n0 + j, N - 1) * K);
#pragma unroll
  for (int m = 0; m < MT; ++m) xr[m] = reinterpret_cast<const char*>(x + (size_t)m * x_stride);
  for (unsigned i = threadIdx.x; i < (unsigned)K / 4; i += 64 * WAVES) {
    const unsigned at = 16 * i;  // (32 bits, so that a row's address stays in the scalar unit)
    f32x4 wv[ROWS_N];
#pragma unroll
    for (int j = 0; j < ROWS_N; ++j) wv[j] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(wr[j] + at));
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const f32x4 xv = *reinterpret_cast<const f32x4*>(xr[m] + at);
#pragma unroll
      for (int j = 0; j < ROWS_N; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[j][m] = fmaf(xv[e], wv[j][e], acc[j][m]);
    }
  }
  // lanes 8 j .. 8 j + 7 end up with row j of w
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    float half[4], row[2];
#pragma unroll
    for (int j = 0; j < 4; ++j) half[j] = sum_halves(acc[j][m], acc[j + 4][m]);
#pragma unroll
    for (int j = 0; j < 2; ++j) row[j] = sum_rows(half[j], half[j + 2]);
    const bool upper = lane & 8;
    const float keep = upper ? row[1] : row[0], give = upper ? row[0] : row[1];
    const float sum = group_sum<8>(keep + dpp_read<0x128>(give));  // row_ror 8
    if (lane % 8 == 0) part[wave][lane / 8 * MT + m] = sum;
  }
  __syncthreads();
  if (threadIdx.x < ROWS_N * MT) {
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < WAVES; ++i) v += part[i][threadIdx.x];
    const int n = n0 + threadIdx.x / MT, m = threadIdx.x % MT;
    if (n < N) out[(size_t)m * out_stride + n] = v;
  }
}

template <int MT = 1>
static int launch_rows_f32(float* out, const float* x, const float* w, int M, int N, int K, int x_stride, int out_stride, hipStream_t stream) {
  if constexpr (MT < ROWS_M)
    if (M > MT) return launch_rows_f32<MT + 1>(out, x, w, M, N, K, x_stride, out_stride, stream);
  const int blocks = (N + ROWS_N - 1) / ROWS_N;
  // Four waves where a row is then one load a lane or two of every lane (the sums of a longer chain are further from 64 bits: K 8,192 1.3e-7 instead of 1.15e-7; of chains of two lengths too: K 1,536
  // 9.37e-8 instead of 9.25e-8; K 2,048 9.49e-8 instead of 9.58e-8) and there are two workgroups for every compute unit: five rows, N 128,256, K 2,048 158 us, with eight waves 169; N 32,000, K 1,024 25 and 32; N 3,072, K 2,048 9.1 and 9.2; N 512 5.2 and 4.4.
  // (The sums depend on this choice, so it is the same for any number of rows.)
  if ((K <= 1024 || K == 2048) && N >= 4096)
    gemm_rows_f32_kernel<MT, 4><<<blocks, 256, 0, stream>>>(out, x, w, N, K, x_stride, out_stride);
  else
    gemm_rows_f32_kernel<MT, 8><<<blocks, 512, 0, stream>>>(out, x, w, N, K, x_stride, out_stride);
  return ns_launch_status();
}

// Many rows in 32-bit on the matrix cores (v_mfma_f32_16x16x4_f32, 32-bit products and sums: 157 TFLOP/s at the boost clock,
// the vector unit's own rate, but 2,048 operations an instruction and far fewer operand reads).  Bound by the matrix unit for many
// rows (the library's best is 131 TFLOP/s at 4,096 cubed), by the latency of a workgroup's loads for few.
// A workgroup of four waves owns TM rows of x and TN rows of w.  A stage is 64 k of both in LDS; wave i multiplies the k
// 16 i .. 16 i + 15 of every stage for the whole tile (so that a fragment from LDS serves as many instructions as the tile has
// rows or columns of 16) and the four waves' sums are added in a fixed order at the end: an output is the same four chains
// over k whatever the tile, so a row's result depends neither on the rows beside it nor on how many there are.  The operand
// lane l of an instruction holds row l % 16 and k = 4 (l / 16) + i in the i-th of four instructions: one 16-byte LDS read each.
// The loads write into LDS themselves (16 bytes a lane, the 64 lanes of an instruction side by side: 4 rows of 64 k), ST stages on their way or in
// use.  The fragments of the next stage are read under the products of this one, behind the barrier at which the next
// stage has come and every wave has read all of this one, whose place is given to a new stage there.
// A row's sixteen pieces of 16 bytes lie in an order of their own, piece p of row r at place p ^ (2 (r % 8)): lanes 0-7 and 16-23, which a
// 16-byte LDS read serves together, then touch all 64 banks once.
// Against the kernel before, whose loads went through registers (the same sums, bit by bit): 777 rows, N 16,384, K 2,048: 558 -> 430 us (121
// TFLOP/s), N 2,048, K 8,192: 276 -> 231 (113), N 3,072, K 2,048: 117 -> 86; 300 rows, N 2,048, K 8,192: 125 -> 101; 16 rows 34 -> 25, 64 rows, N 2,048, K 2,048:
// 12.4 -> 10.0; a short K, 2,048 rows, N 2,048, K 64: 18.7 -> 16.5.  A third of that is addresses: with a 64-bit sum a load in the vector unit the first of these takes 481 us.
// Relative error (2-norm, against 64 bits) 4.1e-7 at K 2,048, 8.1e-7 at K 8,192, half of the tiled kernel's above: four chains for one.
// K and the row strides multiples of 4, 16-byte aligned operands.
#define G32_K 64
#define G32_MAX_BLOCKS 0xffffffL    // workgroups of 256 threads that one dimension of a launch holds
#define G32_MAX_STRIDE (1 << 24)    // 64 rows of fewer floats than this are addressed by 32 bits

// FAR: rows further apart than 32 bits address from a tile's first: every load by a 64-bit address from the vector unit (9 rows 2^24 floats apart
// are 600 MB: such calls are rare, and the plain kernel would add up in one chain instead of four, at twice the error).
template <int TM, int TN, int ST, bool FAR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void gemm_f32_kernel(float* __restrict__ out, const float* __restrict__ x, const float* __restrict__ w, int M, int N,
                                                            int K, int x_stride, int out_stride, int m_tiles, int n_tiles) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef __attribute__((address_space(3))) void* lds_ptr;
  constexpr int ROWS = TM + TN, PER = ROWS / 16, MI = TM / 16, NI = TN / 16, STAGE = ROWS * G32_K, JOIN = 4 * TM * (TN + 4);
  __shared__ __attribute__((aligned(16))) float lds[ST * STAGE > JOIN ? ST * STAGE : JOIN];
  // workgroups are dealt to the eight XCDs in launch order: an XCD takes every eighth tile of w and runs all tiles of x against
  // it one after the other, so that w is read into one L2 only
  const int xcd = blockIdx.x & 7, turn = blockIdx.x >> 3;
  const int nt = (turn / m_tiles) * 8 + xcd, mt = turn % m_tiles;
  if (nt >= n_tiles) return;
  const int m0 = mt * TM, n0 = nt * TN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int piece = 4 * (r ^ (2 * ((wave * 4 + g) & 7)));  // k of a stage that this lane fetches of each of its rows
  // bytes from the tile's first row of x or w to this lane's piece of each row it fetches (32 bits: the launch sees to it); along K the scalar
  // unit counts, so a load costs the vector unit nothing
  typedef typename std::conditional<FAR, size_t, unsigned>::type offset;
  offset from[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int row = (p * 4 + wave) * 4 + g;
    from[p] = (offset)4 * ((p * 16 < TM ? (offset)min(row, M - 1 - m0) * x_stride : (offset)min(row - TM, N - 1 - n0) * K) + piece);
  }
  const float *x0 = x + (size_t)m0 * x_stride, *w0 = w + (size_t)n0 * K;
  const auto xr = __builtin_amdgcn_make_buffer_rsrc((void*)x0, 0, 0xffffffff, 0x00020000);
  const auto wr = __builtin_amdgcn_make_buffer_rsrc((void*)w0, 0, 0xffffffff, 0x00020000);
  const int stages = (K + G32_K - 1) / G32_K;
  auto issue = [&](int buf, int stage) {
    const int k = stage * G32_K;
    if (!FAR && k + G32_K <= K) {
#pragma unroll
      for (int p = 0; p < PER; ++p)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(p * 16 < TM ? xr : wr, (lds_ptr)(lds + buf * STAGE + (p * 4 + wave) * 4 * G32_K), 16, from[p], 4 * k, 0, 0);
    } else {
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        const float* at = k + piece < K ? (p * 16 < TM ? x0 : w0) + from[p] / 4 + k : reinterpret_cast<const float*>(&tile_zeros);
        __builtin_amdgcn_global_load_lds(at, (lds_ptr)(lds + buf * STAGE + (p * 4 + wave) * 4 * G32_K), 16, 0, 0);
      }
    }
  };
  f32x4 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int frag = r * G32_K + 4 * ((4 * wave + g) ^ (2 * (r & 7)));
  auto read = [&](int buf, f32x4* a, f32x4* b) {
    const float* base = &lds[buf * STAGE + frag];
#pragma unroll
    for (int j = 0; j < NI; ++j) a[j] = *reinterpret_cast<const f32x4*>(base + (TM + j * 16) * G32_K);
#pragma unroll
    for (int i = 0; i < MI; ++i) b[i] = *reinterpret_cast<const f32x4*>(base + i * 16 * G32_K);
  };
  int buf = 0;
  // stage s + 1 has come and stage s has been read by all: on with the next, under the products of s
  auto step = [&](int s, const f32x4* a, const f32x4* b, f32x4* a_next, f32x4* b_next) {
    if (s + ST <= stages)
      TILE_WAIT_LOADS((ST - 2) * PER);
    else
      TILE_WAIT_LOADS(0);
    TILE_WAIT_LDS();
    TILE_BARRIER();
    if (s + ST < stages) issue(buf, s + ST);
    buf = buf + 1 == ST ? 0 : buf + 1;
    read(buf, a_next, b_next);  // (behind the last stage: what happens to lie there, not used)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j][e], b[i][e], acc[i][j], 0, 0, 0);
  };
#pragma unroll
  for (int s = 0; s < ST; ++s)
    if (s < stages) issue(s, s);
  if (ST <= stages)
    TILE_WAIT_LOADS((ST - 1) * PER);
  else
    TILE_WAIT_LOADS(0);
  TILE_BARRIER();
  f32x4 a0[NI], b0[MI], a1[NI], b1[MI];
  read(0, a0, b0);
  int s = 0;
  for (; s + 1 < stages; s += 2) {
    step(s, a0, b0, a1, b1);
    step(s + 1, a1, b1, a0, b0);
  }
  if (s < stages) step(s, a0, b0, a1, b1);
  // the waves' sums: [wave][row of x][row of w], rows 16 bytes apart from a multiple of the banks
  __syncthreads();
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
      *reinterpret_cast<f32x4*>(&lds[(wave * TM + i * 16 + r) * (TN + 4) + j * 16 + 4 * g]) = acc[i][j];
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
#endif
}

template <int TM, int TN, int ST, bool FAR = false>
static int launch_gemm_f32(float* out, const float* x, const float* w, int M, int N, int K, int x_stride, int out_stride, hipStream_t stream) {
  const int m_tiles = (M + TM - 1) / TM, n_tiles = (N + TN - 1) / TN;
  const long blocks = (long)m_tiles * ((n_tiles + 7) / 8 * 8);
  if (blocks > G32_MAX_BLOCKS) return NS_ERR_BAD_ARG;
  gemm_f32_kernel<TM, TN, ST, FAR><<<(unsigned)blocks, 256, 0, stream>>>(out, x, w, M, N, K, x_stride, out_stride, m_tiles, n_tiles);
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
    if (M <= ROWS_M && K < 1 << 30) return launch_rows_f32(o, xf, wf, M, N, K, x_stride, out_stride, stream);
    // Tiles of 32 x 64 where there are four for every compute unit (777 rows, N 16,384, K 2,048: 430 against 442 us, 2,048 rows 1,066 against
    // 1,171), of 32 x 32 where they fill the GPU and are not half empty (777 rows, N 2,048, K 8,192: 231 against 253; 100 rows 50 against 57
    // with 16 x 16), of 16 x 16 otherwise (64 rows, N 2,048, K 8,192: 36 against 50).  64 x 64 deals less evenly (443 us in the first of these).
    const long m32 = (M + 31) / 32;
    if (x_stride >= G32_MAX_STRIDE) return launch_gemm_f32<32, 32, 3, true>(o, xf, wf, M, N, K, x_stride, out_stride, stream);
    if (M <= 16 || m32 * ((N + 31) / 32) < 256) {
      // Eight stages of a 16 x 16 tile take 64 KB of LDS, two workgroups a compute unit.  Where an XCD has more of them than that, three stages
      // and up to six workgroups hide the loads better: 96 rows, N 2,048, K 2,048 (768 tiles): 14.8 -> 12.2 us, K 8,192: 47.9 -> 34.4; 2,048 rows, N 64
      // (on four XCDs), K 64: 4.3 -> 3.7; 1,024 rows, N 132, K 4,096: 36.3 -> 25.9.  Up to 16 rows and a long K the weight's bytes bound it,
      // and eight stages bring them faster (16 rows, N 128,256, K 512: 51 us and 41 with three, K 768: 91 and 88, K 2,048: 196 and 206; N 28,672, K 6,144: 135 and 149).
      const long slots = (long)((M + 15) / 16) * (((long)N + 127) / 128 * 8);
      if (slots > 512 && (M > 16 || K <= 960)) return launch_gemm_f32<16, 16, 3>(o, xf, wf, M, N, K, x_stride, out_stride, stream);
      return launch_gemm_f32<16, 16, 8>(o, xf, wf, M, N, K, x_stride, out_stride, stream);
    }
    if (m32 * ((N + 63) / 64) >= 1024) return launch_gemm_f32<32, 64, 3>(o, xf, wf, M, N, K, x_stride, out_stride, stream);
    return launch_gemm_f32<32, 32, 3>(o, xf, wf, M, N, K, x_stride, out_stride, stream);
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

// Products of many bfloat16 rows with a weight in plain rows, out[m][n] = sum_k x[m][k] w[n][k], summed in 32-bit, with what follows the
// product done on its sums: nothing, an activation, the gate of a gated feed-forward (two matrices), the sum into the residual stream, or
// nothing yet (ranges of K side by side, for the kernel that reads them next).  The tile itself is tile_quarters.h's.
// (reference: the nn.Linear calls of model/llama.py:175,184,195)
//
// For products whose tiles come to about one or two a compute unit, where the platform's library has tiles of 256 x 256 for few of the
// units or small ones that read every operand often; products of many more tiles are the library's, whose large tiles read less.  us, the
// library and this kernel, alone and a call beside two others: 2,048 rows of 2,048 x 8,192 76 / 76 and 68 / 60, of 4,096 x 14,336 210 / 216 and 184 / 203, of 4,096 x
// 4,096 60 / 61 and 58 / 58, of 2,048 x 2,048 22.6 / 18.3 and 20.5 / 16.7; 512 rows of 2,048 x 8,192 34.5 / 34.7 and, in four ranges of K, 26.1 / 20.3.
// Bound by the matrix unit for half of the time (2,048 x 2,048 x 8,192: 39 us with the loads and the LDS reads taken out, the clock sinking
// under the products), by the way from L2 to LDS beside it (59 us with the products taken out, 18 TB/s).
#include "common.h"
#include "tile_quarters.h"

enum { MANY_PLAIN, MANY_ACT, MANY_GATED, MANY_ADD, MANY_RANGES };

struct ManyParams {
  void* out;
  const bf16_t *x, *w, *w2;  // w2: the up matrix of a gated product (w: the gate)
  int M, N, K, x_stride, out_stride, m_tiles, n_tiles, ranges, act;
};

// The tiles go to the eight XCDs (workgroups do in launch order) in eighths, range by range of K, and within a range in patches of 4 x 8 tiles, so that what an
// XCD's 32 compute units work on at a time shares rows of both operands in its L2 (loads alone, 16 x 16 tiles of 128 x 128: 24.4 TB/s, row
// by row of tiles 22.3).
#define MANY_PATCH_M 4
#define MANY_PATCH_N 8

template <class T, int EPI>
__global__ __launch_bounds__(T::WAVES * NS_WAVE) __attribute__((amdgpu_waves_per_eu(1))) void gemm_many_kernel(const ManyParams p) {
  constexpr bool DUAL = EPI == MANY_GATED;
  constexpr int HALF = T::BN / 2, CH = DUAL ? HALF : T::BN;  // output channels of a workgroup
  __shared__ __attribute__((aligned(16))) bf16_t many_tiles[T::VALUES];
  const int tiles = p.m_tiles * p.n_tiles, items = tiles * p.ranges, share = (items + 7) / 8;
  const int item = (blockIdx.x & 7) * share + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= share || item >= items) return;
  const int range = item / tiles;
  int tile = item - range * tiles;
  const int band = tile / (MANY_PATCH_M * p.n_tiles);  // of MANY_PATCH_M rows of tiles
  tile -= band * MANY_PATCH_M * p.n_tiles;
  const int high = min(MANY_PATCH_M, p.m_tiles - band * MANY_PATCH_M), patch = tile / (high * MANY_PATCH_N);
  tile -= patch * high * MANY_PATCH_N;
  const int m0 = (band * MANY_PATCH_M + tile % high) * T::BM, n0 = (patch * MANY_PATCH_N + tile / high) * CH;
  const int K = p.K / p.ranges;
  const size_t k0 = (size_t)range * K;

  T t;
  t.init(many_tiles, K);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    // (rows beyond the last are the last; their sums are not written)
    t.x_from(h, p.x + (size_t)m0 * p.x_stride + k0);
    t.w_from(h, (DUAL && h ? p.w2 : p.w) + (size_t)n0 * p.K + k0);
#pragma unroll
    for (int q = 0; q < T::LA; ++q) t.xo[h][q] = 2 * (min(h * (T::BM / 2) + t.row_of(q), p.M - 1 - m0) * p.x_stride + t.piece());
#pragma unroll
    for (int q = 0; q < T::LB; ++q) t.wo[h][q] = 2 * (min((DUAL ? 0 : h * HALF) + t.row_of(q), p.N - 1 - n0) * p.K + t.piece());
  }
  t.run();

  typedef bf16_t bf16x4 __attribute__((ext_vector_type(4)));
  const int r = t.lane % 16, g = t.lane / 16;
#pragma unroll
  for (int i = 0; i < T::MI; ++i) {
    const int row = m0 + 16 * (2 * i + t.wm) + r;
    if (row >= p.M) continue;
#pragma unroll
    for (int j = 0; j < (DUAL ? T::NH : T::NJ); ++j) {
      const int col = n0 + 16 * (2 * j + t.wn) + 4 * g;
      if (col >= p.N) continue;  // (N is a multiple of 4)
      if (EPI == MANY_RANGES) {
        *reinterpret_cast<typename T::f32x4*>((float*)p.out + ((size_t)range * p.M + row) * p.N + col) = t.acc[i][j];
        continue;
      }
      bf16x4* at = reinterpret_cast<bf16x4*>((bf16_t*)p.out + (size_t)row * p.out_stride + col);
      bf16x4 o;
      if (EPI == MANY_ADD) o = *at;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float z = t.acc[i][j][e];
        // (what stands between the product and an activation is rounded as a store would round it)
        if (EPI == MANY_ACT)
          o[e] = from_f<bf16_t>(activation_of(round_to<bf16_t>(z), p.act));
        else if (EPI == MANY_ADD)
          o[e] = from_f<bf16_t>(to_f((bf16_t)o[e]) + z);
        else if (EPI == MANY_GATED) {
          const float gate = round_to<bf16_t>(z), up = round_to<bf16_t>(t.acc[i][T::NH + j][e]);
          o[e] = from_f<bf16_t>(gate / (1.f + expf(-gate)) * up);
        } else
          o[e] = from_f<bf16_t>(z);
      }
      *at = o;
    }
  }
}

// What may follow a product in tiles of T, other pairs are not built: the gate stands behind tiles of 128 columns (half as many channels), ranges of K behind the tile
// that they are for, an activation behind all but the largest tile, whose end costs more than a kernel of its own.
template <class T, int EPI>
static int launch_many(ManyParams p, hipStream_t stream) {
  constexpr bool LARGEST = T::BM == 256, SMALL = T::BN == 64;
  if constexpr ((EPI == MANY_GATED && SMALL) || (EPI == MANY_RANGES && (SMALL || LARGEST)) || (EPI == MANY_ACT && LARGEST))
    return NS_ERR_UNSUPPORTED;
  else {
    const int ch = EPI == MANY_GATED ? T::BN / 2 : T::BN;
    p.m_tiles = (p.M + T::BM - 1) / T::BM, p.n_tiles = (p.N + ch - 1) / ch;
    if (p.K / p.ranges < T::BEHIND * QUARTER_K) return NS_ERR_UNSUPPORTED;
    const long long items = (long long)p.m_tiles * p.n_tiles * p.ranges;
    if (items > (1 << 22)) return NS_ERR_UNSUPPORTED;
    gemm_many_kernel<T, EPI><<<(unsigned)((items + 7) / 8 * 8), T::WAVES * NS_WAVE, 0, stream>>>(p);
    return ns_launch_status();
  }
}

template <class T>
static int launch_many(const ManyParams& p, int epi, hipStream_t stream) {
  switch (epi) {
    case MANY_PLAIN: return launch_many<T, MANY_PLAIN>(p, stream);
    case MANY_ACT: return launch_many<T, MANY_ACT>(p, stream);
    case MANY_GATED: return launch_many<T, MANY_GATED>(p, stream);
    case MANY_ADD: return launch_many<T, MANY_ADD>(p, stream);
    default: return launch_many<T, MANY_RANGES>(p, stream);
  }
}

// ``form``: the tile, rows of x by rows of w: 0 64 x 64, 1 128 x 64, 2 128 x 128, 3 256 x 128.
// ``epi``: 0 out = x w^T; 1 an activation of it (``act`` as common.h numbers them); 2 silu(x w^T) * (x w2^T); 3 out += x w^T (summed in 32-bit,
// rounded once); 4 out: float32 [ranges][M][N], the sums over each of ``ranges`` equal ranges of K (one range in the other four).
// Not every tile with every ``epi``: 1 with forms 0 to 2, 2 with 2 and 3, 4 with 2 (NS_ERR_UNSUPPORTED otherwise).
// K: a multiple of 128 a range and at least 256 (form 0: 384); x_stride a multiple of 8, N and out_stride of 4; x, w, w2 on 16 bytes, out on 8 (on 16 with ranges).
extern "C" int ns_gemm_many_bf16(void* out, const void* x, const void* w, const void* w2, int M, int N, int K, int x_stride, int out_stride, int epi,
                                 int act, int ranges, int form, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0 || x_stride < K || out_stride < N || epi < MANY_PLAIN || epi > MANY_RANGES || ranges < 1) return NS_ERR_BAD_ARG;
  if ((epi == MANY_GATED && !w2) || (epi == MANY_ACT && (act < 0 || act >= NS_ACTIVATIONS)) || (ranges > 1 && epi != MANY_RANGES)) return NS_ERR_BAD_ARG;
  if (K % (QUARTER_K_MULTIPLE * ranges) || x_stride % 8 || N % 4 || out_stride % 4) return NS_ERR_UNSUPPORTED;
  if ((((uintptr_t)x | (uintptr_t)w | (uintptr_t)w2) & 15) || ((uintptr_t)out & (epi == MANY_RANGES ? 15 : 7))) return NS_ERR_UNSUPPORTED;
  if (K >= 1 << 22 || x_stride >= 1 << 22) return NS_ERR_UNSUPPORTED;  // (a tile's rows within 31 bits of bytes)
  const ManyParams p{out, (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)w2, M, N, K, x_stride, out_stride, 0, 0, ranges, act};
  switch (form) {
    // (the smaller tiles' operands come from memory more often than from L2, which takes more stages on their way: 512 rows of 2,048 x 2,048, weights
    // that no cache holds, four stages instead of two 13.2 -> 11.4 us; 512 of 3,072 three 16.0 / 10.4 -> 15.7 / 9.9, four / 11.6)
    case 0: return launch_many<QuarterTile<64, 64, 4>>(p, epi, stream);
    case 1: return launch_many<QuarterTile<128, 64, 3>>(p, epi, stream);
    case 2: return launch_many<QuarterTile<128, 128>>(p, epi, stream);
    case 3: return launch_many<QuarterTile<256, 128>>(p, epi, stream);
  }
  return NS_ERR_BAD_ARG;
}

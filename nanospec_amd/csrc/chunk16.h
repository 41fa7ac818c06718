// What the recurrences that go sixteen tokens at a time share: the order of a chunk's tokens in the matrix instructions' operands, the
// numbering of the chunks, and the product that keeps infinities where they belong.
#pragma once
#include "common.h"

#define DC_T 16  // tokens of a chunk
// Row m of a chunk's matrices is this token: the four rows that a lane holds of a result are what it gives to the four instructions of the next
// product, and each instruction adds four neighbouring tokens, the oldest first, so that the newest, which no decay has
// made smaller yet, are added last, as in the token form.
__device__ __forceinline__ int chunk_token(int m) { return 4 * (m % 4) + m / 4; }
typedef float f32x4 __attribute__((ext_vector_type(4)));

// A request's chunks have numbers of their own without a plan: its first is floor(first row / 16) + its place in the batch, so that no two
// requests' overlap and n / 16 + requests numbers are enough.  The request that a number belongs to (it may have fewer chunks):
__device__ __forceinline__ int chunk_request(const int* __restrict__ qo_indptr, int n_reqs, int chunk) {
  int lo = 0, hi = n_reqs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (qo_indptr[mid] / DC_T + mid <= chunk) lo = mid; else hi = mid - 1;
  }
  return lo;
}

__device__ __forceinline__ bool not_finite(const f32x4 v) { return !(fabsf(v[0]) + fabsf(v[1]) + fabsf(v[2]) + fabsf(v[3]) < INFINITY); }

// sum_j m[row][j] x[j] by the lane that holds rows 4 g .. + 3 of column c of x, without the tokens behind the row's
__device__ __forceinline__ f32x4 lower_product(const float* __restrict__ m, const f32x4 x, int lane) {
  f32x4 r = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int j = 0; j < DC_T; ++j) {
    const float pick = (j & 2) ? ((j & 1) ? x[3] : x[2]) : ((j & 1) ? x[1] : x[0]);
    const float xj = __shfl(pick, j / 4 * 16 + lane % 16, NS_WAVE);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * (lane / 16) + i;
      const bool seen = chunk_token(j) <= chunk_token(row);
      r[i] = fmaf(m[(j / 4 * 16 + row) * 4 + j % 4], seen ? xj : 0.f, r[i]);  // (m is finite where a token is not seen: zero)
    }
  }
  return r;
}


// A workgroup's tile of a bfloat16 product on the matrix cores: BM rows of x times BN rows of w, K in stages of 64, for kernels
// that bring their own rows and do their own thing with the sums.
//
// The loads.  `global_load_lds` writes 16 bytes a lane straight into LDS, the 64 lanes of an instruction side by side: 8 rows of 64
// values.  No register holds a value on its way, so ST stages of both operands can be in flight.  A row's eight pieces of 16
// bytes lie in LDS in an order of their own, piece p of row r at place p ^ (r % 8) (the lane chooses which piece of its row it
// fetches), so that lanes 0-7 and 16-23, which a 16-byte LDS read serves together, touch all 64 banks once.
// The order.  A stage is two halves of 32 k.  While the products of one half run, the fragments of the next are read; the wait for the
// next stage and the barrier stand between the halves, where every wave has work of its own in the matrix unit and the last
// reads of a stage are done, so the stage's place is given to a new one right behind the barrier.
// The waits are counted by hand (lds_loads.h).  No other vector load may be issued between start() and the end of run().
#pragma once
#include "lds_loads.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;

#define TILE_K 64
// WR x WC waves; wave (wm, wn) owns the blocks of 16 rows wm, wm + WR, .. of x (so that a tile whose last blocks are empty keeps all waves
// equally busy) and 16 NJ neighbouring rows of w.  acc[i][j]: lane l holds for row 16 (WR i + wm) + l % 16 of x the sums with rows 16 NJ wn + 16 j +
// 4 (l / 16) .. + 3 of w.
// W_ONCE: most rows of w are read by one workgroup: past the caches.
template <int BM_, int BN_, int WR_, int WC_, int ST_, bool W_ONCE = false>
struct TileBf16 {
  static constexpr int BM = BM_, BN = BN_, WR = WR_, WC = WC_, ST = ST_;
  static constexpr int WAVES = WR * WC, THREADS = WAVES * NS_WAVE, MI = BM / WR / 16, NJ = BN / WC / 16;
  static constexpr int PA = BM / 8 / WAVES, PB = BN / 8 / WAVES, PER = PA + PB;  // loads of a wave for a stage
  static constexpr int STAGE = (BM + BN) * TILE_K;                              // values
  static constexpr int BYTES = ST * STAGE * 2;
  static_assert(PA * 8 * WAVES == BM && PB * 8 * WAVES == BN && MI * 16 * WR == BM && NJ * 16 * WC == BN, "whole loads and whole blocks");
  static_assert(ST >= 2 && (ST - 1) * PER < 64 && BYTES <= 160 * 1024, "stages");

  typedef float f32x4 __attribute__((__vector_size__(4 * sizeof(float))));
  bf16_t* lds;
  int lane, wave, wm, wn, K, stages, turn, next;
  const bf16_t* src[PER];  // this lane's piece of each row it fetches: at k = 0, from start() on at the next stage to fetch
  f32x4 acc[MI][NJ];

  // the row of x (p < PA) or w that load p of this lane fetches
  __device__ __forceinline__ int row_of(int p) const { return ((p < PA ? p : p - PA) * WAVES + wave) * 8 + lane / 8; }
  // the first of the 8 values along a stage that this lane fetches of each of its rows
  __device__ __forceinline__ int piece() const { return 8 * ((lane % 8) ^ (lane / 8)); }

  // ``turn_``: the stage of K to begin with (any number; the sums run over K from there and round)
  __device__ __forceinline__ void init(bf16_t* lds_, int K_, int turn_ = 0) {
    lds = lds_, K = K_, stages = (K + TILE_K - 1) / TILE_K, turn = turn_ % stages;
    lane = threadIdx.x % NS_WAVE;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x / NS_WAVE);
    wm = wave / WC, wn = wave % WC;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  __device__ __forceinline__ void issue(int buf) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(3))) void* lds_ptr;
    bf16_t* to = lds + buf * STAGE + wave * 8 * TILE_K;
    const int k = next;  // of the stage that is issued: they come in order
    auto load = [&](int p, const bf16_t* from) {
      const lds_ptr at = (lds_ptr)(to + (p < PA ? p * WAVES * 8 * TILE_K : (BM + (p - PA) * WAVES * 8) * TILE_K));
      if (W_ONCE && p >= PA)
        __builtin_amdgcn_global_load_lds(from, at, 16, 0, 2);  // (non-temporal)
      else
        __builtin_amdgcn_global_load_lds(from, at, 16, 0, 0);
    };
    if (k + TILE_K <= K) {  // (no selection where none is needed, and one sum a load: the vector unit is short of time here)
#pragma unroll
      for (int p = 0; p < PER; ++p) load(p, src[p]), src[p] += TILE_K;
      next += TILE_K;
      if (next == K) {
        next = 0;
#pragma unroll
        for (int p = 0; p < PER; ++p) src[p] -= K;
      }
    } else {
      const bool in = k + piece() < K;
#pragma unroll
      for (int p = 0; p < PER; ++p) load(p, in ? src[p] : reinterpret_cast<const bf16_t*>(&tile_zeros)), src[p] -= k;
      next = 0;
    }
#endif
  }

  // the rows' addresses to the stage to begin with, and the first stages on their way
  __device__ __forceinline__ void start() {
    next = turn * TILE_K;
#pragma unroll
    for (int p = 0; p < PER; ++p) src[p] += next;
#pragma unroll
    for (int s = 0; s < ST; ++s)
      if (s < stages) issue(s);
  }

  template <int BLOCKS>
  __device__ __forceinline__ void frags(int buf, int half, bf16x8* a, bf16x8* b) const {
    const int r = lane % 16, at = ((4 * half + lane / 16) ^ (r % 8)) * 8;
    const bf16_t* base = lds + buf * STAGE + r * TILE_K + at;
    if constexpr (BLOCKS > 0) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) b[j] = *reinterpret_cast<const bf16x8*>(base + (BM + (wn * NJ + j) * 16) * TILE_K);
    }
#pragma unroll
    for (int i = 0; i < BLOCKS; ++i) a[i] = *reinterpret_cast<const bf16x8*>(base + (WR * i + wm) * 16 * TILE_K);
  }

  template <int BLOCKS>
  __device__ __forceinline__ void multiply(const bf16x8* a, const bf16x8* b) {
#pragma unroll
    for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
    // an LDS read, then its share of the products
    if constexpr (BLOCKS > 0) {
      constexpr int READS = BLOCKS + NJ, SHARE = BLOCKS * NJ / READS;
#pragma unroll
      for (int q = 0; q < READS; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, SHARE, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, BLOCKS * NJ - SHARE * READS, 0);
    }
  }

  template <int BLOCKS>
  __device__ __forceinline__ void loop() {
    bf16x8 a0[MI], b0[NJ], a1[MI], b1[NJ];
    if (ST <= stages)
      TILE_WAIT_LOADS((ST - 1) * PER);
    else
      TILE_WAIT_LOADS(0);
    TILE_BARRIER();
    frags<BLOCKS>(0, 0, a0, b0);
    int buf = 0;
    for (int s = 0; s < stages; ++s) {
      __builtin_amdgcn_sched_barrier(0);
      frags<BLOCKS>(buf, 1, a1, b1);
      multiply<BLOCKS>(a0, b0);
      __builtin_amdgcn_sched_barrier(0);
      if (s + ST <= stages)
        TILE_WAIT_LOADS((ST - 2) * PER);
      else
        TILE_WAIT_LOADS(0);
      TILE_WAIT_LDS();  // this wave has read all of stage s
      TILE_BARRIER();
      if (s + ST < stages) issue(buf);
      buf = buf + 1 == ST ? 0 : buf + 1;
      __builtin_amdgcn_sched_barrier(0);
      frags<BLOCKS>(buf, 0, a0, b0);  // (behind the last stage: what happens to lie there, not used)
      multiply<BLOCKS>(a1, b1);
    }
  }

  // ``blocks``: blocks of 16 rows of x that this wave multiplies (up to MI; the others' sums stay zero)
  template <int BLOCKS = MI>
  __device__ __forceinline__ void run(int blocks) {
    if constexpr (BLOCKS > 0) {
      if (blocks < BLOCKS) return run<BLOCKS - 1>(blocks);
    }
    loop<BLOCKS>();
  }
};

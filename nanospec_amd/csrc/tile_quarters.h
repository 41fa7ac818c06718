// A workgroup's tile of a bfloat16 product on the matrix cores: BM rows of x times BN rows of w, by four waves that hold a quarter of the
// sums each, one wave a SIMD and tile.  For kernels that bring their own rows and do their own thing with the sums.
//
// Why so few waves: a wave reads (BM + BN) / 2 rows from LDS for BM BN / 4 sums, so with two waves on a SIMD instead of one the same tile
// takes up to twice the LDS reads, and LDS (128 bytes a clock) is what the smaller tiles are bound by.  128 x 128, 2,048 x 2,048 x 8,192, one
// tile a compute unit: 111 us with four waves and 79 with eight, both reading a whole stage ahead; as it is here 66.
// The loads.  `buffer_load .. lds` writes 16 bytes a lane straight into LDS, 8 rows of 64 values an instruction, addresses in the scalar
// unit.  ST stages of 64 k lie in LDS, each as four units: the lower and upper half of the rows of x and of w.  A stage's products are
// four quarters, one for each pair of units, in an order in which every quarter wants one new unit:
//     (x low, w low)  (x low, w high)  (x high, w high)  (x high, w low)
// While a quarter's products run, the fragments of the unit that the next one wants are read, and a unit's place is filled anew as soon as
// it has been read: with two stages the loads of six to seven quarters are always on their way, where a ring of whole stages has four.
// One barrier a quarter: behind it a unit has landed for all waves, and another has been read by all.
// The loop has no branches: a merge of two paths makes the compiler move all sums from register to register.
// A row's eight pieces of 16 bytes lie in LDS in an order of their own, piece p of row r at place p ^ (r % 8) (the lane chooses which piece
// of its row it fetches), so that lanes 0-7 and 16-23, which a 16-byte LDS read serves together, touch all 64 banks once.
// The waits are counted by hand (lds_loads.h).  No other vector load may be issued between the first load and the end of run().
#pragma once
#include "lds_loads.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;

#define QUARTER_K 64           // values of K a stage
#define QUARTER_K_MULTIPLE 128  // what K must be a multiple of (an even number of stages)

// What K may be.  PAIRS: an even number of stages.  ODD: an odd one; the first is multiplied ahead of the loop of pairs.  ANY: any multiple of 8 (stages beyond
// K are zeros), and rows anywhere: an address of 64 bits and a choice for every load.
enum QuarterInner { QUARTER_PAIRS, QUARTER_ODD, QUARTER_ANY };

// Wave (wm, wn) of 2 x 2 owns the blocks of 16 rows wm, wm + 2, .. of x and wn, wn + 2, .. of w.  acc[i][j]: lane l holds for row 16 (2 i + wm) + l % 16 of x
// the sums with rows 16 (2 j + wn) + 4 (l / 16) .. + 3 of w.
// W_ONCE: most rows of w are read by one workgroup: past the caches.
template <int BM_, int BN_, int ST_ = 2, bool W_ONCE = false, QuarterInner INNER = QUARTER_PAIRS>
struct QuarterTile {
  static constexpr bool ANY = INNER == QUARTER_ANY;
  static constexpr int BM = BM_, BN = BN_, ST = ST_, WAVES = 4;
  static constexpr int MI = BM / 32, NJ = BN / 32, MH = MI / 2, NH = NJ / 2;
  static constexpr int UA = BM / 2 * QUARTER_K, UB = BN / 2 * QUARTER_K;   // values of a unit of x and of w
  static constexpr int STAGE = 2 * (UA + UB), VALUES = ST * STAGE;         // values of a stage, and of LDS
  static constexpr int LA = BM / 2 / 8 / WAVES, LB = BN / 2 / 8 / WAVES;   // loads of a wave for a unit
  static_assert(MH * 64 == BM && NH * 64 == BN && LA * 64 == BM && LB * 64 == BN, "whole blocks and whole loads");
  static constexpr int BEHIND = ST + 1 + (ST + 1) % 2;                     // stages behind the loop, an even number; K has at least as many (ODD: one more)
  static_assert(ST >= 2 && VALUES * 2 <= 160 * 1024 && 2 * ST * (LA + LB) < 64, "stages");
  enum { X_LOW, W_LOW, W_HIGH, X_HIGH };  // the units, in the order in which they are wanted

  typedef float f32x4 __attribute__((__vector_size__(4 * sizeof(float))));
  bf16_t* lds;
  int lane, wave, wm, wn, stages, at;  // at: the stage of K that is loaded next
  int K;
  int xo[2][LA], wo[2][LB];            // bytes from the halves' first rows to this lane's piece of each row it fetches, at k = 0
  __amdgpu_buffer_rsrc_t xr[2], wr[2];
  const bf16_t *xp[2][LA], *wp[2][LB];  // (ANY: the same as addresses)
  f32x4 acc[MI][NJ];

  // the row of its half that load q of this lane fetches
  __device__ __forceinline__ int row_of(int q) const { return (q * WAVES + wave) * 8 + lane / 8; }
  // the first of the 8 values along a stage that this lane fetches of each of its rows
  __device__ __forceinline__ int piece() const { return 8 * ((lane % 8) ^ (lane / 8)); }

  // ``turn``: the stage of K to begin with (any number; the sums run over K from there and round)
  __device__ __forceinline__ void init(bf16_t* lds_, int K_, int turn = 0) {
    lds = lds_, K = K_, stages = ANY ? max(BEHIND, (K + 2 * QUARTER_K - 1) / (2 * QUARTER_K) * 2) : K / QUARTER_K, at = turn % stages;
    lane = threadIdx.x % NS_WAVE;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x / NS_WAVE % WAVES);
    wm = wave / 2, wn = wave % 2;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // where the low (0) or high (1) half's offsets count from
  __device__ __forceinline__ void x_from(int half, const bf16_t* p) { xr[half] = __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0xffffffff, 0x00020000); }
  __device__ __forceinline__ void w_from(int half, const bf16_t* p) { wr[half] = __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0xffffffff, 0x00020000); }

  // ANY: this lane's piece of the row that its load q fetches
  __device__ __forceinline__ void x_row(int half, int q, const bf16_t* p) { xp[half][q] = p + piece(); }
  __device__ __forceinline__ void w_row(int half, int q, const bf16_t* p) { wp[half][q] = p + piece(); }

  static constexpr bool of_x(int u) { return u == X_LOW || u == X_HIGH; }
  static constexpr int place(int u) { return u == X_LOW ? 0 : u == W_LOW ? UA : u == W_HIGH ? UA + UB : UA + 2 * UB; }
  static constexpr int loads(int u) { return of_x(u % 4) ? LA : LB; }
  static constexpr int loads_of(int first, int last) {  // of units in the order of use
    int n = 0;
    for (int u = first; u <= last; ++u) n += loads(u);
    return n;
  }

  // load q of unit U of stage ``k`` of K, into the stage in LDS that begins at ``slot``
  template <int U>
  __device__ __forceinline__ void load(int q, int slot, int k) const {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(3))) void* lds_ptr;
    const lds_ptr to = (lds_ptr)(lds + slot + place(U) + (q * WAVES + wave) * 8 * QUARTER_K);
    constexpr int half = U == X_HIGH || U == W_HIGH;
    if constexpr (ANY) {
      const bf16_t* from = (of_x(U) ? xp[half][q] : wp[half][q]) + k * QUARTER_K;
      if (k * QUARTER_K + piece() >= K) from = reinterpret_cast<const bf16_t*>(&tile_zeros);
      // (through the caches: rows of no whole 128 bytes share lines with their neighbours.  64 tokens, 32 experts of 2,056, width 1,448, past them 153 us, so 133)
      __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
    } else if constexpr (of_x(U))
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xr[half], to, 16, xo[half][q], k * (QUARTER_K * 2), 0, 0);
    else if constexpr (W_ONCE)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wr[half], to, 16, wo[half][q], k * (QUARTER_K * 2), 0, 2);  // (non-temporal)
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wr[half], to, 16, wo[half][q], k * (QUARTER_K * 2), 0, 0);
#endif
  }
  template <int U>
  __device__ __forceinline__ void load_unit(int slot, int k) const {
#pragma unroll
    for (int q = 0; q < loads(U); ++q) load<U>(q, slot, k);
  }

  // fragment f (block f / 2, half f % 2 of the stage) of unit U
  template <int U>
  __device__ __forceinline__ bf16x8 frag(int f, int slot) const {
    const int r = lane % 16, to = ((4 * (f % 2) + lane / 16) ^ (r % 8)) * 8;
    return *reinterpret_cast<const bf16x8*>(lds + slot + place(U) + (f / 2 * 2 + (of_x(U) ? wm : wn)) * 16 * QUARTER_K + r * QUARTER_K + to);
  }

  // The products of half HI of x's rows and HJ of w's.  Before them: until at most WAIT loads are on their way.  Among them: unit R is
  // read from ``rslot`` (if READ), unit L of stage k loaded into ``lslot`` (if LOAD).
  template <int HI, int HJ, int R, int L, int WAIT, bool READ, bool LOAD>
  __device__ __forceinline__ void quarter(const bf16x8* a, const bf16x8* b, bf16x8* into, int rslot, int lslot, int k) {
    TILE_WAIT_LOADS(WAIT);
    TILE_WAIT_LDS();
    TILE_BARRIER();
    __builtin_amdgcn_sched_barrier(0);
    // reads before every other product, loads before the others from a quarter of them on
    constexpr int NR = 2 * (of_x(R) ? MH : NH), NL = loads(L), NM = 2 * MH * NH, FROM = NM / 4;
    constexpr int AT_READ = (NR + NM / 2 - 1) / (NM / 2), AT_LOAD = (NL + (NM - FROM) / 2 - 1) / ((NM - FROM) / 2);
    int reads = 0, begun = 0;
#pragma unroll
    for (int m = 0; m < NM; ++m) {
#pragma unroll
      for (int q = 0; q < (m % 2 ? 0 : AT_READ); ++q) {
        if constexpr (READ)
          if (reads < NR) into[reads] = frag<R>(reads, rslot);
        ++reads;
      }
#pragma unroll
      for (int q = 0; q < (m % 2 && m >= FROM ? AT_LOAD : 0); ++q) {
        if constexpr (LOAD)
          if (begun < NL) load<L>(begun, lslot, k);
        ++begun;
      }
      const int half = m / (MH * NH), i = m % (MH * NH) / NH, j = m % NH;
      acc[HI * MH + i][HJ * NH + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[2 * j + half], a[2 * i + half], acc[HI * MH + i][HJ * NH + j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    static_assert(AT_READ * (NM / 2) >= NR && AT_LOAD * ((NM - FROM) / 2) >= NL, "a place for every read and load");
  }

  __device__ __forceinline__ int behind(int k) const { return k + 1 == stages ? 0 : k + 1; }
  static __device__ __forceinline__ int slot_behind(int slot) { return slot + STAGE == VALUES ? 0 : slot + STAGE; }
  // the loads that may be on their way at quarter q of a stage behind which LEFT more come: unit q + 2 has landed, those up to q + 4 ST are issued
  static constexpr int open(int q, int left) { return loads_of(q + 3, q + 4 * ST < 4 * left + 3 ? q + 4 * ST : 4 * left + 3); }
  // A stage in ``slot``, with LEFT more behind it; w low is read into ``b0``, and w high into ``b1``, where the next stage finds its w low.
  template <int LEFT>
  __device__ __forceinline__ void stage(int& slot, bf16x8* low, bf16x8* high, bf16x8* b0, bf16x8* b1) {
    const int other = slot_behind(slot);
    quarter<0, 0, W_HIGH, W_LOW, open(0, LEFT), true, LEFT >= ST>(low, b0, b1, slot, slot, at);
    quarter<0, 1, X_HIGH, W_HIGH, open(1, LEFT), true, LEFT >= ST>(low, b1, high, slot, slot, at);
    quarter<1, 1, X_LOW, X_HIGH, open(2, LEFT), LEFT >= 1, LEFT >= ST>(high, b1, low, other, slot, at);
    if constexpr (LEFT >= ST) at = behind(at);
    quarter<1, 0, W_LOW, X_LOW, open(3, LEFT), LEFT >= 1, LEFT >= ST + 1>(high, b0, b1, other, other, at);
    slot = other;
  }
  template <int LEFT>
  __device__ __forceinline__ void last_stages(int& slot, bf16x8* low, bf16x8* high, bf16x8* b0, bf16x8* b1) {
    stage<LEFT>(slot, low, high, b0, b1);
    if constexpr (LEFT > 0) last_stages<LEFT - 1>(slot, low, high, b1, b0);
  }

  // ``count`` stages, an even number
  __device__ __forceinline__ void all_but_odd(int count, int& slot, bf16x8* low, bf16x8* high, bf16x8* b0, bf16x8* b1) {
    for (int s = 0; s + 2 + BEHIND <= count; s += 2) {
      stage<ST + 1>(slot, low, high, b0, b1);
      stage<ST + 1>(slot, low, high, b1, b0);
    }
    last_stages<BEHIND - 1>(slot, low, high, b0, b1);
  }

  __device__ __forceinline__ void run() {
    bf16x8 low[2 * MH], high[2 * MH], b0[2 * NH], b1[2 * NH];
#pragma unroll
    for (int s = 0; s < ST; ++s) {
      load_unit<X_LOW>(s * STAGE, at), load_unit<W_LOW>(s * STAGE, at), load_unit<W_HIGH>(s * STAGE, at), load_unit<X_HIGH>(s * STAGE, at);
      at = behind(at);
    }
    TILE_WAIT_LOADS(loads_of(2, 4 * ST - 1));
    TILE_BARRIER();
#pragma unroll
    for (int f = 0; f < 2 * MH; ++f) low[f] = frag<X_LOW>(f, 0);
#pragma unroll
    for (int f = 0; f < 2 * NH; ++f) b0[f] = frag<W_LOW>(f, 0);
    TILE_WAIT_LDS();
    TILE_BARRIER();
    load_unit<X_LOW>(0, at);
    int slot = 0;
    if constexpr (INNER == QUARTER_ODD) {
      stage<ST + 1>(slot, low, high, b0, b1);
      all_but_odd(stages - 1, slot, low, high, b1, b0);
    } else
      all_but_odd(stages, slot, low, high, b0, b1);
  }
};

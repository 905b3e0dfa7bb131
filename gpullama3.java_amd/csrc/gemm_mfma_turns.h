// A tile of the products in bfloat16 whose waves take turns, for the kernels of one tile (gemm_mfma.hip) and of two (gemm_mfma_two.hip; files of
// their own because the compiler takes minutes over either).
#pragma once
#include "common.h"
#include "lds_loads.h"
#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

enum { MF_STORE = 0, MF_ADD = 1, MF_GATED = 2 };

#define MF_BK 64

// What an epilogue may apply besides a bias: a factor per output column (store and add epilogues, after the bias),
// and the gated rule's bound and shift (gl3_gated; 0, 0: none).
struct MfExtras {
  const float* col_scale;
  float act_limit, act_shift;
};

// ---- tiles of 256 x 256, 128 rows x 256 and 128 x 128 over whole steps of 64 k: operands straight from memory into shared memory, waves in two groups
// that take turns.
//
// Eight waves; wave w's rows of A are 64 of each half of the tile's (group w / 4), its rows of W 32 of each half (gated:
// half 0 holds gate rows, half 1 the up rows of the same columns). A step of 64 k is four phases, one pair of halves
// each: (A0, W0), (A0, W1), (A1, W1), (A1, W0). A phase is a memory part (operands from shared memory to registers, a half
// tile of a later step from memory to shared memory) and sixteen 16x16x32 matrix instructions, with a barrier after each
// part; the second group runs one part behind the first, so on every SIMD one wave's matrix instructions run while the
// other wave's memory part does. Without that lag the same loop is 19% slower (1.24 against 1.50 PFLOP/s at 8,192 x 8,192 x
// 4,096). What bounds it now is the power budget: the clock stands at 1.2 to 1.65 GHz of 2.4, the matrix cores are busy 83 to 85% of
// a CU's cycles (gate/up and plain products of 8,192 rows, K = 4,096), and with the 32x32x16 instruction, whose accumulators pass
// through the registers twice as often per flop, the same loop lost 11%.
// (8,192 x 28,672 x 4,096: the kernel without turns 1,680 us, this one 1,283.)
//
// Halves of A and of W: AH = WH = 2 is the tile of 256 x 256. AH = 1: 128 rows x 256, two phases a step, a third step in shared
// memory instead of registers read ahead (2,048 rows, 3,072 columns, K = 2,048: 42 -> 30 us; 512 rows of the 3B layers' gate/up
// product: 59 -> 48 us). AH = WH = 1: 128 x 128, one phase a step, four steps in shared memory (150 rows of the 1B layers' down
// projection in eight slices of K 31 -> 24 us with its norm; 512 rows, 5,120 columns, K = 3,072 33 -> 25 us).
// The smaller tiles ask the second-level caches for up to twice the bytes per flop: 128 x 128 on every CU for 16 KB a clock, all
// that they give.
//
// AH = 2: registers are read a part or two before they are used: in the memory part of phase 0 W0 and half of A1, of phase 1 the
// rest of A1, of phases 2 and 3 the next step's A0 and W1. A half tile's place in shared memory is written for the step after
// next as soon as both groups have read it (their reads have returned: lgkmcnt before the barrier in front of the part
// that asks), and the loads are only waited for where the next barrier hands them out, so six to eight are on their way
// through a whole step:
//   part of phase 0:                          reads of this step's A0, W1 are behind every wave after it
//   part of phase 1: load A0, W1 of step + 2; wait until 8 are out: A0, W1 of step + 1 have come (read from phase 2 on)
//   part of phase 2: load W0 of step + 2;     reads of this step's A1 are behind every wave after it
//   part of phase 3: load A1 of step + 2;     wait until 8 are out: W0, A1 of step + 1 have come (read from phase 0 on)
// Steps beyond the last read the last again, so that the counts hold; nothing is in flight when a block ends.
//
// In shared memory rows of A (and of W as stored) are 128 bytes in eight pieces of 16, piece c of row r at place
// c ^ (r / 2 % 8): the sixteen rows that sixteen lanes read at one piece meet all banks once. W in a copy's order lies as
// the operands want it, [strip of 16][k-step of 32][lane][16 bytes].
// Byte offset, from the address that mf_w_base gives, of the 16 bytes of W at row `row`, piece k .. k + 7 of the first step,
// and how far a step of 64 k lies behind the one before it.
template <int WT>
__device__ __forceinline__ unsigned mf_w_offset(int row, int k, long ldw, int w_steps, const int* w_pos, int n0) {
  return WT == 1   ? (unsigned)gl3_operand_offset(w_pos ? w_pos[row] : row, k, w_steps) * 2
         : WT == 2 ? (unsigned)gl3_packed_offset(row, k, w_steps) * 2
                   : (unsigned)((long)(row - n0) * ldw + k) * 2;
}

// bytes of shared memory of a tile: its steps in turn, each A's halves, then W's
constexpr int mf_stages(int AH, int WH) { return AH == 2 ? 2 : WH == 2 ? 3 : 4; }
constexpr int mf_lds(int AH, int WH) { return mf_stages(AH, WH) * (AH + WH) * 16384; }

struct MfTurns {
  const bf16_t* A;
  const bf16_t* W;
  void* C;
  int M, N, K;
  long lda, ldw, ldc;
  int k_per_slice;
  float* P;
  long p_stride, ldp;
  const float* bias;
  int act, w_steps;
  const int* w_pos;
  MfExtras ex;
};
// Blocks of tiles_m x tiles_n tiles, the first at row m_first; `tile`: its number in their order (block -> tile as above).
template <int EPI, typename TC, int WT, int AH, int WH>
__device__ __forceinline__ void mf_turns_tile(char* lds, const MfTurns& a, int m_first, int tiles_m, int tiles_n, int group_m, int tile, int slice) {
  const bf16_t* __restrict__ const A = a.A;
  const bf16_t* __restrict__ const W = a.W;
  TC* __restrict__ const C = (TC*)a.C;
  float* __restrict__ const P = a.P;
  const float* __restrict__ const bias = a.bias;
  const int* __restrict__ const w_pos = a.w_pos;
  const int M = a.M, N = a.N, K = a.K, k_per_slice = a.k_per_slice, act = a.act, w_steps = a.w_steps;
  const long lda = a.lda, ldw = a.ldw, ldc = a.ldc, p_stride = a.p_stride, ldp = a.ldp;
  const MfExtras ex = a.ex;
  constexpr int NCOLS = (EPI == MF_GATED ? 64 : 128) * WH;
  constexpr int STAGE = (AH + WH) * 16384;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wm = wave >> 2, wn = wave & 3;
  const int lr = lane & 15, lq = lane >> 4;
  const int band = tile / (group_m * tiles_n), in_band = tile % (group_m * tiles_n);
  const int band_rows = min(group_m, tiles_m - band * group_m);
  const int m0 = m_first + (band * group_m + in_band % band_rows) * (128 * AH);
  const int n0 = (in_band / band_rows) * NCOLS;
  // (the last of many slices may have no step left: it stores zeros)
  const int k_begin = min(slice * k_per_slice, K - 64), steps = max(0, (min(K, (slice + 1) * k_per_slice) - slice * k_per_slice) >> 6);

  // who brings what: a half tile is 16 pieces of 1 KB, two a wave
  const i32x4 a_buf = mf_rsrc(A + (long)m0 * lda + k_begin);
  const i32x4 w_buf = mf_rsrc(WT ? W + (long)(k_begin >> 6) * (WT == 1 ? 1024 : 512) : W + (long)n0 * ldw + k_begin);
  constexpr unsigned W_STEP = WT == 1 ? 2048 : WT == 2 ? 1024 : 128;
  unsigned ao[2][2], wo[2][2];      // (AH 1: the first half of A alone)
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int piece = wave * 2 + i;
      const int row = piece * 8 + (lane >> 3), at = ((lane & 7) ^ ((row >> 1) & 7)) * 8;      // (rows of 128 bytes)
      ao[h][i] = (unsigned)((long)(min(m0 + h * 128 + row, M - 1) - m0) * lda + at) * 2;
      const int w_row = WT ? (piece >> 1) * 16 + lr : row, w_k = WT ? (piece & 1) * 32 + lq * 8 : at;
      // (gated: half 1 are the up rows; with one half every other strip of 16 is, behind the gate rows of its columns)
      const bool up = EPI == MF_GATED && (WH == 2 ? h == 1 : (w_row >> 4) & 1);
      const int col = EPI != MF_GATED ? h * 128 + w_row : WH == 2 ? w_row : (w_row >> 5) * 16 + (w_row & 15);
      const int n = min(n0 + col, N - 1) + (up ? N : 0);
      wo[h][i] = mf_w_offset<WT>(n, w_k, ldw, w_steps, w_pos, n0);
    }
  const unsigned lds0 = (unsigned)(unsigned long)(__attribute__((address_space(3))) char*)lds + wave * 2048;
  // (`place`: the byte where the step lies in shared memory)
  auto load_a = [&](int h, int t, int place) {
    const unsigned s = (unsigned)max(0, min(t, steps - 1)) * 128;
#pragma unroll
    for (int i = 0; i < 2; ++i) mf_dma16(lds0 + place + h * 16384 + i * 1024, ao[h][i], a_buf, s);
  };
  auto load_w = [&](int h, int t, int place) {
    const unsigned s = (unsigned)max(0, min(t, steps - 1)) * W_STEP;
#pragma unroll
    for (int i = 0; i < 2; ++i) mf_dma16(lds0 + place + AH * 16384 + h * 16384 + i * 1024, wo[h][i], w_buf, s);
  };

  f32x4 acc[AH][4][WH][2];    // [half of A][16 rows][half of W][16 rows]
#pragma unroll
  for (int i = 0; i < 8 * AH * WH; ++i) (&acc[0][0][0][0])[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 af[AH][4][2], wf[WH][2][2];      // [half][16 rows][k-step of 32]
  const char* a_at = lds + (wm * 64 + lr) * 128;
  const char* w_at = lds + AH * 16384 + (WT ? wn * 4096 + lane * 16 : (wn * 32 + lr) * 128);
  const int twist = (lr >> 1) & 7;
  auto read_a = [&](int h, int place, int ks) {
#pragma unroll
    for (int tm = 0; tm < 4; ++tm)
      af[h][tm][ks] = *(const bf16x8*)(a_at + place + h * 16384 + tm * 2048 + (((ks * 4 + lq) ^ twist) << 4));
  };
  auto read_w = [&](int h, int place) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int tn = 0; tn < 2; ++tn)
        wf[h][tn][ks] = *(const bf16x8*)(w_at + place + h * 16384 + tn * 2048 + (WT ? ks * 1024 : ((ks * 4 + lq) ^ twist) << 4));
  };
  auto products = [&](int ah, int wh) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int tn = 0; tn < 2; ++tn)
#pragma unroll
        for (int tm = 0; tm < 4; ++tm)
          acc[ah][tm][wh][tn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[wh][tn][ks], af[ah][tm][ks], acc[ah][tm][wh][tn], 0, 0, 0);
  };

  // The rows that an add reads. With one half of A there are registers for all of them beside the sums: they are asked for in the
  // last three steps in the place of loads beyond the last step (as many, so that the counts hold), and come while those are
  // multiplied (beyond the matrix: its last row and columns again). In the slices of their plans, 2,048 rows of the 1B layers: output projection
  // 25.5 -> 23.0 us, down 61.9 -> 60.0; 512 rows of the 3B layers 20.7 -> 19.1 and 32.2 -> 31.4; 4,096 rows x 2,048 x 2,048 38.3 -> 35.5. The tile of
  // 256 x 256 has no registers left and reads them behind the last step.
  const int col0 = n0 + (EPI == MF_GATED && WH == 1 ? wn * 16 : wn * 32), row0 = m0 + wm * 64 + lr;
  // (a row's last columns may be fewer than four; an add in the tile of 256 x 256 has no registers left for that)
  constexpr bool ENDS = EPI != MF_ADD || AH == 1;
  const bool vec = ldc % 4 == 0 && (ENDS ? N >= 4 : N % 4 == 0) && (uintptr_t)C % (4 * sizeof(TC)) == 0;
  typedef TC tc4 __attribute__((ext_vector_type(4)));
  constexpr bool ADDS = EPI == MF_ADD;
  tc4 old[ADDS ? 8 * WH : 1];
  auto ask_old = [&](int ah, int i) {
    const int tm = i / (2 * WH), wh = i / 2 % WH, tn = i % 2;
    old[ADDS ? i : 0] = *(const tc4*)(C + (long)min(row0 + ah * 128 + tm * 16, M - 1) * ldc + min(col0 + wh * 128 + tn * 16 + lq * 4, (N & ~3) - 4));
  };
  const bool early = ADDS && AH == 1 && vec && slice == 0 && steps >= 3;
  // A bias of 32-bit sums is asked for in front of the steps, where there are registers for it (not in the tile of 256 x 256). Read behind them,
  // between the stores, 66 rows of 2,048 x 2,048 took 20.5 us, so 17.7; 2,048 rows of 3,072 x 3,072 47.3 and 40.6.
  constexpr bool BIAS = EPI == MF_STORE && AH == 1 && sizeof(TC) == 4;
  f32x4 bias_at[BIAS ? 2 * WH : 1];
  if constexpr (BIAS) {
    if (bias && N >= 4) {
#pragma unroll
      for (int i = 0; i < 2 * WH; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) bias_at[i][j] = bias[min(col0 + i / 2 * 128 + i % 2 * 16 + lq * 4, N - 4) + j];
    }
  }
  const int plain_steps = early ? steps - 3 : steps;

  if constexpr (AH == 2) {
    load_a(0, 0, 0);
    load_w(1, 0, 0);
    load_w(0, 0, 0);
    load_a(1, 0, 0);
    load_a(0, 1, STAGE);
    load_w(1, 1, STAGE);
    load_w(0, 1, STAGE);
    load_a(1, 1, STAGE);
    mf_wait_loads<8>();
    mf_barrier();
    if (wm == 1) mf_barrier();          // the second group runs a part behind
    read_a(0, 0, 0);
    read_a(0, 0, 1);
    read_w(1, 0);
    for (int t = 0, here = 0; t < steps; ++t, here = STAGE - here) {
      const int there = STAGE - here;
      read_w(0, here);
      __builtin_amdgcn_sched_barrier(0);
      read_a(1, here, 0);
      mf_wait_reads<4>();
      mf_barrier();
      products(0, 0);
      mf_barrier();
      read_a(1, here, 1);
      load_a(0, t + 2, here);
      load_w(1, t + 2, here);
      mf_wait_loads<8>();
      mf_barrier();
      products(0, 1);
      mf_barrier();
      read_a(0, there, 0);
      load_w(0, t + 2, here);
      mf_wait_reads<4>();
      mf_barrier();
      products(1, 1);
      mf_barrier();
      read_a(0, there, 1);
      read_w(1, there);
      load_a(1, t + 2, here);
      mf_wait_loads<8>();
      mf_barrier();
      products(1, 0);
      mf_barrier();
    }
  } else if constexpr (WH == 2) {
    // 128 rows of A: two phases a step, (A, W0) and (A, W1), three steps in shared memory. What a part reads it uses at
    // once; a place is written again, for the step three further, in the part after both groups have read it.
    load_a(0, 0, 0);
    load_w(0, 0, 0);
    load_w(1, 0, 0);
    load_a(0, 1, STAGE);
    load_w(0, 1, STAGE);
    load_w(1, 1, STAGE);
    load_a(0, 2, 2 * STAGE);
    load_w(0, 2, 2 * STAGE);
    mf_wait_loads<12>();
    mf_barrier();
    if (wm == 1) mf_barrier();
    int here = 0, before = 2 * STAGE;
    auto step = [&](int t, auto tail) {       // tail: 0, or the step is the first, second or third of the last three and asks for rows
      constexpr int TAIL = decltype(tail)::value;
      read_a(0, here, 0);
      read_a(0, here, 1);
      read_w(0, here);
      if constexpr (TAIL < 2) load_w(1, t + 2, before);
      else {
#pragma unroll
        for (int i = 0; i < 2; ++i) ask_old(0, (TAIL == 2 ? 4 : 10) + i);
      }
      mf_wait_loads<12>();              // this step's W1 has come
      mf_wait_reads<0>();
      mf_barrier();
      products(0, 0);
      mf_barrier();
      read_w(1, here);
      if constexpr (TAIL == 0) {
        load_a(0, t + 3, here);
        load_w(0, t + 3, here);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) ask_old(0, (TAIL - 1) * 6 + i);
      }
      mf_wait_loads<12>();              // the next step's A and W0 have
      mf_wait_reads<0>();
      mf_barrier();
      products(0, 1);
      mf_barrier();
      before = here;
      here = here == 2 * STAGE ? 0 : here + STAGE;
    };
    for (int t = 0; t < plain_steps; ++t) step(t, std::integral_constant<int, 0>{});
    if constexpr (ADDS) {
      if (early) {
        step(steps - 3, std::integral_constant<int, 1>{});
        step(steps - 2, std::integral_constant<int, 2>{});
        step(steps - 1, std::integral_constant<int, 3>{});
      }
    }
  } else {
    // 128 x 128: one phase a step, four steps in shared memory.
    load_a(0, 0, 0);
    load_w(0, 0, 0);
    load_a(0, 1, STAGE);
    load_w(0, 1, STAGE);
    load_a(0, 2, 2 * STAGE);
    load_w(0, 2, 2 * STAGE);
    mf_wait_loads<8>();
    mf_barrier();
    if (wm == 1) mf_barrier();
    int here = 0, before = 3 * STAGE;
    auto step = [&](int t, auto tail) {       // (tail as above; the third asks for nothing but repeats the last step)
      constexpr int TAIL = decltype(tail)::value;
      read_a(0, here, 0);
      read_w(0, here);
      read_a(0, here, 1);
      if constexpr (TAIL == 1 || TAIL == 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i) ask_old(0, (TAIL - 1) * 4 + i);
      } else {
        load_a(0, t + 3, before);       // (where the step before lay, which both groups have read)
        load_w(0, t + 3, before);
      }
      mf_wait_loads<8>();               // the next step has come
      mf_wait_reads<0>();
      mf_barrier();
      products(0, 0);
      mf_barrier();
      before = here;
      here = here == 3 * STAGE ? 0 : here + STAGE;
    };
    for (int t = 0; t < plain_steps; ++t) step(t, std::integral_constant<int, 0>{});
    if constexpr (ADDS) {
      if (early) {
        step(steps - 3, std::integral_constant<int, 1>{});
        step(steps - 2, std::integral_constant<int, 2>{});
        step(steps - 1, std::integral_constant<int, 3>{});
      }
    }
  }
  if (wm == 0) mf_barrier();
  mf_wait_loads<0>();                 // (what was asked for beyond the last step has landed)

  // The sums go to memory straight from the registers: a lane holds four consecutive columns of a row (4 * (lane / 16) of the 16
  // of a 16 x 16 tile, row lane % 16). Gate and up value of a column are the same lane's, so the gated rule needs nobody else's.
  // 16-bit outputs: two tiles' lanes hand each other half of their columns and store 16 bytes of eight (64 consecutive bytes of
  // sixteen rows an instruction, 32 where a wave has 16 columns); 32-bit ones are 16 bytes a lane as they are. The rule of an
  // epilogue's extras is looked at once, not per element: most products have none, and then the code is short. Against the sums
  // through shared memory, a wave on whole rows: gate/up of 2,048 rows of the 1B layers 123 -> 104 us (93 without any epilogue), of
  // 16,384 910 -> 790, of 8,192 of the 8B layers 1,379 -> 1,283; QKV of 2,048 rows 30.1 -> 27.8, of 512 rows of the 3B layers
  // 26.1 -> 24.7; the output projection of 5,886 rows of the 3B layers, which reads the rows it adds to, 137 -> 132 (110 without);
  // a head's 2,221 x 128,256 floats, bound by their way to memory, 1,048 to 1,090 on both.
  // (plain_t: no extras; whole_t: rows of whole eights of columns, fours if 32 bits wide. Looked at a piece of a row at a time, gate/up took 0.9% longer.)
  auto finish = [&](auto plain_t, auto whole_t) {
    constexpr bool PLAIN = decltype(plain_t)::value, WHOLE = !ENDS || decltype(whole_t)::value;
    // columns n .. n + 3, ready to be stored (an add's old values aside)
    auto sums = [&](int ah, int tm, int wh, int tn, int n) {
      f32x4 v = acc[ah][tm][wh][tn];
      f32x4 u = v;
      if constexpr (EPI == MF_GATED) u = WH == 2 ? acc[ah][tm][WH - 1][tn] : acc[ah][tm][0][1];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (PLAIN) {
          if (EPI == MF_GATED) v[j] = gl3_activation<true>(v[j], GL3_ACT_SILU) * u[j];
        } else {
          const int at = min(n + j, N - 1);
          if (bias) {
            v[j] += BIAS && WHOLE ? bias_at[BIAS ? wh * 2 + tn : 0][j] : bias[at];
            if (EPI == MF_GATED) u[j] += bias[N + at];
          }
          if (EPI == MF_GATED) v[j] = gl3_gated<true>(v[j], u[j], act, ex.act_limit, ex.act_shift);
          else if (ex.col_scale) v[j] *= ex.col_scale[at];
        }
      }
      return v;
    };
    constexpr int HALVES = EPI == MF_GATED ? 1 : WH, TILES = EPI == MF_GATED && WH == 1 ? 1 : 2;      // of output columns
    if constexpr (sizeof(TC) == 2) {
      if (ldc % 8 == 0 && (uintptr_t)C % 16 == 0) {
        auto pack = [&](int ah, int tm, int wh, int tn) {
          const f32x4 v = sums(ah, tm, wh, tn, col0 + wh * 128 + tn * 16 + lq * 4);
          return __builtin_bit_cast(u32x2, bf16x4{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]});
        };
        // (lanes of odd lq get the columns of tile b, of even ones those of a: eight from column 8 * (lq / 2))
        auto put = [&](u32x2 a, u32x2 b, int row, int n) {
          const auto lo = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
          const auto hi = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
          const u32x4 eight = {lo[0], hi[0], lo[1], hi[1]};
          TC* c = C + (long)row * ldc + n;
          if (row >= M || n >= N) return;
          if (WHOLE || n + 8 <= N) *(u32x4*)c = eight;
          else {
            const bf16x8 each = __builtin_bit_cast(bf16x8, eight);
#pragma unroll
            for (int j = 0; j < 7; ++j)
              if (n + j < N) c[j] = each[j];
          }
        };
#pragma unroll
        for (int ah = 0; ah < AH; ++ah) {
          if constexpr (TILES == 1) {
#pragma unroll
            for (int tm = 0; tm < 4; tm += 2)
              put(pack(ah, tm, 0, 0), pack(ah, tm + 1, 0, 0), row0 + ah * 128 + (tm + (lq & 1)) * 16, col0 + (lq >> 1) * 8);
          } else {
#pragma unroll
            for (int tm = 0; tm < 4; ++tm)
#pragma unroll
              for (int wh = 0; wh < HALVES; ++wh)
                put(pack(ah, tm, wh, 0), pack(ah, tm, wh, 1), row0 + ah * 128 + tm * 16, col0 + wh * 128 + (lq & 1) * 16 + (lq >> 1) * 8);
          }
        }
        return;
      }
    }
#pragma unroll
    for (int ah = 0; ah < AH; ++ah) {
      if (ADDS && !early) {             // (all asked for before the first is needed)
#pragma unroll
        for (int i = 0; i < 8 * WH; ++i) ask_old(ah, i);
      }
#pragma unroll
      for (int tm = 0; tm < 4; ++tm)
#pragma unroll
        for (int wh = 0; wh < HALVES; ++wh)
#pragma unroll
          for (int tn = 0; tn < TILES; ++tn) {
            const int n = col0 + wh * 128 + tn * 16 + lq * 4, row = row0 + ah * 128 + tm * 16;
            const f32x4 v = sums(ah, tm, wh, tn, n);
            if (row >= M || n >= N) continue;
            tc4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = from_f32<TC>(ADDS ? to_f32<TC>(old[ADDS ? (tm * WH + wh) * 2 + tn : 0][j]) + v[j] : v[j]);
            TC* c = C + (long)row * ldc + n;
            if (WHOLE || n + 4 <= N) {
              *(tc4*)c = o;
            } else {                    // (their old values are not among those asked for)
#pragma unroll
              for (int j = 0; j < 3; ++j)
                if (n + j < N) c[j] = from_f32<TC>(ADDS ? to_f32<TC>(c[j]) + v[j] : v[j]);
            }
          }
    }
  };
  // Outputs whose rows do not begin at whole fours of columns: single elements from the registers are sixteen rows an
  // instruction, so the sums go through shared memory, half the tile's rows at a time, and a wave stores 64 consecutive columns. Row r's
  // sixteen bytes c lie at place c ^ (r % 16): no two lanes of a write meet in a bank. Against element by element from the registers:
  // 512 x 50,257 x 1,024 100 -> 66 us (58 where rows are whole eights), 2,048 x 32,001 x 2,048 316 -> 238 (239), the same in 16 bits
  // 280 -> 223 (198), an add into 2,048 x 2,050 49 -> 36 (29). Rows of any width whose beginnings are whole fours need none of this: their
  // last columns are stored one by one (2,048 x 32,001, rows 32,008 apart, 313 -> 231).
  auto by_rows = [&](auto before, auto store) {
    constexpr int ROW = 512 * WH, COLS = NCOLS / 64, RPT = 8 / COLS;      // bytes of a row of sums; a lane's columns of a row, rows at a time
#pragma unroll
    for (int ah = 0; ah < AH; ++ah) {
      mf_barrier();                    // (everybody has read what lay here)
#pragma unroll
      for (int tm = 0; tm < 4; ++tm)
#pragma unroll
        for (int wh = 0; wh < WH; ++wh)
#pragma unroll
          for (int tn = 0; tn < 2; ++tn)
            *(f32x4*)(lds + (wm * 64 + tm * 16 + lr) * ROW + (((wh * 32 + wn * 8 + tn * 4 + lq) ^ lr) << 4)) = acc[ah][tm][wh][tn];
      mf_wait_reads<0>();
      mf_barrier();
      const int rows = min(128, M - m0 - ah * 128);
      auto put = [&](int r, int c, float was) {
        const int quad = c >> 2, gate = EPI == MF_GATED && WH == 1 ? (quad >> 2) * 8 + (quad & 3) : quad, up = WH == 1 ? gate + 4 : gate + 32;
        const float v = *(const float*)(lds + r * ROW + ((gate ^ (r & 15)) << 4) + (c & 3) * 4);
        float u = 0.f;
        if constexpr (EPI == MF_GATED) u = *(const float*)(lds + r * ROW + ((up ^ (r & 15)) << 4) + (c & 3) * 4);
        if (n0 + c < N) store(v, u, was, m0 + ah * 128 + r, n0 + c);
      };
      if constexpr (ADDS) {            // (eight old values asked for before the first is needed)
        for (int r0 = wave; r0 < rows; r0 += 8 * RPT) {
          float was[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) was[i] = before(m0 + ah * 128 + min(r0 + i / COLS * 8, rows - 1), min(n0 + lane + i % COLS * 64, N - 1));
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (r0 + i / COLS * 8 < rows) put(r0 + i / COLS * 8, lane + i % COLS * 64, was[i]);
        }
      } else {
#pragma unroll 2
        for (int r = wave; r < rows; r += 8)
#pragma unroll
          for (int c = lane; c < NCOLS; c += 64) put(r, c, 0.f);
      }
    }
  };
  const bool plain = !bias && !ex.col_scale && (EPI != MF_GATED || (act == GL3_ACT_SILU && ex.act_limit <= 0.f && ex.act_shift == 0.f));
  if (EPI != MF_GATED && slice > 0) {
    float* const p = P + (long)(slice - 1) * p_stride;
    if (ldp % 4 != 0 || N % 4 != 0 || (uintptr_t)p % 16 != 0) {
      by_rows([](int, int) { return 0.f; }, [&](float v, float, float, int m, int n) { p[(long)m * ldp + n] = ex.col_scale ? v * ex.col_scale[n] : v; });
      return;
    }
#pragma unroll
    for (int ah = 0; ah < AH; ++ah)
#pragma unroll
      for (int tm = 0; tm < 4; ++tm)
#pragma unroll
        for (int wh = 0; wh < WH; ++wh)
#pragma unroll
          for (int tn = 0; tn < 2; ++tn) {
            const int n = col0 + wh * 128 + tn * 16 + lq * 4, row = row0 + ah * 128 + tm * 16;
            f32x4 v = acc[ah][tm][wh][tn];
            if (row >= M || n >= N) continue;
            if (ex.col_scale) {
#pragma unroll
              for (int j = 0; j < 4; ++j) v[j] *= ex.col_scale[min(n + j, N - 1)];
            }
            *(f32x4*)(p + (long)row * ldp + n) = v;
          }
    return;
  }
  if (!vec) {
    auto before = [&](int m, int n) { return ADDS ? to_f32<TC>(C[(long)m * ldc + n]) : 0.f; };
    by_rows(before, [&](float v, float u, float was, int m, int n) {
      if (bias) v += bias[n];
      if constexpr (EPI == MF_GATED) {
        if (bias) u += bias[N + n];
        v = plain ? gl3_activation<true>(v, GL3_ACT_SILU) * u : gl3_gated<true>(v, u, act, ex.act_limit, ex.act_shift);
      } else if (ex.col_scale) {
        v *= ex.col_scale[n];
      }
      C[(long)m * ldc + n] = from_f32<TC>(ADDS ? was + v : v);
    });
    return;
  }
  if (ENDS && N % (sizeof(TC) == 2 ? 8 : 4) != 0) finish(std::false_type{}, std::false_type{});
  else if (plain) finish(std::true_type{}, std::true_type{});
  else finish(std::false_type{}, std::true_type{});
}

// A launch of gemm_mfma_two_tiles_kernel: W in order w_order (gated: 0 or 1), small tiles of 128 rows x 256 (small 5) or 128 x 128 (1).
template <int EPI, typename TC>
int mf_launch_two_tiles(int w_order, int small, const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc, int slices, float* P,
                        long p_stride, long ldp, const float* bias, int act, int w_steps, const int* w_pos, MfExtras ex, int big_m, hipStream_t stream);

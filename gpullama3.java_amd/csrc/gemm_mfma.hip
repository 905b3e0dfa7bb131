// C[M,N] = A[M,K] . W[N,K]^T in bfloat16 on the matrix cores for many rows of A: the
// products of a prefill step. 32-bit accumulation; W is row-major [out, in]
// (J/core/model/tensor/FloatTensor.java:98-100).
//
// A block is WM x WN waves; each wave owns 64 x 64 (or 32 x 64) of the block's tile of C as
// 2 x 2 (1 x 2) tiles of the 32x32x16 instruction: sixteen waves on 256 x 256 for large products,
// eight waves on 128 x 128 otherwise. For the gated epilogue a W tile holds the gate rows of
// half as many output columns and the matching up rows. K advances in steps of 64 through two
// buffers in shared memory: while a step's products run out of one, the next step's operands go
// from registers into the other and the step after that travels from memory to registers; one
// barrier a step. Rows in shared memory are padded by 16 bytes so that the 32 lanes that read one
// column of 16-byte operands hit different banks.
// Blocks are numbered so that each XCD (whose second-level cache is its own) works on a
// contiguous range of tiles, ordered so that the tiles it holds at one time form a rectangle
// and share their panels of A and of W.
//
// Tiles of 256 x 256, 128 rows x 256 and 128 x 128 over whole steps of 64 k have a kernel of their own (gemm_mfma_turns_kernel, below).
//
// Epilogues as in gemm_generic.hip: store, add into a float matrix, gated.
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
#define MF_LD (MF_BK + 8)   // padded row, in elements

// What an epilogue may apply besides a bias: a factor per output column (store and add epilogues, after the bias),
// and the gated rule's bound and shift (gl3_gated; 0, 0: none).
struct MfExtras {
  const float* col_scale;
  float act_limit, act_shift;
};

// WM x WN waves; a wave owns (32*TM) x 64 of the tile.
template <int EPI, typename TC, int TM, int WM, int WN, int WT = 0>
__global__ __launch_bounds__(64 * WM * WN) void gemm_mfma_kernel(const bf16_t* __restrict__ A,
                                                                  const bf16_t* __restrict__ W, TC* __restrict__ C,
                                                                  int M, int N, int K, long lda, long ldw, long ldc,
                                                                  int tiles_m, int tiles_n, int group_m, int k_per_slice,
                                                                  float* __restrict__ P, long p_stride, long ldp,
                                                                  const float* __restrict__ bias, int act, int w_steps,
                                                                  const int* __restrict__ w_pos, MfExtras ex) {
  constexpr int NT = 64 * WM * WN;                       // threads
  constexpr int BM = 32 * TM * WM;                       // rows of a block
  constexpr int BN = 64 * WN;                            // rows of W of a block
  constexpr int NCOLS = (EPI == MF_GATED) ? BN / 2 : BN; // output columns of a block
  constexpr int NA = BM * 8 / NT;                        // 16-byte chunks of A per thread and k-step
  constexpr int NWC = BN * 8 / NT;                       // and of W
  static_assert(BM * 8 % NT == 0 && BN * 8 % NT == 0, "tile does not divide over the threads");
  __shared__ __attribute__((aligned(16))) bf16_t As[2][BM][MF_LD];
  __shared__ __attribute__((aligned(16))) bf16_t Ws[2][BN][MF_LD];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wm = wave / WN, wn = wave % WN;
  const int lr = lane & 31, lh = lane >> 5;

  // block -> tile: 8 XCDs take turns on consecutive block ids; give each a contiguous range
  const int n_tiles = tiles_m * tiles_n;
  const int per_xcd = (n_tiles + 7) / 8;
  const int tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (tile >= n_tiles) return;
  // the tiles in order: bands of group_m row tiles; inside a band column after column, the band's row
  // tiles of a column one after the other. The tiles that an XCD works on at one time are then a
  // rectangle of group_m row tiles by a few column tiles, which share their rows of A and of W.
  const int band = tile / (group_m * tiles_n), in_band = tile % (group_m * tiles_n);
  const int band_rows = min(group_m, tiles_m - band * group_m);
  const int m0 = (band * group_m + in_band % band_rows) * BM;
  const int n0 = (in_band / band_rows) * NCOLS;

  // global -> register staging in chunks of 16 bytes. An address is a base that the whole block
  // shares (it lives in scalar registers and takes the k-step) plus a 32-bit offset of the thread
  // inside the tile, and every load is unconditional (rows and columns beyond the matrix are
  // clamped to its last ones and their values dropped): no branch around a load, whose registers
  // the compiler would then wait for at once.
  // WT 1: W is the copy in the matrix operands' order alone ([strip of 16 rows][k-step of 32][lane][8], w_steps
  // k-steps a strip, gl3_operand_offset; w_pos, may be null: each row's place in a copy whose strips hold the rows
  // in another order). WT 2: the copy in packed strips of 8 rows (gl3_packed_offset, w_steps steps of 64). A
  // thread's 16 bytes are still 8 consecutive k of one row, only at another place, and go to the same place in
  // shared memory.
  const bf16_t* a_tile = A + (long)m0 * lda;
  const bf16_t* w_tile[2];
  w_tile[0] = WT ? W : W + (long)n0 * ldw;
  w_tile[1] = WT ? W : (EPI == MF_GATED) ? W + ((long)N + n0) * ldw : w_tile[0];
  static_assert(EPI != MF_GATED || (NWC % 2 == 0 && (NT / 8) * (NWC / 2) == BN / 2),
                "gate rows and up rows must fall to different loads of a thread");
  unsigned aoff[NA], woff[NWC];
  int arow_s[NA], wrow_s[NWC], wcol_s[NWC];
  const int scol = (tid & 7) * 8;
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    arow_s[i] = (tid + NT * i) >> 3;
    aoff[i] = (unsigned)(min(m0 + arow_s[i], M - 1) - m0) * (unsigned)lda;
  }
#pragma unroll
  for (int i = 0; i < NWC; ++i) {
    int r = (tid + NT * i) >> 3, c = tid & 7;
    if (WT) {
      // Which 16 bytes of the tile a thread brings is free (they go to their own place in shared memory). In a copy's
      // order 8 rows of a strip at one block of 8 k are a 128-byte line. With the stored order's assignment (eight
      // neighbouring threads: the eight pieces of one row's 64 k) eight threads would touch eight lines, 16 bytes of
      // each, which a CU's first-level cache takes at a third of the rate of whole lines (the products of 2,048 rows
      // were 13 to 20% slower that way). So eight neighbouring threads take one whole line, and a wave the same
      // line of 8 different strips: lane l the row l % 8 of strip l / 8 of its group.
      const int idx = (tid >> 6) * NWC + i, l = tid & 63;
      if (WT == 1) {   // [strip of 16][k-step of 32][k block q][row][8]: 16 lines a strip and step of 64 k
        const int combo = idx & 15;
        r = ((idx >> 4) * 8 + (l >> 3)) * 16 + (combo & 1) * 8 + (l & 7);
        c = (combo >> 3) * 4 + ((combo >> 1) & 3);
      } else {         // [strip of 8][step of 64 k][k block q][half][row][8]: 8 lines a strip and step
        const int combo = idx & 7;
        r = ((idx >> 3) * 8 + (l >> 3)) * 8 + (l & 7);
        c = (combo & 1) * 4 + (combo >> 1);
      }
    }
    wrow_s[i] = r;
    wcol_s[i] = c * 8;
    // (gated: the tile's second half of rows are the up rows of the same columns; in a copy's order which half a
    // load falls into goes by its row, not by its number)
    const bool up = EPI == MF_GATED && (WT ? r >= BN / 2 : i >= NWC / 2);
    const int rel = up ? r - BN / 2 : r;
    const int row = min(n0 + rel, N - 1);
    const int wrow = row + (up ? N : 0);
    // (WT: K is a multiple of 64, so a thread's column inside a k-step of 64 is at the same place of every step)
    woff[i] = WT == 1   ? (unsigned)gl3_operand_offset(w_pos ? w_pos[wrow] : wrow, c * 8, w_steps)
              : WT == 2 ? (unsigned)gl3_packed_offset(wrow, c * 8, w_steps)
                        : (unsigned)(row - n0) * (unsigned)ldw;
  }
  // K in slices (blockIdx.y): slice 0 ends in the epilogue proper, the others store their sums
  // as floats into P[slice - 1], for the reader to add up in slice order
  const int slice = blockIdx.y;
  const int k_begin = slice * k_per_slice;
  K = min(K, k_begin + k_per_slice);
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8 ra[NA], rw[NWC];
  bool r_ok = false;                                   // whether the registers hold columns inside K
  auto fetch = [&](int k0) {
    const int kf = min(k0, K - 8);                     // the step after the last one reads the last again
    r_ok = k0 + scol < K;
    const unsigned col = (unsigned)min(scol, K - 8 - kf);
    const bf16_t* ak = a_tile + kf;
#pragma unroll
    for (int i = 0; i < NA; ++i) ra[i] = *(const bf16x8*)(ak + (aoff[i] + col));
    if (WT) {
      // a k-step of 64 lies 2 KB (the operands' order: two k-steps of 32) or 1 KB (the packed strips of 8) further in
      // every strip: the same step for all threads, whose offsets stay what they are
      const bf16_t* wk = w_tile[0] + (long)(min(k0, K - 64) >> 6) * (WT == 1 ? 1024 : 512);   // (the step after the last reads the last again)
#pragma unroll
      for (int i = 0; i < NWC; ++i) rw[i] = *(const bf16x8*)(wk + woff[i]);
    } else {
#pragma unroll
      for (int i = 0; i < NWC; ++i) {
        const bf16_t* wk = w_tile[(EPI == MF_GATED && i >= NWC / 2) ? 1 : 0] + kf;
        rw[i] = *(const bf16x8*)(wk + (woff[i] + col));
      }
    }
  };
  fetch(k_begin);

  f32x16 acc[TM][2];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int jn = 0; jn < 2; ++jn)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][jn][v] = 0.f;

  const int arow = wm * 32 * TM + lr;
  const int wrow0 = (EPI == MF_GATED) ? wn * 32 + lr : wn * 64 + lr;
  const int wrow1 = (EPI == MF_GATED) ? BN / 2 + wn * 32 + lr : wn * 64 + 32 + lr;

  // registers -> shared memory; a step that reaches beyond K drops the columns from K on
  auto store = [&](int buf, int k0) {
    if (k0 + MF_BK <= K) {   // a whole step (the same for the whole block): nothing to drop
#pragma unroll
      for (int i = 0; i < NA; ++i) *(bf16x8*)&As[buf][arow_s[i]][scol] = ra[i];
#pragma unroll
      for (int i = 0; i < NWC; ++i) *(bf16x8*)&Ws[buf][wrow_s[i]][WT ? wcol_s[i] : scol] = rw[i];
    } else {
#pragma unroll
      for (int i = 0; i < NA; ++i) *(bf16x8*)&As[buf][arow_s[i]][scol] = r_ok ? ra[i] : zero;
#pragma unroll
      for (int i = 0; i < NWC; ++i) *(bf16x8*)&Ws[buf][wrow_s[i]][WT ? wcol_s[i] : scol] = r_ok ? rw[i] : zero;
    }
  };
  auto products = [&](int buf, int kk) {
    const int kc = kk * 16 + lh * 8;
    const bf16x8 b0 = *(const bf16x8*)&Ws[buf][wrow0][kc];
    const bf16x8 b1 = *(const bf16x8*)&Ws[buf][wrow1][kc];
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
      const bf16x8 a = *(const bf16x8*)&As[buf][arow + 32 * tm][kc];
      acc[tm][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b0, acc[tm][0], 0, 0, 0);
      acc[tm][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b1, acc[tm][1], 0, 0, 0);
    }
  };
  // Two buffers in shared memory: while a step's products run out of one, the next step's operands
  // (in registers since the step before) are written to the other and the step after that is asked
  // for; one barrier a step.
  store(0, k_begin);
  fetch(k_begin + MF_BK);
  __syncthreads();
  int buf = 0;
  for (int k0 = k_begin; k0 < K; k0 += MF_BK, buf ^= 1) {
#pragma unroll
    for (int kk = 0; kk < MF_BK / 16; ++kk) {
      products(buf, kk);
      if (kk == 0) {
        // behind the first products (which cover the wait for the registers and the address
        // arithmetic); the scheduler may not move the loads or the writes across the fences
        __builtin_amdgcn_sched_barrier(0);
        if (k0 + MF_BK < K) store(buf ^ 1, k0 + MF_BK);
        fetch(k0 + 2 * MF_BK);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();
  }

  // lane holds C[row(v)][col]: row(v) = 8*(v/4) + 4*(lane/32) + v%4 inside a 32x32 tile, col = lane%32.
  // Whole tiles (all but the matrix's last row and column of tiles) store without a test per element.
  auto finish = [&](auto checked_t) {
    constexpr bool CHECKED = decltype(checked_t)::value;
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = m0 + wm * 32 * TM + tm * 32 + (v >> 2) * 8 + lh * 4 + (v & 3);
        if (CHECKED && m >= M) continue;
        if (slice > 0) {
#pragma unroll
          for (int tn = 0; tn < 2; ++tn) {
            const int n = n0 + wn * 64 + tn * 32 + lr;
            if (!CHECKED || n < N)
              P[(long)(slice - 1) * p_stride + (long)m * ldp + n] = ex.col_scale ? acc[tm][tn][v] * ex.col_scale[n] : acc[tm][tn][v];
          }
          continue;
        }
        if (EPI == MF_GATED) {
          const int n = n0 + wn * 32 + lr;
          if (!CHECKED || n < N) {
            float g = acc[tm][0][v], u = acc[tm][1][v];
            if (bias) { g += bias[n]; u += bias[N + n]; }
            C[(long)m * ldc + n] = from_f32<TC>(gl3_gated<true>(g, u, act, ex.act_limit, ex.act_shift));
          }
        } else {
#pragma unroll
          for (int tn = 0; tn < 2; ++tn) {
            const int n = n0 + wn * 64 + tn * 32 + lr;
            if (!CHECKED || n < N) {
              TC* c = C + (long)m * ldc + n;
              float s = acc[tm][tn][v] + (bias ? bias[n] : 0.f);
              if (ex.col_scale) s *= ex.col_scale[n];
              if (EPI == MF_ADD) *c = from_f32<TC>(to_f32<TC>(*c) + s);
              else *c = from_f32<TC>(s);
            }
          }
        }
      }
    }
  };
  if (m0 + BM <= M && n0 + NCOLS <= N) finish(std::false_type{});
  else finish(std::true_type{});
}

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
// (8,192 x 28,672 x 4,096: the kernel above 1,680 us, this one 1,283.)
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

template <int EPI, typename TC, int WT, int AH, int WH>
__global__ __launch_bounds__(512, 2) void gemm_mfma_turns_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                                  TC* __restrict__ C, int M, int N, int K, long lda, long ldw,
                                                                  long ldc, int tiles_m, int tiles_n, int group_m,
                                                                  int k_per_slice, float* __restrict__ P, long p_stride, long ldp,
                                                                  const float* __restrict__ bias, int act, int w_steps,
                                                                  const int* __restrict__ w_pos, MfExtras ex) {
  __shared__ __attribute__((aligned(1024))) char lds[mf_lds(AH, WH)];
  const int n_tiles = tiles_m * tiles_n, per_xcd = (n_tiles + 7) / 8;
  const int tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;       // (block -> tile as above)
  if (tile >= n_tiles) return;
  const MfTurns a{A, W, C, M, N, K, lda, ldw, ldc, k_per_slice, P, p_stride, ldp, bias, act, w_steps, w_pos, ex};
  mf_turns_tile<EPI, TC, WT, AH, WH>(lds, a, 0, tiles_m, tiles_n, group_m, tile, blockIdx.y);
}

// Tiles of 256 x 256 for the first 256 * big_m rows, smaller ones (128 rows x 256, or 128 x 128) for those behind them, the large
// tiles of all slices first. What bounds a product of a few rounds of the chip is the last one: 2,221 rows of the 1B layers' gate/up product are
// 2.25 rounds of 256 x 256 and took three. Here the small tiles fill the CUs that the last whole round of large ones leaves (one launch: they
// start where a CU is done, not where all are), at a lower rate but for a tenth of the rows: 130.5 -> 112.5 us; 5,886 rows of the
// 3B layers' output projection 126 -> 105, of their QKV product's 3,500 111 -> 89. The same sums, whatever the tile: bit for bit.
template <int EPI, typename TC, int WT, int SWH>
__global__ __launch_bounds__(512, 2) void gemm_mfma_two_tiles_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                                      TC* __restrict__ C, int M, int N, int K, long lda, long ldw,
                                                                      long ldc, int big_m, int big_n, int small_m, int small_n, int slices,
                                                                      int k_per_slice, float* __restrict__ P, long p_stride, long ldp,
                                                                      const float* __restrict__ bias, int act, int w_steps,
                                                                      const int* __restrict__ w_pos, MfExtras ex) {
  constexpr int BIG = mf_lds(2, 2), SMALL = mf_lds(1, SWH);
  __shared__ __attribute__((aligned(1024))) char lds[BIG > SMALL ? BIG : SMALL];
  const MfTurns a{A, W, C, M, N, K, lda, ldw, ldc, k_per_slice, P, p_stride, ldp, bias, act, w_steps, w_pos, ex};
  const int big = big_m * big_n, small = small_m * small_n, big_xcd = (big + 7) / 8, small_xcd = (small + 7) / 8;
  int at = blockIdx.x >> 3;                  // (an XCD's blocks: its large tiles slice by slice, then its small ones)
  const int xcd = blockIdx.x & 7;
  if (at < big_xcd * slices) {
    const int slice = at / big_xcd, tile = xcd * big_xcd + at - slice * big_xcd;
    if (tile < big) mf_turns_tile<EPI, TC, WT, 2, 2>(lds, a, 0, big_m, big_n, min(big_m, 4), tile, slice);
  } else {
    at -= big_xcd * slices;
    const int slice = at / small_xcd, tile = xcd * small_xcd + at - slice * small_xcd;
    if (tile < small) mf_turns_tile<EPI, TC, WT, 1, SWH>(lds, a, big_m * 256, small_m, small_n, min(small_m, 8), tile, slice);
  }
}

// What gemm_mfma_turns_kernel is built for: whole steps of 64 k, and byte offsets of 31 bits inside a tile's rows of A and
// inside W (or, as stored, from the tile's first row of W to its last).
static bool turns_takes(int N, int K, long lda, long ldw, bool gated, int w_order) {
  const long rows = gated ? 2L * N : (long)N;
  return K % 64 == 0 && (255 * lda + K) * 2 < (1L << 31) &&
         (w_order ? rows * K * 2 : ((gated ? (long)N : 0) + 255) * ldw * 2 + 2L * K) < (1L << 31);
}

template <int EPI, typename TC, int SWH, int WT>
static int launch_two_tiles(const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc,
                            int slices, float* P, long p_stride, long ldp, const float* bias, int act, int w_steps,
                            const int* w_pos, MfExtras ex, int big_m, hipStream_t stream) {
  const int big_cols = EPI == MF_GATED ? 128 : 256, small_cols = big_cols * SWH / 2;
  const int big_n = (N + big_cols - 1) / big_cols, small_n = (N + small_cols - 1) / small_cols;
  const int small_m = (M - big_m * 256 + 127) / 128;
  const long blocks = (((long)big_m * big_n + 7) / 8 + ((long)small_m * small_n + 7) / 8) * 8 * slices;
  GL3_REQUIRE(big_m > 0 && small_m > 0 && blocks < (1L << 31), "gl3_gemm_mfma: %d rows of tiles of 256 x 256 for %d rows", big_m, M);
  const int k_per_slice = ((K + MF_BK - 1) / MF_BK + slices - 1) / slices * MF_BK;
  gemm_mfma_two_tiles_kernel<EPI, TC, WT, SWH><<<dim3((unsigned)blocks), dim3(512), 0, stream>>>(
      (const bf16_t*)A, (const bf16_t*)W, (TC*)C, M, N, K, lda, ldw, ldc, big_m, big_n, small_m, small_n, slices, k_per_slice, P, p_stride,
      ldp, bias, act, w_steps, w_pos, ex);
  GL3_LAUNCH_CHECK();
  return 0;
}

template <int EPI, typename TC, int TM, int WM, int WN, int WT = 0>
static int launch_shape(const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc,
                        int slices, float* P, long p_stride, long ldp, const float* bias, int act, int w_steps,
                        const int* w_pos, MfExtras ex, hipStream_t stream) {
  const int bm = 32 * TM * WM;
  const int ncols = (EPI == MF_GATED) ? 32 * WN : 64 * WN;
  const int tiles_n = (N + ncols - 1) / ncols;
  const int tiles_m = (M + bm - 1) / bm;
  const long n_tiles = (long)tiles_m * tiles_n;
  const long blocks = ((n_tiles + 7) / 8) * 8;
  GL3_REQUIRE(blocks < (1L << 31), "gl3_gemm_mfma: too many tiles");
  const int k_per_slice = ((K + MF_BK - 1) / MF_BK + slices - 1) / slices * MF_BK;
  // 32 tiles of 256 x 256 (of 128 x 128 as many on the kernel of turns, 64 on the other) run on an XCD at a time: bands of 4 (8)
  // row tiles make them a rectangle of 4 x 8 (8 x 4, 8 x 8), which asks memory for a third of the bytes that one column of
  // 32 row tiles does (3 to 5% of the time of the large products)
  const int group_m = tiles_m < (bm == 256 ? 4 : 8) ? tiles_m : (bm == 256 ? 4 : 8);
  if constexpr (WM == 4 && (WN == 4 || TM == 1)) {
    if (turns_takes(N, K, lda, ldw, EPI == MF_GATED, WT)) {
      gemm_mfma_turns_kernel<EPI, TC, WT, TM, WN / 2><<<dim3((unsigned)blocks, slices), dim3(512), 0, stream>>>(
          (const bf16_t*)A, (const bf16_t*)W, (TC*)C, M, N, K, lda, ldw, ldc, tiles_m, tiles_n, group_m, k_per_slice, P, p_stride,
          ldp, bias, act, w_steps, w_pos, ex);
      GL3_LAUNCH_CHECK();
      return 0;
    }
  }
  gemm_mfma_kernel<EPI, TC, TM, WM, WN, WT><<<dim3((unsigned)blocks, slices), dim3(64 * WM * WN), 0, stream>>>(
      (const bf16_t*)A, (const bf16_t*)W, (TC*)C, M, N, K, lda, ldw, ldc, tiles_m, tiles_n, group_m, k_per_slice, P,
      p_stride, ldp, bias, act, w_steps, w_pos, ex);
  GL3_LAUNCH_CHECK();
  return 0;
}

// The tile the library takes where the caller names none. Where gemm_mfma_turns_kernel takes the product: the tile whose rounds on
// the chip take the least time, a round (a block on every CU: 32 of an XCD, which has an eighth of the tiles of every slice) being
// 0.40 us a step of 64 k and 0.9 us beside them for 128 x 128, 0.60 and 3.0 for 128 rows x 256, 1.0 and 4.5 for 256 x 256. The
// constants rank the tiles and are no times of their own (at 8,192 rows of 28,672 x 4,096 they say 959 us and it is 1,283).
// Measured at 580 sizes (66 to 8,192 rows; QKV, output, gate/up and down products of five layers' sizes, widths of 1,536 to 4,096, those
// into the residual rows in mfma_plan's slices; profiles/tiled_products_tiles.txt): the tile chosen is the fastest of the three or within 5% at
// all but one (1.07). With 0.42 and 4.0 for the first two, which suited epilogues through shared memory, 17 were beyond 5%, 1,024 rows of
// 2,048 x 2,048 20.3 instead of 17.2 us. With rounds of 256 blocks, whatever their XCD, 300 rows of 3,072 x 8,192 took 47.3 instead of 40.8 us.
//
// Where tiles of 256 x 256 end in a round that is mostly empty, two tiles (gemm_mfma_two_tiles_kernel): 8 * rows of large tiles + the small
// tile. An XCD's small tiles go one after the other to the CUs that are done with their large ones; of all divisions with less than a round
// and a half behind the large tiles the one that ends first, where it saves 4% or more. Small tiles that follow large ones take 0.48 us a step and 4.5
// beside them, or 0.60 and 3.0. Measured at 216 sizes (600 to 13,000 rows, the products of three models, up to six divisions of each): the
// choice is within 4% of the best at all but six (1.11). At 97 other sizes where the rule takes two tiles (300 to 16,000 rows, four models'
// products; profiles/two_tiles.txt) they take 0.78 to 1.02 times as long as the single tile taken before, 0.90 on average.
static int choose_turns_shape(int M, int N, int K, int slices, bool gated, bool two) {
  static const int rows[3] = {128, 128, 256}, cols[3] = {128, 256, 256}, shape[3] = {1, 5, 2};
  static const double step_us[3] = {0.40, 0.60, 1.0}, round_us[3] = {0.9, 3.0, 4.5};
  static const double after_step_us[2] = {0.48, 0.60}, after_us[2] = {4.5, 3.0};
  const int steps = (K / 64 + slices - 1) / slices;
  auto per_xcd = [&](int n_rows, int i) {            // blocks of an XCD
    const int columns = gated ? cols[i] / 2 : cols[i];
    return ((long)((n_rows + rows[i] - 1) / rows[i]) * ((N + columns - 1) / columns) + 7) / 8 * slices;
  };
  int best = 0;
  double least = 0;
  for (int i = 0; i < 3; ++i) {
    const double time = (per_xcd(M, i) + 31) / 32 * (steps * step_us[i] + round_us[i]);
    if (!best || time < least) {
      best = shape[i];
      least = time;
    }
  }
  if (!two) return best;
  least *= 0.96;
  const double large = steps * step_us[2] + round_us[2];
  const int most = (M - 1) / 256;
  for (int r = most; r > 0 && (most - r) * per_xcd(256, 2) <= 48; --r) {
    const long big = per_xcd(r * 256, 2);
    const double early = big / 32 * large, late = early + (big % 32 ? large : 0);      // when an XCD's CUs are done with the large tiles
    if (early >= least) continue;
    for (int i = 0; i < 2; ++i) {
      const long small = per_xcd(M - r * 256, i), late_cus = big % 32;
      const double each = steps * after_step_us[i] + after_us[i];
      // the first end of a small tile by which all of them are done
      double end = 0;
      for (int k = 1; end == 0 && early + k * each < least; ++k)
        for (const double t : {early + k * each, late + (k - 1) * each}) {
          if (t < early || (end != 0 && t >= end)) continue;
          const long done = (32 - late_cus) * (long)((t - early) / each + 1e-6) + (t >= late ? late_cus * (long)((t - late) / each + 1e-6) : 0);
          if (done >= small) end = t < late ? late : t;
        }
      if (end != 0 && end < least) {
        best = 8 * r + shape[i];
        least = end;
      }
    }
  }
  return best;
}

// The same where it does not (K in no whole steps of 64, or offsets beyond its 31 bits), on the kernel without turns: 1 (128 x 128),
// 2 (256 x 256) or 5 (128 rows x 256).
// 256 x 256 tiles of sixteen waves, one block a CU, have half the operand traffic per product, and
// that traffic is what bounds the large products; of the 128 x 128 tiles of eight waves two fit a CU and
// overlap each other's waits. A step of 64 columns takes a chip full of the large tiles 1.7 us and a chip
// full of the small ones (twice as many blocks, a quarter of the work each) 1.05 us, and the blocks need
// rounds on the chip: the tile whose rounds take less time is chosen (240 large tiles are one round
// where 960 small ones are two; 276 large ones are two where 1,104 small ones are three).
// A third tile, 128 rows x 256 of sixteen waves of 32 x 64, is for the products in between: more tiles of 128 x 128
// than one for every CU, but not enough work to fill the chip with the large tiles (2,048 rows of the 1B layers'
// QKV product, 384 tiles of 128 x 128 or 192 of 128 x 256: 45 -> 40 us); a step of it takes a full chip about 0.95 us.
// Tiles of 128 x 128 that are at most one a CU run faster than two that share one (0.8 of the time a step).
static int choose_shape(int M, int N, int slices, bool gated) {
  const long small_n = gated ? (N + 63) / 64 : (N + 127) / 128;
  const long big_n = gated ? (N + 127) / 128 : (N + 255) / 256;
  const long small_tiles = (long)((M + 127) / 128) * small_n * slices, wide_tiles = (long)((M + 127) / 128) * big_n * slices;
  const long big_tiles = (long)((M + 255) / 256) * big_n * slices;
  // rounds on the chip, in thousandths: whole rounds, and a last, partly empty one that costs half a round and
  // half of the share of the places it fills (a chip half full works through its blocks faster, not twice as fast)
  auto rounds = [](long tiles, long places) { return tiles / places * 1000 + (tiles % places ? 500 + tiles % places * 500 / places : 0); };
  const long small_cost = rounds(small_tiles, 512) * (small_tiles <= 256 ? 84 : 105), big_cost = rounds(big_tiles, 256) * 170;
  const long wide_cost = rounds(wide_tiles, 256) * (wide_tiles <= 128 ? 119 : 95);
  if (wide_cost < small_cost && wide_cost < big_cost && slices == 1) return 5;
  return big_cost < small_cost ? 2 : 1;
}

template <int EPI, typename TC>
static int launch_mfma(const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc,
                       int slices, float* P, long p_stride, long ldp, const float* bias, int act, int shape, int w_order,
                       const int* w_pos, MfExtras ex, hipStream_t stream) {
  const int w_steps = w_order == 1 ? (K + 31) / 32 : w_order == 2 ? (K + 63) / 64 : 0;
  if (shape < 0) shape = turns_takes(N, K, lda, ldw, EPI == MF_GATED, w_order) ? 0 : -shape;
  constexpr bool TWO = EPI != MF_GATED || sizeof(TC) == 2;
  if (shape == 0)
    shape = turns_takes(N, K, lda, ldw, EPI == MF_GATED, w_order) ? choose_turns_shape(M, N, K, slices, EPI == MF_GATED, TWO)
                                                                  : choose_shape(M, N, slices, EPI == MF_GATED);
  if (shape > 8) {
    GL3_REQUIRE(TWO && turns_takes(N, K, lda, ldw, EPI == MF_GATED, w_order),
                "gl3_gemm_mfma: two tiles are for whole steps of 64 k (K=%d), and for gated values of 16 bits", K);
#define MF_ARGS A, W, C, M, N, K, lda, ldw, ldc, slices, P, p_stride, ldp, bias, act, w_steps, w_pos, ex, shape / 8, stream
#define MF_TWO(WT) (shape % 8 == 1 ? launch_two_tiles<EPI, TC, 1, WT>(MF_ARGS) : launch_two_tiles<EPI, TC, 2, WT>(MF_ARGS))
    if constexpr (TWO) {
      if (w_order == 0) return MF_TWO(0);
      if (w_order == 1) return MF_TWO(1);
      if constexpr (EPI != MF_GATED) return MF_TWO(2);
    }
#undef MF_TWO
#undef MF_ARGS
  }
#define MF_ARGS A, W, C, M, N, K, lda, ldw, ldc, slices, P, p_stride, ldp, bias, act, w_steps, w_pos, ex, stream
  if (w_order) {
    // W is one of its copies in the matrix cores' order (a weight that is held once): the three tiles that the library
    // chooses between
    GL3_REQUIRE(shape == 1 || shape == 2 || shape == 5, "gl3_gemm_mfma: tile shape %d does not read W in a copy's order", shape);
    if (w_order == 1)
      return shape == 1 ? launch_shape<EPI, TC, 1, 4, 2, 1>(MF_ARGS)
             : shape == 2 ? launch_shape<EPI, TC, 2, 4, 4, 1>(MF_ARGS) : launch_shape<EPI, TC, 1, 4, 4, 1>(MF_ARGS);
    if constexpr (EPI != MF_GATED) {
      return shape == 1 ? launch_shape<EPI, TC, 1, 4, 2, 2>(MF_ARGS)
             : shape == 2 ? launch_shape<EPI, TC, 2, 4, 4, 2>(MF_ARGS) : launch_shape<EPI, TC, 1, 4, 4, 2>(MF_ARGS);
    } else {
      GL3_REQUIRE(false, "gl3_gemm_mfma: the gated epilogue reads the copy in the operands' order, not the packed strips of 8 (order %d)", w_order);
    }
  }
  if (shape == 1) return launch_shape<EPI, TC, 1, 4, 2>(MF_ARGS);
  if (shape == 2) return launch_shape<EPI, TC, 2, 4, 4>(MF_ARGS);
  if (shape == 3) return launch_shape<EPI, TC, 4, 2, 4>(MF_ARGS);
  if (shape == 4) return launch_shape<EPI, TC, 2, 4, 2>(MF_ARGS);
  return launch_shape<EPI, TC, 1, 4, 4>(MF_ARGS);
#undef MF_ARGS
}

// N counts output columns: for the gated epilogue W has 2N rows (gate, then up).
// slices > 1 (not with the gated epilogue): K is cut into that many slices; the first ends in the
// epilogue into C, slice s > 0 stores its sums into P[s - 1] ([slices - 1][M][ldp] floats,
// p_stride elements apart), which the caller adds to C in that order.
// bias (may be null; not with slices): N floats (gated: 2N). act: the gated epilogue's activation, with its bound
// and shift (gl3_gated; 0, 0: none). col_scale (may be null; not gated): N floats, a factor per column (every slice's sums
// are multiplied, so the caller adds up scaled sums).
// shape: 0 lets the library choose the tile; 1: 128 x 128; 2: 256 x 256; 5: 128 rows x 256: eight waves in turns where
// turns_takes says so, else eight waves of 32 x 64, sixteen of 64 x 64 and sixteen of 32 x 64 as the two below; 3: 256 x 256,
// eight waves of 128 x 64; 4: 256 rows x 128, eight waves of 64 x 64. -1, -2, -5: such a tile on the kernel without turns, and the
// library's choice where the product runs on the other (a plan for the former, whose slices hold for both).
// w_order, w_pos: how W lies (see below): as stored, or one of its copies in the matrix cores' order alone.
extern "C" int gl3_gemm_mfma(const void* A, const void* W, void* C, int c_dtype, int M, int N, int K, long lda, long ldw,
                             long ldc, int epilogue, int slices, float* P, long p_stride, long ldp, const float* bias,
                             int act, int shape, int w_order, const int* w_pos, float act_limit, float act_shift,
                             const float* col_scale, hipStream_t stream) {
  if (M == 0 || N == 0) return 0;
  GL3_REQUIRE(A && W && C && M > 0 && N > 0 && K > 0, "gl3_gemm_mfma: bad arguments (M=%d N=%d K=%d)", M, N, K);
  GL3_REQUIRE(K % 8 == 0 && lda % 8 == 0 && ldw % 8 == 0, "gl3_gemm_mfma: K=%d, lda=%ld, ldw=%ld must be multiples of 8",
              K, lda, ldw);
  GL3_REQUIRE(lda > 0 && ldw > 0 && lda < (1L << 22) && ldw < (1L << 22),
              "gl3_gemm_mfma: lda=%ld, ldw=%ld: rows of 2^22 elements or more are not built (32-bit offsets in a tile)",
              lda, ldw);
  GL3_REQUIRE(((uintptr_t)A % 16 == 0) && ((uintptr_t)W % 16 == 0), "gl3_gemm_mfma: operands must be 16-byte aligned");
  GL3_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gl3_gemm_mfma: leading dimensions too small");
  GL3_REQUIRE(epilogue >= 0 && epilogue <= 2, "gl3_gemm_mfma: unknown epilogue %d", epilogue);
  GL3_REQUIRE(epilogue != MF_ADD || c_dtype == GL3_F32, "gl3_gemm_mfma: the add epilogue needs a float output");
  GL3_REQUIRE(slices >= 1 && slices <= 64 && slices <= (K + MF_BK - 1) / MF_BK, "gl3_gemm_mfma: %d slices of K=%d",
              slices, K);
  GL3_REQUIRE(slices == 1 || (epilogue != MF_GATED && P && ldp >= N && p_stride >= (long)(M - 1) * ldp + N),
              "gl3_gemm_mfma: slices need a buffer for their sums and another epilogue than the gated one");
  GL3_REQUIRE(!bias || slices == 1, "gl3_gemm_mfma: a bias goes with one slice of K");
  GL3_REQUIRE(GL3_ACT_KNOWN(act), "gl3_gemm_mfma: unknown activation %d", act);
  GL3_REQUIRE(!col_scale || epilogue != MF_GATED, "gl3_gemm_mfma: a factor per column goes with the store and add epilogues");
  const MfExtras ex{col_scale, act_limit, act_shift};
  GL3_REQUIRE((shape >= -5 && shape <= 5 && shape != -3 && shape != -4) || (shape > 8 && (shape % 8 == 1 || shape % 8 == 5) && shape / 8 <= (M - 1) / 256),
              "gl3_gemm_mfma: unknown tile shape %d", shape);
  // w_order: 0: W holds the rows as stored. 1: W is the copy in the matrix operands' order (lib.tile_weight), w_pos (may be
  // null) naming each row's place in it. 2: the copy in packed strips of 8 rows (lib.tile_weight8).
  {
    const long w_rows = epilogue == MF_GATED ? 2L * N : (long)N;
    GL3_REQUIRE(w_order >= 0 && w_order <= 2 && (w_order == 0 || (K % 64 == 0 && (long)w_rows * K < (1L << 32))) &&
                    (w_order != 1 || (w_rows % 16 == 0 && N % 16 == 0)) && (w_order != 2 || w_rows % 8 == 0) && (w_order == 1 || !w_pos),
                "gl3_gemm_mfma: W in order %d with K=%d (a copy's order is read over whole steps of 64), N=%d", w_order, K, N);
  }
#define ARGS A, W, C, M, N, K, lda, ldw, ldc, slices, P, p_stride, ldp, bias, act, shape, w_order, w_pos, ex, stream
  if (c_dtype == GL3_F32) {
    if (epilogue == MF_STORE) return launch_mfma<MF_STORE, float>(ARGS);
    if (epilogue == MF_ADD) return launch_mfma<MF_ADD, float>(ARGS);
    return launch_mfma<MF_GATED, float>(ARGS);
  } else if (c_dtype == GL3_BF16) {
    if (epilogue == MF_STORE) return launch_mfma<MF_STORE, bf16_t>(ARGS);
    if (epilogue == MF_GATED) return launch_mfma<MF_GATED, bf16_t>(ARGS);
  }
#undef ARGS
  GL3_REQUIRE(false, "gl3_gemm_mfma: unsupported output dtype %d for epilogue %d", c_dtype, epilogue);
  return 0;
}

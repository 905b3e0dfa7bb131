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
#include "gemm_mfma_turns.h"

#define MF_LD (MF_BK + 8)   // padded row, in elements

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

// What gemm_mfma_turns_kernel is built for: whole steps of 64 k, and byte offsets of 31 bits inside a tile's rows of A and
// inside W (or, as stored, from the tile's first row of W to its last).
static bool turns_takes(int N, int K, long lda, long ldw, bool gated, int w_order) {
  const long rows = gated ? 2L * N : (long)N;
  return K % 64 == 0 && (255 * lda + K) * 2 < (1L << 31) &&
         (w_order ? rows * K * 2 : ((gated ? (long)N : 0) + 255) * ldw * 2 + 2L * K) < (1L << 31);
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
// products; profiles/two_tiles.txt) they take 0.78 to 1.02 times as long as the single tile taken before, 0.90 on average. Not for up to 1,024 rows over more than
// 40,000 rows of W: the large tiles and the small ones each read them from memory, which one tile's blocks of the same columns share (65,536 rows of W, K = 2,048: 262
// rows 120 us in one tile and 158 in two, 640 182 and 195; 128,256, K = 4,096, 262 387 and 456; 1,030 to 2,221 rows 0.95 to 1.04 in two, 0.99 on average).
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
  const int most = (M - 1) / 256;
  if (!two || (most < 4 && (gated ? 2L : 1L) * N > 40000)) return best;
  least *= 0.96;
  const double large = steps * step_us[2] + round_us[2];
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

// (for tests: the library's choice where gemm_mfma_turns_kernel takes the product)
extern "C" int gl3_turns_shape(int M, int N, int K, int slices, int gated) { return choose_turns_shape(M, N, K, slices, gated, true); }

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
    if constexpr (TWO)
      return mf_launch_two_tiles<EPI, TC>(w_order, shape % 8, A, W, C, M, N, K, lda, ldw, ldc, slices, P, p_stride, ldp, bias, act, w_steps, w_pos, ex,
                                          shape / 8, stream);
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

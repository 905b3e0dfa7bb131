// Products in bfloat16 of two kinds of tiles in one launch (the tile itself: gemm_mfma_turns.h; where they are taken: choose_turns_shape in gemm_mfma.hip).
#include "gemm_mfma_turns.h"

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

template <int EPI, typename TC>
int mf_launch_two_tiles(int w_order, int small, const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc, int slices, float* P,
                        long p_stride, long ldp, const float* bias, int act, int w_steps, const int* w_pos, MfExtras ex, int big_m, hipStream_t stream) {
#define MF_ARGS A, W, C, M, N, K, lda, ldw, ldc, slices, P, p_stride, ldp, bias, act, w_steps, w_pos, ex, big_m, stream
#define MF_TWO(WT) (small == 1 ? launch_two_tiles<EPI, TC, 1, WT>(MF_ARGS) : launch_two_tiles<EPI, TC, 2, WT>(MF_ARGS))
  if (w_order == 0) return MF_TWO(0);
  if (w_order == 1) return MF_TWO(1);
  if constexpr (EPI != MF_GATED) return MF_TWO(2);
#undef MF_TWO
#undef MF_ARGS
  GL3_REQUIRE(false, "gl3_gemm_mfma: two tiles do not read W in order %d", w_order);
  return 0;
}
#define MF_BUILD(EPI, TC)                                                                                                                  \
  template int mf_launch_two_tiles<EPI, TC>(int, int, const void*, const void*, void*, int, int, int, long, long, long, int, float*, long, \
                                            long, const float*, int, int, const int*, MfExtras, int, hipStream_t)
MF_BUILD(MF_STORE, float);
MF_BUILD(MF_STORE, bf16_t);
MF_BUILD(MF_ADD, float);
MF_BUILD(MF_GATED, bf16_t);
#undef MF_BUILD

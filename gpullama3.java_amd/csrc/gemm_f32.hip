// C[M,N] = A[M,K] . W[N,K]^T with all operands, products and sums in true 32-bit on the matrix cores: the products of a
// float32 engine (a wave's v_mfma_f32_16x16x4_f32 multiplies and adds IEEE floats; nothing is rounded to fewer bits on
// the way). gl3_gemm_generic sends products here whose operands and output are float, K and W's rows in whole 16-byte
// pieces; everything else stays with its own kernel.
//
// A token's result does not depend on how many tokens share the step, nor on the kernel below that works it out: both
// add up an output element in the same order. K is cut into chunks of 256; inside a chunk k advances in blocks of 16,
// a block being four instructions of which the j-th takes k = 4q + j, q = 0..3; each chunk's sum starts from zero, and
// the chunks' sums are added in order. (Short chains of sums are also closer to the 64-bit result than one chain of K.)
//
// Three kernels, by the number of rows of A:
// * up to 64 rows (gated 16 or 32): bound by the weights' way from memory. A block takes 16 rows of W (gated: 16 gate rows and
//   their 16 up rows) and its sixteen waves a chunk of K each (16 KB of weights); the chunks' sums meet in shared memory.
//   One row, weights from memory, 1B layers: gate/up 513 -> 29 us (134 MB: 4.6 TB/s), down projection 950 -> 17 us (67 MB:
//   4.0 TB/s), the head 179 us (5.9 TB/s), against the kernel for any sizes, whose 64 x 64 tiles leave a
//   product of 2,048 columns 32 blocks that walk K in steps of 16 behind two barriers each. Eight waves a block were 1.0
//   to 1.3 times as long.
// * more: bound by the matrix cores (256 flops a clock and CU; 157 TFLOP/s at most). K in whole steps of 32, rows of A at and in whole
//   16 bytes, offsets of 31 bits (f32_streams): gemm_f32_stream_kernel, with its figures. Everything else: tiles through registers into shared
//   memory in steps of 32 k, two buffers, one barrier a step; rows in shared memory are 36 floats apart, so that the sixteen lanes that
//   read 16 bytes of sixteen rows meet all 64 banks once. 4,096 x 4,096 x 4,096, rows of A at an odd float: 1.21 ms, 114 TFLOP/s; 513 rows of
//   the 1B layers 57 to 90 TFLOP/s, against about 20 of the kernel for any sizes.
#include "common.h"
#include "lds_loads.h"
#include <algorithm>
#include <type_traits>

typedef float f32x4 __attribute__((ext_vector_type(4)));

enum { F3_STORE = 0, F3_ADD = 1, F3_GATED = 2 };

#define F3_CHUNK 256

struct F3Out {     // what the epilogues need besides the sums
  const float* bias;
  const float* col_scale;
  int act;
  float act_limit, act_shift;
};

template <int EPI>
__device__ __forceinline__ void f3_finish(float* c, float s, float up, int n, int N, const F3Out& o) {
  if (o.bias) s += o.bias[n];
  if (EPI == F3_GATED) {
    if (o.bias) up += o.bias[N + n];
    *c = gl3_gated<false>(s, up, o.act, o.act_limit, o.act_shift);
    return;
  }
  if (o.col_scale) s *= o.col_scale[n];
  if (EPI == F3_ADD) *c += s;
  else *c = s;
}

typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));     // rows of A may begin at any float

// loads of A for few rows go through a descriptor that ends where A ends: a lane without a token row of its own gives an
// offset beyond it, asks memory for nothing and gets zeros, without a branch around the load
#define F3_NOWHERE 0x80000000u
__device__ __forceinline__ f32x4 f3_load_a(__amdgpu_buffer_rsrc_t buf, unsigned row, unsigned byte) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(buf, row == F3_NOWHERE ? F3_NOWHERE : row + byte, 0, 0));
}

// ---- few rows
#define F3_WAVES 16

// PAIRS (at most 8 rows of A, one tile): strips of 8 rows of W. A tile's rows 8..15 are the same rows of W one chunk of K further and
// its token columns 8..15 the same tokens there, so that a product of the two works out two chunks at once, in its two diagonal
// quarters; every element's sum is the same sum.
//
// FRONT (one tile of tokens): eight blocks of 16 k are asked for, weights and rows, before the first product. Left to itself the compiler has four
// to six loads on their way (43 to 58 registers), which suits products of many blocks, whose waves are in different places; where the
// blocks are at most one a CU all waves start together and the trips to memory add up. One row, weights from memory: 2,048 x 2,048 8.9 ->
// 8.2 us, 3,072 x 2,048 10.3 -> 8.9, 2,048 x 8,192 17.9 -> 17.1; 128,256 x 2,048 188 -> 224. From 8 rows on it is ahead with more blocks too
// (the rows' loads are as many as the weights'): gated 14,336 x 4,096, 8 rows 114 -> 105 us, one row 100 -> 103.
template <int EPI, int TM, bool PAIRS = false, bool FRONT = false>
__global__ __launch_bounds__(64 * F3_WAVES) void gemm_f32_rows_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                                      float* __restrict__ C, int M, int N, int K, long lda,
                                                                      long ldw, long ldc, F3Out o) {
  constexpr int NW = F3_WAVES;
  constexpr int G = EPI == F3_GATED ? 2 : 1;
  constexpr int NE = (256 * TM + 64 * NW - 1) / (64 * NW);     // output elements a thread adds up
  constexpr int SLOTS = 32 / (G * TM) > NW ? 32 / (G * TM) : NW;   // chunks whose sums lie in shared memory at a time
  __shared__ __attribute__((aligned(16))) f32x4 sums[SLOTS][G][TM][64];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int r = lane & 15, q = lane >> 4;
  static_assert(!PAIRS || (TM == 1 && EPI != F3_GATED), "strips of 8: one tile of tokens");
  const int n0 = blockIdx.x * (PAIRS ? 8 : 16);
  const int wrow = min(n0 + (PAIRS ? r & 7 : r), N - 1);
  const float* wp[G];
  wp[0] = W + (long)wrow * ldw + q * 4;
  if (G == 2) wp[G - 1] = W + ((long)N + wrow) * ldw + q * 4;
  const __amdgpu_buffer_rsrc_t a_buf = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, (int)(((long)(M - 1) * lda + K) * 4), 0x00020000);
  unsigned ao[TM];
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    const int row = PAIRS ? r & 7 : t * 16 + r;
    ao[t] = row < M ? (unsigned)(((long)row * lda + q * 4) * 4) : F3_NOWHERE;
  }
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  float total[G][NE] = {};
  constexpr int CPS = PAIRS ? 2 : 1;                             // chunks a slot
  const int chunks = (K + F3_CHUNK - 1) / F3_CHUNK;
  for (int first = 0; first < chunks; first += SLOTS * CPS) {
    const int n_here = min(SLOTS * CPS, chunks - first);
    if (first) __syncthreads();
    for (int slot = wave; slot * CPS < n_here; slot += NW) {
      const int k0 = (first + slot * CPS + (PAIRS ? r >> 3 : 0)) * F3_CHUNK;      // (PAIRS: a lane's own chunk)
      const bool whole = (first + (slot + 1) * CPS) * F3_CHUNK <= K;
      f32x4 acc[G][TM];
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int t = 0; t < TM; ++t) acc[g][t] = zero;
      if (whole) {
        // a whole chunk: sixteen loads of each operand, unrolled, for the scheduler to send ahead
        constexpr int PART = FRONT ? 8 : 16 / G;
#pragma unroll
        for (int p = 0; p < 16; p += PART) {
          f32x4 w[G][PART];
#pragma unroll
          for (int b = 0; b < PART; ++b)
#pragma unroll
            for (int g = 0; g < G; ++g) w[g][b] = *(const f32x4*)(wp[g] + k0 + (p + b) * 16);
          if (FRONT) {
            static_assert(!FRONT || TM == 1, "one tile of tokens");
            f32x4 a[PART];
#pragma unroll
            for (int b = 0; b < PART; ++b) a[b] = f3_load_a(a_buf, ao[0], (unsigned)(k0 + (p + b) * 16) * 4);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int b = 0; b < PART; ++b)
#pragma unroll
              for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int g = 0; g < G; ++g) acc[g][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[g][b][j], a[b][j], acc[g][0], 0, 0, 0);
            continue;
          }
#pragma unroll
          for (int b = 0; b < PART; ++b) {
#pragma unroll
            for (int t = 0; t < TM; ++t) {
              const f32x4 a = f3_load_a(a_buf, ao[t], (unsigned)(k0 + (p + b) * 16) * 4);
#pragma unroll
              for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int g = 0; g < G; ++g) acc[g][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[g][b][j], a[j], acc[g][t], 0, 0, 0);
            }
          }
        }
      } else {
        // (K is a multiple of 4: a lane's four k lie inside it or beyond it; blocks of 16 beyond K add nothing)
        for (int k = k0, b = 0; b < F3_CHUNK / 16; k += 16, ++b) {
          const bool in = k + q * 4 < K;
#pragma unroll
          for (int t = 0; t < TM; ++t) {
            const f32x4 a = f3_load_a(a_buf, in ? ao[t] : F3_NOWHERE, (unsigned)k * 4);
#pragma unroll
            for (int g = 0; g < G; ++g) {
              const f32x4 w = in ? *(const f32x4*)(wp[g] + k) : zero;
#pragma unroll
              for (int j = 0; j < 4; ++j) acc[g][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j], a[j], acc[g][t], 0, 0, 0);
            }
          }
        }
      }
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int t = 0; t < TM; ++t) sums[slot][g][t][lane] = acc[g][t];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const int e = tid + 64 * NW * i;
      if (PAIRS) {
        // element e < 64 (a quarter of a tile): token e / 8, column e % 8; in the other quarter 8 rows and 8 columns further
        if (e < 64) {
          const int m = e >> 3, n = e & 7;
          for (int s = 0; s < n_here; ++s) {
            const int row = n + 8 * (s & 1), col = m + 8 * (s & 1);
            total[0][i] += ((const float*)&sums[s >> 1][0][0][(row >> 2) * 16 + col])[row & 3];
          }
        }
      } else if (e < 256 * TM) {
        for (int s = 0; s < n_here; ++s)
#pragma unroll
          for (int g = 0; g < G; ++g) total[g][i] += ((const float*)&sums[s][g][0][0])[e];
      }
    }
  }
  if (PAIRS) {
    const int m = tid >> 3, n = n0 + (tid & 7);
    if (tid < 64 && m < M && n < N) f3_finish<EPI>(C + (long)m * ldc + n, total[0][0], 0.f, n, N, o);
    return;
  }
  // element e: token tile e / 256, lane (e / 4) % 64, v = e % 4: token lane % 16, column 4 * (lane / 16) + v
#pragma unroll
  for (int i = 0; i < NE; ++i) {
    const int e = tid + 64 * NW * i;
    const int l = (e >> 2) & 63, m = (e >> 8) * 16 + (l & 15), n = n0 + 4 * (l >> 4) + (e & 3);
    if (e < 256 * TM && m < M && n < N) f3_finish<EPI>(C + (long)m * ldc + n, total[0][i], total[G - 1][i], n, N, o);
  }
}

// ---- at most four rows: norm, the product with the stacked q, k, v rows, rotation and cache write in one kernel
//
// A decode step of a few sequences is a chain of short kernels: norm, product and rotation took 4.8, 8.4 and 5.4 us of a layer's 89 under the
// profiler (1B layers, two tokens), this one takes 11.9; without it a step of 16 layers 1.60 -> 1.56 ms, for a small kernel of a replayed graph
// costs some 2 us there. Every block works out the norm of the rows itself (8 KB each, in the second-level cache) while its first weights
// are on their way: the sums of squares by as many threads, in the same order, as gl3_rmsnorm's kernels have a row, so the normalised rows
// are the same bits, and so is everything behind them. They lie in shared memory, where all waves read them: from memory, beside the norm's
// weight, they were as many requests as W's rows (15.6 us). A block's sixteen rows of W are eight pairs that the rotation turns (or
// sixteen rows of a value head), and its sums, turned as rope_cache_kernel turns them, go to the query rows and into the pages of the cache.
// The gated product behind its norm the same way was slower (41 us against 29 and 4.8: its 512 blocks, two a CU, have 64
// registers a lane, too few for the norm's operands beside the weights' loads) and keeps its norm in front.
struct F3Norm {
  const float* w;
  float eps;
  int threads;      // that gl3_rmsnorm's kernels give a row
};
struct F3Rope {
  const int *positions, *table_rows, *block_table;
  int table_stride;
  const float *cos_tab, *sin_tab;      // null: no rotation
  float *k_cache, *v_cache;
  int n_heads, n_kv, head_dim, adjacent, page_size;
};
#define F3_NORM_ROWS 4
#define F3_NORM_PAD 16

__global__ __launch_bounds__(64 * F3_WAVES, 4) void qkv_f32_normed_kernel(
    const float* __restrict__ X, F3Norm norm, const float* __restrict__ W, float* __restrict__ Q, int M, int K, long ldx, long ldw, long ldq,
    F3Rope rope) {
  constexpr int PART = 8;      // blocks of 16 k whose weights are on their way at a time
  // the normalised rows, F3_NORM_PAD floats between two (four rows' sixteen bytes of four q meet all banks once), and later the chunks' sums
  extern __shared__ __attribute__((aligned(16))) float shared_rows[];
  f32x4(*const sums)[64] = (f32x4(*)[64])shared_rows;
  __shared__ __attribute__((aligned(16))) float squares[F3_NORM_ROWS][16];
  __shared__ float turned[16][F3_NORM_ROWS + 1];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int r = lane & 15, q = lane >> 4;
  const int chunks = K / F3_CHUNK;                       // (whole ones, at most one a wave)
  const int hs = rope.head_dim, half = hs / 2, per_head = hs / 16;
  const int head = blockIdx.x / per_head, part = blockIdx.x % per_head, n0 = head * hs;
  const bool turns = rope.cos_tab && head < rope.n_heads + rope.n_kv;
  // the element of the head that column n of the block is
  auto place = [&](int n) {
    return turns && !rope.adjacent ? part * 8 + (n & 7) + (n & 8 ? half : 0) : part * 16 + n;
  };
  // element e = tid < 256 of the block's outputs: token lane' % 16, column 4 * (lane' / 16) + e % 4, lane' = e / 4
  const int em = (tid >> 2) & 15, en = 4 * ((tid >> 6) & 3) + (tid & 3);
  const bool ends = tid < 256 && em < M;
  int pos = 0;
  if (ends) pos = rope.positions[em];

  // the rows, then the first weights: loads come back in order, and the sums of squares need not wait for the weights
  // (a thread has one piece of a row, or, of a row of more than 2,048 with 512 threads, two; a wave four at most either way)
  const int waves_a_row = norm.threads / 64, rows_at_once = F3_WAVES / waves_a_row, two = K > 4 * norm.threads;
  const int group = wave / waves_a_row, piece = (tid & (norm.threads - 1)) * 4;
  f32x4 xv[F3_NORM_ROWS];
#pragma unroll
  for (int i = 0; i < F3_NORM_ROWS; ++i) {
    const int row = min((i >> two) * rows_at_once + group, M - 1), at = piece + (i & two) * 4 * norm.threads;
    xv[i] = *(const f32x4*)(X + (long)row * ldx + min(at, K - 4));
  }
  f32x4 nw[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) nw[i] = *(const f32x4*)(norm.w + min(piece + (i & two) * 4 * norm.threads, K - 4));
  __builtin_amdgcn_sched_barrier(0);
  const int chunk = min(wave, chunks - 1), k0 = chunk * F3_CHUNK;      // (a wave without a chunk reads the last one and drops it)
  const float* const wp = W + (long)(n0 + place(r)) * ldw + k0 + q * 4;
  f32x4 w[PART];
#pragma unroll
  for (int b = 0; b < PART; ++b) w[b] = *(const f32x4*)(wp + b * 16);
  __builtin_amdgcn_sched_barrier(0);
  // what the end needs of the token: its page, its angle
  int page = 0;
  float cosine = 1.f, sine = 0.f;
  const int angle = rope.adjacent ? (part * 16 + en) >> 1 : part * 8 + (en & 7);
  if (ends) {
    if (head >= rope.n_heads) page = rope.block_table[(long)rope.table_rows[em] * rope.table_stride + pos / rope.page_size];
    if (turns) {
      cosine = rope.cos_tab[(long)pos * half + angle];
      sine = rope.sin_tab[(long)pos * half + angle];
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < F3_NORM_ROWS; ++i) {
    const int row = (i >> two) * rows_at_once + group, at = piece + (i & two) * 4 * norm.threads;
    if (row >= M) continue;
    if (!(i & two)) ss = 0.f;
    float more = ss;
#pragma unroll
    for (int e = 0; e < 4; ++e) more = fmaf(xv[i][e], xv[i][e], more);
    if (at < K) ss = more;
    if (two && !(i & 1)) continue;
    const float sum = wave_sum(ss);
    if (lane == 0) squares[row][wave % waves_a_row] = sum;
  }
  __syncthreads();
  const int pitch = K + F3_NORM_PAD;
#pragma unroll
  for (int i = 0; i < F3_NORM_ROWS; ++i) {
    const int row = (i >> two) * rows_at_once + group, at = piece + (i & two) * 4 * norm.threads;
    if (row >= M) continue;
    float scale = 0.f;
    for (int k = 0; k < waves_a_row; k += 4) {
      const f32x4 four = *(const f32x4*)&squares[row][k];
#pragma unroll
      for (int e = 0; e < 4; ++e) scale += four[e];
    }
    scale = scale / (float)K;
    scale = scale + norm.eps;
    scale = 1.0f / sqrtf(scale);
    if (at < K) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (i & two ? nw[1] : nw[0])[e] * (scale * xv[i][e]);
      *(f32x4*)(shared_rows + row * pitch + at) = v;
    }
  }
  __syncthreads();
  // (lanes without a row of their own work on the last one; their sums are dropped)
  const float* const rows = shared_rows + min(r, M - 1) * pitch + k0 + q * 4;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  if (wave < chunks) {
#pragma unroll
    for (int p = 0; p < 16; p += PART) {
#pragma unroll
      for (int b = 0; b < PART; ++b) {
        const f32x4 a = *(const f32x4*)(rows + (p + b) * 16);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[b][j], a[j], acc, 0, 0, 0);
        if (p + PART + b < 16) w[b] = *(const f32x4*)(wp + (p + PART + b) * 16);
      }
    }
  }
  __syncthreads();                     // (everybody has read the rows: the sums lie there now)
  if (wave < chunks) sums[wave][lane] = acc;
  __syncthreads();
  float v = 0.f;
  if (tid < 256)
    for (int s = 0; s < chunks; ++s) v += ((const float*)&sums[s][0])[tid];
  if (ends) turned[en][em] = v;
  __syncthreads();
  if (!ends) return;
  if (turns) {
    const int across = rope.adjacent ? 1 : 8;
    const float other = turned[en ^ across][em];
    v = en & across ? fmaf(other, sine, v * cosine) : fmaf(v, cosine, -(other * sine));      // (rounded as rope_cache_kernel's)
  }
  const int dim = place(en);
  if (head < rope.n_heads) {
    Q[(long)em * ldq + n0 + dim] = v;
    return;
  }
  const int in_page = pos % rope.page_size, c = (head - rope.n_heads) % rope.n_kv;
  const long at = ((long)page * rope.n_kv + c) * rope.page_size * hs;
  if (head < rope.n_heads + rope.n_kv) rope.k_cache[at + gl3_k_offset(in_page, dim, hs)] = v;
  else rope.v_cache[at + gl3_v_offset(dim, in_page, rope.page_size)] = v;
}

// A lane holds four consecutive columns (from n0) of one token (m0) per tile.
template <int EPI, int TW, int TT>
__device__ __forceinline__ void f3_finish_tile(float* __restrict__ C, const f32x4 (&total)[TW][TT], int m0, int n0, int M, int N, long ldc, const F3Out& o) {
#pragma unroll
  for (int y = 0; y < TT; ++y) {
    const int m = m0 + y * 16;
    if (m >= M) continue;
    float* c = C + (long)m * ldc;
#pragma unroll
    for (int x = 0; x < (EPI == F3_GATED ? TW / 2 : TW); ++x) {
      const int n = n0 + x * 16;
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (n + v < N)
          f3_finish<EPI>(c + n + v, total[x][y][v], total[EPI == F3_GATED ? TW / 2 + x : x][y][v], n + v, N, o);
    }
  }
}

// ---- many rows: four waves, 2 x 2, a wave owns 16 * TW rows of W by 16 * TT tokens
#define F3_BK 32
#define F3_LD (F3_BK + 4)

template <int EPI, int TW, int TT>
__global__ __launch_bounds__(256, 2) void gemm_f32_tile_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                               float* __restrict__ C, int M, int N, int K, long lda,
                                                               long ldw, long ldc, int tiles_m, int tiles_n, F3Out o) {
  constexpr int BN = 32 * TW, BM = 32 * TT;
  constexpr int NCOLS = EPI == F3_GATED ? BN / 2 : BN;
  static_assert(EPI != F3_GATED || TW % 2 == 0, "a wave's tiles are gate rows and their up rows");
  __shared__ __attribute__((aligned(16))) float Ws[2][BN][F3_LD];
  __shared__ __attribute__((aligned(16))) float As[2][BM][F3_LD];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int r = lane & 15, q = lane >> 4;
  const int ww = wave & 1, wt = wave >> 1;
  // an XCD (consecutive block ids take turns) works on neighbouring tiles: all token tiles of a column, then the next
  const int n_tiles = tiles_m * tiles_n, per_xcd = (n_tiles + 7) / 8;
  const int tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (tile >= n_tiles) return;
  const int m0 = (tile % tiles_m) * BM, n0 = (tile / tiles_m) * NCOLS;

  // memory -> registers -> shared memory in pieces of 16 bytes, eight a row and step; rows beyond the matrix repeat its
  // last one (their sums are dropped), k beyond K is zero
  constexpr int NW = BN * 8 / 256, NA = BM * 8 / 256;
  const float *wp[NW], *ap[NA];
  const int kc = (tid & 7) * 4;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int row = (tid >> 3) + 32 * i;
    int n = n0 + row;
    if (EPI == F3_GATED) {       // (a wave's rows: TW / 2 tiles of gate rows, then the up rows of the same columns)
      const int sec = row / (16 * TW), in = row % (16 * TW);
      n = min(n0 + sec * 8 * TW + in % (8 * TW), N - 1) + (in >= 8 * TW ? N : 0);
    } else {
      n = min(n, N - 1);
    }
    wp[i] = W + (long)n * ldw;
  }
#pragma unroll
  for (int i = 0; i < NA; ++i) ap[i] = A + (long)min(m0 + (tid >> 3) + 32 * i, M - 1) * lda;
  f32x4 rw[NW], ra[NA];
  bool r_ok = false;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  auto fetch = [&](int k0) {      // (loads without a branch: a piece beyond K reads the row's last one and is not kept)
    r_ok = k0 + kc < K;
    const int k = min(k0 + kc, K - 4);
#pragma unroll
    for (int i = 0; i < NA; ++i) ra[i] = *(const f32x4_any*)(ap[i] + k);
#pragma unroll
    for (int i = 0; i < NW; ++i) rw[i] = *(const f32x4*)(wp[i] + k);
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NA; ++i) *(f32x4*)&As[buf][(tid >> 3) + 32 * i][kc] = r_ok ? ra[i] : zero;
#pragma unroll
    for (int i = 0; i < NW; ++i) *(f32x4*)&Ws[buf][(tid >> 3) + 32 * i][kc] = r_ok ? rw[i] : zero;
  };

  f32x4 acc[TW][TT], total[TW][TT];
#pragma unroll
  for (int a = 0; a < TW; ++a)
#pragma unroll
    for (int b = 0; b < TT; ++b) acc[a][b] = total[a][b] = zero;
  fetch(0);
  store(0);
  fetch(F3_BK);
  __syncthreads();
  for (int k0 = 0, buf = 0; k0 < K; k0 += F3_BK, buf ^= 1) {
    if (k0 + F3_BK < K) {
      store(buf ^ 1);
      fetch(k0 + 2 * F3_BK);
    }
#pragma unroll
    for (int kb = 0; kb < F3_BK; kb += 16) {
      f32x4 w[TW], a[TT];
#pragma unroll
      for (int i = 0; i < TW; ++i) w[i] = *(const f32x4*)&Ws[buf][ww * 16 * TW + i * 16 + r][kb + q * 4];
#pragma unroll
      for (int i = 0; i < TT; ++i) a[i] = *(const f32x4*)&As[buf][wt * 16 * TT + i * 16 + r][kb + q * 4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int x = 0; x < TW; ++x)
#pragma unroll
          for (int y = 0; y < TT; ++y)
            acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[x][j], a[y][j], acc[x][y], 0, 0, 0);
    }
    if ((k0 + F3_BK) % F3_CHUNK == 0 || k0 + F3_BK >= K) {
#pragma unroll
      for (int x = 0; x < TW; ++x)
#pragma unroll
        for (int y = 0; y < TT; ++y) {
          total[x][y] += acc[x][y];
          acc[x][y] = zero;
        }
    }
    __syncthreads();
  }
  f3_finish_tile<EPI, TW, TT>(C, total, m0 + wt * 16 * TT + r, n0 + ww * (EPI == F3_GATED ? 8 : 16) * TW + q * 4, M, N, ldc, o);
}

// ---- many rows, K in whole steps of 32: the same products, operands straight from memory into shared memory
//
// The kernel above keeps one step of operands in registers on the way to shared memory; behind its barrier every wave then waits for
// its reads with little else in flight. Here a block asks for steps ahead (STAGES - 1 of them), no wave writes shared memory, and what a
// tile needs of it is small enough for several blocks a CU, of which one multiplies while another waits. The kernel above and this one at
// 513 rows of the 1B layers: gate/up 381 -> 293 us (118 TFLOP/s), down 276 -> 210, output 75 -> 60, QKV 89 -> 72; at 4,096 rows gate/up
// 2,462 -> 1,974 (139 TFLOP/s; the library's own product of 8,192 cubed reaches 153; profiles/float32_tiles.txt). What bounds the small ones: whole tiles of 32 rows
// and whole rounds of the chip's 256 CUs. Rows in shared memory are 128
// bytes in eight pieces of 16, piece c of row r at place c ^ (r / 2 % 8): the sixteen rows that sixteen lanes read at one piece meet all
// banks once. A step is asked for into the place of the step before, behind the barrier that every wave reaches with that step's
// products issued (its reads have returned); the wait in front of the barrier leaves out the later steps. Steps beyond the last repeat it,
// so that the counts hold; nothing is in flight when a block ends. Sums as above: the same bits.
constexpr int f3_stage(int TW, int TT) { return 32 * (TW + TT) * 128; }      // bytes of a step: rows of W, then rows of A
template <int EPI, int TW, int TT, int STAGES>
__device__ __forceinline__ void f3_stream_tile(char* lds, const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int M, int N,
                                               int K, long lda, long ldw, long ldc, int m0, int n0, const F3Out& o) {
  constexpr int BN = 32 * TW, BM = 32 * TT, PW = (BN + BM) / 32;       // PW: pieces of 1 KB (8 rows) of a step that a wave brings
  constexpr int STAGE = f3_stage(TW, TT);
  static_assert(EPI != F3_GATED || TW % 2 == 0, "a wave's tiles are gate rows and their up rows");
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int r = lane & 15, q = lane >> 4;
  const int ww = wave & 1, wt = wave >> 1;
  const int steps = K / F3_BK;

  const i32x4 a_buf = mf_rsrc(A + (long)m0 * lda), w_buf = mf_rsrc(W + (long)n0 * ldw);
  unsigned from[PW];
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    const int piece = i * 4 + wave, row = piece * 8 + (lane >> 3);             // (rows of W, then rows of A)
    const int at = ((lane & 7) ^ ((row >> 1) & 7)) * 4;
    if (i * 4 * 8 < BN) {
      int n = n0 + row;
      if (EPI == F3_GATED) {       // (a wave's rows: TW / 2 tiles of gate rows, then the up rows of the same columns)
        const int sec = row / (16 * TW), in = row % (16 * TW);
        n = min(n0 + sec * 8 * TW + in % (8 * TW), N - 1) + (in >= 8 * TW ? N : 0);
      } else {
        n = min(n, N - 1);
      }
      from[i] = (unsigned)((long)(n - n0) * ldw + at) * 4;
    } else {
      from[i] = (unsigned)((long)(min(m0 + row - BN, M - 1) - m0) * lda + at) * 4;
    }
  }
  const unsigned lds0 = (unsigned)(unsigned long)(__attribute__((address_space(3))) char*)lds + wave * 1024;
  auto load = [&](int t, int place) {
    const unsigned step = (unsigned)min(t, steps - 1) * (F3_BK * 4);
#pragma unroll
    for (int i = 0; i < PW; ++i) mf_dma16(lds0 + place * STAGE + i * 4096, from[i], i * 4 * 8 < BN ? w_buf : a_buf, step);
  };

  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[TW][TT], total[TW][TT];
#pragma unroll
  for (int a = 0; a < TW; ++a)
#pragma unroll
    for (int b = 0; b < TT; ++b) acc[a][b] = total[a][b] = zero;
  const int twist = (r >> 1) & 7;
  const char* w_at = lds + (ww * 16 * TW + r) * 128;
  const char* a_at = lds + (BN + wt * 16 * TT + r) * 128;
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t) load(t, t);
  for (int t = 0, here = 0, there = STAGES - 1; t < steps; ++t) {
    mf_wait_loads<(STAGES - 2) * PW>();
    mf_barrier();
    load(t + STAGES - 1, there);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      f32x4 w[TW], a[TT];
      const int c = ((kb * 4 + q) ^ twist) << 4;
#pragma unroll
      for (int i = 0; i < TW; ++i) w[i] = *(const f32x4*)(w_at + here * STAGE + i * 2048 + c);
#pragma unroll
      for (int i = 0; i < TT; ++i) a[i] = *(const f32x4*)(a_at + here * STAGE + i * 2048 + c);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int x = 0; x < TW; ++x)
#pragma unroll
          for (int y = 0; y < TT; ++y)
            acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[x][j], a[y][j], acc[x][y], 0, 0, 0);
    }
    if ((t + 1) % (F3_CHUNK / F3_BK) == 0 || t + 1 == steps) {
#pragma unroll
      for (int x = 0; x < TW; ++x)
#pragma unroll
        for (int y = 0; y < TT; ++y) {
          total[x][y] += acc[x][y];
          acc[x][y] = zero;
        }
    }
    there = here;
    here = here + 1 == STAGES ? 0 : here + 1;
  }
  mf_wait_loads<0>();
  f3_finish_tile<EPI, TW, TT>(C, total, m0 + wt * 16 * TT + r, n0 + ww * (EPI == F3_GATED ? 8 : 16) * TW + q * 4, M, N, ldc, o);
}
template <int EPI, int TW, int TT, int STAGES>
__global__ __launch_bounds__(256, 2) void gemm_f32_stream_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                                 float* __restrict__ C, int M, int N, int K, long lda,
                                                                 long ldw, long ldc, int tiles_m, int tiles_n, F3Out o) {
  __shared__ __attribute__((aligned(1024))) char lds[STAGES * f3_stage(TW, TT)];
  const int n_tiles = tiles_m * tiles_n, per_xcd = (n_tiles + 7) / 8;          // (block -> tile as above)
  const int tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (tile >= n_tiles) return;
  f3_stream_tile<EPI, TW, TT, STAGES>(lds, A, W, C, M, N, K, lda, ldw, ldc, tile % tiles_m * (32 * TT), tile / tiles_m * ((EPI == F3_GATED ? 16 : 32) * TW), o);
}

// Two tiles: the first `big_m` rows of tiles are TW x TT, those behind them SW x ST, smaller ones, which the CUs take that are done with the
// large ones, one launch. Whole rounds of the chip are what bounds a product of few tiles: 513 rows of the 1B layers' down projection are 544 tiles of
// 64 x 32, three rounds for the work of 2.1, or one round of 64 x 64 and a row: 223 -> 189 us; their output projection 62 -> 53, gate/up 336 -> 302.
// The same bits: a sum does not know its tile.
template <int EPI, int TW, int TT, int STAGES, int SW, int ST, int SSTAGES>
__global__ __launch_bounds__(256, 2) void gemm_f32_two_tiles_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                                    float* __restrict__ C, int M, int N, int K, long lda, long ldw,
                                                                    long ldc, int big_m, int big_n, int small_m, int small_n, F3Out o) {
  constexpr int BIG = STAGES * f3_stage(TW, TT), SMALL = SSTAGES * f3_stage(SW, ST), COLS = EPI == F3_GATED ? 16 : 32;
  __shared__ __attribute__((aligned(1024))) char lds[BIG > SMALL ? BIG : SMALL];
  const int big = big_m * big_n, small = small_m * small_n, big_xcd = (big + 7) / 8, small_xcd = (small + 7) / 8;
  const int xcd = blockIdx.x & 7, at = blockIdx.x >> 3;
  if (at < big_xcd) {
    const int tile = xcd * big_xcd + at;
    if (tile < big) f3_stream_tile<EPI, TW, TT, STAGES>(lds, A, W, C, M, N, K, lda, ldw, ldc, tile % big_m * (32 * TT), tile / big_m * (COLS * TW), o);
  } else {
    const int tile = xcd * small_xcd + at - big_xcd;
    if (tile < small)
      f3_stream_tile<EPI, SW, ST, SSTAGES>(lds, A, W, C, M, N, K, lda, ldw, ldc, big_m * (32 * TT) + tile % small_m * (32 * ST), tile / small_m * (COLS * SW), o);
  }
}

template <int EPI, int TM, bool PAIRS = false>
static int launch_rows(const float* A, const float* W, float* C, int M, int N, int K, long lda, long ldw, long ldc,
                       const F3Out& o, hipStream_t stream) {
  const dim3 grid(PAIRS ? (N + 7) / 8 : (N + 15) / 16), block(64 * F3_WAVES);
  const bool front = TM == 1 && (grid.x <= 256 || (grid.x <= 1024 && M >= 8));
  if (front) gemm_f32_rows_kernel<EPI, TM, PAIRS, TM == 1><<<grid, block, 0, stream>>>(A, W, C, M, N, K, lda, ldw, ldc, o);
  else gemm_f32_rows_kernel<EPI, TM, PAIRS><<<grid, block, 0, stream>>>(A, W, C, M, N, K, lda, ldw, ldc, o);
  GL3_LAUNCH_CHECK();
  return 0;
}

template <int EPI, int TW, int TT, int STAGES>
static int launch_stream(const float* A, const float* W, float* C, int M, int N, int K, long lda, long ldw, long ldc,
                         const F3Out& o, hipStream_t stream) {
  const int ncols = EPI == F3_GATED ? 16 * TW : 32 * TW;
  const int tiles_m = (M + 32 * TT - 1) / (32 * TT), tiles_n = (N + ncols - 1) / ncols;
  const long blocks = ((long)tiles_m * tiles_n + 7) / 8 * 8;
  GL3_REQUIRE(blocks < (1L << 31), "gl3_gemm_generic: too many tiles");
  gemm_f32_stream_kernel<EPI, TW, TT, STAGES><<<dim3((unsigned)blocks), dim3(256), 0, stream>>>(A, W, C, M, N, K, lda, ldw, ldc, tiles_m,
                                                                                               tiles_n, o);
  GL3_LAUNCH_CHECK();
  return 0;
}

template <int EPI, int TW, int TT, int STAGES, int SW, int ST, int SSTAGES>
static int launch_two_tiles(const float* A, const float* W, float* C, int M, int N, int K, long lda, long ldw, long ldc,
                            const F3Out& o, int big_m, hipStream_t stream) {
  constexpr int COLS = EPI == F3_GATED ? 16 : 32;
  const int big_n = (N + COLS * TW - 1) / (COLS * TW), small_n = (N + COLS * SW - 1) / (COLS * SW);
  const int small_m = (M - big_m * 32 * TT + 32 * ST - 1) / (32 * ST);
  const long blocks = (((long)big_m * big_n + 7) / 8 + ((long)small_m * small_n + 7) / 8) * 8;
  GL3_REQUIRE(big_m > 0 && small_m > 0 && blocks < (1L << 31), "gl3_gemm_generic: too many tiles");
  gemm_f32_two_tiles_kernel<EPI, TW, TT, STAGES, SW, ST, SSTAGES><<<dim3((unsigned)blocks), dim3(256), 0, stream>>>(
      A, W, C, M, N, K, lda, ldw, ldc, big_m, big_n, small_m, small_n, o);
  GL3_LAUNCH_CHECK();
  return 0;
}

template <int EPI, int TW, int TT>
static int launch_tile(const float* A, const float* W, float* C, int M, int N, int K, long lda, long ldw, long ldc,
                       const F3Out& o, hipStream_t stream) {
  const int ncols = EPI == F3_GATED ? 16 * TW : 32 * TW;
  const int tiles_m = (M + 32 * TT - 1) / (32 * TT), tiles_n = (N + ncols - 1) / ncols;
  const long blocks = ((long)tiles_m * tiles_n + 7) / 8 * 8;
  GL3_REQUIRE(blocks < (1L << 31), "gl3_gemm_generic: too many tiles");
  gemm_f32_tile_kernel<EPI, TW, TT><<<dim3((unsigned)blocks), dim3(256), 0, stream>>>(A, W, C, M, N, K, lda, ldw, ldc, tiles_m,
                                                                                    tiles_n, o);
  GL3_LAUNCH_CHECK();
  return 0;
}

// Strips of 8 rows of W for at most 8 rows of A: where strips of 16 leave half of the CUs without a block (a block's loads, 16 rows
// of 64 bytes an instruction, come at 16 bytes a clock and CU) and K has more chunks than a block has waves. 2,048 columns, K =
// 8,192: 25.7 -> 16.7 us; K = 2,048: 8.1 -> 9.3 us (half of the waves find no pair of chunks); 3,072 columns, K = 8,192: 28.6 and 29.1.
static bool f32_pairs(int M, int N, int K) { return M <= 8 && N <= 2048 && K > F3_CHUNK * F3_WAVES; }

// What gemm_f32_stream_kernel is built for: whole steps of 32 k, rows of A in whole 16-byte pieces, and byte offsets of 31 bits inside a
// tile's rows of A (128 at most) and of W (gated: the up rows lie N behind the gate rows).
static bool f32_streams(const void* A, int N, int K, long lda, long ldw, bool gated) {
  return K % F3_BK == 0 && lda % 4 == 0 && (uintptr_t)A % 16 == 0 && 128 * lda * 4 < (1L << 31) && ((gated ? (long)N : 0) + 128) * ldw * 4 < (1L << 31);
}
// Its tile: 1 to 4: 128 rows of W x 128 tokens, 128 x 64, 64 x 64, 64 x 32; 5: 32 x 32 (not gated). As in gl3_f32_shape: one tile alone
// on a CU takes `alone`, a CU with several `each` a tile (us for K = 2,048, both measured; of 85 products of 17 to 4,096 rows
// one is more than 2% from the best of the tiles, 6%: profiles/float32_tiles.txt).
struct F3Cost { int bn, bm; float alone, each; };
static const F3Cost f3_cost[5] = {{128, 128, 144, 124.4f}, {128, 64, 80, 62.5f}, {64, 64, 45.5f, 33.4f}, {64, 32, 28.6f, 17.7f}, {32, 32, 20.5f, 11.f}};
static int f3_best_tile(int M, int N, int gated, float& least) {
  int best = 4;
  least = 0.f;
  for (int i = 0; i < (gated ? 4 : 5); ++i) {
    const F3Cost& t = f3_cost[i];
    const long tiles = (long)((M + t.bm - 1) / t.bm) * (((gated ? 2L : 1L) * N + t.bn - 1) / t.bn);
    const float cu = (float)((tiles + 255) / 256) * t.each, cost = cu < t.alone ? t.alone : cu;
    if (i == 0 || cost < least) {
      least = cost;
      best = i + 1;
    }
  }
  return best;
}
extern "C" int gl3_f32_stream_shape(int M, int N, int gated) {
  float least;
  return f3_best_tile(M, N, gated, least);
}
// Whether two tiles (gemm_f32_two_tiles_kernel) are expected to take less than 0.95 of the best single tile's time, and which: 64 * rows of large
// tiles + 8 * the large tile + the small one; 0: one tile. The blocks are all handed out at once, about as many of either kind to every CU, so a CU's
// time is taken as that of its large tiles and then its small ones. (As if the small ones went to the CUs that have no large tile: of 42 sizes
// seven took 1.03 to 1.08 times as long as one tile, those this rule leaves out.) A small tile beside others takes 1.05 of its time. A single row of large tiles of 64
// rows of A over more than 40,000 rows of W is left out: one tile reads each of them once, for all rows of A, two kinds twice (128,256 rows of W,
// K = 2,048, 96 rows: 1.84 times the bytes from memory, 446 -> 490 us; 70 rows 423 and 461; 210 in three rows of large tiles 931 and 928). Measured at 179 sizes (66
// to 4,096 rows, K of 768 to 14,336, 1,024 to 128,256 rows of W) 0.83 to 1.04 times as long as one tile, 0.920 on average; at 9 with that row 1.04 to 1.10
// (profiles/float32_two_tiles.txt).
extern "C" int gl3_f32_stream_two(int M, int N, int gated) {
  float least;
  f3_best_tile(M, N, gated, least);
  least *= 0.95f;
  const long rows = (gated ? 2L : 1L) * N;
  int best = 0;
  for (int i = 0; i < 3; ++i) {
    const F3Cost& t = f3_cost[i];
    for (int r = (M - 1) / t.bm, first = r - 3; r > (i > 0 && rows > 40000 ? 1 : 0) && r >= first; --r) {
      const float big = (float)((r * ((rows + t.bn - 1) / t.bn) + 255) / 256) * t.each;
      for (int j = i < 2 ? 3 : 4; j < (gated ? 4 : 5); ++j) {      // (64 x 32 behind 64 x 64 never is the best)
        const F3Cost& u = f3_cost[j];
        const long small = (long)((M - r * t.bm + u.bm - 1) / u.bm) * ((rows + u.bn - 1) / u.bn);
        const float cu = big + (float)((small + 255) / 256) * 1.05f * u.each, cost = cu < t.alone ? t.alone : cu;
        if (cost < least) {
          best = r * 64 + (i + 1) * 8 + j + 1;
          least = cost;
        }
      }
    }
  }
  return best;
}

template <int EPI>
static int launch_f32(const float* A, const float* W, float* C, int M, int N, int K, long lda, long ldw, long ldc,
                      const F3Out& o, hipStream_t stream) {
#define F3_ARGS A, W, C, M, N, K, lda, ldw, ldc, o, stream
  int shape = gl3_f32_shape(M, N, EPI == F3_GATED);
  // (gated products of 17 to 32 rows too: 1B layers' gate/up 35 us with the kernel for few rows, 29 in tiles of 64 x 32)
  if ((shape != 1 || (EPI == F3_GATED && M > 16)) && f32_streams(A, N, K, lda, ldw, EPI == F3_GATED)) {
    const int two = gl3_f32_stream_two(M, N, EPI == F3_GATED);
#define F3_TWO_ARGS A, W, C, M, N, K, lda, ldw, ldc, o, two / 64, stream
    switch (two % 64) {
      case 014: return launch_two_tiles<EPI, 4, 4, 2, 2, 1, 3>(F3_TWO_ARGS);
      case 024: return launch_two_tiles<EPI, 4, 2, 2, 2, 1, 3>(F3_TWO_ARGS);
      case 015: if constexpr (EPI != F3_GATED) return launch_two_tiles<EPI, 4, 4, 2, 1, 1, 4>(F3_TWO_ARGS); break;
      case 025: if constexpr (EPI != F3_GATED) return launch_two_tiles<EPI, 4, 2, 2, 1, 1, 4>(F3_TWO_ARGS); break;
      case 035: if constexpr (EPI != F3_GATED) return launch_two_tiles<EPI, 2, 2, 3, 1, 1, 4>(F3_TWO_ARGS); break;
      default: break;
    }
#undef F3_TWO_ARGS
    switch (gl3_f32_stream_shape(M, N, EPI == F3_GATED)) {
      case 1: return launch_stream<EPI, 4, 4, 2>(F3_ARGS);
      case 2: return launch_stream<EPI, 4, 2, 2>(F3_ARGS);
      case 3: return launch_stream<EPI, 2, 2, 3>(F3_ARGS);
      case 5:
        if constexpr (EPI != F3_GATED) return launch_stream<EPI, 1, 1, 4>(F3_ARGS);
      default: return launch_stream<EPI, 2, 1, 3>(F3_ARGS);
    }
  }
  if (shape == 1 && ((long)(M - 1) * lda + K) * 4 >= (1L << 31)) shape = 5;      // (a descriptor's 31 bits)
  switch (shape) {
    case 1:
      if constexpr (EPI != F3_GATED)
        if (f32_pairs(M, N, K)) return launch_rows<EPI, 1, true>(F3_ARGS);
      if (M <= 16) return launch_rows<EPI, 1>(F3_ARGS);
      if (M <= 32) return launch_rows<EPI, 2>(F3_ARGS);
      if constexpr (EPI != F3_GATED) return launch_rows<EPI, 4>(F3_ARGS);
    case 2: return launch_tile<EPI, 4, 4>(F3_ARGS);
    case 3: return launch_tile<EPI, 4, 2>(F3_ARGS);
    case 4: return launch_tile<EPI, 2, 2>(F3_ARGS);
    default: return launch_tile<EPI, 2, 1>(F3_ARGS);
  }
#undef F3_ARGS
}

// 1: the kernel for few rows; 2 to 5: tiles of 128 x 128, 128 x 64, 64 x 64 and 64 rows of W x 32 tokens. Of the tiles the
// one that takes the least time: one tile alone on a CU takes `alone`, a CU with several of them `each` a tile (us for
// K = 2,048, both measured; the sum of a CU's tiles was within 4% of the measured time at 513 to 4,096 rows). Few rows: 48
// rows of the down projection of the 1B layers 136 us in the smallest tile; gated products of more than 32 rows (of more than 16 where
// gemm_f32_stream_kernel takes them) fill the chip with those (48 rows: 55 us, 43 there) where the other kernel would hold 128 KB of sums a block.
extern "C" int gl3_f32_shape(int M, int N, int gated) {
  if (M <= (gated ? 32 : 64)) return 1;
  static const int bn[4] = {128, 128, 64, 64}, bm[4] = {128, 64, 64, 32}, alone[4] = {154, 89, 53, 34}, each[4] = {144, 76, 41, 23};
  int best = 5;
  long least = -1;
  for (int i = 0; i < 4; ++i) {
    const long tiles = (long)((M + bm[i] - 1) / bm[i]) * (((gated ? 2L : 1L) * N + bn[i] - 1) / bn[i]);
    const long cu = (tiles + 255) / 256 * each[i], cost = cu < alone[i] ? alone[i] : cu;
    if (least < 0 || cost < least) {
      least = cost;
      best = i + 2;
    }
  }
  return best;
}

bool gl3_f32_takes(const void* W, int K, long ldw) { return K % 4 == 0 && ldw % 4 == 0 && (uintptr_t)W % 16 == 0; }

int gl3_gemm_f32(const void* A, const void* W, void* C, int M, int N, int K, long lda, long ldw, long ldc, int epi,
                 const float* bias, int act, float act_limit, float act_shift, const float* col_scale, hipStream_t stream) {
  const F3Out o{bias, col_scale, act, act_limit, act_shift};
#define F3_ARGS (const float*)A, (const float*)W, (float*)C, M, N, K, lda, ldw, ldc, o, stream
  if (epi == F3_STORE) return launch_f32<F3_STORE>(F3_ARGS);
  if (epi == F3_ADD) return launch_f32<F3_ADD>(F3_ARGS);
  return launch_f32<F3_GATED>(F3_ARGS);
#undef F3_ARGS
}

// gl3_rmsnorm (weight norm_w, K floats), gl3_gemm_generic with the stacked q, k, v rows W and gl3_rope_cache_write (whole heads rotated; cos_tab null: not)
// of at most four rows, bit for bit: queries to q, keys and values into the cache. K in whole chunks of 256, at most 4,096 and 64 KB of rows; rows of x,
// of W and norm_w at 16 bytes.
extern "C" int gl3_qkv_f32_normed(const float* x, const float* norm_w, float eps, const float* W, float* q, int M, int K, long ldx, long ldw, long ldq,
                                  const int* positions, const int* table_rows, const int* block_table, int table_stride, const float* cos_tab,
                                  const float* sin_tab, float* k_cache, float* v_cache, int n_heads, int n_kv, int head_dim, int adjacent, int page_size,
                                  hipStream_t stream) {
  if (M == 0) return 0;
  GL3_REQUIRE(n_heads > 0 && n_kv > 0 && head_dim > 0 && head_dim % 16 == 0 && page_size > 0 && page_size % 32 == 0 && table_stride > 0,
              "gl3_qkv_f32_normed: %d and %d heads of %d, pages of %d", n_heads, n_kv, head_dim, page_size);
  const int rows = M * (K + F3_NORM_PAD) * 4;      // (bytes of the rows that a block keeps)
  GL3_REQUIRE(x && norm_w && W && M > 0 && M <= F3_NORM_ROWS && K > 0 && K % F3_CHUNK == 0 && K <= F3_CHUNK * F3_WAVES && rows <= 65536,
              "gl3_qkv_f32_normed: %d rows of %d: up to four of whole 256, 4,096 at most, 64 KB together", M, K);
  GL3_REQUIRE(ldx >= K && ldw >= K && ldx % 4 == 0 && ldw % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)norm_w % 16 == 0 && (uintptr_t)W % 16 == 0,
              "gl3_qkv_f32_normed: rows at whole 16 bytes (ldx=%ld ldw=%ld)", ldx, ldw);
  GL3_REQUIRE(q && ldq >= (long)n_heads * head_dim && positions && table_rows && block_table && k_cache && v_cache && (cos_tab == nullptr) == (sin_tab == nullptr),
              "gl3_qkv_f32_normed: outputs, cache or tables missing (ldq=%ld)", ldq);
  const F3Rope rope{positions, table_rows, block_table, table_stride, cos_tab, sin_tab, k_cache, v_cache, n_heads, n_kv, head_dim, adjacent, page_size};
  const F3Norm norm{norm_w, eps, K / 4 >= 1024 ? 1024 : K / 4 > 256 ? 512 : 256};      // (gl3_rmsnorm's rule)
  const int blocks = (n_heads + 2 * n_kv) * (head_dim / 16);
  qkv_f32_normed_kernel<<<dim3(blocks), dim3(64 * F3_WAVES), std::max(rows, K / F3_CHUNK * 1024), stream>>>(x, norm, W, q, M, K, ldx, ldw, ldq, rope);
  GL3_LAUNCH_CHECK();
  return 0;
}

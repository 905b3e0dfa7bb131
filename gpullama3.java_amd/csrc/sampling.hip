// Token selection on the device: a row's softmax by many blocks, its choice by one.
//
// temperature == 0: the first index of the strictly greatest logit
//   (J/inference/sampler/Sampler.java:144-157).
// temperature > 0: p = softmax(logits / temperature) (Sampler.java:87-89), then
//   top_p outside (0,1): the first index whose running sum in index order exceeds
//     u, else the last index (J/inference/sampler/CategoricalSampler.java:31-42);
//   top_p inside (0,1): the tokens in descending order of probability (equal
//     ones by ascending index), cut after the first at which the running sum
//     exceeds top_p; u is scaled by the kept mass and the kept list is walked in
//     that order (J/inference/sampler/ToppSampler.java:116-155).
// The uniform number u in [0,1) comes from the caller, one per row.
//
// No sort: the kept set is {p > v} plus the first k of {p == v}, where v is the
// greatest threshold whose mass {p >= v} still exceeds top_p; v is found digit by
// digit over the float's bit pattern (four passes with histograms), and the walk to
// the drawn token is the same search with u * mass in place of top_p. Masses are
// summed as 64-bit integers (p * 2^62), so the order of a sum cannot move a comparison.
//
// At most 2^13 probabilities are 2^-13 or more. They are gathered while the row is normalised; when
// their mass alone exceeds top_p, the threshold and the drawn token lie among them and both searches
// walk that short list, in shared memory, instead of the row. A flat distribution, whose nucleus
// reaches further down, takes three passes over the whole row, and up to nine where a factor of 1.03 to 1.06 in probability holds more
// than 8,192 values.
#include "common.h"
#include <atomic>
#include <chrono>
#include "gl3_noalloc.h"
#include <mutex>

#define SB 1024
#define SW 16          // waves of a block
#define UN 16          // elements a thread asks for before it uses the first: a pass is bound by trips to memory
#define QSCALE 4611686018427387904.0   // 2^62: probabilities as 64-bit integers, sums exact and in any order
#define CAND_MAX 8192  // candidates kept in shared memory: the probabilities of at least CAND_CUT
#define CAND_CUT 0.0001220703125f      // 2^-13
#define BIN_SHIFT 19   // a flat row's bins: exponent and four bits of the mantissa, of a probability of at most 1 below 2,048
#define BINS 2048

// A probability (0 <= p <= 1) as an integer: floor(p * 2^62), exact for p >= 2^-38, truncated below;
// taken from the float's bits: mantissa shifted by its exponent.
__device__ __forceinline__ unsigned long long to_q(float p) {
  const uint32_t b = __float_as_uint(p);
  const int e = (int)(b >> 23) - 127;                    // p = 1.m * 2^e (e = -127: zero or denormal, taken as 0)
  if (e < -62) return 0ull;
  const unsigned long long m = (unsigned long long)((b & 0x7fffffu) | 0x800000u);   // 24 bits, value m * 2^(e-23)
  const int sh = 62 - 23 + e;                            // q = m * 2^sh
  return sh >= 0 ? m << sh : m >> -sh;
}

struct Found {
  uint32_t bits;               // the threshold value's bit pattern
  unsigned long long above;    // mass of the values greater than it
  unsigned long long each;     // the value as an integer
  int ties;                    // how many values equal it
};

// The greatest value v with mass{p >= v} > thr, found digit by digit over the float's bit pattern
// (8, 8, 8 and 7 bits): per digit one pass builds a histogram of mass and count over the values that
// share the digits found so far, in private per-wave tables (integer adds in shared memory), and
// wave 0 walks the 256 bins from the top. If no prefix of the values exceeds thr (thr is not below
// the total mass), the smallest value is returned. `bits` (of 31): the digits below them are searched, the value's upper digits are
// `prefix` and the mass above all values with that prefix is `above`.
template <typename Src>
__device__ Found radix_search(Src p, int V, unsigned long long thr,
                              unsigned long long (*h_mass)[256], int (*h_cnt)[256], unsigned long long* t_mass,
                              int* t_cnt, unsigned long long* res, int bits = 31, uint32_t prefix = 0, unsigned long long above = 0) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  for (int shift = bits; shift > 0;) {
    const int width = min(8, shift);
    shift -= width;
    const uint32_t mask = (1u << width) - 1u;
    for (int i = tid; i < SW * 256; i += SB) { (&h_mass[0][0])[i] = 0; (&h_cnt[0][0])[i] = 0; }
    __syncthreads();
    for (int base = 0; base < V; base += UN * SB) {   // every lane stays in the loop: the wave votes below
      const int i0 = base + tid;
      float v[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) v[u] = (i0 + u * SB < V) ? p[i0 + u * SB] : -1.f;
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const uint32_t b = __float_as_uint(v[u]);
        const bool in = v[u] >= 0.f && (b >> (shift + width)) == prefix;
        const int bin = (b >> shift) & mask;
        // a wave whose lanes all fall into one bin adds once
        const int first = __builtin_amdgcn_readfirstlane(in ? bin : -1);
        if (__all(in && bin == first)) {
          unsigned long long q = to_q(v[u]);
#pragma unroll
          for (int o = 32; o > 0; o >>= 1) q += __shfl_xor(q, o, 64);
          if (lane == 0) { atomicAdd(&h_mass[wave][bin], q); atomicAdd(&h_cnt[wave][bin], 64); }
        } else if (in) {
          atomicAdd(&h_mass[wave][bin], to_q(v[u]));
          atomicAdd(&h_cnt[wave][bin], 1);
        }
      }
    }
    __syncthreads();
    if (tid < 256) {
      unsigned long long m = 0;
      int c = 0;
      for (int w = 0; w < SW; ++w) { m += h_mass[w][tid]; c += h_cnt[w][tid]; }
      t_mass[tid] = m;
      t_cnt[tid] = c;
    }
    __syncthreads();
    if (wave == 0) {
      // lane l owns bins 255-4l .. 252-4l, walked downwards
      unsigned long long mine = 0;
      int cnt_mine = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) { mine += t_mass[255 - 4 * lane - k]; cnt_mine += t_cnt[255 - 4 * lane - k]; }
      unsigned long long incl = mine;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const unsigned long long y = __shfl_up(incl, o, 64);
        if (lane >= o) incl += y;
      }
      const bool crosses = above + incl > thr;
      const unsigned long long hit = __ballot(crosses);
      const unsigned long long some = __ballot(cnt_mine > 0);
      int who, bin = -1;
      unsigned long long cum = above + incl - mine;
      if (hit) {
        who = __ffsll((long long)hit) - 1;
        if (lane == who) {
          for (int k = 0; k < 4; ++k) {
            const int b = 255 - 4 * lane - k;
            if (cum + t_mass[b] > thr) { bin = b; break; }
            cum += t_mass[b];
          }
        }
      } else {
        who = 63 - __builtin_clzll(some);   // the lowest bins that hold anything
        if (lane == who) {
          for (int k = 3; k >= 0; --k) {
            const int b = 255 - 4 * lane - k;
            if (t_cnt[b] > 0) { bin = b; break; }
          }
          cum = above + incl;
          for (int k = 3; 255 - 4 * lane - k <= bin; --k) cum -= t_mass[255 - 4 * lane - k];
        }
      }
      if (lane == who) { res[0] = (unsigned long long)bin; res[1] = cum; }
    }
    __syncthreads();
    const int bin = (int)res[0];
    above = res[1];
    prefix = (prefix << width) | (uint32_t)bin;
    if (shift == 0) {
      Found f;
      f.bits = prefix;
      f.above = above;
      f.ties = t_cnt[bin];
      f.each = f.ties ? t_mass[bin] / (unsigned long long)f.ties : 0;
      __syncthreads();
      return f;
    }
    __syncthreads();
  }
  return Found{};
}

// How many of the values that equal the threshold are kept: the smallest k with above + k * each > tq.
__device__ __forceinline__ long kept_ties(const Found& f1, unsigned long long tq) {
  long k1 = 1;
  if (f1.each > 0 && tq >= f1.above) k1 = (long)((tq - f1.above) / f1.each) + 1;
  if (k1 > f1.ties) k1 = f1.ties;
  return k1 < 1 ? 1 : k1;
}
// Which of the values that equal the drawn one is drawn, from 0 in ascending order of index.
__device__ __forceinline__ long drawn_tie(const Found& f1, long k1, const Found& f2, unsigned long long target) {
  const long j = (f2.each > 0 && target >= f2.above) ? (long)((target - f2.above) / f2.each) : 0;
  const long limit = (f2.bits == f1.bits) ? k1 : (long)f2.ties;
  return max(0L, min(j, limit - 1));
}
// The same from a list in shared memory that holds all of them (in any order): the index found bit by bit, a count of the equal ones with
// the bits so far for each, so that thousands of equal values cost no more than two. (Every entry against every other: 8,000 equal logits of
// 128,256 5.72 ms a call; so 0.15.) `counts`: 32 integers of shared memory that nobody reads any more. All threads of the block come here.
__device__ __forceinline__ void pick_equal(const float* list_p, const int* list_i, int n, const Found& f1, long k1, const Found& f2,
                                           unsigned long long target, int V, int* counts, int* winner) {
  const int tid = threadIdx.x;
  const float want = __uint_as_float(f2.bits);
  int at[CAND_MAX / SB];      // the indices of the thread's entries with that value; -1 otherwise
#pragma unroll
  for (int e = 0; e < CAND_MAX / SB; ++e) {
    const int a = tid + e * SB;
    at[e] = a < n && list_p[a] == want ? list_i[a] : -1;
  }
  if (f2.ties <= 1) {
#pragma unroll
    for (int e = 0; e < CAND_MAX / SB; ++e)
      if (at[e] >= 0) *winner = at[e];
    return;
  }
  if (tid < 32) counts[tid] = 0;
  __syncthreads();
  long left = drawn_tie(f1, k1, f2, target);
  int index = 0;
  for (int bit = 31 - __clz(max(V - 1, 1)); bit >= 0; --bit) {
    int c = 0;                // of the wave: those whose bits down to this one are the ones found and a zero
#pragma unroll
    for (int e = 0; e < CAND_MAX / SB; ++e) c += __popcll(__ballot(at[e] >> bit == index >> bit));
    if ((tid & 63) == 0 && c) atomicAdd(&counts[bit], c);
    __syncthreads();
    const int below = counts[bit];
    if (left >= below) { left -= below; index |= 1 << bit; }
  }
  if (tid == 0) *winner = index;
}

// A row's softmax is made by many blocks, ST_SLICES slices a row, in two kernels (the slices' maxima and
// sums, the probabilities), before the row's one block picks the token: a single CU draws too few
// bytes a second, and has too little arithmetic, for a row of a hundred thousand logits. Rows with
// temperature 0 are left alone by both.
#define ST_SLICES 64

// Scratch of a call, for every row: the probabilities; per slice the maximum, the sum of the
// exponentials and the mass as an integer; the candidates (probabilities of at least CAND_CUT) with
// their number and mass.
struct SampleWork {
  float* p;                        // [rows, V]
  double* slice_sum;               // [rows, ST_SLICES]
  unsigned long long* slice_mass;  // [rows, ST_SLICES]
  unsigned long long* cand_mass;   // [rows]
  float* slice_max;                // [rows, ST_SLICES]
  int* cand_count;                 // [rows]
  float* cand_p;                   // [rows, CAND_MAX]
  int* cand_i;                     // [rows, CAND_MAX]
};
#define SAMPLE_ROW_FLOATS (ST_SLICES * 5 + 4 + CAND_MAX * 2)   // beside the probabilities, 8-byte units kept whole

static SampleWork carve_sample_work(float* work, int n_rows, int V) {
  SampleWork w;
  w.p = work;
  w.slice_sum = (double*)(work + (((long)n_rows * V + 1) & ~1L));
  w.slice_mass = (unsigned long long*)(w.slice_sum + (long)n_rows * ST_SLICES);
  w.cand_mass = w.slice_mass + (long)n_rows * ST_SLICES;
  w.slice_max = (float*)(w.cand_mass + n_rows);
  w.cand_count = (int*)(w.slice_max + (long)n_rows * ST_SLICES);
  w.cand_p = (float*)(w.cand_count + n_rows);
  w.cand_i = (int*)(w.cand_p + (long)n_rows * CAND_MAX);
  return w;
}

// A call's parameters in host memory travel inside the first kernel's launch, which leaves them in the scratch for the kernels behind it
// (`to`: temperatures, top-p, uniform numbers, n_rows each); with `to` null they are in device memory already.
#define SAMPLE_STAGED 256
#define SAMPLE_LOOK_US 500      // how long a call's tokens are looked for before the stream is waited for
struct SampleArgs { float v[3][SAMPLE_STAGED]; };
struct SampleNoArgs {};

// Every slice's maximum and the sum of its exponentials around that maximum: the logits are read once for both. A slice of at most 2,048
// logits (a vocabulary of 131,072) is one stretch, held in registers between the two. Two kernels, the sum around the row's maximum,
// took 4.3 and 4.6 us (8 rows of 128,256) and the parameters a third of 1.6.
template <typename Args>
__global__ __launch_bounds__(256) void softmax_slices_kernel(const float* __restrict__ logits, long ld,
                                                             const float* __restrict__ temperature, Args args, float* __restrict__ to,
                                                             int n_rows, SampleWork w, int V) {
  __shared__ float fs[16];
  __shared__ double ds[16];
  const int row = blockIdx.x, slice = blockIdx.y, tid = threadIdx.x;
  const int per = (V + ST_SLICES - 1) / ST_SLICES;
  const int lo = min(V, slice * per), hi = min(V, lo + per);
  const float* lg = logits + (long)row * ld;
  float v[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) { const int i = lo + u * 256 + tid; v[u] = lg[min(i, V - 1)]; }      // (asked for before the temperature is known)
  float T;
  if constexpr (sizeof(Args) > 4) {
    T = args.v[0][row];
    if (slice == 0 && tid < 3) to[(long)tid * n_rows + row] = tid == 0 ? T : tid == 1 ? args.v[1][row] : args.v[2][row];
  } else {
    T = temperature[row];
  }
  if (T == 0.f) return;
  if (slice == 0 && tid == 0) { w.cand_count[row] = 0; w.cand_mass[row] = 0ull; }   // for the next kernel
  float m = -INFINITY;
  double z = 0.0;
  for (int base = lo; base < hi; base += 8 * 256) {
    if (base != lo) {
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = lg[min(base + u * 256 + tid, V - 1)];
    }
    float here = -INFINITY;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      v[u] = base + u * 256 + tid < hi ? v[u] / T : -INFINITY;      // the division of the reference, per element
      here = fmaxf(here, v[u]);
    }
    here = fmaxf(m, block_max(here, fs));
    if (base != lo && m > -INFINITY) z *= exp((double)m - (double)here);
    m = here;
    const float around = m > -INFINITY ? m : 0.f;                   // (nothing but -inf so far: no term; NaN stays NaN)
#pragma unroll
    for (int u = 0; u < 8; ++u) z += base + u * 256 + tid < hi ? (double)expf(v[u] - around) : 0.0;
  }
  z = block_sum_f64(z, ds);
  if (tid == 0) { w.slice_max[row * ST_SLICES + slice] = m; w.slice_sum[row * ST_SLICES + slice] = z; }
}

// The row's maximum and sum from its slices', the same bits in every lane: lane k has slice k's.
__device__ __forceinline__ void row_of_slices(float slice_max, double slice_sum, float& m, double& z) {
  m = slice_max;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  z = slice_max > -INFINITY ? slice_sum * exp((double)slice_max - (double)m) : slice_sum;      // (a slice of -inf alone: 0, or NaN)
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) z += __shfl_xor(z, o, 64);
}

// p = softmax(logits / T) into the scratch, each slice's mass as an integer, and the candidates.
__global__ __launch_bounds__(256) void softmax_prob_kernel(const float* __restrict__ logits, long ld,
                                                           const float* __restrict__ temperature,
                                                           const float* __restrict__ top_p, SampleWork w, int V) {
  __shared__ unsigned long long qs[2][4];
  __shared__ float bc_p[8 * 256];
  __shared__ int bc_i[8 * 256];
  __shared__ int bc_n, bc_base;
  const int row = blockIdx.x, slice = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
  // everything that the block reads is asked for before anything is looked at: one trip to memory, not five (8 rows of 128,256: 9.6 -> 8.7 us)
  const int per = (V + ST_SLICES - 1) / ST_SLICES;
  const int lo = min(V, slice * per), hi = min(V, lo + per);
  const float* lg = logits + (long)row * ld;
  float v[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) v[u] = lg[min(lo + u * 256 + tid, V - 1)];
  const float slice_max = w.slice_max[row * ST_SLICES + lane];
  const double slice_sum = w.slice_sum[row * ST_SLICES + lane];
  const float T = temperature[row], tp = top_p[row];
  if (T == 0.f) return;
  float m;
  double z;
  row_of_slices(slice_max, slice_sum, m, z);
  const float zf = (float)z;
  const bool nucleus = tp > 0.f && tp < 1.f;
  float* p = w.p + (long)row * V;
  unsigned long long mass = 0, cmass = 0;
  for (int base = lo; base < hi; base += 8 * 256) {
    if (nucleus) {
      if (tid == 0) bc_n = 0;
      __syncthreads();
    }
    if (base != lo) {
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = lg[min(base + u * 256 + tid, V - 1)];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = base + u * 256 + tid;
      if (i < hi) {
        const float pv = expf(v[u] / T - m) / zf;
        const unsigned long long q = to_q(pv);
        p[i] = pv;
        mass += q;
        if (nucleus && pv >= CAND_CUT) {
          const int slot = atomicAdd(&bc_n, 1);   // at most 8 * 256 of them
          bc_p[slot] = pv;
          bc_i[slot] = i;
          cmass += q;
        }
      }
    }
    if (nucleus) {
      // the block's candidates of this stretch go to the row's list with one addition to its counter
      __syncthreads();
      const int n = bc_n;
      if (tid == 0 && n > 0) bc_base = atomicAdd(&w.cand_count[row], n);
      __syncthreads();
      for (int k = tid; k < n; k += 256) {
        const int slot = bc_base + k;
        if (slot < CAND_MAX) {
          w.cand_p[(long)row * CAND_MAX + slot] = bc_p[k];
          w.cand_i[(long)row * CAND_MAX + slot] = bc_i[k];
        }
      }
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) { mass += __shfl_xor(mass, o, 64); cmass += __shfl_xor(cmass, o, 64); }
  if (lane == 0) { qs[0][tid >> 6] = mass; qs[1][tid >> 6] = cmass; }
  __syncthreads();
  if (tid == 0) {
    w.slice_mass[row * ST_SLICES + slice] = qs[0][0] + qs[0][1] + qs[0][2] + qs[0][3];
    const unsigned long long c = qs[1][0] + qs[1][1] + qs[1][2] + qs[1][3];
    if (c) atomicAdd(&w.cand_mass[row], c);   // integers: the order does not matter
  }
}

// The choice, one block a row. A token is written behind a barrier that follows the block's last look at the scratch: whoever has seen all
// tokens of a call may write there again (gl3_sample_host).
__global__ __launch_bounds__(SB) void sample_kernel(const float* __restrict__ logits, long ld, SampleWork w,
                                                    const float* __restrict__ temperature,
                                                    const float* __restrict__ top_p, const float* __restrict__ uniform,
                                                    int* __restrict__ out, int V, const int* __restrict__ step,
                                                    int uniform_stride) {
  __shared__ float fs[16];
  __shared__ int is[16];
  __shared__ unsigned long long h_mass[SW][256];
  __shared__ int h_cnt[SW][256];
  __shared__ unsigned long long t_mass[256];
  __shared__ int t_cnt[256];
  __shared__ unsigned long long res[2];
  __shared__ unsigned long long w_tot[SW];
  __shared__ int winner;
  __shared__ float cand_p[CAND_MAX];
  __shared__ int cand_i[CAND_MAX];
  __shared__ unsigned long long t_q[SB + 8];
  __shared__ unsigned long long bin_mass[BINS];
  __shared__ int bin_cnt[BINS];
  __shared__ int fill;
  const int row = blockIdx.x, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const float* lg = logits + (long)row * ld;
  // what the row's choice reads is asked for at once, the first candidates too, which are there or not
  // (8 rows, some 20 candidates each: 9.5 -> 6.4 us, with the walk over the candidates eight at a time below)
  const float T = temperature[row], tp = top_p[row];
  const int n_cand = w.cand_count[row];
  const unsigned long long c_mass = w.cand_mass[row];
  const float first_p = w.cand_p[(long)row * CAND_MAX + tid];
  const int first_i = w.cand_i[(long)row * CAND_MAX + tid];
  // in a run of steps replayed from a graph the step's number is read from memory
  const float uf = uniform[(step ? (long)step[0] * uniform_stride : 0) + row];

  if (T == 0.f) {
    float best = -INFINITY;
    int idx = 0x7fffffff;
    for (int i = tid; i < V; i += SB) {
      const float v = lg[i];
      if (v > best) { best = v; idx = i; }
    }
    // reduce (best, idx): greater value wins, equal values: lower index
    for (int o = 32; o > 0; o >>= 1) {
      const float ob = __shfl_xor(best, o, 64);
      const int oi = __shfl_xor(idx, o, 64);
      if (ob > best || (ob == best && oi < idx)) { best = ob; idx = oi; }
    }
    if ((tid & 63) == 0) { fs[tid >> 6] = best; is[tid >> 6] = idx; }
    __syncthreads();
    if (tid == 0) {
      for (int w2 = 1; w2 < SB / 64; ++w2)
        if (fs[w2] > best || (fs[w2] == best && is[w2] < idx)) { best = fs[w2]; idx = is[w2]; }
      out[row] = idx == 0x7fffffff ? 0 : idx;   // all -inf or NaN: index 0, as the reference's loop leaves it
    }
    return;
  }

  const float* p = w.p + (long)row * V;
  const double u = (double)uf;
  if (tid == 0) winner = -1;
  __syncthreads();

  if (tp <= 0.f || tp >= 1.f) {
    // the first index whose running sum in index order exceeds u: first the slice, by the slices' masses
    const unsigned long long uq = (unsigned long long)(u * QSCALE);   // u = k / 2^24: exact
    const unsigned long long sm = w.slice_mass[row * ST_SLICES + lane];
    unsigned long long sincl = sm;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const unsigned long long y = __shfl_up(sincl, o, 64);
      if (lane >= o) sincl += y;
    }
    const unsigned long long shit = __ballot(uq < sincl);
    if (!shit) {                      // u lies beyond the whole mass: the last index
      __syncthreads();
      if (tid == 0) out[row] = V - 1;
      return;
    }
    const int slice = __ffsll((long long)shit) - 1;
    const unsigned long long before_slice = __shfl(sincl - sm, slice, 64);
    const int sper = (V + ST_SLICES - 1) / ST_SLICES;
    const int r_lo = min(V, slice * sper), r_hi = min(V, r_lo + sper);
    // every wave owns a contiguous part of the slice, a multiple of 64 long
    const int per = ((r_hi - r_lo + SW - 1) / SW + 63) / 64 * 64;
    const int lo = min(r_hi, r_lo + wave * per), hi = min(r_hi, lo + per);
    unsigned long long mine = 0;
    for (int i0 = lo + lane; i0 < hi; i0 += 8 * 64) {
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = (i0 + 64 * k < hi) ? p[i0 + 64 * k] : 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) mine += to_q(v[k]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mine += __shfl_xor(mine, o, 64);
    if (lane == 0) w_tot[wave] = mine;
    __syncthreads();
    unsigned long long before = before_slice;
    for (int w2 = 0; w2 < wave; ++w2) before += w_tot[w2];
    if (before <= uq && uq < before + w_tot[wave]) {       // the crossing lies in this wave's part
      for (int base = lo; base < hi; base += 64) {
        const int i = base + lane;
        const unsigned long long q = i < hi ? to_q(p[i]) : 0;
        unsigned long long incl = q;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          const unsigned long long y = __shfl_up(incl, o, 64);
          if (lane >= o) incl += y;
        }
        const unsigned long long hit = __ballot(uq < before + incl);
        if (hit) {
          if (lane == 0) winner = base + __ffsll((long long)hit) - 1;
          break;
        }
        before += __shfl(incl, 63, 64);
      }
    }
    __syncthreads();
    if (tid == 0) out[row] = winner >= 0 ? winner : V - 1;
    return;
  }

  // nucleus: the threshold value, the mass above it, and how many of the equal ones are kept
  const unsigned long long tq = (unsigned long long)((double)tp * QSCALE);
  if (n_cand <= CAND_MAX && c_mass > tq) {
    // the candidates alone exceed top_p: every probability from the threshold upwards is among them
    const int n = n_cand;
    if (tid < n) { cand_p[tid] = first_p; cand_i[tid] = first_i; }
    for (int a = tid + SB; a < n; a += SB) {
      cand_p[a] = w.cand_p[(long)row * CAND_MAX + a];
      cand_i[a] = w.cand_i[(long)row * CAND_MAX + a];
    }
    __syncthreads();
    if (n <= SB) {
      // few candidates, one a thread: the mass that stands before each in the kept order (descending
      // probability, equal ones by ascending index) is summed directly. A candidate is kept if the
      // mass before it does not exceed top_p; the drawn one is that whose stretch holds u * kept mass.
      float pa = 0.f;
      int ia = 0;
      unsigned long long qa = 0;
      if (tid < n) { pa = first_p; ia = first_i; qa = to_q(pa); }
      t_q[tid] = qa;
      if (tid >= n && tid < n + 8) cand_p[tid] = -1.f;      // (n is at most SB: up to eight entries behind the last, that count for nothing)
      if (tid == 0) res[0] = c_mass;
      __syncthreads();
      unsigned long long excl = 0;
      if (tid < n)
        for (int b0 = 0; b0 < n; b0 += 8) {      // (eight at a time: a trip to shared memory for eight, not for each)
          float pb[8];
          int ib[8];
          unsigned long long qb[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) { pb[k] = cand_p[b0 + k]; ib[k] = cand_i[b0 + k]; qb[k] = t_q[b0 + k]; }
#pragma unroll
          for (int k = 0; k < 8; ++k) excl += (pb[k] > pa || (pb[k] == pa && ib[k] < ia)) ? qb[k] : 0ull;
        }
      if (tid < n && excl <= tq && tq < excl + qa) res[0] = excl + qa;   // the last kept one: the kept mass
      __syncthreads();
      const unsigned long long target = (unsigned long long)(u * (double)res[0]);
      if (tid < n && excl <= target && target < excl + qa) winner = ia;
      __syncthreads();
      if (tid == 0) out[row] = winner >= 0 ? winner : V - 1;
      return;
    }
    const Found f1 = radix_search(cand_p, n, tq, h_mass, h_cnt, t_mass, t_cnt, res);
    const long k1 = kept_ties(f1, tq);
    const unsigned long long mass = f1.above + (unsigned long long)k1 * f1.each;
    const unsigned long long target = (unsigned long long)(u * (double)mass);
    const Found f2 = radix_search(cand_p, n, target, h_mass, h_cnt, t_mass, t_cnt, res);
    pick_equal(cand_p, cand_i, n, f1, k1, f2, target, V, h_cnt[0], &winner);
    __syncthreads();
    if (tid == 0) out[row] = winner >= 0 ? winner : V - 1;
    return;
  }

  // A flat row, whose nucleus reaches below the candidates. One pass sorts the row's mass into bins of a factor of 1.03 to 1.06
  // (exponent and four bits of the mantissa); the bin in which the mass exceeds top_p, and then the one that the drawn token lies in,
  // are gathered from the row, and the searches walk those lists in shared memory: three passes over the row in place of nine
  // whose first two put all of a row into a dozen bins (8 rows of 128,256, temperature 1.2, top-p 0.95: a call 324 -> 125 us; one row 312 -> 120,
  // 64 rows 377 -> 163). A bin with more than CAND_MAX values (many equal ones, or a distribution with hardly any) stays in the row, and the
  // search goes on over the row below the bin's digits.
  for (int i = tid; i < BINS; i += SB) { bin_mass[i] = 0; bin_cnt[i] = 0; }
  __syncthreads();
  for (int base = 0; base < V; base += UN * SB) {      // every lane stays in the loop: the wave votes below
    const int i0 = base + tid;
    float v[UN];
#pragma unroll
    for (int k = 0; k < UN; ++k) v[k] = i0 + k * SB < V ? p[i0 + k * SB] : -1.f;
    // A bin that a quarter of the wave's lanes and more share is added to once (twice at most: rows of few values); lane by lane
    // on one counter, 128,256 equal logits took 0.95 ms a call; so 0.67. Whether there are such bins is looked at in two of a thread's values (the
    // first and the last lane's bin); in all sixteen, a call with a row of 128,256 normal logits took 131 us, so 121.
    bool shares = false;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const unsigned long long who = __ballot(v[k] >= 0.f);
      if (!who) break;
      const int b = v[k] >= 0.f ? (int)(__float_as_uint(v[k]) >> BIN_SHIFT) : -1;
      const int lo = __builtin_amdgcn_readlane(b, __ffsll((long long)who) - 1), hi = __builtin_amdgcn_readlane(b, 63 - __builtin_clzll(who));
      shares |= max(__popcll(__ballot(b == lo)), __popcll(__ballot(b == hi))) >= 16;
    }
#pragma unroll
    for (int k = 0; k < UN; ++k) {
      bool in = v[k] >= 0.f;
      const int b = (int)(__float_as_uint(v[k]) >> BIN_SHIFT);
#pragma unroll 1
      for (int turn = 0; shares && turn < 2; ++turn) {
        const unsigned long long who = __ballot(in);
        if (!who) break;
        const int shared = __builtin_amdgcn_readlane(b, __ffsll((long long)who) - 1);
        const bool same = in && b == shared;
        const int count = __popcll(__ballot(same));
        if (count < 16) break;
        unsigned long long q = same ? to_q(v[k]) : 0ull;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) q += __shfl_xor(q, o, 64);
        if (lane == 0) { atomicAdd(&bin_mass[shared], q); atomicAdd(&bin_cnt[shared], count); }
        in = in && !same;
      }
      if (in) {
        atomicAdd(&bin_mass[b], to_q(v[k]));
        atomicAdd(&bin_cnt[b], 1);
      }
    }
  }
  __syncthreads();
  int n = 0, n_bin = -1;
  // the values of the bin where the mass from the top exceeds thr (the lowest bin with any if none does), and the mass above that bin
  auto gather = [&](unsigned long long thr, unsigned long long& above, int& bin) {
    if (wave == 0) {
      // lane l owns bins BINS - 1 - 32 l downwards
      unsigned long long mine = 0;
      int cnt_mine = 0;
      for (int k = 0; k < BINS / 64; ++k) { mine += bin_mass[BINS - 1 - lane * (BINS / 64) - k]; cnt_mine += bin_cnt[BINS - 1 - lane * (BINS / 64) - k]; }
      unsigned long long incl = mine;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const unsigned long long y = __shfl_up(incl, o, 64);
        if (lane >= o) incl += y;
      }
      const unsigned long long hit = __ballot(incl > thr), some = __ballot(cnt_mine > 0);
      const int who = hit ? __ffsll((long long)hit) - 1 : some ? 63 - __builtin_clzll(some) : 0;
      if (lane == who) {
        unsigned long long cum = incl - mine, at = cum;
        int bin = -1;
        for (int k = 0; k < BINS / 64; ++k) {
          const int b = BINS - 1 - lane * (BINS / 64) - k;
          if (bin_cnt[b] > 0) { bin = b; at = cum; }
          if (hit && cum + bin_mass[b] > thr) break;
          cum += bin_mass[b];
        }
        res[0] = (unsigned long long)(long long)bin;
        res[1] = at;
      }
    }
    __syncthreads();
    bin = (int)(long long)res[0];
    above = res[1];
    const int found = bin < 0 ? -1 : bin_cnt[bin];
    if (found < 0 || found > CAND_MAX) {
      __syncthreads();
      return found;
    }
    if (bin != n_bin) {
      n_bin = bin;
      n = found;
      if (tid == 0) fill = 0;
      __syncthreads();
      for (int base = tid; base < V; base += UN * SB) {
        float v[UN];
#pragma unroll
        for (int k = 0; k < UN; ++k) v[k] = base + k * SB < V ? p[base + k * SB] : -1.f;
#pragma unroll
        for (int k = 0; k < UN; ++k)
          if (v[k] >= 0.f && (int)(__float_as_uint(v[k]) >> BIN_SHIFT) == bin) {
            const int slot = atomicAdd(&fill, 1);
            cand_p[slot] = v[k];
            cand_i[slot] = base + k * SB;
          }
      }
    }
    __syncthreads();
    return found;
  };
  unsigned long long over1 = 0, over2 = 0;
  int bin1 = 0, bin2 = 0;
  const int found1 = gather(tq, over1, bin1);
  if (found1 < 0) {                 // (not a number in the row: the last index)
    __syncthreads();
    if (tid == 0) out[row] = V - 1;
    return;
  }
  Found f1;
  if (found1 <= CAND_MAX) f1 = radix_search(cand_p, n, tq, h_mass, h_cnt, t_mass, t_cnt, res, BIN_SHIFT, (uint32_t)bin1, over1);
  else f1 = radix_search(p, V, tq, h_mass, h_cnt, t_mass, t_cnt, res, BIN_SHIFT, (uint32_t)bin1, over1);
  const long k1 = kept_ties(f1, tq);
  const unsigned long long mass = f1.above + (unsigned long long)k1 * f1.each;
  // the drawn token: first in the kept order whose running sum exceeds u * mass
  const unsigned long long target = (unsigned long long)(u * (double)mass);
  if (gather(target, over2, bin2) <= CAND_MAX) {
    const Found f2 = radix_search(cand_p, n, target, h_mass, h_cnt, t_mass, t_cnt, res, BIN_SHIFT, (uint32_t)bin2, over2);
    pick_equal(cand_p, cand_i, n, f1, k1, f2, target, V, h_cnt[0], &winner);
    __syncthreads();
    if (tid == 0) out[row] = winner >= 0 ? winner : V - 1;
    return;
  }
  const Found f2 = radix_search(p, V, target, h_mass, h_cnt, t_mass, t_cnt, res, BIN_SHIFT, (uint32_t)bin2, over2);
  const float want_value = __uint_as_float(f2.bits);   // the drawn token is the `want_index`-th (from 0) with this
  const long want_index = drawn_tie(f1, k1, f2, target);   // probability, in ascending order of index

  // every wave owns a contiguous range of the row, a multiple of 64 long
  const int per = ((V + SW - 1) / SW + 63) / 64 * 64;
  const int lo = min(V, wave * per), hi = min(V, lo + per);
  int mine = 0;
  for (int i0 = lo + lane; i0 < hi; i0 += 8 * 64) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = (i0 + 64 * k < hi) ? p[i0 + 64 * k] : -1.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) mine += (v[k] == want_value) ? 1 : 0;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mine += __shfl_xor(mine, o, 64);
  if (lane == 0) w_tot[wave] = (unsigned long long)mine;
  __syncthreads();
  long before = 0;
  for (int w2 = 0; w2 < wave; ++w2) before += (long)w_tot[w2];
  if (before <= want_index && want_index < before + (long)w_tot[wave]) {
    for (int base = lo; base < hi; base += 64) {
      const int i = base + lane;
      const unsigned long long hit = __ballot(i < hi && p[i] == want_value);
      const int n = __popcll(hit);
      if (want_index < before + n) {
        if (lane == 0) {
          unsigned long long h = hit;
          for (long skip = want_index - before; skip > 0; --skip) h &= h - 1;   // drop the lowest set bits
          winner = base + __ffsll((long long)h) - 1;
        }
        break;
      }
      before += n;
    }
  }
  __syncthreads();
  if (tid == 0) out[row] = winner >= 0 ? winner : V - 1;
}

// Greedy rows only, in two stages so that a row is read by many blocks at once: each block finds the
// first greatest logit of its slice, a second kernel the first greatest of the slices' results.
#define ARG_SLICES 64

__global__ __launch_bounds__(256) void argmax_slice_kernel(const float* __restrict__ logits, long ld,
                                                           float* __restrict__ part_val, int* __restrict__ part_idx,
                                                           int V) {
  __shared__ float fs[4];
  __shared__ int is[4];
  const int row = blockIdx.x, slice = blockIdx.y, tid = threadIdx.x;
  const int per = (V + ARG_SLICES - 1) / ARG_SLICES;
  const int lo = slice * per, hi = min(V, lo + per);
  const float* lg = logits + (long)row * ld;
  float best = -INFINITY;
  int idx = 0x7fffffff;
  for (int i = lo + tid; i < hi; i += 256) {
    const float v = lg[i];
    if (v > best) { best = v; idx = i; }
  }
  for (int o = 32; o > 0; o >>= 1) {
    const float ob = __shfl_xor(best, o, 64);
    const int oi = __shfl_xor(idx, o, 64);
    if (ob > best || (ob == best && oi < idx)) { best = ob; idx = oi; }
  }
  if ((tid & 63) == 0) { fs[tid >> 6] = best; is[tid >> 6] = idx; }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < 4; ++w)
      if (fs[w] > best || (fs[w] == best && is[w] < idx)) { best = fs[w]; idx = is[w]; }
    part_val[row * ARG_SLICES + slice] = best;
    part_idx[row * ARG_SLICES + slice] = idx;
  }
}

__global__ __launch_bounds__(64) void argmax_final_kernel(const float* __restrict__ part_val,
                                                          const int* __restrict__ part_idx, int* __restrict__ out) {
  const int row = blockIdx.x, lane = threadIdx.x;
  float best = part_val[row * ARG_SLICES + lane];
  int idx = part_idx[row * ARG_SLICES + lane];
  for (int o = 32; o > 0; o >>= 1) {
    const float ob = __shfl_xor(best, o, 64);
    const int oi = __shfl_xor(idx, o, 64);
    if (ob > best || (ob == best && oi < idx)) { best = ob; idx = oi; }
  }
  if (lane == 0) out[row] = idx == 0x7fffffff ? 0 : idx;
}

// Every row greedy (J/inference/sampler/Sampler.java:144-157). work: at least 2 * n_rows * 64 floats.
extern "C" int gl3_argmax(const float* logits, long ld, float* work, int* out, int n_rows, int V, hipStream_t stream) {
  if (n_rows == 0) return 0;
  GL3_REQUIRE(logits && work && out && n_rows > 0 && V > 0 && ld >= V, "gl3_argmax: bad arguments");
  GL3_REQUIRE(n_rows <= 65535, "gl3_argmax: too many rows");
  float* pv = work;
  int* pi = (int*)(work + (long)n_rows * ARG_SLICES);
  argmax_slice_kernel<<<dim3(n_rows, ARG_SLICES), dim3(256), 0, stream>>>(logits, ld, pv, pi, V);
  GL3_LAUNCH_CHECK();
  argmax_final_kernel<<<dim3(n_rows), dim3(64), 0, stream>>>(pv, pi, out);
  GL3_LAUNCH_CHECK();
  return 0;
}

// The greedy pick of a decode step inside a run, and what follows it between two steps of the run (as
// gl3_decode_advance does): each row's winner is the sequence's next token, goes into row step[0] of `history`, the
// sequence moves on by one position, and the step counter goes up. One block does the second stage for all rows
// (a wave a row, in turn), so the counter is read by everyone before it changes: one launch instead of two.
__global__ __launch_bounds__(1024) void argmax_final_advance_kernel(const float* __restrict__ part_val,
                                                                    const int* __restrict__ part_idx, int* __restrict__ out,
                                                                    int n_rows, int* __restrict__ token_ids,
                                                                    int* __restrict__ positions, int* __restrict__ kv_before,
                                                                    int* __restrict__ history, int history_stride,
                                                                    int* __restrict__ step) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int s = step[0];
  __syncthreads();
  for (int row = wave; row < n_rows; row += 16) {
    float best = part_val[row * ARG_SLICES + lane];
    int idx = part_idx[row * ARG_SLICES + lane];
    for (int o = 32; o > 0; o >>= 1) {
      const float ob = __shfl_xor(best, o, 64);
      const int oi = __shfl_xor(idx, o, 64);
      if (ob > best || (ob == best && oi < idx)) { best = ob; idx = oi; }
    }
    if (lane == 0) {
      const int t = idx == 0x7fffffff ? 0 : idx;
      out[row] = t;
      token_ids[row] = t;
      history[(long)s * history_stride + row] = t;
      positions[row] += 1;
      kv_before[row] += 1;
    }
  }
  if (threadIdx.x == 0) step[0] = s + 1;
}

extern "C" int gl3_argmax_advance(const float* logits, long ld, float* work, int* out, int n_rows, int V, int* token_ids,
                                  int* positions, int* kv_before, int* history, int history_stride, int* step,
                                  hipStream_t stream) {
  if (n_rows == 0) return 0;
  GL3_REQUIRE(logits && work && out && n_rows > 0 && V > 0 && ld >= V, "gl3_argmax_advance: bad arguments");
  GL3_REQUIRE(token_ids && positions && kv_before && history && step && history_stride >= n_rows && n_rows <= 1024,
              "gl3_argmax_advance: rows=%d stride=%d", n_rows, history_stride);
  float* pv = work;
  int* pi = (int*)(work + (long)n_rows * ARG_SLICES);
  argmax_slice_kernel<<<dim3(n_rows, ARG_SLICES), dim3(256), 0, stream>>>(logits, ld, pv, pi, V);
  GL3_LAUNCH_CHECK();
  argmax_final_advance_kernel<<<dim3(1), dim3(1024), 0, stream>>>(pv, pi, out, n_rows, token_ids, positions, kv_before,
                                                                  history, history_stride, step);
  GL3_LAUNCH_CHECK();
  return 0;
}

// The same without a workspace from the caller (see gl3_noalloc.h): the slices' partial results live
// in a device array of this library. In host code `scratch` is only a handle for the runtime, not a
// device address; the address on each GPU is asked for once, with that GPU current, and kept.
static __device__ __align__(256) float scratch[GL3_ARGMAX_STATIC_ROWS * 2 * ARG_SLICES];
#define GL3_MAX_DEVICES 64
static float* g_scratch_ptr[GL3_MAX_DEVICES];
static std::mutex g_scratch_mutex;

extern "C" int gl3_argmax_static(const float* logits, long ld, int* out, int n_rows, int V, hipStream_t stream) {
  if (n_rows == 0) return 0;
  GL3_REQUIRE(logits && out && n_rows > 0 && V > 0 && ld >= V, "gl3_argmax_static: bad arguments");
  GL3_REQUIRE(n_rows <= GL3_ARGMAX_STATIC_ROWS, "gl3_argmax_static: %d rows exceed the %d that the library's array holds",
              n_rows, GL3_ARGMAX_STATIC_ROWS);
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  GL3_REQUIRE(e == hipSuccess && dev >= 0 && dev < GL3_MAX_DEVICES, "gl3_argmax_static: no current device (%s)",
              hipGetErrorString(e));
  float* work;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
      void* p = nullptr;
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      GL3_REQUIRE(e == hipSuccess && p != nullptr, "gl3_argmax_static: the array's address on device %d: %s", dev,
                  hipGetErrorString(e));
      g_scratch_ptr[dev] = (float*)p;
    }
    work = g_scratch_ptr[dev];
  }
  float* pv = work;
  int* pi = (int*)(work + (long)GL3_ARGMAX_STATIC_ROWS * ARG_SLICES);
  argmax_slice_kernel<<<dim3(n_rows, ARG_SLICES), dim3(256), 0, stream>>>(logits, ld, pv, pi, V);
  GL3_LAUNCH_CHECK();
  argmax_final_kernel<<<dim3(n_rows), dim3(64), 0, stream>>>(pv, pi, out);
  GL3_LAUNCH_CHECK();
  return 0;
}

// Floats of scratch that gl3_sample needs: the rows' probabilities and, per row, what the kernels
// hand to each other.
extern "C" long gl3_sample_work_floats(int n_rows, int V) {
  return (((long)n_rows * V + 1) & ~1L) + (long)n_rows * SAMPLE_ROW_FLOATS;
}

static int launch_choice(const float* logits, long ld, const SampleWork& w, const float* temperature, const float* top_p,
                         const float* uniform, int* out, int n_rows, int V, const int* step, int uniform_stride, hipStream_t stream) {
  softmax_prob_kernel<<<dim3(n_rows, ST_SLICES), dim3(256), 0, stream>>>(logits, ld, temperature, top_p, w, V);
  GL3_LAUNCH_CHECK();
  sample_kernel<<<dim3(n_rows), dim3(SB), 0, stream>>>(logits, ld, w, temperature, top_p, uniform, out, V, step, uniform_stride);
  GL3_LAUNCH_CHECK();
  return 0;
}

// work: gl3_sample_work_floats(n_rows, V) floats of scratch, 8-byte aligned.
// step (may be null): a counter in device memory; row r then takes uniform[step[0] * uniform_stride + r].
extern "C" int gl3_sample(const float* logits, long ld, float* work, const float* temperature, const float* top_p,
                          const float* uniform, int* out, int n_rows, int V, const int* step, int uniform_stride,
                          hipStream_t stream) {
  if (n_rows == 0) return 0;
  GL3_REQUIRE(logits && work && temperature && top_p && uniform && out, "gl3_sample: null argument");
  GL3_REQUIRE(n_rows > 0 && n_rows <= 65535 && V > 0 && ld >= V, "gl3_sample: bad sizes (rows=%d V=%d ld=%ld)", n_rows, V,
              ld);
  GL3_REQUIRE((uintptr_t)work % 8 == 0, "gl3_sample: the scratch must be 8-byte aligned");
  const SampleWork w = carve_sample_work(work, n_rows, V);
  softmax_slices_kernel<<<dim3(n_rows, ST_SLICES), dim3(256), 0, stream>>>(logits, ld, temperature, SampleNoArgs{}, nullptr, n_rows, w, V);
  GL3_LAUNCH_CHECK();
  return launch_choice(logits, ld, w, temperature, top_p, uniform, out, n_rows, V, step, uniform_stride, stream);
}

// A whole call of a sampler whose caller waits for the tokens: parameters in host memory, tokens into host memory. The parameters
// travel inside the first kernel's launch and the tokens are written by the last kernel into pinned memory (`out`: hipHostMalloc's, which
// the GPU reaches under the host's address), where the call looks for them: nothing to copy on either side, and no wait for the stream's end,
// which came 5 us behind the tokens. 8 rows of 128,256 logits 36.8 -> 31.6 us a call, 64 rows 66.7 -> 62.4; greedy 8 rows 22.3 -> 17.5, other logits each
// time 24.4 -> 19.2, after 3 ms without work 31.6 -> 25.4. Behind a decode step, which takes longer than the look, the call waits for the stream as ever and is no shorter
// (both ways of waiting keep the calling thread's core busy: 2,582 us of its time behind 2.6 ms of products).
// work: gl3_sample_work_floats(n_rows, V) floats and 3 * n_rows for the parameters. temperature null: every row greedy (work as
// gl3_argmax's). The stream must not be capturing.
extern "C" int gl3_sample_host(const float* logits, long ld, float* work, const float* temperature, const float* top_p,
                               const float* uniform, int* out, int n_rows, int V, hipStream_t stream) {
  if (n_rows == 0) return 0;
  GL3_REQUIRE(logits && work && out && n_rows > 0 && V > 0, "gl3_sample_host: bad arguments");
  for (int i = 0; i < n_rows; ++i) out[i] = -1;      // (no token yet)
  int rc;
  if (temperature) {
    GL3_REQUIRE(top_p && uniform, "gl3_sample_host: null argument");
    GL3_REQUIRE(n_rows <= 65535 && ld >= V && (uintptr_t)work % 8 == 0, "gl3_sample_host: bad sizes (rows=%d V=%d ld=%ld) or scratch", n_rows, V, ld);
    const SampleWork w = carve_sample_work(work, n_rows, V);
    float* par = work + gl3_sample_work_floats(n_rows, V);
    // (SAMPLE_STAGED rows at a time: their parameters are 3 KB of a launch's arguments)
    for (int first = 0; first < n_rows; first += SAMPLE_STAGED) {
      SampleArgs a;
      const int count = n_rows - first < SAMPLE_STAGED ? n_rows - first : SAMPLE_STAGED;
      for (int i = 0; i < count; ++i) { a.v[0][i] = temperature[first + i]; a.v[1][i] = top_p[first + i]; a.v[2][i] = uniform[first + i]; }
      for (int i = count; i < SAMPLE_STAGED; ++i) a.v[0][i] = a.v[1][i] = a.v[2][i] = 0.f;
      SampleWork part = w;      // (what the slices' kernel writes, from row `first` on)
      part.slice_sum += (long)first * ST_SLICES;
      part.slice_max += (long)first * ST_SLICES;
      part.cand_mass += first;
      part.cand_count += first;
      softmax_slices_kernel<<<dim3(count, ST_SLICES), dim3(256), 0, stream>>>(logits + (long)first * ld, ld, nullptr, a, par + first, n_rows, part, V);
      GL3_LAUNCH_CHECK();
    }
    rc = launch_choice(logits, ld, w, par, par + n_rows, par + 2L * n_rows, out, n_rows, V, nullptr, 0, stream);
  } else {
    rc = gl3_argmax(logits, ld, work, out, n_rows, V, stream);
  }
  if (rc) return rc;
  // The call is over when the tokens are there: they are looked at where the last kernel writes them. (Waiting for the stream takes its end, a
  // packet of its own and that packet's signal.) What ran on the stream before them is done, and the kernel reads no scratch behind a token. A call that
  // takes longer, or whose tokens do not come, waits for the stream.
  const volatile int* tokens = out;
  int seen = 0;
  for (const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(SAMPLE_LOOK_US); std::chrono::steady_clock::now() < until;) {
    for (int spin = 0; spin < 32; ++spin) {
      while (seen < n_rows && tokens[seen] >= 0) ++seen;
      if (seen == n_rows) {
        std::atomic_thread_fence(std::memory_order_acquire);
        return 0;
      }
      __builtin_ia32_pause();
    }
  }
  const hipError_t e = hipStreamSynchronize(stream);
  GL3_REQUIRE(e == hipSuccess, "gl3_sample_host: %s", hipGetErrorString(e));
  return 0;
}

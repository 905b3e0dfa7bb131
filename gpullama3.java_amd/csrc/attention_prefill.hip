// Causal grouped-query attention in bfloat16 for steps that bring many tokens per
// sequence (prompts, chunks), over the paged cache that already holds this step's keys
// and values. Formulas as J/inference/InferenceCore.java:106-145: query head h reads kv
// head h / (H/K); score = q.k * scale over the keys lo..p of the query's own position
// p; softmax; weighted sum of the values.
//
// A block is four waves on 64 consecutive queries of one sequence; a wave owns 16 of them
// and up to GH query heads that share one kv head. The block walks the keys in chunks of
// 32: its 256 threads bring a chunk of keys and of transposed values from the cache into
// shared memory once (the next chunk travels to registers while the current one is
// worked on, and goes into the other of two buffers), and every wave reads its operands
// from there, so the first-level cache carries each key once per block and not once per
// wave. Both products are transposed, as in the decode kernel:
//   S^T[key, query]  = K[key, :] . Q[query, :]^T
//   O^T[dim, query] += V^T[dim, key] . P^T[key, query]
// which makes 16 bytes of a key row, and of a row of the transposed value page, the
// operands as the instruction wants them, and leaves the probabilities in the register
// order the second product takes (row i of the first score tile is key 8*(i/4) + i%4 of
// the chunk, row i of the second the key 4 further, so a quarter of the lanes ends up with
// 8 consecutive keys). The running maximum and sum of the softmax are kept in 32-bit, in
// units of log2: p = 2^(s*scale*log2(e) - m) is one multiply-add and one exponential per
// score; chunks that every query of the wave sees whole skip the mask, and the sums are
// rescaled only when some maximum moved. Rows in shared memory are padded by 16 bytes, which
// spreads the 16 rows that a quarter of the lanes reads over all banks.
#include "common.h"
#include "lds_loads.h"
#include <climits>
#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// max over the four lanes j, j+16, j+32, j+48 (which hold different keys of one query), by the
// row-swap instructions: no trip through shared memory as a general shuffle makes
__device__ __forceinline__ float max_over_quarters(float x) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float m = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// BIAS (both kernels): a bias on the scores that grows with the distance, score - slopes[head] * (p - key), and a
// sink (a key without a value that every query sees with the score `sink`: the running softmax starts from it
// instead of from nothing). A template parameter: the kernels without them are compiled as they were. RULE (with BIAS):
// a Gl3ScoreRule (common.h); each score is then brought into units of log2 by itself, bias and all, where without
// a rule the scale rides in the exponential.
template <int HS, int GH, bool BIAS = false, bool RULE = false>
__global__ __launch_bounds__(256, 2) void attention_prefill_kernel(
    const bf16_t* __restrict__ q, long q_stride, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
    const int* __restrict__ cu_seqlens, const int* __restrict__ kv_before, const int* __restrict__ block_table,
    const int* __restrict__ seq_rows, int table_stride, bf16_t* __restrict__ out, long out_stride, int n_heads, int n_kv, int page_size, int window,
    float scale, int q_blocks, const float* __restrict__ slopes, int has_sink, float sink, int keep_first, int mask_chunk, int maps,
    const float* __restrict__ sinks, Gl3ScoreRule rule) {
  constexpr int KK = HS / 32;
  constexpr int DT = HS / 16;
  constexpr int KROW = HS + 8;            // a key row in shared memory, in elements
  constexpr int VROW = 32 + 8;            // a row of the transposed value chunk
  constexpr int UNITS = HS * 4;           // 16-byte units of a chunk of keys (and of values)
  constexpr int NU = (UNITS + 255) / 256; // units per thread
  __shared__ __attribute__((aligned(16))) bf16_t ks[2][32][KROW];
  __shared__ __attribute__((aligned(16))) bf16_t vs[2][HS][VROW];
  const int g = n_heads / n_kv;
  const int groups = (g + GH - 1) / GH;
  // the longest query blocks first, of all heads and sequences: blockIdx.z counts down through a
  // sequence, the heads (x, which varies fastest as blocks are handed out) and sequences inside it
  const int qb = q_blocks - 1 - blockIdx.z;
  const int b = blockIdx.y;
  const int c = blockIdx.x / groups, hg = blockIdx.x % groups;
  // scalar: what depends on the wave alone (chunk, page) lives in scalar registers
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int j = lane & 15, qd = lane >> 4;
  const int tok0 = __builtin_amdgcn_readfirstlane(cu_seqlens[b]);
  const int q_len = __builtin_amdgcn_readfirstlane(cu_seqlens[b + 1]) - tok0;
  if (qb * 64 >= q_len) return;            // the whole block: no barrier has been passed yet
  const int before = __builtin_amdgcn_readfirstlane(kv_before[b]);
  const int heads_here = min(GH, g - hg * GH);
  const int h0 = c * g + hg * GH;
  // (several score maps over the same values: query and key heads lie head by head as [map 0, map 1, ...]; key head c is
  // map c % maps of group c / maps, read by that map of the group's g heads, and goes with value head c / maps)
  auto head_at = [&](int hh) { return maps > 1 ? ((c / maps) * g + hg * GH + hh) * maps + c % maps : h0 + hh; };
  const int n_v = n_kv / maps, cv = c / maps;
  // the sequence's row of the table: its number in the batch, or what `seq_rows` says (a table with a row per cache slot)
  const int* bt = block_table + (long)(seq_rows ? __builtin_amdgcn_readfirstlane(seq_rows[b]) : b) * table_stride;
  // the block's range of chunks, and the wave's own inside it
  const int blk_first = before + qb * 64, blk_last = before + min(qb * 64 + 63, q_len - 1);
  // the first key that position p sees: its chunk's first (a chunked mask), the window's, or the sequence's
  auto low_of = [&](int p) { return mask_chunk > 0 ? p - p % mask_chunk : (window > 0 && p + 1 > window) ? p + 1 - window : 0; };
  const int blk_lo = low_of(blk_first);
  // With a window, the sequence's first keep_first keys stay visible (BIAS kernels only). Their chunks that lie before
  // the window's first chunk ckw are numbered in front of it: ck0 .. ckw - 1 stand for chunks 0 .. ckw - ck0 - 1.
  const int ckw = blk_lo / 32, ck1 = blk_last / 32;
  const int ck0 = ckw - (BIAS ? min((keep_first + 31) / 32, ckw) : 0);
  auto real = [&](int ck) { return (BIAS && ck < ckw) ? ck - ck0 : ck; };
  const int qi0 = qb * 64 + wave * 16;     // first query of this wave, counted inside the step's tokens
  const bool active = qi0 < q_len;
  const bool q_ok = qi0 + j < q_len;
  const int p_mine = before + qi0 + j;                           // position of this lane's query
  const int p_last = before + min(qi0 + 15, q_len - 1);          // last position of the wave
  const int p_first = before + qi0;
  const int lo_first = low_of(p_first);
  const int lo_last = low_of(p_last);
  const int lo_mine = low_of(p_mine);
  const int ck_first = active ? lo_first / 32 : 1, ck_last = active ? p_last / 32 : 0;

  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8 qt[GH][KK];
#pragma unroll
  for (int hh = 0; hh < GH; ++hh)
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
      qt[hh][kk] = (q_ok && hh < heads_here)
                       ? *(const bf16x8*)(q + (long)(tok0 + qi0 + j) * q_stride + (long)head_at(hh) * HS + kk * 32 + 8 * qd)
                       : zero8;

  float m_run[GH], l_run[GH];
  f32x4 o[GH][DT];
#pragma unroll
  for (int hh = 0; hh < GH; ++hh) {
    m_run[hh] = -INFINITY;
    l_run[hh] = 0.f;
    if (BIAS && (has_sink || sinks)) {          // (a lane holds its quarter's share of the row sum: the sink's 1 once a query)
      m_run[hh] = (sinks ? sinks[min(head_at(hh), n_heads - 1)] : sink) * 1.4426950408889634f;
      l_run[hh] = qd == 0 ? 1.f : 0.f;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[hh][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float sl[GH];                                 // the heads' slopes over the scale: the scores are scaled afterwards
#pragma unroll
  for (int hh = 0; hh < GH; ++hh)
    sl[hh] = (BIAS && slopes && hh < heads_here) ? slopes[head_at(hh)] * (RULE ? 1.4426950408889634f : 1.0f / scale) : 0.f;

  // cache -> registers -> shared memory, 16 bytes a unit: a chunk's keys are 32 consecutive rows
  // of a page, its values 32 consecutive positions of each of the HS rows of the transposed page.
  // Three chunks are on their way in registers while one is worked on: a chunk's work takes a
  // fraction of a trip to memory.
  constexpr int AHEAD = 3;
  bf16x8 rk[AHEAD][NU], rv[AHEAD][NU];
  auto fetch = [&](int ck, bf16x8 (&fk)[NU], bf16x8 (&fv)[NU]) {
    const int key0 = ck * 32;
    const long page = __builtin_amdgcn_readfirstlane(bt[key0 / page_size]);
    const int po = key0 % page_size;
    // (inside a page both lie in tiles, gl3_k_offset and gl3_v_offset: the chunk's keys are still
    // 32 * HS consecutive elements, its values 512 consecutive elements for every 16 dims)
    const bf16_t* kb = k_cache + ((page * n_kv + c) * page_size + po) * HS;
    const bf16_t* vb = v_cache + (page * n_v + cv) * (long)page_size * HS + (long)(po / 8) * 128;
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + 256 * i;
      if (UNITS % 256 == 0 || u < UNITS) {
        fk[i] = *(const bf16x8*)(kb + u * 8);
        fv[i] = *(const bf16x8*)(vb + (long)(u >> 6) * page_size * 16 + (u & 63) * 8);
      }
    }
  };
  auto stage = [&](int buf, const bf16x8 (&fk)[NU], const bf16x8 (&fv)[NU]) {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + 256 * i;
      if (UNITS % 256 == 0 || u < UNITS) {
        // unit u of the keys: tile u / (2 HS) of the two, column block (u / 16) % (HS / 8), row u % 16
        const int row = u & 15, tile = u / (2 * HS);
        *(bf16x8*)&ks[buf][8 * (row >> 2) + 4 * tile + (row & 3)][((u >> 4) % (HS / 8)) * 8] = fk[i];
        // unit u of the values: 16 dims u / 64, positions 8 * ((u % 64) / 16) .., dim u % 16 of the 16
        *(bf16x8*)&vs[buf][(u >> 6) * 16 + (u & 15)][((u >> 4) & 3) * 8] = fv[i];
      }
    }
  };

  const float c2 = RULE ? 1.0f : scale * 1.4426950408889634f;   // scores in units of log2
  const float q_scale = RULE ? scale * gl3_query_temperature(p_mine, rule) : 0.f;
  const float cap2 = RULE ? rule.softcap * 1.4426950408889634f : 0.f;      // the cap in units of log2
  const float rule_in = !RULE ? 0.f : cap2 > 0.f ? 2.8853900817779268f * q_scale / rule.softcap : q_scale * 1.4426950408889634f;
  const int krow = 8 * (j >> 2) + (j & 3);   // which key of a chunk is row j of the first score tile

  // one chunk of one head: scores, running softmax, weighted values. MASKED: some query of the
  // wave does not see some key of the chunk (the diagonal, a window's edge).
  auto head_chunk = [&](int hh, const bf16x8 (&ka)[KK], const bf16x8 (&kb2)[KK], const bf16x8 (&vt)[DT], int key0,
                        bool masked) {
    f32x4 sa = {0.f, 0.f, 0.f, 0.f}, sb = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      sa = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[kk], qt[hh][kk], sa, 0, 0, 0);
      sb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb2[kk], qt[hh][kk], sb, 0, 0, 0);
    }
    float s[8];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      s[v] = sa[v];
      s[4 + v] = sb[v];
    }
    if (RULE) {
      // (the bias as slope * key minus slope * position, so that a score takes one multiply-add for it; the cap's own
      // cap - 2 cap / (1 + e^2y) starts from it)
      const float base = (cap2 > 0.f ? cap2 : 0.f) - sl[hh] * (float)(p_mine - key0 - 8 * qd);
      if (cap2 > 0.f) {
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] = fmaf(-2.0f * cap2, gl3_tanh_part(s[e] * rule_in), fmaf(sl[hh], (float)e, base));
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] = fmaf(s[e], rule_in, fmaf(sl[hh], (float)e, base));
      }
    } else if (BIAS) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int k1 = key0 + 8 * qd + v;
        s[v] = fmaf(-sl[hh], (float)(p_mine - k1), s[v]);
        s[4 + v] = fmaf(-sl[hh], (float)(p_mine - k1 - 4), s[4 + v]);
      }
    }
    if (masked) {                               // (the same for the whole wave: a branch around the tests, one body)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int k1 = key0 + 8 * qd + v, k2 = k1 + 4;
        s[v] = ((k1 >= lo_mine || (BIAS && k1 < keep_first)) && k1 <= p_mine) ? s[v] : -INFINITY;
        s[4 + v] = ((k2 >= lo_mine || (BIAS && k2 < keep_first)) && k2 <= p_mine) ? s[4 + v] : -INFINITY;
      }
    }
    float mx = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
    mx = max_over_quarters(mx);
    mx *= c2;                                   // c2 > 0: the greatest score stays the greatest
    const float m_new = fmaxf(m_run[hh], mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m_run[hh] - m_use);
    float ps = 0.f;
    bf16x8 pb;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float p = __builtin_amdgcn_exp2f(fmaf(s[e], c2, -m_use));
      ps += p;
      pb[e] = static_cast<bf16_t>(p);
    }
    l_run[hh] = l_run[hh] * alpha + ps;
    m_run[hh] = m_new;
    if (!__all(alpha == 1.0f)) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[hh][dt] *= alpha;
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      o[hh][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vt[dt], pb, o[hh][dt], 0, 0, 0);
  };

#pragma unroll
  for (int r = 0; r < AHEAD; ++r)
    if (ck0 + r <= ck1) fetch(real(ck0 + r), rk[r], rv[r]);
  stage(0, rk[0], rv[0]);
  __syncthreads();
  int buf = 0;
  for (int base = ck0; base <= ck1; base += AHEAD) {
#pragma unroll
    for (int r = 0; r < AHEAD; ++r) {
      const int ck = base + r;
      if (ck > ck1) break;
      const int key0 = real(ck) * 32;
      // the registers of this chunk are free (it lies in shared memory): ask for the chunk three further;
      fetch(real(min(ck + AHEAD, ck1)), rk[r], rv[r]);   // unconditional (the last chunk again at the end): a branch
                                                   // around the loads makes the compiler wait for all of them at once
      if (active && (ck >= ck_first || (BIAS && key0 < keep_first)) && ck <= ck_last) {
        bf16x8 ka[KK], kb2[KK], vt[DT];
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          ka[kk] = *(const bf16x8*)&ks[buf][krow][kk * 32 + 8 * qd];
          kb2[kk] = *(const bf16x8*)&ks[buf][krow + 4][kk * 32 + 8 * qd];
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) vt[dt] = *(const bf16x8*)&vs[buf][dt * 16 + j][8 * qd];
        // every query of the wave sees the whole chunk: no mask (the same for the whole wave)
        const bool masked = (BIAS && ck < ckw) || !(key0 + 31 <= p_first && key0 >= lo_last);
#pragma unroll
        for (int hh = 0; hh < GH; ++hh) head_chunk(hh, ka, kb2, vt, key0, masked);
      }
      if (ck < ck1) stage(buf ^ 1, rk[(r + 1) % AHEAD], rv[(r + 1) % AHEAD]);
      __syncthreads();
      buf ^= 1;
    }
  }

#pragma unroll
  for (int hh = 0; hh < GH; ++hh) {
    float l = l_run[hh];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (!q_ok || hh >= heads_here) continue;
    const float inv = 1.0f / l;
    bf16_t* op = out + (long)(tok0 + qi0 + j) * out_stride + (long)head_at(hh) * HS + 4 * qd;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      bf16x4 r;
      if (RULE && rule.gate) {
        const bf16x4 z = *(const bf16x4*)((const bf16_t*)rule.gate + (long)(tok0 + qi0 + j) * rule.gate_ld +
                                          (long)head_at(hh) * HS + 4 * qd + dt * 16);
#pragma unroll
        for (int v = 0; v < 4; ++v) o[hh][dt][v] *= gl3_sigmoid_fast((float)z[v]);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) r[v] = static_cast<bf16_t>(o[hh][dt][v] * inv);
      *(bf16x4*)(op + dt * 16) = r;
    }
  }
}

// The same attention with 32 queries of one head to a wave (128 to a block) on the 32x32x16 instruction, for
// steps that bring enough queries to fill such blocks: a wave reads the chunk's keys and values out
// of shared memory once for twice as many queries, and a block brings a chunk from the cache once
// for twice as many, which is what bounds the kernel above. Tiles as there, transposed:
//   S^T[key, query]  = K[key, :] . Q[query, :]^T     one 32 x 32 tile per chunk of 32 keys
//   O^T[dim, query] += V^T[dim, key] . P^T[key, query]
// A lane holds, of the score tile, query lane % 32 and the rows 8a + 4h + b (h = lane / 32, register
// 4a + b); row r of the tile is made key 16*(a/2) + 8h + 4*(a%2) + b of the chunk by the order in
// which the key rows are read, so that registers 0..7 hold the keys 8h..8h+7 of the chunk's first
// half and registers 8..15 those of its second half: the order in which the second product takes
// its 16 keys a step.
typedef float f32x16 __attribute__((ext_vector_type(16)));

// SPLIT: the chunks of a block's keys are shared out over `splits` blocks; each leaves its sums as they are, with their
// maximum and weight, for attention_prefill_merge_kernel.
#define PF_SPLITS 8      // at most
struct PfSplit {
  int splits;
  int n_tokens;
  float* o;      // [split][token][head][head_dim]
  float* ml;     // [split][token][head][2]: maximum in units of log2, sum
};
template <int HS, int CK, int AHEAD, int OCC, bool BIAS = false, bool RULE = false, bool SPLIT = false>
__global__ __launch_bounds__(256, OCC) void attention_prefill_wide_kernel(
    const bf16_t* __restrict__ q, long q_stride, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
    const int* __restrict__ cu_seqlens, const int* __restrict__ kv_before, const int* __restrict__ block_table,
    const int* __restrict__ seq_rows, int table_stride, bf16_t* __restrict__ out, long out_stride, int n_heads, int n_kv, int page_size, int window,
    float scale, int q_blocks, const float* __restrict__ slopes, int has_sink, float sink, int keep_first, int mask_chunk, int maps,
    const float* __restrict__ sinks, Gl3ScoreRule rule, PfSplit sp) {
  constexpr int KS = HS / 16;             // steps of the score product
  constexpr int DT = HS / 32;             // tiles of 32 dims of the output
  constexpr int NT = CK / 32;             // score tiles of a chunk of CK keys
  constexpr int KROW = HS + 8;
  constexpr int VROW = CK + 8;
  constexpr int VU = CK / 8;              // 16-byte units of a row of the transposed value chunk
  constexpr int UNITS = HS * CK / 8;      // 16-byte units of a chunk of keys (and of values)
  constexpr int NU = (UNITS + 255) / 256;
  constexpr int QB = 128;                 // queries of a block
  __shared__ __attribute__((aligned(16))) bf16_t ks[2][CK][KROW];
  __shared__ __attribute__((aligned(16))) bf16_t vs[2][HS][VROW];
  const int g = n_heads / n_kv;
  const int qb = q_blocks - 1 - blockIdx.z;      // the longest query blocks of all heads and sequences first
  const int b = blockIdx.y;
  const int head = SPLIT ? blockIdx.x % n_heads : blockIdx.x;                 // one query head to a block
  const int c = maps > 1 ? ((head / maps) / g) * maps + head % maps : head / g;      // (its key head: map head % maps of its group)
  const int n_v = n_kv / maps, cv = c / maps;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int n = lane & 31, h = lane >> 5;
  const int tok0 = __builtin_amdgcn_readfirstlane(cu_seqlens[b]);
  const int q_len = __builtin_amdgcn_readfirstlane(cu_seqlens[b + 1]) - tok0;
  if (qb * QB >= q_len) return;            // the whole block: no barrier has been passed yet
  const int before = __builtin_amdgcn_readfirstlane(kv_before[b]);
  // the sequence's row of the table: its number in the batch, or what `seq_rows` says (a table with a row per cache slot)
  const int* bt = block_table + (long)(seq_rows ? __builtin_amdgcn_readfirstlane(seq_rows[b]) : b) * table_stride;
  const int blk_first = before + qb * QB, blk_last = before + min(qb * QB + QB - 1, q_len - 1);
  // the first key that position p sees: its chunk's first (a chunked mask), the window's, or the sequence's
  auto low_of = [&](int p) { return mask_chunk > 0 ? p - p % mask_chunk : (window > 0 && p + 1 > window) ? p + 1 - window : 0; };
  const int blk_lo = low_of(blk_first);
  // (kept first keys: as in the kernel above, their chunks before the window's first chunk are numbered in front of it)
  const int ckw = blk_lo / CK;
  int ck1 = blk_last / CK, ck0 = ckw - (BIAS ? min((keep_first + CK - 1) / CK, ckw) : 0);
  const int split = SPLIT ? blockIdx.x / n_heads : 0;
  if (SPLIT) {
    const int chunks = ck1 - ck0 + 1, lo = ck0;
    ck0 = lo + chunks * split / sp.splits;
    ck1 = lo + chunks * (split + 1) / sp.splits - 1;      // (no chunk: the block leaves a weight of nothing)
  }
  auto real = [&](int ck) { return (BIAS && ck < ckw) ? ck - ck0 : ck; };
  const int qi0 = qb * QB + wave * 32;
  const bool active = qi0 < q_len;
  const bool q_ok = qi0 + n < q_len;
  const int p_mine = before + qi0 + n;
  const int p_last = before + min(qi0 + 31, q_len - 1);
  const int p_first = before + qi0;
  const int lo_first = low_of(p_first);
  const int lo_last = low_of(p_last);
  const int lo_mine = low_of(p_mine);
  const int ck_first = active ? lo_first / CK : 1, ck_last = active ? p_last / CK : 0;

  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8 qt[KS];
#pragma unroll
  for (int kk = 0; kk < KS; ++kk)
    qt[kk] = q_ok ? *(const bf16x8*)(q + (long)(tok0 + qi0 + n) * q_stride + (long)head * HS + kk * 16 + 8 * h) : zero8;

  float m_run = -INFINITY, l_run = 0.f;
  if (BIAS && (has_sink || sinks)) {            // (two lanes share a query's row sum: the sink's 1 once)
    m_run = (sinks ? sinks[head] : sink) * 1.4426950408889634f;
    l_run = h == 0 ? 1.f : 0.f;
  }
  const float sl = (BIAS && slopes) ? slopes[head] * (RULE ? 1.4426950408889634f : 1.0f / scale) : 0.f;
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[dt][v] = 0.f;

  bf16x8 rk[AHEAD][NU], rv[AHEAD][NU];
  auto fetch = [&](int ck, bf16x8 (&fk)[NU], bf16x8 (&fv)[NU]) {
    const int key0 = ck * CK;
    const long page = __builtin_amdgcn_readfirstlane(bt[key0 / page_size]);
    const int po = key0 % page_size;
    // (inside a page both lie in tiles, gl3_k_offset and gl3_v_offset: the chunk's keys are still
    // CK * HS consecutive elements, its values CK * 16 consecutive elements for every 16 dims)
    const bf16_t* kb = k_cache + ((page * n_kv + c) * page_size + po) * HS;
    const bf16_t* vb = v_cache + (page * n_v + cv) * (long)page_size * HS + (long)(po / 8) * 128;
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + 256 * i;
      if (UNITS % 256 == 0 || u < UNITS) {
        fk[i] = *(const bf16x8*)(kb + u * 8);
        fv[i] = *(const bf16x8*)(vb + (long)(u / (2 * CK)) * page_size * 16 + (u % (2 * CK)) * 8);
      }
    }
  };
  auto stage = [&](int buf, const bf16x8 (&fk)[NU], const bf16x8 (&fv)[NU]) {
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = tid + 256 * i;
      if (UNITS % 256 == 0 || u < UNITS) {
        // unit u of the keys: 32 keys u / (4 HS), of their two tiles (u / (2 HS)) % 2, column block
        // (u / 16) % (HS / 8), row u % 16
        const int row = u & 15, tile = (u / (2 * HS)) & 1, group = u / (4 * HS);
        *(bf16x8*)&ks[buf][32 * group + 8 * (row >> 2) + 4 * tile + (row & 3)][((u >> 4) % (HS / 8)) * 8] = fk[i];
        // unit u of the values: 16 dims u / (2 CK), positions 8 * ((u % (2 CK)) / 16) .., dim u % 16 of the 16
        *(bf16x8*)&vs[buf][(u / (2 * CK)) * 16 + (u & 15)][((u % (2 * CK)) >> 4) * 8] = fv[i];
      }
    }
  };

  const float c2 = RULE ? 1.0f : scale * 1.4426950408889634f;   // scores in units of log2
  const float q_scale = RULE ? scale * gl3_query_temperature(p_mine, rule) : 0.f;
  const float cap2 = RULE ? rule.softcap * 1.4426950408889634f : 0.f;      // the cap in units of log2
  const float rule_in = !RULE ? 0.f : cap2 > 0.f ? 2.8853900817779268f * q_scale / rule.softcap : q_scale * 1.4426950408889634f;
  // which key of a chunk is row n of the score tile
  const int krow = 16 * (n >> 4) + 8 * ((n >> 2) & 1) + 4 * ((n >> 3) & 1) + (n & 3);

  // One chunk: scores, running softmax, weighted values. The operands are read from shared memory
  // where they are used, no more than four ahead of their products (the scheduler would read them
  // all first, and they do not fit into the registers beside the sums). MASKED: some query of the
  // wave does not see some key of the chunk (the diagonal, a window's edge).
  auto chunk = [&](int buf, int key0, bool masked) {
    f32x16 s[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) s[t][v] = 0.f;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {      // the tiles' sums do not depend on each other: the matrix cores stay busy
        const bf16x8 a = *(const bf16x8*)&ks[buf][32 * t + krow][kk * 16 + 8 * h];
        s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, qt[kk], s[t], 0, 0, 0);
      }
      if (kk % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    if (RULE) {                                 // (as in the kernel above)
      const float base = (cap2 > 0.f ? cap2 : 0.f) - sl * (float)(p_mine - key0 - 8 * h);
      if (cap2 > 0.f) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            s[t][v] = fmaf(-2.0f * cap2, gl3_tanh_part(s[t][v] * rule_in), fmaf(sl, (float)(32 * t + 16 * (v >> 3) + (v & 7)), base));
      } else {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            s[t][v] = fmaf(s[t][v], rule_in, fmaf(sl, (float)(32 * t + 16 * (v >> 3) + (v & 7)), base));
      }
    } else if (BIAS) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int key = key0 + 32 * t + 16 * (v >> 3) + 8 * h + (v & 7);
          s[t][v] = fmaf(-sl, (float)(p_mine - key), s[t][v]);
        }
    }
    if (masked) {                               // (the same for the whole wave: a branch around the tests, one body)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int key = key0 + 32 * t + 16 * (v >> 3) + 8 * h + (v & 7);
          s[t][v] = ((key >= lo_mine || (BIAS && key < keep_first)) && key <= p_mine) ? s[t][v] : -INFINITY;
        }
    }
    float mx = s[0][0];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) mx = fmaxf(mx, s[t][v]);
    {   // the other half of the keys of this query sits 32 lanes away
      auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    }
    mx *= c2;                                   // c2 > 0: the greatest score stays the greatest
    const float m_new = fmaxf(m_run, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
    float ps = 0.f;
    bf16x8 pb[NT][2];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float p = __builtin_amdgcn_exp2f(fmaf(s[t][e], c2, -m_use));
        ps += p;
        pb[t][e >> 3][e & 7] = static_cast<bf16_t>(p);
      }
    l_run = l_run * alpha + ps;
    m_run = m_new;
    if (!__all(alpha == 1.0f)) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const bf16x8 v0 = *(const bf16x8*)&vs[buf][dt * 32 + n][32 * t + 8 * h];
        const bf16x8 v1 = *(const bf16x8*)&vs[buf][dt * 32 + n][32 * t + 16 + 8 * h];
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v0, pb[t][0], o[dt], 0, 0, 0);
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v1, pb[t][1], o[dt], 0, 0, 0);
        if (dt % 2 == 1) __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

#pragma unroll
  for (int r = 0; r < AHEAD; ++r) fetch(real(SPLIT ? max(ck0, min(ck0 + r, ck1)) : min(ck0 + r, ck1)), rk[r], rv[r]);
  stage(0, rk[0], rv[0]);
  __syncthreads();
  int buf = 0;
  for (int base = ck0; base <= ck1; base += AHEAD) {
#pragma unroll
    for (int r = 0; r < AHEAD; ++r) {
      const int ck = base + r;
      if (ck > ck1) break;
      const int key0 = real(ck) * CK;
      // the registers of this chunk are free (it lies in shared memory): ask for the chunk AHEAD further;
      // unconditional (the last chunk again at the end): a branch around the loads makes the compiler
      // wait for all of them at once
      fetch(real(min(ck + AHEAD, ck1)), rk[r], rv[r]);
      if (active && (ck >= ck_first || (BIAS && key0 < keep_first)) && ck <= ck_last) {
        // every query of the wave sees the whole chunk: no mask (the same for the whole wave)
        chunk(buf, key0, (BIAS && ck < ckw) || !(key0 + CK - 1 <= p_first && key0 >= lo_last));
      }
      if (ck < ck1) stage(buf ^ 1, rk[(r + 1) % AHEAD], rv[(r + 1) % AHEAD]);
      __syncthreads();
      buf ^= 1;
    }
  }

  float l = l_run;
  l += __shfl_xor(l, 32, 64);
  if (!q_ok) return;
  if (SPLIT) {
    const long row = ((long)split * sp.n_tokens + tok0 + qi0 + n) * n_heads + head;
    float* po = sp.o + row * HS + 4 * h;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int a = 0; a < 4; ++a) *(f32x4*)(po + dt * 32 + 8 * a) = f32x4{o[dt][4 * a], o[dt][4 * a + 1], o[dt][4 * a + 2], o[dt][4 * a + 3]};
    if (h == 0) {
      sp.ml[row * 2] = m_run;
      sp.ml[row * 2 + 1] = l;
    }
    return;
  }
  const float inv = 1.0f / l;
  bf16_t* op = out + (long)(tok0 + qi0 + n) * out_stride + (long)head * HS + 4 * h;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      bf16x4 r;
      if (RULE && rule.gate) {
        const bf16x4 z = *(const bf16x4*)((const bf16_t*)rule.gate + (long)(tok0 + qi0 + n) * rule.gate_ld +
                                          (long)head * HS + 4 * h + dt * 32 + 8 * a);
#pragma unroll
        for (int v = 0; v < 4; ++v) o[dt][4 * a + v] *= gl3_sigmoid_fast((float)z[v]);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) r[v] = static_cast<bf16_t>(o[dt][4 * a + v] * inv);
      *(bf16x4*)(op + dt * 32 + 8 * a) = r;
    }
}

// Every earlier key (no window, no bias), heads of 128, pages of whole chunks of 64 keys: eight waves in two groups that take turns.
//
// In the kernel above a wave's matrix instructions (1,024 cycles a chunk of 64 keys and 32 queries) and its softmax (some 900) add up
// although two waves share a SIMD: they come to want the same unit at the same time. Here a barrier ends every turn, and in a turn one
// group has the matrix cores while the other works out its softmax; wave w and wave w + 4, of different groups, share a
// SIMD. A wave's two turns for chunk i:
//   matrix turn i:  scores of chunk i, then the values of chunk i - 1 with its weights
//   vector turn i:  weights of chunk i, the output brought to the new maximum, the first keys of chunk i + 1 read ahead
// The sums are those of the kernel above (chunks of 32 keys there), the same bits: each half of a chunk has its own running maximum
// around which its weights are rounded, the output is brought to the second half's between the values of the two (rarely: only where
// that maximum moved), weights are added up in the order of the keys, and a half that none of a wave's queries sees is left out. One maximum
// for a whole chunk was 2 to 3% faster and its error against 64 bits up to 1.006 times as large.
// Group 0 has matrix turn i in turn 2 i, group 1 in turn 2 i + 1. What bounds it now: the vector instructions of both waves together with
// the matrix instructions (16,384 tokens: vector units busy 61% of the time, matrix cores 58%). With heads of 64, whose matrix part is half as long, such a loop was no faster than the kernel above
// (8,192 tokens 345 and 341 us) and is not built.
// 32 heads, one sequence, the kernel above and this one: 2,048 tokens 75 -> 61 us, 4,096 172 -> 143, 8,192 608 -> 520, 16,384 2,325 -> 1,956
// (1.12 PFLOP/s). Nor has it splits: one block a CU, so that as many splits as the kernel above has are two rounds of the chip (512 tokens
// behind 4,000, 24 heads, 6 splits 68 against 64 us), and fewer splits are longer sums.
//
// HEADS = 2: a block is 128 queries of two heads of one kv head, a group of waves to a head; HEADS = 1: 256 queries of one head.
//
// Keys and values go from memory straight into shared memory, as they lie in the cache (gl3_k_offset and gl3_v_offset are the
// operands' order: sixteen lanes read 256 consecutive bytes), four chunks in turn. In matrix turn i a wave asks for its share of the
// values of chunk i + 2 and of the keys of chunk i + 3; both places were read last in group 1's matrix turn i - 1, a turn that has
// ended (matrix instructions took what was read before its barrier). Keys of chunk i + 1 are read from turn 2 i + 1 on and values of
// chunk i from turn 2 i + 2 on: the wait in front of the barrier that ends turn 2 i leaves out only what was asked for after
// them, two requests of group 0 and one of group 1. Chunks beyond the last repeat it, so that the counts hold; nothing is in flight
// when a block ends.
//
// Score tile: rows 0..15 are the cache's first tile of 32 keys, rows 16..31 the second, so that register 4 a + b of lane (n, h)
// is key 16 (a % 2) + 8 h + 4 (a / 2) + b: eight consecutive keys of each half, as the second product takes them.
template <int HEADS>
__global__ __launch_bounds__(512, 2) void attention_prefill_turns_kernel(
    const bf16_t* __restrict__ q, long q_stride, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
    const int* __restrict__ cu_seqlens, const int* __restrict__ kv_before, const int* __restrict__ block_table,
    const int* __restrict__ seq_rows, int table_stride, bf16_t* __restrict__ out, long out_stride, int n_heads, int n_kv, int page_size,
    float scale, int q_blocks, int n_seqs) {
  constexpr int HS = 128, CK = 64, KS = HS / 16, DT = HS / 32, QB = 256 / HEADS;
  constexpr int KB = CK * HS * 2;                  // bytes of a chunk's keys (and of its values)
  constexpr int STAGE = 2 * KB, STAGES = 4, AHEAD = STAGES - 1;
  constexpr int PW = KB / 8192;                    // pieces of 1 KB of either that a wave brings
  constexpr int NK = 2 * KS, NV = 4 * DT;          // matrix instructions of a chunk: scores, values
  constexpr int RING = 9;                          // operands from shared memory: the next eight, and the one in use
  __shared__ __attribute__((aligned(1024))) char lds[STAGES * STAGE];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  // the y-th query block of all sequences, those behind the most queries first (a grid over sequences and blocks would start blocks
  // that have no query, each on a CU of its own: this kernel's shared memory leaves no room beside another block)
  int b = 0, qb = q_blocks - 1 - blockIdx.y;
  if (n_seqs > 1) {
    const int blocks = lane < n_seqs ? (cu_seqlens[lane + 1] - cu_seqlens[lane] + QB - 1) / QB : 0;
    int left = blockIdx.y;
    unsigned long here = 0;
    qb = q_blocks;
    while (qb > 0) {
      here = __ballot(blocks > --qb);
      const int count = __builtin_popcountl(here);
      if (left < count) break;
      left -= count;
      here = 0;
    }
    if (here == 0) return;                         // the whole block: no barrier has been passed yet
    for (; left > 0; --left) here &= here - 1;
    b = __builtin_ctzl(here);
  }
  const int g = n_heads / n_kv, at = blockIdx.x;
  const int c = at % n_kv;                         // (blocks of one kv head are n_kv apart: on one XCD where n_kv is 8)
  const int group = wave >> 2;
  const int head = c * g + at / n_kv * HEADS + (HEADS == 2 ? group : 0);
  const int n = lane & 31, h = lane >> 5;
  const int tok0 = __builtin_amdgcn_readfirstlane(cu_seqlens[b]);
  const int q_len = __builtin_amdgcn_readfirstlane(cu_seqlens[b + 1]) - tok0;
  if (qb * QB >= q_len) return;                    // (and so here)
  const int before = __builtin_amdgcn_readfirstlane(kv_before[b]);
  const int* bt = block_table + (long)(seq_rows ? __builtin_amdgcn_readfirstlane(seq_rows[b]) : b) * table_stride;
  const int blk_last = before + min(qb * QB + QB - 1, q_len - 1);
  const int ck1 = blk_last / CK, chunks = ck1 + 1;
  const int qi0 = qb * QB + (HEADS == 2 ? (wave & 3) * 32 : wave * 32);
  const bool active = qi0 < q_len;
  const bool q_ok = qi0 + n < q_len;
  const int p_mine = before + qi0 + n;
  const int p_last = before + min(qi0 + 31, q_len - 1), p_first = before + qi0;
  // the wave's chunks: later ones hold no key that one of its queries sees, nor does the last one's second half if its queries end in
  // the first
  const int my_last = active ? p_last / CK : -1;
  const bool half = (p_last & 32) == 0;

  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8 qt[KS];
#pragma unroll
  for (int kk = 0; kk < KS; ++kk)
    qt[kk] = q_ok ? *(const bf16x8*)(q + (long)(tok0 + qi0 + n) * q_stride + (long)head * HS + kk * 16 + 8 * h) : zero8;
  // alpha, beta: what the sums so far are multiplied with in front of the last chunk's first and second half
  float m_run = -INFINITY, l_run = 0.f, alpha = 1.f, beta = 1.f;
  bool moved = false;              // (some query's maximum in the second half)
  f32x16 o[DT], s[2], w[2];      // (w: the weights of the last chunk, in the order of its keys)
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[dt][v] = 0.f;
  bf16x8 pb[2][2], f[RING];        // weights as the second product takes them; operands from shared memory

  // where chunks lie, sixty-four of them in a register (a lane one): keys in units of a chunk, values in units of 1,024 elements
  const int per_page = page_size / CK, v_units = per_page * (HS / 16);
  auto places = [&](int first, int& k_at, int& v_at) {
    const int ck = min(first + lane, ck1), entry = ck / per_page, in_page = ck - entry * per_page;
    const int row = bt[entry] * n_kv + c;
    k_at = row * per_page + in_page;
    v_at = row * v_units + in_page;
  };
  int k_at, v_at, k_later, v_later;
  places(0, k_at, v_at);
  places(64, k_later, v_later);
  const unsigned lds0 = (unsigned)(unsigned long)(__attribute__((address_space(3))) char*)lds + wave * (PW * 1024);
  unsigned k_off[PW], v_off[PW];
#pragma unroll
  for (int i = 0; i < PW; ++i) {
    const int piece = wave * PW + i;               // (of the values: half of sixteen dims' 64 positions)
    k_off[i] = piece * 1024 + lane * 16;
    v_off[i] = (piece >> 1) * (page_size * 32) + (piece & 1) * 1024 + lane * 16;
  }
  // chunks are asked for one after the other: values of chunk x, then keys of chunk x + 1
  i32x4 k_buf, v_buf;
  auto locate = [&](int x) {                       // where chunk x lies; the keys' place is used first
    v_buf = mf_rsrc(v_cache + (long)__builtin_amdgcn_readlane(v_at, (x - 1) & 63) * 1024);
    if (x && (x & 63) == 0) {
      k_at = k_later;
      v_at = v_later;
      places(x + 64, k_later, v_later);
    }
    k_buf = mf_rsrc(k_cache + (long)__builtin_amdgcn_readlane(k_at, x & 63) * (CK * HS));
  };
  auto load_v = [&](int x) {
#pragma unroll
    for (int i = 0; i < PW; ++i) mf_dma16(lds0 + (x % STAGES) * STAGE + KB + i * 1024, v_off[i], v_buf, 0);
  };
  auto load_k = [&](int x) {
#pragma unroll
    for (int i = 0; i < PW; ++i) mf_dma16(lds0 + (x % STAGES) * STAGE + i * 1024, k_off[i], k_buf, 0);
  };

  const char* k_lds = lds + (n >> 4) * (32 * HS) + h * 256 + (n & 15) * 16;
  const char* v_lds = lds + KB + (n >> 4) * 2048 + h * 256 + (n & 15) * 16;
  auto read_k = [&](int x, int m) {                // operand m of the scores: k-step m / 2 of tile m % 2
    f[m % RING] = *(const bf16x8*)(k_lds + (x % STAGES) * STAGE + (m & 1) * (64 * HS) + (m >> 1) * 512);
  };
  auto read_v = [&](int x, int m, int to) {        // operand m of the values: sixteen keys m / DT, dims 32 (m % DT) ..
    f[to % RING] = *(const bf16x8*)(v_lds + (x % STAGES) * STAGE + (m % DT) * 4096 + (m / DT) * 512);
  };
  // What of the softmax does not need a chunk's scores all at once is done beside the matrix instructions, a few instructions behind
  // each (it occupies the matrix core for 32 cycles, the wave's issue for 4): the output brought to the new maximum and
  // the weights rounded beside the scores of the next chunk, the weights added up beside the values; so are the reads of operands
  // and the requests for later chunks, which cost 300 cycles a turn in front of them.
  auto matrix_turn = [&](int i, auto with_scores, auto with_values) {
    constexpr bool QK = decltype(with_scores)::value, PV = decltype(with_values)::value;
    constexpr int K_COUNT = QK ? NK : 0, COUNT = K_COUNT + (PV ? NV : 0), BEFORE = QK ? NK : 1;
    static_assert(NV == 16, "beside an instruction of the values a weight of either half");
    f32x16 zero;
    float sum[2];
#pragma unroll
    for (int v = 0; v < 16; ++v) zero[v] = 0.f;
    auto prepare = [&](int m) {                    // (the m-th of BEFORE parts)
#pragma unroll
      for (int e = m * (32 / BEFORE); e < (m + 1) * (32 / BEFORE); ++e) pb[e >> 4][(e >> 3) & 1][e & 7] = static_cast<bf16_t>(w[e >> 4][e & 15]);
    };
    if (!QK) {
#pragma unroll
      for (int m = 0; m < 8; ++m) read_v(i + STAGES - 1, m, m);
      prepare(0);
    }
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int m = 0; m < COUNT; ++m) {
      const int at = m - K_COUNT;
      if (PV && at == NV / 2) {                    // the second half's values: its maximum may be another
        if (!QK && half) break;
        if (moved) {
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) o[dt] *= beta;
        }
      }
      if (m < K_COUNT) s[m & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[m % RING], qt[m >> 1], m < 2 ? zero : s[m & 1], 0, 0, 0);
      else o[at % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[m % RING], pb[at / DT >> 1][at / DT & 1], o[at % DT], 0, 0, 0);
      if (m + 8 < K_COUNT) read_k(i, m + 8);
      else if (m + 8 < COUNT) read_v(i + STAGES - 1, m + 8 - K_COUNT, m + 8);
      if (m == 1) load_v(i + AHEAD - 1);
      if (m == 3) load_k(i + AHEAD);
      if (PV && m < K_COUNT) prepare(m);
      if (m >= K_COUNT && QK) {
#pragma unroll
        for (int t = 0; t < 2; ++t) sum[t] = at == 0 ? w[t][0] : sum[t] + w[t][at];
        if (at) asm volatile("" : "+v"(sum[0]), "+v"(sum[1]));      // (here, not at the end)
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
    if (PV) {
      if (!QK) {
#pragma unroll
        for (int e = 0; e < 16; ++e)
#pragma unroll
          for (int t = 0; t < 2; ++t) sum[t] = e == 0 ? w[t][0] : sum[t] + w[t][e];
      }
      l_run = l_run * alpha + sum[0];
      l_run = l_run * beta + sum[1];
    }
  };

  const float c2 = scale * 1.4426950408889634f;    // scores in units of log2
  auto max3 = [](float a, float b, float c) { return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c); };
  auto vector_turn = [&](int key0, bool masked) {
    // (register of the lane's e-th key of a tile, in the order of the keys; its key)
    auto reg = [](int e) { return (e & 3) + ((e >> 2) & 1) * 8 + (e >> 3) * 4; };
    if (masked) {                                  // (the same for the whole wave: a branch around the tests, one body)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int key = key0 + 32 * t + 16 * (e >> 3) + 8 * h + (e & 7);
          s[t][reg(e)] = key <= p_mine ? s[t][reg(e)] : -INFINITY;
        }
    }
    // (two chains a half: one would wait for itself, with no other wave of the SIMD at its softmax. v_maximum3, which keeps NaNs: fmaxf of
    // a matrix instruction's results costs one more for each pair to quieten them. A row with a NaN is NaN by its weights either way)
    float top[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float u[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        u[k] = max3(s[t][8 * k], s[t][8 * k + 1], s[t][8 * k + 2]);
        u[k] = max3(u[k], s[t][8 * k + 3], s[t][8 * k + 4]);
        u[k] = max3(u[k], s[t][8 * k + 5], s[t][8 * k + 6]);
      }
      top[t] = max3(max3(u[0], u[1], s[t][7]), s[t][15], s[t][15]);
    }
    {   // the other half of the keys of this query sits 32 lanes away: the greatest of either half of the chunk
      auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(top[0]), __float_as_uint(top[1]), false, false);
      const float mx = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])) * c2;      // c2 > 0: the greatest score stays the greatest
      r = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      top[0] = __uint_as_float(r[0]);
      top[1] = __uint_as_float(r[1]);
    }
    const float m_mid = fmaxf(m_run, top[0]), m_new = fmaxf(m_mid, top[1]);
    const float use_mid = m_mid == -INFINITY ? 0.f : m_mid, use_new = m_new == -INFINITY ? 0.f : m_new;
    alpha = __builtin_amdgcn_exp2f(m_run - use_mid);
    beta = __builtin_amdgcn_exp2f(m_mid - use_new);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) w[t][e] = __builtin_amdgcn_exp2f(fmaf(s[t][reg(e)], c2, t ? -use_new : -use_mid));
    m_run = m_new;
    moved = !__all(beta == 1.0f);
    if (!__all(alpha == 1.0f)) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
    }
    // (the compiler would work the weights out where the next turn first takes them, behind the barrier)
    asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(alpha), "+v"(beta), "+v"(m_run));
  };

#pragma unroll
  for (int x = 0; x < AHEAD; ++x) {
    locate(x);
    if (x) load_v(x - 1);
    load_k(x);
  }
  locate(AHEAD);
  mf_wait_loads<(2 * AHEAD - 2) * PW>();
  mf_barrier();
  // the end of a matrix turn (an even one of group 0) and of a vector turn (an even one of group 1)
  auto end_matrix = [&]() {
    if (group == 0) mf_wait_loads<(2 * AHEAD - 2) * PW>();
    mf_barrier();
  };
  auto end_vector = [&]() {
    if (group == 1) mf_wait_loads<(2 * AHEAD - 4) * PW>();
    mf_barrier();
  };
  if (group == 1) end_vector();                    // the second group runs a turn behind
  int i = 0;
  if (my_last >= 0) {                              // (one body for all chunks: where bodies meet the compiler copies the sums)
#pragma unroll
    for (int m = 0; m < 8; ++m) read_k(i, m);
    matrix_turn(i, std::true_type{}, std::false_type{});
    for (;;) {
      end_matrix();
      locate(i + 1 + AHEAD);
#pragma unroll
      for (int m = 0; m < 8; ++m) read_k(i + 1, m);
      const int key0 = i * CK;
      vector_turn(key0, key0 + CK - 1 > p_first);
      end_vector();
      if (++i > my_last) break;
      matrix_turn(i, std::true_type{}, std::true_type{});
    }
    matrix_turn(i, std::false_type{}, std::true_type{});
  } else {                                         // (none of the block's rows: its share of the loads, and the barriers)
    load_v(AHEAD - 1);
    load_k(AHEAD);
  }
  for (; i < chunks; ++i) {
    end_matrix();
    locate(i + 1 + AHEAD);
    end_vector();
    load_v(i + AHEAD);
    load_k(i + 1 + AHEAD);
  }
  if (group == 0) mf_barrier();
  mf_wait_loads<0>();

  float l = l_run;
  l += __shfl_xor(l, 32, 64);
  if (!q_ok) return;
  const float inv = 1.0f / l;
  bf16_t* op = out + (long)(tok0 + qi0 + n) * out_stride + (long)head * HS + 4 * h;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      bf16x4 r;
#pragma unroll
      for (int v = 0; v < 4; ++v) r[v] = static_cast<bf16_t>(o[dt][4 * a + v] * inv);
      *(bf16x4*)(op + dt * 32 + 8 * a) = r;
    }
}

// Every earlier key, heads of 64 or 128, pages of whole chunks of 64 keys: eight waves a block.
//
// The kernel of 128 queries above carries keys and values through registers into shared memory, and a block walks its keys alone. Here chunks go
// from memory straight into shared memory, as they lie in the cache (the operands' order, as in the kernel of turns).
// GROUPS = 2, for few blocks: 128 queries of one head, four waves of 32 on the even chunks of keys and four on the odd ones, whose sums are
// brought together at the end: a block's way along the keys is half as long. GROUPS = 1: 128 queries of two heads of one kv head, which
// share the chunks: the same sums in the same order as the kernel of 128 queries, bit for bit. Two groups' error against 64 bits is 0.983 to 0.998 times
// that of the kernels beside it at 9 sizes of 333 to 2,048 tokens with scores spread 0.3 to 3, heads of 64 and of 128, the average of 16 sets of inputs each, none of which
// is larger (`profiles/prefill_eight_error.txt`): their maxima are nearer to the weights. (With one maximum for 64 keys heads of 128 took 8 to 15% less time, at up to
// 1.004 times the error.) A value that is not finite spoils the queries that share its 64 keys (heads of 128: 32), as in that kernel.
// Heads of 64: 115 registers where the kernel of 128 queries has 157, so that four waves share a SIMD and while some have its matrix cores others
// work out their softmax (a SIMD has one vector instruction of a wave about every eight cycles, of four waves one every 4.2, an
// exponential 8.2, an addition 2.4); two blocks a CU. Heads of 128: 164, two waves a SIMD and a block a CU.
// What bounds it: one sequence of 16,384 tokens the power (vector and matrix units together; the clock falls below 1.9 GHz), a prompt of
// 2,048 the unequal ways of its blocks, few blocks a wave's chain of scores, softmax and values. Time of the kernel taken before and of this one:
//   32 heads of 64 over 8, one sequence: 1,024 tokens 22.2 -> 15.6 us, 2,048 41.6 -> 29.5, 4,096 97.9 -> 89.1, 8,192 346 -> 308, 16,384 1,313 -> 1,177;
//     317 + 1,203 + 701 tokens 27.5 -> 19.8, 64 of 83 29.4 -> 19.3
//   24 heads of 128 over 8: 512 tokens 17.5 -> 16.1, 1,024 31.1 -> 24.6, 2,048 62.0 -> 52.0; 512 behind 512 29.2 -> 24.3, 512 behind 4,096, unsplit, 112 -> 80
// Heads of 64 with two waves a SIMD and the softmax woven between the matrix instructions (241 registers) took 31.0 us for 2,048 tokens and 1,238 for 16,384, the same
// with 32 queries of two heads a wave 37.7 and 1,223.
//
// A round is a chunk a group; a wave brings a share of its group's chunk (of all, GROUPS = 1). STAGES chunks lie in shared memory in turn: behind
// the barrier of a round the place that was read in the round before is written for the round STAGES - 1 further on, and the wait in
// front of it leaves out the requests for later rounds than its own. Chunks beyond the last repeat it, so that the counts hold; nothing is in
// flight when the sums go through shared memory, or when a block ends.
// SPLIT: as in the kernel of 128 queries.
template <int HS, int GROUPS, bool SPLIT>
__global__ __launch_bounds__(512, HS == 64 ? 4 : 2) void attention_prefill_eight_kernel(
    const bf16_t* __restrict__ q, long q_stride, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
    const int* __restrict__ cu_seqlens, const int* __restrict__ kv_before, const int* __restrict__ block_table,
    const int* __restrict__ seq_rows, int table_stride, bf16_t* __restrict__ out, long out_stride, int n_heads, int n_kv, int page_size,
    float scale, int q_blocks, int folded, int n_seqs, PfSplit sp) {
  static_assert(!SPLIT || GROUPS == 2, "splits are for few blocks");
  constexpr int CK = 64, KS = HS / 16, DT = HS / 32, QB = 128, HEADS = GROUPS == 2 ? 1 : 2;
  constexpr int KB = CK * HS * 2;                  // bytes of a chunk's keys (and of its values)
  constexpr int STAGE = 2 * KB, STAGES = 4 / GROUPS;
  constexpr int PW = KB / 8192 * GROUPS;           // pieces of 1 KB of either that a wave brings
  __shared__ __attribute__((aligned(1024))) char lds[GROUPS * STAGES * STAGE];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, group = wave >> 2;
  // (as in the kernel of 128 queries the longest blocks first; where all blocks are on the chip at once the shortest second, beside them)
  const int half = q_blocks / 2, z = blockIdx.z;
  const int qb = folded && z >= q_blocks - half ? z - (q_blocks - half) : q_blocks - 1 - z;
  const int b = blockIdx.y, g = n_heads / n_kv;
  const int split = SPLIT ? blockIdx.x / n_heads : 0, at = blockIdx.x - split * n_heads;
  const int c = at % n_kv;                         // (blocks of one kv head are n_kv apart: on one XCD where n_kv is 8)
  const int head = c * g + at / n_kv * HEADS + (HEADS == 2 ? group : 0);
  const int n = lane & 31, h = lane >> 5;
  if (b >= n_seqs) return;                         // (a row of the grid that is no sequence's)
  const int tok0 = __builtin_amdgcn_readfirstlane(cu_seqlens[b]);
  const int q_len = __builtin_amdgcn_readfirstlane(cu_seqlens[b + 1]) - tok0;
  if (qb * QB >= q_len) return;                    // the whole block: no barrier has been passed yet
  const int before = __builtin_amdgcn_readfirstlane(kv_before[b]);
  const int* bt = block_table + (long)(seq_rows ? __builtin_amdgcn_readfirstlane(seq_rows[b]) : b) * table_stride;
  int ck0 = 0, ck1 = (before + min(qb * QB + QB - 1, q_len - 1)) / CK;
  if (SPLIT) {                                     // (no chunk: the block leaves a weight of nothing)
    const int chunks = ck1 + 1;
    ck0 = chunks * split / sp.splits;
    ck1 = chunks * (split + 1) / sp.splits - 1;
  }
  const int rounds = (ck1 - ck0 + GROUPS) / GROUPS;
  const int qi0 = qb * QB + (wave & 3) * 32;
  const bool q_ok = qi0 + n < q_len;
  const int p_mine = before + qi0 + n, p_first = before + qi0, p_last = before + min(qi0 + 31, q_len - 1);
  const int my_last = qi0 < q_len ? p_last / CK : -1;      // the last chunk with a key that one of the wave's queries sees

  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  bf16x8 qt[KS];
#pragma unroll
  for (int kk = 0; kk < KS; ++kk)
    qt[kk] = q_ok ? *(const bf16x8*)(q + (long)(tok0 + qi0 + n) * q_stride + (long)head * HS + kk * 16 + 8 * h) : zero8;
  float m_run = -INFINITY, l_run = 0.f;
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[dt][v] = 0.f;

  // where the group's chunks lie, sixty-four of them in a register (a lane one): keys in units of a chunk, values of 1,024 elements
  const int per_page = page_size / CK, v_units = per_page * (HS / 16);
  const int first_ck = ck0 + (GROUPS == 2 ? group : 0);
  auto places = [&](int first, int& k_at, int& v_at) {
    const int ck = max(0, min((first + lane) * GROUPS + first_ck, ck1)), entry = ck / per_page, in_page = ck - entry * per_page;
    const int row = bt[entry] * n_kv + c;
    k_at = row * per_page + in_page;
    v_at = row * v_units + in_page;
  };
  int k_at, v_at;
  places(0, k_at, v_at);
  const int piece0 = (GROUPS == 2 ? wave & 3 : wave) * PW;
  const int base = GROUPS == 2 ? group * STAGES * STAGE : 0;
  const unsigned lds0 = (unsigned)(unsigned long)(__attribute__((address_space(3))) char*)lds + base + piece0 * 1024;
  unsigned v_off[PW];
#pragma unroll
  for (int i = 0; i < PW; ++i) v_off[i] = ((piece0 + i) >> 1) * (page_size * 32) + ((piece0 + i) & 1) * 1024 + lane * 16;
  auto ask = [&](int x) {                          // the group's x-th chunk, one after the other; beyond the last the last again
    if (x && (x & 63) == 0) places(x, k_at, v_at);
    const i32x4 k_buf = mf_rsrc(k_cache + (long)__builtin_amdgcn_readlane(k_at, x & 63) * (CK * HS));
    const i32x4 v_buf = mf_rsrc(v_cache + (long)__builtin_amdgcn_readlane(v_at, x & 63) * 1024);
    const unsigned to = lds0 + (x % STAGES) * STAGE;
#pragma unroll
    for (int i = 0; i < PW; ++i) mf_dma16(to + i * 1024, (piece0 + i) * 1024 + lane * 16, k_buf, 0);
#pragma unroll
    for (int i = 0; i < PW; ++i) mf_dma16(to + KB + i * 1024, v_off[i], v_buf, 0);
  };

  const float c2 = scale * 1.4426950408889634f;    // scores in units of log2
  const char* k_lds = lds + base + (n >> 4) * (32 * HS) + h * 256 + (n & 15) * 16;
  const char* v_lds = lds + base + KB + (n >> 4) * 2048 + h * 256 + (n & 15) * 16;
  auto max3 = [](float a, float b, float c) { return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c); };
  // (register of the lane's e-th key of a tile, in the order of the keys: score tiles as in the kernel of turns)
  auto reg = [](int e) { return (e & 3) + ((e >> 2) & 1) * 8 + (e >> 3) * 4; };
  // The keys of a chunk around whose maximum weights are rounded together: those of a chunk of the kernel of 128 queries.
  constexpr int SUB = HS == 64 ? 64 : 32, NT = SUB / 32;
  auto part = [&](int at, int first, int key0, bool masked) {      // (`first`: the part's first tile of 32 keys)
    f32x16 s[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) s[t][v] = 0.f;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        s[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(k_lds + at + (first + t) * (64 * HS) + kk * 512), qt[kk], s[t], 0, 0, 0);
    if (masked) {                                  // (the same for the whole wave: a branch around the tests, one body)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) s[t][reg(e)] = key0 + 32 * t + 16 * (e >> 3) + 8 * h + (e & 7) <= p_mine ? s[t][reg(e)] : -INFINITY;
    }
    // (v_maximum3, which keeps NaNs: fmaxf of a matrix instruction's results costs one more for each pair to quieten them. A row with a NaN
    // is NaN by its weights either way)
    float top[2 * NT];
#pragma unroll
    for (int k = 0; k < 2 * NT; ++k) {
      const f32x16& v = s[k >> 1];
      const int r = (k & 1) * 8;
      top[k] = max3(max3(max3(v[r], v[r + 1], v[r + 2]), v[r + 3], v[r + 4]), v[r + 5], v[r + 6]);
    }
    float mx = max3(max3(top[0], top[1], s[0][7]), s[0][15], s[0][15]);
    if constexpr (NT == 2) mx = max3(mx, max3(top[2], top[3], s[1][7]), s[1][15]);
    {   // the other half of the keys of this query sits 32 lanes away
      auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
      mx = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    }
    mx *= c2;                                      // c2 > 0: the greatest score stays the greatest
    const float m_new = fmaxf(m_run, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
    float ps = 0.f;
    bf16x8 pb[NT][2];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float p = __builtin_amdgcn_exp2f(fmaf(s[t][reg(e)], c2, -m_use));
        ps += p;
        pb[t][e >> 3][e & 7] = static_cast<bf16_t>(p);
      }
    l_run = l_run * alpha + ps;
    m_run = m_new;
    if (!__all(alpha == 1.0f)) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
    }
#pragma unroll
    for (int j = 0; j < 2 * NT; ++j)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8*)(v_lds + at + dt * 4096 + (2 * first + j) * 512), pb[j >> 1][j & 1], o[dt], 0, 0, 0);
  };
  auto chunk = [&](int at, int key0) {
    part(at, 0, key0, key0 + SUB - 1 > p_first);
    if (SUB < CK && key0 + SUB <= p_last) part(at, 1, key0 + SUB, key0 + CK - 1 > p_first);      // (a half that none of the wave's queries sees is left out)
  };

#pragma unroll
  for (int x = 0; x < STAGES - 1; ++x) ask(x);
  for (int x = 0; x < rounds; ++x) {
    mf_wait_loads<(STAGES - 2) * 2 * PW>();        // this wave's share of chunk x has come, behind the barrier everybody's
    mf_barrier();
    ask(x + STAGES - 1);                           // (into the place that was read last before the barrier)
    const int ck = x * GROUPS + first_ck;
    if (ck <= (SPLIT ? min(my_last, ck1) : my_last)) chunk((x % STAGES) * STAGE, ck * CK);
  }
  mf_wait_loads<0>();

  float l = l_run;
  l += __shfl_xor(l, 32, 64);
  if constexpr (GROUPS == 2) {
    // the second group's sums go through shared memory to the first's waves, which bring both to the greater maximum
    mf_barrier();
    float* const theirs = (float*)lds + (wave & 3) * ((DT * 16 + 2) * 64) + lane;
    if (group == 1) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) theirs[(dt * 16 + v) * 64] = o[dt][v];
      theirs[DT * 16 * 64] = m_run;
      theirs[(DT * 16 + 1) * 64] = l;
    }
    __syncthreads();
    if (group == 1) return;
    const float m1 = theirs[DT * 16 * 64], l1 = theirs[(DT * 16 + 1) * 64];
    if (!(m1 == -INFINITY && l1 == 0.f)) {         // (a query that sees none of their keys; scores that are all NaN have a weight)
      const float m = fmaxf(m_run, m1), f0 = __builtin_amdgcn_exp2f(m_run - m), f1 = __builtin_amdgcn_exp2f(m1 - m);
      l = l * f0 + l1 * f1;
      m_run = m;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[dt][v] = o[dt][v] * f0 + theirs[(dt * 16 + v) * 64] * f1;
    }
  }
  if (!q_ok) return;
  if (SPLIT) {
    const long row = ((long)split * sp.n_tokens + tok0 + qi0 + n) * n_heads + head;
    float* po = sp.o + row * HS + 4 * h;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int a = 0; a < 4; ++a) *(f32x4*)(po + dt * 32 + 8 * a) = f32x4{o[dt][4 * a], o[dt][4 * a + 1], o[dt][4 * a + 2], o[dt][4 * a + 3]};
    if (h == 0) {
      sp.ml[row * 2] = m_run;
      sp.ml[row * 2 + 1] = l;
    }
    return;
  }
  const float inv = 1.0f / l;
  bf16_t* op = out + (long)(tok0 + qi0 + n) * out_stride + (long)head * HS + 4 * h;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      bf16x4 r;
#pragma unroll
      for (int v = 0; v < 4; ++v) r[v] = static_cast<bf16_t>(o[dt][4 * a + v] * inv);
      *(bf16x4*)(op + dt * 32 + 8 * a) = r;
    }
}

// The splits' sums of a row (token, head) brought to the greatest of their maxima, added in the order of the splits, and divided
// by the weight: a thread four dims of a row, its splits' loads all on their way at once.
template <int HS>
__global__ __launch_bounds__(256) void attention_prefill_merge_kernel(PfSplit sp, bf16_t* __restrict__ out, long out_stride, int n_heads) {
  constexpr int TPR = HS / 4;      // threads a row
  const long at = (long)blockIdx.x * 256 + threadIdx.x, rows = (long)sp.n_tokens * n_heads;
  const long row = at / TPR;
  const int d = (int)(at % TPR) * 4;
  if (row >= rows) return;
  f32x4 v[PF_SPLITS];
  float m[PF_SPLITS], l[PF_SPLITS], top = -INFINITY;
#pragma unroll
  for (int s = 0; s < PF_SPLITS; ++s) {
    const long r = min(s, sp.splits - 1) * rows + row;
    v[s] = *(const f32x4*)(sp.o + r * HS + d);
    m[s] = s < sp.splits ? sp.ml[r * 2] : -INFINITY;
    l[s] = s < sp.splits ? sp.ml[r * 2 + 1] : 0.f;
  }
#pragma unroll
  for (int s = 0; s < PF_SPLITS; ++s) top = fmaxf(top, m[s]);
  float weight = 0.f;
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < PF_SPLITS; ++s) {
    if (m[s] == -INFINITY && l[s] == 0.f) continue;      // (a split whose keys the row does not see; scores that are all NaN have a weight)
    const float f = __builtin_amdgcn_exp2f(m[s] - top);
    weight += f * l[s];
    sum += f * v[s];
  }
  bf16x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = static_cast<bf16_t>(sum[j] / weight);
  *(bf16x4*)(out + row / n_heads * out_stride + row % n_heads * HS + d) = o;
}

// Which of the two kernels a step takes, unless the caller says otherwise. Heads of 32 and 64: the one
// with 128 queries a block (chunks of 64 keys) from 33 tokens of the longest sequence on; it was the faster
// one at every length from there (192 tokens, 32 heads of 64: 7.4 against 9.8 us; 1,024: 23 against 33 us).
// Heads of 96 and 128: only where it has at least two blocks for every CU; below that the kernel of 64
// queries a block, with twice the blocks, is ahead (32 heads of 128, one sequence: 1,024 tokens 38 against
// 42 us, 1,536 tokens 59 against 65 us, 2,048 tokens 99 against 84 us).
static bool prefill_wide(int head_dim, int n_heads, int n_seqs, int max_q_len) {
  if (head_dim <= 64) return max_q_len > 32;
  return (long)n_heads * n_seqs * ((max_q_len + 127) / 128) >= 512;
}

// The kernel of turns: what it is built for, and where it is taken instead of the kernel of 128 queries a block (whose bits it gives),
// unless the caller says otherwise: from 1,024 tokens of the longest sequence on, where those are a fifth of the step's tokens at least
// or the sequences are long on average. Its blocks are longer to start (128 KB of shared memory are filled first) and a CU holds one: a
// long sequence is done sooner, many short ones later. Time against the kernel of 128 queries, 24 and 32 heads of 128, one sequence of 1,024 to 8,000 tokens
// beside 1 to 60 of 20 to 1,000 and random batches (profiles/prefill_turns_rule.txt): from a fifth on 0.59 to 1.03 (330
// sizes, 0.80 on average); below 0.98 to 1.25 (60 sizes, 1.08 on average; 1,300 tokens and sixty of 100 58 -> 68 us with 24 heads), but six or eight
// of 1,280 to 2,000 0.92 to 1.01. (What the sequences hold already is not known here: with sixty of 1 to 30 tokens behind 500 beside 1,300
// or 2,048 24 heads take 1.13 to 1.23 times as long, 32 heads 0.82 to 0.87; behind 4,000 0.89 to 0.99 and 0.58 to 0.64.)
#define PF_TURNS INT_MIN
static bool turns_takes(int head_dim, int page_size, int group, int n_seqs, int n_tokens) {
  return head_dim == 128 && page_size % 64 == 0 && (n_seqs == 1 || (n_seqs <= 64 && n_tokens > 0 && n_tokens / (group % 2 ? 256 : 128) + n_seqs <= 65535));
}
static bool turns_wanted(int n_seqs, int max_q_len, int n_tokens) {
  return max_q_len >= 1024 && (n_tokens <= 5L * max_q_len || n_tokens >= 1280L * n_seqs);
}

// The library's choice where it is not the kernel of eight waves (below): 0: 64 queries a block, 1: 128, 2: the kernel of turns. plain: the plain rule (one score map, no window, chunked
// mask, bias, sink, kept keys, cap, temperature or gate), no splits, caches at 16-byte addresses (its loads into shared memory bring
// 16 bytes a lane and want them aligned, where the other kernels' ordinary loads do not).
extern "C" int gl3_prefill_kernel(int head_dim, int page_size, int n_heads, int n_kv, int n_seqs, int max_q_len, int n_tokens, int plain) {
  if (!prefill_wide(head_dim, n_heads, n_seqs, max_q_len)) return 0;
  return plain && turns_takes(head_dim, page_size, n_heads / n_kv, n_seqs, n_tokens) && turns_wanted(n_seqs, max_q_len, n_tokens) ? 2 : 1;
}

// Whether the library takes the kernel of eight waves. 3: with two groups on the keys, 4: with two heads a block, 0: another kernel (`plain` as above).
// All that is known here are the sequences, the longest and the tokens together. Two groups halve a block's way along its keys, which is what a step waits
// for where its blocks are few or one sequence is far longer than the others; two heads a block read half as many keys and values, which pays where many blocks are
// left behind the longest. Measured in every form and on the kernels beside it: 5,843 batches (one sequence, equal and unequal ones, one or two long ones beside
// short ones; 33 to 20,000 tokens) with 16 to 64 heads over 8, 16 over 16 and 32 over 32, of which the limits are, and 3,600 others
// (`profiles/prefill_eight_rule.txt`): at the others, time against the kernel that would be taken without this one, heads of 64 0.846 on average (0.840 with the best
// form everywhere), of 128 0.962 (0.942); above 1.05 of it 3 of them, and 12 of sequences of at most 64 tokens.
// Heads of 64, two blocks a CU at a time. Even numbers of heads a kv head: two heads a block for more than 1,100 blocks of one head, or 400 where the step holds
// five and a half times its longest sequence (32 heads: 4,096 tokens, 1,056 blocks, 86.2 us in two groups and 90.7, 8,192 304 and 293; six of 300 15.5
// and 13.1, 14.3 with 128 queries a block); for sequences of unequal lengths more (1,300 tokens beside twenty of 100 28.2 and 43.4, 34.3). Odd numbers
// have no pairs: two groups but for many short sequences (24 heads: eight of 300 15.7, with 128 queries a block 14.0; six of 1,000 36.5 and 41.9).
// Heads of 128, one block on a CU at a time: two groups from 300 tokens of the longest sequence on (280 tokens 12.9 us, 11.9 with 64 queries a block; 320
// 12.9 and 13.5) to 511 blocks of one sequence, 320 of a short one (24 heads: 2,600 tokens 76 us, with 64 queries a block 101; 32 heads: 2,000 tokens 63.3, with
// turns 58.3; 64 heads: 646 tokens 29.5, with 64 queries 27.7), 512 where the longest has half of the tokens, 256 of others (24 heads: 1,203 beside 317 and
// 701 35.8, with turns 38.7). Two heads a block where the kernel of 128 queries would have them, for 384 tokens a sequence on average and more, of equal length with little of
// their last block empty (a block that is partly empty has its CU for as long; 32 heads: eight of 512 45.9 -> 40.3, ten of 450 43.3 and 46.3), or few (32 heads: 822 tokens
// beside 1,102 of three others 40.7 -> 35.1); with eight heads a kv head unequal ones too (64 heads: 24 of 14,348 tokens, the longest 1,641, 430 -> 392).
#define PF_KEYS (INT_MIN + 1)
#define PF_HEADS (INT_MIN + 2)
static bool eight_takes(int head_dim, int page_size) { return (head_dim == 64 || head_dim == 128) && page_size % 64 == 0; }
extern "C" int gl3_prefill_eight(int head_dim, int page_size, int n_heads, int n_kv, int n_seqs, int max_q_len, int n_tokens, int plain) {
  if (!plain || !eight_takes(head_dim, page_size)) return 0;
  const int group = n_heads / n_kv;
  const bool pairs = group % 2 == 0;
  const long blocks = (long)n_heads * (n_tokens / 128 + (n_seqs + 1) / 2);      // of one head: about as many as there are
  const long most = max_q_len, tokens = n_tokens, padded = most * n_seqs;
  if (head_dim == 64) {
    if (max_q_len <= 32) return 0;
    if (!pairs) return blocks <= 400 || tokens <= 6 * most || (tokens >= 330L * n_seqs && blocks >= 1080) ? 3 : 0;
    if (10 * tokens >= 7 * padded) return blocks > 1100 || (2 * tokens >= 11 * most && blocks > 400) ? 4 : 3;
    if (tokens >= 9 * most) return blocks > 1100 ? 4 : blocks <= 400 ? 3 : 0;
    return blocks > 1800 && tokens >= 5 * most ? 4 : 3;
  }
  if (max_q_len >= 300) {
    const long longest = n_heads * ((most + 127) / 128);
    if (n_seqs == 1 ? longest <= (most >= 700 ? 511 : 320) : blocks <= (tokens <= 2 * most ? 512 : 256)) return 3;
  }
  if (!pairs || tokens < 384L * n_seqs || gl3_prefill_kernel(head_dim, page_size, n_heads, n_kv, n_seqs, max_q_len, n_tokens, plain) != 1) return 0;
  const bool filled = 10 * tokens >= 9 * padded && (most % 128 == 0 || most % 128 >= 96);
  return group % 8 == 0 || (5 * tokens <= 16 * most && blocks <= 700) || (filled && blocks <= 2200) ? 4 : 0;
}

extern "C" int gl3_attention_prefill_supports(int head_dim, int page_size) {
  return (head_dim == 32 || head_dim == 64 || head_dim == 96 || head_dim == 128) && page_size % 32 == 0;
}

// max_q_len: the most tokens any sequence brings in this step (it sizes the grid).
// seq_rows (may be null): the row of `block_table` that holds sequence b's pages; null: row b.
// wide_from: the kernel with 128 queries a block is taken when max_q_len reaches it; <= 0: the library's choice, but for PF_TURNS: the
// kernel of turns, and PF_KEYS, PF_HEADS: the kernel of eight waves in two groups on the keys, or on two heads. Splits: above 0 the kernel of 128 queries,
// else that of eight waves where it is built for the call.
extern "C" int gl3_attention_prefill(const void* q, long q_stride, const void* k_cache, const void* v_cache,
                                     const int* cu_seqlens, const int* kv_before, const int* block_table,
                                     const int* seq_rows, int table_stride, void* out, long out_stride, int n_seqs,
                                     int max_q_len, int n_heads, int n_kv, int head_dim, int page_size, int window,
                                     float scale, int wide_from, const float* slopes, int has_sink, float sink,
                                     int keep_first, int mask_chunk, int maps, const float* sinks, float softcap,
                                     float temp_coef, int temp_every, const void* gate, long gate_ld, int splits,
                                     int n_tokens, float* part_o, float* part_ml, hipStream_t stream) {
  if (n_seqs == 0 || max_q_len == 0) return 0;
  GL3_REQUIRE(q && k_cache && v_cache && cu_seqlens && kv_before && block_table && out,
              "gl3_attention_prefill: null argument");
  GL3_REQUIRE(gl3_attention_prefill_supports(head_dim, page_size),
              "gl3_attention_prefill: head_dim %d / page_size %d is not built (32, 64, 96, 128; pages of a multiple of 32)",
              head_dim, page_size);
  GL3_REQUIRE(n_heads > 0 && n_kv > 0 && n_heads % n_kv == 0, "gl3_attention_prefill: %d heads over %d kv heads",
              n_heads, n_kv);
  GL3_REQUIRE(scale > 0.f, "gl3_attention_prefill: the score scale %g must be positive", (double)scale);
  GL3_REQUIRE(mask_chunk >= 0 && (mask_chunk == 0 || window == 0), "gl3_attention_prefill: a chunked mask has no window");
  GL3_REQUIRE(maps >= 1 && n_kv % maps == 0 && n_heads % maps == 0, "gl3_attention_prefill: %d score maps over %d heads and %d key heads",
              maps, n_heads, n_kv);
  GL3_REQUIRE(q_stride % 8 == 0 && (uintptr_t)q % 16 == 0 && out_stride % 4 == 0 && (uintptr_t)out % 8 == 0,
              "gl3_attention_prefill: queries must be 16-byte aligned, outputs 8-byte aligned");
  const int g = n_heads / n_kv;
  const Gl3ScoreRule rule{softcap, temp_coef, temp_every, gate, gate_ld};
  GL3_CHECK_RULE(rule, "gl3_attention_prefill");
  const bool ruled = rule.any();
  const bool biased = slopes != nullptr || has_sink || sinks != nullptr || keep_first > 0;    // (the kernels that know of kept first keys)
  const bool splits_plain = !ruled && !biased && maps == 1 && window == 0 && mask_chunk == 0 && (uintptr_t)k_cache % 16 == 0 && (uintptr_t)v_cache % 16 == 0;
  const bool plain = splits == 1 && splits_plain;
  const bool eight = plain && eight_takes(head_dim, page_size);
  GL3_REQUIRE((wide_from != PF_KEYS && wide_from != PF_HEADS) || (eight && (wide_from == PF_KEYS || g % 2 == 0)),
              "gl3_attention_prefill: the kernels of eight waves take heads of 64 or 128, pages of whole 64 keys, caches at 16-byte addresses, no splits, the plain rule, and two heads a block an even number of heads a kv head");
  GL3_REQUIRE(wide_from != PF_TURNS || (plain && turns_takes(head_dim, page_size, g, n_seqs, n_tokens)),
              "gl3_attention_prefill: the kernel of turns takes heads of 128, pages of whole 64 keys, caches at 16-byte addresses, at most 64 sequences, no splits, the plain rule");
  const int eights = gl3_prefill_eight(head_dim, page_size, n_heads, n_kv, n_seqs, max_q_len, n_tokens, plain);
  const int kernel = wide_from == PF_TURNS ? 2 : wide_from == PF_KEYS ? 3 : wide_from == PF_HEADS ? 4 : splits > 1 ? 1 : wide_from > 0 ? max_q_len >= wide_from
                     : eights ? eights : gl3_prefill_kernel(head_dim, page_size, n_heads, n_kv, n_seqs, max_q_len, n_tokens, plain);
  const bool wide = kernel > 0;
  // query heads per wave: as many as the registers hold with two blocks on a CU; one with 32 queries a wave
  const int gh = wide ? 1 : head_dim <= 32 ? 4 : head_dim <= 64 ? 2 : 1;
  const long z = (long)n_kv * ((g + gh - 1) / gh);
  const int q_blocks = wide ? (max_q_len + 127) / 128 : (max_q_len + 63) / 64;
  GL3_REQUIRE(n_seqs <= 65535 && q_blocks <= 65535, "gl3_attention_prefill: %d sequences / %d blocks of queries exceed the grid",
              n_seqs, q_blocks);
  dim3 grid((unsigned)z * (splits > 1 ? splits : 1), n_seqs, q_blocks), block(256);
  GL3_REQUIRE(keep_first >= 0 && (keep_first == 0 || window > 0), "gl3_attention_prefill: %d kept first keys without a window", keep_first);
  GL3_REQUIRE(!gate || (gate_ld % 4 == 0 && (uintptr_t)gate % 8 == 0), "gl3_attention_prefill: gate rows must be 8-byte aligned");
  const PfSplit sp{splits, n_tokens, part_o, part_ml};
  GL3_REQUIRE(splits >= 1 && splits <= PF_SPLITS, "gl3_attention_prefill: %d splits (1 to %d)", splits, PF_SPLITS);
  GL3_REQUIRE(splits == 1 || (part_o && part_ml && n_tokens > 0 && !ruled && !biased && maps == 1 && (uintptr_t)part_o % 16 == 0),
              "gl3_attention_prefill: splits need buffers for their sums and the plain rule (one score map, no bias, sink, kept keys, cap, temperature or gate)");
  if (kernel == 2) {
    const int heads = g % 2 == 0 ? 2 : 1, queries = 256 / heads, qbs = (max_q_len + queries - 1) / queries;
    dim3 tgrid((unsigned)(n_heads / heads), n_seqs == 1 ? qbs : n_tokens / queries + n_seqs);
#define GOT(HEADS)                                                                                                    \
  attention_prefill_turns_kernel<HEADS><<<tgrid, dim3(512), 0, stream>>>(                                             \
      (const bf16_t*)q, q_stride, (const bf16_t*)k_cache, (const bf16_t*)v_cache, cu_seqlens, kv_before, block_table, \
      seq_rows, table_stride, (bf16_t*)out, out_stride, n_heads, n_kv, page_size, scale, qbs, n_seqs)
    if (heads == 2) GOT(2);
    else GOT(1);
#undef GOT
    GL3_LAUNCH_CHECK();
    return 0;
  }
  if (kernel >= 3 || (splits > 1 && wide_from <= 0 && splits_plain && eight_takes(head_dim, page_size))) {
    const int heads = kernel == 4 ? 2 : 1;
    const bool folded = n_seqs == 1 && (long)n_heads / heads * q_blocks * splits <= 512;
    // Blocks beyond their sequence's end leave at once. The blocks of an XCD go to its four engines in turn, so where an even number of sequences has one
    // that is far longer than the others, its blocks would meet the same engines again and again: one row more of blocks that leave (16 heads of 128: 3,502 tokens beside
    // three of 17 127 us, so 73; two heads a block 213 and 107).
    const bool uneven = n_seqs % 2 == 0 && 10L * n_tokens < 7L * n_seqs * max_q_len;
    dim3 egrid((unsigned)(n_heads / heads * splits), n_seqs + uneven, q_blocks);
#define GOE(HS, GROUPS, SPLIT)                                                                                        \
  attention_prefill_eight_kernel<HS, GROUPS, SPLIT><<<egrid, dim3(512), 0, stream>>>(                                            \
      (const bf16_t*)q, q_stride, (const bf16_t*)k_cache, (const bf16_t*)v_cache, cu_seqlens, kv_before, block_table, \
      seq_rows, table_stride, (bf16_t*)out, out_stride, n_heads, n_kv, page_size, scale, q_blocks, (int)folded, n_seqs, sp)
#define GOEH(HS)                                                                                                      \
  do {                                                                                                                \
    if (splits > 1) {                                                                                                 \
      GOE(HS, 2, true);                                                                                               \
      const long rows = (long)n_tokens * n_heads * (HS / 4);                                                          \
      attention_prefill_merge_kernel<HS><<<dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, stream>>>(sp, (bf16_t*)out, out_stride, n_heads); \
    } else if (kernel == 3) GOE(HS, 2, false);                                                                        \
    else GOE(HS, 1, false);                                                                                           \
  } while (0)
    if (head_dim == 64) GOEH(64);
    else GOEH(128);
#undef GOEH
#undef GOE
    GL3_LAUNCH_CHECK();
    return 0;
  }
  if (wide) {
#define PF_ARGS                                                                                                     \
  (const bf16_t*)q, q_stride, (const bf16_t*)k_cache, (const bf16_t*)v_cache, cu_seqlens, kv_before, block_table,     \
      seq_rows, table_stride, (bf16_t*)out, out_stride, n_heads, n_kv, page_size, window, scale, q_blocks, slopes, has_sink, sink, keep_first, mask_chunk, maps, sinks, rule
#define GOW(HS, CK, AH, OCC)                                                                                        \
  do {                                                                                                              \
    if (ruled) attention_prefill_wide_kernel<HS, CK, AH, OCC, true, true><<<grid, block, 0, stream>>>(PF_ARGS, sp);     \
    else if (biased) attention_prefill_wide_kernel<HS, CK, AH, OCC, true><<<grid, block, 0, stream>>>(PF_ARGS, sp);     \
    else if (splits > 1) {                                                                                          \
      attention_prefill_wide_kernel<HS, CK, AH, OCC, false, false, true><<<grid, block, 0, stream>>>(PF_ARGS, sp);  \
      const long n = (long)n_tokens * n_heads * (HS / 4);                                                          \
      attention_prefill_merge_kernel<HS><<<dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream>>>(sp, (bf16_t*)out, out_stride, n_heads); \
    } else attention_prefill_wide_kernel<HS, CK, AH, OCC, false><<<grid, block, 0, stream>>>(PF_ARGS, sp);          \
  } while (0)
    // chunks of 64 keys (one barrier for twice the work, two score tiles whose sums do not wait for
    // each other) where the registers hold them and a page holds whole chunks
    const bool ck64 = page_size % 64 == 0;
    switch (head_dim) {
      case 32: if (ck64) { GOW(32, 64, 2, 3); } else { GOW(32, 32, 2, 3); } break;
      case 64: if (ck64) { GOW(64, 64, 2, 2); } else { GOW(64, 32, 2, 3); } break;
      case 96: GOW(96, 32, 2, 2); break;
      default: GOW(128, 32, 1, 2); break;
    }
#undef GOW
    GL3_LAUNCH_CHECK();
    return 0;
  }
#define GO(HS, GH)                                                                                                  \
  do {                                                                                                              \
    if (ruled) attention_prefill_kernel<HS, GH, true, true><<<grid, block, 0, stream>>>(PF_ARGS);                   \
    else if (biased) attention_prefill_kernel<HS, GH, true><<<grid, block, 0, stream>>>(PF_ARGS);                   \
    else attention_prefill_kernel<HS, GH, false><<<grid, block, 0, stream>>>(PF_ARGS);                              \
  } while (0)
  switch (head_dim) {
    case 32: GO(32, 4); break;
    case 64: GO(64, 2); break;
    case 96: GO(96, 1); break;
    default: GO(128, 1); break;
  }
#undef GO
#undef PF_ARGS
  GL3_LAUNCH_CHECK();
  return 0;
}

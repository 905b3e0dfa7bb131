// Causal grouped-query attention over the paged cache in true 32-bit on the matrix cores (v_mfma_f32_16x16x4_f32: IEEE
// products and sums), for the plain rule: every earlier key, values of the keys' size, heads of 32, 64, 96 or 128.
// gl3_attention_generic sends such calls here; anything beside the plain rule stays with its own kernel, which visits
// a key per lane and step and is bound by trips to memory one after the other (two requests of 333 and 180 prompt tokens,
// then 16 tokens each, 1B layers: 185 us a call on average there, 13 us here; 19 before the loads of a step went out together).
//
// A block works on sixteen rows, a row being one (token, query head) of one sequence and kv head, so that the heads of
// a group and neighbouring tokens share the keys and values that it reads; its eight waves take the key steps of 64
// positions in turn (wave w: steps w, w + 8, ...), each with a running softmax of its own, merged in the order of the
// waves. Which positions make a step and which wave takes it depends on the position alone, and a step whose keys a row
// does not see leaves that row's numbers as they are: a token's result is the same bit for bit whether it arrives
// with its whole prompt or alone, and with `per_tile` tokens a block or one (the host's choice: whether the blocks fill the chip).
//
// Operands: a tile of keys in the cache's order (gl3_k_offset: rows i of the two tiles of 32 positions are the positions
// 8 (i / 4) + i % 4 and those 4 further) times the rows' queries gives a lane four consecutive positions of one row,
// which are the weights that the second product takes from that very lane against four consecutive positions of a
// value row: no weight moves between lanes.
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

#define AF_WAVES 8

template <int HB, bool AHEAD>
__global__ __launch_bounds__(64 * AF_WAVES, AHEAD || HB > 4 ? 2 : 4) void attention_f32_kernel(
    const float* __restrict__ Q, long q_stride, const float* __restrict__ k_cache, const float* __restrict__ v_cache,
    const int* __restrict__ positions, const int* __restrict__ table_rows, const int* __restrict__ block_table, int table_stride,
    float* __restrict__ out, long out_stride, int n_tokens, int group, int n_kv, int page_size, float scale, int per_tile) {
  constexpr int HS = 16 * HB;
  __shared__ __attribute__((aligned(16))) f32x4 part[AF_WAVES][HB][64];
  __shared__ float part_m[AF_WAVES][16], part_l[AF_WAVES][16];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int r = lane & 15, q = lane >> 4;
  const int c = blockIdx.y;
  const int tile = gridDim.x - 1 - blockIdx.x;          // (the last tokens have the most keys: they start first)
  int t0 = tile * per_tile;
  const int t1 = min(t0 + per_tile, n_tokens);
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  while (t0 < t1) {
    // tokens of one sequence (at most sixteen: all their rows of the table in one load)
    const int rows = t0 + lane < t1 ? table_rows[t0 + lane] : -1;
    const int row0 = __builtin_amdgcn_readfirstlane(rows);
    const int te = t0 + __builtin_ctzl(~__ballot(t0 + lane < t1 && rows == row0));
    const int* bt = block_table + (long)row0 * table_stride;
    const int flats = (te - t0) * group;
    for (int base = 0; base < flats; base += 16) {
      const int a = base + r;
      const bool have = a < flats;
      const int t = t0 + (have ? a / group : 0), h = c * group + (have ? a % group : 0);
      const int p = have ? positions[t] : -1;
      // AHEAD: the pages of a step's halves are asked for a step ahead (the first before the positions are there: entries beyond the
      // sequence's pages are looked up inside the row and not used)
      int page[2];
      auto look_up = [&](int first) {
#pragma unroll
        for (int b = 0; b < 2; ++b) page[b] = bt[min((first + 32 * b) / page_size, table_stride - 1)];
      };
      if (AHEAD) look_up(wave * 64);
      int p_max = p, p_min = have ? p : 0x7fffffff;
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) {
        p_max = max(p_max, __shfl_xor(p_max, o, 64));
        p_min = min(p_min, __shfl_xor(p_min, o, 64));
      }
      p_max = __builtin_amdgcn_readfirstlane(p_max);
      p_min = __builtin_amdgcn_readfirstlane(p_min);
      f32x4 qf[HB];
#pragma unroll
      for (int d = 0; d < HB; ++d) qf[d] = *(const f32x4_any*)(Q + (long)t * q_stride + (long)h * HS + d * 16 + q * 4);
      float m = -INFINITY, l = 0.f;
      bool had_odd = false;
      f32x4 acc[HB];
#pragma unroll
      for (int d = 0; d < HB; ++d) acc[d] = zero;

      for (int first = wave * 64; first <= p_max; first += 64 * AF_WAVES) {
        const float *kp[2], *vp[2];
        if (!AHEAD) look_up(first);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const bool seen = first + 32 * b <= p_max;     // (a second half that no row sees reads the first again)
          const int pg = page[seen ? b : 0], in_page = (seen ? first + 32 * b : first) % page_size;
          const long at = ((long)pg * n_kv + c) * page_size * HS;
          kp[b] = k_cache + at + (long)in_page * HS + ((q >> 1) << 7) + (r << 3) + (q & 1) * 4;
          vp[b] = v_cache + at + (((in_page >> 3) + q) << 7) + (r << 3);
        }
        // AHEAD (at most one block a CU): all of a step's keys are asked for before the first is waited for, its values in front of the
        // scores or, where the registers do not hold both, of the softmax. Otherwise the compiler waits for one load after
        // the other, 32 trips to memory a step, which the other block of a CU hides. With heads of 128 the registers hold half of the keys or
        // of the values (PART) beside the sums; the other half is asked for when the first is multiplied. (All of them at once went to
        // scratch memory: 2,000 keys for each of four tokens 73 us, in halves 63, without AHEAD 87; 700 for each of two 30, 25 and 26.)
        constexpr int PART = HB > 6 ? HB / 2 : HB;
        f32x4 vf[AHEAD ? HB : 1][2][2];
        auto load_values = [&](int d0, int d1) {
#pragma unroll
          for (int d = d0; d < d1; ++d)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
              for (int e = 0; e < 2; ++e) vf[AHEAD ? d : 0][b][e] = *(const f32x4*)(vp[b] + (((long)d * (page_size >> 3)) << 7) + e * 4);
        };
        f32x4 kf[AHEAD ? HB : 1][2][2];
        auto load_keys = [&](int d0, int d1) {
#pragma unroll
          for (int d = d0; d < d1; ++d)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
              for (int e = 0; e < 2; ++e) kf[AHEAD ? d : 0][b][e] = *(const f32x4*)(kp[b] + ((e * (HS >> 3) + d * 2) << 7));
        };
        if (AHEAD) {
          load_keys(0, PART);
          if (HB <= 4) load_values(0, HB);
        }
        if (AHEAD) look_up(min(first + 64 * AF_WAVES, p_max));
        if (AHEAD) __builtin_amdgcn_sched_barrier(0);
        f32x4 s[2][2] = {{zero, zero}, {zero, zero}};
#pragma unroll
        for (int d = 0; d < HB; ++d) {
          if (AHEAD && PART < HB && d == PART) {
            __builtin_amdgcn_sched_barrier(0);
            load_keys(PART, HB);
            __builtin_amdgcn_sched_barrier(0);
          }
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const f32x4 k = AHEAD ? kf[AHEAD ? d : 0][b][e] : *(const f32x4*)(kp[b] + ((e * (HS >> 3) + d * 2) << 7));
#pragma unroll
              for (int j = 0; j < 4; ++j) s[b][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[j], qf[d][j], s[b][e], 0, 0, 0);
            }
        }
        if (AHEAD && HB > 4) {
          __builtin_amdgcn_sched_barrier(0);
          load_values(0, PART);
          __builtin_amdgcn_sched_barrier(0);
        }
        // a lane's scores: positions first + 32 b + 8 q + 4 e + v of row r
        float most = -INFINITY;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              s[b][e][v] = first + 32 * b + 8 * q + 4 * e + v <= p ? s[b][e][v] * scale : -INFINITY;
              most = fmaxf(most, s[b][e][v]);
            }
        most = fmaxf(most, __shfl_xor(most, 16, 64));
        most = fmaxf(most, __shfl_xor(most, 32, 64));
        const float m_new = fmaxf(m, most);
        const float from = m_new == -INFINITY ? 0.f : m_new;           // (no key seen yet: weights and sums stay zero)
        const float alpha = m == m_new ? 1.f : expf(m - from);
        float sum = 0.f;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              s[b][e][v] = first + 32 * b + 8 * q + 4 * e + v <= p ? expf(s[b][e][v] - from) : 0.f;
              sum += s[b][e][v];
            }
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        l = l * alpha + sum;
        m = m_new;
        const bool edge = first + 63 > p_min;     // some row does not see some of these keys (or they do not exist)
        bool odd = false;
        // a weight of zero does not make nothing of an infinite value: such values are left out here
        auto leave_out = [&](f32x4& val) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const bool fine = fabsf(val[j]) < INFINITY;
            odd |= !fine;
            val[j] = fine ? val[j] : 0.f;
          }
        };
        if (AHEAD) {
          auto multiply = [&](int d0, int d1) {
            if (edge) {
#pragma unroll
              for (int i = 4 * d0; i < 4 * d1; ++i) leave_out((&vf[0][0][0])[i]);
            }
#pragma unroll
            for (int d = d0; d < d1; ++d) acc[d] *= alpha;
            // (an output tile's products one after the other in the order of the keys; the tiles take turns)
#pragma unroll
            for (int i = 0; i < 16; ++i)
#pragma unroll
              for (int d = d0; d < d1; ++d)
                acc[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[AHEAD ? d : 0][i >> 3][(i >> 2) & 1][i & 3], s[i >> 3][(i >> 2) & 1][i & 3], acc[d], 0, 0, 0);
          };
          multiply(0, PART);
          if (PART < HB) {
            __builtin_amdgcn_sched_barrier(0);
            load_values(PART, HB);
            __builtin_amdgcn_sched_barrier(0);
            multiply(PART, HB);
          }
        } else {
#pragma unroll
          for (int d = 0; d < HB; ++d) {
            acc[d] *= alpha;
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
              for (int e = 0; e < 2; ++e) {
                f32x4 val = *(const f32x4*)(vp[b] + (((long)d * (page_size >> 3)) << 7) + e * 4);
                if (edge) leave_out(val);
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(val[j], s[b][e][j], acc[d], 0, 0, 0);
              }
          }
        }
        if (edge && __any(odd)) {
          // and added up apart for the rows that see them (not rescaled later: no factor makes them finite)
          if (!had_odd)
#pragma unroll 1
            for (int d = 0; d < HB; ++d) part[wave][d][lane] = zero;
          had_odd = true;
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
              for (int j = 0; j < 4; ++j) {
#pragma unroll 1
                for (int qq = 0; qq < 4; ++qq) {
                  const float w = __shfl(s[b][e][j], qq * 16 + r, 64);
                  const bool seen = first + 32 * b + 8 * qq + 4 * e + j <= p;
                  const float* at = vp[b] - (q << 7) - (r << 3) + (qq << 7) + e * 4 + j;       // this position, dim 0
#pragma unroll 1
                  for (int i = 0; i < 4 * HB; ++i) {
                    const int d = i >> 2, v = i & 3;
                    const float val = at[(((long)d * (page_size >> 3)) << 7) + ((4 * q + v) << 3)];
                    if (seen && !(fabsf(val) < INFINITY)) part[wave][d][lane][v] += w * val;
                  }
                }
              }
        }
      }
      if (had_odd)
#pragma unroll
        for (int d = 0; d < HB; ++d) acc[d] += part[wave][d][lane];
#pragma unroll
      for (int d = 0; d < HB; ++d) part[wave][d][lane] = acc[d];
      if (q == 0) {
        part_m[wave][r] = m;
        part_l[wave][r] = l;
      }
      __syncthreads();
      for (int e = tid; e < HB * 64; e += 64 * AF_WAVES) {
        const int d = e >> 6, ln = e & 63, rr = ln & 15;
        if (base + rr >= flats) continue;
        float top = part_m[0][rr];
#pragma unroll
        for (int w = 1; w < AF_WAVES; ++w) top = fmaxf(top, part_m[w][rr]);
        float total = 0.f;
        f32x4 o = zero;
#pragma unroll
        for (int w = 0; w < AF_WAVES; ++w) {
          const float mw = part_m[w][rr];
          if (mw == -INFINITY && part_l[w][rr] == 0.f) continue;     // (a wave whose keys the row does not see; scores that are all NaN have a weight)
          const float f = expf(mw - top);
          total += part_l[w][rr] * f;
          o += part[w][d][ln] * f;
        }
        const int fa = base + rr;
        float* op = out + (long)(t0 + fa / group) * out_stride + (long)(c * group + fa % group) * HS + d * 16 + (ln >> 4) * 4;
        *(f32x4_any*)op = o / total;
      }
      __syncthreads();
    }
    t0 = te;
  }
}

bool gl3_attention_f32_takes(int head_dim, int page_size) {
  return (head_dim == 32 || head_dim == 64 || head_dim == 96 || head_dim == 128) && page_size % 32 == 0;
}

int gl3_attention_f32(const float* q, long q_stride, const float* k_cache, const float* v_cache, const int* positions,
                      const int* table_rows, const int* block_table, int table_stride, float* out, long out_stride, int n_tokens,
                      int n_heads, int n_kv, int head_dim, int page_size, float scale, hipStream_t stream) {
  const int group = n_heads / n_kv;
  // tokens a block takes: as many as its sixteen rows hold, but one where the blocks would not fill the chip
  const int most = group >= 16 ? 1 : 16 / group;
  const int per_tile = (long)((n_tokens + most - 1) / most) * n_kv >= 512 ? most : 1;
  const dim3 grid((n_tokens + per_tile - 1) / per_tile, n_kv), block(64 * AF_WAVES);
  // (the loads of a step in registers at once take the room of the other block that a CU would hold: 333 and 180 tokens, 32 heads of
  // 64, 34 us without and 40 with; 2,000 keys for each of four tokens 49 and 34, heads of 32 20.0 and 19.9, of 96 59 and 52, of 128 87 and 63.
  // Of 75 steps of 1 to 32 tokens with 0 to 8,000 keys, heads of 32 to 128, the greatest loss is 0.9 us of 14 (heads of 96, 350 keys))
  const bool ahead = (long)grid.x * grid.y <= 256;
#define AF_GO(HB, AHEAD)                                                                                                        \
  attention_f32_kernel<HB, AHEAD><<<grid, block, 0, stream>>>(q, q_stride, k_cache, v_cache, positions, table_rows, block_table, \
                                                             table_stride, out, out_stride, n_tokens, group, n_kv, page_size, scale, per_tile)
#define AF_RUN(HB)                \
  do {                            \
    if (ahead) AF_GO(HB, true);   \
    else AF_GO(HB, false);        \
  } while (0)
  if (head_dim == 32) AF_RUN(2);
  else if (head_dim == 64) AF_RUN(4);
  else if (head_dim == 96) AF_RUN(6);
  else AF_RUN(8);
#undef AF_RUN
#undef AF_GO
  GL3_LAUNCH_CHECK();
  return 0;
}

// Paged grouped-query attention for portions of prompts (two or more query tokens of one
// sequence in a step), float32 cache, head sizes 64 and 128, on the matrix cores' float32
// instruction (MFMA 16x16x4: products and sums in float32, nothing narrower).
//
// Query token i of the step sits at position p = ctx_before + i and reads keys
// max(0, p - window + 1) .. p (window <= 0: all keys up to p).  Query head h reads kv head
// h / G.  A row is one (query token, query head of the group) pair.
//
// Block = 16 rows of one kv head of one sequence, four waves; units of 32 keys go to the
// waves in turn, every wave keeps its own running maximum, sum and output for all 16 rows,
// and the four meet in LDS at the end, in the order of the waves.  So a walk is a quarter
// as long as its rows' context and no wave waits for another inside it.
//   S^T = K Q^T      A = 16 keys, B = the 16 rows (held in registers for the whole walk).
//                    Keys and values go straight from their pages to the operands' registers:
//                    a lane (r = lane % 16, q = lane / 16) reads dims 16 t + 4 q .. + 3 of key r,
//                    four numbers that are the operands of four MFMAs.
//   softmax          float32, online over units, expf.  A row's 16 keys of a tile sit in four lanes.
//   O^T += V^T P^T   A = 16 dims x 16 keys: value pages are stored transposed ([D][slot]), so the
//                    lane reads slots 4 q .. + 3 of dim r; B = P^T straight from the score
//                    registers: the scores of keys 4 q + s are what MFMA s asks of lane q.
// The next unit's keys are requested when this unit's scores are formed, its values when they are
// requested by the scores' products, page ids a unit earlier.  Heads go to XCDs by blockIdx, so that
// an L2 holds the keys of its own heads; rows with long walks are launched first.
// What bounds it: 2,048 clocks of MFMA against 16 loads of 1 KB a wave and tile, so the matrix pipe where
// the walks are long; at a few hundred tokens the chain of a block's units.  Measured on one MI355X, 16 query
// heads on 8 kv heads of 128, us a launch, the general kernel on the vector ALU -> this: one prompt of
// 100 tokens 57 -> 14; of 700 406 -> 46; of 2,048 2,487 -> 236 (73 TFLOP/s of the causal products); 16 tokens behind
// 4,000 89 -> 29; 200 behind 8,000 2,264 -> 227.
// With few rows and a long context the keys are cut into `splits` runs, a block each, merged by the
// general kernel's merge kernel.
#include "attention_merge.h"

typedef __attribute__((ext_vector_type(4))) float floatx4;

#define UNIT 32       // keys a wave takes at a time
#define WAVES 4

template <int D>
__global__ __launch_bounds__(64 * WAVES, 2) void paged_prefill_f32_kernel(
    const float* __restrict__ q, long long q_stride, const float* __restrict__ key_pages,
    const float* __restrict__ value_pages, float* __restrict__ out, long long out_stride,
    const int* __restrict__ cu_q, const int* __restrict__ ctx_len, const int* __restrict__ block_table,
    int table_stride, int kv_heads, int groups, int block_shift, int num_blocks, int window, float scale,
    int splits, float* __restrict__ part_acc, float* __restrict__ part_ml, int total_tokens) {
  constexpr int T = D / 16;
  __shared__ __attribute__((aligned(16))) floatx4 acc_s[WAVES - 1][T][64];
  __shared__ float ml_s[WAVES][2][16];
  const int seq = blockIdx.y;
  const int hk = blockIdx.x % kv_heads;
  const int split = blockIdx.x / kv_heads % splits;
  const int q0 = cu_q[seq];
  const int q_len = cu_q[seq + 1] - q0;
  const int ctx_before = ctx_len[seq] - q_len;
  const int rows_total = q_len * groups;
  const int tiles = (rows_total + ROWS - 1) / ROWS;
  const int tile = tiles - 1 - (int)(blockIdx.x / kv_heads / splits);
  if (q_len < 2 || tile < 0 || ctx_before < 0) return;

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, lq = lane >> 4;
  const int row0 = tile * ROWS;
  const int my_row = min(row0 + r, rows_total - 1);      // rows beyond the last: the last again, never stored
  const int my_tok = my_row / groups, my_g = my_row - my_tok * groups;
  const int my_pos = ctx_before + my_tok;
  const int pos_min = ctx_before + row0 / groups;
  const int pos_max = ctx_before + (min(rows_total, row0 + ROWS) - 1) / groups;
  const int k_begin = window > 0 ? max(0, pos_min - window + 1) : 0;
  const int k_end = pos_max + 1;
  const int block_mask = (1 << block_shift) - 1;
  const int* table = block_table + (size_t)seq * table_stride;

  // this block's run of units, and of these every WAVES-th for this wave
  const int first = k_begin / UNIT, last = (k_end + UNIT - 1) / UNIT;
  const int each = (last - first + splits - 1) / splits;
  const int my_first = first + split * each + wave, my_last = min(last, first + (split + 1) * each);

  floatx4 qf[T];
  const float* qrow = q + (size_t)(q0 + my_tok) * q_stride + (size_t)(hk * groups + my_g) * D + 4 * lq;
#pragma unroll
  for (int t = 0; t < T; ++t) qf[t] = *(const floatx4*)(qrow + 16 * t);

  // pages of this lane's key and of its four value slots, of the unit's two tiles of 16 keys; a page id outside the pool
  // (a slot that was never written) reads page 0, whose numbers the masks below drop
  int key_page[2], value_page[2];
  auto lookup = [&](int unit) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = unit * UNIT + 16 * h;
      const int kp = table[min(max(at + r, k_begin), k_end - 1) >> block_shift];
      const int vp = table[min(max(at + 4 * lq, k_begin), k_end - 1) >> block_shift];
      key_page[h] = kp >= 0 && kp < num_blocks ? kp : 0;
      value_page[h] = vp >= 0 && vp < num_blocks ? vp : 0;
    }
  };
  floatx4 kf[2][T], vf[2][T];
  auto load_keys = [&](int unit) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int slot = (unit * UNIT + 16 * h + r) & block_mask;
      const float* p = key_pages + ((((size_t)key_page[h] * kv_heads + hk) << block_shift) + slot) * D + 4 * lq;
#pragma unroll
      for (int t = 0; t < T; ++t) kf[h][t] = *(const floatx4*)(p + 16 * t);
    }
  };
  auto load_values = [&](int unit) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int slot = (unit * UNIT + 16 * h + 4 * lq) & block_mask;
      const float* p = value_pages + ((((size_t)value_page[h] * kv_heads + hk) * D + r) << block_shift) + slot;
#pragma unroll
      for (int t = 0; t < T; ++t) vf[h][t] = *(const floatx4*)(p + ((size_t)(16 * t) << block_shift));
    }
  };

  floatx4 acc[T];
#pragma unroll
  for (int t = 0; t < T; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;      // l: this lane's share of the row's sum
  if (my_first < my_last) {
    lookup(my_first);
    load_keys(my_first);
  }
  for (int unit = my_first; unit < my_last; unit += WAVES) {
    load_values(unit);
    if (unit + WAVES < my_last) lookup(unit + WAVES);
    floatx4 s[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int h = 0; h < 2; ++h) s[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[h][t][e], qf[t][e], s[h], 0, 0, 0);
    if (unit + WAVES < my_last) load_keys(unit + WAVES);

    // lane (r, lq) holds the scores of keys 16 h + 4 lq + e of row r
    float top = -INFINITY;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int kp = unit * UNIT + 16 * h + 4 * lq + e;
        const bool visible = kp <= my_pos && (window <= 0 || kp > my_pos - window);
        s[h][e] = visible ? s[h][e] * scale : -INFINITY;
        top = fmaxf(top, s[h][e]);
      }
    top = max_xor32(max_xor16(top));
    const float m_new = fmaxf(m, top);
    const float safe = m_new > -INFINITY ? m_new : 0.f;      // a row that has seen no key yet: every exponential below is zero
    const float corr = expf(m - safe);
    float sum = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[h][e] = expf(s[h][e] - safe);
        sum += s[h][e];
      }
    l = l * corr + sum;
    m = m_new;
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[t][e] *= corr;
    if (unit * UNIT < k_begin || (unit + 1) * UNIT > k_end) {      // slots that hold no key of these rows may hold anything
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int kp = unit * UNIT + 16 * h + 4 * lq + e;
          if (kp < k_begin || kp >= k_end) {
#pragma unroll
            for (int t = 0; t < T; ++t) vf[h][t][e] = 0.f;
          }
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int t = 0; t < T; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[h][t][e], s[h][e], acc[t], 0, 0, 0);
  }
  l = sum_xor32(sum_xor16(l));

  // the waves' shares of the rows; lane (r, lq) holds dims 16 t + 4 lq .. + 3 of row r
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < T; ++t) acc_s[wave - 1][t][lane] = acc[t];
  }
  if (lq == 0) { ml_s[wave][0][r] = m; ml_s[wave][1][r] = l; }
  __syncthreads();
  if (wave > 0) return;
  float m_tot = m;
#pragma unroll
  for (int w = 1; w < WAVES; ++w) m_tot = fmaxf(m_tot, ml_s[w][0][r]);
  const float safe = m_tot > -INFINITY ? m_tot : 0.f;
  float f = expf(m - safe), total = l * f;
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[t][e] *= f;
#pragma unroll
  for (int w = 1; w < WAVES; ++w) {
    f = expf(ml_s[w][0][r] - safe);
    total = fmaf(ml_s[w][1][r], f, total);
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const floatx4 other = acc_s[w - 1][t][lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[t][e] = fmaf(other[e], f, acc[t][e]);
    }
  }
  if (row0 + r >= rows_total) return;
  if (splits == 1) {
    const float inv = total > 0.f ? 1.f / total : 0.f;
    float* orow = out + (size_t)(q0 + my_tok) * out_stride + (size_t)(hk * groups + my_g) * D + 4 * lq;
#pragma unroll
    for (int t = 0; t < T; ++t) {
#pragma unroll
      for (int e = 0; e < 4; ++e) orow[16 * t + e] = acc[t][e] * inv;
    }
  } else {
    const size_t row = ((size_t)split * total_tokens + q0 + my_tok) * (kv_heads * groups) + hk * groups + my_g;
#pragma unroll
    for (int t = 0; t < T; ++t) *(floatx4*)(part_acc + row * D + 16 * t + 4 * lq) = acc[t];
    if (lq == 0) { part_ml[row * 2] = m_tot; part_ml[row * 2 + 1] = total; }
  }
}

// Sequences with fewer than two query tokens are skipped (the decode kernels serve them).  Head size 64 or 128, pages of a
// power of two of at least four slots, q (rows q_stride apart, a multiple of four) and the pages 16-byte aligned; the
// rest, the scratch of `splits` > 1 included, as for the general kernel.
extern "C" int fe_paged_attention_prefill_f32(const float* q, long long q_stride, const float* key_pages,
                                              const float* value_pages, float* out, long long out_stride,
                                              const int* cu_q, const int* ctx_len, const int* block_table,
                                              int table_stride, int num_seqs, int max_q_len, int kv_heads, int groups,
                                              int head_dim, int block_size, int num_blocks, int window, float scale,
                                              int splits, float* part_acc, float* part_ml, int total_tokens,
                                              hipStream_t stream) {
  if (num_seqs <= 0 || max_q_len < 2) return FE_OK;
  if (head_dim != 64 && head_dim != 128) return FE_BAD_ARGUMENT;
  if (block_size < 4 || (block_size & (block_size - 1))) return FE_BAD_ARGUMENT;
  if (kv_heads <= 0 || groups <= 0 || num_blocks <= 0 || table_stride <= 0) return FE_BAD_ARGUMENT;
  if (kv_heads > 65535 || num_seqs > 65535) return FE_BAD_ARGUMENT;
  if (out_stride < (long long)kv_heads * groups * head_dim) return FE_BAD_ARGUMENT;
  if (((((uintptr_t)q) | (uintptr_t)key_pages | (uintptr_t)value_pages) & 15) || q_stride % 4) return FE_BAD_ARGUMENT;
  if (splits < 1 || splits > 64 || (splits > 1 && (!part_acc || !part_ml || total_tokens < 1))) return FE_BAD_ARGUMENT;
  int block_shift = 0;
  while ((1 << block_shift) < block_size) ++block_shift;
  const long long tiles = ((long long)max_q_len * groups + ROWS - 1) / ROWS;
  if (tiles * kv_heads * splits > 0x7fffffffLL) return FE_BAD_ARGUMENT;
  const dim3 grid((unsigned)(tiles * kv_heads * splits), num_seqs);
  if (head_dim == 64)
    paged_prefill_f32_kernel<64><<<grid, 64 * WAVES, 0, stream>>>(q, q_stride, key_pages, value_pages, out, out_stride, cu_q, ctx_len,
        block_table, table_stride, kv_heads, groups, block_shift, num_blocks, window, scale, splits, part_acc, part_ml, total_tokens);
  else
    paged_prefill_f32_kernel<128><<<grid, 64 * WAVES, 0, stream>>>(q, q_stride, key_pages, value_pages, out, out_stride, cu_q, ctx_len,
        block_table, table_stride, kv_heads, groups, block_shift, num_blocks, window, scale, splits, part_acc, part_ml, total_tokens);
  if (splits > 1) {
    const dim3 merge_grid((unsigned)tiles, kv_heads, num_seqs);
    if (head_dim == 64)
      paged_attention_generic_merge_kernel<float, 64, false><<<merge_grid, 256, 0, stream>>>(
          out, out_stride, cu_q, ctx_len, kv_heads, groups, head_dim, 2, max_q_len, splits, part_acc, part_ml, total_tokens);
    else
      paged_attention_generic_merge_kernel<float, 128, false><<<merge_grid, 256, 0, stream>>>(
          out, out_stride, cu_q, ctx_len, kv_heads, groups, head_dim, 2, max_q_len, splits, part_acc, part_ml, total_tokens);
  }
  return fe_check_launch();
}

// The merge of attention's key runs, shared by the kernels that leave their runs in scratch.
#pragma once
#include "common.h"

#define ROWS 16

// The runs of a row's keys, merged in their order: a grid of (tile of ROWS rows, kv head,
// sequence); thread (r = tid / 16, c = tid % 16) owns dims c, c + 16, ... of row r, a row being one (query token,
// query head of the group) pair.  part_acc [split][token][head][dim] holds the runs' unnormalised sums, part_ml their
// (maximum, sum of exponentials) a row.
template <typename T, int DMAX, bool FAST_EXP>
__global__ __launch_bounds__(256) void paged_attention_generic_merge_kernel(
    T* __restrict__ out, long long out_stride, const int* __restrict__ cu_q, const int* __restrict__ ctx_len,
    int kv_heads, int groups, int head_dim, int min_q_len, int max_q_served, int splits,
    const float* __restrict__ part_acc, const float* __restrict__ part_ml, int total_tokens) {
  constexpr int DPT = DMAX / 16;
  const int D = head_dim;
  const int seq = blockIdx.z, hk = blockIdx.y;
  const int q0 = cu_q[seq];
  const int q_len = cu_q[seq + 1] - q0;
  const int rows_total = q_len * groups;
  const int row0 = blockIdx.x * ROWS;
  if (row0 >= rows_total || ctx_len[seq] - q_len < 0 || q_len < min_q_len || q_len > max_q_served) return;
  const int r = threadIdx.x / 16, c = threadIdx.x % 16;
  const int my_row = row0 + r;
  if (my_row >= rows_total) return;
  const int tok = my_row / groups, g = my_row - tok * groups;
  const size_t heads = (size_t)kv_heads * groups;
  const size_t first = ((size_t)(q0 + tok)) * heads + hk * groups + g;
  const size_t step = (size_t)total_tokens * heads;
  // eight runs a round, every load of a round issued before the first is used (the last round reads
  // the last run again where it has fewer; those copies get the weight zero)
  float m_tot = -INFINITY;
  for (int base = 0; base < splits; base += 8) {
    float ms[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) ms[j] = part_ml[(first + min(base + j, splits - 1) * step) * 2];
#pragma unroll
    for (int j = 0; j < 8; ++j) m_tot = fmaxf(m_tot, ms[j]);
  }
  float l = 0.f, acc[DPT];
#pragma unroll
  for (int i = 0; i < DPT; ++i) acc[i] = 0.f;
  for (int base = 0; base < splits; base += 8) {
    float2 ml[8];
    float part[8][DPT];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const size_t row = first + min(base + j, splits - 1) * step;
      ml[j] = *(const float2*)(part_ml + row * 2);
#pragma unroll
      for (int i = 0; i < DPT; ++i) part[j][i] = part_acc[row * D + min(c + 16 * i, D - 1)];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const bool counts = base + j < splits && ml[j].x > -INFINITY;
      const float f = counts ? (FAST_EXP ? __expf(ml[j].x - m_tot) : expf(ml[j].x - m_tot)) : 0.f;
      l = fmaf(f, ml[j].y, l);
#pragma unroll
      for (int i = 0; i < DPT; ++i) acc[i] = fmaf(f, part[j][i], acc[i]);
    }
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  T* orow = out + (size_t)(q0 + tok) * out_stride + (size_t)(hk * groups + g) * D;
#pragma unroll
  for (int i = 0; i < DPT; ++i)
    if (c + 16 * i < D) store_from_float(orow + c + 16 * i, acc[i] * inv);
}

// Paged grouped-query attention for steps in which every sequence brings one token, float32 cache: from the fused projection's raw
// output to the attention's output in one launch, as attention_decode.hip does it in bfloat16.
//
// Block = (key split, kv head, sequence); four waves take blocks of 16 keys in turn, keys and values through a slot of LDS that each
// wave has for one block (requests of whole lines, waits counted by hand).  Scores transposed, S^T = K Q^T, and output transposed,
// O^T = V^T P^T, on the float32 MFMA 16x16x4 with the group's query rows padded to 16: lane (r = l % 16, q = l / 16) supplies a
// key's dims 16 i + 4 q + e (of the keys and of the queries: which four dims an instruction takes does not matter), receives the scores of keys
// 4 q .. + 3 of row r, and these are, after the softmax, what it supplies to the second product.
//
// An error that grows with the length of a chain of sums is what separates this from the kernel for all sizes, whose dot products are trees over
// lanes: so a dot product is sixteen chains of D / 64 instructions, added up as a tree, a block's share of the output is summed from zero and joins the
// run's in one rounding, the exponent takes the scale and the maximum in one, and waves and splits are added up as trees too.  Relative error of 24 launches each of 1 to 8 sequences, 16 heads on
// 8, against 64 bits, the kernel for all sizes -> this: 60 to 200 keys 1.54e-7 -> 1.52e-7, 200 to 1,000 1.64 -> 1.61, 1,000 to 8,000 2.07 ->
// 1.84, with scores four times as large 2.69 -> 2.56, 3.52 -> 3.07, 4.15 -> 3.80.  Heads of 64, whose dot products are short (and whose shares are
// two chains for it), 8 on one, 1.34 -> 1.42, 1.54 -> 1.48, 1.96 -> 1.73, 2.52 -> 2.62, 2.77 -> 2.87, 3.66 -> 3.53.  (Dot products in four chains and
// everything else in a row: 1.95, 2.11, 2.67, 3.64, 4.40, 5.48 with heads of 128, and 4 sequences of 90 to 600 keys 10.0 us where this
// takes 10.3, 1 of 8,000 18.6 and 19.5.)
//
// On the way the block's heads are normalised and rotated, in the arithmetic of the stand-alone kernel (rope_math.h), four elements a
// lane, and the last split's last wave writes the new key and value to their pages and treats them as a partial result of their own.
// The block that finishes last among a (sequence, head)'s splits merges them, eight splits' loads a round, behind a counter as in
// attention_decode.hip.
//
// Bound by latency where contexts are short (start, keys and values, merge one after the other), by the cache's bytes where they are long.
// What it saves are two launches and the trips between them (rotation 4.8, attention 9 and its merge 6.6 us at 4 sequences of 90 to 600
// keys): float32 steps of 1.7B at 4 requests of 90 to 600 tokens 2,090 -> 1,845 us, at 1 of 8,000 2,684 -> 2,089, of 0.6B at 1 of 217 1,349 -> 1,151, 8 of 300 to 800
// 1,714 -> 1,406, 2 of 2,000 to 4,000 2,117 -> 1,422.
#include "agent_access.h"
#include "common.h"
#include "lds_load.h"
#include "lds_tile.h"
#include "rope_math.h"
#include <type_traits>

namespace {

using lds_tile::floatx4;
using lds_tile::uintx4;

constexpr int KEYS = 16, WAVES = 4, GMAX = 8;
constexpr int CHAINS = 16;      // that a dot product is summed in
constexpr int ROUND = 8;        // splits that the merge reads at a time

template <int D>
struct Slot {
  static constexpr int LPH = D / 4;                                  // lanes that share a head
  static constexpr int ROUNDS = ((GMAX + 2) * LPH + 255) / 256;      // how often the block's lanes take heads
  static constexpr int LOADS = D / 16;                               // requests of 1,024 bytes: a block's keys, and its values
  static constexpr int SHARES = D == 64 ? 2 : 1;                     // chains that a block's share of the output is summed in
  static constexpr int VALUES_AT = LOADS * 1024, BYTES = 2 * VALUES_AT;      // the heads come to the values' place before them
  static_assert(ROUNDS <= LOADS, "heads in the values' place");
};

struct Heads {
  const float *q_weight, *k_weight, *inv_freq;      // the norms' weights (null: no norm), the rotation's frequencies [D / 2]
  float eps;
};

// PAST: values are loaded past the caches (pages of 16: a block's values are whole lines that one wave reads)
template <int D, bool PAST>
__global__ __launch_bounds__(256, 2) void paged_decode_f32_kernel(
    const float* __restrict__ qkv, long long q_stride, Heads how, float* key_pages, float* value_pages, float* __restrict__ out,
    long long out_stride, float* part_o, float* part_ml, int* __restrict__ counters, const int* __restrict__ cu_q,
    const int* __restrict__ ctx_len, const int* __restrict__ block_table, int table_stride, int kv_heads, int groups, int block_shift,
    int num_blocks, int window, float scale) {
  using S = Slot<D>;
  constexpr int LPH = S::LPH, ROUNDS = S::ROUNDS, LOADS = S::LOADS, DT = D / 16;
  constexpr int CPR = D / 4, RPI = 64 / CPR;         // 16-byte chunks of a key, keys of a request
  constexpr int PITCH = D + 4;                       // of a finished head in LDS
  extern __shared__ __attribute__((aligned(16))) uintx4 slots[];      // [WAVES] S::BYTES
  __shared__ float Ms[WAVES + 1][GMAX], Ls[WAVES][GMAX];
  __shared__ float cos_s[D / 2], sin_s[D / 2];
  __shared__ __attribute__((aligned(16))) float heads_s[(GMAX + 2) * PITCH];      // queries, the new key, the new value
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lq = lane >> 4;
  const int seq = blockIdx.z, hk = blockIdx.y;

  float frequency = how.inv_freq[max(tid - (256 - D / 2), 0)];       // the last threads': the first ones have heads
  float4 head_w[ROUNDS];
#pragma unroll
  for (int round = 0; round < ROUNDS; ++round)      // (without a norm: any valid address, not used)
    head_w[round] = *(const float4*)(how.q_weight ? ((tid + round * 256) / LPH < groups ? how.q_weight : how.k_weight) + (tid & (LPH - 1)) * 4 : how.inv_freq);
  const int q0 = cu_q[seq], ctx = ctx_len[seq];
  if (cu_q[seq + 1] - q0 != 1 || ctx < 1) return;
  const int cached = ctx - 1;                        // keys that come from the pages
  const int k_begin = window > 0 ? max(0, ctx - window) : 0, first = k_begin / KEYS, last = (cached + KEYS - 1) / KEYS;
  // two blocks a wave need no splits, and no merge
  const int split = blockIdx.x, splits = last - first <= 2 * WAVES ? 1 : gridDim.x;
  if (split >= splits) return;
  const size_t first_part = ((size_t)seq * kv_heads) * gridDim.x + (size_t)hk * splits;
  const int per_split = (last - first + splits - 1) / splits;
  const int my_first = first + split * per_split, my_last = min(last, my_first + per_split);
  uintx4* const slot = slots + wave * (S::BYTES / 16);
  const unsigned int slot_at = __builtin_amdgcn_readfirstlane((unsigned int)(size_t)(const __attribute__((address_space(3))) char*)slot);

  const int block_mask = (1 << block_shift) - 1, table_last = table_stride - 1;
  const int* table = block_table + (size_t)seq * table_stride;
  auto raw_page = [&](int key) -> int { return table[min(key >> block_shift, table_last)]; };
  auto page_of = [&](int b) -> int {                 // a block lies in one page; behind the context maybe in none: page 0 then, masked
    const int id = raw_page(b * KEYS);
    return id >= 0 && id < num_blocks ? id : 0;
  };
  // Keys: a request takes whole rows, chunk p of row r to position p ^ (r % 8), so that the lanes that a read of LDS serves in one
  // cycle hit different banks.
  const int load_row = lane / CPR, load_at = (load_row * D + ((lane & (CPR - 1)) ^ load_row) * 4) * 4;
  auto request_keys = [&](int b, int page) {
    const char* from = (const char*)(key_pages + ((((size_t)page * kv_heads + hk) << block_shift) + ((b * KEYS) & block_mask)) * D);
#pragma unroll
    for (int j = 0; j < LOADS; ++j)
      lds_load::load_to_lds_once(from + j * 1024, load_at ^ ((j * RPI & 7) * 16), slot_at + j * 1024);
  };
  // Values: lane (lr = dim, lq) takes the four keys 4 lq .. + 3 of dims 16 t + lr from the transposed page.
  auto request_values = [&](int b, int page) {
    const float* from = value_pages + ((((size_t)page * kv_heads + hk) * D + lr) << block_shift) + ((b * KEYS) & block_mask) + 4 * lq;
#pragma unroll
    for (int t = 0; t < LOADS; ++t) {
      const float* at = from + ((size_t)(t * 16) << block_shift);
      if constexpr (PAST) lds_load::load_to_lds_once(at, slot_at + S::VALUES_AT + t * 1024);
      else lds_load::load_to_lds(at, slot_at + S::VALUES_AT + t * 1024);
    }
  };
  auto reads_done = []() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };

  // All requests from here to the end of the loop are counted by hand: the compiler's own loads have arrived.
  asm volatile("" : "+v"(frequency));
#pragma unroll
  for (int round = 0; round < ROUNDS; ++round)
    asm volatile("" : "+v"(head_w[round].x), "+v"(head_w[round].y), "+v"(head_w[round].z), "+v"(head_w[round].w));
  int b = my_first + wave;
  const bool has_keys = b < my_last;
  int next = page_of(b);
  const int new_page = raw_page(cached);
#pragma unroll
  for (int round = 0; round < ROUNDS; ++round) {
    if (round * 256 + wave * 64 >= (groups + 2) * LPH) break;
    const int head = min((tid + round * 256) / LPH, groups + 1);
    const int column = (head < groups ? hk * groups + head : kv_heads * groups + (head - groups) * kv_heads + hk) * D + (tid & (LPH - 1)) * 4;
    lds_load::load_to_lds(qkv + (size_t)q0 * q_stride + column, slot_at + S::VALUES_AT + round * 1024);
  }
  if (has_keys) {
    request_keys(b, next);
    lds_tile::wait_loads<LOADS>();
  } else {
    lds_tile::wait_loads<0>();
  }
  float4 raw[ROUNDS];
#pragma unroll
  for (int round = 0; round < ROUNDS; ++round) raw[round] = __builtin_bit_cast(float4, slot[S::VALUES_AT / 16 + round * 64 + lane]);
  reads_done();
  if (has_keys) request_values(b, next);
  next = page_of(b + WAVES);

  // The rotation's cosines and sines once a block, the heads four elements a lane.
  if (tid >= 256 - D / 2) {
    float sn, cs;
    sincosf((float)cached * frequency, &sn, &cs);
    cos_s[tid - (256 - D / 2)] = cs;
    sin_s[tid - (256 - D / 2)] = sn;
  }
  float v[ROUNDS][4];
#pragma unroll
  for (int round = 0; round < ROUNDS; ++round) {
    v[round][0] = raw[round].x; v[round][1] = raw[round].y; v[round][2] = raw[round].z; v[round][3] = raw[round].w;
    if (how.q_weight) {
      float sumsq = __fmaf_rn(v[round][3], v[round][3], __fmaf_rn(v[round][2], v[round][2], __fmaf_rn(v[round][1], v[round][1], v[round][0] * v[round][0])));
#pragma unroll
      for (int offset = LPH / 2; offset > 0; offset >>= 1) sumsq += __shfl_xor(sumsq, offset, FE_WAVE);
      const float inv = inverse_rms(sumsq, D, how.eps);
      const float w4[4] = {head_w[round].x, head_w[round].y, head_w[round].z, head_w[round].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) v[round][e] = normalise(v[round][e], inv, w4[e]);
    }
  }
  __syncthreads();        // cos_s, sin_s (the keys and values requested above stay in flight)
#pragma unroll
  for (int round = 0; round < ROUNDS; ++round) {
    const int head = (tid + round * 256) / LPH, sub = tid & (LPH - 1);
    const bool low = sub * 4 < D / 2;
    float r[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float other = __shfl_xor(v[round][e], LPH / 2, FE_WAVE);
      const int j = (sub * 4 + e) & (D / 2 - 1);
      r[e] = low ? rotate_low(v[round][e], other, cos_s[j], sin_s[j]) : rotate_high(v[round][e], other, cos_s[j], sin_s[j]);
    }
    if (head < groups + 2) *(float4*)&heads_s[head * PITCH + sub * 4] = head == groups + 1 ? raw[round] : make_float4(r[0], r[1], r[2], r[3]);
  }
  __syncthreads();
  floatx4 qb[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) qb[i] = *(const floatx4*)&heads_s[(lr < groups ? lr : 0) * PITCH + 16 * i + 4 * lq];

  // The new token's key and value, in the last wave of the last split: score q.k_new, weight 1, value v_new.
  const bool extra = split == splits - 1;
  float4 fresh = {0.f, 0.f, 0.f, 0.f};      // four elements of the new key (lanes below LPH) or of the new value (the LPH after them)
  if (extra && wave == WAVES - 1) {
    if (lane < 2 * LPH) fresh = *(const float4*)&heads_s[(groups + lane / LPH) * PITCH + (lane & (LPH - 1)) * 4];
    float dot[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const floatx4 k4 = *(const floatx4*)&heads_s[groups * PITCH + 16 * i + 4 * lq];
#pragma unroll
      for (int e = 0; e < 4; ++e) dot[e] = __fmaf_rn(qb[i][e], k4[e], dot[e]);
    }
    const float score = sum_xor32(sum_xor16((dot[0] + dot[1]) + (dot[2] + dot[3])));
    if (lq == 0 && lr < groups) Ms[WAVES][lr] = score * scale;
  }
  // (behind the last load that this wave waits for, whose count the stores would be in)
  auto write_pages = [&]() {
    if (!extra || wave != WAVES - 1 || lane >= 2 * LPH || new_page < 0 || new_page >= num_blocks) return;   // (the host reserves pages before the launch)
    const int sub = lane & (LPH - 1), at = cached & block_mask;
    const size_t page = (size_t)new_page * kv_heads + hk;
    if (lane < LPH) {
      *(float4*)(key_pages + ((page << block_shift) + at) * D + sub * 4) = fresh;
    } else {
      float* to = value_pages + ((page * D) << block_shift) + at;
      const float f4[4] = {fresh.x, fresh.y, fresh.z, fresh.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) to[(size_t)(sub * 4 + e) << block_shift] = f4[e];
    }
  };

  float m_run = -INFINITY, l_run = 0.f;   // of query row lr (the same in the four lanes that share it)
  floatx4 o[DT];                          // O^T: dims 16 t + 4 lq + i of query row lr
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (; b < my_last; b += WAVES) {
    const bool goes_on = b + WAVES < my_last;
    lds_tile::wait_loads<LOADS>();        // the keys; behind them only this block's values are under way
    floatx4 k4[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) k4[i] = __builtin_bit_cast(floatx4, slot[lr * CPR + ((4 * i + lq) ^ (lr & 7))]);
    reads_done();
    if (goes_on) request_keys(b + WAVES, next);
    floatx4 st[CHAINS];
#pragma unroll
    for (int c = 0; c < CHAINS; ++c) st[c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        floatx4& sum = st[(4 * i + e) % CHAINS];
        sum = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[i][e], qb[i][e], sum, 0, 0, 0);
      }
    // lane (lr = query row, lq): score of key b * 16 + 4 lq + i
#pragma unroll
    for (int half = CHAINS / 2; half > 0; half >>= 1)
#pragma unroll
      for (int c = 0; c < half; ++c) st[c] += st[c + half];
    const floatx4 scores = st[0];
    const int key0 = b * KEYS + 4 * lq;
    float s[4], mx = -INFINITY;
    bool owned[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      owned[i] = key0 + i >= k_begin && key0 + i < cached;
      s[i] = owned[i] ? scores[i] * scale : -INFINITY;
      mx = fmaxf(mx, s[i]);
    }
    mx = max_xor32(max_xor16(mx));
    const float m_new = fmaxf(m_run, mx), m_use = m_new > -INFINITY ? m_new : 0.f;
    const float corr = expf(m_run - m_use);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s[i] = owned[i] ? expf(fmaf(scores[i], scale, -m_use)) : 0.f;
      sum += s[i];
    }
    l_run = fmaf(l_run, corr, sum_xor32(sum_xor16(sum)));
    m_run = m_new;
    if (goes_on) lds_tile::wait_loads<LOADS>();      // the values; behind them only the next block's keys
    else lds_tile::wait_loads<0>();
    floatx4 va[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) va[t] = __builtin_bit_cast(floatx4, slot[S::VALUES_AT / 16 + t * 64 + lane]);
    reads_done();
    if (goes_on) {
      request_values(b + WAVES, next);
      next = page_of(b + 2 * WAVES);
    }
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      floatx4 share[S::SHARES];
#pragma unroll
      for (int i = 0; i < S::SHARES; ++i) share[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) {     // slots that no key in reach owns may hold anything: their values count as zero
        floatx4& sum = share[i * S::SHARES / 4];
        sum = __builtin_amdgcn_mfma_f32_16x16x4f32(owned[i] ? va[t][i] : 0.f, s[i], sum, 0, 0, 0);
      }
      if constexpr (S::SHARES == 2) share[0] += share[1];
#pragma unroll
      for (int i = 0; i < 4; ++i) o[t][i] = fmaf(o[t][i], corr, share[0][i]);
    }
  }
  if (splits == 1) write_pages();

  // lane (lr = query row, lq) holds O^T[16 t + 4 lq + i][lr]; the four waves meet in LDS, each in its own slot
  if (lr < groups) {
#pragma unroll
    for (int t = 0; t < DT; ++t) *(floatx4*)((float*)slot + lr * D + t * 16 + lq * 4) = o[t];
    if (lq == 0) { Ms[wave][lr] = m_run; Ls[wave][lr] = l_run; }
  }
  __syncthreads();
  for (int e = tid; e < groups * D; e += 256) {
    const int g = e / D, d = e - g * D;
    float m_tot = extra ? Ms[WAVES][g] : -INFINITY;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) m_tot = fmaxf(m_tot, Ms[w][g]);
    float ov = 0.f, l = 0.f;
    if (m_tot > -INFINITY) {
      float f[WAVES], part[WAVES];
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        f[w] = expf(Ms[w][g] - m_tot);
        part[w] = ((const float*)(slots + w * (S::BYTES / 16)))[g * D + d];
      }
      ov = fmaf(f[0], part[0], f[1] * part[1]) + fmaf(f[2], part[2], f[3] * part[3]);
      l = fmaf(f[0], Ls[0][g], f[1] * Ls[1][g]) + fmaf(f[2], Ls[2][g], f[3] * Ls[3][g]);
      if (extra) {
        const float f = expf(Ms[WAVES][g] - m_tot);
        ov += f * heads_s[(groups + 1) * PITCH + d];
        l += f;
      }
    }
    if (splits == 1) {
      out[(size_t)q0 * out_stride + (size_t)(hk * groups + g) * D + d] = l > 0.f ? ov / l : 0.f;
    } else {
      const size_t at = (first_part + split) * groups + g;
      store_agent(&part_o[at * D + d], ov);
      if (d == 0) {
        store_agent(&part_ml[at * 2], m_tot);
        store_agent(&part_ml[at * 2 + 1], l);
      }
    }
  }
  if (splits == 1) return;

  // The block that counts itself in last merges (attention_decode.hip states what orders the parts before the count).
  __shared__ int is_last;
  __builtin_amdgcn_s_waitcnt((0x0) | (0x7 << 4) | (0xF << 8));    // vmcnt(0): this wave's stores have been acknowledged
  __syncthreads();
  if (tid == 0) {
    int* counter = counters + (size_t)seq * kv_heads + hk;
    is_last = atomicAdd(counter, 1) == splits - 1;
    if (is_last) atomicExch(counter, 0);
  }
  __syncthreads();
  if (is_last) {
    for (int e = tid; e < groups * D; e += 256) {
      const int g = e / D, d = e - g * D;
      float m_tot = -INFINITY, l_tot = 0.f, ov = 0.f;
      for (int base = 0; base < splits; base += ROUND) {
        float m[ROUND], l[ROUND], part[ROUND];
#pragma unroll
        for (int i = 0; i < ROUND; ++i) {
          const size_t at = (first_part + min(base + i, splits - 1)) * groups + g;
          m[i] = load_agent(&part_ml[at * 2]);
          l[i] = load_agent(&part_ml[at * 2 + 1]);
          part[i] = load_agent(&part_o[at * D + d]);
        }
        float m_new = m_tot;
#pragma unroll
        for (int i = 0; i < ROUND; ++i) m_new = fmaxf(m_new, m[i]);
        const float m_use = m_new > -INFINITY ? m_new : 0.f, corr = expf(m_tot - m_use);
#pragma unroll
        for (int i = 0; i < ROUND; ++i) {
          const float f = base + i < splits ? expf(m[i] - m_use) : 0.f;
          l[i] *= f;
          part[i] *= f;
        }
#pragma unroll
        for (int half = ROUND / 2; half > 0; half >>= 1)
#pragma unroll
          for (int i = 0; i < half; ++i) {
            l[i] += l[i + half];
            part[i] += part[i + half];
          }
        l_tot = fmaf(l_tot, corr, l[0]);
        ov = fmaf(ov, corr, part[0]);
        m_tot = m_new;
      }
      out[(size_t)q0 * out_stride + (size_t)(hk * groups + g) * D + d] = l_tot > 0.f ? ov / l_tot : 0.f;
    }
  }
  write_pages();
}

}  // namespace

// A step in which every sequence brings one token: qkv [num_seqs rows of (kv_heads * groups + 2 * kv_heads) * head_dim, row stride
// q_stride] float32; q and k heads are normalised (weights [head_dim], null: no norm) and rotated whole by position ctx_len - 1 (inv_freq
// [head_dim / 2]), each sequence's new key and value are written to slot ctx_len - 1 of its pages, and its attention over them to out.
// Pages: keys [blocks][kv_heads][block_size][D], values transposed [blocks][kv_heads][D][block_size]; head_dim 64 or 128, block_size a power of
// two >= 16.  splits > 1 (at most 64) needs part_o [num_seqs * kv_heads * splits * groups * head_dim] and part_ml [num_seqs * kv_heads *
// splits * groups * 2] floats, and counters [num_seqs * kv_heads]: ints that are zero before the first launch; every launch leaves them
// zero again.  Launches that share counters must not overlap.
extern "C" int fe_paged_attention_decode_f32(const float* qkv, long long q_stride, const float* q_weight, const float* k_weight,
                                             const float* inv_freq, float eps, float* key_pages, float* value_pages, float* out,
                                             long long out_stride, float* part_o, float* part_ml, int* counters, const int* cu_q,
                                             const int* ctx_len, const int* block_table, int table_stride, int num_seqs, int kv_heads,
                                             int groups, int head_dim, int block_size, int num_blocks, int window, float scale, int splits,
                                             hipStream_t stream) {
  if (num_seqs <= 0) return FE_OK;
  if (!inv_freq || (!q_weight) != (!k_weight) || (head_dim != 64 && head_dim != 128)) return FE_BAD_ARGUMENT;
  if (groups < 1 || groups > GMAX || kv_heads < 1 || kv_heads > 65535 || num_seqs > 65535) return FE_BAD_ARGUMENT;
  if (block_size < 16 || (block_size & (block_size - 1)) || num_blocks < 1 || table_stride < 1) return FE_BAD_ARGUMENT;
  if (splits < 1 || splits > 64 || (splits > 1 && (!part_o || !part_ml || !counters))) return FE_BAD_ARGUMENT;
  if (q_stride % 4 || q_stride < (long long)(kv_heads * groups + 2 * kv_heads) * head_dim) return FE_BAD_ARGUMENT;
  if ((((uintptr_t)qkv) | ((uintptr_t)key_pages) | ((uintptr_t)value_pages) | ((uintptr_t)inv_freq) | ((uintptr_t)q_weight) | ((uintptr_t)k_weight)) & 15)
    return FE_BAD_ARGUMENT;
  int block_shift = 0;
  while ((1 << block_shift) < block_size) ++block_shift;
  const Heads how = {q_weight, k_weight, inv_freq, eps};
  const dim3 grid(splits, kv_heads, num_seqs);
#define FE_GO(D, PAST)                                                                                                             \
  do {                                                                                                                             \
    static std::atomic<bool> raised{false};                                                                                        \
    auto kernel = paged_decode_f32_kernel<D, PAST>;                                                                                \
    constexpr int lds_bytes = WAVES * Slot<D>::BYTES;                                                                              \
    const int limit_raised = lds_tile::raise_lds_limit((const void*)kernel, lds_bytes, &raised);                                   \
    if (limit_raised != FE_OK) return limit_raised;                                                                                \
    kernel<<<grid, 256, lds_bytes, stream>>>(qkv, q_stride, how, key_pages, value_pages, out, out_stride, part_o, part_ml, counters, \
                                             cu_q, ctx_len, block_table, table_stride, kv_heads, groups, block_shift, num_blocks,  \
                                             window, scale);                                                                       \
  } while (0)
  if (head_dim == 64) {
    if (block_size == 16) FE_GO(64, true);
    else FE_GO(64, false);
  } else {
    if (block_size == 16) FE_GO(128, true);
    else FE_GO(128, false);
  }
#undef FE_GO
  return fe_check_launch();
}

// A mixture of experts on the device: routing, the sort of (token, choice) pairs by expert, and
// two grouped matrix products over the sorted rows.  Nothing is decided on the host.
//
//   fe_moe_select:   from router logits (float32): bias added, the `top` largest per token, softmax over those alone
//                    (or, scoring 1, each chosen logit's own sigmoid)
//   fe_moe_plan:     counts per expert, their prefix sums, and the pairs ordered by expert
//   fe_moe_select_plan: both for the few tokens of a decode step, in one launch
//   fe_moe_plan_table: the same where a table of token ids names every token's experts and no router is asked;
//                    also the pairs' weights, all alike
//   fe_moe_gate_up:  for every pair, act = min(g, L) * sigmoid(alpha min(g, L)) * (clamp(u, -L, L) + 1) with
//                    g = W_gate[e] x, u = W_up[e] x of the pair's token and expert (form 1: silu(g) * u; with
//                    input weights, g and u are first multiplied by the pair's routing weight); form 2: one matrix
//                    an expert, act = max(u, 0)^2
//   fe_moe_down:     out[choice][token] = weight * W_down[e] act   (float32; one part per choice, so
//                    that the reader adds a token's experts up in a fixed order; the first choice's part
//                    also takes what every token gets beside its experts, a shared expert's output)
//   fe_gated_act:    the same activation over a dense [T, 2F] product (a shared expert)
//
// The grouped products tile the sorted rows within an expert (a tile never spans two experts).  float32, and
// bfloat16 with K no multiple of 32: 32 rows x 64 columns a block, K through LDS in steps of 32, FMA.  bfloat16:
// MFMA 16x16x32 over tiles of 32 x 64 to 256 x 128 with rows and weight straight from memory in LDS.  A launch has as many row-tile slots as the pairs could need at worst (pairs /
// rows a tile + experts); a block whose slot lies beyond the tiles there are returns at once.
#include "common.h"
#include "gate_act.h"
#include "lds_tile.h"
#include <algorithm>

// One thread per token over its row of router logits z [T, E] (float32, the product comes from the
// caller): bias added, the `top` largest chosen one after the other (the largest first; among equals
// the lowest index), weights = softmax over the chosen logits alone.
__global__ void moe_select_kernel(const float* __restrict__ z, const float* __restrict__ bias, int* __restrict__ chosen,
                                  float* __restrict__ weights, int tokens, int E, int top, int scoring) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= tokens) return;
  const float* row = z + (size_t)t * E;
  int picked[16];
  float best[16], raw[16];
  float peak = 0.f, denom = 0.f;
  for (int k = 0; k < top; ++k) {
    int arg = -1;
    float value = -INFINITY;
    for (int e = 0; e < E; ++e) {
      bool taken = false;
      for (int j = 0; j < k; ++j) taken = taken || picked[j] == e;
      const float v = row[e] + (bias ? bias[e] : 0.f);
      if (!taken && (arg < 0 || v > value)) {
        value = v;
        arg = e;
      }
    }
    picked[k] = arg;
    chosen[(size_t)t * top + k] = arg;
    if (k == 0) peak = value;
    raw[k] = value;
    best[k] = expf(value - peak);
    denom += best[k];
  }
  // scoring 1: a chosen expert's weight is the sigmoid of its own logit, whatever the others are
  for (int k = 0; k < top; ++k)
    weights[(size_t)t * top + k] = scoring == 1 ? 1.f / (1.f + expf(-raw[k])) : best[k] / denom;
}

extern "C" int fe_moe_select(const float* logits, const float* bias, int* chosen, float* weights, int tokens, int experts,
                             int top, int scoring, hipStream_t stream) {
  if (tokens <= 0) return FE_OK;
  if (experts <= 0 || experts > 1024 || top < 1 || top > 16 || top > experts || scoring < 0 || scoring > 1) return FE_BAD_ARGUMENT;
  moe_select_kernel<<<(tokens + 63) / 64, 64, 0, stream>>>(logits, bias, chosen, weights, tokens, experts, top, scoring);
  return fe_check_launch();
}

// Selection by corrected scores within the best groups.  Per token: s = softmax(z) over all E experts; an
// expert's choice score is s_e + correction_e; the experts form `groups` equal runs of neighbours, a run's score is
// its largest choice score, and only experts of the `keep` best runs can be chosen (the lowest index among
// equals, for runs and for experts); the `top` largest choice scores among those are chosen, and their weights are
// their own s, divided by the sum of the chosen s (+ 1e-20), times `scale`.  The logits' rows lie `stride`
// floats apart (columns beyond E, a gate's logit say, are not read here).  One thread a token.
#define SELECT_MAX_GROUPS 64
__global__ void moe_select_grouped_kernel(const float* __restrict__ z, size_t stride, const float* __restrict__ correction,
                                          int* __restrict__ chosen, float* __restrict__ weights, int tokens, int E, int top,
                                          int groups, int keep, float scale) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= tokens) return;
  const float* row = z + (size_t)t * stride;
  float peak = -INFINITY;
  for (int e = 0; e < E; ++e) peak = fmaxf(peak, row[e]);
  float denom = 0.f;
  for (int e = 0; e < E; ++e) denom += expf(row[e] - peak);
  const float inv = 1.f / denom;
  auto score = [&](int e) { return expf(row[e] - peak) * inv; };
  auto choice = [&](int e) { return score(e) + (correction ? correction[e] : 0.f); };
  const int each = E / groups;
  unsigned long long open = ~0ull;          // bit g: run g may be chosen from
  if (keep < groups) {
    float best[SELECT_MAX_GROUPS];
    for (int g = 0; g < groups; ++g) {
      float b = -INFINITY;
      for (int e = g * each; e < (g + 1) * each; ++e) b = fmaxf(b, choice(e));
      best[g] = b;
    }
    open = 0ull;
    for (int k = 0; k < keep; ++k) {
      int arg = -1;
      float value = -INFINITY;
      for (int g = 0; g < groups; ++g)
        if (!((open >> g) & 1ull) && (arg < 0 || best[g] > value)) {
          value = best[g];
          arg = g;
        }
      open |= 1ull << arg;
    }
  }
  int picked[16];
  float own[16];
  float total = 0.f;
  for (int k = 0; k < top; ++k) {
    int arg = -1;
    float value = -INFINITY;
    for (int e = 0; e < E; ++e) {
      if (!((open >> (e / each)) & 1ull)) continue;
      bool taken = false;
      for (int j = 0; j < k; ++j) taken = taken || picked[j] == e;
      if (taken) continue;
      const float v = choice(e);
      if (arg < 0 || v > value) {
        value = v;
        arg = e;
      }
    }
    picked[k] = arg;
    own[k] = score(arg);
    total += own[k];
    chosen[(size_t)t * top + k] = arg;
  }
  const float norm = scale / (total + 1e-20f);
  for (int k = 0; k < top; ++k) weights[(size_t)t * top + k] = own[k] * norm;
}

extern "C" int fe_moe_select_grouped(const float* logits, long long stride, const float* correction, int* chosen,
                                     float* weights, int tokens, int experts, int top, int groups, int keep, float scale,
                                     hipStream_t stream) {
  if (tokens <= 0) return FE_OK;
  if (experts <= 0 || experts > 1024 || top < 1 || top > 16 || stride < experts || groups < 1 ||
      groups > SELECT_MAX_GROUPS || experts % groups || keep < 1 || keep > groups || top > (experts / groups) * keep)
    return FE_BAD_ARGUMENT;
  moe_select_grouped_kernel<<<(tokens + 63) / 64, 64, 0, stream>>>(logits, (size_t)stride, correction, chosen, weights, tokens,
                                                                   experts, top, groups, keep, scale);
  return fe_check_launch();
}

// One block: offsets[e] = pairs of experts below e, order[offsets[e] ..] = the pairs of expert e.
// Within an expert the pairs come in no fixed order; a pair's results do not depend on its row.
template <typename Choice>
__device__ __forceinline__ void plan_pairs(Choice choice, int pairs, int E, int* __restrict__ offsets, int* __restrict__ order) {
  extern __shared__ int counts[];   // [E] counts, then [E] cursors
  int* cursor = counts + E;
  for (int e = threadIdx.x; e < E; e += blockDim.x) counts[e] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < pairs; i += blockDim.x) {
    const int e = choice(i);
    if (e >= 0 && e < E) atomicAdd(&counts[e], 1);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int sum = 0;
    for (int e = 0; e < E; ++e) {
      offsets[e] = cursor[e] = sum;
      sum += counts[e];
    }
    offsets[E] = sum;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < pairs; i += blockDim.x) {
    const int e = choice(i);
    if (e >= 0 && e < E) order[atomicAdd(&cursor[e], 1)] = i;
  }
}

__global__ __launch_bounds__(1024) void moe_plan_kernel(const int* __restrict__ chosen, int pairs, int E,
                                                        int* __restrict__ offsets, int* __restrict__ order) {
  plan_pairs([&](int i) { return chosen[i]; }, pairs, E, offsets, order);
}

// Pair i is choice i % top of token i / top: column i % top of the table's row for the token's id.
__global__ __launch_bounds__(1024) void moe_plan_table_kernel(const int* __restrict__ ids, const int* __restrict__ table, int vocab,
                                                              int top, int pairs, int E, int* __restrict__ offsets,
                                                              int* __restrict__ order, float* __restrict__ weights, float weight) {
  plan_pairs([&](int i) {
    const int id = ids[i / top];
    return table[(size_t)(id >= 0 && id < vocab ? id : 0) * top + i % top];
  }, pairs, E, offsets, order);
  for (int i = threadIdx.x; i < pairs; i += blockDim.x) weights[i] = weight;
}

extern "C" int fe_moe_plan(const int* chosen, int pairs, int experts, int* offsets, int* order, hipStream_t stream) {
  if (pairs <= 0) return FE_OK;
  if (experts <= 0 || experts > 1024) return FE_BAD_ARGUMENT;
  moe_plan_kernel<<<1, 1024, 2 * (size_t)experts * sizeof(int), stream>>>(chosen, pairs, experts, offsets, order);
  return fe_check_launch();
}

// ids [tokens]; table [vocab][top] (expert numbers below `experts`); weights [tokens][top] all become `weight`
extern "C" int fe_moe_plan_table(const int* ids, const int* table, int vocab, int tokens, int top, int experts, int* offsets,
                                 int* order, float* weights, float weight, hipStream_t stream) {
  if (tokens <= 0) return FE_OK;
  if (experts <= 0 || experts > 1024 || top < 1 || top > 16 || vocab < 1 || (long long)tokens * top > 0x7fffffffLL) return FE_BAD_ARGUMENT;
  moe_plan_table_kernel<<<1, 1024, 2 * (size_t)experts * sizeof(int), stream>>>(ids, table, vocab, top, tokens * top, experts,
                                                                               offsets, order, weights, weight);
  return fe_check_launch();
}

// fe_moe_select and fe_moe_plan for the few tokens of a decode step, in one block (here the pairs of an expert come in order): two launches
// that are latency alone otherwise.  A thread a token chooses, from LDS, as moe_select_kernel does and with its bits; then a thread a pair
// counts the pairs before it.  8 tokens, 2 of 8 experts each, in a captured step 5.3 -> 3.1 us; 64 tokens, 4 of 32 25.7 -> 13.4.
constexpr int STEP_TOKENS = 64, STEP_EXPERTS = 64, STEP_PAIRS = 256;

__global__ __launch_bounds__(512) void moe_select_plan_kernel(const float* __restrict__ z, const float* __restrict__ bias, int* __restrict__ offsets,
                                                              int* __restrict__ order, float* __restrict__ weights, int tokens, int E, int top,
                                                              int scoring) {
  __shared__ float logits[STEP_TOKENS][STEP_EXPERTS + 1];
  __shared__ int picked[STEP_PAIRS];
  const int tid = threadIdx.x, pairs = tokens * top;
  for (int i = tid; i < tokens * E; i += 512) logits[i / E][i % E] = z[i] + (bias ? bias[i % E] : 0.f);
  __syncthreads();
  if (tid < tokens) {
    unsigned long long taken = 0;
    float best[16], raw[16], peak = 0.f, denom = 0.f;
    for (int k = 0; k < top; ++k) {
      int arg = -1;
      float value = -INFINITY;
      for (int e = 0; e < E; ++e) {
        const float v = logits[tid][e];
        if (!(taken >> e & 1) && (arg < 0 || v > value)) {
          value = v;
          arg = e;
        }
      }
      taken |= 1ull << arg;
      picked[tid * top + k] = arg;
      if (k == 0) peak = value;
      raw[k] = value;
      best[k] = expf(value - peak);
      denom += best[k];
    }
    for (int k = 0; k < top; ++k) weights[tid * top + k] = scoring == 1 ? 1.f / (1.f + expf(-raw[k])) : best[k] / denom;
  }
  __syncthreads();
  if (tid < pairs) {
    const int mine = picked[tid];
    int at = 0;
    for (int j = 0; j < pairs; ++j) at += picked[j] < mine || (picked[j] == mine && j < tid);
    order[at] = tid;
  } else if (tid >= STEP_PAIRS && tid - STEP_PAIRS <= E) {
    int below = 0;
    for (int j = 0; j < pairs; ++j) below += picked[j] < tid - STEP_PAIRS;
    offsets[tid - STEP_PAIRS] = below;
  }
}

// logits [tokens][experts] float32, contiguous, of up to 64 tokens and 64 experts, at most 256 pairs; offsets [experts + 1], order [tokens * top]
extern "C" int fe_moe_select_plan(const float* logits, const float* bias, int* offsets, int* order, float* weights, int tokens, int experts,
                                  int top, int scoring, hipStream_t stream) {
  if (tokens <= 0) return FE_OK;
  if (tokens > STEP_TOKENS || experts < 1 || experts > STEP_EXPERTS || top < 1 || top > 16 || top > experts || tokens * top > STEP_PAIRS ||
      scoring < 0 || scoring > 1)
    return FE_BAD_ARGUMENT;
  moe_select_plan_kernel<<<1, 512, 0, stream>>>(logits, bias, offsets, order, weights, tokens, experts, top, scoring);
  return fe_check_launch();
}

#define CUS 256
#define BM 32
#define BN 64
#define BK 32

// form 0: the bounded activation above; form 1: silu(g) * u; form 2: max(g, 0)^2.  `w` scales both products first (a router's weight
// on the expert's input: W (w x) = w (W x)).
__device__ __forceinline__ float gated(float g, float u, float limit, float alpha, int form, float w) {
  g *= w;
  u *= w;
  if (form == 2) return fmaxf(g, 0.f) * fmaxf(g, 0.f);      // one matrix an expert: g alone
  if (form == 1) return g / (1.f + expf(-g)) * u;
  return gate_bounded(g, u, limit, alpha);
}

// A token's first choice also takes what every token gets beside its experts (a shared expert's output,
// float32 [parts][tokens][N], added up in order first).
__device__ __forceinline__ float with_extra(float v, int choice, const float* __restrict__ extra, int parts,
                                            size_t part_stride, size_t at) {
  if (choice != 0 || !extra) return v;
  float sum = extra[at];
  for (int p = 1; p < parts; ++p) sum += extra[p * part_stride + at];
  return v + sum;
}

// The expert and the first sorted row of this block's row tile; false if the slot is beyond the tiles.
template <int ROWS = BM>
__device__ __forceinline__ bool find_tile(const int* __restrict__ offsets, int E, int slot, int& expert, int& row0,
                                          int& row_end) {
  int tiles = 0;
  for (int e = 0; e < E; ++e) {
    const int begin = offsets[e], end = offsets[e + 1];
    const int mine = (end - begin + ROWS - 1) / ROWS;
    if (slot < tiles + mine) {
      expert = e;
      row0 = begin + (slot - tiles) * ROWS;
      row_end = end;
      return true;
    }
    tiles += mine;
  }
  return false;
}

// MODE 0: rows are tokens' x gathered through the sorted pairs, the weight is [E][2N][K] (gate rows, then
// up rows), the ending is the gated activation into act [pairs, N].  MODE 1: rows are act's sorted rows,
// the weight is [E][N][K], and the result times the pair's routing weight goes to out[choice][token][N].  MODE 2: as
// MODE 0 with one matrix an expert, [E][N][K].
template <typename T, int MODE>
__global__ __launch_bounds__(256) void moe_grouped_kernel(
    const T* __restrict__ a, const T* __restrict__ w, const int* __restrict__ offsets, const int* __restrict__ order,
    const float* __restrict__ pair_weight, T* __restrict__ act, float* __restrict__ out, int E, int N, int K, int top,
    int tokens, float limit, float alpha, int form, const float* __restrict__ extra, int extra_parts) {
  __shared__ float As[BM][BK + 1];
  __shared__ float Ws[BN][BK + 1];
  __shared__ float Us[MODE == 0 ? BN : 1][BK + 1];
  __shared__ int pair_of[BM];
  int expert, row0, row_end;
  if (!find_tile(offsets, E, blockIdx.x, expert, row0, row_end)) return;
  const int tid = threadIdx.x;
  const int n0 = blockIdx.y * BN;
  if (tid < BM) pair_of[tid] = row0 + tid < row_end ? order[row0 + tid] : -1;
  __syncthreads();
  const int ty = tid / 16, tx = tid % 16;
  float acc_g[2][4], acc_u[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc_g[i][j] = acc_u[i][j] = 0.f;
  const size_t w_rows = MODE == 0 ? 2 * (size_t)N : (size_t)N;
  const T* w_expert = w + (size_t)expert * w_rows * K;

  for (int k0 = 0; k0 < K; k0 += BK) {
    for (int e = tid; e < BM * BK; e += 256) {
      const int r = e / BK, k = e % BK;
      float v = 0.f;
      const int pair = pair_of[r];
      if (pair >= 0 && k0 + k < K) {
        const size_t src = MODE != 1 ? (size_t)(pair / top) : (size_t)(row0 + r);
        v = load_as_float(a + src * K + k0 + k);
      }
      As[r][k] = v;
    }
    for (int e = tid; e < BN * BK; e += 256) {
      const int n = e / BK, k = e % BK;
      const bool ok = n0 + n < N && k0 + k < K;
      Ws[n][k] = ok ? load_as_float(w_expert + (size_t)(n0 + n) * K + k0 + k) : 0.f;
      if (MODE == 0) Us[n][k] = ok ? load_as_float(w_expert + ((size_t)N + n0 + n) * K + k0 + k) : 0.f;
    }
    __syncthreads();
#pragma unroll 8
    for (int k = 0; k < BK; ++k) {
      const float a0 = As[ty * 2][k], a1 = As[ty * 2 + 1][k];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float wv = Ws[tx + 16 * j][k];
        acc_g[0][j] = fmaf(a0, wv, acc_g[0][j]);
        acc_g[1][j] = fmaf(a1, wv, acc_g[1][j]);
        if (MODE == 0) {
          const float uv = Us[tx + 16 * j][k];
          acc_u[0][j] = fmaf(a0, uv, acc_u[0][j]);
          acc_u[1][j] = fmaf(a1, uv, acc_u[1][j]);
        }
      }
    }
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = ty * 2 + i;
    const int pair = pair_of[r];
    if (pair < 0) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx + 16 * j;
      if (n >= N) continue;
      if (MODE != 1) {
        store_from_float(act + (size_t)(row0 + r) * N + n, gated(acc_g[i][j], acc_u[i][j], limit, alpha, form, pair_weight ? pair_weight[pair] : 1.f));
      } else {
        const int token = pair / top, choice = pair - token * top;
        out[((size_t)choice * tokens + token) * N + n] =
            with_extra(acc_g[i][j] * (pair_weight ? pair_weight[pair] : 1.f), choice, extra, extra_parts, (size_t)tokens * N, (size_t)token * N + n);
      }
    }
  }
}

// The same two products on the matrix cores, for bfloat16 with K a multiple of 32: the tile product of lds_tile.h, a tile's rows
// gathered through the sorted pairs, its weight rows the expert's; rows and weight go straight from memory into LDS, several
// steps of 64 ahead.  (MODE 0: a fragment of sixteen weight rows is eight gate rows and the eight up rows of the same columns.)
// Blocks go to the eight dies (XCDs, each with an L2 of its own) in turn by their index.  The row tiles of one expert
// under one column tile read the same part of the weight, so they are made neighbours in the order of work (the row
// slot runs fastest) and a die takes a run of that order: a weight tile comes from memory once for all its row tiles.
using lds_tile::floatx4;
using lds_tile::uintx4;

// find_tile by the lanes of a wave: experts 64 at a time, a lane one of them; every lane gets the answer, and whether the tile has all of the
// expert's rows
template <int ROWS>
__device__ __forceinline__ bool find_tile_by_lanes(const int* __restrict__ offsets, int E, int slot, int& expert, int& row0, int& row_end, bool& alone) {
  const int lane = threadIdx.x & 63;
  int before = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int e = min(e0 + lane, E - 1);
    const int begin = offsets[e], end = offsets[e + 1];
    int upto = e0 + lane < E ? (end - begin + ROWS - 1) / ROWS : 0;      // tiles of this lane's expert, then of all up to it
    const int mine = upto;
#pragma unroll
    for (int offset = 1; offset < 64; offset <<= 1) {
      const int below = __shfl_up(upto, offset, FE_WAVE);
      if (lane >= offset) upto += below;
    }
    const unsigned long long past = __ballot(slot < before + upto);
    if (past) {
      const int at = __ffsll((long long)past) - 1;
      expert = e0 + at;
      const int first = __shfl(begin, at, FE_WAVE), tile = slot - before - (__shfl(upto, at, FE_WAVE) - __shfl(mine, at, FE_WAVE));
      row0 = first + tile * ROWS;
      row_end = __shfl(end, at, FE_WAVE);
      alone = __builtin_amdgcn_readfirstlane(row_end - first) <= ROWS;
      return true;
    }
    before += __shfl(upto, 63, FE_WAVE);
  }
  return false;
}

// PAST: weight rows of experts whose pairs are one tile pass the caches.  That is worth it where the blocks are at least one a CU (both products,
// two choices a token, width 2,048, us: 8 tokens, 8 / 16 experts 53.0 -> 48.9 / 69.5 -> 64.9, 32 tokens 54.7 -> 51.8), not where one or two
// experts are a few dozen blocks, which only wait longer (1 token, 2,048 x 1,024 19.7 -> 20.8), nor where experts have more tiles, whose blocks
// share the rows (300 tokens 73.7 -> 75.3, by asking alone).
template <int MI, int NI, int WM, int WN, int KG, int STAGES, int MODE, bool PAST>
__global__ __launch_bounds__(64 * WM * WN * KG) void moe_lds_kernel(
    const bf16_t* __restrict__ a, const bf16_t* __restrict__ w, const int* __restrict__ offsets,
    const int* __restrict__ order, const float* __restrict__ pair_weight, bf16_t* __restrict__ act,
    float* __restrict__ out, int E, int N, int K, int top, int tokens, float limit, float alpha, int form,
    const float* __restrict__ extra, int extra_parts, int slots, int column_tiles) {
  constexpr int TILE_ROWS = 16 * MI * WM, TILE_COLS = 16 * NI * WN, COLUMNS = MODE == 0 ? TILE_COLS / 2 : TILE_COLS;
  extern __shared__ __attribute__((aligned(16))) uintx4 lds[];
  const int items = slots * column_tiles;
  const int per_die = (items + 7) / 8;
  const int item = (int)(blockIdx.x % 8) * per_die + (int)(blockIdx.x / 8);
  if (item >= items) return;
  int expert, row0, row_end;
  bool alone;
  if (!find_tile_by_lanes<TILE_ROWS>(offsets, E, item % slots, expert, row0, row_end, alone)) return;
  const int n0 = (item / slots) * COLUMNS;
  const bf16_t* w_expert = w + (size_t)expert * (MODE == 0 ? 2 * (size_t)N : (size_t)N) * K;
  auto row_of = [&](int row) -> const bf16_t* {      // rows beyond the expert's and columns beyond N: the last again, never stored
    if (row < TILE_ROWS) {
      const int sorted = min(row0 + row, row_end - 1);
      return a + (size_t)(MODE != 1 ? order[sorted] / top : sorted) * K;
    }
    const int j = row - TILE_ROWS;
    if (MODE == 0) return w_expert + ((size_t)min(n0 + (j >> 4) * 8 + (j & 7), N - 1) + ((j & 8) ? N : 0)) * K;
    return w_expert + (size_t)min(n0 + j, N - 1) * K;
  };
  floatx4 acc[MI][NI];
  if (!lds_tile::product<MI, NI, WM, WN, KG, STAGES, true>(lds, row_of, 0, (K + lds_tile::KSTEP - 1) / lds_tile::KSTEP, K, acc, PAST && alone)) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4, wm = wave % WM, wn = wave / WM;
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int row = row0 + (wm * MI + i) * 16 + r;
    const bool live = row < row_end;
    const int pair = live ? order[row] : 0;
    const float weight = pair_weight ? pair_weight[pair] : 1.f;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      if constexpr (MODE != 1) {
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // (MODE 0: lanes q = 0, 1 hold gate columns 4 q .. + 3 of the fragment's eight, lanes q = 2, 3 the up columns of lane - 32)
          float up = 0.f;
          if constexpr (MODE == 0)
            up = __uint_as_float(__builtin_amdgcn_permlane32_swap(__float_as_uint(acc[i][j][e]), __float_as_uint(acc[i][j][e]), false, false)[1]);
          y[e] = gated(acc[i][j][e], up, limit, alpha, form, weight);
        }
        const int n = n0 + (wn * NI + j) * (MODE == 0 ? 8 : 16) + 4 * (MODE == 0 ? q & 1 : q);
        if (!live || (MODE == 0 && q >= 2)) continue;
        bf16_t* to = act + (size_t)row * N + n;
        if (n + 3 < N && (N & 3) == 0 && ((uintptr_t)act & 7) == 0)
          *(uint2*)to = make_uint2((unsigned)float_to_bf16(y[0]) | ((unsigned)float_to_bf16(y[1]) << 16),
                                   (unsigned)float_to_bf16(y[2]) | ((unsigned)float_to_bf16(y[3]) << 16));
        else
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < N) to[e] = float_to_bf16(y[e]);
      } else {
        const int n = n0 + (wn * NI + j) * 16 + 4 * q;
        if (!live) continue;
        const int token = pair / top, choice = pair - token * top;
        float* to = out + ((size_t)choice * tokens + token) * N + n;
        floatx4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[e] = n + e < N ? with_extra(acc[i][j][e] * weight, choice, extra, extra_parts, (size_t)tokens * N, (size_t)token * N + n + e) : 0.f;
        if (n + 3 < N && (N & 3) == 0 && ((uintptr_t)out & 15) == 0) *(floatx4*)to = v;
        else
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < N) to[e] = v[e];
      }
    }
  }
}

template <int MI, int NI, int WM, int WN, int KG, int STAGES, int MODE>
static int launch_moe_tile(const bf16_t* a, const bf16_t* w, const int* offsets, const int* order, const float* pair_weight,
                           bf16_t* act, float* out, int experts, int N, int K, int top, int tokens, float limit, float alpha,
                           int form, const float* extra, int extra_parts, hipStream_t stream) {
  constexpr int TILE_ROWS = 16 * MI * WM, TILE_COLS = 16 * NI * WN, COLUMNS = MODE == 0 ? TILE_COLS / 2 : TILE_COLS;
  constexpr size_t bytes = lds_tile::Shape<MI, NI, WM, WN, KG, STAGES>::BYTES;
  const long long pairs = (long long)tokens * top, slots = pairs / TILE_ROWS + experts, tiles = ((long long)N + COLUMNS - 1) / COLUMNS;
  const long long blocks = (slots * tiles + 7) / 8 * 8;
  if (blocks > 0x7fffffffLL) return FE_BAD_ARGUMENT;
  static std::atomic<bool> raised[2];
  const bool past = std::min<long long>(experts, pairs) * tiles >= CUS && pairs <= (long long)experts * TILE_ROWS;
  auto kernel = past ? moe_lds_kernel<MI, NI, WM, WN, KG, STAGES, MODE, true> : moe_lds_kernel<MI, NI, WM, WN, KG, STAGES, MODE, false>;
  const int limit_raised = lds_tile::raise_lds_limit((const void*)kernel, bytes, &raised[past]);
  if (limit_raised != FE_OK) return limit_raised;
  kernel<<<(unsigned)blocks, 64 * WM * WN * KG, bytes, stream>>>(a, w, offsets, order, pair_weight, act, out, experts, N, K, top, tokens,
                                                                 limit, alpha, form, extra, extra_parts, (int)slots, (int)tiles);
  return fe_check_launch();
}

// Which tile (rows x weight rows) a launch takes, by the rows an expert gets on average: few rows want many blocks with deep
// buffers, each streaming its part of the weight (what bounds them is the weight's bytes), many rows want every weight row read
// for more of them (what bounds them is the lines that a CU's L1 can wait for, see gemm_lds.h).  Measured on one MI355X, both
// products and the plan, us, 8 experts as wide as the model, 2 a token (weight straight in registers, or staged through them
// from 1,024 pairs on -> this): width 2,048 with 1 / 8 / 32 / 100 / 300 / 1,500 / 3,000 tokens 40 -> 26, 57 -> 48, 85 -> 56,
// 93 -> 64, 98 -> 77, 228 -> 141, 379 -> 270; width 1,024 25 -> 18, 27 -> 19, 28 -> 22, 30 -> 23, 35 -> 27, 73 -> 63, 132 -> 100.
// At 300 tokens (75 rows an expert) 64 x 64 takes 27 and 77 us, 64 x 128 31 and 72, 32 x 64 32 and 89; at 1,500 (375 rows)
// 64 x 128 61 and 165, 128 x 128 76 and 199, 256 x 128 63 and 141.
// The largest tile also wants steps enough for its start (its three buffers filled, 256 gathered rows) and blocks for most of the
// CUs: 1,024 x 3,072 of 4 experts at 1,100 tokens, 240 blocks, gate/up 59 us in 256 x 128 against 39 in 64 x 128; 512 x 1,536 at 2,048
// tokens 49 against 30; 2,048 x 2,048 down at 1,500 tokens 41 in the large tile against 53.  And where the smaller tile's blocks
// still leave half the chip idle it is the faster one at any number of rows: 64 x 64 of 4 experts at 400 tokens 6.3 us in 32 x 64, 8.0
// in 64 x 64, 11.3 in 64 x 128.  (Over 1,995 sizes of both products against the kernels before: 1.38 times as fast; at widths of
// 256 and 512 with many tokens those were up to a quarter faster.)
// Returned: 1,000 times the tile's rows + its weight rows.  gated: gate and up rows share a tile's weight rows (MODE 0).
extern "C" int fe_moe_tile(int gated, int tokens, int top, int experts, int N, int K) {
  const long long pairs = (long long)tokens * top, each = pairs / experts;
  // blocks that have work, if the experts share the pairs evenly
  auto busy = [&](int rows, int weight_rows) {
    const int columns = gated ? weight_rows / 2 : weight_rows;
    return (pairs + (long long)rows * experts - 1) / ((long long)rows * experts) * std::min((long long)experts, pairs) * ((N + columns - 1) / columns);
  };
  const int half_the_chip = 128;
  if (each >= 256 && K >= (gated ? 2048 : 768) && busy(256, 128) >= 160) return 256128;
  if (each > 96 && busy(64, 64) > half_the_chip) return 64128;
  if (each > 32 && busy(32, 64) > half_the_chip) return 64064;
  return 32064;
}

template <int MODE>
static int launch_moe(const bf16_t* a, const bf16_t* w, const int* offsets, const int* order, const float* pair_weight,
                      bf16_t* act, float* out, int experts, int N, int K, int top, int tokens, float limit, float alpha,
                      int form, const float* extra, int extra_parts, hipStream_t stream) {
#define FE_GO(...) return launch_moe_tile<__VA_ARGS__, MODE>(a, w, offsets, order, pair_weight, act, out, experts, N, K, top, tokens, \
                                                             limit, alpha, form, extra, extra_parts, stream)
  switch (fe_moe_tile(MODE == 0, tokens, top, experts, N, K)) {
    case 256128: FE_GO(4, 4, 4, 2, 1, 3);
    case 64128: FE_GO(2, 4, 2, 2, 2, 3);
    case 64064: FE_GO(2, 2, 2, 2, 2, 4);
    default: FE_GO(1, 2, 2, 2, 2, 6);       // 32 x 64
  }
#undef FE_GO
}

static bool mfma_fits(const void* a, const void* w, int K) {
  return K % 32 == 0 && ((((uintptr_t)a) | ((uintptr_t)w)) & 15) == 0;
}

extern "C" int fe_moe_gate_up(const void* x, const void* gate_up, int dtype, const int* offsets, const int* order, void* act,
                              int tokens, int top, int experts, int hidden, int inner, float limit, float alpha, int form,
                              const float* input_weight, hipStream_t stream) {
  if (tokens <= 0) return FE_OK;
  if (top < 1 || experts < 1 || experts > 1024 || hidden <= 0 || inner <= 0 || form < 0 || form > 2 ||
      (form == 0 && !(limit > 0.f)))
    return FE_BAD_ARGUMENT;
  const long long pairs = (long long)tokens * top;
  const dim3 grid((unsigned)(pairs / BM + experts), (unsigned)((inner + BN - 1) / BN));
  if (form == 2) {       // one matrix an expert: `gate_up` is [experts][inner][hidden]
    if (dtype == FE_F32)
      moe_grouped_kernel<float, 2><<<grid, 256, 0, stream>>>((const float*)x, (const float*)gate_up, offsets, order, input_weight,
                                                             (float*)act, nullptr, experts, inner, hidden, top, tokens, limit, alpha, form, nullptr, 0);
    else if (dtype == FE_BF16 && mfma_fits(x, gate_up, hidden)) {
      return launch_moe<2>((const bf16_t*)x, (const bf16_t*)gate_up, offsets, order, input_weight, (bf16_t*)act, nullptr, experts, inner, hidden, top,
                           tokens, limit, alpha, form, nullptr, 0, stream);
    } else if (dtype == FE_BF16)
      moe_grouped_kernel<bf16_t, 2><<<grid, 256, 0, stream>>>((const bf16_t*)x, (const bf16_t*)gate_up, offsets, order, input_weight,
                                                              (bf16_t*)act, nullptr, experts, inner, hidden, top, tokens, limit,
                                                              alpha, form, nullptr, 0);
    else
      return FE_BAD_ARGUMENT;
    return fe_check_launch();
  }
  if (dtype == FE_F32)
    moe_grouped_kernel<float, 0><<<grid, 256, 0, stream>>>((const float*)x, (const float*)gate_up, offsets, order, input_weight,
                                                           (float*)act, nullptr, experts, inner, hidden, top, tokens, limit, alpha, form, nullptr, 0);
  else if (dtype == FE_BF16 && mfma_fits(x, gate_up, hidden)) {
    return launch_moe<0>((const bf16_t*)x, (const bf16_t*)gate_up, offsets, order, input_weight, (bf16_t*)act, nullptr, experts, inner, hidden, top,
                         tokens, limit, alpha, form, nullptr, 0, stream);
  } else if (dtype == FE_BF16)
    moe_grouped_kernel<bf16_t, 0><<<grid, 256, 0, stream>>>((const bf16_t*)x, (const bf16_t*)gate_up, offsets, order, input_weight,
                                                            (bf16_t*)act, nullptr, experts, inner, hidden, top, tokens, limit,
                                                            alpha, form, nullptr, 0);
  else
    return FE_BAD_ARGUMENT;
  return fe_check_launch();
}

extern "C" int fe_moe_down(const void* act, const void* down, int dtype, const int* offsets, const int* order,
                           const float* pair_weight, float* out, int tokens, int top, int experts, int hidden, int inner,
                           const float* extra, int extra_parts, hipStream_t stream) {
  if (tokens <= 0) return FE_OK;
  if (top < 1 || experts < 1 || experts > 1024 || hidden <= 0 || inner <= 0 || (extra && extra_parts < 1)) return FE_BAD_ARGUMENT;
  const long long pairs = (long long)tokens * top;
  const dim3 grid((unsigned)(pairs / BM + experts), (unsigned)((hidden + BN - 1) / BN));
  if (dtype == FE_F32)
    moe_grouped_kernel<float, 1><<<grid, 256, 0, stream>>>((const float*)act, (const float*)down, offsets, order, pair_weight,
                                                           nullptr, out, experts, hidden, inner, top, tokens, 0.f, 0.f, 0, extra,
                                                           extra_parts);
  else if (dtype == FE_BF16 && mfma_fits(act, down, inner)) {
    return launch_moe<1>((const bf16_t*)act, (const bf16_t*)down, offsets, order, pair_weight, nullptr, out, experts, hidden, inner, top, tokens, 0.f, 0.f,
                         0, extra, extra_parts, stream);
  } else if (dtype == FE_BF16)
    moe_grouped_kernel<bf16_t, 1><<<grid, 256, 0, stream>>>((const bf16_t*)act, (const bf16_t*)down, offsets, order, pair_weight,
                                                            nullptr, out, experts, hidden, inner, top, tokens, 0.f, 0.f, 0, extra,
                                                           extra_parts);
  else
    return FE_BAD_ARGUMENT;
  return fe_check_launch();
}

// ---------------------------------------------------------------- the activation over a dense product
template <typename T>
__global__ void gated_act_kernel(const T* __restrict__ gate_up, T* __restrict__ out, long long count, int inner, float limit,
                                 float alpha) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  const long long t = i / inner;
  const int n = (int)(i - t * inner);
  const T* row = gate_up + t * 2 * inner;
  store_from_float(out + i, gated(load_as_float(row + n), load_as_float(row + inner + n), limit, alpha, 0, 1.f));
}

extern "C" int fe_gated_act(const void* gate_up, void* out, int dtype, int tokens, int inner, float limit, float alpha,
                            hipStream_t stream) {
  if (tokens <= 0) return FE_OK;
  if (inner <= 0 || !(limit > 0.f)) return FE_BAD_ARGUMENT;
  const long long count = (long long)tokens * inner;
  const int blocks = (int)((count + 255) / 256);
  if (dtype == FE_F32) gated_act_kernel<float><<<blocks, 256, 0, stream>>>((const float*)gate_up, (float*)out, count, inner, limit, alpha);
  else if (dtype == FE_BF16) gated_act_kernel<bf16_t><<<blocks, 256, 0, stream>>>((const bf16_t*)gate_up, (bf16_t*)out, count, inner, limit, alpha);
  else return FE_BAD_ARGUMENT;
  return fe_check_launch();
}

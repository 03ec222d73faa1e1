// Paged grouped-query attention for single decoded tokens, bfloat16 cache.
//
// For every sequence of the batch that brings exactly one query token (others
// are skipped: another kernel serves them), the G query heads that share a kv
// head read that head's keys and values once.  The kernel is bound by the
// cache's bytes, and where contexts are short by the chain of its start and its merge:
//   * grid (key split, kv head, sequence); with few sequences the keys of one
//     (sequence, head) are split over several blocks so that the chip is full,
//     and the block that finishes last merges the splits (a counter per (sequence, head));
//     with a dozen sequences and more, or a few, where contexts may be long, the splits follow the lengths (find_run);
//   * inside a block the four waves take 32-key blocks in turn;
//   * scores transposed, S^T = K Q^T: MFMA 16x16x32 with A = 16 keys (rows) and
//     B = the G query rows padded to 16 (columns).  The 32 keys of a block feed
//     two MFMA tiles whose rows interleave in groups of four, so that lane
//     group lq ends up with the scores of the 8 consecutive keys 8lq .. 8lq+7 of
//     its query row: exactly the B operand of the second product;
//   * softmax statistics per query row in float32 (a row's keys sit in four
//     lanes: two shuffles), base-2 exponent with the scale folded in;
//   * output transposed, O^T = V^T P^T: A = 16 dims x 32 keys from the value
//     pages, which are stored transposed ([D][slot]) for this, B = P^T.  In pages of 16 and 32 keys an instruction takes whole lines,
//     once, and the values are loaded past the caches (64 sequences of 130 to 2,000 keys 52.0 -> 48.4 us, 8 of 1,025 12.3 -> 12.1, two
//     of 30,000 and 20,000 42.8 -> 39.7).  From 64 on a
//     dim's row is a line or more, of which two waves take a half each: past the caches they would both fetch it (the 64 sequences in pages
//     of 64 57.4 -> 60.9, 14 of 14,614 in pages of 128 158 -> 178);
//   * keys and values come through LDS, each wave's to a slot of its own that holds one block (`global_load_lds_dwordx4`, waits counted by
//     hand): a request takes whole rows of keys, which pass the caches too then, the place of a block's keys or values is requested anew
//     as soon as they are in registers, without a branch or a second copy of the block's instructions, and both copies' instructions were
//     what the kernel waited for when it came to them with the memory busy.  us, from registers one and a half blocks ahead -> this: 64
//     sequences of 130 to 2,000 keys 41.5 -> 37.4, 11 of 3,000 39.3 -> 35.1, 4 of 6,000 to 16,000 36.3 -> 34.4, 8 of 1,025 12.4 -> 11.7, 64 of
//     200 to 2,000 with heads of 256 63.5 -> 53.0; whole decode steps of 4B at 8 requests 2,168 -> 2,122, at 64 4,133 -> 4,077, of 1.7B
//     at 4 long contexts 1,930 -> 1,891.  (Two blocks ahead in registers: 64 sequences 40.9, the steps 2,157, 4,120, 1,936.)
// Exactness: scores, max, sum and the weighted value sum are float32; P is
// rounded to bfloat16 for the second product; one rounding at the final store.
//
// The PREPARE variant takes the raw output of the fused q/k/v projection instead of finished
// queries and does on the way what a kernel of its own would do before it: RMSNorm over each
// q and k head, rotation by the token's position, and the write of the new key and value into
// their pages.  The new token's own key never comes back from memory: the last key split
// treats it as a fifth partial result (score q.k_new, weight 1, value v_new) beside those of
// its four waves.  The arithmetic is the stand-alone kernel's (rope_math.h), so the cache
// holds the same bits whichever kernel wrote them.
#include "agent_access.h"
#include "common.h"
#include "lds_load.h"
#include "lds_tile.h"
#include "rope_math.h"
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float floatx4;
typedef __attribute__((ext_vector_type(4))) unsigned int uintx4;

#define KEYS 32          // keys per block of work
#define WAVES 4
#define GMAX 8           // largest group size served
#define SLOT_LAYER 256   // CUs: blocks that land on a CU of their own
#define RUN_LEAST 12     // runs by length: fewest key blocks that a sequence is cut into runs of

typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
__device__ __forceinline__ unsigned int pack_bf16(float lo, float hi) {
  const bf16x2 v = {(__bf16)lo, (__bf16)hi};   // the hardware's round-to-nearest-even conversion
  return __builtin_bit_cast(unsigned int, v);
}

// Two neighbouring output elements from up to N splits: all loads first (the pair of partial
// outputs as one 8-byte load), then the sums in split order.
template <int N>
__device__ __forceinline__ unsigned int merge_few(const float* part_o, const float* part_ml, size_t first_part,
                                                  int splits, int groups, int g, int dim, int d, float sink2) {
  float m[N], l[N];
  unsigned long long o[N];
#pragma unroll
  for (int sp = 0; sp < N; ++sp) {
    const size_t row = (first_part + (sp < splits ? sp : 0)) * groups + g;
    m[sp] = load_agent(&part_ml[row * 2]);
    l[sp] = load_agent(&part_ml[row * 2 + 1]);
    o[sp] = __hip_atomic_load((const unsigned long long*)&part_o[row * dim + d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  float m_tot = -INFINITY;
#pragma unroll
  for (int sp = 0; sp < N; ++sp) m_tot = fmaxf(m_tot, sp < splits ? m[sp] : -INFINITY);
  float l_tot = 0.f, ov0 = 0.f, ov1 = 0.f;
#pragma unroll
  for (int sp = 0; sp < N; ++sp) {
    const float f = (sp < splits && m_tot > -INFINITY) ? __builtin_amdgcn_exp2f(m[sp] - m_tot) : 0.f;
    l_tot += f * l[sp];
    ov0 += f * __uint_as_float((unsigned int)o[sp]);
    ov1 += f * __uint_as_float((unsigned int)(o[sp] >> 32));
  }
  if (sink2 > -INFINITY) l_tot += __builtin_amdgcn_exp2f(sink2 - m_tot);   // a sink joins the denominator once, here
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  return (unsigned int)float_to_bf16(ov0 * inv) | ((unsigned int)float_to_bf16(ov1 * inv) << 16);
}

// What the PREPARE variant needs beyond the plain one: the norms' weights (null: no norm), the
// rotation's frequencies [D / 2], and the pages as writable memory.
struct Prepare {
  const float* q_weight;
  const float* k_weight;
  const float* inv_freq;
  float eps;
  // the projection's output as float32 partial sums [num_sums][rows][q_stride] instead of one
  // bfloat16 matrix (a product whose K was split over blocks): added up in order and rounded here
  const float* sums;
  int num_sums;
  long long sum_stride;
};
#define MAX_SUMS 4

// A wave's sum of ints.
__device__ __forceinline__ int wave_sum_int(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true);    // lane ^ 1
  v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true);    // lane ^ 2
  v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, true);   // 7 - lane within 8
  v += __builtin_amdgcn_update_dpp(0, v, 0x140, 0xF, 0xF, true);   // 15 - lane within 16
  auto r = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
  v = (int)r[0] + (int)r[1];
  r = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
  return __builtin_amdgcn_readfirstlane((int)r[0] + (int)r[1]);
}

// Key blocks that a sequence's token reads: [first, last).  The token at position ctx - 1 reads the last `window` keys, and of
// those the ones of its own run of `chunk` positions (runs counted from position 0); cached: keys that come from the pages.
struct KeyRange {
  int k_begin, first, last;
};
__device__ __forceinline__ KeyRange key_range(int ctx, int cached, int window, int chunk) {
  int k_begin = window > 0 ? max(0, ctx - window) : 0;
  if (chunk > 0) k_begin = max(k_begin, (ctx - 1) / chunk * chunk);
  return {k_begin, k_begin / KEYS, (cached + KEYS - 1) / KEYS};
}

// Runs by length (launches of up to 64 sequences): every wave finds its block's run from the lengths, one sequence a lane.
// A sequence is cut into equal runs of at most max(RUN_LEAST, ceil(all key blocks / more)) key blocks, so a launch of num_seqs + more
// blocks a head has one for each (a run's start and its part in the merge cost about as much as RUN_LEAST blocks of keys: with
// runs of down to 4 blocks 32 sequences of 20 to 200 keys took 13.4 us, whole 9.0; 4 of 1,000 to 8,000 16.9 against 16.1); the runs are handed out longest first, which the order of the blocks then balances: the first
// `layer` blocks of a head land on CUs of their own, the next `layer` beside them, shortest first, what is left goes to
// the slots that come free first.  Where a run for each CU is even to a key block (contexts about equal, and as many as divide
// the CUs), it is taken instead: two runs a CU would only start and merge twice as many (8 of 4,000 keys
// on 8 kv heads 31.1 -> 29.8 us, of 33,000 186.3 -> 185.4; the same runs as splits 28.8 and 184.9).
struct Run {
  int seq, split, splits, part;      // part: where the sequence's partial results begin, in runs of a head
  int q0, tokens, ctx;               // the sequence's query row, how many it brings, and its length
};
__device__ __forceinline__ bool find_run(const int* cu_q, const int* ctx_len, int num_seqs, int more, int own, int window, int chunk,
                                         int layer, int item, Run* run) {
  __shared__ int positions[WAVES][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = min(lane, num_seqs - 1);
  const int q0 = cu_q[i], q1 = cu_q[i + 1], ctx = ctx_len[i];
  const bool mine = lane < num_seqs && q1 - q0 == 1;
  const KeyRange range = key_range(ctx, ctx - own, window, chunk);
  const int blocks = mine ? max(range.last - range.first, 0) : 0;
  const int total = wave_sum_int(blocks), even = (total + layer - 1) / layer + 1;
  int target = max((total + more - 1) / more, RUN_LEAST);
  if (even > target && wave_sum_int(mine ? max((blocks + even - 1) / even, 1) : 0) <= layer) target = even;
  const int runs = mine ? max((blocks + target - 1) / target, 1) : 0;
  const int size = mine ? (blocks + runs - 1) / runs : -1;
  const int key = size * 64 + lane;
  const int all = wave_sum_int(runs);
  if (item >= all) return false;
  int position = 0;           // runs of longer ones; each wave counts among sixteen sequences
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int other = __builtin_amdgcn_readlane(key, wave * 16 + j), count = __builtin_amdgcn_readlane(runs, wave * 16 + j);
    position += other > key ? count : 0;
  }
  positions[wave][lane] = position;
  __syncthreads();
  position = 0;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) position += positions[w][lane];
  if (item >= layer && item < 2 * layer) item = layer + min(all, 2 * layer) - 1 - item;
  const int at = __builtin_ctzll(__ballot(mine && position <= item && item < position + runs));
  run->seq = at;
  run->splits = __builtin_amdgcn_readlane(runs, at);
  run->part = __builtin_amdgcn_readlane(position, at);
  run->split = item - run->part;
  run->q0 = __builtin_amdgcn_readlane(q0, at);
  run->tokens = 1;
  run->ctx = __builtin_amdgcn_readlane(ctx, at);
  return true;
}

// What the output is multiplied by as it is stored: sigmoid(gate) * factor, one gate for `share` neighbouring elements of a row
// (1, or a head's width), rows `stride` apart; no gate: null.  The output is rounded before and after, as by a launch of its own
// behind this one, whose bits these are (8 tokens of 16 heads of 128
// behind 300 keys in a captured graph: 10.2 -> 8.5 us).
struct OutGate : Prepare {
  const bf16_t* gate;
  size_t stride;
  int share;
  float factor;
  __device__ __forceinline__ float at(int row, int column) const { return bf16_to_float(gate[(size_t)row * stride + column / share]); }
  __device__ __forceinline__ bf16_t times(bf16_t y, float g) const { return float_to_bf16(bf16_to_float(y) / (1.f + expf(-g)) * factor); }
  __device__ __forceinline__ unsigned int times(unsigned int two, float g0, float g1) const {
    return (unsigned int)times((bf16_t)(two & 0xffffu), g0) | ((unsigned int)times((bf16_t)(two >> 16), g1) << 16);
  }
};

// A wave's slot of LDS.
template <int D, int MODE>
struct WaveSlot {
  static constexpr int LPH = D / 8;                                   // PREPARE: lanes that share a head, eight elements each
  static constexpr int ROUNDS = ((GMAX + 2) * LPH + 255) / 256;       // ... and how often the block's lanes take heads
  static constexpr int LOADS = D / 16;                                // requests of 1,024 bytes: a block's keys, and its values
  static constexpr int INPUTS = MODE == 2 ? ROUNDS * MAX_SUMS * 2 : MODE == 1 ? ROUNDS : D / 32;      // ... at most, what the queries are made of
  static constexpr int KEYS_AT = 0, VALUES_AT = LOADS * 1024;         // the inputs come to the values' place before them
  static constexpr int BYTES = VALUES_AT + (LOADS > INPUTS ? LOADS : INPUTS) * 1024;
};

// MODE 0: finished queries; 1: PREPARE from the projection's bfloat16 output; 2: PREPARE from its
// float32 partial sums.
// GATED: MODE 0 alone, with an OutGate in the place of Prepare (an argument more and a branch at the stores cost the others .1 us a launch)
// PAST: values are loaded past the caches
template <int D, int MODE, bool CAP = false, int DIST = 0, bool GATED = false, bool PAST = true>
__global__ __launch_bounds__(256, D <= 128 ? 2 : 1) void paged_decode_kernel(
    const bf16_t* __restrict__ q, long long q_stride, const bf16_t* key_pages,
    const bf16_t* value_pages, bf16_t* __restrict__ out, long long out_stride,
    float* part_o, float* part_ml, int* __restrict__ counters, const int* __restrict__ cu_q,
    const int* __restrict__ ctx_len, const int* __restrict__ block_table, int table_stride,
    int kv_heads, int groups, int block_shift, int num_blocks, int window, float scale_log2,
    std::conditional_t<GATED, OutGate, Prepare> prep, int chunk, const float* __restrict__ sink, float cap_ratio, const float* __restrict__ slopes,
    int bias_span, int num_seqs, int more) {
  constexpr bool PREPARE = MODE != 0, FROM_SUMS = MODE == 2;
  const int block_size = 1 << block_shift, block_mask = block_size - 1;
  constexpr int KC = D / 32;        // MFMA k-steps over the head dim (scores)
  constexpr int DT = D / 16;        // 16-dim tiles of the output
  using Slot = WaveSlot<D, MODE>;
  extern __shared__ __attribute__((aligned(16))) uintx4 slots[];      // [WAVES] Slot::BYTES
  // partial results that meet in LDS: the waves' outputs each in its own slot, their statistics, and the new token's score
  __shared__ float Ms[WAVES + 1][GMAX], Ls[WAVES][GMAX];

  const int hk = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lq = lane >> 4;
  // PREPARE: this thread's frequency of the rotation (the last threads': the first ones have heads), and the norms' weights of this
  // lane's elements (without a norm: any valid address, not used)
  float frequency = 0.f;
  float4 head_w[Slot::ROUNDS][2];
  if constexpr (PREPARE) {
    frequency = prep.inv_freq[max(tid - (256 - D / 2), 0)];
#pragma unroll
    for (int round = 0; round < Slot::ROUNDS; ++round) {
      const float* at = prep.q_weight ? ((tid + round * 256) / Slot::LPH < groups ? prep.q_weight : prep.k_weight) + (tid & (Slot::LPH - 1)) * 8 : prep.inv_freq;
      head_w[round][0] = *(const float4*)at;
      head_w[round][1] = *(const float4*)(at + 4);
    }
  }
  Run run;
  if (more > 0) {
    if (!find_run(cu_q, ctx_len, num_seqs, more, PREPARE, window, chunk, max(SLOT_LAYER / kv_heads, 1), blockIdx.z, &run)) return;
  } else {
    const int z = blockIdx.z, q = cu_q[z];
    run = {z, (int)blockIdx.x, (int)gridDim.x, z * (int)gridDim.x, q, cu_q[z + 1] - q, ctx_len[z]};
    // The launch has splits for the longest context that may come; one that four waves read in one block each needs none, and no merge (us,
    // splits and merge -> one run: 1 sequence of 60 keys in a launch of 8 splits 7.5 -> 5.6, 8 of 100 in one of 4 9.0 -> 7.1).
    // Beyond, one run would save more (1 of 217 keys 7.1 -> 5.9), but a wave's second block would be rounded against another maximum than its
    // split's, and so the results of all contexts of 129 to 256 keys; one run that keeps its blocks apart and sums them as the splits do
    // takes as long as they (7.2).
    // Finished queries keep their splits, and with them the order of every sum: they come by the general attention path, which the designs
    // with routers take, whose choice among experts at a near tie another rounding changes (and some without one, for whom it is time left).
    if constexpr (PREPARE) {
      const KeyRange range = key_range(run.ctx, run.ctx - 1, window, chunk);
      if (range.last - range.first <= WAVES) run.splits = 1;
      if (run.split >= run.splits) return;
    }
  }
  const int seq = run.seq, split = run.split, splits = run.splits;
  const size_t first_part = (size_t)run.part * kv_heads + (size_t)hk * splits;
  const int q0 = run.q0, ctx = run.ctx;
  if (run.tokens != 1) return;
  const int cached = PREPARE ? ctx - 1 : ctx;             // keys that the loop below reads from the pages
  const KeyRange range = key_range(ctx, cached, window, chunk);
  const int k_begin = range.k_begin, first = range.first, last = range.last;
  const int per_split = (last - first + splits - 1) / splits;
  const int my_first = first + split * per_split;
  const int my_last = min(last, my_first + per_split);

  // DIST 1: head g's score of key j, after the scale, loses slopes[g] * (ctx - 1 - j); here in base-2 units.
  // DIST 2: it gains table[g][min(ctx - 1 - j, span - 1)] instead, `slopes` being the table, float32 [heads][span]
  float slope2 = 0.f;
  if constexpr (DIST == 1) slope2 = (lr < groups ? slopes[hk * groups + lr] : 0.f) * 1.4426950408889634f;
  const float* bias_row = nullptr;
  if constexpr (DIST == 2) bias_row = slopes + (size_t)(hk * groups + min(lr, groups - 1)) * bias_span;

  // PREPARE: the block's query heads, key head and value head are finished once, eight elements a lane, and handed to all waves through
  // LDS (every wave for itself, all of the heads in the layout of its operand: .7 us a launch where this is .4; 1 sequence of 1,000 keys
  // 9.5 -> 8.6 us, 8 of 100 7.4 -> 6.4, the step of 0.6B at 1 request, with the keys through LDS, 769 -> 760).
  constexpr int LPH = Slot::LPH, ROUNDS = Slot::ROUNDS, LOADS = Slot::LOADS;
  constexpr int PITCH = D + 8;                       // of a finished head in LDS: neighbouring heads' chunks in different banks
  __shared__ float cos_s[PREPARE ? D / 2 : 1], sin_s[PREPARE ? D / 2 : 1];
  __shared__ __attribute__((aligned(16))) bf16_t heads_s[PREPARE ? (GMAX + 2) * PITCH : 8];      // queries, the new key, the new value
  uintx4* const slot = slots + wave * (Slot::BYTES / 16);
  const unsigned int slot_at = __builtin_amdgcn_readfirstlane((unsigned int)(size_t)(const __attribute__((address_space(3))) char*)slot);

  float m_run = -INFINITY, l_run = 0.f;   // of query row lr (the same in the four lanes that share it)
  floatx4 o[DT];                          // O^T: dims 16t + 4lq + i of query row lr
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = floatx4{0.f, 0.f, 0.f, 0.f};

  const int* table = block_table + (size_t)seq * table_stride;
  const int table_last = table_stride - 1;
  // The block's pages, of its first sixteen keys and of the others: the same for the whole wave.  Keys behind the context lie in a page of
  // their own sequence or, where the table has none, in page 0: they are read like the others and masked.
  struct Pages {
    int first, second;
  };
  auto page_of = [&](int key) -> int {
    const int id = table[min(key >> block_shift, table_last)];
    return id >= 0 && id < num_blocks ? id : 0;
  };
  auto pages_of = [&](int b) -> Pages { return {page_of(b * KEYS), page_of(b * KEYS + KEYS / 2)}; };
  // Keys: a request takes whole rows, 16-byte chunk p of row r to position p ^ (r % 4 + 4 (r / 8 % 2)), so that the lanes that a read
  // of LDS serves in one cycle hit different banks.
  constexpr int CPR = D / 8, RPI = 64 / CPR;         // chunks of a row, rows of a request
  const int load_row = lane / CPR, load_at = (load_row * D + ((lane & (CPR - 1)) ^ (load_row & 3)) * 8) * 2;
  auto request_keys = [&](int b, Pages pages) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int slot0 = (b * KEYS + half * (KEYS / 2)) & block_mask;
      const char* from = (const char*)(key_pages + ((((size_t)(half ? pages.second : pages.first) * kv_heads + hk) << block_shift) + slot0) * D);
#pragma unroll
      for (int i = 0; i < LOADS / 2; ++i) {
        const int j = half * (LOADS / 2) + i, row = j * RPI;
        // (rows of a request that lie in different runs of four or of eight differ in load_row alone)
        const int turn = RPI >= 8 ? 4 * (j & 1) : (row & 3 & ~(RPI - 1)) + 4 * ((row >> 3) & 1);
        lds_load::load_to_lds_once(from + i * 1024, load_at ^ (turn * 16), slot_at + Slot::KEYS_AT + j * 1024);
      }
    }
  };
  // Values (A operand of the second product): lane (lr = dim, lq) takes the 8 consecutive keys 8lq .. 8lq+7 of dims 16t + lr from
  // the transposed page, and reads them back from where they came to.
  auto request_values = [&](int b, Pages pages) {
    const size_t page = lq < 2 ? pages.first : pages.second;
    const bf16_t* from = value_pages + (((page * kv_heads + hk) * D + lr) << block_shift) + ((b * KEYS + 8 * lq) & block_mask);
#pragma unroll
    for (int t = 0; t < LOADS; ++t) {
      const bf16_t* at = from + ((size_t)(t * 16) << block_shift);
      if constexpr (PAST) lds_load::load_to_lds_once(at, slot_at + Slot::VALUES_AT + t * 1024);
      else lds_load::load_to_lds(at, slot_at + Slot::VALUES_AT + t * 1024);
    }
  };
  auto reads_done = []() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
  // All requests from here to the end of the loop are counted by hand: the compiler's own loads, which it waits for by a count that knows
  // of no others, have arrived.
  if constexpr (PREPARE) {
    asm volatile("" : "+v"(frequency));
#pragma unroll
    for (int round = 0; round < ROUNDS; ++round)
      asm volatile("" : "+v"(head_w[round][0].x), "+v"(head_w[round][0].y), "+v"(head_w[round][0].z), "+v"(head_w[round][0].w), "+v"(head_w[round][1].x),
                   "+v"(head_w[round][1].y), "+v"(head_w[round][1].z), "+v"(head_w[round][1].w));
  }
  if constexpr (DIST == 1) asm volatile("" : "+v"(slope2));
  int b = my_first + wave;
  const bool has_keys = b < my_last;
  Pages next = pages_of(b);
  const int new_page = PREPARE ? table[min((ctx - 1) >> block_shift, table_last)] : 0;      // of the new token
  // What the queries are made of goes to the slot as well, where the values come later.
  if constexpr (PREPARE) {
#pragma unroll
    for (int round = 0; round < ROUNDS; ++round) {
      if (round * 256 + wave * 64 >= (groups + 2) * LPH) break;
      const int head = min((tid + round * 256) / LPH, groups + 1);
      const size_t column = (size_t)(head < groups ? hk * groups + head : kv_heads * groups + (head - groups) * kv_heads + hk) * D + (tid & (LPH - 1)) * 8;
      const size_t at = (size_t)q0 * q_stride + column;
      if constexpr (FROM_SUMS) {
        for (int i = 0; i < prep.num_sums; ++i)
#pragma unroll
          for (int half = 0; half < 2; ++half)
            lds_load::load_to_lds(prep.sums + at + (size_t)i * prep.sum_stride + half * 4, slot_at + Slot::VALUES_AT + ((round * MAX_SUMS + i) * 2 + half) * 1024);
      } else {
        lds_load::load_to_lds(q + at, slot_at + Slot::VALUES_AT + round * 1024);
      }
    }
  } else {
    // query rows as the B operand: lane (lr = row g, lq) holds q[g][32c + 8lq .. +8]; rows beyond
    // the group read row 0 again, their scores and outputs are never stored
    const bf16_t* qrow = q + (size_t)q0 * q_stride + (size_t)(hk * groups + (lr < groups ? lr : 0)) * D;
#pragma unroll
    for (int c = 0; c < KC; ++c) lds_load::load_to_lds(qrow + c * 32 + lq * 8, slot_at + Slot::VALUES_AT + c * 1024);
  }
  if (has_keys) request_keys(b, next);
  bf16x8 qb[KC];
  uintx4 input[PREPARE ? ROUNDS : 1][FROM_SUMS ? MAX_SUMS : 1][FROM_SUMS ? 2 : 1];
  if (has_keys) lds_tile::wait_loads<LOADS>();
  else lds_tile::wait_loads<0>();
  if constexpr (PREPARE) {
#pragma unroll
    for (int round = 0; round < ROUNDS; ++round)
#pragma unroll
      for (int i = 0; i < (FROM_SUMS ? MAX_SUMS : 1); ++i)
#pragma unroll
        for (int half = 0; half < (FROM_SUMS ? 2 : 1); ++half)
          input[round][i][half] = slot[Slot::VALUES_AT / 16 + (FROM_SUMS ? (round * MAX_SUMS + i) * 2 + half : round) * 64 + lane];
  } else {
#pragma unroll
    for (int c = 0; c < KC; ++c) qb[c] = __builtin_bit_cast(bf16x8, slot[Slot::VALUES_AT / 16 + c * 64 + lane]);
  }
  reads_done();
  if (has_keys) request_values(b, next);
  next = pages_of(b + WAVES);

  // What the requests above brought, while the first keys and values are on their way: the rotation's cosines and sines of this token
  // once per block, and the heads added up, rounded, normalised and rotated as the stand-alone kernel does it (rope_math.h).
  bool extra = false;       // this block also brings the new token's own key and value
  uintx4 fresh = {0u, 0u, 0u, 0u};     // in the last wave: 8 elements of the new key (lanes below LPH) or of the new value (the LPH after them)
  if constexpr (PREPARE) {
    if (tid >= 256 - D / 2) {
      float sn, cs;
      sincosf((float)(ctx - 1) * frequency, &sn, &cs);
      cos_s[tid - (256 - D / 2)] = cs;
      sin_s[tid - (256 - D / 2)] = sn;
    }
    float v[ROUNDS][8];
    uint4 raw[ROUNDS];
#pragma unroll
    for (int round = 0; round < ROUNDS; ++round) {
      if constexpr (FROM_SUMS) {
        float4 a = __builtin_bit_cast(float4, input[round][0][0]), b = __builtin_bit_cast(float4, input[round][0][1]);
#pragma unroll
        for (int i = 1; i < MAX_SUMS; ++i)
          if (i < prep.num_sums) {
            const float4 c = __builtin_bit_cast(float4, input[round][i][0]), d = __builtin_bit_cast(float4, input[round][i][1]);
            a.x += c.x; a.y += c.y; a.z += c.z; a.w += c.w;
            b.x += d.x; b.y += d.y; b.z += d.z; b.w += d.w;
          }
        const float sum[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        uint32_t w4[4];
        pack_bf16x8(sum, w4);
        raw[round] = make_uint4(w4[0], w4[1], w4[2], w4[3]);
      } else {
        raw[round] = __builtin_bit_cast(uint4, input[round][0][0]);
      }
      const uint32_t w4[4] = {raw[round].x, raw[round].y, raw[round].z, raw[round].w};
      unpack_bf16x8(w4, v[round]);
      if (prep.q_weight) {
        float sumsq = sum_squares8(v[round]);
#pragma unroll
        for (int offset = LPH / 2; offset > 0; offset >>= 1) sumsq += __shfl_xor(sumsq, offset, FE_WAVE);
        const float inv = inverse_rms(sumsq, D, prep.eps);
        const float4 wa = head_w[round][0], wb = head_w[round][1];
        const float w8[8] = {wa.x, wa.y, wa.z, wa.w, wb.x, wb.y, wb.z, wb.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) v[round][e] = normalise(v[round][e], inv, w8[e]);
      }
    }
    __syncthreads();        // cos_s, sin_s (the keys and values requested above stay in flight)
#pragma unroll
    for (int round = 0; round < ROUNDS; ++round) {
      const int head = (tid + round * 256) / LPH, sub = tid & (LPH - 1);
      const bool low = sub * 8 < D / 2;
      float r[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float other = __shfl_xor(v[round][e], LPH / 2, FE_WAVE);
        const int j = (sub * 8 + e) & (D / 2 - 1);
        r[e] = low ? rotate_low(v[round][e], other, cos_s[j], sin_s[j]) : rotate_high(v[round][e], other, cos_s[j], sin_s[j]);
      }
      uint32_t w4[4];
      pack_bf16x8(r, w4);
      const uint4 done = head == groups + 1 ? raw[round] : make_uint4(w4[0], w4[1], w4[2], w4[3]);      // a value as it came
      if (head < groups + 2) *(uint4*)&heads_s[head * PITCH + sub * 8] = done;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < KC; ++c) qb[c] = *(const bf16x8*)&heads_s[(lr < groups ? lr : 0) * PITCH + c * 32 + lq * 8];

    // The new token's key and value, in the last wave of the last split (the one with the least other work): a partial result of
    // their own, score q.k_new, weight 1, value v_new.
    extra = split == splits - 1;
    if (extra && wave == WAVES - 1) {
      if (lane < 2 * LPH) fresh = *(const uintx4*)&heads_s[(groups + lane / LPH) * PITCH + (lane & (LPH - 1)) * 8];
      float dot = 0.f;
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const uint4 kraw = *(const uint4*)&heads_s[groups * PITCH + c * 32 + lq * 8];
        const uintx4 qraw = __builtin_bit_cast(uintx4, qb[c]);
        const uint32_t kw[4] = {kraw.x, kraw.y, kraw.z, kraw.w}, qw[4] = {qraw.x, qraw.y, qraw.z, qraw.w};
        float kf[8], qf[8];
        unpack_bf16x8(kw, kf);
        unpack_bf16x8(qw, qf);
#pragma unroll
        for (int e = 0; e < 8; ++e) dot = __fmaf_rn(qf[e], kf[e], dot);
      }
      dot = sum_xor16(dot);
      dot = sum_xor32(dot);
      if (lq == 0 && lr < groups) Ms[WAVES][lr] = dot * scale_log2;
    }
  }

  // The new token's key and value go to their pages behind the last load that this wave waits for: its loads and stores are counted
  // together, so it would wait for these stores (a value's elements lie in as many lines) as well.  That is behind the merge, or, where
  // there is none, behind the keys, so that the stores are under way while the waves meet (217 keys as one run 6.55 -> 6.30 us; with a
  // merge to come 8 of 300 keys 8.4 -> 8.6).
  auto write_pages = [&]() {
    if constexpr (PREPARE) {
      if (!extra || wave != WAVES - 1 || lane >= 2 * LPH || new_page < 0 || new_page >= num_blocks) return;   // (the host reserves pages before the launch)
      const int sub = lane & (LPH - 1), slot = (ctx - 1) & block_mask;
      const size_t page = (size_t)new_page * kv_heads + hk;
      if (lane < LPH) {
        *(uintx4*)(const_cast<bf16_t*>(key_pages) + ((page << block_shift) + slot) * D + sub * 8) = fresh;
      } else {
        bf16_t* vdst = const_cast<bf16_t*>(value_pages) + ((page * D) << block_shift) + slot;
#pragma unroll
        for (int e = 0; e < 8; ++e) vdst[(size_t)(sub * 8 + e) << block_shift] = (bf16_t)(e & 1 ? fresh[e >> 1] >> 16 : fresh[e >> 1] & 0xffffu);
      }
    }
  };

  // MFMA row r of key tile h (h = 0, 1) is key 8*(r/4) + 4h + r%4 of the block
  const int krow = 8 * (lr >> 2) + (lr & 3);
  // One block of 32 keys a turn.  Its keys' place is filled again with the next block's as soon as they are in registers, its values' likewise.
#pragma unroll 1
  for (; b < my_last; b += WAVES) {
    const bool goes_on = b + WAVES < my_last;
    const int vkey = b * KEYS + 8 * lq;
    // Which of these eight keys lie inside [k_begin, cached): the values of the others are set
    // to zero below.  Their probabilities are zero anyway, but a slot that no live key owns may
    // hold anything (a NaN that an earlier request left there), and 0 * NaN is NaN.
    const int v_hi = min(max(cached - vkey, 0), 8), v_lo = min(max(k_begin - vkey, 0), 8);
    const unsigned int v_bits = ((1u << v_hi) - 1u) & ~((1u << v_lo) - 1u);
    uintx4 v_mask;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v_mask[i] = (((v_bits >> (2 * i)) & 1u) ? 0x0000ffffu : 0u) | (((v_bits >> (2 * i + 1)) & 1u) ? 0xffff0000u : 0u);

    lds_tile::wait_loads<LOADS>();        // the keys; behind them only this block's values are under way
    uintx4 k[2][KC];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < KC; ++c) k[h][c] = slot[Slot::KEYS_AT / 16 + (krow + 4 * h) * CPR + ((4 * c + lq) ^ (lr & 7))];
    reads_done();
    if (goes_on) request_keys(b + WAVES, next);
    floatx4 st[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      st[h] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < KC; ++c)
        st[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, k[h][c]), qb[c], st[h], 0, 0, 0);
    }
    // lane (lr = query row, lq): st[h][i] = score of key b*32 + 8lq + 4h + i
    float s[8];
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int key = b * KEYS + 8 * lq + j;
      float raw = st[j >> 2][j & 3];
      // a soft cap: the score after the scale becomes cap * tanh(score / cap); cap_ratio = cap / scale, and
      // tanh(x) = 1 - 2 / (2^(2 x log2 e) + 1)
      if constexpr (CAP)
        raw = cap_ratio * (1.f - 2.f * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(raw * (2.f * 1.4426950408889634f / cap_ratio)) + 1.f));
      float v = raw * scale_log2;
      if constexpr (DIST == 1) v -= slope2 * (float)(ctx - 1 - key);
      if constexpr (DIST == 2) v += bias_row[min(max(ctx - 1 - key, 0), bias_span - 1)] * 1.4426950408889634f;
      s[j] = (key >= k_begin && key < cached) ? v : -INFINITY;
      mx = fmaxf(mx, s[j]);
    }
    mx = max_xor16(mx);
    mx = max_xor32(mx);
    const float m_new = fmaxf(m_run, mx);
    const float m_use = m_new > -INFINITY ? m_new : 0.f;
    const float corr = __builtin_amdgcn_exp2f(m_run - m_use);
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      s[j] = __builtin_amdgcn_exp2f(s[j] - m_use);
      sum += s[j];
    }
    sum = sum_xor16(sum);
    sum = sum_xor32(sum);
    l_run = l_run * corr + sum;
    m_run = m_new;
    uintx4 pw;
    pw.x = pack_bf16(s[0], s[1]); pw.y = pack_bf16(s[2], s[3]);
    pw.z = pack_bf16(s[4], s[5]); pw.w = pack_bf16(s[6], s[7]);
    const bf16x8 pb = __builtin_bit_cast(bf16x8, pw);
    if (goes_on) lds_tile::wait_loads<LOADS>();      // the values; behind them only the next block's keys
    else lds_tile::wait_loads<0>();
    uintx4 va[DT];
#pragma unroll
    for (int t = 0; t < DT; ++t) va[t] = slot[Slot::VALUES_AT / 16 + t * 64 + lane];
    reads_done();
    if (goes_on) {
      request_values(b + WAVES, next);
      next = pages_of(b + 2 * WAVES);
    }
#pragma unroll
    for (int t = 0; t < DT; ++t) {
#pragma unroll
      for (int i = 0; i < 4; ++i) o[t][i] *= corr;
      const uintx4 vt = va[t] & v_mask;
      o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, vt), pb, o[t], 0, 0, 0);
    }
  }

  if (splits == 1) write_pages();

  // lane (lr = query row, lq) holds O^T[16t + 4lq + i][lr]; the four waves meet in LDS
  if (lr < groups) {
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) ((float*)slot)[lr * D + t * 16 + lq * 4 + i] = o[t][i];
    if (lq == 0) { Ms[wave][lr] = m_run; Ls[wave][lr] = l_run; }
  }
  __syncthreads();

  for (int e = tid; e < groups * D; e += 256) {
    const int g = e / D, d = e - g * D;
    float m_tot = -INFINITY;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) m_tot = fmaxf(m_tot, Ms[w][g]);
    if (PREPARE && extra) m_tot = fmaxf(m_tot, Ms[WAVES][g]);
    float ov = 0.f, l = 0.f;
    if (m_tot > -INFINITY) {
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        const float f = __builtin_amdgcn_exp2f(Ms[w][g] - m_tot);
        ov += f * ((const float*)(slots + w * (Slot::BYTES / 16)))[g * D + d];
        l += f * Ls[w][g];
      }
      if (PREPARE && extra) {
        const float f = __builtin_amdgcn_exp2f(Ms[WAVES][g] - m_tot);
        ov += f * bf16_to_float(heads_s[(groups + 1) * PITCH + d]);
        l += f;
      }
    }
    if (splits == 1) {
      // a sink per query head: exp(sink) joins the denominator, with no key and no value
      if (sink) l += __builtin_amdgcn_exp2f(sink[hk * groups + g] * 1.4426950408889634f - m_tot);
      bf16_t y = float_to_bf16(l > 0.f ? ov / l : 0.f);
      if constexpr (GATED) y = prep.times(y, prep.at(q0, (hk * groups + g) * D + d));
      out[(size_t)q0 * out_stride + (size_t)(hk * groups + g) * D + d] = y;
    } else {
      const size_t slot = first_part + split;
      store_agent(&part_o[(slot * groups + g) * D + d], ov);
      if (d == 0) {
        store_agent(&part_ml[(slot * groups + g) * 2], m_tot);        // base-2 exponent units
        store_agent(&part_ml[(slot * groups + g) * 2 + 1], l);
      }
    }
  }
  if (splits == 1) return;

  // The block that finishes last among the splits of this (sequence, kv head) merges them.  The
  // parts are written and read with device-scope accesses that go past the per-die L2 caches,
  // every wave waits until its own stores are acknowledged, the barrier gathers the waves, then
  // one thread counts the block in; whoever counts last reads all parts.  The counter is a
  // relaxed atomic: in the language's memory model nothing orders the parts before the count.
  // What orders them is this hardware: a device-scope store is acknowledged only once it is
  // visible at the memory side that all dies share, so after the wait and the barrier every part
  // of this block is visible there before its count is, and the last block's device-scope loads
  // read from there.  An acquire-release counter at device scope would say the same in the model
  // but costs a cache write-back and invalidate in every block (measured: 16.2 instead of 14.1 us
  // a launch at 8 sequences); a cache-wide fence serialises across all blocks (0.3 us per block).
  // The counter goes back to zero for the next launch.
  // a thread's first two gates come in the meantime
  float g0 = 0.f, g1 = 0.f;
  auto load_gates = [&](int e) {
    if constexpr (GATED) {
      const int g = e / D, d = e - g * D;
      g0 = prep.at(q0, (hk * groups + g) * D + d);
      g1 = prep.at(q0, (hk * groups + g) * D + d + 1);
    }
  };
  if (GATED && 2 * tid < groups * D) load_gates(2 * tid);
  __shared__ int is_last;
  __builtin_amdgcn_s_waitcnt((0x0) | (0x7 << 4) | (0xF << 8));    // vmcnt(0): this wave's stores have been acknowledged
  __syncthreads();
  if (tid == 0) {
    int* counter = counters + (size_t)seq * kv_heads + hk;
    const int arrived = atomicAdd(counter, 1);
    is_last = arrived == splits - 1;
    if (is_last) atomicExch(counter, 0);
  }
  __syncthreads();
  if (!is_last) {
    write_pages();
    return;
  }
  if (splits <= 16) {
    // few splits: every thread reads the statistics of its row itself, together with its share
    // of the partial outputs, so that all loads are in flight at once (same sums, same order)
    for (int e = 2 * tid; e < groups * D; e += 512) {
      const int g = e / D, d = e - g * D;
      unsigned int* dst = (unsigned int*)(out + (size_t)q0 * out_stride + (size_t)(hk * groups + g) * D + d);
      const float sink2 = sink ? sink[hk * groups + g] * 1.4426950408889634f : -INFINITY;
      unsigned int y;
      if (splits <= 4) y = merge_few<4>(part_o, part_ml, first_part, splits, groups, g, D, d, sink2);
      else if (splits <= 8) y = merge_few<8>(part_o, part_ml, first_part, splits, groups, g, D, d, sink2);
      else y = merge_few<16>(part_o, part_ml, first_part, splits, groups, g, D, d, sink2);
      if constexpr (GATED) {
        if (e != 2 * tid) load_gates(e);
        y = prep.times(y, g0, g1);
      }
      *dst = y;
    }
    write_pages();
    return;
  }
  // more: rounds of sixteen, each round's loads all in flight at once, the rounds' shares brought to one maximum as they
  // come (one sequence of 8,000 keys in 32 runs: 17.8 us a launch, 27.6 with the statistics read one after the other)
  for (int e = 2 * tid; e < groups * D; e += 512) {
    const int g = e / D, d = e - g * D;
    float m_tot = -INFINITY, l_tot = 0.f, ov0 = 0.f, ov1 = 0.f;
    for (int base = 0; base < splits; base += 16) {
      float m[16], l[16];
      unsigned long long o[16];
#pragma unroll
      for (int sp = 0; sp < 16; ++sp) {
        const size_t row = (first_part + min(base + sp, splits - 1)) * groups + g;
        m[sp] = load_agent(&part_ml[row * 2]);
        l[sp] = load_agent(&part_ml[row * 2 + 1]);
        o[sp] = __hip_atomic_load((const unsigned long long*)&part_o[row * D + d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      float m_new = m_tot;
#pragma unroll
      for (int sp = 0; sp < 16; ++sp) m_new = fmaxf(m_new, m[sp]);
      const float m_use = m_new > -INFINITY ? m_new : 0.f;
      const float corr = __builtin_amdgcn_exp2f(m_tot - m_use);
      l_tot *= corr; ov0 *= corr; ov1 *= corr;
#pragma unroll
      for (int sp = 0; sp < 16; ++sp) {
        const float f = base + sp < splits ? __builtin_amdgcn_exp2f(m[sp] - m_use) : 0.f;
        l_tot += f * l[sp];
        ov0 += f * __uint_as_float((unsigned int)o[sp]);
        ov1 += f * __uint_as_float((unsigned int)(o[sp] >> 32));
      }
      m_tot = m_new;
    }
    if (sink) l_tot += __builtin_amdgcn_exp2f(sink[hk * groups + g] * 1.4426950408889634f - m_tot);
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    unsigned int y = (unsigned int)float_to_bf16(ov0 * inv) | ((unsigned int)float_to_bf16(ov1 * inv) << 16);
    if constexpr (GATED) {
      if (e != 2 * tid) load_gates(e);
      y = prep.times(y, g0, g1);
    }
    *(unsigned int*)(out + (size_t)q0 * out_stride + (size_t)(hk * groups + g) * D + d) = y;
  }
  write_pages();
}

static int launch_decode(const void* q, long long q_stride, const void* key_pages, const void* value_pages,
                         void* out, long long out_stride, float* part_o, float* part_ml, int* counters,
                         const int* cu_q, const int* ctx_len, const int* block_table, int table_stride,
                         int num_seqs, int kv_heads, int groups, int head_dim, int block_size,
                         int num_blocks, int window, float scale, int splits, const Prepare* prep,
                         int chunk, const float* sink, hipStream_t stream, float softcap = 0.f, const float* slopes = nullptr,
                         int bias_span = 0, const OutGate* gate = nullptr) {
  if (num_seqs <= 0) return FE_OK;
  constexpr int GATED_DIM = 128;      // gates come with heads of up to so many elements
  if (gate && (prep || gate->share < 1 || head_dim > GATED_DIM)) return FE_BAD_ARGUMENT;
  if (softcap < 0.f || (softcap > 0.f && (prep || !(scale > 0.f)))) return FE_BAD_ARGUMENT;
  if (slopes && (prep || softcap > 0.f)) return FE_BAD_ARGUMENT;
  if (bias_span < 0 || (bias_span > 0 && !slopes)) return FE_BAD_ARGUMENT;
  if (head_dim != 64 && head_dim != 128 && head_dim != 256) return FE_BAD_ARGUMENT;
  if (groups < 1 || groups > GMAX || kv_heads < 1 || kv_heads > 65535 || num_seqs > 65535) return FE_BAD_ARGUMENT;
  if (block_size < 16 || (block_size & (block_size - 1)) || num_blocks < 1 || table_stride < 1) return FE_BAD_ARGUMENT;
  int block_shift = 0;
  while ((1 << block_shift) < block_size) ++block_shift;
  if (q_stride % 8 || out_stride % 2 || splits > 64) return FE_BAD_ARGUMENT;
  const int more = splits < 0 ? -splits : 0;     // runs by length: blocks a head beyond the sequences
  if (splits == 0 || more > 4096 || (more > 0 && num_seqs > 64)) return FE_BAD_ARGUMENT;
  if ((((uintptr_t)out) & 3) || (((uintptr_t)part_o) & 7)) return FE_BAD_ARGUMENT;   // pairs of outputs, pairs of partial sums
  if ((((uintptr_t)q) | ((uintptr_t)key_pages) | ((uintptr_t)value_pages)) & 15) return FE_BAD_ARGUMENT;
  if (splits != 1 && (!part_o || !part_ml || !counters)) return FE_BAD_ARGUMENT;
  if (chunk < 0) return FE_BAD_ARGUMENT;
  dim3 grid(more > 0 ? 1 : splits, kv_heads, num_seqs + more);
  const float scale_log2 = scale * 1.4426950408889634f;
  const Prepare none = {nullptr, nullptr, nullptr, 0.f, nullptr, 0, 0};
#define FE_GO_AS(...)                            \
  do {                                           \
    if (block_size <= 32) FE_GO_WITH(true, __VA_ARGS__); \
    else FE_GO_WITH(false, __VA_ARGS__);         \
  } while (0)
#define FE_GO_WITH(PAST, DD, MODE, CAP, DIST, GATED, EXTRA, RATIO, SLOPES, SPAN)                                    \
  do {                                                                                                               \
    static std::atomic<bool> raised{false};                                                                          \
    auto kernel = paged_decode_kernel<DD, MODE, CAP, DIST, GATED, PAST>;                                             \
    constexpr int lds_bytes = WAVES * WaveSlot<DD, MODE>::BYTES;                                                     \
    const int limit_raised = lds_tile::raise_lds_limit((const void*)kernel, lds_bytes, &raised);                     \
    if (limit_raised != FE_OK) return limit_raised;                                                                  \
    kernel<<<grid, 256, lds_bytes, stream>>>((const bf16_t*)q, q_stride, (const bf16_t*)key_pages, \
      (const bf16_t*)value_pages, (bf16_t*)out, out_stride, part_o, part_ml, counters, cu_q, ctx_len, block_table,     \
      table_stride, kv_heads, groups, block_shift, num_blocks, window, scale_log2, EXTRA, chunk, sink, RATIO, SLOPES, SPAN, num_seqs, more); \
  } while (0)
#define FE_GO(DD, MODE) FE_GO_AS(DD, MODE, false, 0, false, MODE ? *prep : none, 0.f, nullptr, 0)
#define FE_GO_FORM(DD, CAP, DIST, RATIO, SLOPES, SPAN)                                \
  do {                                                                                \
    if constexpr (DD <= GATED_DIM)                                                    \
      if (gate) { FE_GO_AS(DD, 0, CAP, DIST, true, *gate, RATIO, SLOPES, SPAN); break; } \
    FE_GO_AS(DD, 0, CAP, DIST, false, none, RATIO, SLOPES, SPAN);                     \
  } while (0)
#define FE_GO_PLAIN(DD) FE_GO_FORM(DD, false, 0, 0.f, nullptr, 0)
#define FE_GO_CAPPED(DD) FE_GO_FORM(DD, true, 0, softcap / scale, nullptr, 0)
#define FE_GO_SLOPED(DD) FE_GO_FORM(DD, false, 1, 0.f, slopes, 0)
#define FE_GO_TABLE(DD) FE_GO_FORM(DD, false, 2, 0.f, slopes, bias_span)
  if (slopes && bias_span > 0) {
    if (head_dim == 64) FE_GO_TABLE(64);
    else if (head_dim == 128) FE_GO_TABLE(128);
    else FE_GO_TABLE(256);
  } else if (slopes) {
    if (head_dim == 64) FE_GO_SLOPED(64);
    else if (head_dim == 128) FE_GO_SLOPED(128);
    else FE_GO_SLOPED(256);
  } else if (softcap > 0.f) {
    if (head_dim == 64) FE_GO_CAPPED(64);
    else if (head_dim == 128) FE_GO_CAPPED(128);
    else FE_GO_CAPPED(256);
  } else if (prep && prep->num_sums > 0) {
    if (head_dim == 64) FE_GO(64, 2);
    else if (head_dim == 128) FE_GO(128, 2);
    else FE_GO(256, 2);
  } else if (prep) {
    if (head_dim == 64) FE_GO(64, 1);
    else if (head_dim == 128) FE_GO(128, 1);
    else FE_GO(256, 1);
  } else {
    if (head_dim == 64) FE_GO_PLAIN(64);
    else if (head_dim == 128) FE_GO_PLAIN(128);
    else FE_GO_PLAIN(256);
  }
#undef FE_GO_AS
#undef FE_GO_WITH
#undef FE_GO
#undef FE_GO_FORM
#undef FE_GO_PLAIN
#undef FE_GO_CAPPED
#undef FE_GO_SLOPED
#undef FE_GO_TABLE
  return fe_check_launch();
}

// Sequences with one query token only; others are left untouched.  Pages: keys
// [blocks][kv_heads][block_size][D], values transposed [blocks][kv_heads][D][block_size];
// block_size a power of two >= 16.  splits > 1 (at most 64) needs part_o [num_seqs * kv_heads * splits * groups * head_dim] and
// part_ml [num_seqs * kv_heads * splits * groups * 2] floats, and counters [num_seqs * kv_heads]; splits = -E (at most
// 4,096, up to 64 sequences): runs by length, at most num_seqs + E of them a head, which is what part_o and part_ml hold then
// in place of num_seqs * splits; the counters alike:
// ints that are zero before the first launch; every launch leaves them zero again.  Launches that
// share counters must not overlap.
extern "C" int fe_paged_attention_decode(const void* q, long long q_stride, const void* key_pages,
                                         const void* value_pages, void* out, long long out_stride,
                                         float* part_o, float* part_ml, int* counters, const int* cu_q,
                                         const int* ctx_len, const int* block_table, int table_stride,
                                         int num_seqs, int kv_heads, int groups, int head_dim,
                                         int block_size, int num_blocks, int window, float scale,
                                         int splits, hipStream_t stream) {
  return launch_decode(q, q_stride, key_pages, value_pages, out, out_stride, part_o, part_ml, counters, cu_q,
                       ctx_len, block_table, table_stride, num_seqs, kv_heads, groups, head_dim, block_size,
                       num_blocks, window, scale, splits, nullptr, 0, nullptr, stream);
}

// The same with the masks and softmax forms beyond the causal one: `chunk` > 0: the token reads
// keys of its own run of `chunk` positions only (runs counted from position 0); `sink` (float32
// [kv_heads * groups], or null): exp(sink_h) joins head h's softmax denominator, with no key and
// no value.
extern "C" int fe_paged_attention_decode_masked(const void* q, long long q_stride, const void* key_pages,
                                                const void* value_pages, void* out, long long out_stride,
                                                float* part_o, float* part_ml, int* counters, const int* cu_q,
                                                const int* ctx_len, const int* block_table, int table_stride,
                                                int num_seqs, int kv_heads, int groups, int head_dim,
                                                int block_size, int num_blocks, int window, int chunk,
                                                const float* sink, float scale, int splits, hipStream_t stream) {
  return launch_decode(q, q_stride, key_pages, value_pages, out, out_stride, part_o, part_ml, counters, cu_q,
                       ctx_len, block_table, table_stride, num_seqs, kv_heads, groups, head_dim, block_size,
                       num_blocks, window, scale, splits, nullptr, chunk, sink, stream);
}

// The same with a soft cap on the scores: after the scale they become softcap * tanh(score / softcap).
extern "C" int fe_paged_attention_decode_capped(const void* q, long long q_stride, const void* key_pages,
                                                const void* value_pages, void* out, long long out_stride,
                                                float* part_o, float* part_ml, int* counters, const int* cu_q,
                                                const int* ctx_len, const int* block_table, int table_stride,
                                                int num_seqs, int kv_heads, int groups, int head_dim,
                                                int block_size, int num_blocks, int window, int chunk,
                                                const float* sink, float scale, float softcap, int splits,
                                                hipStream_t stream) {
  if (!(softcap > 0.f)) return FE_BAD_ARGUMENT;
  return launch_decode(q, q_stride, key_pages, value_pages, out, out_stride, part_o, part_ml, counters, cu_q,
                       ctx_len, block_table, table_stride, num_seqs, kv_heads, groups, head_dim, block_size,
                       num_blocks, window, scale, splits, nullptr, chunk, sink, stream, softcap);
}

// The same with a penalty on distance: head h's score of key j, after the scale, loses slopes[h] * (ctx - 1 - j)
// (slopes: float32 [kv_heads * groups]).
extern "C" int fe_paged_attention_decode_sloped(const void* q, long long q_stride, const void* key_pages,
                                                const void* value_pages, void* out, long long out_stride,
                                                float* part_o, float* part_ml, int* counters, const int* cu_q,
                                                const int* ctx_len, const int* block_table, int table_stride,
                                                int num_seqs, int kv_heads, int groups, int head_dim,
                                                int block_size, int num_blocks, int window, int chunk,
                                                const float* sink, const float* slopes, float scale, int splits,
                                                hipStream_t stream) {
  if (!slopes) return FE_BAD_ARGUMENT;
  return launch_decode(q, q_stride, key_pages, value_pages, out, out_stride, part_o, part_ml, counters, cu_q,
                       ctx_len, block_table, table_stride, num_seqs, kv_heads, groups, head_dim, block_size,
                       num_blocks, window, scale, splits, nullptr, chunk, sink, stream, 0.f, slopes);
}

// The same with a bias by distance: head h's score of key j, after the scale, gains table[h][min(ctx - 1 - j, span - 1)]
// (table: float32 [kv_heads * groups][span]).
extern "C" int fe_paged_attention_decode_biased(const void* q, long long q_stride, const void* key_pages,
                                                const void* value_pages, void* out, long long out_stride,
                                                float* part_o, float* part_ml, int* counters, const int* cu_q,
                                                const int* ctx_len, const int* block_table, int table_stride,
                                                int num_seqs, int kv_heads, int groups, int head_dim,
                                                int block_size, int num_blocks, int window, int chunk,
                                                const float* sink, const float* table, int span, float scale, int splits,
                                                hipStream_t stream) {
  if (!table || span < 1) return FE_BAD_ARGUMENT;
  return launch_decode(q, q_stride, key_pages, value_pages, out, out_stride, part_o, part_ml, counters, cu_q,
                       ctx_len, block_table, table_stride, num_seqs, kv_heads, groups, head_dim, block_size,
                       num_blocks, window, scale, splits, nullptr, chunk, sink, stream, 0.f, table, span);
}

// Any of the forms above (softcap 0, slopes null and span 0 for the ones without; `slopes` is the table where span > 0), the
// output times sigmoid(gate) * factor: gate [tokens] rows gate_stride apart, a number for every `share` elements of a row; heads of 64 or 128.
extern "C" int fe_paged_attention_decode_gated(const void* q, long long q_stride, const void* key_pages,
                                               const void* value_pages, void* out, long long out_stride,
                                               float* part_o, float* part_ml, int* counters, const int* cu_q,
                                               const int* ctx_len, const int* block_table, int table_stride,
                                               int num_seqs, int kv_heads, int groups, int head_dim,
                                               int block_size, int num_blocks, int window, int chunk,
                                               const float* sink, const float* slopes, int span, float scale, float softcap,
                                               int splits, const void* gate, long long gate_stride, int share, float factor,
                                               hipStream_t stream) {
  const long long width = (long long)kv_heads * groups * head_dim;
  OutGate how = {};
  how.gate = (const bf16_t*)gate;
  how.stride = (size_t)gate_stride;
  how.share = share;
  how.factor = factor;
  if (!gate || share < 1 || width % share || gate_stride < width / share) return FE_BAD_ARGUMENT;
  return launch_decode(q, q_stride, key_pages, value_pages, out, out_stride, part_o, part_ml, counters, cu_q,
                       ctx_len, block_table, table_stride, num_seqs, kv_heads, groups, head_dim, block_size,
                       num_blocks, window, scale, splits, nullptr, chunk, sink, stream, softcap, slopes, span, &how);
}

// The same for a batch in which EVERY sequence brings one token, straight from the fused
// projection's output qkv [num_seqs rows of (kv_heads * groups + 2 * kv_heads) * head_dim, row
// stride q_stride]: q and k heads are normalised (weights [head_dim] float32, null: no norm)
// and rotated whole by position ctx_len - 1 (inv_freq [head_dim / 2]), and each sequence's new
// key and value are written to slot ctx_len - 1 of its pages.  qkv itself is not changed.
// qkv_sums > 0 (at most 4): qkv is float32 and holds that many partial sums of the projection,
// sum_stride floats apart, each [num_seqs rows, row stride q_stride]; they are added up in order
// and rounded to bfloat16 first.
extern "C" int fe_paged_attention_decode_prepare(const void* qkv, int qkv_sums, long long sum_stride,
                                                 long long q_stride, const float* q_weight,
                                                 const float* k_weight, const float* inv_freq, float eps,
                                                 void* key_pages, void* value_pages, void* out,
                                                 long long out_stride, float* part_o, float* part_ml,
                                                 int* counters, const int* cu_q, const int* ctx_len,
                                                 const int* block_table, int table_stride, int num_seqs,
                                                 int kv_heads, int groups, int head_dim, int block_size,
                                                 int num_blocks, int window, float scale, int splits,
                                                 hipStream_t stream) {
  if (!inv_freq || (!q_weight) != (!k_weight)) return FE_BAD_ARGUMENT;
  if (q_weight && ((((uintptr_t)q_weight) | ((uintptr_t)k_weight)) & 15)) return FE_BAD_ARGUMENT;
  if (q_stride < (long long)(kv_heads * groups + 2 * kv_heads) * head_dim) return FE_BAD_ARGUMENT;
  if (qkv_sums < 0 || qkv_sums > MAX_SUMS) return FE_BAD_ARGUMENT;
  if (qkv_sums > 0 && (q_stride % 4 || sum_stride % 4 || sum_stride < (long long)num_seqs * q_stride)) return FE_BAD_ARGUMENT;
  const Prepare prep = {q_weight, k_weight, inv_freq, eps, qkv_sums > 0 ? (const float*)qkv : nullptr, qkv_sums, sum_stride};
  return launch_decode(qkv, q_stride, key_pages, value_pages, out, out_stride, part_o, part_ml, counters, cu_q,
                       ctx_len, block_table, table_stride, num_seqs, kv_heads, groups, head_dim, block_size,
                       num_blocks, window, scale, splits, &prep, 0, nullptr, stream);
}

// The tile product that kernels with both operands in LDS share: BM = 16 MI WM rows of one operand times BN = 16 NI WN rows
// of the other (bfloat16, K contiguous in both), WM x WN waves of 16 MI x 16 NI each, in KG groups that share a step's K.
#pragma once
#include "common.h"
#include <atomic>
#include <type_traits>

namespace lds_tile {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float floatx4;
typedef __attribute__((ext_vector_type(4))) unsigned int uintx4;

constexpr int KSTEP = 64;          // elements of K a step

// 16 bytes a lane from `global` to LDS byte address `at` + 16 * lane (`at` the same in every lane).  In assembly, because behind the
// builtin every read of LDS that the compiler forms waits for all loads into LDS that are under way; the statement writes no register,
// so a load under way has nothing of the compiler's to overwrite.  (The other way round, reads of LDS in assembly that are waited for
// later, a register that looks free or is copied meanwhile would be lost; that form was as fast: 1,316 products of 1 to 8,192 rows
// take 0.996 of its time with the compiler's own reads, which it counts and waits for itself.)
__device__ __forceinline__ void load_to_lds(const void* global, unsigned int at) {
  unsigned int m0;       // kept: the compiler takes m0 as untouched by a statement
  asm volatile("s_mov_b32 %0, m0\n s_mov_b32 m0, %2\n s_nop 0\n global_load_lds_dwordx4 %1, off\n s_mov_b32 m0, %0"
               : "=&s"(m0) : "v"(global), "s"(at) : "memory");
}
// The same for lines that no other block reads: they pass the caches without staying there (us, weights from memory,
// with the caches full of something else before: 8 rows x 19,456 x 2,560 19.4 -> 17.9, x 2,560 x 9,728 11.1 -> 10.8, 64 rows x 19,456 x 2,560
// 23.8 -> 22.7; where two blocks share a weight row it is the wrong way: 250 rows 41.3 -> 46.4).
__device__ __forceinline__ void load_to_lds_once(const void* global, unsigned int at) {
  unsigned int m0;
  asm volatile("s_mov_b32 %0, m0\n s_mov_b32 m0, %2\n s_nop 0\n global_load_lds_dwordx4 %1, off nt\n s_mov_b32 m0, %0"
               : "=&s"(m0) : "v"(global), "s"(at) : "memory");
}
// wait until at most PENDING of this wave's loads are outstanding (PENDING < 64; loads of the compiler's in between only make it longer)
template <int PENDING>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(PENDING) : "memory");
}
// the same for min(AHEAD, ahead) steps of PER loads each: the counts of a walk's end are known only when it runs, and a wait takes a constant
template <int PER, int AHEAD>
__device__ __forceinline__ void wait_steps(int ahead) {
  if constexpr (AHEAD <= 0) wait_loads<0>();
  else if (ahead >= AHEAD) wait_loads<PER * AHEAD>();
  else wait_steps<PER, AHEAD - 1>(ahead);
}
// all of this wave's reads of LDS have arrived, and it goes on when every wave of the block is here
__device__ __forceinline__ void reads_done_barrier() {
  __builtin_amdgcn_s_waitcnt(0xF | (0x3 << 14) | (0x7 << 4));      // lgkmcnt(0), and nothing of the other counters
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int MI, int NI, int WM, int WN, int KG, int STAGES>
struct Shape {
  static constexpr int BM = 16 * MI * WM, BN = 16 * NI * WN, THREADS = 64 * WM * WN * KG;
  static constexpr size_t BYTES = (size_t)STAGES * (BM + BN) * 128;
  static_assert(BYTES <= 160 * 1024 && BYTES >= (size_t)(KG - 1) * BM * BN * 4, "LDS of a CU");
};

// Fills acc[i][j] of lane (r = lane % 16, q = lane / 16) of wave (wm, wn) with the products of row 16 (MI wm + i) + r of the first
// operand and rows 16 (NI wn + j) + 4 q .. + 3 of the second, over 64-steps [first, last) of K (a multiple of 64, or, with
// HALF_END, of 32).  row_of(j): where row j of the tile begins, the first operand's BM rows, then the second's BN.  Returns
// whether this wave holds the sums (those of group 0 do); every thread of the block must call it.  once (a bool or a constant): no other
// block reads the rows of the second operand.
//
// LDS holds a step of a tile as [row][8 chunks of 16 bytes], chunk c of row j at position c ^ (j % 8): the lanes that a 16-byte
// read serves in one cycle then hit different bank groups (no conflicts counted).  Both operands go there straight from memory
// (`global_load_lds_dwordx4`), STAGES buffers, all of them in flight; one barrier a step.  A wave requests the fragments of its
// next half step from LDS before it multiplies those of this one.  The last STAGES steps request nothing (until then they fetched
// the last step again, so that one constant served every wait: a quarter more requests at K = 2,560 and ten stages, and a block
// ended when those had landed).  Decode steps: 0.6B, 1 request 947 -> 909 us, 4B, 8 requests 2,532 -> 2,464, 64 requests 4,291 ->
// 4,245; counting the way down at run time, a chain of branches a step, cost more than it saved (1,058 at 1 request).  REFETCH: they
// do fetch the last step again, in a walk of half the instructions, for a tile whose short walks are over before the written out steps
// have been fetched (gemm_lds.h).
template <int MI, int NI, int WM, int WN, int KG, int STAGES, bool HALF_END, bool REFETCH = false, typename Once = std::false_type, typename RowOf>
__device__ __forceinline__ bool product(uintx4* lds, RowOf row_of, int first, int last, int K, floatx4 (&acc)[MI][NI], Once once = {}) {
  constexpr int BM = 16 * MI * WM, BN = 16 * NI * WN, WAVES = WM * WN * KG, T = 2 / KG;
  constexpr int GROUPS = (BM + BN) / 8, LOADS = GROUPS / WAVES, MORE = GROUPS % WAVES;   // groups of eight rows: one load of a wave each
  constexpr int STAGE = (BM + BN) * 8;              // 16-byte units of a stage
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int my_chunk = (lane & 7) ^ (lane >> 3);    // (a group's first row is a multiple of eight)
  const unsigned int base = __builtin_amdgcn_readfirstlane((unsigned int)(size_t)(const __attribute__((address_space(3))) char*)&lds[0]);
  // this lane's place in each of the wave's loads
  const bf16_t* from[LOADS + 1];
#pragma unroll
  for (int i = 0; i <= LOADS; ++i) from[i] = row_of(min((wave + WAVES * i) * 8 + (lane >> 3), BM + BN - 1));
  auto load = [&](int step, int stage) {
    const int k0 = (REFETCH ? min(step, last - 1) : step) * KSTEP;
    const int at = k0 + (HALF_END && k0 + KSTEP > K ? my_chunk & 3 : my_chunk) * 8;
    auto load_one = [&](int i) {
      // a row of the second operand: known here but for the share that may begin inside the first.  (Loads past the caches with a branch at
      // every load, us: 11 x 4,096 x 4,096 7.7 -> 8.5, 5 x 3,776 x 4,480 7.8 -> 9.1; without it 7.5 and 7.6.)
      constexpr int WHOLE = BM / 8 / WAVES, MIXED = BM / 8 % WAVES;
      const bool second = i > WHOLE || (i == WHOLE && (MIXED == 0 || wave >= MIXED));
      if (once && second) load_to_lds_once(from[i] + at, base + (stage * STAGE + (wave + WAVES * i) * 64) * 16);
      else load_to_lds(from[i] + at, base + (stage * STAGE + (wave + WAVES * i) * 64) * 16);
    };
#pragma unroll
    for (int i = 0; i < LOADS; ++i) load_one(i);
    if (MORE > 0 && wave < MORE) load_one(LOADS);
  };
  const int r = lane & 15, q = lane >> 4, group = wave / (WM * WN), wm = wave % WM, wn = wave / WM % WN;
  const uintx4* x_at = lds + (wm * 16 * MI + r) * 8;
  const uintx4* w_at = lds + (BM + wn * 16 * NI + r) * 8;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  if (first < last) {
    uintx4 a0[MI], b0[NI], a1[MI], b1[NI];
    auto fragments = [&](int stage, int t, uintx4* a, uintx4* b) {
      const int at = stage * STAGE + ((4 * (group * T + t) + q) ^ (r & 7));
#pragma unroll
      for (int i = 0; i < MI; ++i) a[i] = x_at[at + 128 * i];
#pragma unroll
      for (int j = 0; j < NI; ++j) b[j] = w_at[at + 128 * j];
    };
    auto multiply = [&](const uintx4* a, const uintx4* b) {
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int i = 0; i < MI; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b[j]), __builtin_bit_cast(bf16x8, a[i]), acc[i][j], 0, 0, 0);
    };
    int stage = 0;
    // a half: the next half's fragments are requested, then this half's are multiplied.
    auto half = [&](int step, bool ends_step, auto ahead, bool loads, int t_next, const uintx4* a, const uintx4* b, uintx4* a_next, uintx4* b_next) {
      const int t = T == 1 ? 0 : ends_step;
      int from_stage = stage;
      if (ends_step) {
        // this wave's share of the next step has landed, and behind the barrier everyone's; everyone has read all of
        // this step, whose buffer is filled again
        constexpr int AHEAD = decltype(ahead)::value;
        if (MORE > 0 && wave < MORE) wait_loads<(LOADS + 1) * AHEAD>();
        else wait_loads<LOADS * AHEAD>();
        reads_done_barrier();
        if (loads) load(step + STAGES, stage);
        stage = stage + 1 == STAGES ? 0 : stage + 1;
        from_stage = stage;
      }
      fragments(from_stage, t_next, a_next, b_next);
      __builtin_amdgcn_sched_barrier(0);
      if (!HALF_END || step * KSTEP + (group * T + t) * 32 < K) multiply(a, b);
      __builtin_amdgcn_sched_barrier(0);
    };
    const std::integral_constant<int, STAGES - 2> full;
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
      if (REFETCH || first + s < last) load(first + s, s);
    const int behind = REFETCH ? STAGES - 1 : last - 1 - first;
    if (MORE > 0 && wave < MORE) wait_steps<LOADS + 1, STAGES - 1>(behind);
    else wait_steps<LOADS, STAGES - 1>(behind);
    reads_done_barrier();
    fragments(0, 0, a0, b0);
    int step = first;
    if constexpr (REFETCH) {
      static_assert(T == 1, "two steps a round");
      for (; step + 1 < last; step += 2) {
        half(step, true, full, true, 0, a0, b0, a1, b1);
        half(step + 1, true, full, true, 0, a1, b1, a0, b0);
      }
      if (step < last) half(step, true, full, true, 0, a0, b0, a1, b1);
      wait_loads<0>();
    } else if constexpr (T == 2) {
      for (; last - step > STAGES; ++step) {
        half(step, false, full, true, 1, a0, b0, a1, b1);
        half(step, true, full, true, 0, a1, b1, a0, b0);
      }
    } else {
      for (; last - step > STAGES + 1; step += 2) {
        half(step, true, full, true, 0, a0, b0, a1, b1);
        half(step + 1, true, full, true, 0, a1, b1, a0, b0);
      }
      if ((last - step) % 2 == 0) fragments(stage, 0, a1, b1);      // below, an odd count of steps left finds its fragments in a0
    }
    // The last STAGES steps (STAGES + 1 where two steps make a round) request nothing, or no further step: fewer and fewer loads
    // are under way, and a wait takes a constant, so each of them is written out.
    const int rest = REFETCH ? 0 : last - step;
    auto end = [&](auto self, auto left) {
      constexpr int L = decltype(left)::value;
      if constexpr (L > 0) {
        const std::integral_constant<int, (L < STAGES ? (L > 1 ? L - 2 : 0) : STAGES - 2)> ahead;
        if (rest >= L) {
          if constexpr (T == 2) {
            half(last - L, false, ahead, false, 1, a0, b0, a1, b1);
            if constexpr (L > 1) half(last - L, true, ahead, false, 0, a1, b1, a0, b0);
            else if (!HALF_END || (last - 1) * KSTEP + (group * T + 1) * 32 < K) multiply(a1, b1);
          } else {
            const uintx4 *a = L % 2 ? a0 : a1, *b = L % 2 ? b0 : b1;
            if constexpr (L > 1) half(last - L, true, ahead, L > STAGES, 0, a, b, L % 2 ? a1 : a0, L % 2 ? b1 : b0);
            else if (!HALF_END || (last - 1) * KSTEP + group * 32 < K) multiply(a, b);
          }
        }
        self(self, std::integral_constant<int, L - 1>{});
      }
    };
    end(end, std::integral_constant<int, REFETCH ? 0 : T == 2 ? STAGES : STAGES + 1>{});
  }
  if constexpr (KG > 1) {
    reads_done_barrier();
    floatx4* meet = (floatx4*)lds;
    if (group > 0) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) meet[((wave % (WM * WN)) * MI * NI + i * NI + j) * 64 + lane] = acc[i][j];
    }
    __syncthreads();
    if (group > 0) return false;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] += meet[(wave * MI * NI + i * NI + j) * 64 + lane];
  }
  return true;
}

// Lets a kernel use more LDS than a launch may by default; once a kernel (asked for from several threads at a time it is only
// done again).
static inline int raise_lds_limit(const void* kernel, size_t lds_bytes, std::atomic<bool>* raised) {
  if (raised->load(std::memory_order_relaxed)) return FE_OK;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes) != hipSuccess) return FE_LAUNCH_FAILED;
  raised->store(true, std::memory_order_relaxed);
  return FE_OK;
}

}  // namespace lds_tile

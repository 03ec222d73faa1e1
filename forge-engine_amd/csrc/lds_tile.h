// The tile product that kernels with both operands in LDS share: BM = 16 MI WM rows of one operand times BN = 16 NI WN rows
// of the other (bfloat16, K contiguous in both), WM x WN waves of 16 MI x 16 NI each, in KG groups that share a step's K.
#pragma once
#include "common.h"

namespace lds_tile {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float floatx4;
typedef __attribute__((ext_vector_type(4))) unsigned int uintx4;

constexpr int KSTEP = 64;          // elements of K a step

// wait until at most n of this wave's vector memory operations are outstanding (n < 64)
#define FE_WAIT_VMEM(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | ((((n) >> 4) & 0x3) << 14) | (0x7 << 4) | (0xF << 8))

__device__ __forceinline__ void load_to_lds(const void* global, void* lds) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)global,
                                   (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}

// 16 bytes from LDS byte address `at` + OFFSET (a constant below 65536); nothing waits for them here (the compiler's own
// reads of LDS would wait for every load into LDS that is under way, too)
template <int OFFSET>
__device__ __forceinline__ uintx4 lds_read16(unsigned int at) {
  uintx4 v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(OFFSET) : "memory");
  return v;
}
// COUNT fragments of sixteen rows, 2,048 bytes apart
template <int COUNT, int FROM = 0>
__device__ __forceinline__ void lds_read_rows(unsigned int at, uintx4* v) {
  if constexpr (FROM < COUNT) {
    v[FROM] = lds_read16<2048 * FROM>(at);
    lds_read_rows<COUNT, FROM + 1>(at, v);
  }
}
// every read of LDS of this wave has arrived; `v` are the registers that the wait is for
template <int COUNT>
__device__ __forceinline__ void lds_arrived(uintx4* v) {
#pragma unroll
  for (int i = 0; i < COUNT; ++i) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v[i]));
}

template <int MI, int NI, int WM, int WN, int KG, int STAGES>
struct Shape {
  static constexpr int BM = 16 * MI * WM, BN = 16 * NI * WN, THREADS = 64 * WM * WN * KG;
  static constexpr size_t BYTES = (size_t)STAGES * (BM + BN) * 128;
  static_assert(BYTES <= 160 * 1024 && BYTES >= (size_t)(KG - 1) * BM * BN * 4, "LDS of a CU");
};

// Fills acc[i][j] of lane (r = lane % 16, q = lane / 16) of wave (wm, wn) with the products of row 16 (MI wm + i) + r of the first
// operand and rows 16 (NI wn + j) + 4 q .. + 3 of the second, over 64-steps [first, last) of K (a multiple of 64, or, with
// HALF_END, of 32).  row_of(j): where
// row j of the tile begins, the first operand's BM rows, then the second's BN.  Returns whether this wave holds the sums
// (those of group 0 do); every thread of the block must call it.
//
// LDS holds a step of a tile as [row][8 chunks of 16 bytes], chunk c of row j at position c ^ (j % 8): the lanes that a 16-byte
// read serves in one cycle then hit different bank groups (no conflicts counted).  Both operands go there straight from memory
// (`global_load_lds_dwordx4`), STAGES buffers, all of them in flight; one barrier a step.  A wave requests the fragments of its
// next half step from LDS before it multiplies those of this one.
template <int MI, int NI, int WM, int WN, int KG, int STAGES, bool HALF_END, typename RowOf>
__device__ __forceinline__ bool product(uintx4* lds, RowOf row_of, int first, int last, int K, floatx4 (&acc)[MI][NI]) {
  constexpr int BM = 16 * MI * WM, BN = 16 * NI * WN, WAVES = WM * WN * KG, T = 2 / KG;
  constexpr int GROUPS = (BM + BN) / 8, LOADS = GROUPS / WAVES, MORE = GROUPS % WAVES;   // groups of eight rows: one load of a wave each
  constexpr int STAGE = (BM + BN) * 8;              // 16-byte units of a stage
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int my_chunk = (lane & 7) ^ (lane >> 3);    // (a group's first row is a multiple of eight)
  // this lane's place in each of the wave's loads
  const bf16_t* from[LOADS + 1];
#pragma unroll
  for (int i = 0; i <= LOADS; ++i) from[i] = row_of(min((wave + WAVES * i) * 8 + (lane >> 3), BM + BN - 1));
  auto load = [&](int step, int stage) {       // past the end the last step again, so that the waits can count
    const int k0 = min(step, last - 1) * KSTEP;
    const int at = k0 + (HALF_END && k0 + KSTEP > K ? my_chunk & 3 : my_chunk) * 8;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) load_to_lds(from[i] + at, &lds[stage * STAGE + (wave + WAVES * i) * 64]);
    if (MORE > 0 && wave < MORE) load_to_lds(from[LOADS] + at, &lds[stage * STAGE + (wave + WAVES * LOADS) * 64]);
  };
  const int r = lane & 15, q = lane >> 4, group = wave / (WM * WN), wm = wave % WM, wn = wave / WM % WN;
  const unsigned int base = (unsigned int)(size_t)(const __attribute__((address_space(3))) char*)&lds[0];
  const unsigned int x_at = base + (wm * 16 * MI + r) * 128, w_at = base + (BM + wn * 16 * NI + r) * 128;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  if (first < last) {
    uintx4 a0[MI], b0[NI], a1[MI], b1[NI];
    auto fragments = [&](int stage, int t, uintx4* a, uintx4* b) {
      const unsigned int at = stage * (STAGE * 16) + (((4 * (group * T + t) + q) ^ (r & 7)) * 16);
      lds_read_rows<MI>(x_at + at, a);
      lds_read_rows<NI>(w_at + at, b);
    };
    auto multiply = [&](const uintx4* a, const uintx4* b) {
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int i = 0; i < MI; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b[j]), __builtin_bit_cast(bf16x8, a[i]), acc[i][j], 0, 0, 0);
    };
    int stage = 0;
    // a half: the next half's fragments are requested, then this half's are multiplied
    auto half = [&](int step, bool ends_step, int t_next, const uintx4* a, const uintx4* b, uintx4* a_next, uintx4* b_next) {
      const int t = T == 1 ? 0 : ends_step;
      int from_stage = stage;
      if (ends_step) {
        // this wave's share of the next step has landed, and behind the barrier everyone's; everyone has read all of
        // this step, whose buffer is filled again
        if (MORE > 0 && wave < MORE) FE_WAIT_VMEM((LOADS + 1) * (STAGES - 2));
        else FE_WAIT_VMEM(LOADS * (STAGES - 2));
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        load(step + STAGES, stage);
        stage = stage + 1 == STAGES ? 0 : stage + 1;
        from_stage = stage;
      }
      fragments(from_stage, t_next, a_next, b_next);
      __builtin_amdgcn_sched_barrier(0);
      if (!HALF_END || step * KSTEP + (group * T + t) * 32 < K) multiply(a, b);
      __builtin_amdgcn_sched_barrier(0);
      lds_arrived<MI>(a_next);
      lds_arrived<NI>(b_next);
    };
#pragma unroll
    for (int s = 0; s < STAGES; ++s) load(first + s, s);
    if (MORE > 0 && wave < MORE) FE_WAIT_VMEM((LOADS + 1) * (STAGES - 1));
    else FE_WAIT_VMEM(LOADS * (STAGES - 1));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    fragments(0, 0, a0, b0);
    lds_arrived<MI>(a0);
    lds_arrived<NI>(b0);
    if constexpr (T == 2) {
      for (int step = first; step < last; ++step) {
        half(step, false, 1, a0, b0, a1, b1);
        half(step, true, 0, a1, b1, a0, b0);
      }
    } else {
      int step = first;
      for (; step + 1 < last; step += 2) {
        half(step, true, 0, a0, b0, a1, b1);
        half(step + 1, true, 0, a1, b1, a0, b0);
      }
      if (step < last) half(step, true, 0, a0, b0, a1, b1);
    }
    FE_WAIT_VMEM(0);
  }
  if constexpr (KG > 1) {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
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

// The fragments' reads are waited for by hand: a build that spills registers would move values that are still in flight,
// and is never launched.  Also raises the kernel's LDS limit.  0: not yet asked, 1: fit, -1: refused.
static inline int fit_to_launch(const void* kernel, size_t lds_bytes, int* checked) {
  if (*checked == 0) {
    hipFuncAttributes attributes;
    if (hipFuncGetAttributes(&attributes, kernel) != hipSuccess) return FE_LAUNCH_FAILED;
    if (attributes.localSizeBytes != 0) { *checked = -1; return FE_BAD_ARGUMENT; }
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes) != hipSuccess)
      return FE_LAUNCH_FAILED;
    *checked = 1;                 // (a race here only repeats the calls)
  }
  return *checked < 0 ? FE_BAD_ARGUMENT : FE_OK;
}

}  // namespace lds_tile

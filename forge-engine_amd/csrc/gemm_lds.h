// The product for portions (gemm_wide.hip) with both operands in LDS: dozens to hundreds of rows of x (many requests
// decoding, a portion of a prompt):
//   out[M, N] = x[M, K] * W[N, K]^T
// with one of three endings: float32 partial sums over parts of K ([parts][M, N]; the consumer, the next norm or the
// attention launch, adds them in order), bfloat16, or act(gate) * up as bfloat16 for a fused gate/up weight.
//
// Block = BM rows of x x BN weight rows x a part of K, WM x WN waves of 16 MI x 16 NI each, in KG groups that share a
// step's K (the groups' sums meet in LDS at the end, in order).  Both operands go from memory straight into LDS by
// `global_load_lds_dwordx4`, 64 elements of K a step, STAGES buffers deep, all of them in flight; one barrier a step.  A
// wave requests the fragments of its next half step from LDS before it multiplies those of this one.
//
// What bounds it: a CU's L1 holds about 80 lines that it waits for (128 x 160 tiles, 256 rows x 19,456 weight rows x
// 2,560: 2.94 M requests of 128 bytes, 547 clocks each, over 256 CUs and 80,000 clocks), 17 to 19 bytes a clock and CU at
// that latency, 9 to 10 TB/s for the chip, and a tile needs (BM + BN) x 128 bytes a step.  So the tile that wins is the
// one whose blocks fill rounds of one a CU with the fewest bytes for the fullest CU.  The same product with the weight
// straight in registers and x through registers into LDS (gemm_wide) has a wave's own few loads in flight instead.
// Measured on one MI355X, us a product (what took the sizes before -> this): gate/up of 9,728 x 2,560 at 64 rows
// 26.7 -> 24.1, at 256 54 -> 42 (the matrix library and the gate kernel); q/k/v of 6,144 x 2,560 at 256 rows
// 21 -> 15; down projection of 2,560 x 9,728 at 64 / 256 / 512 rows 14.6 -> 12, 25.5 -> 22, 48 -> 32; gate/up of
// 3,072 x 1,024 at 384 rows 18.0 -> 13.5.  Starting the blocks' walks over K at different places changes nothing (no
// memory channel is hot), nor do four stages instead of three.  From 1,500 rows on the matrix library is ahead.
//
// MFMA 16x16x32 bf16 with A = W (16 weight rows), B = x^T (16 rows of x): lane l (r = l % 16, q = l / 16) supplies row r,
// k = 8 q .. + 8 of either and receives D[weight row 4 q + i][row of x r]: four neighbouring output columns of a row.
#pragma once
#include "common.h"
#include "gate_act.h"

namespace through_lds {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float floatx4;
typedef __attribute__((ext_vector_type(4))) unsigned int uintx4;

constexpr int KSTEP = 64;          // elements of K a step
constexpr int XCDS = 8;
constexpr int END_PARTS = 0, END_BF16 = 1, END_GATED = 2;

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

// LDS holds a step of a tile as [row][8 chunks of 16 bytes], x's rows and then the weight's, chunk c of row j at position
// c ^ (j % 8): the lanes that a 16-byte read serves in one cycle then hit different bank groups (no conflicts counted).
// With the gated ending a fragment of sixteen weight rows is eight gate rows and the eight up rows of the same columns.
template <int MI, int NI, int WM, int WN, int KG, int STAGES, int END>
__global__ __launch_bounds__(64 * WM * WN * KG) void gemm_lds_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, void* __restrict__ out, int M, int N, int K,
    long long ldw, long long ldo, int tiles_m, int tiles_n, int parts, int steps_per_part, long long part_stride,
    long long up_offset, GateAct act) {
  constexpr int BM = 16 * MI * WM, BN = 16 * NI * WN, WAVES = WM * WN * KG, T = 2 / KG;
  constexpr int GROUPS = (BM + BN) / 8, LOADS = GROUPS / WAVES, MORE = GROUPS % WAVES;   // groups of eight rows: one load of a wave each
  constexpr int STAGE = (BM + BN) * 8;              // 16-byte units of a stage
  constexpr int COLUMNS = END == END_GATED ? BN / 2 : BN;
  extern __shared__ __attribute__((aligned(16))) uintx4 lds[];     // [STAGES][BM + BN rows][8]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Block b runs on XCD b % 8.  An XCD takes a run of neighbouring tiles, rows of x fastest, so that the blocks that
  // share weight rows find them in their L2.
  const int tiles = tiles_m * tiles_n * parts;
  const int xcd = blockIdx.x % XCDS, per = tiles / XCDS, rest = tiles % XCDS;
  int tile = xcd * per + min(xcd, rest) + blockIdx.x / XCDS;
  const int m0 = tile % tiles_m * BM;
  tile /= tiles_m;
  const int n0 = tile % tiles_n * COLUMNS, part = tile / tiles_n;
  const int steps = K / KSTEP, first = part * steps_per_part, last = min(steps, first + steps_per_part);

  // this lane's place in each of the wave's loads; rows beyond M and N read the last row again (never stored)
  const bf16_t* from[LOADS + 1];
#pragma unroll
  for (int i = 0; i <= LOADS; ++i) {
    const int row = min((wave + WAVES * i) * 8 + (lane >> 3), BM + BN - 1);
    const int chunk = (lane & 7) ^ (row & 7);
    if (row < BM) from[i] = x + (size_t)min(m0 + row, M - 1) * K + chunk * 8;
    else {
      const int j = row - BM;
      if (END == END_GATED) from[i] = w + (size_t)min(n0 + (j >> 4) * 8 + (j & 7), N - 1) * ldw + ((j & 8) ? up_offset : 0) + chunk * 8;
      else from[i] = w + (size_t)min(n0 + j, N - 1) * ldw + chunk * 8;
    }
  }
  auto load = [&](int step, int stage) {       // past the end the last step again, so that the waits can count
    const int k0 = min(step, last - 1) * KSTEP;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) load_to_lds(from[i] + k0, &lds[stage * STAGE + (wave + WAVES * i) * 64]);
    if (MORE > 0 && wave < MORE) load_to_lds(from[LOADS] + k0, &lds[stage * STAGE + (wave + WAVES * LOADS) * 64]);
  };
  const int r = lane & 15, q = lane >> 4, group = wave / (WM * WN), wm = wave % WM, wn = wave / WM % WN;
  const unsigned int base = (unsigned int)(size_t)(const __attribute__((address_space(3))) char*)&lds[0];
  const unsigned int x_at = base + (wm * 16 * MI + r) * 128, w_at = base + (BM + wn * 16 * NI + r) * 128;
  floatx4 acc[MI][NI];
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
      multiply(a, b);
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
    if (group > 0) return;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] += meet[(wave * MI * NI + i * NI + j) * 64 + lane];
  }
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int m = m0 + (wm * MI + i) * 16 + r;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      if constexpr (END == END_GATED) {
        // lanes q = 0, 1 hold gate columns 4 q .. + 3 of the fragment's eight, lanes q = 2, 3 the up columns of lane - 32
        bf16_t y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[i][j][e]), __float_as_uint(acc[i][j][e]), false, false);
          y[e] = float_to_bf16(gate_times(acc[i][j][e], __uint_as_float(sw[1]), act));
        }
        const int n = n0 + (wn * NI + j) * 8 + 4 * (q & 1);
        if (q < 2 && m < M) {
          bf16_t* to = (bf16_t*)out + (size_t)m * ldo + n;
          if (n + 3 < N && (ldo & 3) == 0 && ((uintptr_t)out & 7) == 0)
            *(uint2*)to = make_uint2((unsigned)y[0] | ((unsigned)y[1] << 16), (unsigned)y[2] | ((unsigned)y[3] << 16));
          else
            for (int e = 0; e < 4; ++e) if (n + e < N) to[e] = y[e];
        }
      } else {
        const int n = n0 + (wn * NI + j) * 16 + 4 * q;
        if (m >= M) continue;
        if constexpr (END == END_PARTS) {
          float* to = (float*)out + (size_t)part * part_stride + (size_t)m * ldo + n;
          if (n + 3 < N && (ldo & 3) == 0 && (part_stride & 3) == 0 && ((uintptr_t)out & 15) == 0) *(floatx4*)to = acc[i][j];
          else
            for (int e = 0; e < 4; ++e) if (n + e < N) to[e] = acc[i][j][e];
        } else {
          bf16_t* to = (bf16_t*)out + (size_t)m * ldo + n;
          bf16_t y[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = float_to_bf16(acc[i][j][e]);
          if (n + 3 < N && (ldo & 3) == 0 && ((uintptr_t)out & 7) == 0)
            *(uint2*)to = make_uint2((unsigned)y[0] | ((unsigned)y[1] << 16), (unsigned)y[2] | ((unsigned)y[3] << 16));
          else
            for (int e = 0; e < 4; ++e) if (n + e < N) to[e] = y[e];
        }
      }
    }
  }
}

// The fragments' reads are waited for by hand: a build that spills registers would move values that are still in flight,
// and is never launched.  Also raises the kernel's LDS limit.  0: not yet asked, 1: fit, -1: refused.
static int fit_to_launch(const void* kernel, size_t lds_bytes, int* checked) {
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

template <int MI, int NI, int WM, int WN, int KG, int STAGES, int END>
static int launch_tile(const void* x, const void* w, void* out, int M, int N, int K, long long ldw, long long ldo, int parts,
                       long long part_stride, GateAct act, hipStream_t stream) {
  constexpr int BM = 16 * MI * WM, BN = 16 * NI * WN, COLUMNS = END == END_GATED ? BN / 2 : BN;
  constexpr size_t bytes = (size_t)STAGES * (BM + BN) * 128;
  static_assert(bytes <= 160 * 1024 && bytes >= (size_t)(KG - 1) * BM * BN * 4, "LDS of a CU");
  static int checked = 0;
  auto kernel = gemm_lds_kernel<MI, NI, WM, WN, KG, STAGES, END>;
  const int fit = fit_to_launch((const void*)kernel, bytes, &checked);
  if (fit != FE_OK) return fit;
  const long long tiles_m = ((long long)M + BM - 1) / BM, tiles_n = ((long long)N + COLUMNS - 1) / COLUMNS;
  if (tiles_m * tiles_n * parts > 0x7fffffffLL) return FE_BAD_ARGUMENT;
  const int steps = K / KSTEP, per_part = (steps + parts - 1) / parts;
  kernel<<<(unsigned)(tiles_m * tiles_n * parts), 64 * WM * WN * KG, bytes, stream>>>(
      (const bf16_t*)x, (const bf16_t*)w, out, M, N, K, ldw, ldo, (int)tiles_m, (int)tiles_n, parts, per_part, part_stride,
      (long long)N * ldw, act);
  return fe_check_launch();
}

// Operands and endings as fe_gemm_wide's (ending 0: parts, 1: bfloat16, 2: gated); the caller has checked them.
// tile: rows of x x weight rows a block takes: 0: 32 x 32, 1: 64 x 32, 2: 64 x 64, 3: 64 x 80, 4: 64 x 96, 5: 128 x 64,
//   6: 128 x 128, 7: 128 x 160, 8: 32 x 64.
// FE_BAD_ARGUMENT also if the library was built with registers spilled to scratch memory: the kernel then never runs.
static int launch(const void* x, const void* w, void* out, int M, int N, int K, long long ldw, long long ldo, int ending,
                  int parts, long long part_stride, int tile, GateAct act, hipStream_t stream) {
#define FE_END(END, ...) return launch_tile<__VA_ARGS__, END>(x, w, out, M, N, K, ldw, ldo, parts, part_stride, act, stream)
#define FE_TILE(I, ...)                                                \
  case I:                                                              \
    if (ending == END_PARTS) FE_END(END_PARTS, __VA_ARGS__);           \
    else if (ending == END_BF16) FE_END(END_BF16, __VA_ARGS__);        \
    else if (ending == END_GATED) FE_END(END_GATED, __VA_ARGS__);      \
    break;
  switch (tile) {
    FE_TILE(0, 1, 2, 2, 1, 2, 10)
    FE_TILE(1, 2, 2, 2, 1, 2, 8)
    FE_TILE(2, 2, 2, 2, 2, 2, 4)
    FE_TILE(3, 1, 5, 4, 1, 2, 6)
    FE_TILE(4, 2, 3, 2, 2, 2, 4)
    FE_TILE(5, 4, 2, 2, 2, 2, 4)
    FE_TILE(6, 4, 4, 2, 2, 2, 4)
    FE_TILE(7, 4, 5, 2, 2, 2, 3)
    FE_TILE(8, 1, 2, 2, 2, 2, 6)
  }
#undef FE_TILE
#undef FE_END
  return FE_BAD_ARGUMENT;
}

}  // namespace through_lds

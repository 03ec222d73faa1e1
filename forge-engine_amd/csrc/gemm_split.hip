// float32 matrix product C[M,N] = A[M,K] * B[N,K]^T (+ bias[N]) of more rows than a decode step, on the matrix cores' bfloat16
// instruction, each operand in three bfloat16 parts (split_f32.h).
//
// The float32 MFMA does 154 TFLOP/s here, the bfloat16 one 1,440, which six products make 240.  What bounds this kernel is that, the
// splitting (3.5 instructions an element: a conversion of two, and a dot product with (-1, 0) that subtracts a part exactly) and
// what a CU's L1 delivers: of 56 us for 700 x 4,096 x 1,024 in tiles of 128 x 128 the products alone take 42, all else alone 32.
//
// Block = 16 MI WM rows of A x 16 NI WN rows of B, KG groups of WM x WN waves (16 MI x 16 NI each).  K is walked in steps of 32 KG
// through STAGES buffers in LDS, a group's 32 of a step each; the groups' sums meet at the end in their order.  A tile comes by
// `global_load_lds_dwordx4` straight from memory as float32, waited for by count; a wave splits the fragments that it reads.
// Large tiles have two groups that alternate, one splitting while the other multiplies (96 x 128 tiles of the product above 49 -> 43
// us); small ones, bound by latency, four groups that do the same at the same time (32 x 32, 20 rows: 12.2 -> 10.5).
// Measured on one MI355X against the float32 MFMA: 700 x 4,096 x 1,024 63 -> 48 us, 700 x 6,144 x 1,024 98 -> 71, 1,024 x 4,096 x
// 2,048 152 -> 110 (156 TFLOP/s), and against the weight streamed past registers once for every eight rows 60 x 4,096 x 1,024
// 52 -> 11.  Error against 64 bits 1.5e-7 of 4.1e-7 (700 x 4,096 x 1,024).
#include "split_f32.h"
#include "lds_tile.h"

namespace {

using lds_tile::bf16x8;
using lds_tile::floatx4;
using lds_tile::uintx4;
using lds_tile::load_to_lds;
using lds_tile::wait_loads;

constexpr int XCDS = 8;

template <int MI, int NI, int WM, int WN, int STAGES, int KG>
__global__ __launch_bounds__(64 * WM * WN * KG) void gemm_split_kernel(
    const float* __restrict__ A, const float* __restrict__ B, const float* __restrict__ bias, float* __restrict__ C,
    int M, int N, int K, long long lda, long long ldb, long long ldc, int tiles_m, int tiles_n, int parts, int steps_per_part,
    long long part_stride, int wide_store) {
  constexpr int BM = 16 * MI * WM, BN = 16 * NI * WN, BK = 32 * KG, CH = BK / 4, WAVES = WM * WN * KG;
  constexpr int LOADS = (BM + BN) * CH / (64 * WAVES);          // loads a wave and step
  constexpr bool ALTERNATE = KG == 2;
  static_assert((BM + BN) * CH % (64 * WAVES) == 0, "every wave loads as much as every other");
  static_assert(STAGES * (BM + BN) * BK >= (KG - 1) * BM * BN, "the groups' sums meet in the same LDS");
  extern __shared__ __attribute__((aligned(16))) floatx4 lds[];      // [STAGES][BM + BN rows][CH]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Block b runs on XCD b % 8.  An XCD takes a run of neighbouring tiles, rows of A fastest, so that the blocks that
  // share rows of B find them in their L2.
  const int tiles = tiles_m * tiles_n * parts, xcd = blockIdx.x % XCDS, per = tiles / XCDS, more = tiles % XCDS;
  int tile = xcd * per + min(xcd, more) + blockIdx.x / XCDS;
  const int m0 = (tile % tiles_m) * BM;
  tile /= tiles_m;
  const int n0 = (tile % tiles_n) * BN, part = tile / tiles_n;
  const int first = part * steps_per_part, steps = min((K + BK - 1) / BK, first + steps_per_part), whole = K / BK;      // this part's steps
  // the unit of a row that holds a chunk: sixteen lanes that read one chunk of sixteen rows touch every bank once
  auto swizzle = [](int row) { return row & 15; };

  const unsigned int base = __builtin_amdgcn_readfirstlane((unsigned int)(size_t)(const __attribute__((address_space(3))) char*)&lds[0]);
  const float* from[LOADS];      // this lane's row of each of the wave's loads (A's rows, then B's)
  int chunk[LOADS];              // ... and its place in that row
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int unit = (wave * LOADS + i) * 64 + lane, row = unit / CH;
    from[i] = row < BM ? A + (size_t)min(m0 + row, M - 1) * lda : B + (size_t)min(n0 + row - BM, N - 1) * ldb;
    chunk[i] = ((unit % CH) ^ swizzle(row)) * 4;
  }
  auto load = [&](int step, int stage) {       // chunks beyond K read the row's first
    const int k0 = step * BK;
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      load_to_lds(from[i] + (step < whole || k0 + chunk[i] < K ? k0 + chunk[i] : 0), base + (stage * (BM + BN) * CH + (wave * LOADS + i) * 64) * 16);
  };

  const int r = lane & 15, q = lane >> 4, group = wave / (WM * WN), wm = wave % WM, wn = wave / WM % WN;
  const split_f32::Minus minus = split_f32::minus();
  floatx4 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  bf16x8 a[MI][3], b[NI][3];
  // a group's 32 of a step: from LDS, split
  auto take = [&](int step, int stage) {
    const floatx4* at = lds + stage * (BM + BN) * CH;
    const int c = 8 * group + q;        // a lane's eight k: chunks c and c + 4, for A and B alike
    auto fragment = [&](int row, bf16x8 (&parts)[3]) {
      floatx4 u = at[row * CH + (c ^ swizzle(r))], v = at[row * CH + ((c + 4) ^ swizzle(r))];
      if (step >= whole) {        // chunks beyond K: nothing
        if (step * BK + c * 4 >= K) u = floatx4{0.f, 0.f, 0.f, 0.f};
        if (step * BK + c * 4 + 16 >= K) v = floatx4{0.f, 0.f, 0.f, 0.f};
      }
      split_f32::split8(u, v, minus, parts);
    };
#pragma unroll
    for (int i = 0; i < MI; ++i) fragment((wm * MI + i) * 16 + r, a[i]);
#pragma unroll
    for (int j = 0; j < NI; ++j) fragment(BM + (wn * NI + j) * 16 + r, b[j]);
  };
  auto multiply = [&]() {
#pragma unroll
    for (int j = 0; j < NI; ++j) split_f32::add_products<MI>(a, b[j], [&](int i) -> floatx4& { return acc[i][j]; });
  };
  auto barrier = []() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto landed = [&](int step, auto ahead) {      // this wave's share of `step`, behind which up to `ahead` further ones are under way
    constexpr int AHEAD = decltype(ahead)::value;
    if (step + AHEAD < steps) wait_loads<LOADS * AHEAD>();
    else wait_loads<0>();
  };
  int stage = 0, before = STAGES - 1;
  if constexpr (ALTERNATE) {
    // While one group takes its half of a step, the other multiplies its own, one phase behind: group 0 takes step s (counted from
    // the part's first) in phase 2 s and multiplies it in 2 s + 1, group 1 in 2 s + 1 and 2 s + 2.  A buffer is read for the last time in
    // phase 2 s + 1, so every wave fills it again from phase 2 s + 2 on, and every wave's share of step s must have landed at the end
    // of phase 2 s - 1.
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
      if (first + s < steps) load(first + s, s);
    landed(first, std::integral_constant<int, STAGES - 1>{});
    barrier();
    if (group == 1) barrier();
    for (int step = first; step < steps; ++step) {
      if (group == 0 && step > first && step - 1 + STAGES < steps) load(step - 1 + STAGES, before);
      take(step, stage);
      if (group == 1) landed(step + 1, std::integral_constant<int, STAGES - 2>{});
      barrier();
      if (group == 1 && step + STAGES < steps) load(step + STAGES, stage);
      __builtin_amdgcn_s_setprio(1);
      multiply();
      __builtin_amdgcn_s_setprio(0);
      if (group == 0) landed(step + 1, std::integral_constant<int, STAGES - 2>{});
      barrier();
      before = stage;
      stage = stage + 1 == STAGES ? 0 : stage + 1;
    }
    if (group == 0) barrier();
  } else {
    // The small tiles are what up to 64 rows take, whose sums were FMAs before: theirs go into the whole every four steps, so that the
    // instruction's cutting off stays small (20 rows through the 1.7B sizes: error against 64 bits 6.5e-7 -> 4.9e-7, with FMAs 4.9e-7).
    floatx4 whole_sum[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) whole_sum[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    auto gather = [&]() {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          whole_sum[i][j] += acc[i][j];
          acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    };
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
      if (first + s < steps) load(first + s, s);
    for (int step = first; step < steps; ++step) {
      landed(step, std::integral_constant<int, STAGES - 2>{});
      barrier();       // everyone's share is there, and everyone is done with the buffer that is filled next
      if (step + STAGES - 1 < steps) load(step + STAGES - 1, before);
      take(step, stage);
      multiply();
      if ((step - first) % 4 == 3) gather();
      before = stage;
      stage = stage + 1 == STAGES ? 0 : stage + 1;
    }
    gather();
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] = whole_sum[i][j];
  }
  if constexpr (KG > 1) {       // the groups' sums, added in the order of the groups
    __syncthreads();
    if (group > 0) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) lds[(((group - 1) * WM * WN + wave % (WM * WN)) * MI * NI + i * NI + j) * 64 + lane] = acc[i][j];
    }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int g = 1; g < KG; ++g)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] += lds[(((g - 1) * WM * WN + wave) * MI * NI + i * NI + j) * 64 + lane];
  }

  // lane (r, q) holds rows of B n0 + 16 j + 4 q .. + 3 for row of A m0 + 16 i + r: four neighbouring columns of C
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int m = m0 + (wm * MI + i) * 16 + r;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int n = n0 + (wn * NI + j) * 16 + 4 * q;
      floatx4 v = acc[i][j];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (!split_f32::finite(v[e]) && n + e < N) {
          const int k = first * BK;
          v[e] = split_f32::dot(A + (size_t)m * lda + k, B + (size_t)(n + e) * ldb + k, min(K, steps * BK) - k);
        }
      float* dst = C + (size_t)part * part_stride + (size_t)m * ldc + n;
      if (bias)
        for (int e = 0; e < 4; ++e) if (n + e < N) v[e] += bias[n + e];
      if (wide_store && n + 3 < N) *(floatx4*)dst = v;
      else
        for (int e = 0; e < 4; ++e) if (n + e < N) dst[e] = v[e];
    }
  }
}

template <int MI, int NI, int WM, int WN, int STAGES, int KG>
int launch(const float* A, const float* B, const float* bias, float* C, int M, int N, int K, long long lda, long long ldb,
           long long ldc, int parts, long long part_stride, hipStream_t stream) {
  constexpr int BM = 16 * MI * WM, BN = 16 * NI * WN, BK = 32 * KG;
  constexpr size_t bytes = (size_t)STAGES * (BM + BN) * BK * 4;
  static_assert(bytes <= 160 * 1024, "LDS of a CU");
  static std::atomic<bool> raised{false};
  auto kernel = gemm_split_kernel<MI, NI, WM, WN, STAGES, KG>;
  const int limit_raised = lds_tile::raise_lds_limit((const void*)kernel, bytes, &raised);
  if (limit_raised != FE_OK) return limit_raised;
  const long long tiles_m = ((long long)M + BM - 1) / BM, tiles_n = ((long long)N + BN - 1) / BN;
  if (tiles_m * tiles_n * parts > 0x7fffffffLL) return FE_BAD_ARGUMENT;
  const int wide_store = ldc % 4 == 0 && part_stride % 4 == 0 && (((uintptr_t)C) & 15) == 0;
  const int steps = (K + BK - 1) / BK;
  kernel<<<dim3((unsigned)(tiles_m * tiles_n * parts)), 64 * WM * WN * KG, bytes, stream>>>(
      A, B, bias, C, M, N, K, lda, ldb, ldc, (int)tiles_m, (int)tiles_n, parts, (steps + parts - 1) / parts, part_stride, wide_store);
  return fe_check_launch();
}

}  // namespace

// A [M, K], B [N, K] float32, rows 16-byte aligned (strides lda, ldb), K a multiple of four; bias [N] or null; C holds `parts` matrices
// [M, N] (row stride ldc) part_stride floats apart, each the sum over a run of whole steps of K (zeros where it has none), whose sum
// is the product; with a bias one.  tile: rows of A x rows of B a block takes: 0: 128 x 160, 1: 128 x 128, 2: 96 x 128, 3: 128 x 64,
// 4: 96 x 64, 5: 64 x 64, 6: 32 x 32.
extern "C" int fe_gemm_split(const float* A, const float* B, const float* bias, float* C, int M, int N, int K, long long lda,
                             long long ldb, long long ldc, int parts, long long part_stride, int tile, hipStream_t stream) {
  if (M <= 0 || N <= 0) return FE_OK;
  if (K < 4 || K % 4 || lda < K || ldb < K || ldc < N || lda % 4 || ldb % 4 || ((((uintptr_t)A) | ((uintptr_t)B)) & 15)) return FE_BAD_ARGUMENT;
  if (parts < 1 || parts > 64 || (parts > 1 && (bias || part_stride < (long long)M * ldc))) return FE_BAD_ARGUMENT;
#define FE_TILE(I, ...) case I: return launch<__VA_ARGS__>(A, B, bias, C, M, N, K, lda, ldb, ldc, parts, part_stride, stream);
  switch (tile) {
    FE_TILE(0, 4, 5, 2, 2, 2, 2)
    FE_TILE(1, 4, 4, 2, 2, 2, 2)
    FE_TILE(2, 3, 4, 2, 2, 2, 2)
    FE_TILE(3, 4, 2, 2, 2, 3, 2)
    FE_TILE(4, 3, 2, 2, 2, 3, 2)
    FE_TILE(5, 2, 2, 2, 2, 2, 4)
    FE_TILE(6, 1, 1, 2, 2, 2, 4)
  }
#undef FE_TILE
  return FE_BAD_ARGUMENT;
}

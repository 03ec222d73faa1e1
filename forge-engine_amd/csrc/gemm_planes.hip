// float32 matrix product C[M,N] = A[M,K] * B[N,K]^T (+ bias[N]) of the rows of prompts, each operand in three bfloat16 parts (split_f32.h) and
// A split ahead, by a launch of its own: [3][M][K] planes of bfloat16, which a block then fetches like any bfloat16 operand.
// (gemm_split splits a fragment wherever it is used: every element of A by every block of its rows, in two waves of each.)
//
// Block = 16 MI rows of A x 64 NI rows of B, two groups of four waves, a wave 16 MI x 16 NI of them; K in steps of 64, 32 a group.  Planes and weight
// come by `global_load_lds_dwordx4`, two buffers each, the weight a step ahead of the planes: while a step's products are formed, its
// successor's weight is read, split and kept in registers, once for all rows.  The order of a step is written out: a row tile's planes are
// read two ahead, the step's loads go out one after the other over the first rows (their addresses pass one by one: issued at once they held
// everything up), and between two MFMAs stand two vector instructions of the sums of the row before or of the splitting.
//
// What bounds it: a step of 128 x 128 takes 1.7 us (1.9 with the weight coming from memory) of 1.28 that its MFMAs do (2.1 with the small products added to the long sum at every step
// and loads issued at once; without loads .16 less, without the planes' reads .3, without splitting .2), a round of tiles another 4 to 7 us:
// the first loads' way, the groups' meeting, the stores.  Measured on one MI355X against gemm_split, us, both with the pass over A: 700 x
// 4,096 x 1,024 48 -> 42, x 6,144 x 1,024 68 -> 59, x 12,288 x 2,048 257 -> 190, x 2,048 x 6,144 130 -> 100.  Error against 64 bits
// 8.2e-8 of 1.49e-7 (700 x 6,144 x 1,024; 1.31e-7 in the tiles that do not gather, below): the products of the first parts and the others'
// are summed apart, to the end.
#include "split_f32.h"
#include "lds_load.h"
#include "lds_tile.h"

namespace {

using lds_load::load_to_lds;
using split_f32::bf16x2;
using split_f32::bf16x8;
using split_f32::split2;
using split_f32::split8;
using lds_tile::floatx4;
using lds_tile::wait_loads;

constexpr int XCDS = 8, KSTEP = 64, GROUPS = 2, WAVES = 8;

// A [M, K] float32 as planes [3][M][KP] bfloat16, zeros beyond K: eight elements a thread
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ A, bf16_t* __restrict__ planes, int M, int K, int KP, long long lda) {
  const long long unit = (long long)blockIdx.x * 256 + threadIdx.x, per_row = KP / 8;
  const int row = (int)(unit / per_row), k = (int)(unit % per_row) * 8;
  if (row >= M) return;
  const float* from = A + (size_t)row * lda + k;
  floatx4 u = {0.f, 0.f, 0.f, 0.f}, v = u;
  if (k < K) u = *(const floatx4*)from;
  if (k + 4 < K) v = *(const floatx4*)(from + 4);
  bf16x8 parts[3];
  split8(u, v, parts);
#pragma unroll
  for (int i = 0; i < 3; ++i) *(bf16x8*)(planes + ((size_t)i * M + row) * KP + k) = parts[i];
}

template <int MI, int NI>
__global__ __launch_bounds__(64 * WAVES) void gemm_planes_kernel(
    const bf16_t* __restrict__ planes, const float* __restrict__ A, const float* __restrict__ B, const float* __restrict__ bias, float* __restrict__ C,
    int M, int N, int K, int KP, long long lda, long long ldb, long long ldc, int tiles_m, int tiles_n, int parts, long long part_stride, int wide_store) {
  constexpr int BM = 16 * MI, BN = 64 * NI;
  constexpr int X_BYTES = 3 * BM * 128, W_BYTES = BN * 256;
  constexpr int DEPTH = MI * NI >= 16 ? 2 : 3;      // row tiles of planes in registers: the largest tile has no room for three
  constexpr int X_GROUPS = 3 * BM / 8, X_LOADS = (X_GROUPS + WAVES - 1) / WAVES, W_LOADS = BN / 4 / WAVES;
  static_assert(X_LOADS + W_LOADS <= 3 * MI, "a step's loads are spread over its rows");
  extern __shared__ __attribute__((aligned(16))) char lds[];      // [2][3 planes][BM rows][8 chunks], then [2][BN rows][16 chunks]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tiles = tiles_m * tiles_n * parts, xcd = blockIdx.x % XCDS, per = tiles / XCDS, more = tiles % XCDS;
  int tile = xcd * per + min(xcd, more) + blockIdx.x / XCDS;
  const int m0 = (tile % tiles_m) * BM;
  tile /= tiles_m;
  const int n0 = (tile % tiles_n) * BN, part = tile / tiles_n;
  const int all = KP / KSTEP, first = (int)((long long)part * all / parts), last = (int)((long long)(part + 1) * all / parts);
  const unsigned int lds_at = __builtin_amdgcn_readfirstlane((unsigned int)(size_t)(const __attribute__((address_space(3))) char*)lds);

  unsigned int x_off[X_LOADS], x_to[X_LOADS], w_off[W_LOADS];
#pragma unroll
  for (int i = 0; i < X_LOADS; ++i) {
    const int rows8 = min(wave + WAVES * i, X_GROUPS - 1), row = rows8 * 8 + (lane >> 3), plane = row / BM;
    x_off[i] = ((unsigned int)plane * M + min(m0 + row - plane * BM, M - 1)) * (unsigned int)(KP * 2) + ((lane & 7) ^ (lane >> 3)) * 16;
    x_to[i] = lds_at + rows8 * 1024;
  }
  const int w_row = wave * W_LOADS * 4 + (lane >> 4);
#pragma unroll
  for (int i = 0; i < W_LOADS; ++i)
    w_off[i] = (unsigned int)min(w_row + 4 * i, N - 1 - n0) * (unsigned int)(ldb * 4) + ((lane & 15) ^ ((w_row + 4 * i) & 15)) * 16;
  auto load_x = [&](int i, int step, int stage) { load_to_lds(planes + (size_t)step * KSTEP, x_off[i], x_to[i] + stage * X_BYTES); };
  auto load_w = [&](int i, int step, int stage) {
    const float* from = B + (size_t)n0 * ldb + (size_t)step * KSTEP;
    unsigned int off = w_off[i];
    if ((step + 1) * KSTEP > K) {      // chunks beyond K read the step's first: the planes hold zeros there
      const unsigned int k = ((lane & 15) ^ ((w_row + 4 * i) & 15)) * 4;
      if (step * KSTEP + k >= K) off -= k * 4;
    }
    load_to_lds(from, off, lds_at + 2 * X_BYTES + stage * W_BYTES + (wave * W_LOADS + i) * 1024);
  };

  const int r = lane & 15, q = lane >> 4, group = wave >> 2, wn = wave & 3;
  floatx4 acc[MI][NI], small[MI][NI] = {};
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  const char* a_at = lds + r * 128 + ((4 * group + q) ^ (r & 7)) * 16;
  const char* b_at = lds + 2 * X_BYTES + (wn * 16 * NI + r) * 256;
  const int b_chunk = 8 * group + 2 * q;
  auto take_w = [&](int stage, floatx4 (&raw)[NI][2]) {
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int e = 0; e < 2; ++e) raw[j][e] = *(const floatx4*)(b_at + stage * W_BYTES + j * 4096 + ((b_chunk + e) ^ r) * 16);
  };
  auto take_x = [&](int stage, int i, bf16x8 (&a)[3]) {
#pragma unroll
    for (int p = 0; p < 3; ++p) a[p] = *(const bf16x8*)(a_at + stage * X_BYTES + (p * BM + 16 * i) * 128);
  };

  floatx4 raw[NI][2];
  bf16x8 b0[NI][3], b1[NI][3];
  // The instruction cuts off what an addend has below the last bit of a larger sum: where registers are left, a sum goes into the whole every
  // four steps (700 x 1,024 x 3,072 in three parts: error against 64 bits 1.30e-7 -> 1.0e-7; gemm_split in four 1.29e-7).
  constexpr bool GATHER = MI * NI <= 10;
  floatx4 whole[GATHER ? MI : 1][NI] = {};
  auto gather = [&]() {
#pragma unroll
    for (int i = 0; i < (GATHER ? MI : 0); ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        whole[i][j] += acc[i][j];
        acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
  };
  // a step: its products of b, the weight of the next one into `b_next`
  auto step_of = [&](int step, int stage, bf16x8 (&b)[NI][3], bf16x8 (&b_next)[NI][3]) {
    wait_loads<0>();
    lds_tile::reads_done_barrier();
    constexpr int OF_X[5] = {2, 0, 1, 1, 0}, OF_W[5] = {0, 2, 1, 0, 1};
    bf16x8 a[DEPTH][3];

    take_x(stage, 0, a[0]);
    if (DEPTH == 3) take_x(stage, 1, a[1]);
    take_w(1 - stage, raw);      // (behind the last step: what is there, for nobody)
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      if (i + DEPTH - 1 < MI) take_x(stage, i + DEPTH - 1, a[(i + DEPTH - 1) % DEPTH]);
      // the loads' addresses pass one after the other: spread over the first rows, they do not hold up the products
#pragma unroll
      for (int n = 0; n < X_LOADS + W_LOADS; ++n)
        if (n / 3 == i) {
          if (n < X_LOADS) { if (step + 1 < last) load_x(n, step + 1, 1 - stage); }
          else if (step + 2 < last) load_w(n - X_LOADS, step + 2, stage);
        }
      __builtin_amdgcn_sched_barrier(0);
      bf16x8 (&x)[3] = a[i % DEPTH];
#pragma unroll
      for (int p = 0; p < 5; ++p)
#pragma unroll
        for (int j = 0; j < NI; ++j)
          small[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j][OF_W[p]], x[OF_X[p]], small[i][j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j][0], x[0], acc[i][j], 0, 0, 0);
      if (i >= 1 && i <= NI) {
        split8(raw[i - 1][0], raw[i - 1][1], b_next[i - 1]);
#pragma unroll
        for (int p = 0; p < 3; ++p) asm volatile("" : "+v"(b_next[i - 1][p]));
      }
#pragma unroll
      for (int z = 0; z < 6 * NI; ++z) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);      // an MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);      // two vector instructions
      }
    }
  };
#pragma unroll
  for (int i = 0; i < W_LOADS; ++i) load_w(i, first, 0);
#pragma unroll
  for (int i = 0; i < X_LOADS; ++i) load_x(i, first, 0);
  if (first + 1 < last)
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) load_w(i, first + 1, 1);
  wait_loads<0>();
  lds_tile::reads_done_barrier();
  take_w(0, raw);
#pragma unroll
  for (int j = 0; j < NI; ++j) split8(raw[j][0], raw[j][1], b0[j]);
  int step = first;
  for (; step + 1 < last; step += 2) {
    step_of(step, 0, b0, b1);
    step_of(step + 1, 1, b1, b0);
    if (GATHER && ((step - first) & 2)) gather();
  }
  if (step < last) step_of(step, 0, b0, b1);
  if constexpr (GATHER) {
    gather();
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] = whole[i][j];
  }

#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] += small[i][j];
  // The groups' sums meet: each hands the other the rows that it does not store, the first group the rows from FIRST on.  The first
  // group's sum is the first addend everywhere.
  constexpr int FIRST_ROWS = (MI + 1) / 2;
  lds_tile::reads_done_barrier();
  floatx4* meet = (floatx4*)lds + wn * MI * NI * 64 + lane;
  static_assert(2 * (X_BYTES + W_BYTES) >= 4 * MI * NI * 64 * 16, "the groups' sums meet in the same LDS");
  auto in_mine = [&](int i) { return (i < FIRST_ROWS) == (group == 0); };
#pragma unroll
  for (int i = 0; i < MI; ++i)
    if (!in_mine(i))
#pragma unroll
      for (int j = 0; j < NI; ++j) meet[(i * NI + j) * 64] = acc[i][j];
  __syncthreads();
  // lane (r, q) holds rows of B n0 + 16 j + 4 q .. + 3 for row of A m0 + 16 i + r: four neighbouring columns of C
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    if (!in_mine(i)) continue;
    const int m = m0 + i * 16 + r;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const floatx4 other = meet[(i * NI + j) * 64];
      floatx4 v = group ? other + acc[i][j] : acc[i][j] + other;
      const int n = n0 + (wn * NI + j) * 16 + 4 * q;
      if (m >= M) continue;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (!split_f32::finite(v[e]) && n + e < N) {
          const int k = first * KSTEP;
          v[e] = split_f32::dot(A + (size_t)m * lda + k, B + (size_t)(n + e) * ldb + k, min(K, last * KSTEP) - k);
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

template <int MI, int NI>
int launch(const bf16_t* planes, const float* A, const float* B, const float* bias, float* C, int M, int N, int K, long long lda, long long ldb,
           long long ldc, int parts, long long part_stride, hipStream_t stream) {
  constexpr int BM = 16 * MI, BN = 64 * NI;
  constexpr size_t bytes = 2 * (3 * BM * 128 + BN * 256);
  static_assert(bytes <= 160 * 1024, "LDS of a CU");
  static std::atomic<bool> raised{false};
  auto kernel = gemm_planes_kernel<MI, NI>;
  const int limit_raised = lds_tile::raise_lds_limit((const void*)kernel, bytes, &raised);
  if (limit_raised != FE_OK) return limit_raised;
  const long long tiles_m = ((long long)M + BM - 1) / BM, tiles_n = ((long long)N + BN - 1) / BN;
  if (tiles_m * tiles_n * parts > 0x7fffffffLL) return FE_BAD_ARGUMENT;
  const int wide_store = ldc % 4 == 0 && part_stride % 4 == 0 && (((uintptr_t)C) & 15) == 0;
  kernel<<<dim3((unsigned)(tiles_m * tiles_n * parts)), 64 * WAVES, bytes, stream>>>(
      planes, A, B, bias, C, M, N, K, (K + KSTEP - 1) / KSTEP * KSTEP, lda, ldb, ldc, (int)tiles_m, (int)tiles_n, parts, part_stride, wide_store);
  return fe_check_launch();
}

}  // namespace

// A [M, K], B [N, K] float32, rows 16-byte aligned (strides lda, ldb), K a multiple of four; planes: room for 3 M bfloat16 rows of K rounded up
// to 64, less than 4 GB; bias [N] or null; C holds `parts` matrices [M, N] (row stride ldc) part_stride floats apart, each the sum over a run of whole
// steps of K, whose sum is the product; with a bias one.  A block takes 16 rows16 rows of A x 64 columns64 rows of B.
// ready: the planes hold A's parts already (who made A stored them beside it).
extern "C" int fe_gemm_planes(const float* A, void* planes, const float* B, const float* bias, float* C, int M, int N, int K, long long lda,
                              long long ldb, long long ldc, int parts, long long part_stride, int rows16, int columns64, int ready, hipStream_t stream) {
  if (M < 1 || N < 1) return FE_OK;
  if (K < 4 || K % 4 || lda < K || ldb < K || ldc < N || lda % 4 || ldb % 4 || ldb >= (1 << 22)) return FE_BAD_ARGUMENT;
  if ((((uintptr_t)planes) | ((uintptr_t)A) | ((uintptr_t)B)) & 15) return FE_BAD_ARGUMENT;
  const int KP = (K + KSTEP - 1) / KSTEP * KSTEP;
  if (parts < 1 || parts > 64 || parts > KP / KSTEP || (parts > 1 && (bias || part_stride < (long long)M * ldc))) return FE_BAD_ARGUMENT;
  if (6LL * M * KP >= (1LL << 32)) return FE_BAD_ARGUMENT;
  if (!ready) {
    const long long blocks = ((long long)M * (KP / 8) + 255) / 256;
    split_rows_kernel<<<(unsigned)blocks, 256, 0, stream>>>(A, (bf16_t*)planes, M, K, KP, lda);
    const int split = fe_check_launch();
    if (split != FE_OK) return split;
  }
#define FE_TILE(MI, NI) \
  if (rows16 == MI && columns64 == NI) return launch<MI, NI>((const bf16_t*)planes, A, B, bias, C, M, N, K, lda, ldb, ldc, parts, part_stride, stream);
  FE_TILE(4, 1) FE_TILE(4, 2) FE_TILE(5, 2) FE_TILE(6, 1) FE_TILE(6, 2) FE_TILE(7, 2) FE_TILE(8, 1) FE_TILE(8, 2) FE_TILE(9, 1) FE_TILE(10, 1)
#undef FE_TILE
  return FE_BAD_ARGUMENT;
}

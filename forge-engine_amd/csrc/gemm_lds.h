// The product for portions (gemm_wide.hip) with both operands in LDS: one to hundreds of rows of x (requests decoding, a
// portion of a prompt):
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
// memory channel is hot), nor do four stages instead of three, nor loads that go out one by one between the MFMAs; without loads that product
// takes 25 of its 41.5 us, with lines that the L2 holds 34.  From 1,500 rows on tiles of 256 x 256 (gemm_big.hip) and the matrix library are ahead.
//
// Tiles of 96 rows (gemm_lds96.hip) stand between those of 64 and 128: they are the ones that fill a round with the fewest bytes where 64 make
// too many blocks and 128 too few (361 rows: 3,072 columns of gate/up, K = 1,024, 256 blocks of 96 x 96, 14.4 -> 12.0 us, 4,096 x 1,024
// stored in 96 x 64 9.8 -> 8.9, 2,048 x 6,144 in four parts in 96 x 128 22.6 -> 18.5).
//
// Up to 16 rows of x, tiles of 16 rows with one fragment a wave: the weight's bytes are nearly all of the tile's, so the widths
// (16 to 80 weight rows) only choose how evenly the CUs share them, and 8 to 12 stages keep 64 KB and more of a CU's share in
// flight; the kernels with the weight in registers had a wave's two to four steps, and read x again for every 16 weight rows
// (gemm_skinny) or gave a block 64 weight rows whatever the weight (gemm_wide).  8 rows, before -> this: gate/up of 3,072 x
// 1,024 8.3 -> 5.7, of 6,144 x 2,048 14.4 -> 12.8, of 9,728 x 2,560 22.4 -> 21.1; updates of 1,024 x 2,048 5.0 -> 3.1,
// of 2,560 x 9,728 12.2 -> 11.6; q/k/v of 4,096 x 1,024 4.7 -> 4.2; 6,144 x 2,048 stored 9.2 -> 7.7.
//
// MFMA 16x16x32 bf16 with A = W (16 weight rows), B = x^T (16 rows of x): lane l (r = l % 16, q = l / 16) supplies row r,
// k = 8 q .. + 8 of either and receives D[weight row 4 q + i][row of x r]: four neighbouring output columns of a row.
#pragma once
#include "common.h"
#include "gate_act.h"
#include "lds_tile.h"

namespace through_lds {

using lds_tile::floatx4;
using lds_tile::uintx4;
using lds_tile::KSTEP;

constexpr int XCDS = 8;
constexpr int END_PARTS = 0, END_BF16 = 1, END_GATED = 2, END_BOUNDED = 3;

// Rows whose norm's factor was left out (gemm_ring.hip): the sums of row m are multiplied by rsqrt(sum of squares[m][.] / width +
// eps) before anything else is done with them.  The factors are made from LDS, where the row's 256 partial sums of squares went
// ahead of the walk over K.
struct RowFactors {
  const float* squares;       // [M][256]
  float width, eps;
};
constexpr int SQUARES = 256, SQUARES_PITCH = SQUARES * 4 + 16;      // bytes from row to row in LDS: sixteen rows in different banks

// The tile of 32 x 32, of which a CU holds two: its last ten steps written out cost walks of 16 to 48 steps more than the requests that they
// save (us, written out -> fetched again: gate/up of 512 columns, K = 2,048 at 25 rows 6.95 -> 6.58, 768 of 2,560 at 53 8.09 -> 7.59, of K =
// 12,288 27.5 -> 27.0; every other tile 1 to 7 % the other way).
template <int MI, int NI, int WM, int WN>
constexpr bool refetches() {
  return MI == 1 && NI == 2 && WM == 2 && WN == 1;
}

// END_BOUNDED: `gate_bounded` of gate and up, both rounded to bfloat16 first, with the limit in act.cubic and alpha in act.linear: the bits of
// the bfloat16 ending and a launch of the activation behind it (8 rows of 2,048 through 4,096 in a captured graph:
// 6.6 -> 5.0 us).
// With a gated ending a fragment of sixteen weight rows is eight gate rows and the eight up rows of the same columns.
template <int MI, int NI, int WM, int WN, int KG, int STAGES, int END, bool SCALED, bool ONCE>
__global__ __launch_bounds__(64 * WM * WN * KG) void gemm_lds_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, void* __restrict__ out, int M, int N, int K,
    long long ldw, long long ldo, int tiles_m, int tiles_n, int parts, int steps_per_part, long long part_stride,
    long long up_offset, GateAct act, RowFactors factors) {
  constexpr int BM = 16 * MI * WM, BN = 16 * NI * WN;
  constexpr bool PAIRS = END == END_GATED || END == END_BOUNDED;
  constexpr int COLUMNS = PAIRS ? BN / 2 : BN;
  extern __shared__ __attribute__((aligned(16))) uintx4 lds[];     // [STAGES][BM + BN rows][8]
  // Block b runs on XCD b % 8.  An XCD takes a run of neighbouring tiles, rows of x fastest, so that the blocks that
  // share weight rows find them in their L2.
  const int tiles = tiles_m * tiles_n * parts;
  const int xcd = blockIdx.x % XCDS, per = tiles / XCDS, rest = tiles % XCDS;
  int tile = xcd * per + min(xcd, rest) + blockIdx.x / XCDS;
  const int m0 = tile % tiles_m * BM;
  tile /= tiles_m;
  const int n0 = tile % tiles_n * COLUMNS, part = tile / tiles_n;
  const int steps = K / KSTEP, first = part * steps_per_part, last = min(steps, first + steps_per_part);

  // rows beyond M and N read the last row again (never stored)
  auto row_of = [&](int row) -> const bf16_t* {
    if (row < BM) return x + (size_t)min(m0 + row, M - 1) * K;
    const int j = row - BM;
    if (PAIRS) return w + (size_t)min(n0 + (j >> 4) * 8 + (j & 7), N - 1) * ldw + ((j & 8) ? up_offset : 0);
    return w + (size_t)min(n0 + j, N - 1) * ldw;
  };
  constexpr int STAGE_BYTES = STAGES * (BM + BN) * 128;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4, wm = wave % WM, wn = wave / WM;
  if constexpr (SCALED) {
    static_assert(MI == 1 && WM == 1, "rows of x in one tile of sixteen");
    const unsigned int base = __builtin_amdgcn_readfirstlane((unsigned int)(size_t)(const __attribute__((address_space(3))) char*)&lds[0]);
    for (int m = __builtin_amdgcn_readfirstlane(wave); m < M; m += WN * KG)
      lds_tile::load_to_lds(factors.squares + m * SQUARES + lane * 4, base + STAGE_BYTES + m * SQUARES_PITCH);
  }
  floatx4 acc[MI][NI];
  if (!lds_tile::product<MI, NI, WM, WN, KG, STAGES, false, refetches<MI, NI, WM, WN>()>(lds, row_of, first, last, K, acc,
                                                                                         std::integral_constant<bool, ONCE>())) return;
  if constexpr (SCALED) {
    // Lane (r, q) adds up a quarter of row r's squares.  A wave's loads arrive in order, so its rows were there before its first
    // step of K, and behind that step's barrier everyone's.
    if (first < last) {
      const floatx4* from = (const floatx4*)((const char*)lds + STAGE_BYTES + min(r, M - 1) * SQUARES_PITCH) + q * (SQUARES / 16);
      floatx4 sum = from[0];
#pragma unroll
      for (int j = 1; j < SQUARES / 16; ++j) sum += from[j];
      const float factor = rsqrtf(sum_xor32(sum_xor16((sum[0] + sum[1]) + (sum[2] + sum[3]))) / factors.width + factors.eps);
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[0][j] *= factor;
    }
  }
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int m = m0 + (wm * MI + i) * 16 + r;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      if constexpr (PAIRS) {
        // lanes q = 0, 1 hold gate columns 4 q .. + 3 of the fragment's eight, lanes q = 2, 3 the up columns of lane - 32
        bf16_t y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[i][j][e]), __float_as_uint(acc[i][j][e]), false, false);
          if constexpr (END == END_BOUNDED)
            y[e] = float_to_bf16(gate_bounded(bf16_to_float(float_to_bf16(acc[i][j][e])), bf16_to_float(float_to_bf16(__uint_as_float(sw[1]))), act.cubic, act.linear));
          else
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

template <int MI, int NI, int WM, int WN, int KG, int STAGES, int END, bool SCALED = false>
static int launch_tile(const void* x, const void* w, void* out, int M, int N, int K, long long ldw, long long ldo, int parts,
                       long long part_stride, GateAct act, hipStream_t stream, RowFactors factors = {}) {
  constexpr int BM = 16 * MI * WM, BN = 16 * NI * WN, COLUMNS = END == END_GATED || END == END_BOUNDED ? BN / 2 : BN;
  const size_t bytes = lds_tile::Shape<MI, NI, WM, WN, KG, STAGES>::BYTES + (SCALED ? (M <= 8 ? 8 : 16) * SQUARES_PITCH : 0);
  static_assert(!SCALED || lds_tile::Shape<MI, NI, WM, WN, KG, STAGES>::BYTES + 16 * SQUARES_PITCH <= 160 * 1024, "LDS of a CU");
  const long long tiles_m = ((long long)M + BM - 1) / BM, tiles_n = ((long long)N + COLUMNS - 1) / COLUMNS;
  if (tiles_m * tiles_n * parts > 0x7fffffffLL) return FE_BAD_ARGUMENT;
  // one tile of x: no block reads another's weight rows (an instance of its own: asked at every load it cost prompts of 361 rows .3 %).  The
  // tile that fetches a walk's last step again does so past the caches too: by itself its walks of 4 to 16 steps are .3 to 3 % slower for it
  // in the mean and those of 32 2 % faster, but whole prompts gain (32 steps of 17 to 32 rows, its rows past the caches to in them, mean
  // ratio of the times at 0.6B, 1.7B and 4B: prompts .951, 1.004 and .967; decode 1.004, 1.007 and .999, at most 1.009).  Likely because the
  // last cache is left to rows that are read again; at 0.6B all of a layer's products have to pass, at 4B the first one is enough.
  static std::atomic<bool> raised[2];
  const bool once = tiles_m == 1;
  auto kernel = once ? gemm_lds_kernel<MI, NI, WM, WN, KG, STAGES, END, SCALED, true> : gemm_lds_kernel<MI, NI, WM, WN, KG, STAGES, END, SCALED, SCALED>;
  const int limit_raised = lds_tile::raise_lds_limit(
      (const void*)kernel, lds_tile::Shape<MI, NI, WM, WN, KG, STAGES>::BYTES + (SCALED ? 16 * SQUARES_PITCH : 0), &raised[once]);
  if (limit_raised != FE_OK) return limit_raised;
  const int steps = K / KSTEP, per_part = (steps + parts - 1) / parts;
  kernel<<<(unsigned)(tiles_m * tiles_n * parts), 64 * WM * WN * KG, bytes, stream>>>(
      (const bf16_t*)x, (const bf16_t*)w, out, M, N, K, ldw, ldo, (int)tiles_m, (int)tiles_n, parts, per_part, part_stride,
      (long long)N * ldw, act, factors);
  return fe_check_launch();
}

// Operands and endings as fe_gemm_wide's (ending 0: parts, 1: bfloat16, 2: gated); the caller has checked them.
#define FE_END(END, ...) return launch_tile<__VA_ARGS__, END>(x, w, out, M, N, K, ldw, ldo, parts, part_stride, act, stream)
#define FE_TILE(I, ...)                                                \
  case I:                                                              \
    if (ending == END_PARTS) FE_END(END_PARTS, __VA_ARGS__);           \
    else if (ending == END_BF16) FE_END(END_BF16, __VA_ARGS__);        \
    else if (ending == END_GATED) FE_END(END_GATED, __VA_ARGS__);      \
    break;
// tile: rows of x x weight rows a block takes: 0: 32 x 32, 1: 64 x 32, 2: 64 x 64, 3: 64 x 80, 4: 64 x 96, 5: 128 x 64,
//   6: 128 x 128, 7: 128 x 160, 8: 32 x 64, 9 to 13: 16 x 16, 32, 48, 64, 80.  (Templates: a source holds the tiles that it launches.)
template <typename T>
static int launch(const T* x, const T* w, void* out, int M, int N, int K, long long ldw, long long ldo, int ending,
                  int parts, long long part_stride, int tile, GateAct act, hipStream_t stream) {
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
    FE_TILE(9, 1, 1, 1, 1, 2, 12)
    FE_TILE(10, 1, 1, 1, 2, 2, 12)
    FE_TILE(11, 1, 1, 1, 3, 2, 9)
    FE_TILE(12, 1, 1, 1, 4, 2, 8)
    FE_TILE(13, 1, 1, 1, 5, 2, 10)
  }
  return FE_BAD_ARGUMENT;
}

// tile: 96064, 96096, 96128: 96 x 64, 96, 128.
template <typename T>
static int launch_96(const T* x, const T* w, void* out, int M, int N, int K, long long ldw, long long ldo, int ending,
                     int parts, long long part_stride, int tile, GateAct act, hipStream_t stream) {
  switch (tile) {
    FE_TILE(96064, 3, 2, 2, 2, 2, 4)
    FE_TILE(96096, 3, 3, 2, 2, 2, 4)
    FE_TILE(96128, 3, 4, 2, 2, 2, 4)
  }
  return FE_BAD_ARGUMENT;
}
#undef FE_TILE
#undef FE_END

// The bounded ending: tiles 9 to 13.
template <typename T>
static int launch_bounded(const T* x, const T* w, void* out, int M, int N, int K, long long ldw, long long ldo, int tile,
                          float limit, float alpha, hipStream_t stream) {
#define FE_TILE(I, ...) \
  case I: return launch_tile<__VA_ARGS__, END_BOUNDED>(x, w, out, M, N, K, ldw, ldo, 1, 0, GateAct{alpha, limit}, stream);
  switch (tile) {
    FE_TILE(9, 1, 1, 1, 1, 2, 12)
    FE_TILE(10, 1, 1, 1, 2, 2, 12)
    FE_TILE(11, 1, 1, 1, 3, 2, 9)
    FE_TILE(12, 1, 1, 1, 4, 2, 8)
    FE_TILE(13, 1, 1, 1, 5, 2, 10)
  }
#undef FE_TILE
  return FE_BAD_ARGUMENT;
}

// The same for up to 16 rows of x with row factors: tiles 9 to 13, endings parts and gated.  Two buffers fewer where two blocks
// share a CU's LDS, which the squares would keep from it.
template <typename T>
static int launch_scaled(const T* x, const T* w, void* out, int M, int N, int K, long long ldw, long long ldo, int ending,
                         int parts, long long part_stride, int tile, GateAct act, hipStream_t stream, RowFactors factors) {
#define FE_END(END, ...) return launch_tile<__VA_ARGS__, END, true>(x, w, out, M, N, K, ldw, ldo, parts, part_stride, act, stream, factors)
#define FE_TILE(I, ...)                                                \
  case I:                                                              \
    if (ending == END_PARTS) FE_END(END_PARTS, __VA_ARGS__);           \
    else if (ending == END_GATED) FE_END(END_GATED, __VA_ARGS__);      \
    break;
  switch (tile) {
    FE_TILE(9, 1, 1, 1, 1, 2, 12)
    FE_TILE(10, 1, 1, 1, 2, 2, 10)
    FE_TILE(11, 1, 1, 1, 3, 2, 7)
    FE_TILE(12, 1, 1, 1, 4, 2, 6)
    FE_TILE(13, 1, 1, 1, 5, 2, 10)
  }
#undef FE_TILE
#undef FE_END
  return FE_BAD_ARGUMENT;
}

}  // namespace through_lds

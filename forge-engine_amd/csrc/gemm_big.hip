// bfloat16 matrix products of whole prompts, x[M, K] * w[N, K]^T with hundreds to thousands of rows of x, with one of two endings:
// act(gate) * up as bfloat16 for a fused gate/up weight (gate rows first), or float32 sums of parts of K ([parts][M, N], the next
// norm adds them in order).
//
// Block = 256 rows of x x 256 weight rows (gated: 128 gate rows and their 128 up rows) x 64 of K a step, one block a CU, which takes
// tile after tile (its loads run on into the next tile while this one's sums leave).  Eight waves in two groups of four; a wave
// holds 128 x 64 sums as four quadrants of 64 x 32, the groups other rows of x.  Both operands go straight from memory into LDS
// (two buffers of four parts: rows 0 and 1, weight rows 0 and 1 of 128 each).
//
// A step is four phases, a phase half memory and half matrix: reads of one part from LDS and one part's loads from memory, then
// the sixteen MFMAs of a quadrant.  The two groups are half a phase apart: each SIMD has one wave of each, and while one
// multiplies the other reads (8 and 4 reads of 16 bytes a lane in turn, which is what a phase's MFMAs hide).  Two barriers a phase
// keep them there.  A part is loaded two phases after its buffer was last read and six phases before it is read again.
// 2,480 clocks a step, of which the MFMAs are 2,048, in a launch of any size.
//
// What bounds it: power.  With all CUs at work the clock falls from 2.4 to 1.7 GHz (4,096 x 4,096 x 8,192: 317,000 clocks are 132 us
// with 16 blocks of the launch and 181 with 256: 1.52 PFLOP/s), so fewer instructions are what helps: m0 not saved around a load (1.43 ->
// 1.44 PFLOP/s), no priorities (1.44 -> 1.456), a sum's two halves of K one after the other (1.52 -> 1.54, another card).  The same
// tile in four waves of 128 x 128 reads a third less from LDS, but its one wave a SIMD waits at every load that it issues: 2,960
// clocks a step, 1.39.
//
// The last round of tiles is rarely full: a tile of 128 rows of x (two phases a step, three buffers) takes .62 of a whole one's
// time, and the columns beyond whole rounds go in such tiles where that is less.
//
// Measured on one MI355X, us, before (gemm_tile, or the matrix library and the gate kernel) -> this: gate/up of 9,728 columns, K = 2,560 at
// 768 / 2,048 / 4,096 / 6,001 rows 83 -> 68, 214 -> 175, 388 -> 310, 574 -> 477 (1.25 PFLOP/s), of 3,072 columns, K = 1,024 at 8,192
// 116 -> 96, of 12,288, K = 4,096 at 3,000 608 -> 468; an update of 2,560 x 9,728 with its norm at 2,048 rows in three parts 117 -> 100.
//
// MFMA 16x16x32 bf16 with A = W (16 weight rows), B = x^T (16 rows of x): lane l (r = l % 16, q = l / 16) supplies row r,
// k = 8 q .. + 8 of either and receives D[weight row 4 q + i][row of x r]: four neighbouring output columns of a row.
#include "common.h"
#include "gate_act.h"
#include "lds_load.h"
#include "lds_tile.h"
#include <algorithm>

namespace {

using lds_load::load_to_lds;
using lds_tile::bf16x8;
using lds_tile::floatx4;
using lds_tile::uintx4;
using lds_tile::wait_loads;

constexpr int CUS = 256, XCDS = 8, KSTEP = 64, THREADS = 512;
constexpr int HALF = 128, PART_BYTES = HALF * 128;
constexpr int END_PARTS = 0, END_GATED = 1;

__device__ __forceinline__ void barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

struct Product {
  const bf16_t *x, *w;
  void* out;
  int M, N, steps;
  unsigned int row_bytes, weight_row_bytes;      // from row to row
  long long ldo, part_stride, up_bytes;          // up_bytes: from a gate row to its up row
  GateAct act;
};
// Tiles of 128 HEIGHT rows and `columns` columns each, from column `n0` on: `band` tiles of rows at a time (neighbouring tiles, which an
// XCD takes together, share rows and weight rows in its L2), part by part of K.
struct Region {
  int tiles_m, tiles_n, parts, band, n0;
};

template <int END, int HEIGHT>
__device__ __forceinline__ void walk(const Product& p, const Region& region, char* lds) {
  constexpr int ROWS = HALF * HEIGHT, COLUMNS = END == END_GATED ? HALF : 2 * HALF;
  constexpr int STAGES = HEIGHT == 2 ? 2 : 3, PARTS = HEIGHT + 2, STAGE_BYTES = PARTS * PART_BYTES;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4, group = wave >> 2, wc = wave & 3;
  const unsigned int lds_at = __builtin_amdgcn_readfirstlane((unsigned int)(size_t)(const __attribute__((address_space(3))) char*)lds);

  // Block b runs on XCD b % 8, which takes a run of a round's neighbouring tiles.
  const int tiles = region.tiles_m * region.tiles_n * region.parts, rounds = (tiles + CUS - 1) / CUS;
  struct Tile { int m0, n0, part, first, count; };      // count: steps of K, none if this block has no tile in the round
  auto tile_of = [&](int round) -> Tile {
    const int base = round * CUS, here = min(CUS, tiles - base);
    const int xcd = blockIdx.x % XCDS, per = here / XCDS, rest = here % XCDS, slot = blockIdx.x / XCDS;
    if (slot >= per + (xcd < rest)) return Tile{0, 0, 0, 0, 0};
    int id = base + xcd * per + min(xcd, rest) + slot;
    const int each = region.tiles_m * region.tiles_n, part = id / each;
    id -= part * each;
    const int band = id / (region.band * region.tiles_n), in_band = id - band * region.band * region.tiles_n;
    const int rows = min(region.band, region.tiles_m - band * region.band);
    const int first = part * p.steps / region.parts;
    return Tile{(band * region.band + in_band % rows) * ROWS, region.n0 + in_band / rows * COLUMNS, part, first,
                (part + 1) * p.steps / region.parts - first};
  };
  Tile tile = tile_of(0);
  if (tile.count == 0) return;

  // Where the loads are.  A part is two loads of a wave, eight rows each; rows beyond M and N read the last row again (never stored).
  // LDS holds a row as eight chunks of 16 bytes, chunk c of row j at c ^ (j % 8).
  int load_round = 0, load_left;
  const char *x_at, *w_at;
  unsigned int x_off[2 * HEIGHT], w_off[4];
  const unsigned int chunk = ((lane & 7) ^ (lane >> 3)) * 16;
  auto aim = [&](const Tile& t) {
    x_at = (const char*)p.x + (size_t)t.m0 * p.row_bytes + t.first * (KSTEP * 2);
    w_at = (const char*)p.w + (size_t)t.n0 * p.weight_row_bytes + t.first * (KSTEP * 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = (i >> 1) * HALF + (i & 1) * 64 + wave * 8 + (lane >> 3);
      if (i < 2 * HEIGHT) x_off[i] = (unsigned int)min(row, p.M - 1 - t.m0) * p.row_bytes + chunk;
      w_off[i] = (unsigned int)min(END == END_GATED ? row & (HALF - 1) : row, p.N - 1 - t.n0) * p.weight_row_bytes + chunk;
    }
    load_left = t.count;
  };
  auto load_x = [&](auto half, unsigned int stage) {
    constexpr int H = decltype(half)::value;
#pragma unroll
    for (int i = 0; i < 2; ++i) load_to_lds(x_at, x_off[2 * H + i], lds_at + stage + H * PART_BYTES + i * 8192 + wave * 1024);
  };
  auto load_w = [&](auto half, unsigned int stage) {
    constexpr int G = decltype(half)::value;
    const char* from = END == END_GATED && G ? w_at + p.up_bytes : w_at;
#pragma unroll
    for (int i = 0; i < 2; ++i) load_to_lds(from, w_off[2 * G + i], lds_at + stage + (HEIGHT + G) * PART_BYTES + i * 8192 + wave * 1024);
  };
  auto advance = [&]() {      // behind the block's last step it stays there: that step's loads are issued again, for nobody
    if (load_left > 1) {
      --load_left;
      x_at += KSTEP * 2;
      w_at += KSTEP * 2;
    } else if (load_round + 1 < rounds) {
      const Tile t = tile_of(load_round + 1);
      if (t.count > 0) {
        ++load_round;
        aim(t);
      }
    }
  };
  auto next = [&](unsigned int stage) { return stage + STAGE_BYTES == STAGES * STAGE_BYTES ? 0u : stage + STAGE_BYTES; };
  const std::integral_constant<int, 0> zero;
  const std::integral_constant<int, 1> one;

  floatx4 acc[HEIGHT][2][4][2];      // [half of the rows][half of the weight rows][16 rows][16 weight rows]
  uintx4 a[4][2], b[2][2][2];        // [16 rows][half of K], [half][16 weight rows][half of K]
  auto clear = [&]() {
#pragma unroll
    for (int h = 0; h < HEIGHT; ++h)
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[h][g][i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  };
  const unsigned int a_lane[2] = {(group * 64 + r) * 128 + (q ^ (r & 7)) * 16u, (group * 64 + r) * 128 + ((4 + q) ^ (r & 7)) * 16u};
  const unsigned int b_lane[2] = {(wc * 32 + r) * 128 + (q ^ (r & 7)) * 16u, (wc * 32 + r) * 128 + ((4 + q) ^ (r & 7)) * 16u};
  auto read_a = [&](auto half, unsigned int stage) {
    constexpr int H = decltype(half)::value;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i][t] = *(const uintx4*)(lds + (a_lane[t] + stage) + H * PART_BYTES + i * 2048);
  };
  auto read_b = [&](auto half, unsigned int stage) {
    constexpr int G = decltype(half)::value;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 2; ++j) b[G][j][t] = *(const uintx4*)(lds + (b_lane[t] + stage) + (HEIGHT + G) * PART_BYTES + j * 2048);
  };
  // The end of a phase's memory half, and its matrix half.  PENDING: this wave's loads of the phases behind the one whose part is
  // read next, so that part has landed for every wave behind the barrier.  All reads of LDS have arrived before the second one.
  auto multiply = [&](auto h_, auto g_, auto pending) {
    constexpr int H = decltype(h_)::value, G = decltype(g_)::value;
    wait_loads<decltype(pending)::value>();
    barrier();
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          acc[H][G][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b[G][j][t]), __builtin_bit_cast(bf16x8, a[i][t]),
                                                                    acc[H][G][i][j], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
    __builtin_amdgcn_s_waitcnt(0xF | (0x3 << 14) | (0x7 << 4));      // lgkmcnt(0)
    barrier();
  };

  // The loads' order, a part each: weight 0, rows 0, weight 1 and (two halves of rows) rows 1 of step 0, then of step 1 ...; a phase
  // of two halves issues one part, six phases before it is read; of one half, the first phase one and the second two, four before.
  aim(tile);
  if constexpr (HEIGHT == 2) {
    load_w(zero, 0);
    load_x(zero, 0);
    load_w(one, 0);
    load_x(one, 0);
    advance();
    load_w(zero, STAGE_BYTES);
    load_x(zero, STAGE_BYTES);
    load_w(one, STAGE_BYTES);
    wait_loads<10>();
  } else {
    load_w(zero, 0);
    load_x(zero, 0);
    load_w(one, 0);
    advance();
    load_w(zero, STAGE_BYTES);
    load_x(zero, STAGE_BYTES);
    load_w(one, STAGE_BYTES);
    advance();
    load_w(zero, 2 * STAGE_BYTES);
    wait_loads<10>();
  }
  clear();
  barrier();
  if (group) barrier();
  read_b(zero, 0);
  unsigned int stage = 0;
  for (int round = 0;;) {
    for (int left = tile.count; left > 0; --left) {
      const unsigned int ahead = next(stage);
      if constexpr (HEIGHT == 2) {
        const std::integral_constant<int, 10> pending;
        read_a(zero, stage);
        load_x(one, ahead);
        multiply(zero, zero, pending);
        advance();
        read_b(one, stage);
        load_w(zero, stage);
        multiply(zero, one, pending);
        read_a(one, stage);
        load_x(zero, stage);
        multiply(one, zero, pending);
        read_b(zero, ahead);
        load_w(one, stage);
        multiply(one, one, pending);
      } else {
        const unsigned int before = next(ahead);
        read_a(zero, stage);
        load_x(zero, before);
        multiply(zero, zero, std::integral_constant<int, 8>{});
        read_b(one, stage);
        read_b(zero, ahead);
        load_w(one, before);
        advance();
        load_w(zero, stage);
        multiply(zero, one, std::integral_constant<int, 10>{});
      }
      stage = ahead;
    }
    // the tile's sums leave
#pragma unroll
    for (int h = 0; h < HEIGHT; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = tile.m0 + h * HALF + group * 64 + i * 16 + r;
        if (m >= p.M) continue;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int g = 0; g < (END == END_GATED ? 1 : 2); ++g) {
            const int n = tile.n0 + g * HALF + wc * 32 + j * 16 + 4 * q;
            if (n >= p.N) continue;
            if constexpr (END == END_PARTS) {
              *(floatx4*)((float*)p.out + (size_t)tile.part * p.part_stride + (size_t)m * p.ldo + n) = acc[h][g][i][j];
            } else {
              bf16_t y[4];
#pragma unroll
              for (int e = 0; e < 4; ++e) y[e] = float_to_bf16(gate_times(acc[h][0][i][j][e], acc[h][1][i][j][e], p.act));
              *(uint2*)((bf16_t*)p.out + (size_t)m * p.ldo + n) =
                  make_uint2((unsigned)y[0] | ((unsigned)y[1] << 16), (unsigned)y[2] | ((unsigned)y[3] << 16));
            }
          }
      }
    if (++round >= rounds) break;
    tile = tile_of(round);
    if (tile.count == 0) break;
    clear();
  }
  // the groups meet again, with no load under way
  wait_loads<0>();
  if (!group) barrier();
  barrier();
}

template <int END>
__global__ __launch_bounds__(THREADS) void gemm_big_kernel(Product p, Region whole, Region half) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  if (whole.tiles_n > 0) walk<END, 2>(p, whole, lds);
  if constexpr (END == END_GATED)
    if (half.tiles_n > 0) walk<END, 1>(p, half, lds);
}

constexpr int BAND_ROWS = 2048;      // eight tiles of 256: 32 neighbouring tiles of an XCD share 8 tiles of rows and 4 of weight rows
constexpr double HALF_TILE = 0.62;   // of a whole tile's time

template <int END>
int launch(const Product& p, int parts, hipStream_t stream) {
  constexpr int COLUMNS = END == END_GATED ? HALF : 2 * HALF;
  constexpr size_t LDS_BYTES = END == END_GATED ? 9 * PART_BYTES : 8 * PART_BYTES;
  static std::atomic<bool> raised{false};
  const int limit_raised = lds_tile::raise_lds_limit((const void*)gemm_big_kernel<END>, LDS_BYTES, &raised);
  if (limit_raised != FE_OK) return limit_raised;
  const long long tiles_m = (p.M + 2 * HALF - 1) / (2 * HALF), halves_m = (p.M + HALF - 1) / HALF, tiles_n = (p.N + COLUMNS - 1) / COLUMNS;
  if (halves_m * tiles_n * parts > 0x3fffffffLL) return FE_BAD_ARGUMENT;
  // columns of whole tiles: all of them, or what fills whole rounds, the rest in tiles of half the rows
  long long whole_n = tiles_n;
  if (END == END_GATED) {
    auto rounds = [](long long tiles) { return (double)((tiles + CUS - 1) / CUS); };
    const long long fill = tiles_m * tiles_n / CUS * CUS / tiles_m;
    if (rounds(tiles_m * fill) + HALF_TILE * rounds(halves_m * (tiles_n - fill)) < rounds(tiles_m * tiles_n)) whole_n = fill;
  }
  const Region whole{(int)tiles_m, (int)whole_n, parts, BAND_ROWS / (2 * HALF), 0};
  const Region half{(int)halves_m, (int)(tiles_n - whole_n), parts, BAND_ROWS / HALF, (int)whole_n * COLUMNS};
  const long long most = std::max(tiles_m * whole_n, halves_m * (tiles_n - whole_n)) * parts;
  gemm_big_kernel<END><<<(unsigned)std::min<long long>(CUS, most), THREADS, LDS_BYTES, stream>>>(p, whole, half);
  return fe_check_launch();
}

}  // namespace

// x [M, K] bf16 contiguous, K a multiple of 64; w [N, K] (gated: [2 N, K], gate rows first) bf16 with row stride ldw (a multiple of 8,
// less than 2^22); rows of out `ldo` elements apart.  ending 0: float32 sums of `parts` parts of K, part_stride elements apart; 1: gated,
// bfloat16, by `activation` (gate_act.h).  N, ldo and part_stride are multiples of four and all three pointers 16-byte aligned.
extern "C" int fe_gemm_big(const void* x, const void* w, void* out, int M, int N, int K, long long ldw, long long ldo, int ending, int parts,
                           long long part_stride, int activation, hipStream_t stream) {
  if (M < 1) return FE_OK;
  GateAct act;
  if (!gate_act(activation, &act)) return FE_BAD_ARGUMENT;
  if (N < 4 || N % 4 || K < KSTEP || K % KSTEP || ldw < K || ldw % 8 || ldo < N || ldo % 4 || part_stride % 4) return FE_BAD_ARGUMENT;
  if (parts < 1 || parts > K / KSTEP || (parts > 1 && ending != END_PARTS) || ldw >= (1 << 22)) return FE_BAD_ARGUMENT;
  if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15) return FE_BAD_ARGUMENT;
  const Product p{(const bf16_t*)x, (const bf16_t*)w, out, M, N, K / KSTEP, (unsigned int)K * 2, (unsigned int)ldw * 2, ldo, part_stride,
                  (long long)N * ldw * 2, act};
  switch (ending) {
    case END_PARTS: return launch<END_PARTS>(p, parts, stream);
    case END_GATED: return launch<END_GATED>(p, 1, stream);
  }
  return FE_BAD_ARGUMENT;
}

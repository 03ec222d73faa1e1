// Products of up to 16 rows of x (a decode step) in which a block holds finished sums:
//   s[M, N] = x[M, K] * W[N, K]^T
// with one of five endings:
//   update: h += s (float32 stream), y = bfloat16(h * weight), squares[M, b] = sum over block b's columns of h^2: the product back to
//           the residual stream with the next norm behind it.  The norm's own factor rsqrt(mean(h^2) + eps) is one number a row,
//           which the product that reads y multiplies its sums by, so the norm needs no launch of its own and y is rounded once
//           as before;
//   float32, bfloat16: stored; gated: act(gate) * up as bfloat16 for a fused gate/up weight;
//   several: stored bfloat16, up to four weights of one size with rows of x of their own each, side by side in one launch;
// float32, bfloat16 and gated with the rows' factors of such a y (SCALED) or without.
//
// Block = N / 256 weight rows (gated: pairs; one block a CU, all with the same bytes to read: 2,560 rows are 256 blocks of ten) and the
// whole of K, so no partial sums go through memory; eight waves take chunks of 64 of K in turn, each with a ring of its own in LDS
// that it fills straight from memory (`global_load_lds_dwordx4`) and empties into MFMA operands, so that no wave waits for another
// before the sums meet at the end, in the waves' order.
//
// What bounds it: the weight's bytes, and latency at the small sizes.  No block reads another's weight rows, so they pass the caches
// (lds_tile::load_to_lds_once; us: 4 rows x 12,288 x 2,048 gated 11.4 -> 10.6, 8 x 6,144 x 2,560 7.4 -> 7.1, 1 x 4,096 x 1,024 3.7 either way).  What the update ending saves is the norm's launch (4.0 to 4.7
// us in a captured step) and the parts that went through memory: 2,560 x 9,728 with its norm 13.7 -> 11.2 us at 8 rows (4.5 TB/s),
// 2,560 x 4,096 9.2 -> 6.5, 1,024 x 2,048 at 1 row 5.4 -> 3.2; a decode step of 0.6B at 1 request 909 -> 799 us, of 4B at 8 requests
// 2,464 -> 2,300.  The stored endings beside what took such sizes before (420 random products): bfloat16 1.36 times as fast, gated 1.41;
// 2,048 x 2,048 stored at 8 rows 4.6 -> 3.9 us, 6,144 x 2,048 gated 12.4 -> 11.8, of K = 4,096 25.1 -> 20.1; the same steps 793 -> 768 us
// and 2,297 -> 2,262.
//
// float32 operands go through the same rings, 32 of K a chunk, and through the bfloat16 instruction in three parts each (split_f32.h).
// At 4 rows, product, norm or gate in launches of their own before: 2,048 x 2,048 with its norm 11 -> 7.5 us, 2,048 x 6,144 17 -> 16 (the
// splitting of 16 rows where 8 are a block's), 3,072 gated columns of K = 1,024 12.3 -> 7.9, 6,144 of 2,048 24 -> 20.7; 16 rows, which
// took the weight twice, 42 -> 20.7.
//
// MFMA 16x16x32 bf16 with A = W, B = x^T: lane l (r = l % 16, q = l / 16) supplies row r, k = 8 q .. + 8 of either and receives
// D[weight row 4 q + i][row of x r].  Rows of either tile that the block has not (weight rows of its neighbour, rows of x beyond
// M) are not fetched: what lies in LDS there only reaches sums that are not stored.
#include "gate_act.h"
#include "lds_tile.h"
#include "split_f32.h"

namespace {

using lds_tile::bf16x8;
using lds_tile::floatx4;
using lds_tile::uintx4;
using lds_tile::load_to_lds;
using lds_tile::load_to_lds_once;
using lds_tile::wait_loads;

constexpr int WAVES = 8, SQUARES = 256;
constexpr int UPDATE = 0, FLOAT = 1, BFLOAT = 2, GATED = 3, SEVERAL = 4, TANH = 5;      // TANH: BFLOAT and `Ending::tanh`

// XI, WI: requests of eight rows a chunk for x and for the weight; PAIRED: a buffer holds two chunks
template <int XI, int WI, bool SCALED, bool PAIRED>
struct Ring {
  static constexpr int LOADS = (PAIRED ? 2 : 1) * (XI + WI), STAGES = (SCALED ? 17 : 19) / LOADS, TILES = (WI + 1) / 2;
  static constexpr int WAVE_BYTES = STAGES * LOADS * 1024;
  static constexpr int BYTES = WAVES * (WAVE_BYTES + (SCALED ? XI * 1024 : 0));      // behind the rings, the rows' squares
  static_assert((PAIRED ? 2 : 1) * TILES * 1024 <= WAVE_BYTES && STAGES >= 2 && BYTES <= 152 * 1024, "LDS of a CU");
};

struct Ending {
  float* h;                 // UPDATE: the stream, the norm's weight, what is left of the norm (of the operands' type)
  const float* weight;
  void* y;
  float* squares;
  void* out;                // the others: [M, N], row stride N
  const float* row_squares; // SCALED: [M][256], the factors' row length and eps
  float width, eps;
  GateAct act;
  const void* more[3];      // SEVERAL: the weights behind the first, and each one's blocks; x and out [weights][M][.]
  int each;
  bool tanh;                // BFLOAT: tanh of what is stored otherwise, rounded again
};

// float32, up to eight weight rows a block: they and up to eight rows of x fill a quarter of the instruction's tile, whose operands are split
// whatever they hold.  So it takes two chunks at a time, the second one's rows in its rows 8 to 15: sums [n][m] and [8 + n][8 + m]
// are the result's halves, the others are nobody's.  4 rows: 2,048 x 6,144 with its norm 17.0 -> 12.6 us, 2,048 x 2,048 8.4 -> 6.9, 1 row: 1,024 x
// 3,072 9.6 -> 7.3.  With 9 to 16 rows of x two sets of sums take the chunks in turn, so that a row's sums stay the same.
template <typename T, int WI>
constexpr bool pairs() {
  return sizeof(T) == 4 && WI == 1;
}

template <typename T, int XI, int WI, int END, bool SCALED>
__global__ __launch_bounds__(64 * WAVES) void gemm_ring_kernel(
    const T* __restrict__ x, const T* __restrict__ w, Ending ending, int M, int N, int K, long long ldw, int block_rows) {
  constexpr bool WIDE = sizeof(T) == 4, PAIRED = pairs<T, WI>(), FOLD = PAIRED && XI == 1;
  constexpr int CHUNKS = PAIRED ? 2 : 1, SETS = PAIRED && !FOLD ? 2 : 1;      // chunks of a buffer, sets of sums
  using R = Ring<XI, WI, SCALED, PAIRED>;
  constexpr int CHUNK = 128 / sizeof(T), PIECE = 16 / sizeof(T);      // elements of a row's 128 bytes, and of 16
  constexpr int TILES = R::TILES, PAIR = END == GATED ? 2 : 1;
  constexpr int VALUES = TILES * 256 / PAIR;          // results of a block, one a thread
  static_assert(VALUES <= 64 * WAVES && (END != GATED || WI % 2 == 0), "a thread a result");
  extern __shared__ __attribute__((aligned(16))) uintx4 lds[];
  __shared__ float per_row[END == UPDATE ? TILES * 4 : 1][16];        // UPDATE: sums of squares; SCALED: the factors
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  int block = blockIdx.x;
  if constexpr (END == SEVERAL) {
    const int which = block / ending.each;
    block -= which * ending.each;
    x += (size_t)which * M * K;
    if (which > 0) w = (const T*)ending.more[which - 1];
    ending.out = (T*)ending.out + (size_t)which * M * N;
  }
  const int n0 = block * block_rows, rows = min(block_rows, N - n0);       // columns of the result

  // thread v ends sum v: of tile v / 256 (gated: v / 128, gate columns 0 .. 7 of a tile of eight), element v % 4 of lane group v / 64 % 4
  // (gated: % 2), row v / 4 % 16
  const int tile = tid / (256 / PAIR), group = (tid >> 6) & (4 / PAIR - 1);
  const int column = tile * (16 / PAIR) + group * 4 + (tid & 3), row = (tid >> 2) & 15;
  const bool mine = tid < VALUES && row < M && column < rows;
  const size_t place = (size_t)row * N + n0 + column;
  float before = 0.f, gain = 0.f;
  if constexpr (END == UPDATE) {
    if (mine) {
      before = ending.h[place];
      gain = ending.weight[n0 + column];
    }
  }

  const unsigned int lds_at = __builtin_amdgcn_readfirstlane((unsigned int)(size_t)(const __attribute__((address_space(3))) char*)&lds[0]);
  const unsigned int squares_at = WAVES * R::WAVE_BYTES + wave * XI * 1024;
  if constexpr (SCALED) {
#pragma unroll
    for (int i = 0; i < XI; ++i)       // a row beyond M: the last one again
      load_to_lds(ending.row_squares + min(wave + WAVES * i, M - 1) * SQUARES + lane * 4, lds_at + squares_at + i * 1024);
  }

  const int chunks = K / CHUNK, own = (chunks - wave + WAVES - 1) / WAVES;       // this wave's chunks: wave, wave + 8, ..
  const int count = (own + CHUNKS - 1) / CHUNKS;      // buffers full of them
  const unsigned int base = lds_at + wave * R::WAVE_BYTES;
  // a request: eight rows of 128 bytes, 16-byte piece c of a row at c ^ (row % 8)
  const int of_group = lane >> 3, at = wave * CHUNK + ((lane & 7) ^ of_group) * PIECE;
  const T *x_from[XI], *w_from[WI];
  bool x_has[XI], w_has[WI];
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    x_has[i] = i * 8 + of_group < M;
    x_from[i] = x + (size_t)min(i * 8 + of_group, M - 1) * K + at;
  }
#pragma unroll
  for (int i = 0; i < WI; ++i) {       // gated: eight gate rows, then the eight up rows of the same columns
    const int j = (END == GATED ? i / 2 : i) * 8 + of_group;
    w_has[i] = j < rows;
    w_from[i] = w + (size_t)(n0 + min(j, rows - 1) + (END == GATED && i % 2 ? N : 0)) * ldw + at;
  }
  // every request is issued whatever the rows, so that the waits can count: where all eight rows lie beyond the block's last one (the
  // last block's), that one is fetched again
  auto load = [&](int index, int stage) {
#pragma unroll
    for (int part = 0; part < CHUNKS; ++part) {
      const int k = (PAIRED ? min(2 * index + part, own - 1) : index) * WAVES * CHUNK;      // a chunk too few: the last one again
      const unsigned int to = base + (stage * R::LOADS + part * (XI + WI)) * 1024;
#pragma unroll
      for (int i = 0; i < XI; ++i)
        if (x_has[i] || of_group == 0) load_to_lds(x_from[i] + k, to + i * 1024);
#pragma unroll
      for (int i = 0; i < WI; ++i)
        if (w_has[i] || of_group == 0) load_to_lds_once(w_from[i] + k, to + (XI + i) * 1024);
    }
  };
  floatx4 acc[SETS * TILES];
#pragma unroll
  for (int t = 0; t < SETS * TILES; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  // float32 operands: the products of the first parts, added to the whole every four chunks, and all others, a 2^8th of their size: so
  // the long sum is rounded a quarter as often and a long K costs no accuracy
  floatx4 large[SETS * TILES], small[SETS * TILES];
  int turn = 0;
#pragma unroll
  for (int t = 0; t < SETS * TILES; ++t) large[t] = small[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  const uintx4* ring = lds + wave * (R::WAVE_BYTES / 16);
  const split_f32::Minus minus = split_f32::minus();
  uintx4 a[2], b[TILES][2];
  auto fragments = [&](int stage, int part) {
    const uintx4* from = ring + (stage * R::LOADS + (FOLD ? r >> 3 : part) * (XI + WI)) * 64;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int piece = (4 * half + q) ^ (r & 7);
      a[half] = from[(XI == 1 ? r & 7 : r) * 8 + piece];
#pragma unroll
      for (int t = 0; t < TILES; ++t) b[t][half] = from[XI * 64 + (FOLD ? r & 7 : min(t * 16 + r, WI * 8 - 8 + (r & 7))) * 8 + piece];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // read before the buffer is filled again
  };
  auto multiply = [&](int set) {
    if constexpr (WIDE) {       // the two pieces are a lane's eight elements of 32
      bf16x8 x_parts[1][3], w_parts[3];
      split_f32::split8(__builtin_bit_cast(floatx4, a[0]), __builtin_bit_cast(floatx4, a[1]), minus, x_parts[0]);
#pragma unroll
      for (int t = 0; t < TILES; ++t) {
        split_f32::split8(__builtin_bit_cast(floatx4, b[t][0]), __builtin_bit_cast(floatx4, b[t][1]), minus, w_parts);
        split_f32::add_products_apart(x_parts[0], w_parts, large[set * TILES + t], small[set * TILES + t]);
        if (turn == 3) {
          acc[set * TILES + t] += large[set * TILES + t];
          large[set * TILES + t] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
      }
      if (set == SETS - 1) turn = (turn + 1) & 3;
      return;
    }
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int t = 0; t < TILES; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b[t][half]), __builtin_bit_cast(bf16x8, a[half]), acc[t], 0, 0, 0);
  };
#pragma unroll
  for (int s = 0; s < R::STAGES; ++s)
    if (s < count) load(s, s);
  if constexpr (SCALED) {       // the factors, while the first chunks are on their way
    lds_tile::wait_steps<R::LOADS, R::STAGES>(count);
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const floatx4 v = *(const floatx4*)((const char*)lds + squares_at + i * 1024 + lane * 16);
      const float sum = wave_sum_dpp((v[0] + v[1]) + (v[2] + v[3]));
      if (lane == 0) per_row[0][wave + WAVES * i] = rsqrtf(sum / ending.width + ending.eps);
    }
  }
  int stage = 0, i = 0;
  for (; count - i > R::STAGES; ++i) {
    wait_loads<R::LOADS*(R::STAGES - 1)>();
    if constexpr (SETS == 2) {
      fragments(stage, 0);
      multiply(0);
    }
    fragments(stage, SETS - 1);
    load(i + R::STAGES, stage);
    multiply(SETS - 1);
    stage = stage + 1 == R::STAGES ? 0 : stage + 1;
  }
  // the last chunks, with fewer and fewer requests under way: each with its own wait
  const int rest = count - i;
  auto end = [&](auto self, auto left) {
    constexpr int L = decltype(left)::value;
    if constexpr (L > 0) {
      if (rest >= L) {
        wait_loads<R::LOADS*(L - 1)>();
        if constexpr (SETS == 2) {
          fragments(stage, 0);
          multiply(0);
        }
        fragments(stage, SETS - 1);
        if (PAIRED && L == 1 && own % 2 && (!FOLD || r >= 8)) a[0] = a[1] = uintx4{0, 0, 0, 0};      // an odd chunk, here twice
        multiply(SETS - 1);
        stage = stage + 1 == R::STAGES ? 0 : stage + 1;
      }
      self(self, std::integral_constant<int, L - 1>{});
    }
  };
  end(end, std::integral_constant<int, R::STAGES>{});

  // the waves' sums meet, each in its wave's own ring, which nobody else reads and which it has emptied
  floatx4* meet = (floatx4*)(lds + wave * (R::WAVE_BYTES / 16));
#pragma unroll
  for (int t = 0; t < SETS * TILES; ++t) meet[t * 64 + lane] = WIDE ? acc[t] + (large[t] + small[t]) : acc[t];
  __syncthreads();
  auto total = [&](int lane_group) {       // of the eight columns' gate or up rows, or of all sixteen: lane group of the tile
    const float* from = (const float*)lds + tile * 256 + (lane_group * 16 + row) * 4 + (tid & 3);
    float sum = 0.f;
    if constexpr (FOLD) from = (const float*)lds + ((lane_group & 1) * 16 + (row & 7)) * 4 + (tid & 3);
    constexpr int OTHER = FOLD ? (2 * 16 + 8) * 4 : 256;      // from the first chunks' sum to the second ones'
#pragma unroll
    for (int v = 0; v < WAVES; ++v) {
      if constexpr (PAIRED) sum += from[v * (R::WAVE_BYTES / 4)] + from[v * (R::WAVE_BYTES / 4) + OTHER];
      else sum += from[v * (R::WAVE_BYTES / 4)];
    }
    if constexpr (WIDE) {
      if (!split_f32::finite(sum) && mine)
        sum = split_f32::dot(x + (size_t)row * K, w + (size_t)(n0 + column + (lane_group != group ? N : 0)) * ldw, K);
    }
    return sum;
  };
  if constexpr (END == UPDATE) {
    if (tid < VALUES) {
      const float sum = total(group) + before;
      float square = mine ? sum * sum : 0.f;
      square += __shfl_xor(square, 1, 64);
      square += __shfl_xor(square, 2, 64);
      if ((tid & 3) == 0) per_row[tid >> 6][row] = square;
      if (mine) {
        ending.h[place] = sum;
        store_from_float((T*)ending.y + place, sum * gain);
      }
    }
    __syncthreads();
    if (tid < M) {
      float square = 0.f;
#pragma unroll
      for (int j = 0; j < TILES * 4; ++j) square += per_row[j][tid];
      ending.squares[tid * SQUARES + blockIdx.x] = square;
      if (blockIdx.x == gridDim.x - 1)
        for (int j = gridDim.x; j < SQUARES; ++j) ending.squares[tid * SQUARES + j] = 0.f;
    }
  } else if (mine) {
    const float factor = SCALED ? per_row[0][row] : 1.f;
    float sum = total(group);
    if (SCALED) sum *= factor;
    if constexpr (END == GATED) {
      float up = total(group + 2);
      if (SCALED) up *= factor;
      if constexpr (WIDE) ((float*)ending.out)[place] = gate_times_exact(sum, up, ending.act);
      else ((bf16_t*)ending.out)[place] = float_to_bf16(gate_times(sum, up, ending.act));
    } else if constexpr (END == FLOAT) {
      ((float*)ending.out)[place] = sum;
    } else {
      bf16_t y = float_to_bf16(sum);
      if (END == BFLOAT && ending.tanh) y = float_to_bf16(tanhf(bf16_to_float(y)));      // the bits of a launch of its own behind this one
      ((bf16_t*)ending.out)[place] = y;
    }
  }
}

template <typename T, int XI, int WI, int END, bool SCALED>
int launch(const void* x, const void* w, const Ending& ending, int M, int N, int K, long long ldw, int block_rows, int weights, hipStream_t stream) {
  static std::atomic<bool> raised{false};
  using R = Ring<XI, WI, SCALED, pairs<T, WI>()>;
  auto kernel = gemm_ring_kernel<T, XI, WI, END, SCALED>;
  const int limit_raised = lds_tile::raise_lds_limit((const void*)kernel, R::BYTES, &raised);
  if (limit_raised != FE_OK) return limit_raised;
  kernel<<<ending.each * weights, 64 * WAVES, R::BYTES, stream>>>(
      (const T*)x, (const T*)w, ending, M, N, K, ldw, block_rows);
  return fe_check_launch();
}

template <typename T, int END, bool SCALED>
int pick(const void* x, const void* w, Ending ending, int M, int N, int K, long long ldw, hipStream_t stream, int weights = 1) {
  const int block_rows = (N * weights + SQUARES - 1) / SQUARES;
  ending.each = (N + block_rows - 1) / block_rows;
#define FE_PICK(XI, WI) return launch<T, XI, WI, END, SCALED>(x, w, ending, M, N, K, ldw, block_rows, weights, stream)
  const int groups = (block_rows + 7) / 8;
  if constexpr (END == GATED) {
    switch (groups) {
      case 1: if (M <= 8) FE_PICK(1, 2); FE_PICK(2, 2);
      case 2: if (M <= 8) FE_PICK(1, 4); FE_PICK(2, 4);
      case 3: if (M <= 8) FE_PICK(1, 6); FE_PICK(2, 6);
    }
  } else {
    switch (groups) {
      case 1: if (M <= 8) FE_PICK(1, 1); FE_PICK(2, 1);
      case 2: if (M <= 8) FE_PICK(1, 2); FE_PICK(2, 2);
      case 3: if (M <= 8) FE_PICK(1, 3); FE_PICK(2, 3);
      case 4: if (M <= 8) FE_PICK(1, 4); FE_PICK(2, 4);
    }
  }
#undef FE_PICK
  return FE_BAD_ARGUMENT;
}

bool operands_fit(const void* x, const void* w, int dtype, int M, int N, int K, long long ldw) {
  if (dtype != FE_F32 && dtype != FE_BF16) return false;
  const int chunk = dtype == FE_F32 ? 32 : 64, piece = dtype == FE_F32 ? 4 : 8;
  return M <= 16 && N >= 1 && K >= chunk && K % chunk == 0 && ldw >= K && ldw % piece == 0 && x && w && ((((uintptr_t)x) | ((uintptr_t)w)) & 15) == 0;
}

}  // namespace

// x [M, K], contiguous, 1 <= M <= 16, and w [N, K] with row stride ldw, rows 16-byte aligned, N up to 8,192: bfloat16, K a multiple of
// 64, or float32, K a multiple of 32; h [M, N] float32, contiguous, is replaced by h + x w^T; weight [N] float32; y [M, N] of x's type;
// squares [M][256] float32, whose sum over a row is that row's sum of squares of the new h (entries beyond the blocks are zero).
extern "C" int fe_gemm_update_norm(const void* x, const void* w, int dtype, float* h, const float* weight, void* y, float* squares,
                                   int M, int N, int K, long long ldw, hipStream_t stream) {
  if (M < 1) return FE_OK;
  if (!operands_fit(x, w, dtype, M, N, K, ldw) || N > 32 * SQUARES || !h || !weight || !y || !squares) return FE_BAD_ARGUMENT;
  const Ending how = {h, weight, y, squares, nullptr, nullptr, 0.f, 0.f, {}, {}, 0, false};
  if (dtype == FE_F32) return pick<float, UPDATE, false>(x, w, how, M, N, K, ldw, stream);
  return pick<bf16_t, UPDATE, false>(x, w, how, M, N, K, ldw, stream);
}

// The same operands; ending 1: out [M, N] float32, 2: bfloat16, of bfloat16 operands (N up to 8,192), 3: out [M, N] of x's type =
// act(x gate^T) * (x up^T) for a fused weight [2 N, K], gate rows first (N up to 6,144; act by `activation`, gate_act.h), 5: tanh of ending 2.  squares
// (null: none) [M][256] float32: the sums of row m are multiplied by rsqrt(sum of squares[m] / K + eps) before anything else is done
// with them.
extern "C" int fe_gemm_ring(const void* x, const void* w, int dtype, void* out, int M, int N, int K, long long ldw, int ending,
                            int activation, const float* squares, float eps, hipStream_t stream) {
  if (M < 1) return FE_OK;
  GateAct act;
  if (!gate_act(activation, &act)) return FE_BAD_ARGUMENT;
  if (!operands_fit(x, w, dtype, M, N, K, ldw) || !out || N > (ending == GATED ? 24 : 32) * SQUARES) return FE_BAD_ARGUMENT;
  if (squares && (!(eps > 0.f) || (((uintptr_t)squares) & 15))) return FE_BAD_ARGUMENT;
  const bool tanh = ending == TANH;
  if (tanh) ending = BFLOAT;
  const Ending how = {nullptr, nullptr, nullptr, nullptr, out, squares, (float)K, eps, act, {}, 0, tanh};
#define FE_PICK(TYPE, T, END)                                                       \
  if (dtype == TYPE && ending == END) {                                             \
    if (squares) return pick<T, END, true>(x, w, how, M, N, K, ldw, stream);        \
    return pick<T, END, false>(x, w, how, M, N, K, ldw, stream);                    \
  }
  FE_PICK(FE_BF16, bf16_t, FLOAT)
  FE_PICK(FE_BF16, bf16_t, BFLOAT)
  FE_PICK(FE_BF16, bf16_t, GATED)
  FE_PICK(FE_F32, float, FLOAT)
  FE_PICK(FE_F32, float, GATED)
#undef FE_PICK
  return FE_BAD_ARGUMENT;
}

// out [weights][M][N] bfloat16: rows x [weights][M][K], contiguous, each against its own weight of w[0 .. weights) (host array of device
// addresses; [N, K], contiguous, 16-byte aligned), 2 to 4 of them of N up to 8,192 together, K a multiple of 64.
// What it saves is the starts: four weights of 2,048 x 2,048 at 6 rows 15.33 -> 12.35 us, of 1,024 x 1,024 10.30 -> 6.06.
extern "C" int fe_gemm_ring_several(const void* x, const void* const* w, void* out, int weights, int M, int N, int K, hipStream_t stream) {
  if (M < 1) return FE_OK;
  if (weights < 2 || weights > 4 || !w || !out || N < 1 || (long long)N * weights > 32 * SQUARES) return FE_BAD_ARGUMENT;
  Ending how = {nullptr, nullptr, nullptr, nullptr, out, nullptr, 0.f, 0.f, {}, {}, 0, false};
  for (int i = 0; i < weights; ++i) {
    if (!operands_fit(x, w[i], FE_BF16, M, N, K, K)) return FE_BAD_ARGUMENT;
    if (i > 0) how.more[i - 1] = w[i];
  }
  return pick<bf16_t, SEVERAL, false>(x, w[0], how, M, N, K, K, stream, weights);
}

// A decode step's product back to the residual stream with the next norm behind it, for up to 16 rows:
//   h[M, N] += x[M, K] * W[N, K]^T                 (float32 sums and stream)
//   y[M, N] = bfloat16(h * weight),  squares[M, b] = sum over block b's columns of h^2
// The norm's own factor rsqrt(mean(h^2) + eps) is one number a row: the product that reads y multiplies its sums by it
// (gemm_lds.h), so the norm needs no launch of its own, and y is rounded once as before.
//
// Block = N / 256 weight rows (one block a CU, all with the same bytes to read: 2,560 rows are 256 blocks of ten) and the whole
// of K, so that a block holds finished sums and no partial ones go through memory; eight waves take chunks of 64 of K in turn,
// each with a ring of its own in LDS that it fills straight from memory (`global_load_lds_dwordx4`) and empties into MFMA
// operands, so that no wave waits for another before the sums meet at the end, in the waves' order.
//
// What bounds it: the weight's bytes, and latency at the small sizes.  What it saves is the norm's launch (4.0 to 4.7 us in a
// captured step) and the parts that went through memory: 2,560 x 9,728 with its norm 13.7 -> 11.2 us at 8 rows (4.5 TB/s), 2,560 x
// 4,096 9.2 -> 6.5, 1,024 x 2,048 at 1 row 5.4 -> 3.2; a decode step of 0.6B at 1 request 909 -> 799 us, of 4B at 8 requests
// 2,464 -> 2,300.
//
// MFMA 16x16x32 bf16 with A = W, B = x^T: lane l (r = l % 16, q = l / 16) supplies row r, k = 8 q .. + 8 of either and receives
// D[weight row 4 q + i][row of x r].  Rows of either tile that the block has not (weight rows of its neighbour, rows of x beyond
// M) are not fetched: what lies in LDS there only reaches sums that are not stored.
#include "lds_tile.h"

namespace {

using lds_tile::bf16x8;
using lds_tile::floatx4;
using lds_tile::uintx4;
using lds_tile::load_to_lds;
using lds_tile::wait_loads;

constexpr int WAVES = 8, CHUNK = 64, SQUARES = 256;

// XI, WI: requests of eight rows a chunk for x and for the weight
template <int XI, int WI>
struct Ring {
  static constexpr int LOADS = XI + WI, STAGES = 19 / LOADS, TILES = (WI + 1) / 2;
  static constexpr int WAVE_BYTES = STAGES * LOADS * 1024;
  static constexpr int BYTES = WAVES * WAVE_BYTES;
  static_assert(TILES * 1024 <= WAVE_BYTES && BYTES <= 160 * 1024, "LDS of a CU");
};

template <int XI, int WI>
__global__ __launch_bounds__(64 * WAVES) void gemm_update_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, float* __restrict__ h, const float* __restrict__ weight,
    bf16_t* __restrict__ y, float* __restrict__ squares, int M, int N, int K, long long ldw, int block_rows) {
  using R = Ring<XI, WI>;
  constexpr int TILES = R::TILES, VALUES = TILES * 256;
  extern __shared__ __attribute__((aligned(16))) uintx4 lds[];
  __shared__ float row_squares[TILES * 4][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int n0 = blockIdx.x * block_rows, rows = min(block_rows, N - n0);

  // what the ending adds to and multiplies by; thread v stores sum v: column 16 (v / 256) + 4 (v / 64 % 4) + v % 4, row v / 4 % 16
  const int column = (tid >> 8) * 16 + ((tid >> 6) & 3) * 4 + (tid & 3), row = (tid >> 2) & 15;
  const bool mine = tid < VALUES && row < M && column < rows;
  float before = 0.f, gain = 0.f;
  if (mine) {
    before = h[(size_t)row * N + n0 + column];
    gain = weight[n0 + column];
  }

  const int chunks = K / CHUNK, count = (chunks - wave + WAVES - 1) / WAVES;       // this wave's chunks: wave, wave + 8, ..
  const unsigned int base = __builtin_amdgcn_readfirstlane((unsigned int)(size_t)(const __attribute__((address_space(3))) char*)&lds[0]) + wave * R::WAVE_BYTES;
  // a request: eight rows of 128 bytes, 16-byte piece c of a row at c ^ (row % 8)
  const int of_group = lane >> 3, at = wave * CHUNK + ((lane & 7) ^ of_group) * 8;
  const bf16_t *x_from[XI], *w_from[WI];
  bool x_has[XI], w_has[WI];
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    x_has[i] = i * 8 + of_group < M;
    x_from[i] = x + (size_t)min(i * 8 + of_group, M - 1) * K + at;
  }
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    w_has[i] = i * 8 + of_group < rows;
    w_from[i] = w + (size_t)(n0 + min(i * 8 + of_group, rows - 1)) * ldw + at;
  }
  // every request is issued whatever the rows, so that the waits can count: a wave's first row of eight may lie beyond the block's
  // last one (the last block's), and then that one is fetched again
  auto load = [&](int index, int stage) {
    const int k = index * WAVES * CHUNK;
    const unsigned int to = base + stage * R::LOADS * 1024;
#pragma unroll
    for (int i = 0; i < XI; ++i)
      if (x_has[i] || of_group == 0) load_to_lds(x_from[i] + k, to + i * 1024);
#pragma unroll
    for (int i = 0; i < WI; ++i)
      if (w_has[i] || of_group == 0) load_to_lds(w_from[i] + k, to + (XI + i) * 1024);
  };
  floatx4 acc[TILES];
#pragma unroll
  for (int t = 0; t < TILES; ++t) acc[t] = floatx4{0.f, 0.f, 0.f, 0.f};
  const uintx4* ring = lds + wave * (R::WAVE_BYTES / 16);
  uintx4 a[2], b[TILES][2];
  auto fragments = [&](int stage) {
    const uintx4* from = ring + stage * R::LOADS * 64;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int piece = (4 * half + q) ^ (r & 7);
      a[half] = from[(XI == 1 ? r & 7 : r) * 8 + piece];
#pragma unroll
      for (int t = 0; t < TILES; ++t) b[t][half] = from[XI * 64 + min(t * 16 + r, WI * 8 - 1 - (7 - (r & 7))) * 8 + piece];
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // read before the buffer is filled again
  };
  auto multiply = [&]() {
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int t = 0; t < TILES; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b[t][half]), __builtin_bit_cast(bf16x8, a[half]), acc[t], 0, 0, 0);
  };
#pragma unroll
  for (int s = 0; s < R::STAGES; ++s)
    if (s < count) load(s, s);
  int stage = 0, i = 0;
  for (; count - i > R::STAGES; ++i) {
    wait_loads<R::LOADS*(R::STAGES - 1)>();
    fragments(stage);
    load(i + R::STAGES, stage);
    multiply();
    stage = stage + 1 == R::STAGES ? 0 : stage + 1;
  }
  // the last chunks, with fewer and fewer requests under way: each with its own wait
  const int rest = count - i;
  auto end = [&](auto self, auto left) {
    constexpr int L = decltype(left)::value;
    if constexpr (L > 0) {
      if (rest >= L) {
        wait_loads<R::LOADS*(L - 1)>();
        fragments(stage);
        multiply();
        stage = stage + 1 == R::STAGES ? 0 : stage + 1;
      }
      self(self, std::integral_constant<int, L - 1>{});
    }
  };
  end(end, std::integral_constant<int, R::STAGES>{});

  // the waves' sums meet, each in its wave's own ring, which nobody else reads and which it has emptied
  floatx4* meet = (floatx4*)(lds + wave * (R::WAVE_BYTES / 16));
#pragma unroll
  for (int t = 0; t < TILES; ++t) meet[t * 64 + lane] = acc[t];
  __syncthreads();
  float sum = 0.f;
  if (tid < VALUES) {
    // sum v of a tile lies at lane 16 (v / 64 % 4) + v / 4 % 16, element v % 4
    const float* from = (const float*)lds + (tid >> 8) * 256 + (((tid >> 6) & 3) * 16 + row) * 4 + (tid & 3);
#pragma unroll
    for (int v = 0; v < WAVES; ++v) sum += from[v * (R::WAVE_BYTES / 4)];
    sum += before;
    float square = mine ? sum * sum : 0.f;
    square += __shfl_xor(square, 1, 64);
    square += __shfl_xor(square, 2, 64);
    if ((tid & 3) == 0) row_squares[tid >> 6][row] = square;
  }
  if (mine) {
    h[(size_t)row * N + n0 + column] = sum;
    y[(size_t)row * N + n0 + column] = float_to_bf16(sum * gain);
  }
  __syncthreads();
  if (tid < M) {
    float square = 0.f;
#pragma unroll
    for (int j = 0; j < TILES * 4; ++j) square += row_squares[j][tid];
    squares[tid * SQUARES + blockIdx.x] = square;
    if (blockIdx.x == gridDim.x - 1)
      for (int j = gridDim.x; j < SQUARES; ++j) squares[tid * SQUARES + j] = 0.f;
  }
}

template <int XI, int WI>
int launch(const void* x, const void* w, float* h, const float* weight, void* y, float* squares, int M, int N, int K,
           long long ldw, int block_rows, hipStream_t stream) {
  static std::atomic<bool> raised{false};
  auto kernel = gemm_update_kernel<XI, WI>;
  const int limit_raised = lds_tile::raise_lds_limit((const void*)kernel, Ring<XI, WI>::BYTES, &raised);
  if (limit_raised != FE_OK) return limit_raised;
  kernel<<<(N + block_rows - 1) / block_rows, 64 * WAVES, Ring<XI, WI>::BYTES, stream>>>(
      (const bf16_t*)x, (const bf16_t*)w, h, weight, (bf16_t*)y, squares, M, N, K, ldw, block_rows);
  return fe_check_launch();
}

}  // namespace

// x [M, K] bfloat16, contiguous, 1 <= M <= 16, K a multiple of 64; w [N, K] bfloat16 with row stride ldw, rows 16-byte aligned, N up to
// 8,192; h [M, N] float32, contiguous, is replaced by h + x w^T; weight [N] float32; y [M, N] bfloat16; squares [M][256] float32,
// whose sum over a row is that row's sum of squares of the new h (entries beyond the blocks are zero).
extern "C" int fe_gemm_update_norm(const void* x, const void* w, float* h, const float* weight, void* y, float* squares, int M,
                                   int N, int K, long long ldw, hipStream_t stream) {
  if (M < 1) return FE_OK;
  if (M > 16 || N < 1 || N > 32 * SQUARES || K < CHUNK || K % CHUNK || ldw < K || ldw % 8) return FE_BAD_ARGUMENT;
  if (!x || !w || !h || !weight || !y || !squares || ((((uintptr_t)x) | ((uintptr_t)w)) & 15)) return FE_BAD_ARGUMENT;
  const int block_rows = (N + SQUARES - 1) / SQUARES;
#define FE_PICK(XI, WI) return launch<XI, WI>(x, w, h, weight, y, squares, M, N, K, ldw, block_rows, stream)
  switch ((block_rows + 7) / 8) {
    case 1: if (M <= 8) FE_PICK(1, 1); FE_PICK(2, 1);
    case 2: if (M <= 8) FE_PICK(1, 2); FE_PICK(2, 2);
    case 3: if (M <= 8) FE_PICK(1, 3); FE_PICK(2, 3);
    default: if (M <= 8) FE_PICK(1, 4); FE_PICK(2, 4);
  }
#undef FE_PICK
}

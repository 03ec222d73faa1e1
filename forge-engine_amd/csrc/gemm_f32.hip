// True float32 matrix product C[M,N] = A[M,K] * B[N,K]^T (+ bias[N]), both
// operands K-contiguous (activations times a weight in [out, in] layout).
// float32 products and float32 accumulation throughout, in an order that depends
// on K alone within a variant.  Up to 16 rows of A (64 where K is 1,024 or more) stream the
// weight past registers on the vector ALU; more rows are tiled on the matrix cores'
// float32 instruction, whose products and sums are not rounded to anything narrower;
// operands that are not 16-byte aligned rows take the plain 64x64 tile.
#include "common.h"
#include <algorithm>

#define TILE_M 64
#define TILE_N 64
#define TILE_K 16

__global__ __launch_bounds__(256) void gemm_nt_f32_kernel(
    const float* __restrict__ A, const float* __restrict__ B, const float* __restrict__ bias,
    float* __restrict__ C, int M, int N, int K, long long lda, long long ldb, long long ldc) {
  // [k][row], padded so that the transposing stores spread over banks
  __shared__ float As[TILE_K][TILE_M + 4];
  __shared__ float Bs[TILE_K][TILE_N + 4];
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * TILE_M;
  const int n0 = blockIdx.x * TILE_N;
  const int tx = tid % 16;  // 4 columns each
  const int ty = tid / 16;  // 4 rows each
  // loader: thread -> (row = tid / 4, k quad = tid % 4)
  const int lrow = tid / 4;
  const int lk = (tid % 4) * 4;

  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

  for (int k0 = 0; k0 < K; k0 += TILE_K) {
    float a[4] = {0.f, 0.f, 0.f, 0.f};
    float b[4] = {0.f, 0.f, 0.f, 0.f};
    const int am = m0 + lrow;
    const int bn = n0 + lrow;
    const int kk = k0 + lk;
    if (am < M) {
      const float* p = A + (size_t)am * lda + kk;
#pragma unroll
      for (int i = 0; i < 4; ++i) if (kk + i < K) a[i] = p[i];
    }
    if (bn < N) {
      const float* p = B + (size_t)bn * ldb + kk;
#pragma unroll
      for (int i = 0; i < 4; ++i) if (kk + i < K) b[i] = p[i];
    }
    __syncthreads();  // previous tile fully consumed
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      As[lk + i][lrow] = a[i];
      Bs[lk + i][lrow] = b[i];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < TILE_K; ++k) {
      const float4 av = *(const float4*)&As[k][ty * 4];
      const float4 bv = *(const float4*)&Bs[k][tx * 4];
      const float ar[4] = {av.x, av.y, av.z, av.w};
      const float br[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(ar[i], br[j], acc[i][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n < N) C[(size_t)m * ldc + n] = acc[i][j] + (bias ? bias[n] : 0.f);
    }
  }
}

// The same product for up to 16 rows of A (a decode step), where the work is reading B once:
// a block takes R rows of B and MR rows of A; its four waves split K in interleaved steps of
// 256 (a lane reads 16 contiguous bytes of every row, a wave 1 KB), each lane keeps R x MR
// sums over its own k, the sums meet by a butterfly over the lanes and then over the waves in
// LDS, in a fixed order.  The order of a row's sum depends on K alone: not on M, not on the
// rows beside it, not on R or MR.  Needs K % 4 == 0 and 16-byte aligned rows.
template <int MR, int R>
__global__ __launch_bounds__(256) void gemm_rows_f32_kernel(
    const float* __restrict__ A, const float* __restrict__ B, const float* __restrict__ bias,
    float* __restrict__ C, int M, int N, int K, long long lda, long long ldb, long long ldc) {
  __shared__ float red[4][R * MR];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n0 = blockIdx.x * R, m0 = blockIdx.y * MR;
  const float* arow[MR];
  const float* brow[R];
#pragma unroll
  for (int m = 0; m < MR; ++m) arow[m] = A + (size_t)min(m0 + m, M - 1) * lda;     // rows beyond M: the last again, never stored
#pragma unroll
  for (int r = 0; r < R; ++r) brow[r] = B + (size_t)min(n0 + r, N - 1) * ldb;
  float acc[R][MR];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int m = 0; m < MR; ++m) acc[r][m] = 0.f;

  // Loads are unconditional (a load under a per-lane condition becomes a branch, and where
  // branches meet every load in flight is waited for): a step beyond K reads the row's last
  // four elements again and is never used, because the loop ends first.
  int k = (wave * 64 + lane) * 4;
  float4 bnext[R];
#pragma unroll
  for (int r = 0; r < R; ++r) bnext[r] = *(const float4*)(brow[r] + min(k, K - 4));
  for (; k < K; k += 1024) {
    float4 bv[R], av[MR];
#pragma unroll
    for (int r = 0; r < R; ++r) bv[r] = bnext[r];
#pragma unroll
    for (int m = 0; m < MR; ++m) av[m] = *(const float4*)(arow[m] + k);
    const int kn = min(k + 1024, K - 4);           // the next step's rows of B fly during this step's sums
#pragma unroll
    for (int r = 0; r < R; ++r) bnext[r] = *(const float4*)(brow[r] + kn);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int m = 0; m < MR; ++m) {
        float s = acc[r][m];
        s = fmaf(av[m].x, bv[r].x, s);
        s = fmaf(av[m].y, bv[r].y, s);
        s = fmaf(av[m].z, bv[r].z, s);
        s = fmaf(av[m].w, bv[r].w, s);
        acc[r][m] = s;
      }
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const float total = wave_sum(acc[r][m]);
      if (lane == 0) red[wave][r * MR + m] = total;
    }
  __syncthreads();
  if (tid < R * MR) {
    const int r = tid / MR, m = tid - r * MR;
    const int n = n0 + r, row = m0 + m;
    if (n < N && row < M) {
      const float total = ((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid];
      C[(size_t)row * ldc + n] = total + (bias ? bias[n] : 0.f);
    }
  }
}

// The same product for up to 8 rows of A with the rows of A held in registers: a lane's places in K
// are its own for the whole launch (k = 4 (64 wave + lane) + 256 WAVES step), so a block fetches its
// slices of A once and then walks tiles of two rows of B (blocks are persistent: tile b, b + blocks,
// ...), reading nothing but B: the streaming kernel above pulls every row of A through L1 again for
// every four rows of B, twice the bytes of B itself.  The next tile's rows of B fly while this tile
// is multiplied.  The 16 sums of a tile (2 rows of B x 8 of A) meet across the 64 lanes by a
// butterfly that halves the values a lane holds at every exchange (one exchange a value instead of
// six), then across the waves in LDS, in wave order.  K beyond 768 WAVES elements takes further
// passes over the tiles, each adding to what the pass before stored (the same thread wrote it).
// The order of a row's sum depends on K alone.
template <int XS, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void gemm_rows_resident_f32_kernel(
    const float* __restrict__ A, const float* __restrict__ B, const float* __restrict__ bias,
    float* __restrict__ C, int M, int N, int K, long long lda, long long ldb, long long ldc) {
  constexpr int MR = 8, R = 2, SPAN = 256 * WAVES * XS;     // SPAN: elements of K a pass covers
  __shared__ float red[2][WAVES][R * MR];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int k_lane = (wave * 64 + lane) * 4;
  const int tiles = (N + R - 1) / R;
  for (int k0 = 0; k0 < K; k0 += SPAN) {
    // this pass's slices of A: zero beyond K, rows beyond M the last row again (never stored)
    float4 xr[XS][MR];
    int kk[XS];
#pragma unroll
    for (int s = 0; s < XS; ++s) {
      const int k = k0 + k_lane + 256 * WAVES * s;
      kk[s] = min(k, K - 4);
#pragma unroll
      for (int m = 0; m < MR; ++m) {
        const float4 v = *(const float4*)(A + (size_t)min(m, M - 1) * lda + kk[s]);
        xr[s][m] = k < K ? v : make_float4(0.f, 0.f, 0.f, 0.f);
      }
    }
    const bool last_pass = k0 + SPAN >= K;
    float4 bnext[R][XS];
    auto fetch = [&](int tile) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float* brow = B + (size_t)min(tile * R + r, N - 1) * ldb;
#pragma unroll
        for (int s = 0; s < XS; ++s) bnext[r][s] = *(const float4*)(brow + kk[s]);
      }
    };
    fetch(min((int)blockIdx.x, tiles - 1));
    int round = 0;
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x, round ^= 1) {
      float4 bv[R][XS];
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int s = 0; s < XS; ++s) bv[r][s] = bnext[r][s];
      fetch(min(tile + (int)gridDim.x, tiles - 1));       // unconditional: past the end the last tile again, never used
      float acc[R * MR];
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < MR; ++m) {
          float sum = 0.f;
#pragma unroll
          for (int s = 0; s < XS; ++s) {
            sum = fmaf(xr[s][m].x, bv[r][s].x, sum);
            sum = fmaf(xr[s][m].y, bv[r][s].y, sum);
            sum = fmaf(xr[s][m].z, bv[r][s].z, sum);
            sum = fmaf(xr[s][m].w, bv[r][s].w, sum);
          }
          acc[r * MR + m] = sum;
        }
      // 16 values over 64 lanes: lanes 32 apart exchange halves (each keeps eight sums of two lanes), lanes
      // 16 apart quarters, then 8 and 4 apart, and the last two exchanges add what the four lanes of a
      // quad hold: lane l ends with value 8 b5 + 4 b4 + 2 b3 + b2 of its bits, summed over all lanes.
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[i]), __float_as_uint(acc[i + 8]), false, false);
        acc[i] = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[i]), __float_as_uint(acc[i + 4]), false, false);
        acc[i] = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
      }
      const bool up8 = lane & 8, up4 = lane & 4;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float keep = up8 ? acc[i + 2] : acc[i], send = up8 ? acc[i] : acc[i + 2];
        acc[i] = keep + __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(send), 0x128, 0xF, 0xF, true));   // lane ^ 8: a row rotated by 8
      }
      {
        const float keep = up4 ? acc[1] : acc[0], send = up4 ? acc[0] : acc[1];
        acc[0] = keep + __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(send), 0x141, 0xF, 0xF, true));   // 7 - lane within 8
      }
      acc[0] += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(acc[0]), 0x4E, 0xF, 0xF, true));   // lane ^ 2
      acc[0] += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(acc[0]), 0xB1, 0xF, 0xF, true));   // lane ^ 1
      if ((lane & 3) == 0) red[round][wave][((lane >> 5) & 1) * 8 + ((lane >> 4) & 1) * 4 + ((lane >> 3) & 1) * 2 + ((lane >> 2) & 1)] = acc[0];
      __syncthreads();
      if (tid < R * MR) {
        const int r = tid / MR, m = tid - r * MR;
        const int n = tile * R + r;
        if (n < N && m < M) {
          float total = red[round][0][tid];
#pragma unroll
          for (int w = 1; w < WAVES; ++w) total += red[round][w][tid];
          float* dst = C + (size_t)m * ldc + n;
          if (k0 > 0) total += *dst;
          *dst = total + (last_pass && bias ? bias[n] : 0.f);
        }
      }
    }
    __syncthreads();    // the last tile's sums are read before the next pass writes over them
  }
}

// ---- more rows than a decode step: matrix cores ----------------------------------------------------------------
//
// The float32 MFMA 16x16x4 multiplies and adds in float32 (no bfloat16 or tf32 form), 256 flops a clock and CU like
// the vector ALU's FMAs, but an operand that is read from LDS once feeds a whole row of a 16x16 tile: the plain tile
// above needs an LDS read for every two FMAs a thread does, and that is what bound it.
// Block = 32 MI rows of A x 32 NI rows of B, KG groups of four waves (2 x 2 of 16 MI x 16 NI each).  K is walked in
// steps of BK through STAGES buffers in LDS, a share of a step for each group, whose sums meet at the end in the order
// of the groups: with two to four waves a SIMD one wave's reads of LDS and its wait at the step's barrier pass behind
// the others' MFMAs (one group, 700 x 4,096 x 1,024: 83 us, two 68), and shorter chains of sums round less.  A
// tile comes by `global_load_lds_dwordx4` straight from memory, STAGES - 1 steps ahead, waited for by count, one barrier
// a step.  A lane (r = lane % 16, q = lane / 16) reads a chunk of four neighbouring k of its row, which are the operands
// of four MFMAs: MFMA s of a sixteen of K adds the products at k = 4 q + s for q = 0..3, for A and B alike.
// Measured on one MI355X, plain tile -> this, us, for 700 rows: N = 4,096, K = 1,024 108 -> 68; N = 1,024, K = 2,048
// 133 -> 41; N = 6,144, K = 1,024 150 -> 105; N = 1,024, K = 3,072 190 -> 57; for 2,048 rows, N = 6,144, K = 2,560
// 870 -> 556 (116 TFLOP/s; the chip's large products reach 154).  What is left is the last, partly filled round of
// blocks and the waits at the steps' barriers.  Staging through registers instead (the compiler then counts the LDS
// reads' waits itself) was slower everywhere: 44 to 58 us where this takes 41.
typedef __attribute__((ext_vector_type(4))) float floatx4;

#define FE_XCDS 8
// wait until at most n of this wave's vector memory operations are outstanding
#define FE_WAIT_VMEM(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | ((((n) >> 4) & 0x3) << 14) | (0x7 << 4) | (0xF << 8))

__device__ __forceinline__ void load_to_lds(const void* global, void* lds) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)global,
                                   (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}

// COUNT times 16 bytes from LDS byte address `at`, STEP bytes apart, arrived when this returns (the compiler's own
// reads of LDS would wait for every load into LDS that is under way, too)
template <int COUNT, int STEP>
__device__ __forceinline__ void lds_read_rows(unsigned int at, floatx4* v) {
  if constexpr (COUNT == 1) asm volatile("ds_read_b128 %0, %1\n s_waitcnt lgkmcnt(0)" : "=&v"(v[0]) : "v"(at) : "memory");
  if constexpr (COUNT == 2)
    asm volatile("ds_read_b128 %0, %2\n ds_read_b128 %1, %2 offset:%3\n s_waitcnt lgkmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1]) : "v"(at), "n"(STEP) : "memory");
  if constexpr (COUNT == 4)
    asm volatile("ds_read_b128 %0, %4\n ds_read_b128 %1, %4 offset:%5\n ds_read_b128 %2, %4 offset:%6\n"
                 " ds_read_b128 %3, %4 offset:%7\n s_waitcnt lgkmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "v"(at), "n"(STEP), "n"(2 * STEP), "n"(3 * STEP) : "memory");
}

template <int MI, int NI, int STAGES, int KG, int BK>
__global__ __launch_bounds__(256 * KG) void gemm_tile_f32_kernel(
    const float* __restrict__ A, const float* __restrict__ B, const float* __restrict__ bias, float* __restrict__ C,
    int M, int N, int K, long long lda, long long ldb, long long ldc, int tiles_m, int tiles, int wide_store) {
  constexpr int BM = 32 * MI, BN = 32 * NI, CH = BK / 4, T = BK / (16 * KG);      // 16-byte chunks a row; sixteens of K a wave and step
  constexpr int LOADS = (BM + BN) * CH / (256 * KG);                              // loads a wave and step
  static_assert(T >= 1 && (BM + BN) * CH % (256 * KG) == 0, "every wave loads as much as every other");
  static_assert(STAGES * (BM + BN) * BK >= (KG - 1) * BM * BN, "the groups' sums meet in the same LDS");
  __shared__ __attribute__((aligned(16))) floatx4 lds[STAGES * (BM + BN) * CH];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Block b runs on XCD b % 8.  An XCD takes a run of neighbouring tiles, rows of A fastest, so that the blocks that
  // share rows of B find them in their L2.
  const int xcd = blockIdx.x % FE_XCDS, per = tiles / FE_XCDS, more = tiles % FE_XCDS;
  const int tile = xcd * per + min(xcd, more) + blockIdx.x / FE_XCDS;
  const int m0 = (tile % tiles_m) * BM, n0 = (tile / tiles_m) * BN;
  // the unit of a row that holds a chunk: sixteen lanes that read one chunk of sixteen rows touch every bank once
  auto swizzle = [](int row) { return CH == 8 ? (row >> 1) & 7 : row & 15; };

  const float* from[LOADS];      // this lane's row of each of the wave's loads (A's rows, then B's)
  int chunk[LOADS];              // ... and its place in that row
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int unit = (wave * LOADS + i) * 64 + lane, row = unit / CH;
    from[i] = row < BM ? A + (size_t)min(m0 + row, M - 1) * lda : B + (size_t)min(n0 + row - BM, N - 1) * ldb;
    chunk[i] = ((unit % CH) ^ swizzle(row)) * 4;
  }
  const int steps = (K + BK - 1) / BK;
  auto load = [&](int step, int stage) {       // past the end the last step again, so that the waits can count; chunks beyond K read the row's first
    const int k0 = min(step, steps - 1) * BK;
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      load_to_lds(from[i] + (k0 + chunk[i] < K ? k0 + chunk[i] : 0), &lds[stage * (BM + BN) * CH + (wave * LOADS + i) * 64]);
  };

  const int r = lane & 15, q = lane >> 4, group = wave >> 2, wm = wave & 1, wn = (wave >> 1) & 1;
  const unsigned int base = (unsigned int)(size_t)(const __attribute__((address_space(3))) char*)&lds[0];
  const unsigned int a_at = base + (wm * 16 * MI + r) * BK * 4, b_at = base + (BM + wn * 16 * NI + r) * BK * 4;
  floatx4 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  auto multiply = [&](int stage, int k0, bool partial) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int c = 4 * (group * T + t) + q;
      const unsigned int at = stage * ((BM + BN) * BK * 4) + ((c ^ swizzle(r)) * 16);
      floatx4 a[MI], b[NI];
      lds_read_rows<MI, BK * 64>(a_at + at, a);
      lds_read_rows<NI, BK * 64>(b_at + at, b);
      if (partial && k0 + c * 4 >= K) {      // chunks beyond K: nothing of either operand
#pragma unroll
        for (int i = 0; i < MI; ++i) a[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < NI; ++j) b[j] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j][s], a[i][s], acc[i][j], 0, 0, 0);
    }
  };

#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) load(s, s);
  const int whole = K / BK;
  int stage = 0, fill = STAGES - 1;
  for (int step = 0; step < steps; ++step) {
    FE_WAIT_VMEM(LOADS * (STAGES - 2));      // this wave's share of the step's tile has landed ...
    __builtin_amdgcn_s_barrier();            // ... and everyone's; everyone is done with the buffer that is filled next
    asm volatile("" ::: "memory");
    load(step + STAGES - 1, fill);
    if (step < whole) multiply(stage, step * BK, false);
    else multiply(stage, step * BK, true);
    stage = stage + 1 == STAGES ? 0 : stage + 1;
    fill = fill + 1 == STAGES ? 0 : fill + 1;
  }
  FE_WAIT_VMEM(0);       // the loads past the end have landed: the LDS is free
  if constexpr (KG > 1) {       // the groups' sums, added in the order of the groups
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (group > 0) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) lds[(((group - 1) * 4 + (wave & 3)) * MI * NI + i * NI + j) * 64 + lane] = acc[i][j];
    }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int g = 1; g < KG; ++g)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] += lds[(((g - 1) * 4 + wave) * MI * NI + i * NI + j) * 64 + lane];
  }

  // lane (r, q) holds rows of B n0 + 16 j + 4 q .. + 3 for row of A m0 + 16 i + r: four neighbouring columns of C
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int m = m0 + (wm * MI + i) * 16 + r;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int n = n0 + (wn * NI + j) * 16 + 4 * q;
      float* dst = C + (size_t)m * ldc + n;
      if (wide_store && n + 3 < N) {
        floatx4 v = acc[i][j];
        if (bias) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += bias[n + e];
        }
        *(floatx4*)dst = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) dst[e] = acc[i][j][e] + (bias ? bias[n + e] : 0.f);
      }
    }
  }
}

template <int MI, int NI, int STAGES, int KG, int BK>
static int launch_tile_f32(const float* A, const float* B, const float* bias, float* C, int M, int N, int K, long long lda,
                           long long ldb, long long ldc, hipStream_t stream) {
  const long long tiles_m = (M + 32 * MI - 1) / (32 * MI), tiles = tiles_m * ((N + 32 * NI - 1) / (32 * NI));
  if (tiles > 0x7fffffffLL) return FE_BAD_ARGUMENT;
  const int wide_store = ldc % 4 == 0 && (((uintptr_t)C) & 15) == 0;
  gemm_tile_f32_kernel<MI, NI, STAGES, KG, BK><<<dim3((unsigned)tiles), 256 * KG, 0, stream>>>(
      A, B, bias, C, M, N, K, lda, ldb, ldc, (int)tiles_m, (int)tiles, wide_store);
  return fe_check_launch();
}

#define FE_ROWS_F32_MAX 16     // most rows of A that the weight-streaming variant takes
#define FE_ROWS_F32_RESIDENT_MAX 64   // most rows of A that go through the variant with A in registers, eight at a time

// The tile (1,000 times its rows of A + its rows of B) that a product of more rows than the few-rows variants takes: the one that
// loads the fullest CU least.  A launch takes as long as the CU with the most tiles, so smaller tiles win where larger ones leave
// CUs idle or start a round of few blocks; a small tile takes somewhat longer for its area (more bytes from LDS and L2 a product).
// The factors are fitted to fourteen shapes of 70 to 2,048 rows, where the rule picks the fastest of the three or one within 2 %
// of it.
extern "C" int fe_gemm_nt_f32_tile(int M, int N) {
  auto rounds = [](long long tiles) { return (double)((tiles + 255) / 256); };
  const long long m64 = (M + 63LL) / 64, m32 = (M + 31LL) / 32, n64 = (N + 63LL) / 64, n32 = (N + 31LL) / 32;
  const double large = 4.0 * rounds(m64 * n64), half = 2.24 * rounds(m64 * n32), small = 1.22 * rounds(m32 * n32);
  if (large <= half && large <= small) return 64064;
  return half <= small ? 64032 : 32032;
}

extern "C" int fe_gemm_nt_f32(const float* A, const float* B, const float* bias, float* C,
                              int M, int N, int K, long long lda, long long ldb, long long ldc,
                              hipStream_t stream) {
  if (M <= 0 || N <= 0) return FE_OK;
  if (K <= 0 || lda < K || ldb < K || ldc < N) return FE_BAD_ARGUMENT;
  const bool rows_ok = M <= FE_ROWS_F32_MAX && K % 4 == 0 && lda % 4 == 0 && ldb % 4 == 0 &&
                       ((((uintptr_t)A) | ((uintptr_t)B)) & 15) == 0;
  const bool aligned = K % 4 == 0 && lda % 4 == 0 && ldb % 4 == 0 && ((((uintptr_t)A) | ((uintptr_t)B)) & 15) == 0;
  if (aligned && M <= FE_ROWS_F32_RESIDENT_MAX && K >= 1024) {
    // persistent blocks, two a CU with four waves (K up to 3,072 a pass), one with eight; more than
    // eight rows in groups of eight, a launch each: the weight is streamed once a group, which up to
    // 64 rows still beats the tiles below (measured at the 4B sizes, a decode step: 9 rows 11.7 ->
    // 8.2 ms, 17 rows 50.4 -> 11.8 ms, 32 rows 51.5 -> 16.2 ms; 64 rows 31.2 ms), and a row's sums
    // are those of the row alone
    const int tiles = (N + 1) / 2;
    for (int m0 = 0; m0 < M; m0 += 8) {
      const float* a = A + (size_t)m0 * lda;
      float* c = C + (size_t)m0 * ldc;
      const int rows = std::min(8, M - m0);
      if (K <= 2048) gemm_rows_resident_f32_kernel<2, 4><<<std::min(tiles, 512), 256, 0, stream>>>(a, B, bias, c, rows, N, K, lda, ldb, ldc);
      else if (K <= 3072) gemm_rows_resident_f32_kernel<3, 4><<<std::min(tiles, 512), 256, 0, stream>>>(a, B, bias, c, rows, N, K, lda, ldb, ldc);
      else if (K <= 4096) gemm_rows_resident_f32_kernel<2, 8><<<std::min(tiles, 256), 512, 0, stream>>>(a, B, bias, c, rows, N, K, lda, ldb, ldc);
      else gemm_rows_resident_f32_kernel<3, 8><<<std::min(tiles, 256), 512, 0, stream>>>(a, B, bias, c, rows, N, K, lda, ldb, ldc);
    }
    return fe_check_launch();
  }
  if (rows_ok) {
    if (M <= 4) gemm_rows_f32_kernel<4, 8><<<dim3((N + 7) / 8, 1), 256, 0, stream>>>(A, B, bias, C, M, N, K, lda, ldb, ldc);
    else if (M <= 8) gemm_rows_f32_kernel<8, 4><<<dim3((N + 3) / 4, 1), 256, 0, stream>>>(A, B, bias, C, M, N, K, lda, ldb, ldc);   // measured: four rows of B a block beat eight (more waves in flight)
    else gemm_rows_f32_kernel<16, 4><<<dim3((N + 3) / 4, 1), 256, 0, stream>>>(A, B, bias, C, M, N, K, lda, ldb, ldc);
    return fe_check_launch();
  }
  if (aligned) {
    switch (fe_gemm_nt_f32_tile(M, N)) {
      case 64064: return launch_tile_f32<2, 2, 2, 2, 64>(A, B, bias, C, M, N, K, lda, ldb, ldc, stream);
      case 64032: return launch_tile_f32<2, 1, 3, 2, 64>(A, B, bias, C, M, N, K, lda, ldb, ldc, stream);
      default: return launch_tile_f32<1, 1, 4, 4, 64>(A, B, bias, C, M, N, K, lda, ldb, ldc, stream);
    }
  }
  const long long grid_y = (M + TILE_M - 1) / TILE_M;
  if (grid_y > 65535) return FE_BAD_ARGUMENT;
  dim3 grid((N + TILE_N - 1) / TILE_N, (unsigned)grid_y);
  gemm_nt_f32_kernel<<<grid, 256, 0, stream>>>(A, B, bias, C, M, N, K, lda, ldb, ldc);
  return fe_check_launch();
}

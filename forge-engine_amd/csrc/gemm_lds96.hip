// The product through LDS (gemm_lds.h) in tiles of 96 rows of x, which stand between those of 64 and 128: a library of their own, since
// gemm_wide's is the one that takes longest to compile.
#include "common.h"
#include "gate_act.h"
#include "gemm_lds.h"

// x [M][K], w [N][K] (gated: [2N][K], gate rows first), bfloat16, rows of x whole and of w ldw apart; ending 0: float32 partial sums [parts][M][N]
// (part_stride apart, rows ldo), 1: bfloat16, 2: act(gate) * up as bfloat16 (activation: gate_act.h); tile 96064, 96096 or 96128.  K a multiple of 64.
extern "C" int fe_gemm_lds96(const void* x, const void* w, void* out, int M, int N, int K, long long ldw, long long ldo, int ending,
                             int parts, long long part_stride, int tile, int activation, hipStream_t stream) {
  if (M < 1) return FE_OK;
  GateAct act;
  if (!gate_act(activation, &act)) return FE_BAD_ARGUMENT;
  if (N < 1 || K < lds_tile::KSTEP || K % lds_tile::KSTEP || ldw < K || ldw % 8 || ldo < N) return FE_BAD_ARGUMENT;
  if (((((uintptr_t)x) | ((uintptr_t)w)) & 15) || parts < 1 || parts > 64 || (ending != through_lds::END_PARTS && parts != 1)) return FE_BAD_ARGUMENT;
  if (parts > 1 && part_stride < (long long)M * ldo) return FE_BAD_ARGUMENT;
  return through_lds::launch_96((const bf16_t*)x, (const bf16_t*)w, out, M, N, K, ldw, ldo, ending, parts, part_stride, tile, act, stream);
}

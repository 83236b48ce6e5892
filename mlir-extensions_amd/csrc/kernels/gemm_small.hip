// Entry points of the small-tile MFMA GEMM (gemm_small.h): the operators of gemm.hip, same arguments and results,
// with tiles of 128 x 128, 128 x 64, 64 x 64, 32 x 64 and 16 x 64 outputs.  imexHipKernelVariant says which of them a
// problem should take.
//
// Launch: block (512,1,1); grid (ceil(M / TM) * ceil(N / TN),1,1); workgroups stride, so any grid is correct.

#include "gemm_small.h"

using namespace imexhip;
using namespace imexhip_gemm;

using Tile128 = SmallShape<128, 128, 2, 2, 2, 4>;
using Tile128x64 = SmallShape<128, 64, 2, 2, 2, 6>;
using Tile64 = SmallShape<64, 64, 2, 2, 2, 5>;
using Tile32 = SmallShape<32, 64, 1, 2, 4, 6>;
using Tile16 = SmallShape<16, 64, 1, 1, 8, 4>;

#define IMEX_GEMM_SMALL(BASE, TILE, SHAPE, T, AT, BT, OUT, EPI)                                                       \
  extern "C" __global__ __launch_bounds__(kThreads, SHAPE::kWavesPerEu) void BASE##TILE(const uint16_t *A, const uint16_t *B, OUT *C,     \
                                                                    int64_t M, int64_t N, int64_t K) {                \
    gemm_small_entry<T, AT, BT, SHAPE>(A, B, M, N, K, EPI{C});                                                        \
  }
#define IMEX_GEMM_SMALL_BIAS(BASE, TILE, SHAPE)                                                                       \
  extern "C" __global__ __launch_bounds__(kThreads, SHAPE::kWavesPerEu) void BASE##TILE(const uint16_t *A, const uint16_t *B,             \
                                                                    const float *bias, uint16_t *out, int64_t M,      \
                                                                    int64_t N, int64_t K) {                           \
    gemm_small_entry<BF16, false, false, SHAPE>(A, B, M, N, K, BiasSiluBF16{out, bias});                              \
  }
#define IMEX_GEMM_SMALL_ALL(TILE, SHAPE)                                                                              \
  IMEX_GEMM_SMALL(imex_gemm_f16_f16_f32, TILE, SHAPE, F16, false, false, float, StoreF32)                             \
  IMEX_GEMM_SMALL(imex_gemm_f16_f16_f32_acc, TILE, SHAPE, F16, false, false, float, AccumulateF32)                    \
  IMEX_GEMM_SMALL(imex_gemm_bf16_bf16_f32, TILE, SHAPE, BF16, false, false, float, StoreF32)                          \
  IMEX_GEMM_SMALL(imex_gemm_bf16_bf16_f32_acc, TILE, SHAPE, BF16, false, false, float, AccumulateF32)                 \
  IMEX_GEMM_SMALL(imex_gemm_f16_f16_f16, TILE, SHAPE, F16, false, false, uint16_t, StoreF16)                          \
  IMEX_GEMM_SMALL(imex_gemm_f16_f16_f32_tb, TILE, SHAPE, F16, false, true, float, StoreF32)                           \
  IMEX_GEMM_SMALL(imex_gemm_f16_f16_f32_ta, TILE, SHAPE, F16, true, false, float, StoreF32)                           \
  IMEX_GEMM_SMALL_BIAS(imex_gemm_bf16_bias_silu_bf16, TILE, SHAPE)

IMEX_GEMM_SMALL_ALL(_t128, Tile128)
IMEX_GEMM_SMALL_ALL(_t128x64, Tile128x64)
IMEX_GEMM_SMALL_ALL(_t64, Tile64)
IMEX_GEMM_SMALL_ALL(_t32, Tile32)
IMEX_GEMM_SMALL_ALL(_t16, Tile16)

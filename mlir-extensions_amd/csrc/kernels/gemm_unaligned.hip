// Entry points of the MFMA GEMM for rows that are not 16-byte aligned (gemm_unaligned.h): the operators of gemm.hip,
// same arguments, with tiles of 128 x 128 and 64 x 64 outputs.  imexHipKernelVariant says which problems take them.
//
// Launch: block (512,1,1); grid (ceil(M / TM) * ceil(N / TN),1,1); workgroups stride, so any grid is correct.

#include "gemm_unaligned.h"

using namespace imexhip;
using namespace imexhip_gemm;

using Tile128 = SmallShape<128, 128, 2, 2, 2, 2>;
using Tile64 = SmallShape<64, 64, 2, 2, 2, 2>;

#define IMEX_GEMM_UNALIGNED(BASE, TILE, SHAPE, D, T, AT, BT, OUT, EPI)                                                 \
  extern "C" __global__ __launch_bounds__(kThreads, SHAPE::kWavesPerEu) void BASE##TILE(                              \
      const uint16_t *A, const uint16_t *B, OUT *C, int64_t M, int64_t N, int64_t K) {                                \
    gemm_unaligned_entry<T, AT, BT, SHAPE, D>(A, B, M, N, K, EPI{C});                                                 \
  }
#define IMEX_GEMM_UNALIGNED_BIAS(BASE, TILE, SHAPE, D)                                                                 \
  extern "C" __global__ __launch_bounds__(kThreads, SHAPE::kWavesPerEu) void BASE##TILE(                              \
      const uint16_t *A, const uint16_t *B, const float *bias, uint16_t *out, int64_t M, int64_t N, int64_t K) {      \
    gemm_unaligned_entry<BF16, false, false, SHAPE, D>(A, B, M, N, K, BiasSiluBF16{out, bias});                       \
  }
#define IMEX_GEMM_UNALIGNED_ALL(TILE, SHAPE, D)                                                                        \
  IMEX_GEMM_UNALIGNED(imex_gemm_f16_f16_f32, TILE, SHAPE, D, F16, false, false, float, StoreF32)                      \
  IMEX_GEMM_UNALIGNED(imex_gemm_f16_f16_f32_acc, TILE, SHAPE, D, F16, false, false, float, AccumulateF32)             \
  IMEX_GEMM_UNALIGNED(imex_gemm_bf16_bf16_f32, TILE, SHAPE, D, BF16, false, false, float, StoreF32)                   \
  IMEX_GEMM_UNALIGNED(imex_gemm_bf16_bf16_f32_acc, TILE, SHAPE, D, BF16, false, false, float, AccumulateF32)          \
  IMEX_GEMM_UNALIGNED(imex_gemm_f16_f16_f16, TILE, SHAPE, D, F16, false, false, uint16_t, StoreF16)                   \
  IMEX_GEMM_UNALIGNED(imex_gemm_f16_f16_f32_tb, TILE, SHAPE, D, F16, false, true, float, StoreF32)                    \
  IMEX_GEMM_UNALIGNED(imex_gemm_f16_f16_f32_ta, TILE, SHAPE, D, F16, true, false, float, StoreF32)                    \
  IMEX_GEMM_UNALIGNED_BIAS(imex_gemm_bf16_bias_silu_bf16, TILE, SHAPE, D)

// slabs in flight: four where a slab is two 16-byte pieces per lane, two where it is four and a step takes longer
IMEX_GEMM_UNALIGNED_ALL(_u128, Tile128, 2)
IMEX_GEMM_UNALIGNED_ALL(_u64, Tile64, 4)

// Entry points of the MFMA GEMM for rows that are not 16-byte aligned (gemm_unaligned.h): the operators of gemm.hip,
// same arguments, with tiles of 128 x 128, 64 x 64, 32 x 64, 16 x 32 and 16 x 16 outputs.  imexHipKernelVariant says which
// problems take them.
//
// Launch: block (512,1,1); grid (ceil(M / TM) * ceil(N / TN),1,1); workgroups stride, so any grid is correct.

#include "gemm_unaligned.h"

using namespace imexhip;
using namespace imexhip_gemm;

using Tile128 = SmallShape<128, 128, 2, 2, 2, 2>;
using Tile64 = SmallShape<64, 64, 2, 2, 2, 2>;
// Few rows and columns: tiles of which every CU gets one, k shared by four or eight wavefronts (us with 64 x 64 / so):
//   32 x 64           441 x 441 x 351 5.6 / 4.8, 333 x 777 x 555 6.8 / 6.1
//   16 x 32, 16 x 16  131 x 133 x 999 8.8 / 5.5 / 4.7, 200 x 301 x 901 9.0 / 5.8 / 4.8
// (32 x 32: 6.5, 6.9.)  128 x 64 would spill at two workgroups per CU: 1500 x 1501 x 997 24.0, 17.4 with 128 x 128.
using Tile32 = SmallShape<32, 64, 1, 2, 4, 2>;
using Tile16x32 = SmallShape<16, 32, 1, 1, 8, 2>;
using Tile16x16 = SmallShape<16, 16, 1, 1, 8, 2>;

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

// slabs in flight: four where a slab is two 16-byte pieces per lane, two where it is more and a step takes longer (32 x 64
// with four 8.9 us on 333 x 777 x 555), or where a step is 256 k
IMEX_GEMM_UNALIGNED_ALL(_u128, Tile128, 2)
IMEX_GEMM_UNALIGNED_ALL(_u64, Tile64, 4)
IMEX_GEMM_UNALIGNED_ALL(_u32, Tile32, 2)
IMEX_GEMM_UNALIGNED_ALL(_u16x32, Tile16x32, 2)
IMEX_GEMM_UNALIGNED_ALL(_u16x16, Tile16x16, 2)

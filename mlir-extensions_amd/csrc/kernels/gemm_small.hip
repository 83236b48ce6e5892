// Entry points of the small-tile MFMA GEMM (gemm_small.h): the operators of gemm.hip, same arguments and results,
// with tiles of 256 x 128, 128 x 128, 128 x 64, 64 x 64, 32 x 64, 16 x 64, 16 x 32 and 16 x 16 outputs.
// imexHipKernelVariant says which of them a problem should take.
//
// Launch: block (512,1,1); grid (ceil(M / TM) * ceil(N / TN),1,1), or 256 workgroups where those without a tile pay as ones
// that fetch for the others (fetch_ahead; fetchesAhead in KernelCatalog.cpp); workgroups stride, so any grid is correct.

#include "gemm_small.h"

using namespace imexhip;
using namespace imexhip_gemm;

// The last number is the ring's stages.  More of them do not make a K step shorter -- a CU's requests beyond its L2 are
// what bounds the small tiles (16 x 16 on N = 1680: 0.36 us per 256 k with 3, 4, 8 and 9 stages) -- but the first result
// later (K = 1024: 3.4, 3.7, 3.8, 4.0 us), so: what lets workgroups share a CU, or what hides the latency of a step.
// "true" refills a slot in the step that has its fragments in registers, a step sooner than the rest, and so does with a
// stage less: 128 x 128 (4 stages before) 1616 x 1760 x 3616 33.2 -> 31.9 us, 1064 x 2200 x 424 9.2 -> 8.9; 64 x 64 (5
// before) 912 x 944 x 520 5.33 -> 5.14, 1000 x 1592 x 1168 the same; 128 x 64 and narrower tiles gain nothing or lose 1 %.
//   256 x 128  between 128 x 128 tiles for two rounds and 256 x 256 for less than half the chip: 2414 x 2104 x 2208 44.4 us
//              with 128 x 128, 36.4 so; 892 x 4768 x 3096 60.6 / 47.1; 1704 x 2648 x 4088 A^T 97.6 (64 x 64) / 59.3
//   128 x 64 s two workgroups on a CU for problems of more than one round: 1542 x 4000 x 720 32.8 -> 26.6
//   16 x 32, 16 x 16  few rows: a CU gets 40 .. 60 GB/s from beyond its L2, so narrow outputs bring more CUs to the weights:
//              16 x 1680 x 3992 13.8 us with 16 x 64, 9.8 so; 5 x 2200 x 1160 5.8 -> 4.0
using Tile256x128 = SmallShape<256, 128, 2, 2, 2, 3>;
using Tile128 = SmallShape<128, 128, 2, 2, 2, 3, true>;
using Tile128x64 = SmallShape<128, 64, 2, 2, 2, 4>;
using Tile128x64Shared = SmallShape<128, 64, 2, 2, 2, 3>;
using Tile64 = SmallShape<64, 64, 2, 2, 2, 4, true>;
using Tile32 = SmallShape<32, 64, 1, 2, 4, 4>;
using Tile16 = SmallShape<16, 64, 1, 1, 8, 3>;
using Tile16x32 = SmallShape<16, 32, 1, 1, 8, 3>;
using Tile16x16 = SmallShape<16, 16, 1, 1, 8, 3>;

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

IMEX_GEMM_SMALL_ALL(_t256x128, Tile256x128)
IMEX_GEMM_SMALL_ALL(_t128, Tile128)
IMEX_GEMM_SMALL_ALL(_t128x64, Tile128x64)
IMEX_GEMM_SMALL_ALL(_t128x64s, Tile128x64Shared)
IMEX_GEMM_SMALL_ALL(_t64, Tile64)
IMEX_GEMM_SMALL_ALL(_t32, Tile32)
IMEX_GEMM_SMALL_ALL(_t16, Tile16)
IMEX_GEMM_SMALL_ALL(_t16x32, Tile16x32)
IMEX_GEMM_SMALL_ALL(_t16x16, Tile16x16)

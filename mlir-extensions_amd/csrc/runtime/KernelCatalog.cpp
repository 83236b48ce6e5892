//===- KernelCatalog.cpp - embedded gfx950 code objects + launch shapes ----===//
//
// Host-side table of the hand-written kernels: which embedded code object
// holds each one and the grid/block it is launched with.  This plays the part
// of the `gpu.binary` blob plus the `blocks in (...) threads in (...)` operands
// that IMEX's lowering bakes into host code
// (lib/Conversion/GPUXToLLVM/GPUXToLLVMPass.cpp:456-713).
//
//===----------------------------------------------------------------------===//

#include "imex_hip_kernels.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <iterator>

// Blob symbols come from the assembler stub generated at build time
// (one .incbin per code object).
extern "C" {
extern const unsigned char imex_blob_eltwise[], imex_blob_eltwise_end[];
extern const unsigned char imex_blob_softmax[], imex_blob_softmax_end[];
extern const unsigned char imex_blob_reduce[], imex_blob_reduce_end[];
extern const unsigned char imex_blob_transpose[], imex_blob_transpose_end[];
extern const unsigned char imex_blob_gemm[], imex_blob_gemm_end[];
extern const unsigned char imex_blob_gemm_small[], imex_blob_gemm_small_end[];
extern const unsigned char imex_blob_gemm_unaligned[], imex_blob_gemm_unaligned_end[];
extern const unsigned char imex_blob_fusion[], imex_blob_fusion_end[];
extern const unsigned char imex_blob_attention[], imex_blob_attention_end[];
}

namespace {

enum class Module { Eltwise, Softmax, Reduce, Transpose, Gemm, GemmSmall, GemmUnaligned, Fusion, Attention };
enum class Shape {
  Eltwise32, Eltwise16, Fusion32, Fusion16, SoftmaxRows32, SoftmaxRows16, SoftmaxShared32, SoftmaxShared16,
  RowSum, RowSumShort, ReduceOuter, ReduceOuter16, ReduceTall32, ReduceTall16, ReduceDeep32, ReduceDeep16,
  Transpose2D32, Transpose2D16, Transpose3D32, Transpose3D16, TransposeAny32, TransposeAny16, Gemm,
  GemmStreamK, GemmTA, GemmTB, GemmSmall, GemmUnaligned, GemmFixed4k, ColumnThreads, ColumnThreads16,
  ColumnChains, ColumnChains16, Attention, AttentionTiling
};

struct Entry {
  const char *name;
  const char *signature;
  Module module;
  Shape shape;
  int ndims;
};

// The operators that exist with smaller tiles too (gemm_small.hip), and for rows that are not 16-byte aligned
// (gemm_unaligned.hip), one entry per tile.
#define IMEX_GEMM_SMALL_TILES(NAME, SIGNATURE)                                                                        \
  {NAME "_t128", SIGNATURE, Module::GemmSmall, Shape::GemmSmall, 3},                                                  \
      {NAME "_t128x64", SIGNATURE, Module::GemmSmall, Shape::GemmSmall, 3},                                           \
      {NAME "_t64", SIGNATURE, Module::GemmSmall, Shape::GemmSmall, 3},                                               \
      {NAME "_t32", SIGNATURE, Module::GemmSmall, Shape::GemmSmall, 3},                                               \
      {NAME "_t16", SIGNATURE, Module::GemmSmall, Shape::GemmSmall, 3},                                               \
      {NAME "_t256x128", SIGNATURE, Module::GemmSmall, Shape::GemmSmall, 3},                                          \
      {NAME "_t128x64s", SIGNATURE, Module::GemmSmall, Shape::GemmSmall, 3},                                          \
      {NAME "_t16x32", SIGNATURE, Module::GemmSmall, Shape::GemmSmall, 3},                                            \
      {NAME "_t16x16", SIGNATURE, Module::GemmSmall, Shape::GemmSmall, 3},                                            \
      {NAME "_u128", SIGNATURE, Module::GemmUnaligned, Shape::GemmUnaligned, 3},                                      \
      {NAME "_u64", SIGNATURE, Module::GemmUnaligned, Shape::GemmUnaligned, 3},                                       \
      {NAME "_u32", SIGNATURE, Module::GemmUnaligned, Shape::GemmUnaligned, 3},                                       \
      {NAME "_u16x32", SIGNATURE, Module::GemmUnaligned, Shape::GemmUnaligned, 3},                                    \
      {NAME "_u16x16", SIGNATURE, Module::GemmUnaligned, Shape::GemmUnaligned, 3}

const Entry kEntries[] = {
    {"imex_relu_f32", "(in: f32*, out: f32*, n: i64)", Module::Eltwise, Shape::Eltwise32, 1},
    {"imex_relu_f16", "(in: f16*, out: f16*, n: i64)", Module::Eltwise, Shape::Eltwise16, 1},
    {"imex_relu_bf16", "(in: bf16*, out: bf16*, n: i64)", Module::Eltwise, Shape::Eltwise16, 1},
    {"imex_silu_f32", "(in: f32*, out: f32*, n: i64)", Module::Eltwise, Shape::Fusion32, 1},
    {"imex_silu_f16", "(in: f16*, out: f16*, n: i64)", Module::Eltwise, Shape::Fusion16, 1},
    {"imex_silu_bf16", "(in: bf16*, out: bf16*, n: i64)", Module::Eltwise, Shape::Fusion16, 1},
    {"imex_exp_f32", "(in: f32*, out: f32*, n: i64)", Module::Eltwise, Shape::Fusion32, 1},
    {"imex_maximum_f32", "(a: f32*, b: f32*, out: f32*, n: i64)", Module::Eltwise, Shape::Eltwise32, 1},
    {"imex_softmax_f32", "(in: f32*, out: f32*, rows: i64, cols: i64)", Module::Softmax, Shape::SoftmaxRows32, 2},
    {"imex_softmax_f16", "(in: f16*, out: f16*, rows: i64, cols: i64)", Module::Softmax, Shape::SoftmaxRows16, 2},
    {"imex_softmax_bf16", "(in: bf16*, out: bf16*, rows: i64, cols: i64)", Module::Softmax, Shape::SoftmaxRows16, 2},
    {"imex_softmax_f32_shared", "(in: f32*, out: f32*, rows: i64, cols: i64)", Module::Softmax, Shape::SoftmaxShared32, 2},
    {"imex_softmax_f16_shared", "(in: f16*, out: f16*, rows: i64, cols: i64)", Module::Softmax, Shape::SoftmaxShared16, 2},
    {"imex_softmax_bf16_shared", "(in: bf16*, out: bf16*, rows: i64, cols: i64)", Module::Softmax, Shape::SoftmaxShared16, 2},
    {"imex_rowsum_f32", "(in: f32*, out: f32*, rows: i64, cols: i64, init: f32)", Module::Reduce, Shape::RowSum, 2},
    {"imex_rowmean_f32", "(in: f32*, out: f32*, rows: i64, cols: i64)", Module::Reduce, Shape::RowSum, 2},
    {"imex_rowsum_f32_short", "(in: f32*, out: f32*, rows: i64, cols: i64, init: f32)", Module::Reduce, Shape::RowSumShort, 2},
    {"imex_rowmean_f32_short", "(in: f32*, out: f32*, rows: i64, cols: i64)", Module::Reduce, Shape::RowSumShort, 2},
    {"imex_reduce_outer_f32", "(in: f32*, out: f32*, outer: i64, inner: i64, init: f32)", Module::Reduce,
     Shape::ReduceOuter, 2},
    {"imex_reduce_outer_f16", "(in: f16*, out: f16*, outer: i64, inner: i64, init: f32)", Module::Reduce,
     Shape::ReduceOuter16, 2},
    {"imex_reduce_outer_bf16", "(in: bf16*, out: bf16*, outer: i64, inner: i64, init: f32)", Module::Reduce,
     Shape::ReduceOuter16, 2},
    {"imex_reduce_outer_f32_tall", "(in: f32*, out: f32*, outer: i64, inner: i64, init: f32)", Module::Reduce,
     Shape::ReduceTall32, 2},
    {"imex_reduce_outer_f16_tall", "(in: f16*, out: f16*, outer: i64, inner: i64, init: f32)", Module::Reduce,
     Shape::ReduceTall16, 2},
    {"imex_reduce_outer_bf16_tall", "(in: bf16*, out: bf16*, outer: i64, inner: i64, init: f32)", Module::Reduce,
     Shape::ReduceTall16, 2},
    {"imex_reduce_outer_f32_deep", "(in: f32*, out: f32*, outer: i64, inner: i64, init: f32)", Module::Reduce,
     Shape::ReduceDeep32, 2},
    {"imex_reduce_outer_f16_deep", "(in: f16*, out: f16*, outer: i64, inner: i64, init: f32)", Module::Reduce,
     Shape::ReduceDeep16, 2},
    {"imex_reduce_outer_bf16_deep", "(in: bf16*, out: bf16*, outer: i64, inner: i64, init: f32)", Module::Reduce,
     Shape::ReduceDeep16, 2},
    {"imex_transpose2d_b32", "(in: b32*, out: b32*, rows: i64, cols: i64)", Module::Transpose, Shape::Transpose2D32, 2},
    {"imex_transpose2d_b16", "(in: b16*, out: b16*, rows: i64, cols: i64)", Module::Transpose, Shape::Transpose2D16, 2},
    {"imex_transpose3d_b32", "(in: b32*, out: b32*, d0: i64, d1: i64, d2: i64)", Module::Transpose,
     Shape::Transpose3D32, 3},
    {"imex_transpose3d_b16", "(in: b16*, out: b16*, d0: i64, d1: i64, d2: i64)", Module::Transpose,
     Shape::Transpose3D16, 3},
    {"imex_transpose2d_b32_any", "(in: b32*, out: b32*, rows: i64, cols: i64)", Module::Transpose, Shape::TransposeAny32, 2},
    {"imex_transpose2d_b16_any", "(in: b16*, out: b16*, rows: i64, cols: i64)", Module::Transpose, Shape::TransposeAny16, 2},
    {"imex_transpose3d_b32_any", "(in: b32*, out: b32*, d0: i64, d1: i64, d2: i64)", Module::Transpose,
     Shape::TransposeAny32, 3},
    {"imex_transpose3d_b16_any", "(in: b16*, out: b16*, d0: i64, d1: i64, d2: i64)", Module::Transpose,
     Shape::TransposeAny16, 3},
    {"imex_loop_fusion_f32", "(a: f32*, b: f32*, out: f32*, n: i64)", Module::Fusion, Shape::Fusion32, 1},
    {"imex_loop_fusion_f16", "(a: f16*, b: f16*, out: f16*, n: i64)", Module::Fusion, Shape::Fusion16, 1},
    {"imex_loop_fusion_bf16", "(a: bf16*, b: bf16*, out: bf16*, n: i64)", Module::Fusion, Shape::Fusion16, 1},
    {"imex_input_fusion_f32", "(a: f32*, b: f32*, out: f32*, rows: i64, cols: i64)", Module::Fusion,
     Shape::ColumnThreads, 2},
    {"imex_input_fusion_f16", "(a: f16*, b: f16*, out: f16*, rows: i64, cols: i64)", Module::Fusion,
     Shape::ColumnThreads16, 2},
    {"imex_input_fusion_bf16", "(a: bf16*, b: bf16*, out: bf16*, rows: i64, cols: i64)", Module::Fusion,
     Shape::ColumnThreads16, 2},
    {"imex_input_fusion_f32_tall", "(a: f32*, b: f32*, out: f32*, rows: i64, cols: i64)", Module::Fusion,
     Shape::ColumnChains, 2},
    {"imex_input_fusion_f16_tall", "(a: f16*, b: f16*, out: f16*, rows: i64, cols: i64)", Module::Fusion,
     Shape::ColumnChains16, 2},
    {"imex_input_fusion_bf16_tall", "(a: bf16*, b: bf16*, out: bf16*, rows: i64, cols: i64)", Module::Fusion,
     Shape::ColumnChains16, 2},
    {"imex_flash_attention_fwd_f16",
     "(Q: f16*, K: f16*, V: f16*, Out: f16*, sm_scale: f32, ZH: i64, N_CTX: i64)", Module::Attention,
     Shape::Attention, 2},
    {"imex_flash_attention_fwd_f16_q32",
     "(Q: f16*, K: f16*, V: f16*, Out: f16*, sm_scale: f32, ZH: i64, N_CTX: i64)", Module::Attention,
     Shape::AttentionTiling, 2},
    {"imex_flash_attention_fwd_f16_q64",
     "(Q: f16*, K: f16*, V: f16*, Out: f16*, sm_scale: f32, ZH: i64, N_CTX: i64)", Module::Attention,
     Shape::AttentionTiling, 2},
    {"imex_flash_attention_fwd_f16_q128",
     "(Q: f16*, K: f16*, V: f16*, Out: f16*, sm_scale: f32, ZH: i64, N_CTX: i64)", Module::Attention,
     Shape::AttentionTiling, 2},
    {"imex_flash_attention_fwd_f16_q256",
     "(Q: f16*, K: f16*, V: f16*, Out: f16*, sm_scale: f32, ZH: i64, N_CTX: i64)", Module::Attention,
     Shape::AttentionTiling, 2},
    {"imex_gemm_f16_f16_f32", "(A: f16*, B: f16*, C: f32*, M: i64, N: i64, K: i64)", Module::Gemm, Shape::Gemm, 3},
    {"imex_gemm_f16_f16_f32_acc", "(A: f16*, B: f16*, C: f32*, M: i64, N: i64, K: i64)", Module::Gemm, Shape::Gemm, 3},
    {"imex_gemm_bf16_bf16_f32", "(A: bf16*, B: bf16*, C: f32*, M: i64, N: i64, K: i64)", Module::Gemm, Shape::Gemm, 3},
    {"imex_gemm_bf16_bf16_f32_acc", "(A: bf16*, B: bf16*, C: f32*, M: i64, N: i64, K: i64)", Module::Gemm,
     Shape::Gemm, 3},
    {"imex_gemm_f16_f16_f16", "(A: f16*, B: f16*, C: f16*, M: i64, N: i64, K: i64)", Module::Gemm, Shape::Gemm, 3},
    {"imex_gemm_bf16_bias_silu_bf16", "(A: bf16*, B: bf16*, bias: f32*, out: bf16*, M: i64, N: i64, K: i64)",
     Module::Gemm, Shape::Gemm, 3},
    {"imex_gemm_bf16_bias_silu_bf16_streamk",
     "(A: bf16*, B: bf16*, bias: f32*, out: bf16*, M: i64, N: i64, K: i64, workspace: i8*, epoch: i64, spin_limit: i64)",
     Module::Gemm, Shape::GemmStreamK, 3},
    {"imex_gemm_f16_f16_f32_tb", "(A: f16*, Bt: f16* [N,K], C: f32*, M: i64, N: i64, K: i64)", Module::Gemm,
     Shape::GemmTB, 3},
    {"imex_gemm_f16_f16_f32_ta", "(At: f16* [K,M], B: f16*, C: f32*, M: i64, N: i64, K: i64)", Module::Gemm,
     Shape::GemmTA, 3},
    IMEX_GEMM_SMALL_TILES("imex_gemm_f16_f16_f32", "(A: f16*, B: f16*, C: f32*, M: i64, N: i64, K: i64)"),
    IMEX_GEMM_SMALL_TILES("imex_gemm_f16_f16_f32_acc", "(A: f16*, B: f16*, C: f32*, M: i64, N: i64, K: i64)"),
    IMEX_GEMM_SMALL_TILES("imex_gemm_bf16_bf16_f32", "(A: bf16*, B: bf16*, C: f32*, M: i64, N: i64, K: i64)"),
    IMEX_GEMM_SMALL_TILES("imex_gemm_bf16_bf16_f32_acc", "(A: bf16*, B: bf16*, C: f32*, M: i64, N: i64, K: i64)"),
    IMEX_GEMM_SMALL_TILES("imex_gemm_f16_f16_f16", "(A: f16*, B: f16*, C: f16*, M: i64, N: i64, K: i64)"),
    IMEX_GEMM_SMALL_TILES("imex_gemm_bf16_bias_silu_bf16",
                          "(A: bf16*, B: bf16*, bias: f32*, out: bf16*, M: i64, N: i64, K: i64)"),
    IMEX_GEMM_SMALL_TILES("imex_gemm_f16_f16_f32_tb", "(A: f16*, Bt: f16* [N,K], C: f32*, M: i64, N: i64, K: i64)"),
    IMEX_GEMM_SMALL_TILES("imex_gemm_f16_f16_f32_ta", "(At: f16* [K,M], B: f16*, C: f32*, M: i64, N: i64, K: i64)"),
    {"imex_gemm_4kx4kx4k_f16_f16_f32", "(A: f16*, B: f16*, C: f32*)", Module::Gemm, Shape::GemmFixed4k, 0},
    {"imex_gemm_4kx4kx4k_transpose_b", "(A: f16*, Bt: f16* [N,K], C: f32*)", Module::Gemm, Shape::GemmFixed4k, 0},
    {"imex_gemm_4kx4kx4k_transpose_a", "(At: f16* [K,M], B: f16*, C: f32*)", Module::Gemm, Shape::GemmFixed4k, 0},
    {"imex_gemm_4kx4kx4k_f16_f16_f32_bias", "(bias: f32*, C: f32*, A: f16*, B: f16*)", Module::Gemm,
     Shape::GemmFixed4k, 0},
};
constexpr int kEntryCount = sizeof(kEntries) / sizeof(kEntries[0]);

const Entry *find(const char *name) {
  if (!name)
    return nullptr;
  for (const Entry &e : kEntries)
    if (strcmp(e.name, name) == 0)
      return &e;
  return nullptr;
}

size_t ceilDiv(int64_t a, int64_t b) { return static_cast<size_t>((a + b - 1) / b); }

// The grid of a form whose problem has `groups` workgroups of work.  HIP takes fewer than 2^32 lanes per dimension of a
// launch, and the kernels stride over what a smaller grid leaves out.  (A multiple of 8: as many for each XCD.)
size_t gridFor(size_t groups, size_t block) { return std::min(groups, ((size_t(1) << 32) - 1) / block / 8 * 8); }

// How many 32-byte segments of a row a workgroup of column chains takes (chain_lanes in column_chain.h).
int chainWidth(size_t segments) { return segments <= 256 ? 1 : segments <= 512 ? 2 : 4; }

// What the MFMA paths of the GEMM kernels take (mfma_takes in gemm_tile.h): 16-byte aligned rows, and operands
// addressed through one 32-bit-offset buffer descriptor below 2 GiB.
bool mfmaTakes(bool transA, bool transB, int64_t M, int64_t N, int64_t K) {
  const int64_t twoGiB = int64_t(1) << 31, maxRow = int64_t(1) << 22;
  const bool fitsA = transA ? K * M * 2 < twoGiB : K < maxRow;
  const bool fitsB = transB ? K < maxRow : K * N * 2 < twoGiB;
  return M > 0 && N > 0 && K > 0 && K % 8 == 0 && (transB || N % 8 == 0) && (!transA || M % 8 == 0) && fitsA && fitsB;
}

// What the MFMA path for unaligned rows takes (unaligned_takes in gemm_unaligned.h).
bool unalignedTakes(bool transA, bool transB, int64_t M, int64_t N, int64_t K) {
  const int64_t maxRow = int64_t(1) << 22;
  return M > 0 && N > 0 && K >= 8 && K < maxRow && (!transA || (M >= 8 && M < maxRow)) &&
         (transB || (N >= 8 && N < maxRow));
}

} // namespace

extern "C" int imexHipKernelCount(void) { return kEntryCount; }

extern "C" const char *imexHipKernelName(int index) {
  return (index >= 0 && index < kEntryCount) ? kEntries[index].name : nullptr;
}

extern "C" const char *imexHipKernelSignature(int index) {
  return (index >= 0 && index < kEntryCount) ? kEntries[index].signature : nullptr;
}

extern "C" const void *imexHipKernelModule(const char *kernel, size_t *size) {
  const Entry *e = find(kernel);
  if (!e)
    return nullptr;
  const unsigned char *begin = nullptr, *end = nullptr;
  switch (e->module) {
  case Module::Eltwise: begin = imex_blob_eltwise; end = imex_blob_eltwise_end; break;
  case Module::Softmax: begin = imex_blob_softmax; end = imex_blob_softmax_end; break;
  case Module::Reduce: begin = imex_blob_reduce; end = imex_blob_reduce_end; break;
  case Module::Transpose: begin = imex_blob_transpose; end = imex_blob_transpose_end; break;
  case Module::Gemm: begin = imex_blob_gemm; end = imex_blob_gemm_end; break;
  case Module::GemmSmall: begin = imex_blob_gemm_small; end = imex_blob_gemm_small_end; break;
  case Module::GemmUnaligned: begin = imex_blob_gemm_unaligned; end = imex_blob_gemm_unaligned_end; break;
  case Module::Fusion: begin = imex_blob_fusion; end = imex_blob_fusion_end; break;
  case Module::Attention: begin = imex_blob_attention; end = imex_blob_attention_end; break;
  }
  if (size)
    *size = static_cast<size_t>(end - begin);
  return begin;
}

// Which tile a GEMM should take.  What one workgroup costs was fitted to 4400 random problems (M 1 .. 8192, N 64 ..
// 11008, K 32 .. 4096, all eight operators, operands from the caches and from beyond the L2s, every tile timed on each): a
// launch takes `constant`, a workgroup `setup` (first slab) and `store` per byte of a result (storeBytes()) plus `step` per K
// step, and every further workgroup that a CU gets costs these again and `stepMore` per step -- less than the sum of the two
// where workgroups share a CU (64 x 64: counted by the fraction, the others by whole rounds of 256 workgroups).
// Nanoseconds.  The tile with the least estimate is within 0.7 % of the fastest one in the mean over those problems (1.2 %
// with constants from problems of K >= 64 alone and nothing per byte, which gave short sums too small a share of their time
// to the result: 2168 x 4064 x 312 with A^T 18.8 us on 128 x 64, 16.6 on 256 x 256; 771 x 880 x 112 4.2 / 3.5 on 64 x 64);
// examples, 256 x 256 / chosen: 256 x 256 x 256 10.5 / 3.5 us (16 x 16), 1000^3 27.5 / 7.4 (64 x 64), 16 x 1680 x 3992 67.6 /
// 9.8 (16 x 16), 2414 x 2104 x 2208 49.1 / 36.4 (256 x 128); 4096 x 4096 x 1024 36.6, against 53.3 with 128 x 128 tiles.
//
// Workgroups that fetch for others (fetch_ahead in gemm_small.h) change what a step costs: stepAhead per step, aheadMib per
// MiB of operands and `ahead` once, where it is worth more than the launch of 256 workgroups (fitted to 2100 other problems,
// operands from beyond the L2s; us without / with, from HBM: 16 x 1024 x 4096 10.9 / 6.2, 16 x 2048 x 4096 14.0 / 7.2, 16 x
// 1680 x 3992 11.8 / 7.3, 128 x 2048 x 4096 15.3 / 10.8; from the 256 MiB cache 11.3 / 7.1 for the second).  On 900 further ones
// the launches that get them, with the tiles chosen by these numbers, take 0.84 of the time without from that cache (more than
// 1.04 on 15, 1.12 at most) and 0.94 where the L2s have the operands (more than 1.1 on 29).  Not below 3.75 MiB and 1024 k, 16 x
// 16 tiles 1400, or 2 MiB and 2560 k with half of the CUs free, which the L2s may have (there 2 x 1560 x 1080 1.21, 391 x 176 x
// 1928 1.17, 141 x 544 x 2800 1.08; 5 x 1720 x 1184 1.18, from the cache 1.11), nor above 32 MiB, which HBM's rate bounds (32 ..
// 48 MiB: 1.01; 128 x 64 tiles 16 MiB: B^T 3409 x 296 x 3776 1.21), with fewer than 96 helpers (176 .. 192 tiles: up to 1.5) or for
// 128 x 128 tiles and larger, which their own steps bound (above 16 MiB 1.03 .. 1.04).  An XCD's share of the operands beyond
// its 4 MiB L2 is gone before it is read: from 6 MiB on there are none (1560 x 168 x 9680 1.06), and they draw a problem to
// other tiles below 4 MiB only (above, 12 of 12 that went from 16 x 64 to 32 x 64 1.03 .. 1.18, 640 x 600 x 12064 to 64 x 64
// 1.32; below 0.87 in the mean), and only where that holds from the L2s too: from 3.75 MiB of all operands on (405 x 144 x 2920
// 1.09), not to 16 x 64 (from 16 x 32 1.03 of the time in the mean, 151 x 576 x 3456 1.21) and not to 16 x 32 with B^T (48 x 1000
// x 2064 1.12).
struct GemmTile {
  const char *suffix;
  int tileM, tileN, stepK, constant, setup, store, step, stepMore;
  bool shared;
  int stepAhead, aheadMib, ahead; // (0: chosen as without)
};
constexpr GemmTile kGemmTiles[] = {{"", 256, 256, 32, 3705, 5101, 691, 581, 810, false, 0, 0, 0},
                                   {"_t256x128", 256, 128, 64, 1238, 5315, 773, 717, 956, false, 0, 0, 0},
                                   {"_t128", 128, 128, 64, 1068, 3318, 313, 494, 454, false, 0, 0, 0},
                                   {"_t128x64", 128, 64, 64, 558, 2586, 125, 258, 391, false, 0, 0, 0},
                                   {"_t128x64s", 128, 64, 64, 1616, 1283, 100, 399, 311, false, 0, 0, 0},
                                   {"_t64", 64, 64, 64, 1621, 1410, 100, 259, 332, true, 181, 23, -171},
                                   {"_t32", 32, 64, 128, 814, 1512, 50, 375, 339, false, 225, 52, 966},
                                   {"_t16", 16, 64, 256, 837, 2121, 25, 574, 722, false, 0, 0, 0},
                                   {"_t16x32", 16, 32, 256, 1799, 466, 37, 489, 397, false, 196, 70, 889},
                                   {"_t16x16", 16, 16, 256, 2031, 385, 25, 379, 282, false, 146, 94, 761}};

double operandMib(int64_t M, int64_t N, int64_t K) { return 2.0 * double(K) * (double(M) + double(N)) / (1 << 20); }

// MiB that the tiles of one XCD, an eighth of them in bands of four tile rows (small_tile_origin), read.
double operandMibOfXcd(const GemmTile &t, int64_t M, int64_t N, int64_t K) {
  const double tilesM = double(ceilDiv(M, t.tileM)), tilesN = double(ceilDiv(N, t.tileN)), tiles = std::ceil(tilesM * tilesN / 8.0);
  const double rows = std::min(4.0, tilesM), cols = std::min(tilesN, std::ceil(tiles / rows));
  const double bands = std::ceil(tiles / (rows * tilesN));
  return operandMib(std::min(M, int64_t(bands * rows) * t.tileM), std::min(N, int64_t(cols) * t.tileN), K);
}

// Whether workgroups without a tile are launched to fetch what the others read.
bool fetchesAhead(const GemmTile &t, int64_t M, int64_t N, int64_t K) {
  const double mib = operandMib(M, N, K), tiles = double(ceilDiv(M, t.tileM)) * double(ceilDiv(N, t.tileN));
  const int64_t from = t.tileM * t.tileN <= 16 * 16 ? 1400 : 1024;
  return ((K >= from && mib >= 3.75 && tiles <= 160) || (K >= 2560 && mib >= 2.0 && tiles <= 128)) &&
         t.tileM * t.tileN <= 128 * 64 && mib <= (t.tileM == 128 ? 16.0 : 32.0) && operandMibOfXcd(t, M, N, K) < 6.0;
}
// Whether they count in the choice of a tile.
bool drawnByFetching(const GemmTile &t, bool transB, int64_t M, int64_t N, int64_t K) {
  return t.stepAhead && fetchesAhead(t, M, N, K) && operandMib(M, N, K) >= 3.75 && operandMibOfXcd(t, M, N, K) < 4.0 &&
         !(transB && t.tileM * t.tileN == 16 * 32);
}

// Bytes moved for an element of the result: read and written again, or written; the 16-bit result of bias and SiLU counts
// double for its arithmetic.
int storeBytes(const Entry *e) {
  return strstr(e->name, "_acc") ? 8 : strstr(e->name, "f16_f16_f16") ? 2 : 4;
}

// The same for rows that are not 16-byte aligned, fitted to 2600 random problems of the seven operators without a bias (M 1 ..
// 4096, N 64 .. 4096, K 64 .. 2048, N and K odd); over 420 others the choice is 0.5 % from the fastest tile in the mean, and
// 20 % faster than the better one of 128 x 128 and 64 x 64.  The operator itself is a loop on the vector ALUs there, 4.4 us
// for every sixteen k: 1001 x 1003 x 999 276 us, 9.5 here (64 x 64); 131 x 133 x 999 8.8 with 64 x 64, 4.7 with 16 x 16.
constexpr GemmTile kUnalignedTiles[] = {{"_u128", 128, 128, 64, -568, 4171, 645, 731, 589, false, 0, 0, 0},
                                        {"_u64", 64, 64, 64, 2399, 413, 233, 350, 306, false, 0, 0, 0},
                                        {"_u32", 32, 64, 128, 2564, 464, 141, 492, 456, false, 0, 0, 0},
                                        {"_u16x32", 16, 32, 256, 2842, 0, 105, 591, 611, false, 0, 0, 0},
                                        {"_u16x16", 16, 16, 256, 2485, 50, 96, 467, 471, false, 0, 0, 0}};
// Products that are small and whose sums are short stay with that loop, which adds in the sequential order bit for bit; small
// ones of longer sums take 0.70 of the time of 64 x 64 tiles in the mean (1350 of fewer than 2^21 products, at most 0.97).
constexpr double kUnalignedFrom = double(1 << 23);
constexpr int64_t kUnalignedFromK = 192;
// From 129 k to there the second step of 128 or the first of 256 k is part empty: narrow tiles where they should gain 6 %.  Of
// 260 such problems 31 were more than 2 % slower with less (A^T 798 x 549 x 185 1.09 of the time with 64 x 64, B^T 1233 x 137
// x 189 1.07), none is so (0.92 in the mean); not those of bias and SiLU, whose results weigh more in the wide ones.
constexpr double kUnalignedNarrowGain = 0.94;

// The tile that the name of a GemmSmall or GemmUnaligned entry ends in.
const GemmTile &tileOf(const Entry *e) {
  const char *suffix = strrchr(e->name, '_');
  for (const GemmTile &t : kUnalignedTiles)
    if (strcmp(t.suffix, suffix) == 0)
      return t;
  return *std::find_if(std::begin(kGemmTiles), std::end(kGemmTiles), [&](const GemmTile &t) { return strcmp(t.suffix, suffix) == 0; });
}

const char *gemmVariant(const Entry *e, int64_t M, int64_t N, int64_t K) {
  const bool transA = e->shape == Shape::GemmTA, transB = e->shape == Shape::GemmTB;
  const GemmTile *first = std::begin(kGemmTiles), *last = std::end(kGemmTiles);
  if (!mfmaTakes(transA, transB, M, N, K)) {
    if (!unalignedTakes(transA, transB, M, N, K) ||
        (K < kUnalignedFromK && double(M) * double(N) * double(K) < kUnalignedFrom))
      return e->name;
    first = std::begin(kUnalignedTiles), last = std::end(kUnalignedTiles);
  }
  const bool partEmpty = first == std::begin(kUnalignedTiles) && K > 128 && K < kUnalignedFromK && !strstr(e->name, "silu");
  const GemmTile *best = nullptr;
  double least = 0.0;
  for (; first != last; ++first) {
    const GemmTile &t = *first;
    const double tiles = double(ceilDiv(M, t.tileM)) * double(ceilDiv(N, t.tileN)), steps = double(ceilDiv(K, t.stepK));
    const double load = t.shared ? std::max(1.0, tiles / 256.0) : std::ceil(tiles / 256.0);
    const double once = t.constant + load * (t.setup + t.store * storeBytes(e));
    double ns = once + steps * (t.step + (load - 1.0) * t.stepMore);
    if (drawnByFetching(t, transB, M, N, K))
      ns = std::min(ns, once + steps * t.stepAhead + operandMib(M, N, K) * t.aheadMib + t.ahead);
    if (partEmpty && t.tileM * t.tileN < 64 * 64)
      ns /= kUnalignedNarrowGain;
    if (!best || ns < least) {
      best = &t;
      least = ns;
    }
  }
  if (!*best->suffix)
    return e->name;
  char name[96];
  snprintf(name, sizeof name, "%s%s", e->name, best->suffix);
  const Entry *variant = find(name);
  return variant ? variant->name : e->name;
}

// Which form of the outer-dimension sum a problem should take, from two estimates in microseconds fitted to 1000
// timed problems (1 .. 20000 slices of 1 .. 8 Mi outputs, all types, whole vectors and not, from HBM and not; the choice is
// within 0.2 % of the faster of tall and deep in the mean, at worst 12 %; over 350 others within 0.6 % of the fastest form).
//   plain  whole vectors and slices of 5 MiB (16-bit: 8 MiB) and more, for up to four slices 4 MiB (f32 4 x 1359872 6.8,
//          deep 8.5; f16 2 x 2999824 8.1, 8.7; f32 7 x 2071552 15.4, 13.5; 12 x 1051744 11.7, 10.4; 6 x 1500000 16.4, 16.0;
//          f16 15 x 2283888 18.3, 12.6);
//   tall   a launch, a slice's share of the chain, and what a CU pays for further workgroups; 4.9 TB/s at most;
//   deep   a slice costs its share of sixteen slices' latency, which its bytes hide little of; 8.0 (5.1) TB/s at most.
// 8192 x 4096 f32: plain 980, tall 34, deep 540 us; 62 x 32296: tall 3.7, deep 7.0; 568 x 197848: 102, 66.  With three tiles
// in flight tall is up to 0.87 of its estimate, where deep is far off: of 150 problems of 200 .. 3000 segments the choice is the
// faster one of the two on all, but for what two runs differ (0.4 % in the mean).  Below 64
// outputs (1 .. 15, 8 .. 10^5 slices) tall is never slower than deep by more than 0.1 us: 64 x 4 both 3.3, 256 x 4 3.3 / 8.5.
const char *reduceVariant(const Entry *e, int64_t outer, int64_t inner) {
  const bool f32 = e->shape == Shape::ReduceOuter;
  const int64_t perVec = f32 ? 4 : 8, slice = inner * (f32 ? 4 : 2);
  const bool vec = inner % perVec == 0;
  if (outer == 0 || inner == 0 || (vec && slice >= (outer <= 4 ? int64_t(4) << 20 : f32 ? int64_t(5) << 20 : int64_t(8) << 20)))
    return e->name;
  const double bytes = double(outer) * double(slice);
  const size_t segments = ceilDiv(slice, 32);
  const int width = chainWidth(segments);
  const double more = std::max(0.0, double(ceilDiv(segments, width)) / 256.0 - 1.0);
  const double step = width == 1 ? 0.00252 : width == 2 ? 0.00363 : f32 ? 0.00112 : 0.00458;
  const double tall = 3.28 + std::max(0.744 * more + double(outer) * step * (1.0 + (f32 ? 1.77 : 1.17) * more), bytes / 4.91e6);
  const double wait = double(outer) * (vec ? 0.0375 : f32 ? 0.0236 : 0.0139), move = bytes / (vec ? 8.02e6 : 5.13e6);
  const double deep = 3.26 + std::max(wait, move) + (vec ? 0.88 : 0.098) * std::min(wait, move);
  const bool chains = bytes >= 8.0 && slice < int64_t(1) << 26 && outer < int64_t(1) << 31; // chains_take in column_chain.h
  char name[96];
  snprintf(name, sizeof name, "%s%s", e->name, chains && tall < deep ? "_tall" : "_deep");
  return find(name)->name;
}

// The operator's own launch is one for wavefronts (four per workgroup) or workgroups of 256 that have a row each: right
// for rows of 65 .. 128 whole 16-byte pieces -- the f16 ones that wavefronts walk; f32 and bf16 up to 8192 rows, 16384 from
// 96 pieces on (f32 16384 x 384: 9.0 us, 10.8 with shared wavefronts; 30000 x 512: 23.9 / 22.6) -- and for rows that fit
// nobody's registers (more than 4096 pieces).  Every other row goes to as many lanes as suit its length: 65536 x 32 bf16
// 20.5 us with a wavefront per row, 3.2 so; 2500 x 8191 55.3 with 256 lanes of the streaming form, 18.8.
const char *softmaxVariant(const Entry *e, int64_t rows, int64_t cols) {
  const int64_t perVec = e->shape == Shape::SoftmaxRows16 ? 8 : 4, pieces = (cols + perVec - 1) / perVec;
  const bool f16 = strcmp(e->name, "imex_softmax_f16") == 0;
  const bool own = cols % perVec == 0 && pieces <= 128 && pieces > 64 && (f16 || rows <= (pieces >= 96 ? 16384 : 8192));
  if (rows == 0 || cols == 0 || own || pieces > 4096)
    return e->name;
  char name[96];
  snprintf(name, sizeof name, "%s_shared", e->name);
  return find(name)->name;
}

// Transposes whose rows are no whole 16-byte vectors on one side or the other go to the kernels with tiles for these,
// from one vector each way on (16-bit 1203 x 1777: 29.4 -> 4.1 us; 32-bit 333 x 17 x 501: 17.0 -> 5.8).  So do those whose
// result has rows that are no whole 64 bytes: there neighbouring segments share lines, which those kernels' order of tiles
// brings together in one L2 (16-bit 6000 x 6000 42.0 -> 34.1 us, 4104 x 4096 18.4 -> 16.1, 11472 x 3312 43.1 -> 37.2, 32-bit
// 3000 x 2000 14.8 -> 11.7; 98 of 260 timed problems, 0.82 of their time in the mean).  With whole halves of lines it is as
// often the other way (16-bit 13280 x 2048 22.5, 24.9, 32-bit 6000 x 6000 62.8, 62.4), and so it is with a few columns, which
// tiles of 64 fit badly (16-bit 63352 x 280 18.3, 22.0): tall 16-bit ones of 5.5 .. 15 MB, of 500 timed problems the only ones
// that were more than 4 % slower (16336 x 200 1.14 of the time, 20568 x 264 6.9, 7.3, 20360 x 232 6.0, 6.4; 16336 x 256 0.74).
const char *transposeVariant(const Entry *e, const int64_t *dims) {
  const int64_t perVec = e->shape == Shape::Transpose2D32 || e->shape == Shape::Transpose3D32 ? 4 : 8;
  const int64_t rows = dims[0], cols = dims[e->ndims - 1], planes = e->ndims == 3 ? dims[1] : 1;
  const bool halves = uint64_t(rows) * uint64_t(planes) % uint64_t(4 * perVec) == 0; // of cache lines, in the result
  const double bytes = 16.0 / double(perVec) * double(rows) * double(cols);
  const bool tall = rows / 128 > cols ||
                    (perVec == 8 && planes == 1 && rows / 12 > cols && cols % 64 != 0 && bytes >= 5.5e6 && bytes <= 15e6);
  if (rows < perVec || cols < perVec || (rows % perVec == 0 && cols % perVec == 0 && (halves || tall)))
    return e->name;
  char name[96];
  snprintf(name, sizeof name, "%s_any", e->name);
  return find(name)->name;
}

// The operator's own launch takes the most queries per workgroup that give every CU a workgroup.  That leaves CUs idle
// where 64 queries are too many for it, and runs a second, partly empty round where the next larger tiling would do in
// one.  A tiling costs its rounds of 256 workgroups, in microseconds at 4096 keys: 32 queries wherever they fit one round
// (1 x 4096 27.6 -> 14.8 us, 8 x 1024 10.0 -> 7.6, 16 x 512 7.1 -> 6.0, 4 x 64 6.0 -> 4.2; at 264 workgroups 24 x 333
// 7.6, 7.7, at 288 48 x 192 6.2, 7.1), 128 where 64 take two (12 x 1500 27.0 -> 20.1, 6 x 4096 53.1 -> 42.5, 64 x 320 14.2
// -> 9.2, 200 x 128 11.6 -> 7.0), 256 where 128 take two (12 x 4096 85.1 -> 68.3, 100 x 333 19.1 -> 14.1).  Of the two
// forms with 64 queries the one whose wavefronts have keys of their own from 768 keys on (4 x 4096 30.8 -> 27.6, 16 x 1000
// 11.6 -> 11.4) and where the last 256 keys are no more than half there (16 x 600 9.1 -> 8.6, 32 x 320 7.7 -> 6.8; it merges
// more for its few tiles elsewhere: 24 x 512 7.5, 7.8, 40 x 256 6.0, 6.5).
// Problems that fill more than one round with 256 queries stay.
struct Tiling {
  const char *suffix;
  int64_t queries;
  double cost;
};
constexpr Tiling kTilings[] = {{"_q32", 32, 15.5}, {"_q64", 64, 26.0}, {"_q128", 128, 43.0}, {"_q256", 256, 68.0}};

const char *attentionVariant(const Entry *e, int64_t ZH, int64_t N) {
  auto workgroups = [&](int64_t queries) { return (N + queries - 1) / queries * ZH; };
  if (N <= 0 || N >= (int64_t(1) << 24) || ZH == 0 || ZH > 256 || workgroups(256) > 256)
    return e->name;
  int64_t own = 256; // as imexHipKernelLaunchShape
  while (own > 64 && workgroups(own) < 256)
    own /= 2;
  const Tiling *best = nullptr;
  double least = 0.0;
  for (const Tiling &t : kTilings) {
    const double cost = double((workgroups(t.queries) + 255) / 256) * t.cost;
    if (!best || cost < least) {
      best = &t;
      least = cost;
    }
  }
  const bool ownKeys = own == 64 && (N >= 768 || (N > 256 && N % 256 >= 1 && N % 256 <= 128));
  if (best->queries == own && !ownKeys)
    return e->name;
  char name[96];
  snprintf(name, sizeof name, "%s%s", e->name, best->suffix);
  return find(name)->name;
}

// The fused chain with column sums: column chains, but for a few rows, where the operator's own launch has a shorter way to
// its first and only additions.  By 300 timed problems (2 .. 12000 rows of 16 .. 300000 columns): below 2048 columns
// from 128 rows on (f16 124 x 81: own 4.1 us, chains 4.4; f32 827 x 1592 23.2 / 6.2), from 256 on for 16-bit rows of less
// than a segment (f16 128 x 1 3.9 / 4.8, 300 x 12 5.4 / 4.1, 9124 x 8 84 / 34; f32 100000 x 4 857 / 267); rows that take workgroups of 128-byte
// segments more than one round from 72 (f32) or 24 rows on (f32 33 x 25520 9.9 / 10.8; f16 20 x 37008 8.7 / 9.5; bf16 5550 x
// 5932 449 / 42; f32 72 x 1074784 494 / 299); rows in between always (f32 2 x 7024 6.6 / 3.8).
const char *inputFusionVariant(const Entry *e, int64_t rows, int64_t cols) {
  const bool f32 = e->shape == Shape::ColumnThreads;
  const int64_t bytes = cols * (f32 ? 4 : 2);
  if (rows == 0 || rows >= int64_t(1) << 31 || bytes >= int64_t(1) << 26 || // chains_take in column_chain.h
      (cols < 2048 ? rows < (f32 || bytes >= 32 ? 128 : 256) : bytes > 256 * 128 && rows < (f32 ? 72 : 24)))
    return e->name;
  char name[96];
  snprintf(name, sizeof name, "%s_tall", e->name);
  return find(name)->name;
}

extern "C" const char *imexHipKernelVariant(const char *kernel, const int64_t *dims, int ndims) {
  const Entry *e = find(kernel);
  if (!e || ndims != e->ndims || (ndims > 0 && !dims))
    return e ? e->name : nullptr;
  for (int i = 0; i < ndims; ++i)
    if (dims[i] < 0 || dims[i] > (int64_t(1) << 40))
      return e->name;
  switch (e->shape) {
  case Shape::Gemm:
  case Shape::GemmTA:
  case Shape::GemmTB:
    return gemmVariant(e, dims[0], dims[1], dims[2]);
  case Shape::ReduceOuter:
  case Shape::ReduceOuter16:
    return reduceVariant(e, dims[0], dims[1]);
  case Shape::SoftmaxRows32:
  case Shape::SoftmaxRows16:
    return softmaxVariant(e, dims[0], dims[1]);
  case Shape::RowSum: // rows that fit a wavefront's four pieces per lane (131072 x 32: 20.9 -> 4.1 us; 1000 x 1000: 3.6 -> 3.3)
    if (dims[1] < 4 || dims[1] > 1024)
      return e->name;
    return strcmp(e->name, "imex_rowsum_f32") == 0 ? "imex_rowsum_f32_short" : "imex_rowmean_f32_short";
  case Shape::Transpose2D32:
  case Shape::Transpose2D16:
  case Shape::Transpose3D32:
  case Shape::Transpose3D16:
    return transposeVariant(e, dims);
  case Shape::ColumnThreads:
  case Shape::ColumnThreads16:
    return inputFusionVariant(e, dims[0], dims[1]);
  case Shape::Attention:
    return attentionVariant(e, dims[0], dims[1]);
  default:
    return e->name;
  }
}

extern "C" size_t imexHipStreamKWorkspaceBytes(size_t workgroups) { return 4096 + (size_t(256) * 256 * 4) * workgroups; }

extern "C" int imexHipKernelLaunchShape(const char *kernel, const int64_t *dims, int ndims, size_t grid[3],
                                        size_t block[3], size_t *sharedMemBytes) {
  const Entry *e = find(kernel);
  if (!e)
    return -1;
  if (ndims != e->ndims || (ndims > 0 && !dims))
    return -2;
  for (int i = 0; i < ndims; ++i)
    if (dims[i] < 0 || dims[i] > (int64_t(1) << 40))
      return -2;
  grid[0] = grid[1] = grid[2] = 1;
  block[0] = 256;
  block[1] = block[2] = 1;
  if (sharedMemBytes)
    *sharedMemBytes = 0;
  switch (e->shape) {
  case Shape::Eltwise32: // 256 lanes x 4 vectors x 4 elements
    grid[0] = ceilDiv(dims[0], 4096);
    break;
  case Shape::Eltwise16: // 256 lanes x 4 vectors x 8 elements
    grid[0] = ceilDiv(dims[0], 8192);
    break;
  case Shape::Fusion32: // SiLU and the fused chains: as Eltwise32 / 16, but one vector per lane below 4 Mi elements
    grid[0] = ceilDiv(dims[0], dims[0] < (int64_t(1) << 22) ? 1024 : 4096);
    break;
  case Shape::Fusion16:
    grid[0] = ceilDiv(dims[0], dims[0] < (int64_t(1) << 22) ? 2048 : 8192);
    break;
  case Shape::SoftmaxRows32:
  case Shape::SoftmaxRows16: {
    // Any grid is correct, the kernels stride over the rows.  f16 rows of 65 .. 128 whole 16-byte pieces: a
    // wavefront walks its rows with the next row's loads in flight, and 2048 workgroups give every wavefront
    // slot of the chip (256 CUs x 4 SIMDs x 8) one wavefront.
    const int64_t regCols = e->shape == Shape::SoftmaxRows16 ? 1024 : 512;
    const bool f16 = std::strcmp(e->name, "imex_softmax_f16") == 0;
    if (dims[1] > regCols)
      grid[0] = static_cast<size_t>(dims[0] < 1048560 ? dims[0] : 1048560);
    else if (f16)
      grid[0] = std::min<size_t>(ceilDiv(dims[0], 4), 2048);
    else
      grid[0] = ceilDiv(dims[0], dims[0] >= 16384 ? 8 : 4);
    if (dims[1] == 0)
      grid[0] = 0;
    break;
  }
  case Shape::SoftmaxShared32:
  case Shape::SoftmaxShared16: { // one row for every group of lanes: the kernels' own rule (softmax_kernel in softmax.hip)
    const int64_t rows = dims[0], cols = dims[1], perVec = e->shape == Shape::SoftmaxShared16 ? 8 : 4;
    const int64_t pieces = (cols + perVec - 1) / perVec;
    if (cols == 0)
      grid[0] = 0;
    else if (cols < perVec)
      grid[0] = gridFor(ceilDiv(rows, 256), 256);
    else if (pieces <= 256 && (pieces <= 64 || rows >= 1024)) {
      int64_t lanes = 4;
      while (lanes < 64 && (4 * lanes < pieces || (lanes < pieces && rows * lanes <= 2048 * 64) ||
                            (cols % perVec == 0 && pieces > 48 && pieces != 64 && 2 * lanes < pieces)))
        lanes *= 2;
      grid[0] = gridFor(ceilDiv(rows, 256 / lanes), 256);
    } else {
      grid[0] = static_cast<size_t>(std::min<int64_t>(rows, 1048560));
      const int64_t most = pieces <= 1024 ? 256 : pieces <= 2048 ? 512 : 1024, per = (pieces + most - 1) / most;
      block[0] = pieces > 4096 ? 256 : ceilDiv((pieces + per - 1) / per, 64) * 64;
    }
    break;
  }
  case Shape::RowSum: // workgroup per row above 2048 columns, else wavefront per row
    grid[0] = dims[1] > 2048 ? static_cast<size_t>(dims[0]) : ceilDiv(dims[0], 4);
    break;
  case Shape::RowSumShort: { // up to four 16-byte pieces of a row per lane
    int64_t lanes = 4;
    while (lanes < 64 && 16 * lanes < dims[1])
      lanes *= 2;
    grid[0] = gridFor(dims[1] >= 4 && dims[1] <= 1024 ? ceilDiv(dims[0], 256 / lanes)
                                                      : dims[1] > 2048 ? static_cast<size_t>(dims[0]) : ceilDiv(dims[0], 4),
                      256);
    break;
  }
  case Shape::ReduceOuter:
  case Shape::ReduceOuter16: { // 256 lanes x v vectors of 4 (8) outputs, v = 8, 4, 2, 1: the widest that leaves 512 workgroups
    const int64_t inner = dims[1], perVec = e->shape == Shape::ReduceOuter ? 1024 : 2048;
    const int64_t v = inner >= 512 * 8 * perVec ? 8 : inner >= 512 * 4 * perVec ? 4 : inner >= 512 * 2 * perVec ? 2 : 1;
    grid[0] = ceilDiv(inner, perVec * v);
    break;
  }
  case Shape::ReduceDeep32:
  case Shape::ReduceDeep16: { // a lane per 16-byte vector, or per output
    const int64_t perVec = e->shape == Shape::ReduceDeep32 ? 4 : 8;
    grid[0] = gridFor(ceilDiv(dims[1], dims[1] % perVec == 0 ? 256 * perVec : 256), 256);
    break;
  }
  case Shape::Transpose2D32:
  case Shape::Transpose2D16:
  case Shape::Transpose3D32:
  case Shape::Transpose3D16: {
    // One workgroup per R x C tile.  Problems of 2^24 elements and more use the
    // large tiles (512-byte row segments): 128 x 128 for 32-bit, 256 x 256 for
    // 16-bit elements; smaller ones 64 x 64 / 128 x 128.  The kernels apply the same
    // rule, and stride over the tiles if the grid is any different.
    const bool is32 = e->shape == Shape::Transpose2D32 || e->shape == Shape::Transpose3D32;
    const bool is3d = e->shape == Shape::Transpose3D32 || e->shape == Shape::Transpose3D16;
    const int64_t rows = dims[0], cols = is3d ? dims[2] : dims[1], planes = is3d ? dims[1] : 1;
    const bool big = rows * cols * planes >= (int64_t(1) << 24);
    const int64_t tileR = is32 ? (big ? 128 : 64) : (big ? 256 : 128);
    const int64_t tileC = is32 ? (big ? 128 : 64) : (big ? 256 : 128);
    grid[0] = ceilDiv(cols, tileC);
    grid[1] = ceilDiv(rows, tileR);
    grid[2] = static_cast<size_t>(planes);
    if (grid[1] > 65535) // the kernels stride over the tiles a smaller grid leaves out
      grid[1] = 65535;
    if (grid[2] > 65535)
      grid[2] = 65535;
    // 32-bit problems made of whole 128 x 128 tiles: 512 workgroups (two per CU), each of which walks its
    // share of the tiles with the next tile's loads in flight while the current one is written
    if (is32 && big && rows % 128 == 0 && cols % 128 == 0) {
      const size_t budget = 512;
      if (grid[0] >= budget) {
        grid[0] = budget;
        grid[1] = grid[2] = 1;
      } else {
        grid[1] = std::min(grid[1], std::max<size_t>(1, budget / grid[0]));
        grid[2] = std::min(grid[2], std::max<size_t>(1, budget / (grid[0] * grid[1])));
      }
    }
    break;
  }
  case Shape::TransposeAny32:
  case Shape::TransposeAny16: { // a workgroup per tile of 512 bytes of output rows x 128 bytes of input rows, for each XCD the same number
    const int64_t bytes = e->shape == Shape::TransposeAny32 ? 4 : 2, planes = e->ndims == 3 ? dims[1] : 1;
    const size_t perPlane = ceilDiv(dims[0], 512 / bytes) * ceilDiv(dims[e->ndims - 1], 128 / bytes);
    const size_t most = size_t(1) << 24; // (the product of two large counts would overflow)
    grid[0] = gridFor(planes == 0 ? 0 : perPlane >= most ? most : (perPlane * size_t(planes) + 7) / 8 * 8, 256);
    break;
  }
  case Shape::Attention: {
    // dims = {ZH, N_CTX}.  A workgroup takes 64, 128 or 256 queries of one (batch, head); the kernel reads
    // the choice off the grid and the block.  More queries per workgroup mean less K / V traffic, so: the
    // largest of the three that still gives every one of the 256 CUs a workgroup.  256 queries run as
    // sixteen wavefronts (8 query blocks x 2 key groups), the others as eight.  N_CTX need not divide.
    const int64_t ZH = dims[0], N = dims[1];
    block[0] = 512;
    if (N > 0 && N < (int64_t(1) << 24) && ZH > 0 && ZH <= 65535) {
      int64_t queries = 256;
      while (queries > 64 && ((N + queries - 1) / queries) * ZH < 256)
        queries /= 2;
      grid[0] = ceilDiv(N, queries);
      grid[1] = static_cast<size_t>(ZH);
      if (queries == 256)
        block[0] = 1024;
    } else {
      grid[0] = ceilDiv(ZH * N, 512); // one lane per query
    }
    break;
  }
  case Shape::AttentionTiling: { // the tiling that the name ends in
    const int64_t ZH = dims[0], N = dims[1];
    const int64_t queries = std::find_if(std::begin(kTilings), std::end(kTilings), [&](const Tiling &t) {
                              return strcmp(t.suffix, strrchr(e->name, '_')) == 0;
                            })->queries;
    block[0] = queries == 256 ? 1024 : 512;
    if (N > 0 && N < (int64_t(1) << 24) && ZH > 0 && ZH <= 65535) {
      grid[0] = ceilDiv(N, queries);
      grid[1] = static_cast<size_t>(ZH);
    } else {
      grid[0] = gridFor(ceilDiv(ZH * N, 512), block[0]); // one lane per query
    }
    break;
  }
  case Shape::ColumnThreads:
  case Shape::ColumnThreads16: {
    const int64_t rows = dims[0], cols = dims[1];
    // From 2048 rows and 128 row segments of 128 bytes on: column chains with 576 lanes per segment's
    // columns (32 f32 or 64 16-bit ones).  The kernel applies the same rule.
    const int64_t segment_cols = e->shape == Shape::ColumnThreads ? 32 : 64;
    if (rows >= 2048 && cols >= segment_cols * 128) {
      block[0] = 576;
      grid[0] = ceilDiv(cols, segment_cols);
      break;
    }
    // Fewer than 4096 columns (the reference's 512 x 1024): 256 workers and the adder wavefront = 320 lanes per
    // four columns.
    if (cols < 8 * 512) {
      block[0] = 320;
      grid[0] = ceilDiv(cols, 4);
      break;
    }
    // otherwise a workgroup per block of 64 .. 8 columns: the widest that leaves 512 workgroups
    const int64_t block_cols = cols >= 64 * 512 ? 64 : cols >= 32 * 512 ? 32 : cols >= 16 * 512 ? 16 : cols >= 8 * 512 ? 8 : 4;
    grid[0] = ceilDiv(cols, block_cols);
    break;
  }
  case Shape::ReduceTall32:
  case Shape::ReduceTall16:
  case Shape::ColumnChains:
  case Shape::ColumnChains16: { // a workgroup per segment of 16 .. 128 bytes: the kernels' own rule (chain_lanes in column_chain.h)
    const bool f32 = e->shape == Shape::ReduceTall32 || e->shape == Shape::ColumnChains;
    const bool reduce = e->shape == Shape::ReduceTall32 || e->shape == Shape::ReduceTall16;
    const int64_t perSegment = f32 ? 8 : 16;
    const size_t segments = ceilDiv(dims[1], perSegment);
    const int64_t times = chainWidth(segments);
    block[0] = (times == 4 && segments <= 4 * 256) || (times == 2 && !reduce) ? 576 : 320; // eight workers or four
    // (the fused chain, half_segments in fusion.hip)
    const bool half = !reduce && dims[1] >= perSegment && dims[1] <= 128 * perSegment && dims[0] >= (f32 ? 4096 : 2048);
    grid[0] = gridFor(ceilDiv(dims[1], half ? perSegment / 2 : times * perSegment), block[0]);
    break;
  }
  case Shape::Gemm:
  case Shape::GemmTA:
  case Shape::GemmTB: {
    // 512 lanes: eight wavefronts per 256 x 256 tile of C, edge tiles included.  The MFMA path
    // needs 16-byte aligned rows in memory, i.e. K % 8 == 0, N % 8 == 0 where B is [K,N] and
    // M % 8 == 0 where A is [K,M]; everything else runs 128 x 128 tiles on the vector ALUs.
    const int64_t M = dims[0], N = dims[1], K = dims[2];
    const bool tileable = mfmaTakes(e->shape == Shape::GemmTA, e->shape == Shape::GemmTB, M, N, K);
    block[0] = 512;
    grid[0] = tileable ? ceilDiv(M, 256) * ceilDiv(N, 256) : ceilDiv(M, 128) * ceilDiv(N, 128);
    break;
  }
  case Shape::GemmSmall: { // one workgroup per tile of the size that the name ends in
    const int64_t M = dims[0], N = dims[1], K = dims[2];
    const GemmTile &tile = tileOf(e);
    block[0] = 512;
    if (mfmaTakes(strstr(e->name, "_ta_") != nullptr, strstr(e->name, "_tb_") != nullptr, M, N, K)) {
      const size_t tiles = ceilDiv(M, tile.tileM) * ceilDiv(N, tile.tileN);
      grid[0] = fetchesAhead(tile, M, N, K) ? 256 : gridFor(tiles, 512);
    } else {
      grid[0] = gridFor(ceilDiv(M, 128) * ceilDiv(N, 128), 512);
    }
    break;
  }
  case Shape::GemmUnaligned: {
    const int64_t M = dims[0], N = dims[1], K = dims[2];
    const GemmTile &tile = tileOf(e);
    block[0] = 512;
    grid[0] = gridFor(unalignedTakes(strstr(e->name, "_ta_") != nullptr, strstr(e->name, "_tb_") != nullptr, M, N, K)
                          ? ceilDiv(M, tile.tileM) * ceilDiv(N, tile.tileN)
                          : ceilDiv(M, 128) * ceilDiv(N, 128),
                      512);
    break;
  }
  case Shape::GemmStreamK: {
    // One workgroup per CU at most (256 on this part): the kernel's finishing workgroups wait for partial sums
    // of others, which have to be resident.  A problem with fewer tiles than CUs still gets more workgroups
    // than tiles -- its K loops are split -- as long as each one has 1024 k or more to do.
    const int64_t M = dims[0], N = dims[1], K = dims[2];
    const bool streams = M > 0 && N > 0 && K > 0 && K % 64 == 0 && N % 8 == 0;
    const size_t tiles = ceilDiv(M, 256) * ceilDiv(N, 256);
    const size_t shares = K >= 2048 ? static_cast<size_t>(K / 1024) : 1;
    block[0] = 512;
    grid[0] = !streams ? (K % 8 == 0 && N % 8 == 0 ? tiles : ceilDiv(M, 128) * ceilDiv(N, 128))
                       : std::min<size_t>(imexHipStreamKMaxWorkgroups, tiles * shares);
    break;
  }
  case Shape::GemmFixed4k: // the reference's own launch: blocks (16,16,1), threads (512,1,1)
    block[0] = 512;
    grid[0] = 16;
    grid[1] = 16;
    break;
  }
  // A grid component of 0 means there is nothing to launch.
  return 0;
}

// Tile code of the MFMA GEMM for problems that leave most of the chip idle under the 256 x 256 tiles of
// gemm_tile.h: C[M,N] = A[M,K] . B[K,N], A and B f16 or bf16 (also A stored [K,M], B stored [N,K]), f32 sums.
// Entry points: gemm_small.hip.  The reference kernels these stand for are those of gemm_tile.h.
//
// What bounds such a problem is not arithmetic but a chain: a workgroup walks its K loop alone, and with few
// workgroups the chip waits for that walk.  So: smaller tiles (more workgroups), and inside a workgroup the
// eight wavefronts share the tile's k as well as its rows and columns -- KG key groups each multiply their own
// 32-wide slices of every K step -- which makes the walk shorter without a workspace or a second launch.
//
//   workgroup   512 lanes = WMC x WNC x KG wavefronts on a TM x TN tile; a K step is BK = 32 KG k;
//   operands    global -> LDS directly (16 bytes per lane), a ring of S stages, S - 1 of them in flight; the
//               images and their swizzles follow the LDS service rules of gemm_tile.h: k-contiguous operands as
//               64-k slabs of 128-byte rows, group c of row r at c ^ ((r >> 1) & 7); strided ones as k rows of TM
//               (TN) elements whose 32-byte pairs trade places with the k row (pair_swizzle);
//   registers   the fragments of step t + 1 are read while step t is multiplied (one barrier per step);
//   result      the product is taken transposed (a lane holds four consecutive columns of a row); the KG partial
//               tiles meet in LDS (pitch TN + 4 floats: no bank conflicts on either side; one after the other where
//               they do not fit side by side), are added in group order and leave as four consecutive columns per
//               lane, whole lines per row.
//   edges       rows and columns past the end go out of the descriptor's range: nothing moves for them.
//
// Steps past the end of K are fetched through a descriptor of size zero (nothing moves, LDS gets zeros).
// Operands whose rows are not 16-byte aligned take gemm_blocked, as in gemm_tile.h, or the kernels of gemm_unaligned.h.

#ifndef IMEX_HIP_GEMM_SMALL_H
#define IMEX_HIP_GEMM_SMALL_H

#include "gemm_tile.h"

namespace imexhip_gemm {

// Which 32-byte pair of a strided operand's k row `row` holds pair 0: a transpose read takes, for sixteen lanes,
// four k rows (row & 3) and, for the next sixteen, the rows eight further; all eight must lie in different banks
// (256 bytes apart repeats).  NP = pairs per row.
template <int NP> __device__ __forceinline__ int pair_swizzle(int row) {
  if constexpr (NP >= 8)
    return (row & 3) | (((row >> 3) & 1) << 2);
  else if constexpr (NP == 4) // 128-byte rows: odd and even rows are apart already
    return ((row >> 1) & 1) | (((row >> 3) & 1) << 1);
  else if constexpr (NP == 2)
    return (row >> 3) & 1;
  else
    return 0;
}

// One operand's TR x BK (rows x k) slab per step.
template <typename T, bool kStrided, int TR, int BK> struct SmallOperand {
  static constexpr int kBytes = TR * BK * 2;
  static constexpr int kCopies = kBytes / 1024 / kWaves; // 1 KiB copies per wavefront and step
  static_assert(kBytes % (1024 * kWaves) == 0, "every wavefront makes the same number of whole copies");
  const uint16_t *base;
  int range;          // bytes the descriptor covers
  int voff[kCopies];  // per-lane byte offsets at step 0
  int voffT[kCopies]; // the same for the last step, pieces at k >= K sent out of range
  int step;           // bytes per step in memory
  int dst;            // this wavefront's copies inside the image
  int rd;             // per-lane LDS address of fragment 0, slice 0 (strided: without the pair)
  int swz;            // strided: pair swizzle of this lane's k rows

  // where a wavefront whose fragments start at row w0 of the slab reads them
  __device__ __forceinline__ void setup_read(int w0, int lane) {
    if constexpr (!kStrided) {
      const int r = lane & 15;
      rd = (w0 + r) * 128 + (((lane >> 4) ^ ((r >> 1) & 7)) << 4);
      swz = 0;
    } else {
      const int t = lane & 15, row = (lane >> 4) * 8 + (t >> 2);
      rd = row * (TR * 2) + (t & 3) * 8;
      swz = pair_swizzle<TR / 16>(row) ^ (w0 / 16);
    }
  }
  __device__ __forceinline__ void setup(const uint16_t *ptr, int64_t ld, int64_t first, int w0, int64_t extent,
                                        int wave, int lane, int kRem) {
    dst = wave * kCopies * 1024;
    setup_read(w0, lane);
    if constexpr (!kStrided) {
      const int64_t rows = extent / ld - first;
      const int last = rows < TR ? int(rows) - 1 : TR - 1;
      base = ptr + first * ld;
      range = int(int64_t(last + 1) * ld * 2);
#pragma unroll
      for (int q = 0; q < kCopies; ++q) {
        const int id = wave * kCopies + q, slab = id / (TR / 8), row = (id % (TR / 8)) * 8 + (lane >> 3);
        const int k = slab * 64 + (((lane & 7) ^ ((row >> 1) & 7)) << 3);
        voff[q] = row <= last ? int((int64_t(row) * ld + k) * 2) : kOutOfRange;
        voffT[q] = k < kRem ? voff[q] : kOutOfRange;
      }
      step = BK * 2;
    } else {
      constexpr int kRow = TR * 2, kChunks = kRow / 16; // bytes and 16-byte chunks per k row
      base = ptr + first;
      const int64_t bytes = (extent - first) * 2;
      range = bytes > 0x7fffffff ? 0x7fffffff : int(bytes);
#pragma unroll
      for (int q = 0; q < kCopies; ++q) {
        const int row = (wave * kCopies + q) * (1024 / kRow) + lane / kChunks, chunk = lane % kChunks;
        const int pair = (chunk >> 1) ^ pair_swizzle<TR / 16>(row);
        const int64_t col = pair * 16 + (chunk & 1) * 8; // ld % 8 == 0: a piece is inside or not
        voff[q] = first + col < ld ? int((int64_t(row) * ld + col) * 2) : kOutOfRange;
        voffT[q] = row < kRem ? voff[q] : kOutOfRange;
      }
      step = int(BK * ld * 2);
    }
  }
  // step `kt` of `steps` into the image at `image`
  __device__ __forceinline__ void dma(LdsChar *lds, int image, int kt, int steps) const {
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(base), 0, kt < steps ? range : 0, 0x00020000);
    const bool tail = kt == steps - 1;
    const int at = kt < steps ? kt * step : 0; // (never beyond the descriptor's range)
#pragma unroll
    for (int q = 0; q < kCopies; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, lds + image + dst + q * 1024, 16, tail ? voffT[q] : voff[q], at, 0, 0);
  }
  // fragment f (16 rows from w0 + 16 f), 32-wide slice s of the step
  __device__ __forceinline__ typename T::Frag read(const char *lds, int image, int f, int s) const {
    if constexpr (!kStrided) {
      return *reinterpret_cast<const typename T::Frag *>(lds + image + (s >> 1) * (TR * 128) +
                                                         ((rd ^ ((s & 1) * 64)) + f * 16 * 128));
    } else {
      const char *p = lds + image + s * (32 * TR * 2) + rd + ((f ^ swz) << 5);
      const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4 *)(p));
      const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4 *)(p + 4 * TR * 2));
      return __builtin_bit_cast(typename T::Frag, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  }
};

template <int TMv, int TNv, int WMCv, int WNCv, int KGv, int Sv, bool kRefillv = false> struct SmallShape {
  static constexpr int TM = TMv, TN = TNv, WMC = WMCv, WNC = WNCv, KG = KGv, S = Sv;
  static constexpr bool kRefill = kRefillv; // a slot is filled again in the step whose fragments were the last read of it
  static constexpr int BK = 32 * KG;
  static constexpr int FI = TM / WMC / 16, FJ = TN / WNC / 16;
  static constexpr int kStageBytes = (TM + TN) * BK * 2;
  static constexpr int kPitch = TN + 4; // floats per row of a partial tile in LDS
  // the partial tiles of all key groups side by side, or one after the other where these would not fit
  static constexpr bool kMergeInPlace = KG * TM * kPitch * 4 > 160 * 1024;
  static constexpr int kMergeBytes = (kMergeInPlace ? 1 : KG) * TM * kPitch * 4;
  static constexpr int kLds = S * kStageBytes > kMergeBytes ? S * kStageBytes : kMergeBytes;
  static constexpr int kWavesPerEu = kLds <= 80 * 1024 ? 4 : 2; // two workgroups on a CU where LDS has room for two
  static_assert(WMC * WNC * KG == kWaves && BK % 64 == 0 && kLds <= 160 * 1024, "eight wavefronts, one CU's LDS");
};

// The end of a tile: the KG partial tiles meet in LDS (which nobody reads or writes any more: a barrier has been
// passed since), are added in group order, and what lies inside C goes through the epilogue.
template <typename P, typename Epi>
__device__ __forceinline__ void merge_and_store(const f32x4 (&acc)[P::FI][P::FJ], char *lds, int64_t M, int64_t N,
                                                const Epi &epi, int64_t m0, int64_t n0, int kg, int wm, int wn,
                                                int lane) {
  constexpr int FI = P::FI, FJ = P::FJ;
  const int tid = threadIdx.x;
  // partial tiles side by side in LDS: lane holds row lane % 16, columns (lane / 16) * 4 .. + 3 of a block
  float *part = reinterpret_cast<float *>(lds);
  {
    float *mine = part + (P::kMergeInPlace ? 0 : kg) * (P::TM * P::kPitch) +
                  (wm * (P::TM / P::WMC) + (lane & 15)) * P::kPitch + wn * (P::TN / P::WNC) + (lane >> 4) * 4;
    auto put = [&](bool add) {
#pragma unroll
      for (int i = 0; i < FI; ++i)
#pragma unroll
        for (int j = 0; j < FJ; ++j) {
          f32x4 *at = reinterpret_cast<f32x4 *>(mine + i * 16 * P::kPitch + j * 16);
          *at = add ? acc[i][j] + *at : acc[i][j];
        }
    };
    if constexpr (P::kMergeInPlace) {
      static_assert(P::KG == 2);
      if (kg == 1) // uniform over the wavefront
        put(false);
      __syncthreads();
      if (kg == 0)
        put(true);
    } else {
      put(false);
    }
  }
  __syncthreads();
  constexpr int kVecs = P::TM * P::TN / 4;
#pragma unroll
  for (int u = 0; u < (kVecs + kThreads - 1) / kThreads; ++u) {
    const int v = u * kThreads + tid;
    if (kVecs % kThreads == 0 || v < kVecs) {
      const int r = v / (P::TN / 4), c = (v % (P::TN / 4)) * 4;
      f32x4 sum = *reinterpret_cast<const f32x4 *>(part + r * P::kPitch + c);
#pragma unroll
      for (int g = 1; g < (P::kMergeInPlace ? 1 : P::KG); ++g)
        sum += *reinterpret_cast<const f32x4 *>(part + g * (P::TM * P::kPitch) + r * P::kPitch + c);
      if (m0 + r < M && n0 + c < N)
        store_columns(epi, m0 + r, n0 + c, N, sum);
    }
  }
}

template <typename T, bool kAT, bool kBT, typename P, typename Epi>
__device__ __forceinline__ void gemm_small_tile(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B,
                                                int64_t M, int64_t N, int64_t K, Epi epi, char *lds, int64_t m0,
                                                int64_t n0) {
  constexpr int FI = P::FI, FJ = P::FJ, S = P::S;
  LdsChar *ldsBase = (LdsChar *)lds;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave / (P::WMC * P::WNC), wmn = wave % (P::WMC * P::WNC);
  const int wm = wmn / P::WNC, wn = wmn % P::WNC;
  const int steps = int((K + P::BK - 1) / P::BK), kRem = int(K - int64_t(steps - 1) * P::BK);
  SmallOperand<T, kAT, P::TM, P::BK> opA;
  SmallOperand<T, !kBT, P::TN, P::BK> opB;
  opA.setup(A, kAT ? M : K, m0, wm * (P::TM / P::WMC), M * K, wave, lane, kRem);
  opB.setup(B, kBT ? K : N, n0, wn * (P::TN / P::WNC), K * N, wave, lane, kRem);
  constexpr int kImageA = 0, kImageB = P::TM * P::BK * 2;
  constexpr int kCopies = decltype(opA)::kCopies + decltype(opB)::kCopies;

  f32x4 acc[FI][FJ];
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j)
      acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // With eight A fragments per wavefront there is room for one set of them: each is replaced by the next step's as soon
  // as its products are issued.
  constexpr bool kOneA = FI >= 8;
  static_assert(!(kOneA && P::kRefill), "with one set of A fragments the ring is filled in front of a step's barrier only");
  typename T::Frag af[kOneA ? 1 : 2][FI], bf[2][FJ];
  auto dma = [&](int kt, int slot) {
    opA.dma(ldsBase, slot * P::kStageBytes + kImageA, kt, steps);
    opB.dma(ldsBase, slot * P::kStageBytes + kImageB, kt, steps);
  };
  auto read_a = [&](int p, int slot, int i) { af[kOneA ? 0 : p][i] = opA.read(lds, slot * P::kStageBytes + kImageA, i, kg); };
  auto read_b = [&](int p, int slot) {
#pragma unroll
    for (int j = 0; j < FJ; ++j)
      bf[p][j] = opB.read(lds, slot * P::kStageBytes + kImageB, j, kg);
  };
  auto read = [&](int p, int slot) {
#pragma unroll
    for (int i = 0; i < FI; ++i)
      read_a(p, slot, i);
    read_b(p, slot);
  };
#pragma unroll
  for (int t = 0; t < (P::kRefill ? S : S - 1); ++t)
    dma(t, t);
  wait_vmcnt<(P::kRefill ? S - 1 : S - 2) * kCopies>();
  __builtin_amdgcn_s_barrier();
  IMEX_FENCE();
  read(0, 0);
  // Step t: everybody's fragments of step t - 1 were in registers before the barrier of that step, so its slot takes slab
  // t + S - 1; slab t + 1 has landed at the barrier of this one.  With kRefill the slot of step t takes slab t + S behind
  // the barrier of step t, at which everybody's fragments of it are in registers.
  int cur = 0; // slot of step t
  auto step = [&](int p, int t) {
    const int nxt = cur + 1 == S ? 0 : cur + 1, free = cur == 0 ? S - 1 : cur - 1;
    if constexpr (!P::kRefill)
      dma(t + S - 1, free);
    wait_vmcnt<(S - 2) * kCopies>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    IMEX_FENCE();
    if constexpr (kOneA) {
      read_b(p ^ 1, nxt);
      IMEX_FENCE();
#pragma unroll
      for (int i = 0; i < FI; ++i) {
#pragma unroll
        for (int s = 0; s < FJ; ++s) {
          const int j = (i & 1) ? FJ - 1 - s : s;
          acc[i][j] = T::mfma(bf[p][j], af[0][i], acc[i][j]);
        }
        read_a(0, nxt, i);
        IMEX_FENCE();
      }
    } else {
      read(p ^ 1, nxt);
      if constexpr (P::kRefill)
        dma(t + S, cur);
      IMEX_FENCE();
#pragma unroll
      for (int j = 0; j < FJ; ++j)
#pragma unroll
        for (int s = 0; s < FI; ++s) {
          const int i = (j & 1) ? FI - 1 - s : s;
          acc[i][j] = T::mfma(bf[p][j], af[p][i], acc[i][j]);
        }
    }
    cur = nxt;
  };
  int t = 0;
  for (; t + 1 < steps; t += 2) {
    step(0, t);
    step(1, t + 1);
  }
  if (t < steps)
    step(0, t);
  wait_vmcnt<0>();
  __syncthreads(); // the ring is free

  merge_and_store<P>(acc, lds, M, N, epi, m0, n0, kg, wm, wn, lane);
}

// Tile number -> tile, as tile_origin of gemm_tile.h: the workgroups of an XCD (ids congruent mod 8) take a compact
// band of tiles, four tile rows high; as many tiles for each XCD, or one more.  (With the last tiles % 8 in launch order behind
// eight equal shares instead, 411 products that 8 does not divide take 1.006 of the time in the mean, 0.93 .. 1.11.)
constexpr uint32_t kXcds = 8;
__device__ __forceinline__ uint32_t first_tile_of_xcd(uint32_t xcd, uint32_t tiles) {
  return xcd * (tiles / kXcds) + min(xcd, tiles % kXcds);
}
template <typename P> __device__ __forceinline__ TileOrigin small_tile_origin(uint32_t id, uint32_t tilesM, uint32_t tilesN) {
  const uint32_t pid = first_tile_of_xcd(id % kXcds, tilesM * tilesN) + id / kXcds;
  const uint32_t group = kGroupM * tilesN, band = pid / group, in = pid - band * group;
  const uint32_t rows = min(tilesM - band * kGroupM, uint32_t(kGroupM));
  uint32_t row = in % kGroupM, col = in / kGroupM;
  // Fewer rows in the last band only.  A signed division here for every tile, and signed ones above, were 0.13 us on the
  // way to the first load: f16 B^T 1000 x 1000 x 1000 7.50 -> 7.36 us, over 20 problems of 7 .. 30 us 0.3 .. 2 %.
  if (rows != kGroupM) {
    col = in / rows;
    row = in - col * rows;
  }
  return TileOrigin{int64_t(band * kGroupM + row) * P::TM, int64_t(col) * P::TN};
}

// Workgroups without a tile fetch what the other workgroups of their XCD are going to read.  A CU draws no more than 50
// GB/s from beyond its L2 (a limit on requests: 16 GB/s in 32-byte pieces of rows, 29 in 64-byte ones, 51 in lines) but 180
// from it, so a few workgroups that walk a long K alone wait for memory while the rest of the chip is idle: that rest brings
// the operands of an XCD's tiles into its L2, in the order of K, 512 k at a time, as copies into LDS that nobody reads.
// bf16 16 x 2048 x 4096 from HBM 14.0 -> 7.2 us (6.0 when the L2s have it), from the 256 MiB cache 11.3 -> 7.1; 16 x 1680 x
// 3992 9.2 -> 6.6.  Nothing depends on it but the time: if workgroups lay elsewhere than on XCD id % 8, lines would be
// fetched that nobody asks for.
template <bool kAT, bool kBT, typename P>
__device__ __forceinline__ void fetch_ahead(const uint16_t *A, const uint16_t *B, uint32_t M, uint32_t N, uint32_t K,
                                            char *lds, uint32_t id, uint32_t tilesM, uint32_t tilesN, uint32_t workgroups) {
  constexpr uint32_t kChunk = 512;
  const uint32_t tiles = tilesM * tilesN, xcd = id % kXcds;
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the XCD's tiles, this workgroup's number among those of the XCD that fetch, and their wavefronts
  const uint32_t from = first_tile_of_xcd(xcd, tiles), to = first_tile_of_xcd(xcd + 1, tiles);
  const uint32_t rank = id / kXcds - (to - from), turns = ((workgroups + kXcds - 1 - xcd) / kXcds - (to - from)) * kWaves;
  if (turns < 8 * kWaves) // too few: the others would wait for them (200 x 301 x 901 on 247 of 256 workgroups 5 us, 34 so)
    return;
  LdsChar *sink = (LdsChar *)lds + wave * 1024;
  // What the tiles read: rows m0 .. m1 - 1 of A, columns n0 .. n1 - 1 of B, for those of the first band of tile rows and for
  // the others (of one band, or all columns of more).
  struct Block {
    uint32_t m0, m1, n0, n1;
  };
  const uint32_t band = kGroupM * tilesN, turnover = min((from / band + 1) * band, to);
  auto block = [&](uint32_t p, uint32_t end) {
    if (p >= end)
      return Block{0, 0, 0, 0};
    const uint32_t first = p / band, last = (end - 1) / band, rows = min(tilesM - first * kGroupM, uint32_t(kGroupM));
    const uint32_t col = (p - first * band) / rows, lastCol = first == last ? (end - 1 - first * band) / rows : tilesN - 1;
    return Block{first * kGroupM * P::TM, min((last + 1) * kGroupM * P::TM, M), first == last ? col * P::TN : 0,
                 min((lastCol + 1) * P::TN, N)};
  };
  const Block blocks[2] = {block(from, turnover), block(turnover, to)};
  uint32_t turn;
  // Rows (k-contiguous) or columns (strided) first .. last - 1 of an operand, ks of its k from k0 on: a row for each wavefront
  // in turn, or as many k rows as 64 pieces of 16 bytes hold.  (Few instructions per copy, and few copies, 0.15 us each: with
  // addresses in 64 bits, or one k row of 200 bytes and less in each, they took longer than the tiles.  One k row each, operands
  // in the L2s: A^T 112 x 72 x 6760 8.7 us without workgroups that fetch, 13.7 with them.)
  auto fetch = [&](const uint16_t *ptr, bool strided, uint32_t ld, uint32_t first, uint32_t last, uint32_t k0, uint32_t ks) {
    const uint32_t count = strided ? ks : last - first, bytes = (strided ? last - first : ks) * 2, pitch = ld * 2;
    if (first >= last || uint64_t(count) * pitch >= kOutOfRange)
      return;
    const uint16_t *base = ptr + (strided ? uint64_t(k0) * ld + first : uint64_t(first) * ld + k0);
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(base), 0, int((count - 1) * pitch + bytes), 0x00020000);
    if (strided && bytes <= 512) {
      const uint32_t pieces = bytes / 16, rows = 64 / pieces, row = lane / pieces, off = row * pitch + (lane - row * pieces) * 16;
      const uint32_t copies = (count + rows - 1) / rows;
      for (; turn < copies; turn += turns)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, sink, 16, row < min(rows, count - turn * rows) ? turn * rows * pitch + off : kOutOfRange,
                                                 0, 0, 0);
      turn -= copies;
      return;
    }
    for (; turn < count; turn += turns)
      for (uint32_t b = 0; b < bytes; b += 1024)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, sink, 16, b + lane * 16 < bytes ? b + lane * 16 : kOutOfRange,
                                                 turn * pitch, 0, 0);
    turn -= count;
  };
  for (uint32_t k0 = 0; k0 < K; k0 += kChunk) {
    const uint32_t ks = min(K - k0, kChunk);
    turn = rank * kWaves + wave;
#pragma unroll
    for (const Block &b : blocks) {
      fetch(A, kAT, kAT ? M : K, b.m0, b.m1, k0, ks);
      fetch(B, !kBT, kBT ? K : N, b.n0, b.n1, k0, ks);
    }
  }
  wait_vmcnt<0>(); // the copies' place in LDS is given back with the workgroup
}

template <typename T, bool kAT, bool kBT, typename P, typename Epi>
__device__ __forceinline__ void gemm_small_entry(const uint16_t *A, const uint16_t *B, int64_t M, int64_t N, int64_t K,
                                                 Epi epi) {
  __shared__ __attribute__((aligned(16))) char lds[P::kLds];
  if (!mfma_takes<kAT, kBT>(A, B, M, N, K)) {
    gemm_blocked<T, kAT, kBT, Epi>(A, B, M, N, K, epi, lds);
    return;
  }
  const int tilesM = int((M + P::TM - 1) / P::TM), tilesN = int((N + P::TN - 1) / P::TN);
  const int tiles = tilesM * tilesN, workgroups = gridDim.x * gridDim.y;
  int id = blockIdx.y * gridDim.x + blockIdx.x;
  if (id >= tiles) {
    fetch_ahead<kAT, kBT, P>(A, B, uint32_t(M), uint32_t(N), uint32_t(K), lds, id, tilesM, tilesN, workgroups);
    return;
  }
  for (; id < tiles; id += workgroups) {
    const TileOrigin o = small_tile_origin<P>(id, tilesM, tilesN);
    gemm_small_tile<T, kAT, kBT, P, Epi>(A, B, M, N, K, epi, lds, o.m0, o.n0);
    if (id + workgroups < tiles)
      __syncthreads(); // the partial tiles are read before the ring is filled again
  }
}

} // namespace imexhip_gemm

#endif

// Tile code of the MFMA GEMM for operands whose rows are not 16-byte aligned in memory (K, or the N of a B [K,N], or
// the M of an A [K,M], no multiple of 8): C[M,N] = A[M,K] . B[K,N], A and B f16 or bf16, f32 sums.  Entry points:
// gemm_unaligned.hip.  The reference kernels these stand for are those of gemm_tile.h.
//
// The tiles, the sharing of k between wavefronts, the LDS images and the end of a tile are those of gemm_small.h.
// What differs is how a slab gets into LDS: the direct global -> LDS copies want aligned pieces, ordinary 16-byte
// loads take any address, so a slab goes through registers.
//
//   loads       16 bytes per lane at the element's own (2-byte aligned) address, D slabs in flight in registers;
//   edges       in the last step, a piece that would stick out of its row is loaded from the last 16 bytes of the row and
//               shifted down, zeros following: no address leaves the matrix, and nothing beyond K is multiplied by
//               anything but zero.  In the steps before it a strided operand's last pieces run into the next row: what
//               they find there lies in columns that are never stored.  (Shifting them in every step held up the whole
//               launch for the last tile column: f16 1001 x 1003 x 999 10.45 us, 9.5 so; A^T 11.7 / 9.7);
//   LDS         two slots: slab t + 2 is written to the slot that step t's fragments have been read from.
//
// Bound by the latency of a step (load, LDS write, barrier, fragment reads), as gemm_small.h is; the vector-ALU loop
// that took these shapes before spent 4.4 us on every sixteen k, most of it waiting for one element's load after the
// other.  A step of 64 k takes 0.37 us on 64 x 64 tiles (0.27 with direct copies; as the rules of
// KernelCatalog.cpp have them).  1001 x 1003 x 999 f16: 276 us before, 9.5 here.

#ifndef IMEX_HIP_GEMM_UNALIGNED_H
#define IMEX_HIP_GEMM_UNALIGNED_H

#include "gemm_small.h"

namespace imexhip_gemm {

typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(2))); // 8 halves at any half address

// The eight 16-bit elements of v moved down by s (0 .. 7) places, zeros following; s >= 8: all zero.
__device__ __forceinline__ u32x4 shift_down(u32x4 v, int s) {
  uint32_t d0 = v.x, d1 = v.y, d2 = v.z, d3 = v.w;
  const bool by4 = s & 4, by2 = s & 2, by1 = s & 1;
  d0 = by4 ? d2 : d0, d1 = by4 ? d3 : d1, d2 = by4 ? 0 : d2, d3 = by4 ? 0 : d3;
  d0 = by2 ? d1 : d0, d1 = by2 ? d2 : d1, d2 = by2 ? d3 : d2, d3 = by2 ? 0 : d3;
  const uint32_t e0 = (d0 >> 16) | (d1 << 16), e1 = (d1 >> 16) | (d2 << 16), e2 = (d2 >> 16) | (d3 << 16);
  d0 = by1 ? e0 : d0, d1 = by1 ? e1 : d1, d2 = by1 ? e2 : d2, d3 = by1 ? d3 >> 16 : d3;
  const bool none = s >= 8;
  return u32x4{none ? 0 : d0, none ? 0 : d1, none ? 0 : d2, none ? 0 : d3};
}

// One operand's TR x BK (rows x k) slab per step, through registers.
template <typename T, bool kStrided, int TR, int BK> struct UnalignedOperand : SmallOperand<T, kStrided, TR, BK> {
  using Base = SmallOperand<T, kStrided, TR, BK>;
  using Base::kCopies;
  const char *from;        // the operand (strided) or its row `first` (k-contiguous)
  int64_t stepBytes;       // bytes per step in memory
  uint32_t off[kCopies];   // per-lane byte offsets from the step's base
  uint32_t offT[kCopies];  // the same for the last step (k-contiguous: from step 0's base)
  int shift[kCopies];      // places by which the piece has to move down in the last step
  int put;                 // per-lane LDS address of copy 0 inside the image

  // K >= 8, and ld >= 8 where kStrided.  ld < 2^22 keeps a strided operand's offsets, (BK - 1) rows and one row's columns, below
  // 2^31 with BK = 256, and a k-contiguous one's, TR - 1 rows and the last step's end, below 2^30.
  static_assert((uint64_t(kStrided ? BK : TR) << 22) * 2 <= uint64_t(1) << 31, "rows of up to 2^22 elements within 32-bit offsets");
  __device__ __forceinline__ void setup(const uint16_t *ptr, int64_t ld, int64_t first, int64_t rows, int w0, int wave,
                                        int lane, int steps, int kRem) {
    this->setup_read(w0, lane);
    put = wave * kCopies * 1024 + lane * 16;
    if constexpr (!kStrided) {
      const int last = int(min(rows - first, int64_t(TR))) - 1;
      from = reinterpret_cast<const char *>(ptr + first * ld);
      stepBytes = BK * 2;
#pragma unroll
      for (int q = 0; q < kCopies; ++q) {
        const int id = wave * kCopies + q, slab = id / (TR / 8), row = (id % (TR / 8)) * 8 + (lane >> 3);
        const int k = slab * 64 + (((lane & 7) ^ ((row >> 1) & 7)) << 3);
        const uint32_t rowOff = uint32_t(min(row, last)) * uint32_t(ld) * 2;
        off[q] = rowOff + k * 2;
        const int kT = min(k, kRem - 8); // may lie in the step before
        shift[q] = k - kT;
        offT[q] = rowOff + uint32_t((steps - 1) * BK + kT) * 2;
      }
    } else {
      constexpr int kRow = TR * 2, kChunks = kRow / 16; // bytes and 16-byte chunks per k row
      from = reinterpret_cast<const char *>(ptr);
      stepBytes = BK * ld * 2;
#pragma unroll
      for (int q = 0; q < kCopies; ++q) {
        const int row = (wave * kCopies + q) * (1024 / kRow) + lane / kChunks, chunk = lane % kChunks;
        const int pair = (chunk >> 1) ^ pair_swizzle<TR / 16>(row);
        const int64_t col = first + pair * 16 + (chunk & 1) * 8, at = min(col, ld - 8);
        shift[q] = int(col - at);
        off[q] = (uint32_t(row) * uint32_t(ld) + uint32_t(col < ld ? col : at)) * 2; // (another row follows this one)
        offT[q] = (uint32_t(min(row, kRem - 1)) * uint32_t(ld) + uint32_t(at)) * 2;
      }
    }
  }
  // A slab past the last one is not needed; it is loaded all the same, every lane the operand's first 16 bytes, so that
  // the number of loads in flight is known at every wait.
  __device__ __forceinline__ void fetch(u32x4 (&r)[kCopies], int slab, int steps) const {
    const bool tail = slab == steps - 1, past = slab >= steps;
    const char *base = from + (past || (tail && !kStrided) ? 0 : slab * stepBytes);
#pragma unroll
    for (int q = 0; q < kCopies; ++q) {
      uint32_t o = past ? 0u : tail ? offT[q] : off[q];
      asm volatile("" : "+v"(o)); // (one load per piece, selected by its address: no branches around equal ones)
      r[q] = *reinterpret_cast<const u32x4u *>(base + o);
    }
  }
  __device__ __forceinline__ void store(u32x4 (&r)[kCopies], char *image, int slab, int steps, int kRem) const {
    const bool tail = slab == steps - 1;
    if (tail) {
#pragma unroll
      for (int q = 0; q < kCopies; ++q) {
        int s = shift[q];
        if constexpr (kStrided) {
          constexpr int kRow = TR * 2;
          const int row = (put + q * 1024) / kRow;
          s = row >= kRem ? 8 : s;
        }
        r[q] = shift_down(r[q], s);
      }
    }
#pragma unroll
    for (int q = 0; q < kCopies; ++q)
      *reinterpret_cast<u32x4 *>(image + put + q * 1024) = r[q];
  }
};

template <int I> struct Phase { static constexpr int value = I; };

template <typename T, bool kAT, bool kBT, typename P, int D, typename Epi>
__device__ __forceinline__ void gemm_unaligned_tile(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B,
                                                    int64_t M, int64_t N, int64_t K, Epi epi, char *lds, int64_t m0,
                                                    int64_t n0) {
  static_assert(D % 2 == 0 && P::S == 2, "a slab's registers, its LDS slot and its fragments' parity follow from its number mod D");
  constexpr int FI = P::FI, FJ = P::FJ;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave / (P::WMC * P::WNC), wmn = wave % (P::WMC * P::WNC);
  const int wm = wmn / P::WNC, wn = wmn % P::WNC;
  const int steps = int((K + P::BK - 1) / P::BK), kRem = int(K - int64_t(steps - 1) * P::BK);
  UnalignedOperand<T, kAT, P::TM, P::BK> opA;
  UnalignedOperand<T, !kBT, P::TN, P::BK> opB;
  opA.setup(A, kAT ? M : K, m0, M, wm * (P::TM / P::WMC), wave, lane, steps, kRem);
  opB.setup(B, kBT ? K : N, n0, N, wn * (P::TN / P::WNC), wave, lane, steps, kRem);
  constexpr int kImageB = P::TM * P::BK * 2;

  f32x4 acc[FI][FJ];
#pragma unroll
  for (int i = 0; i < FI; ++i)
#pragma unroll
    for (int j = 0; j < FJ; ++j)
      acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  typename T::Frag af[2][FI], bf[2][FJ];
  u32x4 ra[D][decltype(opA)::kCopies], rb[D][decltype(opB)::kCopies];
  auto fetch = [&](int q, int slab) {
    opA.fetch(ra[q], slab, steps);
    opB.fetch(rb[q], slab, steps);
  };
  auto store = [&](int q, int slab) {
    char *slot = lds + (q & 1) * P::kStageBytes;
    opA.store(ra[q], slot, slab, steps, kRem);
    opB.store(rb[q], slot + kImageB, slab, steps, kRem);
  };
  auto read = [&](int p) { // fragments of a slab of parity p
#pragma unroll
    for (int i = 0; i < FI; ++i)
      af[p][i] = opA.read(lds, p * P::kStageBytes, i, kg);
#pragma unroll
    for (int j = 0; j < FJ; ++j)
      bf[p][j] = opB.read(lds, p * P::kStageBytes + kImageB, j, kg);
  };
  auto meet = [&] { // everybody's LDS accesses are done
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    IMEX_FENCE();
  };
#pragma unroll
  for (int q = 0; q < D; ++q)
    fetch(q, q);
  store(0, 0);
  fetch(0, D);
  meet();
  read(0);
  store(1, 1);
  fetch(1, D + 1);
  meet();
  // Step t: its fragments are in registers, slab t + 1 is in LDS, slabs t + 2 .. t + D + 1 are in flight.
  auto step = [&](auto phase, int t) {
    constexpr int ph = decltype(phase)::value, p = ph & 1, q = (ph + 2) % D;
    store(q, t + 2);
    fetch(q, t + 2 + D);
    IMEX_FENCE();
    read(p ^ 1);
    IMEX_FENCE();
#pragma unroll
    for (int j = 0; j < FJ; ++j)
#pragma unroll
      for (int s = 0; s < FI; ++s) {
        const int i = (j & 1) ? FI - 1 - s : s;
        acc[i][j] = T::mfma(bf[p][j], af[p][i], acc[i][j]);
      }
    meet();
  };
  // (whole rounds of D steps as one straight line: the loads in flight at every wait are then known exactly)
  int t = 0;
  for (; t + D <= steps; t += D) {
    step(Phase<0>{}, t);
    step(Phase<1>{}, t + 1);
    if constexpr (D == 4) {
      step(Phase<2>{}, t + 2);
      step(Phase<3>{}, t + 3);
    }
  }
  if (t < steps) {
    step(Phase<0>{}, t);
    if constexpr (D == 4) {
      if (t + 1 < steps) {
        step(Phase<1>{}, t + 1);
        if (t + 2 < steps)
          step(Phase<2>{}, t + 2);
      }
    }
  }
  merge_and_store<P>(acc, lds, M, N, epi, m0, n0, kg, wm, wn, lane);
}

// What this path takes: 16 bytes fit into every row that a piece is loaded from, and the offsets fit 32 bits.
template <bool kAT, bool kBT> __device__ __forceinline__ bool unaligned_takes(int64_t M, int64_t N, int64_t K) {
  constexpr int64_t kMaxRow = int64_t(1) << 22;
  return M > 0 && N > 0 && K >= 8 && K < kMaxRow && (!kAT || (M >= 8 && M < kMaxRow)) && (kBT || (N >= 8 && N < kMaxRow));
}

template <typename T, bool kAT, bool kBT, typename P, int D, typename Epi>
__device__ __forceinline__ void gemm_unaligned_entry(const uint16_t *A, const uint16_t *B, int64_t M, int64_t N,
                                                     int64_t K, Epi epi) {
  __shared__ __attribute__((aligned(16))) char lds[P::kLds];
  if (!unaligned_takes<kAT, kBT>(M, N, K)) {
    gemm_blocked<T, kAT, kBT, Epi>(A, B, M, N, K, epi, lds);
    return;
  }
  const int tilesM = int((M + P::TM - 1) / P::TM), tilesN = int((N + P::TN - 1) / P::TN);
  const int tiles = tilesM * tilesN, workgroups = gridDim.x * gridDim.y;
  for (int id = blockIdx.y * gridDim.x + blockIdx.x; id < tiles; id += workgroups) {
    const TileOrigin o = small_tile_origin<P>(id, tilesM, tilesN);
    gemm_unaligned_tile<T, kAT, kBT, P, D, Epi>(A, B, M, N, K, epi, lds, o.m0, o.n0);
    if (id + workgroups < tiles)
      __syncthreads(); // the partial tiles are read before the slots are filled again
  }
}

} // namespace imexhip_gemm

#endif

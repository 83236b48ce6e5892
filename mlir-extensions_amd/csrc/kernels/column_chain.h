// Sums down the columns of a row-major matrix, added in row order: out[c] = ((init + x[0,c]) + x[1,c]) + ..., where x
// is the matrix itself or a function of two of them evaluated on the way (the outer-dimension sums of reduce.hip, the
// fused chain of fusion.hip).  For matrices with too few columns to give every lane of the chip one.
//
// What bounds it is the chain of dependent additions of a column: a lone wavefront issues one instruction every four
// cycles or so whatever it is, so a row costs four cycles for its addition and four for every other instruction that
// the adding wavefront runs per row (measured, cycles per row: additions alone 4.2; with a 32-bit LDS read each 8.8 ..
// 10; with a 128-bit read per four rows and one wait per sixteen 5.3; a 16-bit value widened by the adder 10.9).  So
// the work is split between wavefronts of one workgroup: workers load, widen, evaluate and write f32 values to LDS
// COLUMN by column, and one wavefront does nothing but add, a lane per column, four rows per LDS read.  A lane of a
// worker loads the same 8 or 16 bytes of four consecutive rows and so holds four consecutive values of every column it
// touches: the change of layout costs no instruction.  One barrier per tile of rows hands a tile over and the other one
// back.  Workgroups of neighbouring segments run on one XCD, whose L2 then fetches a 128-byte line once for all of them.
#ifndef IMEX_HIP_COLUMN_CHAIN_H
#define IMEX_HIP_COLUMN_CHAIN_H

#include "device_common.h"

namespace imexhip {

// kInputs matrices; kLanes lanes of a worker cover a row's segment with kWords 32-bit words each; kWorkers wavefronts of
// workers; loads run kAhead tiles ahead of the one that is evaluated.
template <io::Dt D, int kInputs_, int kLanes_, int kWords_, int kWorkers_, int kAhead_> struct ColumnChain {
  using E = io::Elem<D>;
  static constexpr int kInputs = kInputs_, kLanes = kLanes_, kWords = kWords_, kWorkers = kWorkers_, kAhead = kAhead_;
  static constexpr int kPer = kWords * 4 / E::kBytes;           // columns per lane
  static constexpr int kCols = kLanes * kPer;                   // columns per workgroup, a lane of the adder each
  static constexpr int kRowsPerWave = 4 * (kWave / kLanes);     // rows of a tile that one worker wavefront takes
  static constexpr int kTileRows = kWorkers * kRowsPerWave;
  static constexpr int kThreads = (kWorkers + 1) * kWave;
  // Floats from one column of a tile to the next.  128-bit LDS accesses are served sixteen lanes at a time over 64
  // banks.  The adder's lanes read at c * pitch: an odd number of 4-word groups serves sixteen lanes without conflict,
  // two for eight.  A worker's sixteen lanes write four rows-of-four of four column groups, kPer * pitch apart: with
  // 16 words (modulo 64) between these they land on sixteen different groups.
  static constexpr int kPad = kCols <= 8 ? 8 : 4;
  static constexpr int kPitch = kTileRows + kPad;
  static constexpr int kTileFloats = kCols * kPitch;
  static constexpr int kLdsFloats = 2 * kTileFloats;
  static_assert(kCols <= kWave && kTileRows % 64 == 0, "a lane per column; the adder takes sixteen rows at a time, four deep");

  typedef uint32_t Raw __attribute__((ext_vector_type(kWords), aligned(E::kBytes))); // at any element's address
  struct Tile {
    Raw v[kInputs][4];
  };

  static __device__ __forceinline__ bool takes(int64_t rows, int64_t cols) {
    // a tile's rows are addressed with 32-bit offsets from its first one
    return cols >= kCols && cols * E::kBytes < (int64_t(1) << 31) / kTileRows && rows < (int64_t(1) << 40);
  }

  // prologue(): run by every thread while the first loads are in flight; what it leaves in LDS is there for eval.
  // eval(const Raw (&words)[kInputs], float (&f)[kPer]): one row's values of this lane's columns.
  template <typename Prologue, typename Eval>
  static __device__ __forceinline__ void run(const void *a, const void *b, void *out, int64_t rows, int64_t cols, float init,
                                             float *lds, Prologue prologue, Eval eval) {
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t pitch = static_cast<uint32_t>(cols * E::kBytes);
    const int64_t tiles = (rows + kTileRows - 1) / kTileRows;
    const int lastRows = static_cast<int>(rows - (tiles - 1) * kTileRows); // of the last tile
    const int64_t blocks = (cols + kCols - 1) / kCols;
    bool first = true;
    for (int64_t w = blockIdx.x; w < blocks; w += gridDim.x) {
      // Workgroup w runs on XCD w % 8: the XCDs take contiguous shares of the segments.  (The last block of columns
      // starts early enough to be whole; columns that two workgroups share get the same value from both.)
      const int64_t share = blocks / 8, extra = blocks % 8, x = w % 8;
      const int64_t block = x * share + min(x, extra) + w / 8;
      const int64_t c0 = min(block * kCols, cols - kCols);
      if (wave < kWorkers) {
        const int quad = wave * (kWave / kLanes) + lane / kLanes; // rows 4 quad .. 4 quad + 3 of a tile
        const int col = (lane % kLanes) * kPer;
        const char *base[2] = {static_cast<const char *>(a) + c0 * E::kBytes, static_cast<const char *>(b) + c0 * E::kBytes};
        uint32_t at[4], atLast[4]; // rows past the end re-read the last one; they are never added
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          at[i] = static_cast<uint32_t>(4 * quad + i) * pitch + col * E::kBytes;
          atLast[i] = static_cast<uint32_t>(min(4 * quad + i, lastRows - 1)) * pitch + col * E::kBytes;
        }
        auto load = [&](int64_t t, Tile &tile) { // tiles past the end: the last one again, never evaluated
          const bool last = t >= tiles - 1;
          const int64_t start = (last ? tiles - 1 : t) * kTileRows * int64_t(pitch);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint32_t o = last ? atLast[i] : at[i];
#pragma unroll
            for (int n = 0; n < kInputs; ++n)
              tile.v[n][i] = __builtin_nontemporal_load(reinterpret_cast<const Raw *>(base[n] + start + o));
          }
        };
        auto put = [&](int64_t t, const Tile &tile) {
          if (t < tiles - 1 || 4 * (quad - lane / kLanes) < lastRows) { // uniform: a wavefront wholly past the end has nothing to do
            float *dst = lds + (t & 1) * kTileFloats + col * kPitch + 4 * quad;
            float f[4][kPer];
            eval(tile.v, f);
#pragma unroll
            for (int e = 0; e < kPer; ++e)
              *reinterpret_cast<f32x4 *>(dst + e * kPitch) = f32x4{f[0][e], f[1][e], f[2][e], f[3][e]};
          }
          handover(); // tile t is complete; the adder is done with tile t - 1, whose place tile t + 1 goes to
        };
        Tile ring[kAhead + 1];
        if (tiles > 0) {
#pragma unroll
          for (int u = 0; u < kAhead; ++u)
            load(u, ring[u]);
        }
        if (first) {
          prologue();
          handover();
        }
        for (int64_t t = 0; t < tiles; t += kAhead + 1) {
#pragma unroll
          for (int u = 0; u <= kAhead; ++u) {
            if (t + u < tiles) { // uniform
              load(t + u + kAhead, ring[(u + kAhead) % (kAhead + 1)]);
              put(t + u, ring[u]);
            }
          }
        }
      } else {
        if (first) {
          prologue();
          handover();
        }
        __builtin_amdgcn_s_setprio(3); // the chain is the critical path
        const int col = lane % kCols;
        float acc = init;
        if (tiles > 0) {
          constexpr int kGroups = kTileRows / 16; // of sixteen rows, four LDS reads each, three groups ahead
          f32x4 x[4][4];
          const float *p = lds + col * kPitch;
          auto read = [&](f32x4(&v)[4], int g) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
              v[q] = *reinterpret_cast<const f32x4 *>(p + g * 16 + q * 4);
          };
          auto add = [&](f32x4(&v)[4]) {
            asm volatile("" : "+v"(v[3])); // one wait, for the youngest of the four reads
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              acc = acc + v[q].x;
              acc = acc + v[q].y;
              acc = acc + v[q].z;
              acc = acc + v[q].w;
            }
          };
          handover(); // tile 0 is complete
#pragma unroll
          for (int g = 0; g < 3; ++g)
            read(x[g], g);
          for (int64_t t = 0; t + 1 < tiles; ++t) {
#pragma unroll
            for (int g = 0; g < kGroups; ++g) {
              if (g + 3 == kGroups) {
                handover(); // everything of tile t is in registers; tile t + 1 is complete
                p = lds + ((t + 1) & 1) * kTileFloats + col * kPitch;
              }
              read(x[(g + 3) % 4], (g + 3) % kGroups);
              add(x[g % 4]);
              __builtin_amdgcn_sched_barrier(0);
            }
          }
          // the last tile: 1 .. kTileRows rows
          int g = 0;
          for (; 16 * g + 64 <= lastRows; g += 4) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              read(x[(u + 3) % 4], min(g + u + 3, kGroups - 1));
              add(x[u]);
            }
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if (u == 0 && 16 * g + 48 < lastRows)
              read(x[3], g + 3);
            if (16 * (g + u) + 16 <= lastRows) { // uniform, as the others
              add(x[u]);
            } else {
#pragma unroll
              for (int r = 0; r < 15; ++r)
                if (16 * (g + u) + r < lastRows)
                  acc = acc + x[u][r / 4][r % 4];
            }
          }
        }
        __builtin_amdgcn_s_setprio(0);
        if (lane < kCols)
          E::put(out, c0 + lane, acc);
      }
      first = false;
      __syncthreads(); // both tiles are free for the next block of columns
    }
  }

private:
  // The hand-over of a tile between the workers and the adder.  The two run different code and meet here from different
  // places, which the hardware barrier allows (it counts wavefronts that have arrived, wherever each one arrives from);
  // what makes it correct is that both pass it exactly once per tile, and the barriers before and after the tiles once
  // per block of columns (the one after the prologue once per launch).  Written as the instruction with the LDS release
  // / acquire around it, not as a call the compiler may treat as convergent across the two branches.
  static __device__ __forceinline__ void handover() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  }
};

} // namespace imexhip
#endif

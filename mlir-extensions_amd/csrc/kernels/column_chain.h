// Sums down the columns of a row-major matrix, added in row order: out[c] = ((init + x[0,c]) + x[1,c]) + ..., where x
// is the matrix itself or a function of two of them evaluated on the way (the outer-dimension sums of reduce.hip, the
// fused chain of fusion.hip).  For matrices with too few columns to give every lane of the chip one.
//
// What bounds it is the chain of dependent additions of a column: a lone wavefront issues one instruction every four
// cycles or so whatever it is, so a row costs four cycles for its addition and four for every other instruction that
// the adding wavefront runs per row (measured, cycles per row: additions alone 4.2; with a 32-bit LDS read each 8.8 ..
// 10; with a 128-bit read per four rows 7.4, and here, with one wait per sixteen rows, 6.3; a 16-bit value widened by the
// adder 10.9).  So the work is split between the wavefronts of a workgroup: workers load, widen, evaluate and write f32
// values to LDS COLUMN by column, and one wavefront does nothing but add, a lane per column, four rows per LDS read.  A
// lane of a worker loads the same 8 bytes of four consecutive rows and so holds four consecutive values of every column
// it touches: the change of layout costs no instruction.  One barrier per tile of rows hands a tile over and the other
// one back; loads run one tile ahead or three (kAhead).
// Workgroups of neighbouring segments run on one XCD, whose L2 then fetches a 128-byte line once for all of them (in launch
// order / so: f32 sums of 8192 x 4096, one tile ahead, 42.7 / 37.0 us, 8192 x 2048 44.1 / 25.3, bf16 8192 x 4096 44.5 / 26.3; ordinary loads:
// non-temporal ones lose the line, fused chain of f32 8192 x 512 50 us against 32).
// What is left: f32 8192 x 8, one workgroup, takes 23.7 us, 2.6 ns a row behind the launch.  8192 x 2048 hides its loads
// behind that (24.7); 8192 x 4096 does not, 33.6 us, 4.0 TB/s in 64-byte pieces of rows 16 KiB apart (rows of 16000 bytes 29.1).
#ifndef IMEX_HIP_COLUMN_CHAIN_H
#define IMEX_HIP_COLUMN_CHAIN_H

#include "device_common.h"

namespace imexhip {

// Lanes per row segment (of 8 bytes each), by the 32-byte segments of a row.  Chains on one CU get in each other's way
// (their additions fill a SIMD each, whether 8 or 64 lanes have a column), so: the narrowest segments of which every CU
// gets one.  f32 sums of 8192 x 256 25.1 us with 4 lanes, 26.6 with 8, 29.5 with 16; 6481 x 2832 40.4, 21.9, 23.8; 964 x
// 26136 61.8, 37.6, 27.0.
__device__ __forceinline__ int chain_lanes(int64_t segments) { return segments <= 256 ? 4 : segments <= 512 ? 8 : 16; }
// Eight workers where a CU gets one segment of 128 bytes (f16 sums of 5914 x 13936: 45.3 us with four, 31.8 with eight),
// four where it gets more of them, so that these share it (128 x 32768: 6.5 with eight, 3.9 with four).
__device__ __forceinline__ int wide_chain_workers(int64_t segments) { return segments <= 4 * 256 ? 8 : 4; }

// Whether a matrix of 64-byte segments is taken three tiles ahead: from 84 MiB on, a third of the 256 MiB cache, where
// matrices in use together come from HBM (three in turn: from 92 MB on 0.91 .. 1.00 of the time with one tile, to 82 MB 1.00 ..
// 1.15).
__device__ __forceinline__ bool ahead_of(int64_t rows, int64_t pitch) { return rows * pitch >= int64_t(84) << 20; }

// What the chains take: a tile's rows -- 64 where a row has more than 1024 segments, 512 at most -- within 32-bit offsets of
// its first one.
template <io::Dt D> __device__ __forceinline__ bool chains_take(int64_t rows, int64_t cols) {
  return rows > 0 && cols > 0 && cols * io::Elem<D>::kBytes < int64_t(1) << 26 && rows < int64_t(1) << 31;
}

// blockDim.x of a launch by workgroups that are all of one size, as one scalar load of the kernel's hidden arguments (whose
// layout is the code object's, version 5): blockDim.x itself is a vector load that every wavefront waits for before it
// knows its form, 0.2 .. 0.3 us of a launch (fused chain of bf16 26 x 880 3.54 -> 3.28 us, f16 105 x 328 4.15 -> 3.87).
__device__ __forceinline__ int lanes_launched() {
  return ((const uint32_t *)__builtin_amdgcn_implicitarg_ptr())[3] & 0xffff;
}

// kInputs matrices; kLanes lanes of a worker cover a row's segment with 8 bytes each; kWorkers wavefronts of workers.
template <io::Dt D, int kInputs_, int kLanes_, int kWorkers_, int kAhead_ = 1> struct ColumnChain {
  using E = io::Elem<D>;
  static constexpr int kInputs = kInputs_, kLanes = kLanes_, kWorkers = kWorkers_;
  static constexpr int kPer = 8 / E::kBytes;                    // columns per lane
  static constexpr int kCols = kLanes * kPer;                   // columns per workgroup, a lane of the adder each
  static constexpr int kRowsPerWave = 4 * (kWave / kLanes);     // rows of a tile that one worker wavefront takes
  static constexpr int kTileRows = kWorkers * kRowsPerWave;
  static constexpr int kThreads = (kWorkers + 1) * kWave;
  // Tiles whose loads are in flight while one is evaluated.  Three for 64-byte segments of one input from HBM, of which a CU
  // has one workgroup: one 8 KiB tile at a time left it waiting for memory, f32 7449 x 3680 27.4 us, 25.2 so, bf16 8192 x 8000
  // 31.6 / 29.1 (five: 30.2).  One where the caches have the matrix (ahead_of): f32 3745 x 4096 13.8, with three 14.5, f16 1261
  // x 8192 6.4 / 7.0, 126 problems under 50 MB 1.06 times as long with three in the mean.  One elsewhere: 32-byte segments wait
  // for their additions (4041 x 1792 13.3, with three 14.2), 128-byte ones of whole 4 KiB rows ask too much of the same channels
  // (8192 x 8192 45.7 / 50.9, of other pitches 5 % faster), several workgroups on a CU have tiles of each other's in flight
  // (8192 x 12000 65.0 / 75.1) and two inputs take the registers (fused chain of f32 1500 x 2048 9.1 / 10.0).
  static constexpr int kAhead = kAhead_;
  static constexpr bool kNarrow = kLanes == 4; // takes rows of less than a segment too
  // Floats from one column of a tile to the next, and where a column keeps its rows: four rows (a "quad") are 16 bytes,
  // and quad q of a column that lane group j wrote is at place q ^ swizzle(j) within its four.  128-bit LDS accesses
  // are served sixteen lanes at a time over 64 banks.  The adder's sixteen lanes read one quad of sixteen columns:
  // conflict-free with 4 words (modulo 64) from column to column, and with 8 where there are eight columns.  A worker's
  // sixteen lanes write 16 / kLanes quads of min(16, kLanes) column groups, kPer columns apart: 4 kPer words (or 16), and
  // groups that meet after 16 / kPer of them (there are no more than four per place) trade quads.
  static constexpr int kPad = kCols <= 8 ? 8 : 4;
  static constexpr int kPitch = kTileRows + kPad;
  static constexpr bool kSwizzled = kLanes * kPer > 16;
  static __device__ __forceinline__ int swizzle(int group) {
    return kSwizzled ? group * kPer / 16 * (kLanes < 16 ? 16 / kLanes : 1) : 0;
  }
  static constexpr int kTileFloats = kCols * kPitch;
  static constexpr int kLdsFloats = 2 * kTileFloats;
  static_assert(kLanes < 16 || kWorkers > 4 || kTileRows <= 64, "chains_take");
  static_assert(kCols <= kWave && kTileRows % 64 == 0 && kTileRows <= 512, "a lane per column; the adder takes sixteen rows at a time, four deep");

  typedef uint32_t Raw __attribute__((ext_vector_type(2), aligned(2))); // at any element's address
  struct Tile {
    Raw v[kInputs][4];
  };

  // kShort: rows of fewer than 8 bytes, which a lane's loads run past: what it finds there is never stored, and at the
  // matrix's end it loads the last 8 bytes instead and moves its row's to the front.  (Rows of 8 .. 31 bytes: lanes whose
  // columns would lie past the end take the row's last ones once more.)  f32 sums of 8192 x 4 24.9 us, with a lane per column
  // 222; 100000 x 1 266, 1766; bf16 8192 x 8 26.1, 335; fused chain, four columns per workgroup before, f16 9124 x 8 84 -> 34.
  // prologue(): run by every thread while the first loads are in flight; what it leaves in LDS is there for eval.
  // eval(const Raw (&words)[kInputs][4], float (&f)[4][kPer]): four rows' values of this lane's columns.
  template <bool kShort = false, typename Prologue, typename Eval>
  static __device__ __forceinline__ void run(const void *a, const void *b, void *out, int64_t rows, int64_t cols, float init,
                                             float *lds, Prologue prologue, Eval eval) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t pitch = static_cast<uint32_t>(cols * E::kBytes);
    const int tiles = static_cast<int>((rows + kTileRows - 1) / kTileRows);
    const int lastRows = static_cast<int>(rows - int64_t(tiles - 1) * kTileRows); // of the last tile
    const uint32_t blocks = static_cast<uint32_t>((cols + kCols - 1) / kCols);
    // Each role walks the blocks in a loop of its own: in one loop around both, the compiler keeps a role's addresses and
    // tiles in registers under the other role, 16 of the f32 sums' 109 and 13 of the bf16 fused chain's 135.  Four
    // workgroups of five wavefronts on a CU leave a wavefront 96 -- f32 sums of 128 x 32768 8.0 us with three of them, 5.7
    // so -- and three 128: fused chain of f16 1606 x 17080 48.5, 33.8; bf16 382 x 47034 21.7, 16.9.
    const int lane = threadIdx.x & (kWave - 1);
    auto for_blocks = [&](auto &&role) {
      bool first = true;
      for (uint32_t w = blockIdx.x; w < blocks; w += gridDim.x) {
        // Workgroup w runs on XCD w % 8: the XCDs take contiguous shares of the segments.  (The last block of columns
        // starts early enough to be whole.  The columns that it shares with the block before it are stored by that one
        // only, and what it reads of them is not used: so the result may lie in a row of the matrix itself.)
        const uint32_t xcd = w % 8, block = xcd * (blocks / 8) + min(xcd, blocks % 8) + w / 8;
        const int64_t c0 = min(block * kCols, static_cast<uint32_t>(kNarrow ? max(cols, int64_t(kCols)) : cols) - kCols);
        role(block, c0, first);
        first = false;
        handover(); // both tiles are free for the next block of columns
      }
    };
    if (wave < kWorkers) {
      for_blocks([&](uint32_t, int64_t c0, bool first) {
        const int quad = wave * (kWave / kLanes) + lane / kLanes; // rows 4 quad .. 4 quad + 3 of a tile
        const int col = kShort ? 0 : kNarrow ? min((lane % kLanes) * kPer, static_cast<int>(cols) - kPer) : (lane % kLanes) * kPer;
        const char *base[2] = {static_cast<const char *>(a) + c0 * E::kBytes, static_cast<const char *>(b) + c0 * E::kBytes};
        const uint32_t at = static_cast<uint32_t>(4 * quad) * pitch;
        const int64_t end = rows * int64_t(pitch) - 8; // kShort: the last address of a load
        auto load = [&](int t, Tile &tile) { // tiles past the end: the last one again, never evaluated
          const bool last = t >= tiles - 1;
          const int64_t start = int64_t(last ? tiles - 1 : t) * kTileRows * int64_t(pitch);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            // rows past the end re-read the last one; they are never added
            const uint32_t row = last ? static_cast<uint32_t>(min(4 * quad + i, lastRows - 1)) * pitch : at + i * pitch;
#pragma unroll
            for (int n = 0; n < kInputs; ++n)
              tile.v[n][i] = *reinterpret_cast<const Raw *>(base[n] + (kShort ? min(start + row, end) : start + (row + col * E::kBytes)));
          }
        };
        auto put = [&](int t, Tile &tile) {
          if (t < tiles - 1 || 4 * (quad - lane / kLanes) < lastRows) { // uniform: a wavefront wholly past the end has nothing to do
            float *dst = lds + (t & 1) * kTileFloats + col * kPitch + 4 * (quad ^ swizzle(lane % kLanes));
            float f[4][kPer];
            if constexpr (kShort) {
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const int64_t past = min(int64_t(t) * kTileRows + 4 * quad + i, rows - 1) * pitch - end;
#pragma unroll
                for (int n = 0; n < kInputs; ++n)
                  if (past > 0)
                    tile.v[n][i] = __builtin_bit_cast(Raw, __builtin_bit_cast(uint64_t, tile.v[n][i]) >> (past * 8));
              }
            }
            eval(tile.v, f);
            // Sixteen rows are added or none: -0 behind the last one leaves a sum as it is, whatever it is.
            if (t == tiles - 1) { // uniform
#pragma unroll
              for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int e = 0; e < kPer; ++e)
                  f[i][e] = 4 * quad + i < lastRows ? f[i][e] : -0.0f;
            }
#pragma unroll
            for (int e = 0; e < kPer; ++e)
              *reinterpret_cast<f32x4 *>(dst + e * kPitch) = f32x4{f[0][e], f[1][e], f[2][e], f[3][e]};
          }
          handover(); // tile t is complete; the adder is done with tile t - 1, whose place tile t + 1 goes to
        };
        Tile ring[kAhead + 1]; // the loads of kAhead tiles are on their way while the one before them is evaluated
#pragma unroll
        for (int i = 0; i < kAhead; ++i)
          load(i, ring[i]);
        if (first) {
          prologue();
          handover();
        }
        // (whole rounds as one straight line: the loads in flight at every wait are then known exactly)
        int t = 0;
        for (; t + kAhead < tiles; t += kAhead + 1) {
#pragma unroll
          for (int i = 0; i <= kAhead; ++i) {
            load(t + i + kAhead, ring[(i + kAhead) % (kAhead + 1)]);
            put(t + i, ring[i]);
          }
        }
#pragma unroll
        for (int i = 0; i < kAhead; ++i)
          if (t + i < tiles) // uniform
            put(t + i, ring[i]);
      });
    } else {
      for_blocks([&](uint32_t block, int64_t c0, bool first) {
        if (first) {
          prologue();
          handover();
        }
        __builtin_amdgcn_s_setprio(3); // the chain is the critical path
        const int col = lane % kCols;
        float acc = init;
        // Four groups of sixteen rows in registers: while one is added, the three after it are on their way.
        typedef __attribute__((address_space(3))) const float LdsFloat;
        typedef __attribute__((address_space(3))) const f32x4 LdsVec;
        f32x4 x[4][4];
        LdsFloat *place[4]; // of the first four quads of the 64 rows that are read
        auto start = [&](int t) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            place[q] = (LdsFloat *)lds + (t & 1) * kTileFloats + col * kPitch + 4 * (q ^ swizzle(col / kPer));
        };
        auto read = [&](int g, int at = 0) { // the g-th group of the 64 rows `at` rows on
#pragma unroll
          for (int q = 0; q < 4; ++q)
            x[g][q] = *(LdsVec *)(place[q] + at + g * 16);
          __builtin_amdgcn_sched_barrier(0);
        };
        auto add = [&](int g) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            acc = acc + x[g][q].x;
            acc = acc + x[g][q].y;
            acc = acc + x[g][q].z;
            acc = acc + x[g][q].w;
          }
          __builtin_amdgcn_sched_barrier(0);
        };
        auto landed = [] { // all reads but those of the three youngest groups: one wait per group, not one per read
          __builtin_amdgcn_s_waitcnt(0xc07f | 12 << 8);
          __builtin_amdgcn_sched_barrier(0);
        };
        start(0);
        handover(); // tile 0 is complete
        read(0);
        read(1);
        read(2);
        for (int t = 0; t + 1 < tiles; ++t) {
#pragma unroll
          for (int at = 0; at < kTileRows; at += 64) {
            read(3, at);
            landed();
            add(0);
            if (at + 64 == kTileRows) {
              handover(); // everything of tile t is in registers; tile t + 1 is complete
              start(t + 1);
            }
            const int next = (at + 64) % kTileRows;
            read(0, next);
            landed();
            add(1);
            read(1, next);
            landed();
            add(2);
            read(2, next);
            landed();
            add(3);
          }
        }
        int left = lastRows;
#pragma unroll 1
        for (; left >= 64; left -= 64) {
          read(3);
          landed();
          add(0);
          if (left > 64) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
              place[q] += 64;
          }
          read(0); // (past the last row: some rows again, not added)
          landed();
          add(1);
          read(1);
          landed();
          add(2);
          read(2);
          landed();
          add(3);
        }
        read(3);
#pragma unroll
        for (int g = 0; g < 4; ++g)
          if (left > 16 * g) // uniform; what the last of them has past the end is -0
            add(g);
        __builtin_amdgcn_s_setprio(0);
        if (lane < kCols && c0 + lane >= int64_t(block) * kCols && (!kNarrow || lane < cols))
          E::put(out, c0 + lane, acc);
      });
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

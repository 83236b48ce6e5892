// Fused element-wise chains of the reference's kLoopFusion / kInputFusion
// benchmarks, each as ONE pass over HBM.
//
// Reference op bodies:
//   benchmarks/kLoopFusion/kLoopFusion.mlir.in:4-30
//       t1 = log(a); t2 = |b|; t3 = t1 + t2; out = t3 - a          (four generics,
//       three full-size temporaries in the reference's lowering)
//   benchmarks/kInputFusion/kInputFusion.mlir.in:6-40
//       t = log(b) + |a|  (same first three generics, on swapped arguments), then
//       out[j] = 0 + sum_i t[i][j]: a reduction over the ROWS, one output per
//       column, added in ascending i (indexing maps (d1,d0) -> (d0), :29-39).
//
// Every operation is a separately rounded f32 one, as in the reference; log is
// the host libm's logf (benchmarks/pipelines/linalg-to-cpu.pp:18-19 lowers
// math.log to it), restated below so that the device lands on the same bits.
// 16-bit variants widen to f32, run the same chain and round once at the end
// (the policy the reference applies to 16-bit types on the GPU,
// docs/Transforms/BF16ToGpu.md:17-26).
//
// Arguments:  loop fusion  (a, b, out, n: i64)              dims = {n}
//             input fusion (a, b, out, rows: i64, cols: i64) dims = {rows, cols}
// Launch: block (256,1,1); loop fusion grid ceil(n / 4096) (f32) or ceil(n / 8192)
// (16-bit), a quarter of that per workgroup below 4 Mi elements.  Input fusion, by shape: below 4096 columns
// block (320,1,1), grid ceil(cols / 4); from 2048 rows and 128 row segments of 128 bytes on block (576,1,1),
// grid ceil(cols * element bytes / 128); otherwise block (256,1,1), grid ceil(cols / c), a workgroup per
// block of c = 64 .. 8 columns (the widest that leaves 512 workgroups).  A launch with 256 lanes always gets
// the last form, one with fewer a lane per column.  The _tall forms, by the 32-byte segments of a row (chain_lanes in
// column_chain.h): up to 256 block (320,1,1), up to 1024 (576,1,1), beyond that (320,1,1); grid a workgroup per segment
// of 32, 64 (257 .. 512) or 128 bytes, of 16 where half_segments() says so.  With any other block they go as the forms with 256 lanes or fewer.  Workgroups
// stride, so any grid is correct.

#include "column_chain.h"
#include "device_common.h"

using namespace imexhip;
using namespace imexhip::io;

namespace {

constexpr int kThreads = 256;

// ---------------------------------------------------------------------------
// logf as glibc computes it (Arm Optimized Routines logf: x = 2^k z with z in
// [0x3f330000, ...), c = table centre of z's 1/16 sub-interval, r = z/c - 1,
// log x = k ln2 + log c + r + r^2 (A2 + A1 r + A0 r^2); all in f64 with IEEE
// operations, one final rounding).  A host build of this function agrees with
// libm's logf on every positive finite f32, with its products and sums rounded
// separately and fused: fused it is five f64 instructions shorter.
// ---------------------------------------------------------------------------
struct alignas(16) LogfEntry {
  double invc, logc;
};
__device__ const LogfEntry kLogfTable[16] = {
    {0x1.661ec79f8f3bep+0, -0x1.57bf7808caadep-2}, {0x1.571ed4aaf883dp+0, -0x1.2bef0a7c06ddbp-2},
    {0x1.49539f0f010bp+0, -0x1.01eae7f513a67p-2},  {0x1.3c995b0b80385p+0, -0x1.b31d8a68224e9p-3},
    {0x1.30d190c8864a5p+0, -0x1.6574f0ac07758p-3}, {0x1.25e227b0b8eap+0, -0x1.1aa2bc79c81p-3},
    {0x1.1bb4a4a1a343fp+0, -0x1.a4e76ce8c0e5ep-4}, {0x1.12358f08ae5bap+0, -0x1.1973c5a611cccp-4},
    {0x1.0953f419900a7p+0, -0x1.252f438e10c1ep-5}, {0x1p+0, 0x0p+0},
    {0x1.e608cfd9a47acp-1, 0x1.aa5aa5df25984p-5},  {0x1.ca4b31f026aap-1, 0x1.c5e53aa362eb4p-4},
    {0x1.b2036576afce6p-1, 0x1.526e57720db08p-3},  {0x1.9c2d163a1aa2dp-1, 0x1.bc2860d22477p-3},
    {0x1.886e6037841edp-1, 0x1.1058bc8a07ee1p-2},  {0x1.767dcf5534862p-1, 0x1.4043057b6ee09p-2},
};

// The arithmetic of logf on the bits of a positive normal number (libm's main path), before its one rounding to f32.
constexpr double kLn2 = 0x1.62e42fefa39efp-1;
__device__ __forceinline__ double logf_libm_core(uint32_t ix, const LogfEntry *table) {
  const uint32_t tmp = ix - 0x3f330000u;
  const int i = (tmp >> 19) & 15;
  const int k = static_cast<int32_t>(tmp) >> 23;
  const uint32_t iz = ix - (tmp & 0xff800000u);
  const double invc = table[i].invc, logc = table[i].logc;
  const double z = static_cast<double>(u2f(iz));
  const double r = __builtin_fma(z, invc, -1.0);
  const double y0 = __builtin_fma(static_cast<double>(k), kLn2, logc);
  const double r2 = r * r;
  double y = __builtin_fma(0x1.5575b0be00b6ap-2, r, -0x1.ffffef20a4123p-2);
  y = __builtin_fma(-0x1.00ea348b88334p-2, r2, y);
  return __builtin_fma(y, r2, y0 + r);
}

// Positive, normal and finite: what libm sends down its main path, and 1.0, for which that path gives its +0 too.
__device__ __forceinline__ bool logf_ordinary(float x) { return f2u(x) - 0x00800000u < 0x7f800000u - 0x00800000u; }

// Any x, without a branch: libm's special cases are selected at the end.
__device__ __forceinline__ float logf_libm(float x, const LogfEntry *table) {
  const uint32_t ix = f2u(x);
  const uint32_t normal = ix < 0x00800000u ? f2u(x * 0x1p23f) - (23u << 23) : ix; // subnormals: normalised
  float y = static_cast<float>(logf_libm_core(normal, table));
  y = ix >= 0x7f800000u ? u2f(0xffc00000u) : y; // log of a negative number: libm's (x - x) / 0, the x86 default NaN
  y = ix == 0x7f800000u ? x : y;                // log(inf)
  y = ix * 2 > 0xff000000u ? x + x : y;         // NaN: quieted, sign and payload kept
  return ix * 2 == 0 ? -__builtin_inff() : y;   // log(+-0)
}

// The logarithms of a kernel, with what they need in LDS.  kMantissa is 0 for any f32.  A value widened from a 16-bit
// type has a mantissa of 7 (bf16) or 10 (f16) bits, and log x = k ln2 + log m: the f64 logarithms of all 128 (1024)
// mantissas, from the arithmetic above, leave one fused multiply-add and the rounding per element, where the general
// form has twelve f64 instructions and conversions (a host build agrees with libm's logf on every bf16 and f16 value).
// Without them the logarithms bound the 16-bit chains: loop fusion of 64 M bf16 78.3 -> 64.0 us (6.0 TB/s), of 11.3 M
// 20.5 -> 15.1, of 4.6 M f16 11.2 -> 8.7.
template <int kMantissa> struct Logarithms {
  LogfEntry entry[16];
  double mantissa[kMantissa ? 1 << kMantissa : 1];

  // by all threads of the workgroup, 16 or more; readable after a barrier
  __device__ __forceinline__ void stage() {
    if (threadIdx.x < 16)
      entry[threadIdx.x] = kLogfTable[threadIdx.x];
    if constexpr (kMantissa != 0)
      for (uint32_t m = threadIdx.x; m < 1u << kMantissa; m += lanes_launched())
        mantissa[m] = logf_libm_core(0x3f800000u | m << (23 - kMantissa), kLogfTable);
  }
  // kOrdinary: the caller has checked logf_ordinary() in every lane of the wavefront, so that this is straight-line code
  // (libm's special cases cost a masked region per element, which keeps the f64 chains of a vector's elements from
  // interleaving).
  template <bool kOrdinary> __device__ __forceinline__ float of(float x) const {
    if constexpr (!kOrdinary)
      return logf_libm(x, entry);
    else if constexpr (kMantissa == 0)
      return static_cast<float>(logf_libm_core(f2u(x), entry));
    const uint32_t ix = f2u(x);
    const double k = static_cast<int32_t>(ix >> 23) - 127;
    return static_cast<float>(__builtin_fma(k, kLn2, mantissa[ix >> (23 - kMantissa) & ((1u << kMantissa) - 1)]));
  }
};
template <Dt D> constexpr int kMantissaOf = D == Dt::F32 ? 0 : D == Dt::F16 ? 10 : 7;

// the chains, on f32 values
template <bool kOrdinary = false, typename Logs>
__device__ __forceinline__ float loop_chain(float a, float b, const Logs &logs) {
  const float t1 = logs.template of<kOrdinary>(a);
  const float t2 = __builtin_fabsf(b);
  const float t3 = t1 + t2;
  return t3 - a;
}
template <bool kOrdinary = false, typename Logs>
__device__ __forceinline__ float input_chain(float a, float b, const Logs &logs) {
  const float t1 = logs.template of<kOrdinary>(b);
  const float t2 = __builtin_fabsf(a);
  return t1 + t2;
}

// Elem<Dt>: element access, 16-byte vector unpack / pack to f32 (device_common.h).

// ---- kLoopFusion: two streams in, one out ------------------------------------------
// kVecs 16-byte vectors per lane and pass: four for tensors that stream from HBM, one for small
// ones, where the logarithms of a lane are the critical path and spreading them over more
// workgroups is what shortens it.
constexpr int64_t kSmallFusion = int64_t(1) << 22; // elements

template <Dt D, int kVecs, typename Logs>
__device__ __forceinline__ void loop_fusion_pass(const void *__restrict__ a, const void *__restrict__ b,
                                                 void *__restrict__ out, int64_t n, const Logs &logs) {
  using E = Elem<D>;
  constexpr int kVecsPerThread = kVecs;
  constexpr int64_t kElemsPerBlock = int64_t(kThreads) * kVecsPerThread * E::kPerVec;
  const bool aligned = ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) |
                         reinterpret_cast<uintptr_t>(out)) & 15) == 0;
  // workgroups stride over the blocks, so any grid covers n
  for (int64_t base = int64_t(blockIdx.x) * kElemsPerBlock; base < n; base += int64_t(gridDim.x) * kElemsPerBlock) {
    const u32x4 *pa = reinterpret_cast<const u32x4 *>(static_cast<const char *>(a) + base * E::kBytes);
    const u32x4 *pb = reinterpret_cast<const u32x4 *>(static_cast<const char *>(b) + base * E::kBytes);
    u32x4 *po = reinterpret_cast<u32x4 *>(static_cast<char *>(out) + base * E::kBytes);
    u32x4 va[kVecsPerThread], vb[kVecsPerThread];
    auto result = [&](int j) {
      float fa[E::kPerVec], fb[E::kPerVec];
      E::unpack(va[j], fa);
      E::unpack(vb[j], fb);
      bool ordinary = true;
#pragma unroll
      for (int i = 0; i < E::kPerVec; ++i)
        ordinary = ordinary && logf_ordinary(fa[i]);
      if (__builtin_amdgcn_ballot_w64(!ordinary) == 0) { // uniform over the wavefront
#pragma unroll
        for (int i = 0; i < E::kPerVec; ++i)
          fa[i] = loop_chain<true>(fa[i], fb[i], logs);
      } else {
#pragma unroll
        for (int i = 0; i < E::kPerVec; ++i)
          fa[i] = loop_chain(fa[i], fb[i], logs);
      }
      return E::pack(fa);
    };
    if (aligned && base + kElemsPerBlock <= n) {
#pragma unroll
      for (int j = 0; j < kVecsPerThread; ++j) {
        va[j] = load128<true>(pa + j * kThreads + threadIdx.x);
        vb[j] = load128<true>(pb + j * kThreads + threadIdx.x);
      }
#pragma unroll
      for (int j = 0; j < kVecsPerThread; ++j)
        store128<true>(result(j), po + j * kThreads + threadIdx.x);
    } else if (aligned) {
      // The last block: lanes past its last vector take that one again, and their results go nowhere.  (Element by element
      // it was up to 32 loads and chains one after the other, which the whole launch waited for: bf16 4701392 11.5 -> 8.2 us.)
      const int vecs = static_cast<int>((n - base) / E::kPerVec), lane = static_cast<int>(threadIdx.x);
      if (vecs > 0) {
#pragma unroll
        for (int j = 0; j < kVecsPerThread; ++j) {
          va[j] = load128<true>(pa + min(j * kThreads + lane, vecs - 1));
          vb[j] = load128<true>(pb + min(j * kThreads + lane, vecs - 1));
        }
#pragma unroll
        for (int j = 0; j < kVecsPerThread; ++j)
          if (j * kThreads + __builtin_amdgcn_readfirstlane(lane) < vecs) { // uniform
            const u32x4 r = result(j);
            if (j * kThreads + lane < vecs)
              store128<true>(r, po + j * kThreads + lane);
          }
      }
      const int64_t i = base + int64_t(vecs) * E::kPerVec + lane;
      if (i < n)
        E::put(out, i, loop_chain(E::get(a, i), E::get(b, i), logs));
    } else {
      for (int64_t i = base + threadIdx.x; i < base + kElemsPerBlock && i < n; i += kThreads)
        E::put(out, i, loop_chain(E::get(a, i), E::get(b, i), logs));
    }
  }
}

template <Dt D>
__device__ __forceinline__ void loop_fusion(const void *__restrict__ a, const void *__restrict__ b,
                                            void *__restrict__ out, int64_t n) {
  __shared__ Logarithms<kMantissaOf<D>> logs;
  if (n < kSmallFusion) {
    // (f16: 1024 mantissas are as many logarithms as a workgroup of 2048 elements saves)
    if constexpr (D == Dt::F16) {
      __shared__ Logarithms<0> plain;
      plain.stage();
      __syncthreads();
      loop_fusion_pass<D, 1>(a, b, out, n, plain);
    } else {
      logs.stage();
      __syncthreads();
      loop_fusion_pass<D, 1>(a, b, out, n, logs);
    }
    return;
  }
  logs.stage();
  __syncthreads();
  loop_fusion_pass<D, 4>(a, b, out, n, logs);
}

// ---- kInputFusion: chain + column sums ------------------------------------------------
// out[j] = sum over rows i, in ascending order from +0.0, of chain(a[i,j], b[i,j]) -- the
// reference's order of additions, so the f32 result is the same bits.  Only the additions are
// ordered; the chain (a logarithm per element) is not.  A workgroup owns kCols adjacent columns
// and walks the rows in tiles of 4096 / kCols: all 256 lanes evaluate the chain of a tile into
// LDS (coalesced along the rows), then lane j < kCols adds column j's values of the tile to its
// running sum, in row order.  The tile is double-buffered, so the ordered additions of one tile
// run under the loads and logarithms of the next, with one barrier per tile.  Short matrices
// (up to 1024 rows, the reference's 512 x 1024 among them) use tiles of 1024 elements, so that
// there is a next tile to overlap with; tall ones are faster with fewer barriers.
constexpr int kTileElems = 4096, kSmallTileElems = 1024;

// acc + t[0] + t[stride] + ... + t[(n-1) stride], added in that order: sixteen LDS reads are in flight
// while the previous sixteen values are added.
__device__ __forceinline__ float add_in_row_order(float acc, const float *t, int n, int stride) {
  float v[16], w[16];
  int r = 0;
  if (n >= 16) {
#pragma unroll
    for (int u = 0; u < 16; ++u)
      v[u] = t[u * stride];
    for (r = 16; r + 16 <= n; r += 16) {
#pragma unroll
      for (int u = 0; u < 16; ++u)
        w[u] = t[(r + u) * stride];
#pragma unroll
      for (int u = 0; u < 16; ++u)
        acc = acc + v[u];
#pragma unroll
      for (int u = 0; u < 16; ++u)
        v[u] = w[u];
    }
#pragma unroll
    for (int u = 0; u < 16; ++u)
      acc = acc + v[u];
  }
  for (; r < n; ++r)
    acc = acc + t[r * stride];
  return acc;
}

// A lane per column, for launches with fewer lanes than the tiles below are filled by.
template <Dt D, typename Logs>
__device__ __forceinline__ void input_fusion_by_element(const void *__restrict__ a, const void *__restrict__ b,
                                                        void *__restrict__ out, int64_t rows, int64_t cols, Logs &logs) {
  using E = Elem<D>;
  for (int i = threadIdx.x; i < 16; i += lanes_launched())
    logs.entry[i] = kLogfTable[i];
  __syncthreads();
  for (int64_t c = int64_t(blockIdx.x) * lanes_launched() + threadIdx.x; c < cols; c += int64_t(gridDim.x) * lanes_launched()) {
    float acc = 0.0f;
    for (int64_t r = 0; r < rows; ++r)
      acc = acc + input_chain(E::get(a, r * cols + c), E::get(b, r * cols + c), logs);
    E::put(out, c, acc);
  }
}

template <Dt D, int kCols, int kTileElems = ::kTileElems, typename Logs>
__device__ __forceinline__ void input_fusion_cols(const void *__restrict__ a, const void *__restrict__ b,
                                                  void *__restrict__ out, int64_t rows, int64_t cols,
                                                  const Logs &logs, float *tile) {
  using E = Elem<D>;
  constexpr int kTileRows = kTileElems / kCols;
  constexpr int kPerLane = kTileElems / kThreads;
  const int tid = threadIdx.x;
  const bool worker = tid < kThreads; // a launch with more lanes: the others only take part in the barriers
  for (int64_t c0 = int64_t(blockIdx.x) * kCols; c0 < cols; c0 += int64_t(gridDim.x) * kCols) {
    float acc = 0.0f;
    int buf = 0;
    for (int64_t r0 = 0; r0 < rows; r0 += kTileRows, buf ^= 1) {
      float *t = tile + buf * kTileElems;
      float xa[kPerLane], xb[kPerLane];
#pragma unroll
      for (int u = 0; u < kPerLane; ++u) {
        const int e = u * kThreads + tid;
        const int64_t r = r0 + e / kCols, c = c0 + e % kCols;
        const bool ok = worker && r < rows && c < cols;
        xa[u] = ok ? E::get(a, r * cols + c) : 2.0f; // positions outside the matrix: any ordinary value, never added
        xb[u] = ok ? E::get(b, r * cols + c) : 2.0f;
      }
      bool ordinary = true;
#pragma unroll
      for (int u = 0; u < kPerLane; ++u)
        ordinary = ordinary && logf_ordinary(xb[u]);
      if (__builtin_amdgcn_ballot_w64(!ordinary) == 0) { // uniform over the wavefront
#pragma unroll
        for (int u = 0; u < kPerLane; ++u)
          if (worker && r0 + (u * kThreads) / kCols < rows) // passes that lie wholly below the last row are skipped
            t[u * kThreads + tid] = input_chain<true>(xa[u], xb[u], logs);
      } else {
#pragma unroll
        for (int u = 0; u < kPerLane; ++u)
          if (worker && r0 + (u * kThreads) / kCols < rows)
            t[u * kThreads + tid] = input_chain(xa[u], xb[u], logs);
      }
      __syncthreads(); // the tile is complete; the other buffer was consumed before the previous barrier
      if (tid < kCols && c0 + tid < cols) {
        const int n = rows - r0 < kTileRows ? int(rows - r0) : kTileRows;
        acc = add_in_row_order(acc, t + tid, n, kCols);
      }
    }
    if (tid < kCols && c0 + tid < cols)
      E::put(out, c0 + tid, acc);
    __syncthreads(); // both buffers are free for the next block of columns
  }
}

// ---- kInputFusion on narrow matrices: the streaming form ------------------------------------
// With 4 columns per workgroup the form above reads 16-byte row segments, computes and adds in turn, and is bound by
// memory latency.  Here 256 workers + one adder wavefront = 320 lanes own 4 columns, one element per lane and access, 64
// rows per tile (a lane's first result is ready after ONE chain), the loads of eight tiles -- 512 rows -- in flight
// together.  The next group's loads are issued before this group's chains are evaluated; the results go into one of two
// LDS tiles.  The fifth wavefront does nothing but the ordered additions, one lane per column, a tile behind the
// workers: one barrier per tile, passed by everybody, hands a tile over and returns the other one.  The ordered additions
// are the critical path (a lone wavefront issues a dependent addition every ~8 cycles), and what this form buys is that
// nothing else is ever on it.  Taller matrices go by column chains (below).
constexpr int kNarrowWorkers = 256, kNarrowThreads = kNarrowWorkers + 64;
constexpr int kNarrowCols = 4, kNarrowRows = kNarrowWorkers / kNarrowCols, kNarrowTilesAhead = 8;
// A tile lies in LDS COLUMN by column, and row r of column c sits at position r ^ 4 c: the adder still reads four
// consecutive rows of its column with one 128-bit access.  A 32-bit write is served 32 lanes at a time (0-31, 32-63) over
// banks that repeat every 32 words: eight rows of four columns, of which the pitch (16 modulo 32 words) puts odd and even
// ones 16 banks apart and the swizzle the two of a kind 8.
constexpr int kNarrowPitch = kNarrowRows + 16, kNarrowTileFloats = kNarrowCols * kNarrowPitch;
// 576 lanes, from 2048 rows and 128 row segments of 128 bytes on: column chains of such segments, eight workers
constexpr int kStreamThreads = 576;
constexpr int64_t kStreamFromRows = 2048;

// what the launch and the kernel both decide on: enough column blocks for the chip, enough rows for a pipeline
template <Dt D> __device__ __forceinline__ bool input_fusion_streams(int64_t rows, int64_t cols) {
  return rows >= kStreamFromRows && cols * Elem<D>::kBytes >= 128 * 128;
}
// ... and the narrow form wherever the form above would take four columns per workgroup
__device__ __forceinline__ bool input_fusion_narrow(int64_t cols) { return cols < 8 * 512; }

// acc + c[0] + c[1] + ... + c[n-1], added in that order, for a column c of kNarrowRows consecutive floats
// (16-byte aligned, all of them readable): sixteen rows arrive as four 128-bit LDS reads while the previous
// sixteen are added, so the adder issues 1.25 instructions per row.
// swz: row r is kept at position r ^ swz (a multiple of 4 below 32: blocks of four rows trade places).
__device__ __forceinline__ float add_column_in_row_order(float acc, const float *c, int n, int swz) {
  f32x4 x[4], y[4];
  auto read16 = [&](f32x4(&v)[4], int r) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      v[q] = *reinterpret_cast<const f32x4 *>(c + ((r + 4 * q) ^ swz));
  };
  auto add16 = [&](const f32x4(&v)[4]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      acc = acc + v[q].x;
      acc = acc + v[q].y;
      acc = acc + v[q].z;
      acc = acc + v[q].w;
    }
  };
  int r = 0;
  read16(x, 0);
  for (; r + 32 <= n; r += 32) {
    read16(y, r + 16);
    add16(x);
    read16(x, r + 32 < kNarrowRows ? r + 32 : 0); // past the tile's last row: any readable rows, not added
    add16(y);
  }
  // x holds rows r .. r + 15; fewer than 32 rows are left
  if (r + 16 <= n) {
    read16(y, r + 16);
    add16(x);
    r += 16;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (r + 4 * q + e < n)
          acc = acc + y[q][e];
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (r + 4 * q + e < n)
          acc = acc + x[q][e];
  }
  return acc;
}

// The hand-over of a tile between the worker wavefronts and the adder wavefront.  The two roles run
// different code and meet here from different places, which the hardware barrier allows (it counts
// wavefronts that have arrived, wherever each one arrives from); what makes it correct is that both roles
// pass it exactly once per tile -- `tiles` times per block of columns, the workers after writing tile t,
// the adder before reading it -- and once more together when the block of columns is done.  Written as
// the instruction with the LDS release / acquire around it, not as a call the compiler may treat as
// convergent across the two branches.  The workgroup must be exactly kNarrowThreads lanes (the entry checks).
__device__ __forceinline__ void tile_handover() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

template <Dt D>
__device__ __forceinline__ void input_fusion_stream(const void *__restrict__ a, const void *__restrict__ b,
                                                    void *__restrict__ out, int64_t rows, int64_t cols,
                                                    const Logarithms<0> &logs, float *tile) {
  using E = Elem<D>;
  const int tid = threadIdx.x;
  const int64_t tiles = (rows + kNarrowRows - 1) / kNarrowRows;
  const int64_t groups = (tiles + kNarrowTilesAhead - 1) / kNarrowTilesAhead;
  for (int64_t c0 = int64_t(blockIdx.x) * kNarrowCols; c0 < cols; c0 += int64_t(gridDim.x) * kNarrowCols) {
    if (tid < kNarrowWorkers) {
      const int lr = tid / kNarrowCols, lc = tid % kNarrowCols; // row within a tile, column
      // Rows past the end and, in a partial last block, columns past the end re-read a position inside the
      // matrix instead (their results are never added): the loads are then unconditional, straight-line
      // code, and the wait for a tile's data leaves the next group's loads in flight.
      const int64_t col = c0 + lc < cols ? c0 + lc : c0;
      float ca[kNarrowTilesAhead], cb[kNarrowTilesAhead], na[kNarrowTilesAhead], nb[kNarrowTilesAhead];
      auto load_group = [&](int64_t g, float(&va)[kNarrowTilesAhead], float(&vb)[kNarrowTilesAhead]) {
#pragma unroll
        for (int p = 0; p < kNarrowTilesAhead; ++p) {
          const int64_t r = min((g * kNarrowTilesAhead + p) * kNarrowRows + lr, rows - 1);
          va[p] = E::get(a, r * cols + col);
          vb[p] = E::get(b, r * cols + col);
        }
      };
      if (groups > 0) // (no rows: nothing to read, the sums are +0.0)
        load_group(0, ca, cb);
      for (int64_t g = 0; g < groups; ++g) {
        load_group(g + 1 < groups ? g + 1 : g, na, nb); // past the last group: the last one again, unused
#pragma unroll
        for (int j = 0; j < kNarrowTilesAhead; ++j) {
          const int64_t t = g * kNarrowTilesAhead + j;
          if (t < tiles) { // uniform
            float *dst = tile + (t & 1) * kNarrowTileFloats + lc * kNarrowPitch + (lr ^ 4 * lc);
            if (__builtin_amdgcn_ballot_w64(!logf_ordinary(cb[j])) == 0) // uniform over the wavefront
              *dst = input_chain<true>(ca[j], cb[j], logs);
            else
              *dst = input_chain(ca[j], cb[j], logs);
            tile_handover(); // tile t is complete; the adder is done with tile t-1, whose buffer tile t+1 goes into
          }
        }
#pragma unroll
        for (int p = 0; p < kNarrowTilesAhead; ++p) {
          ca[p] = na[p];
          cb[p] = nb[p];
        }
      }
    } else {
      const int col = tid - kNarrowWorkers;
      const bool active = col < kNarrowCols && c0 + col < cols;
      float acc = 0.0f;
      for (int64_t t = 0; t < tiles; ++t) {
        tile_handover(); // tile t is complete
        const int n = rows - t * kNarrowRows < kNarrowRows ? int(rows - t * kNarrowRows) : kNarrowRows;
        if (active)
          acc = add_column_in_row_order(acc, tile + (t & 1) * kNarrowTileFloats + col * kNarrowPitch, n, 4 * col);
      }
      if (active)
        E::put(out, c0 + col, acc);
    }
    __syncthreads(); // both tiles are free for the next block of columns
  }
}

// ---- kInputFusion by column chains (column_chain.h) -------------------------------------------
// Any number of columns and rows, at any address: the forms above read 4 .. 64 columns of a row per workgroup element by
// element and are bound by the latency of those loads or, 16-bit inputs, by the logarithms.  bf16 5550 x 5932 449 -> 42 us (floor 21 for its
// bytes), f32 3785 x 3480 155 -> 27 (17), f16 1052 x 5433 76 -> 11, f32 8192 x 512 87 -> 31 (the chain alone: 22), f32
// 8192 x 8192 106 -> 91 (85).  Two workers per SIMD on segments of 64 and 128 bytes: one took 29 and 82 us on f16 3785 x
// 3480 and f32 5550 x 5932, two take 19 and 60.
template <Dt D, int kLanes, int kWorkers, bool kShort = false, typename Logs>
__device__ __forceinline__ void input_fusion_chains(const void *__restrict__ a, const void *__restrict__ b,
                                                    void *__restrict__ out, int64_t rows, int64_t cols, Logs &logs, float *lds) {
  using C = ColumnChain<D, 2, kLanes, kWorkers>;
  using E = Elem<D>;
  constexpr int kPer = C::kPer;
  C::template run<kShort>(a, b, out, rows, cols, 0.0f, lds, [&] { logs.stage(); }, [&](const typename C::Raw(&v)[2][4], float(&f)[4][kPer]) {
    float x[4][kPer]; // under the logarithm
    uint32_t least = ~0u, most = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        if constexpr (D == Dt::F32) {
          f[i][w] = u2f(v[0][i][w]);
          x[i][w] = u2f(v[1][i][w]);
        } else {
          f[i][2 * w] = E::widen(v[0][i][w] & 0xffffu);
          f[i][2 * w + 1] = E::widen(v[0][i][w] >> 16);
          x[i][2 * w] = E::widen(v[1][i][w] & 0xffffu);
          x[i][2 * w + 1] = E::widen(v[1][i][w] >> 16);
        }
      }
#pragma unroll
      for (int e = 0; e < kPer; ++e) {
        least = min(least, f2u(x[i][e]));
        most = max(most, f2u(x[i][e]));
      }
    }
    // uniform over the wavefront: all of them logf_ordinary()
    if (__builtin_amdgcn_ballot_w64(least < 0x00800000u || most >= 0x7f800000u) == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < kPer; ++e)
          f[i][e] = input_chain<true>(f[i][e], x[i][e], logs);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < kPer; ++e)
          f[i][e] = input_chain(f[i][e], x[i][e], logs);
    }
  });
}

// Segments of 16 bytes where they still fit one round and the rows are many: with 32 a CU's logarithms, not its additions, set
// the pace (four instructions' cycles for each on four SIMDs, 3.4 .. 4 ns a row against 2.6), and half of the columns are half
// of them: f16 6750 x 448 27.3 -> 22.2 us, bf16 8192 x 1024 32.5 -> 27.0, f32 8192 x 512 31.1 -> 26.6, and of rows of 4 KiB,
// which crowd a few channels, f32 8192 x 1024 53.4 -> 42.5.  Fewer rows wait for the first tile instead: f16 2100 x 1100
// 0.91 of the time, bf16 2100 x 1500 0.96, 1200 x 1500 1.03; f32 5000 x 700 0.92, 2100 x 700 0.98, 900 x 700 1.07.
template <Dt D> __device__ __forceinline__ bool half_segments(int64_t rows, int64_t row) {
  return row >= 32 && row <= 128 * 32 && rows >= (D == Dt::F32 ? 4096 : 2048);
}
// Four workers for segments of 16 and 32 bytes, eight for 64 (wide_chain_workers() for 128).  Other launches, and what the
// chains do not take, go by blocks of columns, or a lane per column.
template <Dt D>
__device__ __forceinline__ void input_fusion_tall(const void *__restrict__ a, const void *__restrict__ b,
                                                  void *__restrict__ out, int64_t rows, int64_t cols) {
  __shared__ __attribute__((aligned(16))) float lds[ColumnChain<D, 2, 16, 8>::kLdsFloats];
  __shared__ Logarithms<kMantissaOf<D>> logs;
  const int64_t row = cols * Elem<D>::kBytes, segments = (row + 31) / 32;
  const int lanes = half_segments<D>(rows, row) ? 2 : chain_lanes(segments);
  const int workers = lanes <= 4 ? 4 : lanes == 8 ? 8 : wide_chain_workers(segments);
  if (!chains_take<D>(rows, cols) || (row < 8 && rows * row < 8) || lanes_launched() != (workers + 1) * kWave) {
    if (lanes_launched() < kThreads) {
      input_fusion_by_element<D>(a, b, out, rows, cols, logs);
      return;
    }
    logs.stage();
    __syncthreads();
    input_fusion_cols<D, 4, kSmallTileElems>(a, b, out, rows, cols, logs, lds);
  } else if (lanes == 2) {
    input_fusion_chains<D, 2, 4>(a, b, out, rows, cols, logs, lds);
  } else if (lanes == 4 && row < 8) {
    input_fusion_chains<D, 4, 4, true>(a, b, out, rows, cols, logs, lds);
  } else if (lanes == 4) {
    input_fusion_chains<D, 4, 4>(a, b, out, rows, cols, logs, lds);
  } else if (lanes == 8) {
    input_fusion_chains<D, 8, 8>(a, b, out, rows, cols, logs, lds);
  } else if (workers == 8) {
    input_fusion_chains<D, 16, 8>(a, b, out, rows, cols, logs, lds);
  } else {
    input_fusion_chains<D, 16, 4>(a, b, out, rows, cols, logs, lds);
  }
}

// Columns per workgroup: as many as still leave every CU a couple of workgroups (wide blocks read
// longer row segments), down to 4.
__device__ __forceinline__ int input_fusion_block_cols(int64_t cols) {
  return cols >= 64 * 512 ? 64 : cols >= 32 * 512 ? 32 : cols >= 16 * 512 ? 16 : cols >= 8 * 512 ? 8 : 4;
}

template <Dt D>
__device__ __forceinline__ void input_fusion(const void *__restrict__ a, const void *__restrict__ b,
                                             void *__restrict__ out, int64_t rows, int64_t cols) {
  constexpr int kLdsFloats = ColumnChain<D, 2, 16, 8>::kLdsFloats;
  static_assert(kLdsFloats >= 2 * kTileElems && kLdsFloats >= 2 * kNarrowTileFloats);
  __shared__ Logarithms<0> logs;
  __shared__ __attribute__((aligned(16))) float tile[kLdsFloats];
  if (lanes_launched() < kThreads) {
    input_fusion_by_element<D>(a, b, out, rows, cols, logs);
    return;
  }
  // The launch says which form.
  if (lanes_launched() == kStreamThreads && chains_take<D>(rows, cols) && input_fusion_streams<D>(rows, cols)) {
    __shared__ Logarithms<kMantissaOf<D>> all;
    input_fusion_chains<D, 16, 8>(a, b, out, rows, cols, all, tile);
    return;
  }
  logs.stage();
  __syncthreads();
  if (lanes_launched() == kNarrowThreads && input_fusion_narrow(cols)) {
    input_fusion_stream<D>(a, b, out, rows, cols, logs, tile);
    return;
  }
  switch (input_fusion_block_cols(cols)) {
  case 64: input_fusion_cols<D, 64>(a, b, out, rows, cols, logs, tile); break;
  case 32: input_fusion_cols<D, 32>(a, b, out, rows, cols, logs, tile); break;
  case 16: input_fusion_cols<D, 16>(a, b, out, rows, cols, logs, tile); break;
  case 8: input_fusion_cols<D, 8>(a, b, out, rows, cols, logs, tile); break;
  default:
    if (rows <= 1024)
      input_fusion_cols<D, 4, kSmallTileElems>(a, b, out, rows, cols, logs, tile);
    else
      input_fusion_cols<D, 4>(a, b, out, rows, cols, logs, tile);
    break;
  }
}

} // namespace

#define IMEX_FUSION_KERNELS(SUFFIX, DT, CTYPE)                                                                       \
  extern "C" __global__ __launch_bounds__(kThreads) void imex_loop_fusion_##SUFFIX(                                  \
      const CTYPE *a, const CTYPE *b, CTYPE *out, int64_t n) {                                                       \
    loop_fusion<DT>(a, b, out, n);                                                                                   \
  }                                                                                                                  \
  extern "C" __global__ __launch_bounds__(kStreamThreads) void imex_input_fusion_##SUFFIX(                                 \
      const CTYPE *a, const CTYPE *b, CTYPE *out, int64_t rows, int64_t cols) {                                      \
    input_fusion<DT>(a, b, out, rows, cols);                                                                         \
  }                                                                                                                  \
  extern "C" __global__ __launch_bounds__(576) void imex_input_fusion_##SUFFIX##_tall(          \
      const CTYPE *a, const CTYPE *b, CTYPE *out, int64_t rows, int64_t cols) {                                      \
    input_fusion_tall<DT>(a, b, out, rows, cols);                                                                    \
  }

IMEX_FUSION_KERNELS(f32, Dt::F32, float)
IMEX_FUSION_KERNELS(f16, Dt::F16, uint16_t)
IMEX_FUSION_KERNELS(bf16, Dt::BF16, uint16_t)

// Sum reductions, f32.
//
//  * imex_rowsum_f32: out[r] = init + sum_c in[r, c]  (row-sum / last-dim form:
//    test/Integration/Dialect/XeGPU/WG/reduction_2D_1D_cross_sg_cross_lane.mlir:31-37,
//    benchmarks/kInputFusion/kInputFusion.mlir.in:29-39).
//    The reference's linalg path runs the whole sum in one work-item
//    (test/SPIRV/OpTest.Sum_FLOAT32.mlir:39); here a workgroup (or a wavefront,
//    for short rows) owns a row, streams it once with 128-bit loads, and
//    combines partial sums with wavefront-64 butterflies and one LDS hop.
//  * imex_reduce_outer_f32 / _f16 / _bf16: out[i] = init + sum_o in[o, i], the OUTERMOST
//    dimension reduced (benchmarks/reduce/reduce_gpu.mlir.in:4-21).  Each lane
//    owns groups of four adjacent outputs and adds the `outer` slices in order,
//    which is the reference's summation order, so this one is bit-exact.
//
//    imex_reduce_outer_*_tall and _deep are the same sums for shapes that leave most of the chip idle in that form.
//
//  * imex_rowmean_f32: out[r] = (0 + sum_c in[r, c]) / cols, the same reduction with the
//    division the reference applies afterwards
//    (WG/reduction_4D_3D_mean_intra_sg_intra_lane.mlir:51-52, 1x24x1024x64 -> 1x24x1024x1).
//
// Arguments: rowsum (in, out, rows: i64, cols: i64, init: f32); rowmean (in, out, rows: i64, cols: i64);
//            reduce_outer (in, out, outer: i64, inner: i64, init: f32).
// Launch: block (256,1,1);
//   rowsum: cols > 2048 -> grid (rows,1,1) [workgroup per row],
//           else grid (ceil(rows/4),1,1)  [wavefront per row]; the _short forms (4 .. 1024 columns) give a row
//           4 .. 64 lanes, grid (ceil(rows * lanes / 256),1,1);
//   reduce_outer: grid (ceil(inner / (1024 v)), 1, 1), v = 8, 4, 2 or 1: the largest that leaves
//           512 workgroups (any other grid works too, the workgroups stride).

#include "column_chain.h"
#include "device_common.h"

using namespace imexhip;

namespace {

constexpr int kThreads = 256;
constexpr int kWavesPerBlock = kThreads / kWave;
constexpr int64_t kWavePerRowMaxCols = 2048;

// 16 bytes at any float's address
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ float sum4(f32x4 v) { return (v.x + v.y) + (v.z + v.w); }

// Partial sum of one row over the lanes [tid, tid+stride, ...).  Four independent 16-byte loads in flight per lane, in
// the last round as well (a vector past the end is loaded as the row's last one and counts as zero); no alignment
// needed: 2500 x 8191 33.0 -> 14.0 us, 300 x 16001 19.4 -> 5.8 (element by element where a row's start was not aligned).
template <bool kStream>
__device__ __forceinline__ float row_partial(const float *__restrict__ row, int64_t cols, int tid, int stride) {
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  const int64_t vecs = cols / 4;
  const f32x4u *src = reinterpret_cast<const f32x4u *>(row);
  const float rest = vecs * 4 + tid < cols ? row[vecs * 4 + tid] : 0.0f; // fewer than four elements in all
  auto load = [&](int64_t v) -> f32x4 {
    if constexpr (kStream)
      return __builtin_nontemporal_load(src + v);
    else
      return src[v];
  };
  int64_t v = tid;
  for (; v + 3 * int64_t(stride) < vecs; v += 4 * int64_t(stride)) {
    f32x4 x[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      x[k] = load(v + k * int64_t(stride));
#pragma unroll
    for (int k = 0; k < 4; ++k)
      acc[k] += sum4(x[k]);
  }
  if (v < vecs) {
    f32x4 x[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      x[k] = load(min(v + k * int64_t(stride), vecs - 1));
#pragma unroll
    for (int k = 0; k < 4; ++k)
      acc[k] += v + k * int64_t(stride) < vecs ? sum4(x[k]) : 0.0f;
  }
  return ((acc[0] + acc[1]) + (acc[2] + acc[3])) + rest;
}

} // namespace

// kMean: the sum (from `init`) divided by the row length, the post-op of
// WG/reduction_4D_3D_mean_intra_sg_intra_lane.mlir:51-52.
template <bool kMean>
__device__ __forceinline__ void row_reduce(const float *in, float *out, int64_t rows, int64_t cols, float init) {
  const float divisor = static_cast<float>(cols);
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  // the input is read exactly once: stream it past the caches (non-temporal)
  constexpr bool stream = true;
  // workgroups (wavefronts) stride over the rows, so any grid covers all of them
  if (cols > kWavePerRowMaxCols) {
    __shared__ float partial[kWavesPerBlock];
    for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
      const float p = stream ? row_partial<true>(in + row * cols, cols, threadIdx.x, kThreads)
                             : row_partial<false>(in + row * cols, cols, threadIdx.x, kThreads);
      float s = wave_sum(p);
      if (lane == 0)
        partial[wave] = s;
      __syncthreads();
      if (threadIdx.x == 0)
        out[row] = kMean ? (init + ((partial[0] + partial[1]) + (partial[2] + partial[3]))) / divisor
                         : init + ((partial[0] + partial[1]) + (partial[2] + partial[3]));
      __syncthreads(); // `partial` is reused by the next row
    }
  } else {
    for (int64_t row = int64_t(blockIdx.x) * kWavesPerBlock + wave; row < rows;
         row += int64_t(gridDim.x) * kWavesPerBlock) {
      const float p = stream ? row_partial<true>(in + row * cols, cols, lane, kWave)
                             : row_partial<false>(in + row * cols, cols, lane, kWave);
      float s = wave_sum(p);
      if (lane == 0)
        out[row] = kMean ? (init + s) / divisor : init + s;
    }
  }
}

extern "C" __global__ __launch_bounds__(kThreads) void imex_rowsum_f32(const float *in, float *out, int64_t rows,
                                                                      int64_t cols, float init) {
  row_reduce<false>(in, out, rows, cols, init);
}

extern "C" __global__ __launch_bounds__(kThreads) void imex_rowmean_f32(const float *in, float *out, int64_t rows,
                                                                       int64_t cols) {
  row_reduce<true>(in, out, rows, cols, 0.0f);
}

// Short rows: kLanes lanes of a wavefront share one, up to four 16-byte pieces each, so a wavefront reads up to sixteen
// rows at once; the last piece of a row that is no whole number of pieces starts at cols - 4 and counts only the
// elements the piece before does not hold.  Bound by HBM; with a wavefront per row most lanes had nothing to load
// (131072 x 32: 20.9 -> 4.1 us; 10^6 x 40: 145 -> 27.9, 5.7 TB/s), and rows off the 16-byte grid went element by element
// (60000 x 255: 22.0 -> 10.8).
template <bool kMean, int kLanes>
__device__ __forceinline__ void row_reduce_by_lanes(const float *in, float *out, int64_t rows, int cols, float init) {
  const int lane = threadIdx.x % kLanes, per = (cols + 4 * kLanes - 1) / (4 * kLanes);
  int start[4], repeated[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int at = (k * kLanes + lane) * 4;
    start[k] = min(at, cols - 4);
    repeated[k] = at - start[k];
  }
  for (int64_t row = int64_t(blockIdx.x) * (kThreads / kLanes) + threadIdx.x / kLanes; row < rows;
       row += int64_t(gridDim.x) * (kThreads / kLanes)) {
    const float *src = in + row * cols;
    f32x4 x[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (k < per) {
        if constexpr (kLanes == kWave) // rows of 2 KiB and more stream past the caches: 10^5 x 1024 59 us, 65 without
          x[k] = __builtin_nontemporal_load(reinterpret_cast<const f32x4u *>(src + start[k]));
        else
          x[k] = *reinterpret_cast<const f32x4u *>(src + start[k]);
      }
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (k < per) {
        const int r = repeated[k];
        sum += ((r > 0 ? 0.0f : x[k].x) + (r > 1 ? 0.0f : x[k].y)) + ((r > 2 ? 0.0f : x[k].z) + (r > 3 ? 0.0f : x[k].w));
      }
    sum = init + lanes_sum<kLanes>(sum);
    if (lane == 0)
      out[row] = kMean ? sum / static_cast<float>(cols) : sum;
  }
}

template <bool kMean>
__device__ __forceinline__ void row_reduce_short(const float *in, float *out, int64_t rows, int64_t cols, float init) {
  if (cols < 4 || cols > 16 * kWave) {
    row_reduce<kMean>(in, out, rows, cols, init);
    return;
  }
  const int n = int(cols);
  if (n <= 64)
    row_reduce_by_lanes<kMean, 4>(in, out, rows, n, init);
  else if (n <= 128)
    row_reduce_by_lanes<kMean, 8>(in, out, rows, n, init);
  else if (n <= 256)
    row_reduce_by_lanes<kMean, 16>(in, out, rows, n, init);
  else if (n <= 512)
    row_reduce_by_lanes<kMean, 32>(in, out, rows, n, init);
  else
    row_reduce_by_lanes<kMean, 64>(in, out, rows, n, init);
}

extern "C" __global__ __launch_bounds__(kThreads) void imex_rowsum_f32_short(const float *in, float *out, int64_t rows,
                                                                            int64_t cols, float init) {
  row_reduce_short<false>(in, out, rows, cols, init);
}

extern "C" __global__ __launch_bounds__(kThreads) void imex_rowmean_f32_short(const float *in, float *out, int64_t rows,
                                                                             int64_t cols) {
  row_reduce_short<true>(in, out, rows, cols, 0.0f);
}

// Outer-dimension sum: lane owns kVecs vectors of four adjacent outputs, 4 KiB apart, so a
// workgroup reads kVecs * 4 KiB contiguous bytes of every slice.  With `outer` slices a power-of-two
// number of bytes apart, all of a lane's loads fall into the same DRAM channel; wide contiguous
// spans per workgroup are what keeps the channels streaming (measured on 32 x 4 Mi: 111 us with
// 4 KiB spans, 83 us with 32 KiB).  Four slices' loads are kept in flight (a register ring), adds
// kept in slice order.  Workgroups stride over the blocks of outputs, so any grid covers everything.
template <io::Dt D, int kVecs>
__device__ __forceinline__ void reduce_outer_vec(const void *__restrict__ in, void *__restrict__ out, int64_t outer,
                                                 int64_t inner, float init) {
  using E = io::Elem<D>;
  constexpr int kPer = E::kPerVec;                             // outputs per 16-byte vector: 4 or 8
  constexpr int64_t kSpan = int64_t(kThreads) * kPer * kVecs;  // outputs per workgroup and pass
  const u32x4 *src = static_cast<const u32x4 *>(in);
  const int64_t strideVecs = inner / kPer;
  for (int64_t base = int64_t(blockIdx.x) * kSpan; base < inner; base += int64_t(gridDim.x) * kSpan) {
    const int64_t i0 = base + threadIdx.x * kPer;
    float acc[kVecs][kPer];
#pragma unroll
    for (int v = 0; v < kVecs; ++v)
#pragma unroll
      for (int e = 0; e < kPer; ++e)
        acc[v][e] = init;
    auto add = [&](int v, u32x4 raw) {
      float f[kPer];
      E::unpack(raw, f);
#pragma unroll
      for (int e = 0; e < kPer; ++e)
        acc[v][e] = acc[v][e] + f[e];
    };
    // Lanes past the end of the last block read the last vector instead (and store nothing): the loads
    // are unconditional, so the wait for one slice leaves the loads of the next three in flight.
    int64_t at[kVecs];
#pragma unroll
    for (int v = 0; v < kVecs; ++v) {
      const int64_t i = i0 + v * (kThreads * kPer);
      at[v] = (i < inner ? i : inner - kPer) / kPer;
    }
    // A ring of four slices: slice o is added, in slice order, and its registers are at once reloaded with
    // slice o + 4, so three to four slices' loads are in flight all the time.
    constexpr int kRing = 4;
    int64_t o = 0;
    if (outer >= kRing) {
      u32x4 t[kRing][kVecs];
#pragma unroll
      for (int u = 0; u < kRing; ++u)
#pragma unroll
        for (int v = 0; v < kVecs; ++v)
          t[u][v] = __builtin_nontemporal_load(src + at[v] + u * strideVecs);
      for (; o + 2 * kRing <= outer; o += kRing) {
#pragma unroll
        for (int u = 0; u < kRing; ++u) {
#pragma unroll
          for (int v = 0; v < kVecs; ++v)
            add(v, t[u][v]);
#pragma unroll
          for (int v = 0; v < kVecs; ++v)
            t[u][v] = __builtin_nontemporal_load(src + at[v] + (o + kRing + u) * strideVecs);
        }
      }
#pragma unroll
      for (int u = 0; u < kRing; ++u)
#pragma unroll
        for (int v = 0; v < kVecs; ++v)
          add(v, t[u][v]);
      o += kRing;
    }
    for (; o < outer; ++o)
#pragma unroll
      for (int v = 0; v < kVecs; ++v)
        add(v, __builtin_nontemporal_load(src + at[v] + o * strideVecs));
#pragma unroll
    for (int v = 0; v < kVecs; ++v) {
      const int64_t i = i0 + v * (kThreads * kPer);
      if (i < inner)
        static_cast<u32x4 *>(out)[i / kPer] = E::pack(acc[v]);
    }
  }
}

template <io::Dt D>
__device__ __forceinline__ void reduce_outer_by_element(const void *in, void *out, int64_t outer, int64_t inner, float init) {
  using E = io::Elem<D>;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < inner; i += int64_t(gridDim.x) * blockDim.x) {
    float acc = init;
    for (int64_t o = 0; o < outer; ++o)
      acc = acc + E::get(in, o * inner + i);
    E::put(out, i, acc);
  }
}

// 16-bit inputs widen to f32, are added in f32 in slice order and rounded once at the end (the
// reference's policy for 16-bit element types on the GPU, docs/Transforms/BF16ToGpu.md:17-26;
// benchmarks/reduce/reduce.dtypes.in lists f32, f16, bf16).
template <io::Dt D>
__device__ __forceinline__ void reduce_outer(const void *in, void *out, int64_t outer, int64_t inner, float init) {
  using E = io::Elem<D>;
  const bool vec = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0 &&
                   (inner % E::kPerVec) == 0;
  if (vec) {
    // the widest span that still leaves 512 workgroups (two per CU): 32, 16, 8 or 4 KiB per slice
    const int64_t perVec = int64_t(kThreads) * E::kPerVec;
    if (inner >= 512 * 8 * perVec)
      reduce_outer_vec<D, 8>(in, out, outer, inner, init);
    else if (inner >= 512 * 4 * perVec)
      reduce_outer_vec<D, 4>(in, out, outer, inner, init);
    else if (inner >= 512 * 2 * perVec)
      reduce_outer_vec<D, 2>(in, out, outer, inner, init);
    else
      reduce_outer_vec<D, 1>(in, out, outer, inner, init);
  } else {
    reduce_outer_by_element<D>(in, out, outer, inner, init);
  }
}

extern "C" __global__ __launch_bounds__(kThreads) void imex_reduce_outer_f32(const float *in, float *out,
                                                                            int64_t outer, int64_t inner,
                                                                            float init) {
  reduce_outer<io::Dt::F32>(in, out, outer, inner, init);
}

extern "C" __global__ __launch_bounds__(kThreads) void imex_reduce_outer_f16(const uint16_t *in, uint16_t *out,
                                                                            int64_t outer, int64_t inner,
                                                                            float init) {
  reduce_outer<io::Dt::F16>(in, out, outer, inner, init);
}

extern "C" __global__ __launch_bounds__(kThreads) void imex_reduce_outer_bf16(const uint16_t *in, uint16_t *out,
                                                                             int64_t outer, int64_t inner,
                                                                             float init) {
  reduce_outer<io::Dt::BF16>(in, out, outer, inner, init);
}

// ---- outer-dimension sum, sixteen slices in flight ------------------------------------------------------
// A lane owns one piece: a vector of four (eight) outputs, or one output where the slices are no whole 16-byte vectors
// (kVec false).  For outputs that are too few to fill the chip with the wide spans above but enough for a lane each:
// what bounds it is how many loads are in flight, so the ring is sixteen slices deep, the remaining slices' loads are in
// flight together too, and it is a kernel of its own with few registers (eight wavefronts per SIMD, where the wide spans
// leave room for one).  512 x 131072 f32: 73 -> 45 us (floor 42 for its bytes); slices of no whole vectors, one load
// at a time before: f32 238 x 209827 350 -> 40 us, bf16 64 x 524291 210 -> 15.
constexpr int kDeepRing = 16;
template <bool kFirst, typename A, typename B> struct Select { using Type = A; };
template <typename A, typename B> struct Select<false, A, B> { using Type = B; };
template <io::Dt D, bool kVec>
__device__ __forceinline__ void reduce_outer_deep(const void *__restrict__ in, void *__restrict__ out, int64_t outer,
                                                  int64_t inner, float init) {
  using E = io::Elem<D>;
  constexpr int kPer = kVec ? E::kPerVec : 1; // outputs per piece
  constexpr int kRing = kDeepRing;
  using Raw = typename Select<kVec, u32x4, uint32_t>::Type; // as it comes from memory: widening an element here would wait for it
  const int64_t pitch = inner * E::kBytes;
  for (int64_t base = int64_t(blockIdx.x) * kThreads * kPer; base < inner; base += int64_t(gridDim.x) * kThreads * kPer) {
    // Lanes past the end read the last piece instead (and store nothing): the loads are unconditional, so the wait for
    // one slice leaves the loads of the next ones in flight.
    const int64_t i = base + threadIdx.x * kPer;
    const uint32_t at = static_cast<uint32_t>(min(i, inner - kPer) - base) * E::kBytes;
    const char *slice = static_cast<const char *>(in) + base * E::kBytes; // of the slice that is fetched next
    float acc[kPer];
#pragma unroll
    for (int e = 0; e < kPer; ++e)
      acc[e] = init;
    auto load = [&]() -> Raw {
      if constexpr (kVec)
        return __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(slice + at));
      else if constexpr (D == io::Dt::F32)
        return *reinterpret_cast<const uint32_t *>(slice + at);
      else
        return *reinterpret_cast<const uint16_t *>(slice + at);
    };
    auto add = [&](const Raw &raw) {
      float f[kPer];
      if constexpr (kVec)
        E::unpack(raw, f);
      else if constexpr (D == io::Dt::F32)
        f[0] = u2f(raw);
      else
        f[0] = E::widen(raw);
#pragma unroll
      for (int e = 0; e < kPer; ++e)
        acc[e] = acc[e] + f[e];
    };
    // Slice o is added, in slice order, and its register is at once reloaded with slice o + kRing.
    if (outer > 0) {
      Raw t[kRing];
#pragma unroll
      for (int u = 0; u < kRing; ++u) { // fewer slices than the ring holds: the last one again, not added
        t[u] = load();
        slice += u + 1 < outer ? pitch : 0;
      }
      int64_t o = 0;
      for (; o + 2 * kRing <= outer; o += kRing) {
#pragma unroll
        for (int u = 0; u < kRing; ++u) {
          add(t[u]);
          t[u] = load();
          slice += pitch;
          __builtin_amdgcn_sched_barrier(0); // slice by slice: gathered up, the widened values cost 100 registers
        }
      }
      const int left = int(outer - o) - kRing; // beyond those in registers; negative: not all of those exist
      if (left > 0) { // the remaining slices' loads together, the last one's standing in for those past it
#pragma unroll
        for (int u = 0; u < kRing; ++u) {
          add(t[u]);
          t[u] = load();
          slice += u + 1 < left ? pitch : 0;
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      const int last = left > 0 ? left : left + kRing;
#pragma unroll
      for (int u = 0; u < kRing; ++u) {
        if (u < last)
          add(t[u]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (i < inner) {
      if constexpr (kVec)
        static_cast<u32x4 *>(out)[i / kPer] = E::pack(acc);
      else
        E::put(out, i, acc[0]);
    }
  }
}

template <io::Dt D>
__device__ __forceinline__ void reduce_outer_deep_entry(const void *in, void *out, int64_t outer, int64_t inner, float init) {
  using E = io::Elem<D>;
  if (((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15) == 0 && inner % E::kPerVec == 0)
    reduce_outer_deep<D, true>(in, out, outer, inner, init);
  else if (outer <= 2 && inner % E::kPerVec == 0)
    // a buffer off the 16-byte grid under the vectors' launch: a lane walks several outputs, and sixteen loads of one or
    // two slices each cost more than they hide (bf16 1 x 65536: 5.4 us, 3.3 so)
    reduce_outer_by_element<D>(in, out, outer, inner, init);
  else
    reduce_outer_deep<D, false>(in, out, outer, inner, init);
}

extern "C" __global__ __launch_bounds__(kThreads) void imex_reduce_outer_f32_deep(const float *in, float *out,
                                                                                 int64_t outer, int64_t inner,
                                                                                 float init) {
  reduce_outer_deep_entry<io::Dt::F32>(in, out, outer, inner, init);
}

extern "C" __global__ __launch_bounds__(kThreads) void imex_reduce_outer_f16_deep(const uint16_t *in, uint16_t *out,
                                                                                 int64_t outer, int64_t inner,
                                                                                 float init) {
  reduce_outer_deep_entry<io::Dt::F16>(in, out, outer, inner, init);
}

extern "C" __global__ __launch_bounds__(kThreads) void imex_reduce_outer_bf16_deep(const uint16_t *in, uint16_t *out,
                                                                                  int64_t outer, int64_t inner,
                                                                                  float init) {
  reduce_outer_deep_entry<io::Dt::BF16>(in, out, outer, inner, init);
}

// ---- outer-dimension sum, many slices of few outputs -------------------------------------------------
// With 4 .. 32 KiB of every slice per workgroup, a tall matrix (column sums of [8192, 4096]: 4 workgroups of the
// form above) leaves the chip idle and waits for one slice's latency per four slices.  Column chains instead
// (column_chain.h), whose workers have nothing to do but widen: the additions of one output are ordered, so a column costs
// `outer` dependent additions whatever is done, 2.7 ns each here.  f32 8192 x 4096: 980 us in the plain form, 45.2 with a
// 32-bit LDS read for every addition, 33.6 so (floor 21.3 for its bytes, 22 for the chain); 4041 x 1792 24.1 -> 13.9;
// bf16 8192 x 4096 58.0 -> 26.3, where the adder widened as well; f16 2000 x 1001 16.6 -> 8.1, 500 x 20000 9.5 -> 5.8.
template <io::Dt D, int kLanes, int kWorkers, bool kShort = false, int kAhead = 1>
__device__ __forceinline__ void reduce_outer_chains(const void *in, void *out, int64_t outer, int64_t inner, float init, float *lds) {
  using C = ColumnChain<D, 1, kLanes, kWorkers, kAhead>;
  using E = io::Elem<D>;
  C::template run<kShort>(in, nullptr, out, outer, inner, init, lds, [] {}, [](const typename C::Raw(&v)[1][4], float(&f)[4][C::kPer]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        if constexpr (D == io::Dt::F32) {
          f[i][w] = u2f(v[0][i][w]);
        } else {
          f[i][2 * w] = E::widen(v[0][i][w] & 0xffffu);
          f[i][2 * w + 1] = E::widen(v[0][i][w] >> 16);
        }
      }
  });
}

// Four workers for segments of 32 and 64 bytes, wide_chain_workers() for 128.  Other launches, and what the chains do not
// take, add slice by slice as the kernel without the suffix does.
template <io::Dt D>
__device__ __forceinline__ void reduce_outer_tall(const void *in, void *out, int64_t outer, int64_t inner, float init) {
  __shared__ __attribute__((aligned(16))) float lds[ColumnChain<D, 1, 16, 8>::kLdsFloats];
  const int64_t segments = (inner * io::Elem<D>::kBytes + 31) / 32;
  const int lanes = chain_lanes(segments), workers = lanes == 16 ? wide_chain_workers(segments) : 4;
  const int64_t slice = inner * io::Elem<D>::kBytes;
  if (!chains_take<D>(outer, inner) || lanes_launched() != (workers + 1) * kWave || (slice < 8 && outer * slice < 8))
    reduce_outer_by_element<D>(in, out, outer, inner, init);
  else if (lanes == 4 && slice < 8)
    reduce_outer_chains<D, 4, 4, true>(in, out, outer, inner, init, lds);
  else if (lanes == 4)
    reduce_outer_chains<D, 4, 4>(in, out, outer, inner, init, lds);
  else if (lanes == 8 && ahead_of(outer, slice))
    reduce_outer_chains<D, 8, 4, false, 3>(in, out, outer, inner, init, lds);
  else if (lanes == 8)
    reduce_outer_chains<D, 8, 4>(in, out, outer, inner, init, lds);
  else if (workers == 8)
    reduce_outer_chains<D, 16, 8>(in, out, outer, inner, init, lds);
  else
    reduce_outer_chains<D, 16, 4>(in, out, outer, inner, init, lds);
}

extern "C" __global__ __launch_bounds__(576) void imex_reduce_outer_f32_tall(const float *in, float *out, int64_t outer,
                                                                            int64_t inner, float init) {
  reduce_outer_tall<io::Dt::F32>(in, out, outer, inner, init);
}

extern "C" __global__ __launch_bounds__(576) void imex_reduce_outer_f16_tall(const uint16_t *in, uint16_t *out, int64_t outer,
                                                                            int64_t inner, float init) {
  reduce_outer_tall<io::Dt::F16>(in, out, outer, inner, init);
}

extern "C" __global__ __launch_bounds__(576) void imex_reduce_outer_bf16_tall(const uint16_t *in, uint16_t *out, int64_t outer,
                                                                            int64_t inner, float init) {
  reduce_outer_tall<io::Dt::BF16>(in, out, outer, inner, init);
}

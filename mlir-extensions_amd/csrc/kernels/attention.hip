// Flash-attention forward, f16 in / f16 out, head dimension 64, no mask.
//
// Reference: test/Integration/Dialect/XeGPU/WG/flash_attention_fwd.mlir
//   kernel :25-307 -- per workgroup a 128 x 64 Q tile, K/V walked in 64-key
//   blocks, online softmax (running max m, running sum l, accumulator rescaled by
//   exp(m_old - m_new)), P truncated to f16 before P.V, O = acc / l at the end;
//   CPU check :332-421 -- softmax(scale * Q K^T) V per (batch, head), Q/K/V/O stored
//   as [(Z*H*N_CTX), 64] row-major.
//
// On MI355X the products are formed TRANSPOSED, so that a lane owns one query:
//   S^T[key, q] = K_tile . Q^T     A operand = K rows (k-contiguous in LDS),
//                                  B operand = Q rows, loaded once into registers;
//   O^T[d, q]  += V_tile^T . P^T   A operand = V^T via the LDS transpose read,
//                                  B operand = P^T straight from the S^T
//                                  accumulator registers (no shuffles: the MFMA's
//                                  k index is bound to the keys in the order the
//                                  accumulator holds them, and V^T is read in
//                                  the same order).
// With v_mfma_f32_32x32x16_f16 a lane holds query q = lane % 32 and, per 32-key
// block, keys (r/4)*8 + (lane/32)*4 + r%4: the softmax max and sum over keys are
// plain register loops plus ONE exchange between lane l and l+32 per block of
// keys.
//
// Workgroup = QB query blocks of 32 x KG key groups, one wavefront each: 64, 128 or 256
// queries of one (batch, head) as (QB, KG) = (2,4), (4,2), (8,1) with 512 threads, or 256
// queries as (8,2) with 1024 threads.  Wavefront w takes query block w % QB and every KG-th
// key tile of 64 keys, group w / QB; partial (m, l, O) of the key groups are merged through LDS
// at the end.  (_q32 and _q64 have eight key groups: "every wavefront its own keys" below.)  Every
// workgroup walks all keys of its head, so K / V traffic from L2 falls with the
// queries per workgroup; key groups exist to keep all CUs busy on small problems (the
// reference's 2 x 2 x 4096 x 64 gives one 64-query workgroup per CU) and, in the 1024-thread
// form, to put four wavefronts on every SIMD (the tiled path needs 114 registers).  The launch
// says which: N_CTX / gridDim.x queries per workgroup, blockDim.x threads.  K and V blocks of
// 64 KG keys go from global memory straight into an LDS ring (buffer_load ... lds) of 2, 4 or
// 8 stages, up to seven blocks ahead.
//
// Arguments: (Q, K, V, Out, sm_scale: f32, ZH: i64, N_CTX: i64)   dims = {ZH, N_CTX}
//   ZH = batch * heads; all four tensors [(ZH*N_CTX), 64]; sm_scale > 0.  N_CTX need not divide the
//   tiles: queries past the end are not stored, keys past the end get a score of -inf.
// imex_flash_attention_fwd_f16_q32 / _q64 / _q128 / _q256 are the operator with one tiling each.
// Launch: grid (ceil(N_CTX / q), ZH, 1) with q = 64, 128 or 256 and block (512,1,1), or q = 256
// and block (1024,1,1); the forms with one tiling take theirs only, _q256 with block (1024,1,1).  Other launches (and a
// scale <= 0, or misaligned tensors) take the one-query-per-lane reference loop of the same kernel (grid-stride, any grid and block).

#include "device_common.h"

using namespace imexhip;

namespace {

constexpr int kMaxThreads = 1024; // 8 or 16 wavefronts per workgroup
constexpr int D = 64;                 // head dimension
constexpr int kRingBytes = 128 * 1024;          // 2 stages of 64 KiB, 4 of 32 KiB or 8 of 16 KiB
constexpr int kLdsBytes = kRingBytes;           // the ring, and after it the partial results of up to eight wavefronts
static_assert(kLdsBytes >= 8 * 34 * 64 * 4, "two key groups hand eight of them over, four or eight meet from eight wavefronts");

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 LdsI16x4;
typedef __attribute__((address_space(3))) char LdsChar;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *base, int64_t bytes) {
  const int range = bytes > 0x7fffffff ? 0x7fffffff : int(bytes);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, range, 0x00020000);
}
template <int N> __device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));
}
// the larger of this lane's value and the one that lane l+32 (or l-32) holds
__device__ __forceinline__ float max_of_halves(float v) {
  const auto both = __builtin_amdgcn_permlane32_swap(f2u(v), f2u(v), false, false); // the lower half's, the upper half's
  return fmaxf(u2f(both[0]), u2f(both[1]));
}
// the value lane l+32 (or l-32) holds
__device__ __forceinline__ float other_half(float v) { return __shfl_xor(v, 32, 64); }

// Workgroups go to the 8 XCDs round-robin in launch order, and each XCD has its own L2.  Renumber them so that one XCD gets
// consecutive query blocks -- whole heads, or a contiguous part of one; as many as the others or one more -- and its L2
// holds the K / V of a few heads instead of a slice of the traffic of all of them.  A launch that 8 does not divide only
// where `uneven` says so: the way there takes 0.1 .. 0.3 us longer than launch order, which 32 queries, whose one round has
// little to share, and few keys do not get back (1 x 52 with it 4.50 us, 3.89 so; 28 such problems of 32 queries of 1024 keys
// and more 1.00 .. 1.02 of the time with it; others from 256 keys on 0.85 .. 1.00: 165 x 513 38.4 in launch order, 35.3).
__device__ __forceinline__ void place_of_workgroup(uint32_t &x, uint32_t &y, bool uneven) {
  const uint32_t total = gridDim.x * gridDim.y;
  x = blockIdx.x;
  y = blockIdx.y;
  if (total % 8 == 0 || uneven) {
    const uint32_t launched = y * gridDim.x + x, xcd = launched & 7;
    const uint32_t logical = xcd * (total >> 3) + min(xcd, total & 7) + (launched >> 3);
    y = logical / gridDim.x;
    x = logical - y * gridDim.x;
  }
}

// ---- any-shape path: one lane per query, the reference loop ----------------------------
__device__ __forceinline__ void attention_scalar(const uint16_t *Q, const uint16_t *K, const uint16_t *V,
                                                 uint16_t *Out, float scale, int64_t ZH, int64_t N) {
  const int64_t block = int64_t(blockIdx.z) * gridDim.y * gridDim.x + int64_t(blockIdx.y) * gridDim.x + blockIdx.x;
  const int64_t stride = int64_t(gridDim.x) * gridDim.y * gridDim.z * blockDim.x;
  const float c = scale * 1.44269504088896341f;
  for (int64_t row = block * blockDim.x + threadIdx.x; row < ZH * N; row += stride) {
    const int64_t head0 = (row / N) * N;
    float o[D]; // the query row is re-read per key (it stays in cache): 64 registers, not 128
    for (int d = 0; d < D; ++d)
      o[d] = 0.0f;
    float m = -__builtin_inff(), l = 0.0f;
    for (int64_t j = 0; j < N; ++j) {
      float s = 0.0f;
      for (int d = 0; d < D; ++d)
        s += half_bits_to_float(Q[row * D + d]) * half_bits_to_float(K[(head0 + j) * D + d]);
      s *= c;
      const float mNew = fmaxf(m, s);
      const float alpha = exp2f(m - mNew);
      const float p = half_bits_to_float(float_to_half_bits(exp2f(s - mNew)));
      l = l * alpha + p;
      for (int d = 0; d < D; ++d)
        o[d] = o[d] * alpha + p * half_bits_to_float(V[(head0 + j) * D + d]);
      m = mNew;
    }
    for (int d = 0; d < D; ++d)
      Out[row * D + d] = static_cast<uint16_t>(float_to_half_bits(o[d] / l));
  }
}

// ---- results ---------------------------------------------------------------------------------
// The partial results of the key groups meet in LDS (whose tiles nobody copies or reads any more), and every wavefront
// merges its share of them: 8 / KG of the eight groups of four rows that a query block of 32 has.  (One wavefront per
// query block merging all of it is as fast for two key groups, 8 x 3000 35.0 against 35.8 us, but not for four, 16 x 768
// 8.93 against 8.74, or eight.)
constexpr int kSlot = 33 * 64; // floats of one partial result: 32 accumulator rows, four to a vector; m, l of every query
__device__ __forceinline__ void put_partial(const f32x16 (&o)[2], float m, float l, float *slot, int lane) {
#pragma unroll
  for (int u = 0; u < 8; ++u) // rows of the accumulator's block u / 4
    *reinterpret_cast<f32x4 *>(slot + (u * 64 + lane) * 4) =
        f32x4{o[u >> 2][(u & 3) * 4], o[u >> 2][(u & 3) * 4 + 1], o[u >> 2][(u & 3) * 4 + 2], o[u >> 2][(u & 3) * 4 + 3]};
  if (lane < 32)
    *reinterpret_cast<float2 *>(slot + 32 * 64 + lane * 2) = float2{m, l};
}
// Units first .. first + kUnits - 1 of a query block whose KG partial results begin at `of`.
template <int KG, int kUnits>
__device__ __forceinline__ void merge_partials(const float *of, uint16_t *__restrict__ Out, int64_t firstRow, int64_t endRow,
                                               int first, int lane, bool ragged) {
  float a[KG], mAll = -__builtin_inff(), lAll = 0.0f;
  float2 ml[KG];
#pragma unroll
  for (int g = 0; g < KG; ++g) {
    ml[g] = *reinterpret_cast<const float2 *>(of + g * kSlot + 32 * 64 + (lane & 31) * 2);
    mAll = fmaxf(mAll, ml[g].x);
  }
#pragma unroll
  for (int g = 0; g < KG; ++g) {
    a[g] = __builtin_amdgcn_exp2f(ml[g].x - mAll); // a group without a key: 0
    lAll += ml[g].y * a[g];
  }
  const float inv = 1.0f / lAll;
  const int64_t row = firstRow + (lane & 31);
#pragma unroll
  for (int j = 0; j < kUnits; ++j) {
    const int u = first + j; // lane holds, for its query, d = u*8 + (lane/32)*4 .. +3
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int g = 0; g < KG; ++g)
      acc += *reinterpret_cast<const f32x4 *>(of + g * kSlot + (u * 64 + lane) * 4) * a[g];
    f16x4 out4;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      out4[e] = static_cast<_Float16>(acc[e] * inv);
    if (!ragged || row < endRow)
      *reinterpret_cast<f16x4 *>(Out + row * D + u * 8 + (lane >> 5) * 4) = out4;
  }
}
template <int QB, int KG>
__device__ __forceinline__ void merge_and_store(const f32x16 (&o)[2], float m, float l, uint16_t *__restrict__ Out,
                                                int64_t firstRow, int64_t endRow, char *lds, int wave, int wq, int wk,
                                                int lane, bool ragged) {
  constexpr int kUnits = 8 / KG; // of four rows, per wavefront
  float *all = reinterpret_cast<float *>(lds);
  __syncthreads(); // the ring is free
  put_partial(o, m, l, all + (wq * KG + wk) * kSlot, lane);
  __syncthreads();
  const int qb = wave / KG; // the query block of which this wavefront merges a share
  merge_partials<KG, kUnits>(all + qb * (KG * kSlot), Out, firstRow + qb * 32, endRow, wave % KG * kUnits, lane, ragged);
}

// ---- MFMA path ---------------------------------------------------------------------------
// QB = 32-query blocks per workgroup, KG = key groups: QB x KG wavefronts (8 or 16).  More query
// blocks mean fewer workgroups but proportionally less K / V traffic from L2 (every workgroup walks
// all keys of its head); fewer key groups mean smaller ring stages and therefore a deeper ring.
// kRagged: N_CTX is not a multiple of the workgroup's 32 QB queries or of its 64 KG-key blocks; the
// padding logic below is compiled in only then.
template <int QB, int KG, bool kRagged, bool kScoresAhead = false>
__device__ __forceinline__ void attention_tiled(const uint16_t *__restrict__ Q, const uint16_t *__restrict__ K,
                                                const uint16_t *__restrict__ V, uint16_t *__restrict__ Out,
                                                float scale, int64_t N, char *lds) {
  LdsChar *ldsBase = (LdsChar *)lds;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int kWaves = QB * KG;
  constexpr int KB = 2, BN = 32 * KB;              // keys per tile
  constexpr int kTileBytes = BN * D * 2;           // 8 KiB
  constexpr int kStageBytes = 2 * KG * kTileBytes; // K tiles of all key groups, then their V tiles
  constexpr int kStages = kRingBytes / kStageBytes; // 2, 4 or 8
  constexpr int kAhead = kStages - 1;              // blocks in flight ahead of the one being multiplied
  constexpr int kCopies = BN * KG / (8 * kWaves);  // 1 KiB (8-row) copies per wavefront, stage and operand
  const int wq = wave % QB, wk = wave / QB;
  const int qi = lane & 31, half = lane >> 5;
  uint32_t bx, by;
  place_of_workgroup(bx, by, N >= 256);
  const int64_t head0 = int64_t(by) * N;                 // first row of this (batch, head)
  const int64_t q0 = head0 + int64_t(bx) * (32 * QB) + wq * 32;
  // N_CTX need not divide the tiles.  Queries past the end of the head are computed on a copy of
  // its last row and not stored; keys past the end are copies of the last key whose scores are
  // set to -inf before the softmax (below), so no address ever leaves the head.
  const int64_t qRow = kRagged ? min(q0 + qi, head0 + N - 1) : q0 + qi;

  // Q^T operand: lane (q, half) keeps Q[q][ds*16 + half*8 .. +7] for the four 16-wide steps
  f16x8 qf[4];
#pragma unroll
  for (int ds = 0; ds < 4; ++ds)
    qf[ds] = *reinterpret_cast<const f16x8 *>(Q + qRow * D + ds * 16 + half * 8);

  // -- global -> LDS copies.  A stage is [K tile 0 .. KG-1][V tile 0 .. KG-1], each BN
  // rows of 128 bytes; one copy = 8 rows.  16-byte chunk c of row r is stored at
  //   K: c ^ ((r ^ (r>>3 & 3)) & 7)   (conflict-free 128-bit fragment reads; same for r and r+32)
  //   V: c ^ (((r>>1) & 1) << 2)     (conflict-free transpose reads)
  // applied on the global side, since a direct copy fixes the lane's LDS position.
  const __amdgpu_buffer_rsrc_t kRsrc = make_rsrc(K + head0 * D, N * D * 2);
  const __amdgpu_buffer_rsrc_t vRsrc = make_rsrc(V + head0 * D, N * D * 2);
  const __amdgpu_buffer_rsrc_t nothing = make_rsrc(K + head0 * D, 0);
  const int iters = int((N + KG * BN - 1) / (KG * BN));            // key blocks of BN KG keys
  const int lastRows = int(N - int64_t(iters - 1) * (KG * BN));    // keys in the last block: 1 .. BN KG
  const bool raggedKeys = kRagged && lastRows != KG * BN;
  int kVoff[kCopies], vVoff[kCopies];   // per-lane byte offsets inside a block
  int kVoffT[kCopies], vVoffT[kCopies]; // the same for the last block, rows clamped to its last key
#pragma unroll
  for (int c = 0; c < kCopies; ++c) {
    // wavefront w copies rows [8 kCopies w, 8 kCopies (w+1)) of the stage's BN KG K rows and of its V rows
    const int row = wave * (8 * kCopies) + c * 8 + (lane >> 3); // key within the stage's block of BN KG keys
    const int r = row & (BN - 1);                          // row within its tile
    const int kc = (lane & 7) ^ ((r ^ ((r >> 3) & 3)) & 7);
    const int vc = (lane & 7) ^ (((r >> 1) & 1) << 2);
    kVoff[c] = (row * D + kc * 8) * 2;
    vVoff[c] = (row * D + vc * 8) * 2;
    const int rowT = kRagged ? min(row, lastRows - 1) : row;
    kVoffT[c] = (rowT * D + kc * 8) * 2;
    vVoffT[c] = (rowT * D + vc * 8) * 2;
  }
  // Blocks past the end: through a descriptor of size zero with four key groups (nothing moves, but the copies count: 4 x
  // 4096 28.5 -> 28.2 us); the last block again with fewer, whose two query blocks and more per key group hide it, and
  // which the choice of a descriptor costs more (12 x 1500 20.1, 20.3).
  constexpr bool kSkip = KG >= 4;
  auto dma_k = [&](int block, int stage) { // keys [BN KG block, BN KG (block + 1)) into ring stage `stage`
    LdsChar *dst = ldsBase + stage * kStageBytes + wave * (kCopies * 1024);
    const int b = kSkip ? block : min(block, iters - 1);
    const bool tail = raggedKeys && b == iters - 1; // uniform
#pragma unroll
    for (int c = 0; c < kCopies; ++c)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b < iters ? kRsrc : nothing, dst + c * 1024, 16, tail ? kVoffT[c] : kVoff[c],
                                               b < iters ? b * (KG * BN * D * 2) : 0, 0, 0);
  };
  auto dma_v = [&](int block, int stage) { // the same keys' rows of V
    LdsChar *dst = ldsBase + stage * kStageBytes + KG * kTileBytes + wave * (kCopies * 1024);
    const int b = kSkip ? block : min(block, iters - 1);
    const bool tail = raggedKeys && b == iters - 1;
#pragma unroll
    for (int c = 0; c < kCopies; ++c)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b < iters ? vRsrc : nothing, dst + c * 1024, 16, tail ? vVoffT[c] : vVoff[c],
                                               b < iters ? b * (KG * BN * D * 2) : 0, 0, 0);
  };

  // -- LDS read addresses (relative to this wavefront's K / V tile of a stage)
  // K fragment (key block kb, step ds): row kb*32 + qi, logical chunk ds*2 + half
  int kRd[4];
#pragma unroll
  for (int ds = 0; ds < 4; ++ds) {
    const int r = qi; // the swizzle term is the same for rows r and r + 32
    kRd[ds] = wk * kTileBytes + r * 128 + ((((ds * 2 + half) ^ r ^ ((r >> 3) & 3)) & 7) << 4);
  }
  // V^T fragment (d block db, key step kk): two transpose reads.  Lane t of a 16-lane group
  // supplies the address of 4 consecutive d at key row (base + t/4) and receives 4 consecutive
  // key rows of d = t.  Key rows of element e of the operand: kk*16 + (e/4)*8 + half*4 + e%4 --
  // the order in which the S^T accumulator holds the keys.
  int vRd[2];
  {
    const int t = lane & 15, blk = (lane >> 4) & 1;
    const int row = half * 4 + (t >> 2);
#pragma unroll
    for (int db = 0; db < 2; ++db) {
      const int chunk = ((db ^ ((t >> 3) & 1)) << 2) | (blk << 1) | ((t & 3) >> 1);
      vRd[db] = KG * kTileBytes + wk * kTileBytes + row * 128 + chunk * 16 + (t & 1) * 8;
    }
  }

  f32x16 o[2];
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      o[db][r] = 0.0f;
  float m = -__builtin_inff(); // running max of scale*log2(e)*s over this lane's query (both halves agree)
  float l = 0.0f;              // running sum of p over THIS lane's keys only
  const float c = scale * 1.44269504088896341f;

  // S^T = K . Q^T for this wavefront's BN keys of a stage (the first product of each chain takes a
  // literal zero accumulator, so no registers are cleared)
  auto scores = [&](f32x16(&s)[KB], const char *st) {
    const f32x16 zero = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    f16x8 kf[KB][4];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int ds = 0; ds < 4; ++ds)
        kf[kb][ds] = *reinterpret_cast<const f16x8 *>(st + kRd[ds] + kb * 32 * 128);
    // the two accumulator chains alternate, so no MFMA waits for the one just issued
#pragma unroll
    for (int ds = 0; ds < 4; ++ds)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[kb][ds], qf[ds], ds == 0 ? zero : s[kb], 0, 0, 0);
  };
  // block `it`, its scores in s and its V tile in stage st: online softmax, O^T += V^T . P^T
  auto attend = [&](f32x16(&s)[KB], int it, const char *st) {
    // keys of this wavefront's tile that exist: fewer than BN only in the last block of a ragged N_CTX
    const int nValid = int(N) - (it * (KG * BN) + wk * BN);
    if (kRagged && nValid < BN) { // uniform over the wavefront
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          s[kb][r] = kb * 32 + (r >> 2) * 8 + half * 4 + (r & 3) < nValid ? s[kb][r] : -__builtin_inff();
    }
    // online softmax over the keys; this lane owns half of the query's BN scores
    // four chains of additions and maxima where few wavefronts would wait for one; one where many issue (16 x 4096: 83 us, 86)
    constexpr int kChains = kScoresAhead ? 4 : 1;
    float part[kChains];
#pragma unroll
    for (int r = 0; r < kChains; ++r)
      part[r] = s[0][r];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int r = kb ? 0 : kChains; r < 16; ++r)
        part[r % kChains] = fmaxf(part[r % kChains], s[kb][r]);
    float mx = part[0];
#pragma unroll
    for (int r = 1; r < kChains; ++r)
      mx = fmaxf(mx, part[r]);
    mx = max_of_halves(mx);
    const float mRun = fmaxf(m, mx * c);
    // a key group that has seen no key yet (ragged N_CTX shorter than its first tile) stays at -inf;
    // 0 stands in for it below so that -inf - -inf never forms: every p and alpha is then exp2(-inf) = 0
    const float mNew = kRagged && mRun == -__builtin_inff() ? 0.0f : mRun;
    const float alpha = __builtin_amdgcn_exp2f(m - mNew);
    m = mRun;
    float sum[kChains];
#pragma unroll
    for (int r = 0; r < kChains; ++r)
      sum[r] = 0.0f;
    f16x8 pf[2 * KB];
#pragma unroll
    for (int kk = 0; kk < 2 * KB; ++kk) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kk >> 1][(kk & 1) * 8 + e], c, -mNew)); // one fused op per score
        pf[kk][e] = static_cast<_Float16>(p); // the reference truncates P to f16 before P.V (:262-265)
        sum[e % kChains] += p;                      // ... and sums the untruncated f32 values (:243-247)
      }
    }
    #pragma unroll
    for (int r = 1; r < kChains; ++r)
      sum[0] += sum[r];
    l = l * alpha + sum[0];
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) { // the running max moved for some query of this wavefront
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          o[db][r] *= alpha;
    }
    // O^T += V^T . P^T
#pragma unroll
    for (int kk = 0; kk < 2 * KB; ++kk) {
#pragma unroll
      for (int db = 0; db < 2; ++db) {
        const char *p = st + vRd[db] + kk * 16 * 128;
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4 *)(p));
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4 *)(p + 8 * 128));
        const f16x8 vf = __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pf[kk], o[db], 0, 0, 0);
      }
    }
  };

  if constexpr (kScoresAhead) {
    // The scores of block it + 1 are formed before block `it` goes through the softmax, so the softmax does not wait for
    // the last products of its own scores.  The K reads are still waited for, in front of the products of either
    // order: a wavefront issues in order, and these come first.  K(it + 1) and V(it) are there when block `it` begins;
    // the copies in flight are pairs of these.  Past the end as below.
    dma_k(0, 0);
#pragma unroll
    for (int b = 0; b < kAhead; ++b) {
      dma_k(b + 1, b + 1);
      dma_v(b, b);
    }
    wait_vmcnt<kAhead * 2 * kCopies>(); // K(0) has landed
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    f32x16 s[KB], next[KB];
    scores(s, lds);
    int cur = 0; // ring stage of V(it)
    for (int it = 0; it < iters; ++it) {
      __builtin_amdgcn_sched_barrier(0);        // everything read from LDS so far has been used
      wait_vmcnt<(kAhead - 1) * 2 * kCopies>(); // K(it + 1), V(it) have landed
      __builtin_amdgcn_s_barrier();             // ... everyone's; and everyone is done with K(it), V(it - 1) ...
      __builtin_amdgcn_sched_barrier(0);
      dma_k(it + kStages, cur); // ... whose places these go to
      dma_v(it + kAhead, cur == 0 ? kStages - 1 : cur - 1);
      const int after = cur == kStages - 1 ? 0 : cur + 1;
      scores(next, lds + after * kStageBytes); // (past the last block: of whatever the ring holds, not used)
      attend(s, it, lds + cur * kStageBytes);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        s[kb] = next[kb];
      cur = after;
    }
  } else {
    // The ring always holds kAhead blocks in flight (also past the end), so "block `it` has landed" is one fixed vmcnt.
#pragma unroll
    for (int b = 0; b < kAhead; ++b) {
      dma_k(b, b);
      dma_v(b, b);
    }
    int cur = 0; // ring stage of block `it`
    for (int it = 0; it < iters; ++it) {
      wait_vmcnt<(kAhead - 1) * 2 * kCopies>(); // block `it` has landed (this wavefront's copies)
      __builtin_amdgcn_s_barrier();             // ... everyone's; and everyone is done reading block it-1
      __builtin_amdgcn_sched_barrier(0);
      const int before = cur == 0 ? kStages - 1 : cur - 1; // the stage block it-1 occupied
      dma_k(it + kAhead, before);
      dma_v(it + kAhead, before);
      f32x16 s[KB];
      scores(s, lds + cur * kStageBytes);
      attend(s, it, lds + cur * kStageBytes);
      cur = cur == kStages - 1 ? 0 : cur + 1;
    }
  }
  wait_vmcnt<0>();
  l += other_half(l); // both key halves of the lane pair

  if constexpr (KG >= 4) {
    merge_and_store<QB, KG>(o, m, l, Out, q0 - wq * 32, head0 + N, lds, wave, wq, wk, lane, kRagged);
    return;
  }

  // -- two key groups: group 1 hands (m, l, O^T) to group 0 through LDS
  __syncthreads(); // the ring is free
  constexpr int kHand = 34 * 64; // floats per query block and key group: 32 accumulator rows, m, l
  float *xchg = reinterpret_cast<float *>(lds) + wq * (KG - 1) * kHand;
  if (wk != 0) {
    float *mine = xchg + (wk - 1) * kHand;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        mine[(db * 16 + r) * 64 + lane] = o[db][r];
    mine[32 * 64 + lane] = m;
    mine[33 * 64 + lane] = l;
  }
  __syncthreads();
  if (wk == 0) {
    float mAll = m;
#pragma unroll
    for (int g = 0; g < KG - 1; ++g)
      mAll = fmaxf(mAll, xchg[g * kHand + 32 * 64 + lane]);
    float a[KG];
    a[0] = exp2f(m - mAll);
    float lAll = l * a[0];
#pragma unroll
    for (int g = 0; g < KG - 1; ++g) {
      a[g + 1] = exp2f(xchg[g * kHand + 32 * 64 + lane] - mAll);
      lAll += xchg[g * kHand + 33 * 64 + lane] * a[g + 1];
    }
    const float inv = 1.0f / lAll;
    // lane holds, for query q = qi, d = db*32 + (r/4)*8 + half*4 + r%4
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        f16x4 out4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = g4 * 4 + e;
          float acc = o[db][r] * a[0];
#pragma unroll
          for (int g = 0; g < KG - 1; ++g)
            acc += xchg[g * kHand + (db * 16 + r) * 64 + lane] * a[g + 1];
          out4[e] = static_cast<_Float16>(acc * inv);
        }
        if (!kRagged || q0 + qi < head0 + N)
          *reinterpret_cast<f16x4 *>(Out + (q0 + qi) * D + db * 32 + g4 * 8 + half * 4) = out4;
      }
  }
}

// ---- every wavefront its own keys ------------------------------------------------------------
// Eight wavefronts on 32 queries; wavefront w takes every eighth 32-key tile.  Nobody else reads its tiles, so it
// copies them into LDS of its own (a place of 4 KiB for K and one for V, filled again as soon as the fragments are in
// registers) and waits for its own copies only: no barrier in the loop, and the wavefronts of a SIMD drift apart, so that
// one's products run under the others' exponentials, where the shared ring keeps all of them in step.  (68 KiB of LDS and
// at most 128 registers leave room for a second workgroup on the CU, which the catalogue's rule never puts there: from a
// second one on, 64 queries walk half the keys.)  Against the 32-query form of attention_tiled that it replaced
// (1 x 4096, 128 workgroups: 20.0 us) and 64 queries (the others): 1 x 4096 14.8 us, 4 x 2048 14.0 -> 11.0, 8 x 1024 10.0
// -> 7.6, 4 x 512 7.1 -> 5.9, 4 x 264 7.8 -> 5.2, 256 x 32 7.3 -> 4.3; it ends where a CU gets more than one workgroup
// (16 x 768 8.75 -> 10.0).  Bound by the softmax's instructions (about 460
// cycles of issue per tile, two wavefronts on a SIMD) and, at one wavefront's 8 KiB in flight, by the copies' latency.
// Sixteen wavefronts, or 64 queries per wavefront, were not faster.
constexpr int kOwnKeys = 32, kOwnTile = kOwnKeys * D * 2;
constexpr int kOwnWaves = 8, kOwnLds = kOwnWaves * kSlot * 4; // the partial results; the tiles are 8 KiB per wavefront

template <bool kRagged>
__device__ __forceinline__ void attention_own_keys(const uint16_t *__restrict__ Q, const uint16_t *__restrict__ K,
                                                   const uint16_t *__restrict__ V, uint16_t *__restrict__ Out,
                                                   float scale, int64_t N, char *lds) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int qi = lane & 31, half = lane >> 5;
  uint32_t bx, by;
  place_of_workgroup(bx, by, false);
  const int64_t head0 = int64_t(by) * N, q0 = head0 + int64_t(bx) * 32;
  const int tiles = int((N + kOwnKeys - 1) / kOwnKeys), lastRows = int(N - int64_t(tiles - 1) * kOwnKeys);
  const int iters = tiles > wave ? (tiles - wave + kOwnWaves - 1) / kOwnWaves : 0;

  // copies, places and fragment addresses: the layouts of attention_tiled for 32-key tiles
  const __amdgpu_buffer_rsrc_t kRsrc = make_rsrc(K + head0 * D, N * D * 2), vRsrc = make_rsrc(V + head0 * D, N * D * 2);
  const __amdgpu_buffer_rsrc_t nothing = make_rsrc(K + head0 * D, 0); // past the last tile: nothing moves, but the copies count
  int kVoff[4], vVoff[4], kVoffT[4], vVoffT[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int r = c * 8 + (lane >> 3), rT = kRagged ? min(r, lastRows - 1) : r;
    const int kc = (lane & 7) ^ ((r ^ ((r >> 3) & 3)) & 7), vc = (lane & 7) ^ (((r >> 1) & 1) << 2);
    kVoff[c] = (r * D + kc * 8) * 2;
    vVoff[c] = (r * D + vc * 8) * 2;
    kVoffT[c] = (rT * D + kc * 8) * 2;
    vVoffT[c] = (rT * D + vc * 8) * 2;
  }
  char *own = lds + wave * (2 * kOwnTile); // K, V
  auto dma_k = [&](int i) {
    LdsChar *dst = (LdsChar *)own;
    const int tile = wave + i * kOwnWaves;
    const bool tail = kRagged && tile == tiles - 1;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(i < iters ? kRsrc : nothing, dst + c * 1024, 16, tail ? kVoffT[c] : kVoff[c],
                                               i < iters ? tile * kOwnTile : 0, 0, 0);
  };
  auto dma_v = [&](int i) {
    LdsChar *dst = (LdsChar *)own + kOwnTile;
    const int tile = wave + i * kOwnWaves;
    const bool tail = kRagged && tile == tiles - 1;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(i < iters ? vRsrc : nothing, dst + c * 1024, 16, tail ? vVoffT[c] : vVoff[c],
                                               i < iters ? tile * kOwnTile : 0, 0, 0);
  };
  dma_k(0);
  const int64_t qRow = kRagged ? min(q0 + qi, head0 + N - 1) : q0 + qi;
  f16x8 qf[4]; // loaded between the first copies: the wait for the keys covers them
#pragma unroll
  for (int ds = 0; ds < 4; ++ds)
    qf[ds] = *reinterpret_cast<const f16x8 *>(Q + qRow * D + ds * 16 + half * 8);
  __builtin_amdgcn_sched_barrier(0);
  dma_v(0);
  int kRd[4], vRd[2];
#pragma unroll
  for (int ds = 0; ds < 4; ++ds)
    kRd[ds] = qi * 128 + ((((ds * 2 + half) ^ qi ^ ((qi >> 3) & 3)) & 7) << 4);
  {
    const int t = lane & 15, blk = (lane >> 4) & 1, row = half * 4 + (t >> 2);
#pragma unroll
    for (int db = 0; db < 2; ++db)
      vRd[db] = row * 128 + ((((db ^ ((t >> 3) & 1)) << 2) | (blk << 1) | ((t & 3) >> 1)) * 16) + (t & 1) * 8;
  }
  f32x16 o[2];
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      o[db][r] = 0.0f;
  float m = -__builtin_inff(), l = 0.0f;
  const float c = scale * 1.44269504088896341f;
  auto landed = [] { // all but the four youngest copies, of one tile
    wait_vmcnt<4>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto read_done = [] { // the fragments are in registers: their place may be filled again
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  for (int i = 0; i < iters; ++i) {
    landed(); // K(i); V(i) may be on its way
    f16x8 kf[4];
#pragma unroll
    for (int ds = 0; ds < 4; ++ds)
      kf[ds] = *reinterpret_cast<const f16x8 *>(own + kRd[ds]);
    read_done();
    dma_k(i + 1);
    const f32x16 zero = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    f32x16 s;
#pragma unroll
    for (int ds = 0; ds < 4; ++ds)
      s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[ds], qf[ds], ds == 0 ? zero : s, 0, 0, 0);
    if (kRagged && wave + i * kOwnWaves == tiles - 1 && lastRows < kOwnKeys) { // uniform over the wavefront
#pragma unroll
      for (int r = 0; r < 16; ++r)
        s[r] = (r >> 2) * 8 + half * 4 + (r & 3) < lastRows ? s[r] : -__builtin_inff();
    }
    // online softmax, as in attention_tiled; while every score so far is -inf, 0 stands in for the maximum
    float part[2] = {s[0], s[1]};
#pragma unroll
    for (int r = 2; r < 16; ++r)
      part[r & 1] = fmaxf(part[r & 1], s[r]);
    const float mRun = fmaxf(m, max_of_halves(fmaxf(part[0], part[1])) * c);
    const float mNew = mRun == -__builtin_inff() ? 0.0f : mRun;
    const float alpha = __builtin_amdgcn_exp2f(m - mNew);
    m = mRun;
    f16x8 pf[2];
    float sum[2] = {0.0f, 0.0f};
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], c, -mNew));
      pf[r >> 3][r & 7] = static_cast<_Float16>(p);
      sum[r & 1] += p;
    }
    l = l * alpha + (sum[0] + sum[1]);
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) { // the running max moved for some query of this wavefront
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          o[db][r] *= alpha;
    }
    landed(); // V(i); K(i + 1) may be on its way
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int db = 0; db < 2; ++db) {
        const char *p = own + kOwnTile + vRd[db] + kk * 16 * 128;
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4 *)(p));
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4 *)(p + 8 * 128));
        const f16x8 vf = __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pf[kk], o[db], 0, 0, 0);
      }
    read_done();
    dma_v(i + 1);
  }
  wait_vmcnt<0>();

  merge_and_store<1, kOwnWaves>(o, m, l + other_half(l), Out, q0, head0 + N, lds, wave, 0, wave, lane, kRagged);
}

template <typename T> __device__ __forceinline__ void pin(T &v) { asm volatile("" : "+v"(v)); }

// ---- every wavefront its own keys, for two blocks of 32 queries -------------------------------
// 64 queries, eight wavefronts, each of which takes every eighth 32-key tile through both blocks of 32 queries, A and B: a
// fragment is read from LDS once for two products (half the LDS reads of attention_tiled's two query blocks x four key
// groups, which this replaced), and no barrier stands between the first and the merge.  The two blocks are half a tile
// apart: while one's scores go through the softmax, the matrix cores take the other's eight products, one between every two
// exponentials (a wavefront issues in order: products in a row hold it for 32 cycles each, and a SIMD has two wavefronts
// here).  The exponentials are taken against the running maximum itself, though a reference that lags it by up to 2^8 would
// rescale the accumulators in the first tiles only and be 10 % faster (4 x 4096 24.2 us): the largest weights, which are 1 and
// just below it here, would be rounded anywhere in their binade, and the error against 64 bits grows by as much (2-norm,
// 4 x 4096: 2.62e-4 before, 2.88e-4 lagging, 2.56e-4 so; a reference half a power of two ahead, 2.69e-4, saves nothing).
// The queries come through LDS, 1 KiB a wavefront: as fragments from memory (32 rows a load) and behind three tiles of
// copies they held the first product up for 5000 cycles, now 2800.
//   4 x 4096 28.1 -> 27.6 us, 3 x 3500 25.0 -> 24.3, 5 x 3001 23.5 -> 23.0, 16 x 1000 11.4, 11.4, 16 x 600 9.1 -> 8.6, 20 x
//   640 9.2 -> 8.1.  (128 queries as two pairs and four key groups 48.9 on 8 x 4096, by the form above 46.8.)
// What bounds it: about 1.4 us per tile of two wavefronts on a SIMD, issue of 2 x (32 exponentials, 16 products, about 210
// others) at 12, 13 and 3.2 cycles at the clock that random operands leave, and about 6 us around the loop,
// 2.5 of them the launch, 1.9 the merge of eight partial results.  Taken back: a barrier per tile or per four (the
// wavefronts of a SIMD end within 1000 cycles of each other instead of 10000, 4 x 4096 25.5 -> 26.0), s_setprio (none).
constexpr int kPairWave = 4 * kOwnTile; // two places for K, two for V
constexpr int kPairLds = kOwnWaves * kPairWave + 64 * D * 2; // the tiles, the queries
static_assert(kPairLds >= 2 * kOwnWaves * kSlot * 4, "the partial results fit");

template <bool kRagged>
__device__ __forceinline__ void attention_pairs(const uint16_t *__restrict__ Q, const uint16_t *__restrict__ K,
                                                const uint16_t *__restrict__ V, uint16_t *__restrict__ Out, float scale,
                                                int64_t N, char *lds) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int qi = lane & 31, half = lane >> 5;
  uint32_t bx, by;
  place_of_workgroup(bx, by, N >= 256);
  const int64_t head0 = int64_t(by) * N, q0 = head0 + int64_t(bx) * 64;
  const int tiles = int((N + kOwnKeys - 1) / kOwnKeys), lastRows = int(N - int64_t(tiles - 1) * kOwnKeys);
  const int iters = tiles > wave ? (tiles - wave + kOwnWaves - 1) / kOwnWaves : 0;

  // copies, places and fragment addresses: as in attention_own_keys
  const __amdgpu_buffer_rsrc_t kRsrc = make_rsrc(K + head0 * D, N * D * 2), vRsrc = make_rsrc(V + head0 * D, N * D * 2);
  const __amdgpu_buffer_rsrc_t nothing = make_rsrc(K + head0 * D, 0); // past the last tile: nothing moves, but the copies count
  int kVoff[4], vVoff[4], kVoffT[4], vVoffT[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int r = c * 8 + (lane >> 3), rT = kRagged ? min(r, lastRows - 1) : r;
    const int kc = (lane & 7) ^ ((r ^ ((r >> 3) & 3)) & 7), vc = (lane & 7) ^ (((r >> 1) & 1) << 2);
    kVoff[c] = (r * D + kc * 8) * 2;
    vVoff[c] = (r * D + vc * 8) * 2;
    kVoffT[c] = (rT * D + kc * 8) * 2;
    vVoffT[c] = (rT * D + vc * 8) * 2;
  }
  char *own = lds + wave * kPairWave; // K, K, V, V
  auto dma = [&](const __amdgpu_buffer_rsrc_t &rsrc, const int (&off)[4], const int (&offT)[4], int i, int place) {
    LdsChar *dst = (LdsChar *)own + place * kOwnTile;
    const int tile = wave + i * kOwnWaves;
    const bool tail = kRagged && tile == tiles - 1;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(i < iters ? rsrc : nothing, dst + c * 1024, 16, tail ? offT[c] : off[c],
                                               i < iters ? tile * kOwnTile : 0, 0, 0);
  };
  auto dma_k = [&](int i) { dma(kRsrc, kVoff, kVoffT, i, i & 1); };
  auto dma_v = [&](int i) { dma(vRsrc, vVoff, vVoffT, i, 2 + (i & 1)); };
  int kRd[4], vRd[2];
#pragma unroll
  for (int ds = 0; ds < 4; ++ds)
    kRd[ds] = qi * 128 + ((((ds * 2 + half) ^ qi ^ ((qi >> 3) & 3)) & 7) << 4);
  {
    const int t = lane & 15, blk = (lane >> 4) & 1, row = half * 4 + (t >> 2);
#pragma unroll
    for (int db = 0; db < 2; ++db)
      vRd[db] = 2 * kOwnTile + row * 128 + ((((db ^ ((t >> 3) & 1)) << 2) | (blk << 1) | ((t & 3) >> 1)) * 16) + (t & 1) * 8;
  }
  const f32x16 zero = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  f32x16 oA[2] = {zero, zero}, oB[2] = {zero, zero}, sA, sB;
  constexpr float kNoKey = -3.40282347e38f; // a reference that every score is above, or -inf
  float mA = kNoKey, mB = kNoKey, lA = 0.0f, lB = 0.0f;
  const float c = scale * 1.44269504088896341f;
  f16x8 qf[2][4], kf[4], vf[2][2], pA[2], pB[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    pA[kk] = pB[kk] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
    vf[kk][0] = vf[kk][1] = f16x8{0, 0, 0, 0, 0, 0, 0, 0};
  }
  auto read_k = [&](int i) {
#pragma unroll
    for (int ds = 0; ds < 4; ++ds)
      kf[ds] = *reinterpret_cast<const f16x8 *>(own + (i & 1) * kOwnTile + kRd[ds]);
  };
  auto read_v = [&](int i) {
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int db = 0; db < 2; ++db) {
        const char *p = own + (i & 1) * kOwnTile + vRd[db] + kk * 16 * 128;
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4 *)(p));
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsI16x4 *)(p + 8 * 128));
        vf[kk][db] = __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
  };
  auto read_done = [] { // the fragments are in registers: their places may be filled again
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // computed here, not where it is used
  auto stay = [](auto &...v) { (pin(v), ...); };
  // One block's tile `i` through the softmax, step(0) .. step(7), the other block's products, between its exponentials, and
  // middle() behind the last of them.
  auto softmax = [&](f32x16 &s, f16x8 (&p)[2], f32x16 (&o)[2], float &m, float &l, int i, auto &&step, auto &&middle) {
    if (kRagged && wave + i * kOwnWaves == tiles - 1 && lastRows < kOwnKeys) { // uniform over the wavefront
#pragma unroll
      for (int r = 0; r < 16; ++r)
        s[r] = (r >> 2) * 8 + half * 4 + (r & 3) < lastRows ? s[r] : -__builtin_inff();
    }
    float part[2] = {s[0], s[1]};
#pragma unroll
    for (int r = 2; r < 16; ++r)
      part[r & 1] = fmaxf(part[r & 1], s[r]);
    const float mx = max_of_halves(fmaxf(part[0], part[1])) * c;
    if (__builtin_amdgcn_ballot_w64(mx > m) != 0) { // the running max moved for some query
      const float mNew = fmaxf(m, mx), alpha = __builtin_amdgcn_exp2f(m - mNew);
      m = mNew;
      l *= alpha;
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          o[db][r] *= alpha;
    }
    float x[2], e[2], sum[2] = {0.0f, 0.0f};
    u32x4 w[2];
    x[0] = __builtin_fmaf(s[0], c, -m);
    x[1] = __builtin_fmaf(s[1], c, -m);
    auto take = [&](int j) { // the exponentials of step j
      const f16x2 h = {static_cast<_Float16>(e[0]), static_cast<_Float16>(e[1])};
      uint32_t word = __builtin_bit_cast(uint32_t, h);
      sum[0] += e[0];
      sum[1] += e[1];
      stay(word, sum[0], sum[1]);
      w[j >> 2][j & 3] = word;
    };
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      step(j);
      if (j > 0)
        take(j - 1);
      e[0] = __builtin_amdgcn_exp2f(x[0]);
      e[1] = __builtin_amdgcn_exp2f(x[1]);
      if (j < 7) {
        x[0] = __builtin_fmaf(s[2 * j + 2], c, -m);
        x[1] = __builtin_fmaf(s[2 * j + 3], c, -m);
      }
      stay(x[0], x[1], e[0], e[1]);
      if (j == 7)
        middle();
      __builtin_amdgcn_sched_barrier(0);
    }
    take(7);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
      p[kk] = __builtin_bit_cast(f16x8, w[kk]);
    l += sum[0] + sum[1];
  };

  // The queries, 8 rows a wavefront, laid out as K's.
  {
    const int row = wave * 8 + (lane >> 3), there = kRagged ? int(min(int64_t(row), N - 1 - int64_t(bx) * 64)) : row;
    const int chunk = (lane & 7) ^ ((row ^ ((row >> 3) & 3)) & 7);
    const __amdgpu_buffer_rsrc_t qRsrc = make_rsrc(Q + q0 * D, (head0 + N - q0) * D * 2);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(qRsrc, (LdsChar *)lds + kOwnWaves * kPairWave + wave * 1024, 16,
                                             (there * D + chunk * 8) * 2, 0, 0, 0);
  }
  dma_k(0);
  dma_k(1);
  dma_v(0);
  wait_vmcnt<8>(); // the queries, K(0)
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  if (iters > 0) { // uniform over the wavefront
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int ds = 0; ds < 4; ++ds)
        qf[b][ds] = *reinterpret_cast<const f16x8 *>(lds + kOwnWaves * kPairWave + b * (32 * 128) + kRd[ds]);
    read_k(0);
    read_done();
    dma_v(1);
    dma_k(2);
#pragma unroll
    for (int ds = 0; ds < 4; ++ds)
      sA = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[ds], qf[0][ds], ds == 0 ? zero : sA, 0, 0, 0);
    for (int i = 0; i < iters; ++i) {
      // A's softmax; B's last tile times V(i - 1), B's scores of tile i
      softmax(sA, pA, oA, mA, lA, i, [&](int j) {
        if (j < 4)
          oB[j & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[j >> 1][j & 1], pB[j >> 1], oB[j & 1], 0, 0, 0);
        else
          sB = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[j - 4], qf[1][j - 4], j == 4 ? zero : sB, 0, 0, 0);
      }, [&] {
        wait_vmcnt<8>(); // K(i + 1), V(i)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        read_v(i);
        read_k(i + 1);
      });
      // B's softmax; A's tile i times V(i), A's scores of tile i + 1 (past the end of whatever is there, not used)
      softmax(sB, pB, oB, mB, lB, i, [&](int j) {
        if (j == 0) {
          read_done();
          dma_k(i + 3);
          dma_v(i + 2);
        }
        if (j < 4)
          oA[j & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[j >> 1][j & 1], pA[j >> 1], oA[j & 1], 0, 0, 0);
        else
          sA = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[j - 4], qf[0][j - 4], j == 4 ? zero : sA, 0, 0, 0);
      }, [] {});
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      oB[j & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[j >> 1][j & 1], pB[j >> 1], oB[j & 1], 0, 0, 0);
  }
  wait_vmcnt<0>();
  float *all = reinterpret_cast<float *>(lds);
  __syncthreads(); // everyone's tiles are done with
  put_partial(oA, mA, lA + other_half(lA), all + wave * kSlot, lane);
  put_partial(oB, mB, lB + other_half(lB), all + (kOwnWaves + wave) * kSlot, lane);
  __syncthreads();
  const int block = wave / 4; // four wavefronts merge a block of 32 queries
  merge_partials<kOwnWaves, 2>(all + block * (kOwnWaves * kSlot), Out, q0 + block * 32, head0 + N, wave % 4 * 2, lane, kRagged);
}

// What the tiled path takes, of the arguments and of the launch.
__device__ __forceinline__ bool attention_shaped(const uint16_t *Q, const uint16_t *K, const uint16_t *V,
                                                 const uint16_t *Out, float scale, int64_t ZH, int64_t N) {
  return N > 0 && N < (int64_t(1) << 24) && scale > 0.0f && gridDim.y == ZH && gridDim.z == 1 &&
         ((reinterpret_cast<uintptr_t>(Q) | reinterpret_cast<uintptr_t>(K) | reinterpret_cast<uintptr_t>(V) |
           reinterpret_cast<uintptr_t>(Out)) & 15) == 0;
}

} // namespace

extern "C" __global__ __launch_bounds__(kMaxThreads) void imex_flash_attention_fwd_f16(const uint16_t *Q,
                                                                                   const uint16_t *K,
                                                                                   const uint16_t *V,
                                                                                   uint16_t *Out, float sm_scale,
                                                                                   int64_t ZH, int64_t N_CTX) {
  __shared__ __attribute__((aligned(16))) char lds[kLdsBytes];
  // The launch says how many queries a workgroup takes (ceil(N_CTX / gridDim.x) = 64, 128 or 256) and
  // with how many wavefronts.  The tiled path assumes a positive scale (it takes the row maximum
  // before scaling) and 32-bit byte offsets inside one head.
  const bool shaped = attention_shaped(Q, K, V, Out, sm_scale, ZH, N_CTX);
  const int64_t gx = gridDim.x;
  const bool even = N_CTX % 256 == 0; // every tiling divides it
  if (shaped && blockDim.x == 512 && gx == (N_CTX + 63) / 64) {
    if (even)
      attention_tiled<2, 4, false>(Q, K, V, Out, sm_scale, N_CTX, lds);
    else
      attention_tiled<2, 4, true>(Q, K, V, Out, sm_scale, N_CTX, lds);
  } else if (shaped && blockDim.x == 512 && gx == (N_CTX + 127) / 128) {
    if (even)
      attention_tiled<4, 2, false>(Q, K, V, Out, sm_scale, N_CTX, lds);
    else
      attention_tiled<4, 2, true>(Q, K, V, Out, sm_scale, N_CTX, lds);
  } else if (shaped && blockDim.x == 512 && gx == (N_CTX + 255) / 256) {
    if (even)
      attention_tiled<8, 1, false>(Q, K, V, Out, sm_scale, N_CTX, lds);
    else
      attention_tiled<8, 1, true>(Q, K, V, Out, sm_scale, N_CTX, lds);
  } else if (shaped && blockDim.x == 1024 && gx == (N_CTX + 255) / 256) {
    if (even)
      attention_tiled<8, 2, false>(Q, K, V, Out, sm_scale, N_CTX, lds);
    else
      attention_tiled<8, 2, true>(Q, K, V, Out, sm_scale, N_CTX, lds);
  } else {
    attention_scalar(Q, K, V, Out, sm_scale, ZH, N_CTX);
  }
}

// One tiling each, for problems whose tilings by the rule above leave CUs idle or run a nearly empty last round
// (attentionVariant in KernelCatalog.cpp).  128 queries are the form above with the next block's scores formed ahead.
template <int QB, int KG, bool kScoresAhead>
__device__ __forceinline__ void attention_one_tiling(const uint16_t *Q, const uint16_t *K, const uint16_t *V,
                                                     uint16_t *Out, float scale, int64_t ZH, int64_t N, char *lds) {
  constexpr int64_t kQueries = 32 * QB;
  if (!attention_shaped(Q, K, V, Out, scale, ZH, N) || blockDim.x != QB * KG * kWave ||
      gridDim.x != (N + kQueries - 1) / kQueries)
    attention_scalar(Q, K, V, Out, scale, ZH, N);
  else if (N % 256 == 0)
    attention_tiled<QB, KG, false, kScoresAhead>(Q, K, V, Out, scale, N, lds);
  else
    attention_tiled<QB, KG, true, kScoresAhead>(Q, K, V, Out, scale, N, lds);
}

#define IMEX_ATTENTION_TILING(QUERIES, QB, KG, AHEAD)                                                                  \
  extern "C" __global__ __launch_bounds__(QB *KG *kWave) void imex_flash_attention_fwd_f16_q##QUERIES(                \
      const uint16_t *Q, const uint16_t *K, const uint16_t *V, uint16_t *Out, float sm_scale, int64_t ZH,             \
      int64_t N_CTX) {                                                                                                \
    __shared__ __attribute__((aligned(16))) char lds[kLdsBytes];                                                      \
    attention_one_tiling<QB, KG, AHEAD>(Q, K, V, Out, sm_scale, ZH, N_CTX, lds);                                      \
  }
extern "C" __global__ __launch_bounds__(kOwnWaves *kWave, 4) void imex_flash_attention_fwd_f16_q32(
    const uint16_t *Q, const uint16_t *K, const uint16_t *V, uint16_t *Out, float sm_scale, int64_t ZH, int64_t N_CTX) {
  __shared__ __attribute__((aligned(16))) char lds[kOwnLds];
  if (!attention_shaped(Q, K, V, Out, sm_scale, ZH, N_CTX) || blockDim.x != kOwnWaves * kWave || gridDim.x != (N_CTX + 31) / 32)
    attention_scalar(Q, K, V, Out, sm_scale, ZH, N_CTX);
  else if (N_CTX % 32 == 0)
    attention_own_keys<false>(Q, K, V, Out, sm_scale, N_CTX, lds);
  else
    attention_own_keys<true>(Q, K, V, Out, sm_scale, N_CTX, lds);
}
extern "C" __global__ __launch_bounds__(kOwnWaves *kWave) void imex_flash_attention_fwd_f16_q64(
    const uint16_t *Q, const uint16_t *K, const uint16_t *V, uint16_t *Out, float sm_scale, int64_t ZH, int64_t N_CTX) {
  __shared__ __attribute__((aligned(16))) char lds[kPairLds];
  if (!attention_shaped(Q, K, V, Out, sm_scale, ZH, N_CTX) || blockDim.x != kOwnWaves * kWave || gridDim.x != (N_CTX + 63) / 64)
    attention_scalar(Q, K, V, Out, sm_scale, ZH, N_CTX);
  else if (N_CTX % 64 == 0)
    attention_pairs<false>(Q, K, V, Out, sm_scale, N_CTX, lds);
  else
    attention_pairs<true>(Q, K, V, Out, sm_scale, N_CTX, lds);
}
IMEX_ATTENTION_TILING(128, 4, 2, true)
IMEX_ATTENTION_TILING(256, 8, 2, false)

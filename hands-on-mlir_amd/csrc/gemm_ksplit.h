#pragma once

#include "gemm_staged.h"
#include "rectangles.h"

namespace hom {
namespace gemmk {

// ================================================================== ksplit ==
// GEMMs with few output tiles: the wavefronts of a workgroup split K.
//
// Where a problem gives a CU one tile or less, the slab pipelines of
// gemm_pipe.h are a chain of latencies: K / 64 slabs one after the other, each
// behind a barrier (0.16 us a slab, 64 slabs at K = 4096).  Here each of the
// eight wavefronts computes the WHOLE tile over its own share of K, slab w, w +
// 8, .. of 64 k, out of LDS that no other wavefront touches.  The main loop has
// no barrier; two slabs per wavefront, sixteen per workgroup, are on their way
// at once; and a fragment is read from LDS once per slab instead of once per
// wavefront row or column of the tile.  The eight partial tiles meet in LDS
// behind the only barrier and are added in wavefront order.
//
// Slab pipeline before, this kernel, three sets of operands in turn, us: 100 x 768 x
// 768 5.6 -> 4.5, 256 x 704 x 1504 9.4 -> 6.2, 256 x 700 x 1500 10.0 -> 7.4, 64 x 1001 x
// 1003 6.6 -> 5.3, 1000 x 333 x 2777 14.3 -> 13.4; 3.5 us of a launch are not the K loop.
// On rows on 16 bytes it takes seven slabs for that, see ksplitPays() in runners.cpp.
//
// A tile is 16 MB x 16 NB.  What bounds it is the CU's L1 (60 bytes a clock where
// whole 128-byte lines are asked for), so a row-major B is not cut into tiles
// of fewer than 64 columns: 32 columns are half a line at the price of a whole one.
//
// LDS of a wavefront: A rows, and rows of a [N, K] B, of 64 k in 16-byte chunks
// permuted by swzK(); a row-major B as it lies in memory, 64 rows of 2 NT bytes,
// its 32-byte blocks of 16 columns permuted by ksplitSlot() so that the eight rows
// that half a transposing read touches fall into different banks.
//
// VEC: rows on 16-byte boundaries and K a multiple of 8; otherwise rows of any length
// from 8 values up.  Every load is of whole dwords, in the tensor or, as part of
// its first or last dword, two bytes in front of it or behind it; what a vector of A
// (or of a [N, K] B) holds behind the row's end is masked.  ODD_A, ODD_B: rows may start in the middle of a
// dword.  16-byte loads from there run at 17 bytes a clock instead of 46, so such a
// row is read from two bytes earlier and shifted into place, the last value of a
// vector coming from the next lane's.  The last value of a row's 128 bytes would be
// missing: slabs are of 63 k then, or tiles of a row-major B of 63 columns (a load of
// that value for each row cost more: 64 lines for 128 bytes).
// 33 x 1001 x 3001 unsplit on 16 x 64 tiles: 13.5 -> 8.7 us (33 x 1002 x 3002: 7.9 us).
//
// Split-K across workgroups (gridDim.y): the slices of a tile share an XCD (the
// grid's x extent is a multiple of eight) and the last to arrive adds them in
// slice order; see arriveAtTile().

constexpr int kKsplitWaves = 8, kKsplitThreads = kKsplitWaves * kWave;

// Position of 32-byte block `block` in row k of a row-major B slab of 64 columns.  A
// transposing read takes 32 bytes of rows r .. r+3 and r+8 .. r+11 (r a multiple
// of four) with its first 32 lanes: eight blocks that must differ modulo 256 bytes.
__device__ __forceinline__ int ksplitSlot(int k, int block) {
  return block ^ (((k >> 1) & 1) | ((k >> 3) & 1) << 1);
}

template <int MB, int NB> constexpr int ksplitWaveBytes() {
  constexpr int kSlab = (MB + NB) * 16 * 128, kPartial = MB * 16 * (NB * 64 + 16);
  return kSlab > kPartial ? kSlab : kPartial;
}
// Consecutive columns a thread finishes (all threads of a 32 x 64 tile have some).
constexpr int kKsplitOut = 4;

// alpha * v + beta * c, activated and stored: consecutive columns of row m, those
// in front of nEnd.  onVectors: rows of D start on whole vectors.
__device__ __forceinline__ void ksplitFinish(const GemmParams &p, int activation, int m, int n,
                                             int nEnd, bool onVectors, const float (&v)[kKsplitOut],
                                             const _Float16 (&c)[kKsplitOut]) {
  typedef _Float16 vec __attribute__((ext_vector_type(kKsplitOut)));
  vec o;
#pragma unroll
  for (int e = 0; e < kKsplitOut; e++) {
    float x = p.alpha * v[e];
    if (p.beta != 0.f)
      x += p.beta * float(c[e]);
    if (activation == int(Epilogue::kGeluErf))
      x = geluErf(x);
    else if (activation == int(Epilogue::kGeluTanh))
      x = geluTanh(x);
    o[e] = _Float16(x);
  }
  _Float16 *d = p.D + int64_t(m) * p.ldd + n;
  if (n + kKsplitOut <= nEnd) {
    // (8 bytes a lane, but sixteen lanes write a whole line: written through, 200 x
    // 2048 x 768 5.40 -> 5.35 us, 500 x 1024 x 512 5.04 -> 4.99, tiles of 16 rows equal.  Rows
    // that do not start on whole vectors: default policy, see store_policy.h)
    if (onVectors)
      storeWriteThrough(d, o);
    else
      asm volatile("global_store_dwordx2 %0, %1, off"
                   :
                   : "v"(d), "v"(__builtin_bit_cast(float2v, o))
                   : "memory");
  } else {
#pragma unroll
    for (int e = 0; e < kKsplitOut; e++)
      if (n + e < nEnd)
        d[e] = o[e];
  }
}
// The source of the same outputs (zeros without one).
__device__ __forceinline__ void ksplitSource(const GemmParams &p, int m, int n, int nEnd,
                                             _Float16 (&c)[kKsplitOut]) {
  typedef _Float16 vec __attribute__((ext_vector_type(kKsplitOut)));
  typedef vec vecAny __attribute__((aligned(2)));
#pragma unroll
  for (int e = 0; e < kKsplitOut; e++)
    c[e] = _Float16(0);
  if (p.beta == 0.f || m >= p.M || n >= nEnd)
    return;
  const _Float16 *src = p.C + int64_t(rowInPeriod(p, m)) * p.ldc + n;
  if (n + kKsplitOut <= nEnd) {
    const vec x = *reinterpret_cast<const vecAny *>(src);
#pragma unroll
    for (int e = 0; e < kKsplitOut; e++)
      c[e] = x[e];
  } else {
#pragma unroll
    for (int e = 0; e < kKsplitOut; e++)
      if (n + e < nEnd)
        c[e] = src[e];
  }
}

template <int MB, int NB, bool B_NK, bool VEC, bool ODD_A, bool ODD_B>
__global__ __launch_bounds__(kKsplitThreads, 2) void gemmKsplitKernel(
    const _Float16 *A, const _Float16 *B, int M, int N, int K, int lda, int ldb, int chunkM,
    uint32_t chunkMMagic, int chunkN, int xmLog, int slabsPerSlice, int activation,
    GemmParams rest) {
  (void)rest; // (through the argument pointer, behind the first loads)
  constexpr int MT = MB * 16, NT = NB * 16;
  constexpr bool ODD_K = ODD_A || (B_NK && ODD_B), ODD_N = !B_NK && ODD_B;
  constexpr int SLAB = ODD_K ? 63 : 64, COLS = ODD_N ? NT - 1 : NT; // used
  constexpr int A_VECS = MT / 8, B_VECS = NT / 8; // 16-byte vectors per lane and slab
  constexpr int A_BYTES = MT * 128;
  static_assert(B_NK || NT == 64, "rows of a row-major B slab are one cache line");
  constexpr int WAVE_BYTES = ksplitWaveBytes<MB, NB>();
  constexpr uint32_t kOob = 0x80000000u;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  unsigned char *const mine = smem + wave * WAVE_BYTES;
  // XCD id % 8 owns a rectangle of chunkM x chunkN tiles (chooseRectangles()).
  const int id = blockIdx.x, slice = blockIdx.y;
  const int xcd = id % 8, loc = id / 8, xm = xcd & ((1 << xmLog) - 1), xn = xcd >> xmLog;
  const int ln = int(divByMagic(uint32_t(loc), uint32_t(chunkM), chunkMMagic));
  const int m0 = (xm * chunkM + loc - ln * chunkM) * MT, n0 = (xn * chunkN + ln) * COLS;
  if (ln >= chunkN || m0 >= M || n0 >= N)
    return;
  const int slabs = (K + SLAB - 1) / SLAB, first = slice * slabsPerSlice;
  const int last = first + slabsPerSlice < slabs ? first + slabsPerSlice : slabs;
  // Descriptors based at this tile's first row (A, [N, K] B) or column block, on a
  // dword: rows past the edge of the tensor are outside and read as zero.
  struct Source {
    uint64_t base;
    int32_t bytes;
    uint32_t odd; // the tile starts in the middle of a dword
  };
  auto source = [](const _Float16 *tile, int64_t values, bool odd) {
    Source r;
    const uint64_t at = reinterpret_cast<uint64_t>(tile);
    r.odd = odd ? uint32_t(at >> 1) & 1u : 0u;
    r.base = at - r.odd * 2;
    const int64_t bytes = (values * 2 + r.odd * 2 + 3) & ~int64_t(3);
    r.bytes = bytes > 0x7ffffffcLL ? 0x7ffffffc : int32_t(bytes);
    return r;
  };
  const Source srcA = source(A + int64_t(m0) * lda, int64_t(M - m0) * lda, ODD_A);
  const Source srcB = B_NK ? source(B + int64_t(n0) * ldb, int64_t(N - n0) * ldb, ODD_B)
                           : source(B + n0, int64_t(K) * ldb - n0, ODD_B);
  const auto rsrcA = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(srcA.base), 0, srcA.bytes, 0x00020000);
  const auto rsrcB = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(srcB.base), 0, srcB.bytes, 0x00020000);
  // This lane's 16 bytes of an instruction's eight rows of 128 bytes.
  const uint32_t r8 = uint32_t(lane / 8), c8 = uint32_t(lane % 8 * 8);
  const uint32_t aFirst = r8 * uint32_t(lda) + c8 + srcA.odd, bFirst = r8 * uint32_t(ldb) + c8 + srcB.odd;
  auto onDword = [](uint32_t value, bool odd) { return (odd ? value & ~1u : value) * 2u; };

  // Slab s into register set setC: every lane adds one scalar per vector, and what
  // lies outside gets an offset outside the descriptor, which reads as zero
  // without touching memory: lanes past the end of a row, slabs past the last one.
  // (Rows past K of a row-major B end up behind the tensor by themselves.)
  half8 ra[2][A_VECS], rb[2][B_VECS];
  auto request = [&](auto setC, int s) {
    constexpr int S = decltype(setC)::value;
    const int k0 = s * SLAB;
    // (odd rows: the vector's first dword may hold the row's last value)
    const bool live = s < last, kIn = live && k0 + int(c8) < K + (ODD_K ? 1 : 0);
    const uint32_t aAt = kIn ? onDword(aFirst + uint32_t(k0), ODD_A) : kOob;
    const uint32_t bAt = B_NK   ? (kIn ? onDword(bFirst + uint32_t(k0), ODD_B) : kOob)
                         : live ? onDword(bFirst + uint32_t(k0) * uint32_t(ldb), ODD_B)
                                : kOob;
#pragma unroll
    for (int i = 0; i < A_VECS; i++)
      ra[S][i] = __builtin_bit_cast(
          half8, __builtin_amdgcn_raw_buffer_load_b128(rsrcA, aAt + uint32_t(i * 16) * uint32_t(lda), 0, 0));
#pragma unroll
    for (int i = 0; i < B_VECS; i++) {
      uint32_t at = bAt + uint32_t(i * 16) * uint32_t(ldb);
      if (ODD_K && !B_NK && i == B_VECS - 1) // (row 63: not of this slab)
        at = r8 == 7 ? kOob : at;
      rb[S][i] = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(rsrcB, at, 0, 0));
    }
  };
  // A vector read from two bytes early, by `shift` bits (0 or 16) into place.
  auto shiftIn = [](half8 v, uint32_t shift) {
    const uint4v w = __builtin_bit_cast(uint4v, v);
    // (lane + 1's first dword; what the last lane of eight gets is not used)
    const uint32_t next = uint32_t(__builtin_amdgcn_update_dpp(0, int(w[0]), 0x101, 0xf, 0xf, false));
    uint4v o;
    o[0] = __builtin_amdgcn_alignbit(w[1], w[0], shift);
    o[1] = __builtin_amdgcn_alignbit(w[2], w[1], shift);
    o[2] = __builtin_amdgcn_alignbit(w[3], w[2], shift);
    o[3] = __builtin_amdgcn_alignbit(next, w[3], shift);
    return __builtin_bit_cast(half8, o);
  };
  // The first `count` values of a vector, zeros behind them.
  auto keep = [](half8 v, int count) {
    uint4v w = __builtin_bit_cast(uint4v, v);
#pragma unroll
    for (int d = 0; d < 4; d++)
      w[d] &= count >= 2 * d + 2 ? 0xffffffffu : count == 2 * d + 1 ? 0xffffu : 0u;
    return __builtin_bit_cast(half8, w);
  };
  // LDS addresses: a few per lane, the rest are immediates.
  const int l16 = lane % 16, kb = lane / 16;
  unsigned char *aWrite[2], *bWrite[2];
  const unsigned char *aRead[2], *bRead[B_NK ? 2 : NB];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int r = lane / 8 + h * 8, c = lane % 8;
    aWrite[h] = mine + r * 128 + swzK(r, c) * 16;
    bWrite[h] = mine + A_BYTES + r * 128 + (B_NK ? swzK(r, c) * 16 : ksplitSlot(r, c / 2) * 32 + c % 2 * 16);
    aRead[h] = mine + l16 * 128 + swzK(l16, h * 4 + kb) * 16;
    if (B_NK)
      bRead[h] = mine + A_BYTES + l16 * 128 + swzK(l16, h * 4 + kb) * 16;
  }
  if (!B_NK) {
#pragma unroll
    for (int j = 0; j < NB; j++) { // (steps of 32 k and the second four rows: the same block)
      const int r = kb * 8 + l16 / 4;
      bRead[j] = mine + A_BYTES + r * 128 + ksplitSlot(r, j) * 32 + l16 % 4 * 8;
    }
  }
  auto stage = [&](auto setC, int s) {
    constexpr int S = decltype(setC)::value;
    const int k0 = s * SLAB;
    // (rows eight apart start alike)
    if constexpr (ODD_A) {
      const uint32_t shift = (aFirst + uint32_t(k0)) % 2 * 16;
#pragma unroll
      for (int i = 0; i < A_VECS; i++)
        ra[S][i] = shiftIn(ra[S][i], shift);
    }
    if constexpr (ODD_B) {
      const uint32_t shift = (bFirst + uint32_t(k0) * (B_NK ? 1u : uint32_t(ldb))) % 2 * 16;
#pragma unroll
      for (int i = 0; i < B_VECS; i++)
        rb[S][i] = shiftIn(rb[S][i], shift);
    }
    if (!VEC && k0 + SLAB > K) { // (the last slab of K)
      const int count = K - k0 - int(c8);
#pragma unroll
      for (int i = 0; i < A_VECS; i++)
        ra[S][i] = keep(ra[S][i], count);
      if (B_NK) {
#pragma unroll
        for (int i = 0; i < B_VECS; i++)
          rb[S][i] = keep(rb[S][i], count);
      } else if (ODD_B) { // (what follows the tensor in its last dword)
#pragma unroll
        for (int i = 0; i < B_VECS; i++)
          rb[S][i] = keep(rb[S][i], k0 + int(r8) + i * 8 < K ? 8 : 0);
      }
    } else if (ODD_K) { // 63 k
      const half8 none = {};
#pragma unroll
      for (int i = 0; i < A_VECS; i++)
        ra[S][i][7] = c8 == 56 ? none[7] : ra[S][i][7];
      if (B_NK) {
#pragma unroll
        for (int i = 0; i < B_VECS; i++)
          rb[S][i][7] = c8 == 56 ? none[7] : rb[S][i][7];
      }
    }
    // (vectors i and i + 2 are sixteen rows apart, which leaves the swizzles alone)
#pragma unroll
    for (int i = 0; i < A_VECS; i++)
      *reinterpret_cast<half8 *>(aWrite[i % 2] + i / 2 * (16 * 128)) = ra[S][i];
#pragma unroll
    for (int i = 0; i < B_VECS; i++)
      *reinterpret_cast<half8 *>(bWrite[i % 2] + i / 2 * (16 * 128)) = rb[S][i];
  };

  float4v acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; i++)
#pragma unroll
    for (int j = 0; j < NB; j++)
      acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&]() {
    // (a wavefront's LDS operations run in order: what other lanes wrote is there)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int kk = 0; kk < 2; kk++) {
      half8 fa[MB], fb[NB];
#pragma unroll
      for (int i = 0; i < MB; i++)
        fa[i] = *reinterpret_cast<const half8 *>(aRead[kk] + i * (16 * 128));
#pragma unroll
      for (int j = 0; j < NB; j++) {
        if constexpr (B_NK) {
          fb[j] = *reinterpret_cast<const half8 *>(bRead[kk] + j * (16 * 128));
        } else {
          typedef short short8v __attribute__((ext_vector_type(8)));
          short8v both;
#pragma unroll
          for (int h = 0; h < 2; h++) {
            const short4v t = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) short4v *)(bRead[j] + (kk * 32 + h * 4) * 128));
#pragma unroll
            for (int e = 0; e < 4; e++)
              both[h * 4 + e] = t[e];
          }
          fb[j] = __builtin_bit_cast(half8, both);
        }
      }
#pragma unroll
      for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < NB; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[j], fa[i], acc[i][j], 0, 0, 0);
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
  };

  using Set0 = std::integral_constant<int, 0>;
  using Set1 = std::integral_constant<int, 1>;
  int s = first + wave;
  request(Set0{}, s);
  request(Set1{}, s + kKsplitWaves);
  __builtin_amdgcn_sched_barrier(0);
  GemmParams p = {};
#if defined(__HIP_DEVICE_COMPILE__) // (the host pass only needs the kernel's stub)
  {
    constexpr int kLeading = 2 * 8 + 11 * 4, kAlign = alignof(GemmParams);
    constexpr int kRestOffset = (kLeading + kAlign - 1) / kAlign * kAlign;
    typedef const __attribute__((address_space(4))) GemmParams *RestPtr;
    RestPtr late = (RestPtr)((const __attribute__((address_space(4))) char *)
                                 __builtin_amdgcn_kernarg_segment_ptr() + kRestOffset);
    asm volatile("" : "+s"(late));
    p = *late;
  }
#endif
  // What this thread finishes: some columns of one row of the tile.
  constexpr int OPR = NT / kKsplitOut, kFinish = MT * OPR;
  static_assert(kFinish <= kKsplitThreads, "one thread per outputs");
  const bool out = tid < kFinish;
  const int row = tid / OPR, col = tid % OPR * kKsplitOut;
  _Float16 c[kKsplitOut];
  const int nEnd = n0 + COLS < N ? n0 + COLS : N;
  ksplitSource(p, out ? m0 + row : M, n0 + col, nEnd, c);
#pragma unroll 1
  for (; s < last; s += 2 * kKsplitWaves) {
    stage(Set0{}, s);
    request(Set0{}, s + 2 * kKsplitWaves);
    multiply();
    if (s + kKsplitWaves < last) {
      stage(Set1{}, s + kKsplitWaves);
      request(Set1{}, s + 3 * kKsplitWaves);
      multiply();
    }
  }

  // The partial tiles meet: rows of NT floats and 16 bytes.
  constexpr int ROW_B = NT * 4 + 16;
#pragma unroll
  for (int i = 0; i < MB; i++)
#pragma unroll
    for (int j = 0; j < NB; j++)
      *reinterpret_cast<float4v *>(mine + (i * 16 + l16) * ROW_B + (j * 16 + kb * 4) * 4) = acc[i][j];
  __syncthreads();
  float4v v = {0.f, 0.f, 0.f, 0.f};
  if (out) {
#pragma unroll
    for (int w = 0; w < kKsplitWaves; w++)
      v += *reinterpret_cast<const float4v *>(smem + w * WAVE_BYTES + row * ROW_B + col * 4);
  }
  const int numSlices = gridDim.y;
  if (numSlices > 1) {
    // (workspace: a vector per finishing thread, slices of a tile one after the other)
    const int tile = m0 / MT + n0 / COLS * p.tilesM;
    float4v *part = reinterpret_cast<float4v *>(p.workspace) + int64_t(tile) * numSlices * kFinish;
    if (out)
      part[slice * kFinish + tid] = v;
    if (p.tileArrivals == nullptr || !arriveAtTile(p, tile, numSlices, tid, smem))
      return;
    if (out) {
      v = float4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
      for (int sl = 0; sl < numSlices; sl++)
        v += part[sl * kFinish + tid];
    }
  }
  if (out && m0 + row < M && n0 + col < nEnd)
    ksplitFinish(p, activation, m0 + row, n0 + col, nEnd, COLS == NT && p.ldd % 8 == 0,
                 {v[0], v[1], v[2], v[3]}, c);
}

// The slices of a split-K launch, where the last workgroup to arrive does not add
// them: the same sums in the same order, a thread per finishing thread.
template <int MB, int NB>
__global__ __launch_bounds__(256) void ksplitReduceKernel(GemmParams p, int numSlices, int activation,
                                                       int cols) {
  constexpr int MT = MB * 16, NT = NB * 16;
  constexpr int OPR = NT / kKsplitOut, kFinish = MT * OPR;
  const int64_t idx = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (idx >= int64_t(p.tilesM) * p.tilesN * kFinish)
    return;
  const int tile = int(idx / kFinish), t = int(idx % kFinish);
  const int m = tile % p.tilesM * MT + t / OPR, n0 = tile / p.tilesM * cols, n = n0 + t % OPR * kKsplitOut;
  const int nEnd = n0 + cols < p.N ? n0 + cols : p.N;
  if (m >= p.M || n >= nEnd)
    return;
  _Float16 c[kKsplitOut];
  ksplitSource(p, m, n, nEnd, c);
  const float4v *part = reinterpret_cast<const float4v *>(p.workspace) + int64_t(tile) * numSlices * kFinish;
  float4v v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int sl = 0; sl < numSlices; sl++)
    v += part[sl * kFinish + t];
  ksplitFinish(p, activation, m, n, nEnd, cols == NT && p.ldd % 8 == 0, {v[0], v[1], v[2], v[3]}, c);
}

template <int MB, int NB, bool B_NK>
Status launchKsplit(const GemmProblem &pr, int activation, hipStream_t s) {
  constexpr int MT = MB * 16, NT = NB * 16;
  // (a row-major B is as well read from dwords as from 16-byte boundaries)
  auto rowsOn = [](const void *q, int64_t ld, int values) {
    return ld % values == 0 && reinterpret_cast<uintptr_t>(q) % uintptr_t(2 * values) == 0;
  };
  const bool vec = pr.K % 8 == 0 && rowsOn(pr.A, pr.lda, 8) && rowsOn(pr.B, pr.ldb, B_NK ? 8 : 2);
  // ([N, K]: rows of A and B have the same length, and one kernel for both)
  bool oddA = !rowsOn(pr.A, pr.lda, 2), oddB = !rowsOn(pr.B, pr.ldb, 2);
  if (B_NK)
    oddA = oddB = oddA || oddB;
  const int cols = !B_NK && oddB ? NT - 1 : NT, slab = oddA ? 63 : 64; // used
  LaunchPlan plan;
  Status st = planTiles(pr, MT, cols, slab, MT * NT, &plan);
  if (st != Status::kSuccess)
    return st;
  // (32-bit offsets: a row-major B is addressed from the matrix base, in whole slabs)
  HOM_CHECK_RET(B_NK || (pr.K + 63) / 64 * 64 * pr.ldb * 2 < (int64_t(1) << 31), Status::kInvalidArgument,
                "gemm: B larger than 2 GiB is not supported by this kernel");
  HOM_CHECK_RET((int64_t(MT) * pr.lda + pr.K) * 2 < (int64_t(1) << 31) &&
                    (int64_t(NT) * pr.ldb + pr.K) * 2 < (int64_t(1) << 31),
                Status::kInvalidArgument, "gemm: leading dimension too large");
  if (plan.nTiles == 0)
    return Status::kSuccess;
  constexpr int kLds = kKsplitWaves * ksplitWaveBytes<MB, NB>();
  auto kernel = vec            ? gemmKsplitKernel<MB, NB, B_NK, true, false, false>
                : oddA && oddB ? gemmKsplitKernel<MB, NB, B_NK, false, true, true>
                               : gemmKsplitKernel<MB, NB, B_NK, false, false, false>;
  if constexpr (!B_NK) {
    if (oddA != oddB)
      kernel = oddA ? gemmKsplitKernel<MB, NB, B_NK, false, true, false>
                    : gemmKsplitKernel<MB, NB, B_NK, false, false, true>;
  }
  static bool attrSet[5] = {};
  st = allowLds(kernel, kLds, &attrSet[vec ? 4 : 2 * oddA + oddB]);
  if (st != Status::kSuccess)
    return st;
  const int cus = deviceInfo().computeUnits > 0 ? deviceInfo().computeUnits : 256;
  const Rectangles r = chooseRectangles(plan.p.tilesM, plan.p.tilesN, MB, NB, pr.K, cus);
  GemmParams q = plan.p;
  bool sumInKernel = false;
  if (plan.splitK > 1 && plan.splitK <= 64 && !plan.callerWorkspace &&
      plan.nTiles <= kMaxArrivalTiles) {
    SplitKArrival arr;
    if (splitKArrival(s, &arr)) {
      q.tileArrivals = arr.words;
      q.misplaced = arr.misplaced;
      sumInKernel = true;
    }
  }
  kernel<<<dim3((unsigned)(8 * r.chunkM * r.chunkN), (unsigned)plan.splitK), dim3(kKsplitThreads), kLds, s>>>(
      q.A, q.B, q.M, q.N, q.K, int(q.lda), int(q.ldb), r.chunkM, magicFor(uint32_t(r.chunkM)),
      r.chunkN, r.xmLog, q.kTilesPerSlice, activation, q);
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  if (plan.splitK > 1 && !sumInKernel) {
    const int64_t threads = plan.nTiles * (MT * NT / kKsplitOut);
    ksplitReduceKernel<MB, NB><<<dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s>>>(
        plan.p, plan.splitK, activation, cols);
    HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  }
  return Status::kSuccess;
}

// (rows shorter than a vector: the scalar kernel)
template <int MB, int NB, int EPI, bool B_NK>
Status launchKsplitEntry(const GemmProblem &p, hipStream_t s) {
  if (p.K < 8 || p.N < 8)
    return launchStaged<64, 64, 32, 2, 2, EPI, B_NK, 1>(p, s);
  return launchKsplit<MB, NB, B_NK>(p, EPI, s);
}

} // namespace gemmk
} // namespace hom

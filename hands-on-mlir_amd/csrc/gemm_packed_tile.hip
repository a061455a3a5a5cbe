// GEMMs against packed weights for hundreds of rows and more: the counterpart of
// gemm_packed.hip whose workgroups share operands through LDS.
//
// Both operands arrive in fragment order (packedOffset() in kernels.h), so a slab
// of a tile is a row of whole kilobytes: buffer_load ... lds copies them in lane
// order, 1 KiB per instruction with one scalar offset, without a swizzle, and
// the fragment reads (32 rows x 16 k of v_mfma_f32_32x32x16_f16 = four runs of
// 256 bytes) have no bank conflicts.  Results in fragment order leave the
// accumulators as they are, in whole 256-byte runs, with no pass through LDS.
// That leaves LDS to the slab ring also while a tile is finished: workgroups are
// persistent and the ring runs on into the next tile, so its first slabs arrive
// under the epilogue instead of behind it.
//
// A layer norm in front of the GEMM is folded as in gemm_packed.hip.  The row
// sums are divided between the wavefronts of a tile row: each reads its share of
// the slab's A fragments once more (one LDS read in seven) and sums them between
// its MFMAs.  That costs a large GEMM more than a layer norm kernel of its own
// (16384 x 4096 x 1024: 126 -> 142 us), so the callers fold only where a launch
// is what counts.
#include "cross_lane.h"
#include "fast_div.h"
#include "packed_args.h"
#include "store_policy.h"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace hom {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float2v __attribute__((ext_vector_type(2)));

constexpr int kWave = 64;

template <class F, int... I>
__device__ __forceinline__ void unrolledImpl(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F> __device__ __forceinline__ void unrolled(F &&f) {
  unrolledImpl(f, std::make_integer_sequence<int, N>{});
}

#define HOM_LDS_PTR(p) ((__attribute__((address_space(3))) void *)(p))

// BM x BN tile, WM x WN wavefronts, slabs of SB * 32 k in a ring of NBUF LDS
// buffers.  ACT: 0 linear, 1 erf GELU, 2 tanh GELU; SRC: a residual source.
template <int BM, int BN, int WM, int WN, int SB, int NBUF, bool NORM_A, int ACT, bool SRC>
__global__ __launch_bounds__(WM *WN *kWave, NBUF *(BM + BN) * SB > 1280 ? 1 : WM *WN / 2) void packedTileKernel(
    const _Float16 *A, const _Float16 *B, int rowBlocks, int colBlocks, int slabs, int tilesN,
    int xcdQ, uint32_t groupMagic, int walk, int workers, int tiles, PackedArgs p) {
  constexpr int WAVES = WM * WN, WTM = BM / WM, WTN = BN / WN;
  constexpr int MI = WTM / 32, NI = WTN / 32, NM = MI * NI;
  constexpr int kBlocksA = BM / 16, kBlocksB = BN / 16;  // 16-row blocks of a tile
  constexpr int kKilo = (kBlocksA + kBlocksB) * SB;      // KiB of a slab
  constexpr int NV = kKilo / WAVES;                      // requests of a wavefront per slab
  constexpr int kStage = kKilo * 1024;
  constexpr int KSTEPS = 2 * SB; // k16 steps of a slab
  static_assert(kKilo % WAVES == 0 && kBlocksA * SB % WAVES == 0, "whole kilobytes per wavefront");
  constexpr uint32_t kOob = 0x80000000u;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid % kWave;
  if (int(blockIdx.x) >= workers) {
    readAhead<WAVES * kWave>(p.ahead, p.aheadBytes, int(blockIdx.x) - workers,
                             int(gridDim.x) - workers, tid);
    return;
  }
  const int xcdR = walk & 15, lastRows = (walk >> 4) & 15, fullGroups = walk >> 8;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int waveM = wave / WN, waveN = wave % WN;
  const int l32 = lane % 32, kb = lane / 32;
  const int steps = slabs * SB; // 32-k blocks of K

  [[maybe_unused]] const auto rsrcA = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<_Float16 *>(A), 0, rowBlocks * steps * 1024, 0x00020000);
  [[maybe_unused]] const auto rsrcB = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<_Float16 *>(B), 0, colBlocks * steps * 1024, 0x00020000);

  // Tile of workgroup number v: XCD v % 8 owns a contiguous run of tiles, which
  // walks groups of 8 tile rows column by column (both operands of the tiles an
  // XCD works on at a time then fit its L2).
  auto tileOf = [&](int v, int *tm, int *tn) {
    const int xcd = v % 8, loc = v / 8;
    const uint32_t tile = uint32_t(xcd * xcdQ + (xcd < xcdR ? xcd : xcdR) + loc);
    const uint32_t groupSize = uint32_t(8 * tilesN);
    const uint32_t g = divByMagic(tile, groupSize, groupMagic);
    const uint32_t in = tile - g * groupSize;
    if (int(g) < fullGroups) {
      *tm = int(g * 8 + in % 8);
      *tn = int(in / 8);
    } else {
      const uint32_t q = in / uint32_t(lastRows);
      *tm = int(g * 8 + in - q * uint32_t(lastRows));
      *tn = int(q);
    }
  };

  // ---- the requesting side: slab `reqSlab` of tile `reqV`, NBUF - 1 slabs ahead ----
  // Kilobyte c of a slab: 16-row block c / SB (of A, then of B), 32-k block c % SB.
  int reqV = blockIdx.x, reqSlab = 0, reqBuf = 0;
  uint32_t reqOff[NV]; // this wavefront's kilobytes: block offset + lane's 16 bytes
  auto aimAt = [&](int v) {
    int tm, tn;
    tileOf(v, &tm, &tn);
#pragma unroll
    for (int i = 0; i < NV; i++) {
      const int c = i * WAVES + wave;
      const bool isA = i * WAVES < kBlocksA * SB;
      const int block = isA ? tm * kBlocksA + c / SB : tn * kBlocksB + c / SB - kBlocksA;
      const bool in = block < (isA ? rowBlocks : colBlocks);
      reqOff[i] =
          in ? uint32_t(block * steps + c % SB) * 1024u + uint32_t(lane) * 16u : kOob;
    }
  };
  auto requestOne = [&](auto iC) {
#if defined(__HIP_DEVICE_COMPILE__) // (the builtin's LDS pointer type exists only for the GPU target)
    constexpr int I = decltype(iC)::value;
    unsigned char *dst = smem + reqBuf * kStage + (I * WAVES + wave) * 1024;
    if constexpr (I * WAVES < kBlocksA * SB)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcA, HOM_LDS_PTR(dst), 16, reqOff[I],
                                               uint32_t(reqSlab) * uint32_t(SB * 1024), 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrcB, HOM_LDS_PTR(dst), 16, reqOff[I],
                                               uint32_t(reqSlab) * uint32_t(SB * 1024), 0, 0);
#endif
  };
  auto advance = [&]() {
    reqBuf = reqBuf + 1 == NBUF ? 0 : reqBuf + 1;
    if (reqSlab + 1 < slabs) {
      reqSlab++;
    } else if (reqV + workers < tiles) {
      reqV += workers;
      reqSlab = 0;
      aimAt(reqV);
    } // (behind the last slab: the same one again, into a buffer nobody reads;
      // every slab then has the same number of requests behind it)
  };
  aimAt(reqV);
#pragma unroll 1
  for (int i = 0; i < NBUF - 1; i++) {
    unrolled<NV>(requestOne);
    advance();
  }

  // ---- the multiplying side ----
  // Fragment of 32-row pair i at k16 step s: the two blocks of the pair lie SB
  // KiB apart, step s is half s % 2 of k block s / 2.
  const int fragLane = (l32 / 16) * (SB * 1024) + kb * 256 + (lane % 16) * 16;
  const int aLane = waveM * (WTM / 16) * (SB * 1024) + fragLane;
  const int bLane = (kBlocksA + waveN * (WTN / 16)) * (SB * 1024) + fragLane;
  // Wave tiles of one or two MFMA blocks keep a whole slab's fragments: with a
  // set per step parity every k16 step would be an LDS round trip.
  constexpr bool kWhole = NM <= 2;
  constexpr int FSETS = kWhole ? KSTEPS : 2;
  half8 fa[FSETS][MI], fb[FSETS][NI];
  auto readFrag = [&](int buf, auto sC, auto uC) {
    constexpr int S = decltype(sC)::value, U = decltype(uC)::value;
    const unsigned char *st = smem + buf * kStage;
    constexpr int at = (S / 2) * 1024 + (S % 2) * 512;
    if constexpr (U < MI)
      fa[S % FSETS][U] =
          *reinterpret_cast<const half8 *>(st + aLane + U * (2 * SB * 1024) + at);
    else
      fb[S % FSETS][U - MI] =
          *reinterpret_cast<const half8 *>(st + bLane + (U - MI) * (2 * SB * 1024) + at);
  };
  float16v acc[MI][NI];
  // Row statistics: of the MI x KSTEPS fragments of A that a tile row's
  // wavefronts share, this one sums number r * WN + waveN for r = 0 .. NSTAT - 1,
  // which are all of the same rows (those of 32-row pair waveN % MI).
  static_assert(!NORM_A || (WN % MI == 0 && MI * KSTEPS % WN == 0), "shares of the row sums");
  constexpr int NSTAT = NORM_A ? MI * KSTEPS / WN : 0;
  half8 fs[NSTAT > 0 ? NSTAT : 1];
  float sum = 0.f, sq = 0.f;
  auto readStat = [&](int buf, auto rC) {
    constexpr int R = decltype(rC)::value;
    const int f = R * WN + waveN, i = waveN % MI, S = f / MI;
    fs[R] = *reinterpret_cast<const half8 *>(smem + buf * kStage + aLane + i * (2 * SB * 1024) +
                                             (S / 2) * 1024 + (S % 2) * 512);
  };
  auto addStat = [&](auto dC) { // quarter D % 4 of fragment D / 4
    constexpr int D = decltype(dC)::value, R = D / 4, E = D % 4;
    const half2v one = {_Float16(1), _Float16(1)};
    const half2v x = {fs[R][2 * E], fs[R][2 * E + 1]};
    sum = __builtin_amdgcn_fdot2(x, one, sum, false);
    sq = __builtin_amdgcn_fdot2(x, x, sq, false);
  };
  int buf = 0;
  bool landed = false; // the ring's slabs are known to be there
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NBUF - 2) * NV) : "memory");
  unrolled<kWhole ? KSTEPS : 1>([&](auto sC) {
    unrolled<MI + NI>([&](auto uC) { readFrag(0, sC, uC); });
  });

  // MFMAs of k16 step S with N memory operations and the quarters D0 .. D1 of
  // the row sums spread between them
  auto multiply = [&](auto sC, auto nC, auto d0C, auto d1C, auto &&op) {
    constexpr int S = decltype(sC)::value % FSETS, N = decltype(nC)::value;
    constexpr int D0 = decltype(d0C)::value, ND = decltype(d1C)::value - D0;
    unrolled<NM>([&](auto mC) {
      constexpr int m = decltype(mC)::value;
      unrolled<N>([&](auto qC) {
        constexpr int q = decltype(qC)::value;
        if constexpr (q * NM / (N > 0 ? N : 1) == m) {
          __builtin_amdgcn_sched_barrier(0);
          op(qC);
          __builtin_amdgcn_sched_barrier(0);
        }
      });
      acc[m / NI][m % NI] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
          fb[S][m % NI], fa[S][m / NI], acc[m / NI][m % NI], 0, 0, 0);
      unrolled<ND>([&](auto dC) {
        constexpr int d = decltype(dC)::value;
        if constexpr (d * NM / (ND > 0 ? ND : 1) == m) {
          __builtin_amdgcn_sched_barrier(0);
          addStat(std::integral_constant<int, D0 + d>{});
        }
      });
    });
    __builtin_amdgcn_sched_barrier(0);
  };
  // Every wavefront has its fragments of this slab, and the next one has landed
  // once its requests are all but the NBUF - 2 newest.  (Behind an epilogue the
  // ring is known to be there already, and the newest operations are the
  // epilogue's stores, which need not be waited for.)
  auto slabBarrier = [&](int it) {
    if (landed && it < NBUF - 2)
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NBUF - 2) * NV)
                   : "memory");
  };

  for (int v = blockIdx.x; v < tiles; v += workers) {
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
      for (int j = 0; j < NI; j++)
#pragma unroll
        for (int e = 0; e < 16; e++)
          acc[i][j][e] = 0.f;
    sum = sq = 0.f;
#pragma unroll 1
    for (int it = 0; it < slabs; it++) {
      const int next = buf + 1 == NBUF ? 0 : buf + 1;
      unrolled<KSTEPS>([&](auto sC) {
        constexpr int S = decltype(sC)::value;
        constexpr bool kLast = S == KSTEPS - 1;
        // this step's share of the requests that refill the buffer the previous
        // slab left
        constexpr int V0 = kLast ? NV : S * NV / (KSTEPS - 1);
        constexpr int V1 = kLast ? NV : (S + 1) * NV / (KSTEPS - 1);
        constexpr int kReads = kWhole ? 0 : MI + NI;
        // row sums: fragments read in this step (none in the last, whose reads
        // are the next slab's), and those summed in it, read a step earlier
        constexpr int R0 = kLast ? NSTAT : S * NSTAT / (KSTEPS - 1);
        constexpr int R1 = kLast ? NSTAT : (S + 1) * NSTAT / (KSTEPS - 1);
        constexpr int P0 = S > 0 ? (S - 1) * NSTAT / (KSTEPS - 1) : 0;
        constexpr int P1 = S > 0 ? S * NSTAT / (KSTEPS - 1) : 0;
        if constexpr (kLast) {
          advance();
          slabBarrier(it);
          if constexpr (kWhole) // (their sets are free)
            unrolled<KSTEPS - 1>([&](auto rC) {
              unrolled<MI + NI>([&](auto uC) { readFrag(next, rC, uC); });
            });
        }
        multiply(sC, std::integral_constant<int, kReads + (R1 - R0) + (V1 - V0)>{},
                 std::integral_constant<int, 4 * P0>{}, std::integral_constant<int, 4 * P1>{},
                 [&](auto qC) {
                   constexpr int q = decltype(qC)::value;
                   if constexpr (q < kReads)
                     readFrag(kLast ? next : buf,
                              std::integral_constant<int, kLast ? 0 : S + 1>{}, qC);
                   else if constexpr (q < kReads + R1 - R0)
                     readStat(buf, std::integral_constant<int, R0 + q - kReads>{});
                   else
                     requestOne(std::integral_constant<int, V0 + q - kReads - (R1 - R0)>{});
                 });
        if constexpr (kLast && kWhole)
          unrolled<MI + NI>([&](auto uC) { readFrag(next, sC, uC); });
      });
      buf = next;
    }

    // ---- epilogue: D in fragment order straight from the accumulators ----
    // acc[i][j][4 g + e]: row l32 of 32-row pair i, column 8 g + 4 kb + e of
    // 32-column block j: 8 bytes at g * 256 + (l32 % 16) * 16 + kb * 8 of the
    // kilobyte (row block, column block).  Rows past M in the last row block are
    // padding; row blocks past it fall outside the descriptors.
    int tm, tn;
    tileOf(v, &tm, &tn);
    const int wideBlocks = p.N / 32; // 32-column blocks of C and D
    const int block0 = tm * kBlocksA + waveM * (WTM / 16) + l32 / 16;
    const int col0 = (tn * BN + waveN * WTN) / 32;
    // ... in accumulator order; lane and lane ^ 32 swap halves, so that each loads and
    // stores whole 16 bytes, of the even (kb = 0) or odd g.
    const uint32_t laneOff = uint32_t(lane % 16) * 16u + uint32_t(kb) * 256u;
    const uint32_t bytesCD = uint32_t(rowBlocks) * uint32_t(wideBlocks) * 1024u;
    const auto rsrcD = __builtin_amdgcn_make_buffer_rsrc(p.D, 0, int32_t(bytesCD), 0x00020000);
    auto offsetOf = [&](int i, int j) {
      return (uint32_t(block0 + 2 * i) * uint32_t(wideBlocks) + uint32_t(col0 + j)) * 1024u +
             laneOff;
    };
    lanes4 cw[SRC ? MI : 1][SRC ? NI : 1][2];
    float2v rowStat[MI];
    float4v cs[NORM_A ? NI : 1][4];
    if constexpr (SRC) {
      const auto rsrcC = __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16 *>(p.C), 0,
                                                           int32_t(bytesCD), 0x00020000);
#pragma unroll
      for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NI; j++)
#pragma unroll
          for (int g = 0; g < 2; g++)
            cw[i][j][g] = __builtin_amdgcn_raw_buffer_load_b128(
                rsrcC, col0 + j < wideBlocks ? offsetOf(i, j) + g * 512u : kOob, 0, 0);
#pragma unroll
      for (int i = 0; i < MI; i++) {
        rowStat[i] = float2v{1.f, 0.f};
        const int m = (block0 + 2 * i) * 16 + lane % 16;
        if (p.statsIn)
          rowStat[i] = *reinterpret_cast<const float2v *>(p.statsIn +
                                                          int64_t(m < p.M ? m : p.M - 1) * 2);
      }
    }
    if constexpr (NORM_A) {
#pragma unroll
      for (int j = 0; j < NI; j++)
#pragma unroll
        for (int g = 0; g < 4; g++)
          cs[j][g] = *reinterpret_cast<const float4v *>(
              p.colSum + (col0 + j < wideBlocks ? (col0 + j) * 32 + g * 8 + kb * 4 : 0));
      float2v *stat = reinterpret_cast<float2v *>(smem + NBUF * kStage); // [WN][BM]
      {
        const float s = pairSum(sum), q = pairSum(sq);
        if (kb == 0)
          stat[waveN * BM + waveM * WTM + (waveN % MI) * 32 + l32] = float2v{s, q};
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
      for (int i = 0; i < MI; i++) {
        float2v t{0.f, 0.f};
#pragma unroll
        for (int w = i; w < WN; w += MI)
          t += stat[w * BM + waveM * WTM + i * 32 + l32];
        const float mu = t[0] * p.invK;
        const int m = (block0 + 2 * i) * 16 + lane % 16;
        // the difference cancels to a small negative number for near-constant
        // rows; clamped so that a tiny eps cannot turn it into a NaN
        float var = fmaxf(t[1] * p.invK - mu * mu, 0.f);
        const bool again = m < p.M && meanDominates(mu, var);
        if (__builtin_expect(__any(again), 0)) { // the 32 rows once more, the two halves of the wavefront in turn
          float d2 = 0.f;
          const uint32_t row = uint32_t((block0 + 2 * i) * steps) * 1024u +
                               uint32_t(lane % 16) * 16u + uint32_t(kb) * 256u;
#pragma unroll 2
          for (int s = 0; s < 2 * steps; s++) { // 16 k each
            const half8 x = __builtin_bit_cast(
                half8,
                __builtin_amdgcn_raw_buffer_load_b128(rsrcA, row + uint32_t(s) * 512u, 0, 0));
#pragma unroll
            for (int e = 0; e < 8; e++) {
              const float d = float(x[e]) - mu;
              d2 = fmaf(d, d, d2);
            }
          }
          d2 = pairSum(d2);
          var = again ? d2 * p.invK : var;
        }
        const float rstd = 1.0f / sqrtf(var + p.eps);
        rowStat[i] = float2v{rstd, -mu * rstd};
        if (p.statsOut && tn == 0 && waveN == 0 && kb == 0 && m < p.M)
          *reinterpret_cast<float2v *>(p.statsOut + int64_t(m) * 2) = rowStat[i];
      }
    }
    // Everything requested so far is there before the first store goes out: the
    // ring is then known to be complete for the next tile's first slabs.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    landed = true;
#pragma unroll
    for (int j = 0; j < NI; j++) {
      if (col0 + j >= wideBlocks)
        continue; // (the same for the whole wavefront)
#pragma unroll
      for (int i = 0; i < MI; i++)
#pragma unroll
        for (int g = 0; g < 4; g += 2) {
          half4 o[2];
          [[maybe_unused]] half8 c = {}; // g, then g + 1
          if constexpr (SRC)
            c = __builtin_bit_cast(half8, splitHalves(cw[i][j][g / 2]));
#pragma unroll
          for (int h = 0; h < 2; h++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
              float x = acc[i][j][4 * (g + h) + e];
              if constexpr (NORM_A)
                x = fmaf(rowStat[i][0], x, rowStat[i][1] * cs[j][g + h][e]);
              if constexpr (ACT == 1)
                x = geluErf(x);
              if constexpr (ACT == 2)
                x = geluTanh(x);
              if constexpr (SRC)
                x += float(_Float16(fmaf(float(c[4 * h + e]), rowStat[i][0], rowStat[i][1])));
              o[h][e] = _Float16(x);
            }
          // (written through, see store_policy.h: a wavefront's store is whole runs of
          // 256 bytes.  BERT-base 32 x 128 1430 -> 1379 us, 8 x 128 597 -> 585,
          // BERT-large 32 x 512 11.54 -> 11.42 ms)
          typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
          const u32x2 even = __builtin_bit_cast(u32x2, o[0]), odd = __builtin_bit_cast(u32x2, o[1]);
          __builtin_amdgcn_raw_buffer_store_b128(joinHalves(even[0], even[1], odd[0], odd[1]), rsrcD,
                                                 offsetOf(i, j) + g * 256u, 0, kWriteThroughAux);
        }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // (no request outlives the workgroup)
}

// NORMS: normalised A as well (tiles that only share a CU never get one).
template <int BM, int BN, int WM, int WN, int SB, int NBUF, bool NORMS = true>
Status launchTile(const PackedGemm &g, const PackedArgs &p, hipStream_t s) {
  if (g.only) {
    *g.only = {true, BM, BN, SB * 32};
    return Status::kSuccess;
  }
  constexpr int kLds = NBUF * (BM + BN) * 64 * SB + WN * BM * 8;
  const int tilesM = int((g.M + BM - 1) / BM), tilesN = int((g.N + BN - 1) / BN);
  const int tiles = tilesM * tilesN;
  const int cus = deviceInfo().computeUnits > 0 ? deviceInfo().computeUnits : 256;
  using Kernel = void (*)(const _Float16 *, const _Float16 *, int, int, int, int, int, uint32_t,
                          int, int, int, PackedArgs);
  constexpr auto normalised = [](auto act) -> Kernel {
    if constexpr (NORMS)
      return packedTileKernel<BM, BN, WM, WN, SB, NBUF, true, decltype(act)::value, false>;
    else
      return nullptr;
  };
  // [normalised A][linear, erf GELU, tanh GELU, linear + source]
  static const Kernel kernels[2][4] = {
      {packedTileKernel<BM, BN, WM, WN, SB, NBUF, false, 0, false>,
       packedTileKernel<BM, BN, WM, WN, SB, NBUF, false, 1, false>,
       packedTileKernel<BM, BN, WM, WN, SB, NBUF, false, 2, false>,
       packedTileKernel<BM, BN, WM, WN, SB, NBUF, false, 0, true>},
      {normalised(std::integral_constant<int, 0>{}), normalised(std::integral_constant<int, 1>{}),
       normalised(std::integral_constant<int, 2>{}), nullptr}};
  const int kind = g.C ? 3 : g.activation;
  HOM_CHECK_RET(kernels[g.normA][kind], Status::kInternal,
                "packed gemm: no %d x %d kernel of this kind", BM, BN);
  const Kernel kernel = kernels[g.normA][kind];
  static int resident[2][4] = {};
  int &res = resident[g.normA][kind];
  if (res == 0) {
    HOM_HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, kLds),
                Status::kInternal);
    int perCu = 0;
    HOM_HIP_RET(hipOccupancyMaxActiveBlocksPerMultiprocessor(
                    &perCu, reinterpret_cast<const void *>(kernel), WM * WN * kWave, kLds),
                Status::kInternal);
    res = std::max(8, perCu * cus / 8 * 8);
  }
  // (workgroups that read ahead go to CUs without a tile)
  const int workers = std::min(tiles, res);
  const int extra = aheadGroups<WM * WN * kWave>(p.aheadBytes, cus - tiles);
  const int lastRows = tilesM % 8 ? tilesM % 8 : 8;
  kernel<<<dim3((unsigned)(workers + extra)), dim3(WM * WN * kWave), kLds, s>>>(
      g.A, g.packedB, int((g.M + 15) / 16), int(g.N / 16), int(g.K / (32 * SB)), tilesN,
      tiles / 8, magicFor(uint32_t(8 * tilesN)), tiles % 8 | lastRows << 4 | (tilesM / 8) << 8,
      workers, tiles, p);
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}

} // namespace

namespace {
struct Tile {
  int bm, bn;
  double fixedUs; // per tile of a CU: first slab, epilogue
  double slabUs;  // per 64 k, one tile per CU
  double rate;    // bytes per us that all tiles together load at most
  // the same of workgroups that share a CU and fill each other's gaps
  double sharedFactor, sharedRate;
};
constexpr Tile kTiles[] = {{256, 256, 4.5, 1.09, 11.5e6, 1.0, 11.5e6},
                           {256, 128, 2.5, 0.57, 11.5e6, 0.93, 14.5e6},
                           {128, 128, 1.1, 0.43, 14.5e6, 0.88, 18.0e6},
                           {64, 128, 0.7, 0.27, 18.5e6, 0.8, 18.5e6},
                           {64, 64, 0.4, 0.20, 22.5e6, 0.8, 22.5e6},
                           {64, 192, 0.9, 0.40, 14.5e6, 1.0, 14.5e6}};
// (Row sums between the MFMAs cost a quarter of the main loop; least where a
// wavefront has three MFMAs to a fragment of A.)
constexpr double kRowSumFactor[] = {1.25, 1.25, 1.25, 1.25, 1.25, 1.1};

// More tiles than CUs: slabs of 32 k, so that two rings fit a CU and one
// workgroup's epilogue runs beside the other's main loop (128 x 128: 4096 x 3072 x 768
// with GELU 27.7 -> 24.9 us; 256 x 128: 27.1 -> 25.4, 8192 rows 46.9 -> 44.0).
// Otherwise 64 k per barrier (128 x 128: 4096 x 768 x 3072 28.1 -> 26.7), and also
// with the row sums of a folded layer norm, which need the registers.
bool sharesCu(const PackedGemm &g, int64_t tiles, int cus) { return tiles > cus && !g.normA; }
} // namespace

// Model of a tile's time in a chain of launches (us), fitted to M = 512 .. 16384
// x the shapes of BERT-base and -large (most within 10 %): launch, then per tile of
// the fullest CU a fixed part and its slabs, these no faster than all tiles'
// operands arrive or the matrix cores multiply at the clock the power allows
// (1.2 PFLOP/s).
PackedTileChoice choosePackedTile(const PackedGemm &g) {
  PackedTileChoice best{-1, 1e300};
  if (!g.aPacked || !g.dPacked || (g.C && !g.cPacked) || g.K % 64 != 0 || g.N % 32 != 0 ||
      (g.C && g.normA))
    return best;
  const int cus = deviceInfo().computeUnits > 0 ? deviceInfo().computeUnits : 256;
  for (int i = 0; i < int(sizeof(kTiles) / sizeof(kTiles[0])); i++) {
    const Tile &t = kTiles[i];
    const int64_t tiles = ((g.M + t.bm - 1) / t.bm) * ((g.N + t.bn - 1) / t.bn);
    const double perCu = double((tiles + cus - 1) / cus);
    const bool shared = i == 3 || i == 4 ? perCu > 1 : sharesCu(g, tiles, cus);
    const double loop =
        std::max({perCu * double(g.K) / 64 * t.slabUs * (shared ? t.sharedFactor : 1.0),
                  double(tiles) * (t.bm + t.bn) * double(g.K) * 2 / (shared ? t.sharedRate : t.rate),
                  2.0 * double(g.M) * double(g.N) * double(g.K) / 1.2e9});
    const double us = 2.2 + loop * (g.normA ? kRowSumFactor[i] : 1.0) +
                      perCu * (t.fixedUs + (g.activation ? 5e-5 * t.bm * t.bn : 0));
    if (us < best.us)
      best = {i, us};
  }
  return best;
}

Status launchPackedTile(int tile, const PackedGemm &g, const PackedArgs &p, hipStream_t s) {
  const int cus = deviceInfo().computeUnits > 0 ? deviceInfo().computeUnits : 256;
  auto shared = [&](int bm, int bn) {
    return sharesCu(g, ((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn), cus);
  };
  switch (tile) {
  case 0:
    return launchTile<256, 256, 2, 4, 1, 4>(g, p, s);
  case 1:
    return shared(256, 128) ? launchTile<256, 128, 4, 2, 1, 3, false>(g, p, s)
                            : launchTile<256, 128, 4, 2, 2, 3>(g, p, s);
  case 2:
    // (and not for so few slabs that the first one counts: 1024 x 3072 x 768 9.7 us
    // against 10.3)
    return shared(128, 128) || (g.K <= 1024 && !g.normA)
               ? launchTile<128, 128, 2, 4, 1, 4, false>(g, p, s)
               : launchTile<128, 128, 2, 4, 2, 4>(g, p, s);
  case 3:
    return launchTile<64, 128, 1, 4, 2, 4>(g, p, s);
  case 4:
    return launchTile<64, 64, 2, 2, 2, 4>(g, p, s);
  default: // (between 128 x 128 and 64 x 128: 1024 x 3072 x 768 11.5 -> 10.4 us, 2304 columns 10.0 -> 8.9)
    return launchTile<64, 192, 2, 2, 2, 3>(g, p, s);
  }
}

} // namespace hom

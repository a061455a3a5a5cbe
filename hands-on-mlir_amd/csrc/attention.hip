// Packed-QKV BERT self-attention with a key-padding mask, for gfx950.
//
//   QKV [bs, seq, 3, heads, 64] fp16 (per token: Q of all heads, then K, then V
//   -- the packing produced by the weight concatenation in
//   lib/Dialect/HOM/HOMFusionPass.cpp:317-346, TransformerEngine layout BS3HD),
//   cu_seqlens int32 [bs+1], Out [bs, seq, heads, 64].
//   Per (b, h):  S = scale * Q K^T over keys < len_b;  P = softmax(S) in fp32;
//   O = P V.  Query rows >= len_b are written as zeros.
// Replaces the cuDNN fused attention reached through
// include/NVGPUKernels/BertAttentionRunner.h:113-136.
//
// A workgroup of four wavefronts handles 128 or 64 query rows of one (batch,
// head): each wavefront owns 32 rows and walks every key block (long
// sequences, many workgroups), or two wavefronts share 32 rows and take every
// other key block (short sequences: fewer workgroups than CUs, the key walk of
// one wavefront is the critical path; the two halves are merged through LDS).
// Keys are walked in chunks of 128 (64 where they are copied straight into LDS): the
// whole workgroup stages the chunk's K and V rows into LDS (one barrier), then the
// wavefronts run over it in blocks of 64 keys (32 each) without further
// synchronisation.
// Both contractions run on v_mfma_f32_32x32x16_f16 and are issued transposed:
//   S^T = K Q^T   (A operand = K rows from LDS, B operand = Q rows in registers)
//   O^T = V^T P^T (A operand = V columns, B operand = P rows)
// With that orientation a lane holds, for ONE query row, 16 of the 32 scores of
// a key sub-block, so the online-softmax row reductions are in-lane plus one
// exchange with lane^32, and the probabilities already have the layout of the
// second MFMA's B operand: P never leaves registers.  The MFMA k index is free
// as long as both operands agree, so V is read in the key order the score
// accumulators happen to have: two runs of 4 consecutive keys per lane, each one
// ds_read_b64_tr_b16 (the transposing LDS read) from the row-major V tile.
// LDS rows are 128 bytes, unpadded; 16-byte chunks (K) / 64-byte groups (V) are
// XOR-permuted by row so that the fragment reads are bank-conflict free.
#include "attention_way.h"
#include "cross_lane.h"
#include "fast_div.h"
#include "packed_args.h"

#include <cstring>
#include <type_traits>

namespace hom {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef short short8v __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWave = 64;
#define HOM_LDS_PTR(p) ((__attribute__((address_space(3))) void *)(p))
// Head sizes 64, 128, 192 and 256 (template parameter D; the reference's
// contract is head size % 64 == 0).  A K or V row in LDS is D halves: 128 bytes = 8
// chunks of 16 bytes = 2 groups of 64 bytes for D = 64.  Two wavefronts share a
// SIMD up to head size 192: held to 256 registers, head size 128 went from 292
// registers and one wavefront to 212 and two, 138 -> 82 us at 32 x 512 x 16 heads
// and 24.6 -> 17.9 us at 8 x 384 x 16.
//
// Keys staged per barrier: 128, or 64 where two tiles of 128 rows would not fit
// the 64 KB of static LDS.
template <int D> struct Chunk {
  static constexpr int value = D <= 128 ? 128 : 64;
};
// chunk c (16 bytes) of K row r lives at position c ^ ((r >> 1) & 7) (rows of
// 128 bytes: two consecutive rows cover all banks once) or c ^ (r & 15) (rows
// of 256 or 512 bytes: every row starts at bank 0), so that the 128-bit
// fragment reads of 16 consecutive rows hit 16 distinct bank groups; rows of
// 384 bytes (24 chunks) permute inside groups of 8 chunks so that a position
// never leaves the row
template <int D> __device__ __forceinline__ int swzK(int row, int chunk) {
  return D == 64    ? chunk ^ ((row >> 1) & 7)
         : D == 192 ? chunk ^ (row & 7)
                    : chunk ^ (row & 15);
}
// 64-byte group g of V row k lives at position g ^ ((k >> 1) & 1), or
// g ^ (k & 3) for rows whose group count is a multiple of 4: a transposing read
// touches 64 bytes of each of rows k..k+3
template <int D> __device__ __forceinline__ int swzV(int k, int group) {
  return D == 64 || D == 192 ? group ^ ((k >> 1) & 1) : group ^ (k & 3);
}

// Kernels whose launches may have all first query tiles first (attentionTilesOutside).  On eight wavefronts
// 32:512:12 of 192 takes 104.8 us so instead of 102.1.
template <int NW, int KS, int D, bool DMA>
constexpr bool kTilesOutside = DMA && KS == 2 && NW == 4 && D >= 128;

// 16 bytes of the result, which starts on an 8-byte boundary: the hardware takes that,
// and the type promises no more.  (As inline assembly the stores stay in source order
// with an address each: 39 x 35 x 1 heads of 64 3.31 us, 3.27 so.)  Default policy:
// written through, BERT-base 1 x 64 took 265 us a request instead of 263.
__device__ __forceinline__ void storeVector(_Float16 *p, u32x4 v) {
  typedef u32x4 onEight __attribute__((aligned(8)));
  *reinterpret_cast<onEight *>(p) = v;
}

// NW wavefronts per workgroup, KS of them share each group of 32 query rows
// and split its key blocks between them (KS = 1: every wavefront walks all
// keys of its own 32 rows; KS = 2: half the serial work per wavefront, for
// short sequences where there are fewer workgroups than CUs and the key walk
// of one wavefront is the critical path; the halves are merged through LDS).
// PACKED_IN: QKV in fragment order (packedOffset() in kernels.h): the 8 values of
// a token row that a vector takes are contiguous there as well, only the address
// of a row differs.
// PIPE: the next chunk's scores between this chunk's exponentials, so that one
// wavefront has the matrix cores and the vector ALU at work at once (a kernel that
// takes them in turn is bound by the sum of both, also with two wavefronts on a SIMD).
// It costs the registers of another block's scores; from how many tokens on it pays:
// attentionOverlapsScores().  Not for head size 64 with whole rows (us, lengths uniform in [seq / 4,
// seq], 32:512:16 37.2 -> 40.1: two wavefronts a SIMD instead of four), 192 (32:512:12 102.1
// -> 104.7, spills) and fragment order (requests, BERT-base 8 x 384 1315 -> 1328, 2 x 700 equal).
template <int D, int KS, bool PACKED_IN, bool DMA>
constexpr bool kPipe = DMA && !PACKED_IN && (D == 128 || (KS == 2 && (D == 64 || D == 256)));
template <int NW, int KS, int D, bool PACKED_IN, bool DMA, bool PIPE>
__global__ __launch_bounds__(NW *kWave)
__attribute__((amdgpu_waves_per_eu(D <= 128 || NW == 8 ? 2 : 1, D == 64 && KS == 1 ? 4 : (D <= 128 || NW == 8 ? 2 : 1)))) void bertAttentionKernel(
    const _Float16 *__restrict__ qkv, const int32_t *__restrict__ cu,
    _Float16 *__restrict__ out, int seq, int heads, int numQTiles, int bs,
    float scale, int packedOut, uint32_t numQMagic, uint32_t headsMagic, const char *ahead,
    int64_t aheadBytes) {
  static_assert(D == 64 || D == 128 || D == 192 || D == 256, "head size");
  static_assert(D <= 128 || KS == 1 || DMA, "the key-split variant stages 128 keys per chunk");
  static_assert(!PACKED_IN || D == 64, "fragment order is read at head size 64");
  constexpr int kChunk = DMA ? 64 : Chunk<D>::value;
  constexpr int SBW = DMA && KS == 2 ? 1 : 2; // 32-key sub-blocks a wavefront takes at a time
  // A wavefront at its MFMAs goes first, so that the other one of the SIMD is at its
  // softmax meanwhile (head size 64, chunks by DMA: 20 x 700 x 12 30.2 -> 29.1 us, 32 x 512
  // x 16 equal; through registers 8 x 128 x 12 4.18 -> 4.25; head size 128: equal; 192:
  // 52.9 -> 53.3).
  auto priority = [](auto pC) {
    if constexpr (D == 64 && DMA)
      __builtin_amdgcn_s_setprio(decltype(pC)::value);
  };
  using First = std::integral_constant<int, 1>;
  using Even = std::integral_constant<int, 0>;
  constexpr int kHeadDim = D;
  constexpr int kRowB = D * 2;               // bytes of a K or V row
  constexpr int CPR = D / 8;                 // 16-byte chunks per row
  constexpr int kTileBytes = kChunk * kRowB; // one K or V chunk in LDS
  constexpr int kThreads = NW * kWave;
  constexpr int QG = NW / KS; // groups of 32 query rows per workgroup
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  unsigned char *sK = smem, *sV = smem + kTileBytes;

  const int tid = threadIdx.x, lane = tid % kWave;
  // (the same for every lane: what depends on it stays in scalar registers)
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int l32 = lane % 32, hb = lane / 32;
  const int qg = wave % QG, kh = wave / QG; // query group, key share
  // Workgroup id -> (query tile, head, batch).  Workgroups are dealt to the 8
  // XCDs round-robin by id, and the query tiles of one (batch, head) read the
  // same K and V: ids that differ by 8 (same XCD, launched back to back) walk
  // the query tiles of one pair, so K/V are fetched into one L2 once instead
  // of once per XCD.  Needs the pair count to be a multiple of 8; the
  // 2-wavefront variant (few workgroups, launch-bound) keeps the plain order.
  // The key-split variant is launched on a (query tile, head, batch) grid: the
  // same order of workgroups as a flat id, without the divisions that would
  // stand between the kernel's entry and its first loads.
  const int pairs = bs * heads;
  int qTile, head, b;
  if (KS == 1 || DMA) {
    const int id = blockIdx.x;
    if constexpr (PACKED_IN) {
      if (id >= numQTiles * pairs) {
        readAhead<kThreads>(ahead, aheadBytes, id - numQTiles * pairs,
                            int(gridDim.x) - numQTiles * pairs, tid);
        return;
      }
    }
    int pair;
    if (kTilesOutside<NW, KS, D, DMA> && attentionTilesOutside(pairs, numQTiles)) {
      qTile = int(divByMagic(uint32_t(id), uint32_t(pairs), numQMagic));
      pair = id - qTile * pairs;
    } else if (pairs % 8 == 0) {
      const uint32_t t = uint32_t(id) / 8, g = divByMagic(t, uint32_t(numQTiles), numQMagic);
      qTile = int(t - g * uint32_t(numQTiles));
      pair = int(g * 8 + uint32_t(id) % 8);
    } else {
      pair = int(divByMagic(uint32_t(id), uint32_t(numQTiles), numQMagic));
      qTile = id - pair * numQTiles;
    }
    b = int(divByMagic(uint32_t(pair), uint32_t(heads), headsMagic));
    head = pair - b * heads;
  } else {
    qTile = blockIdx.x;
    head = blockIdx.y;
    b = blockIdx.z;
    if constexpr (PACKED_IN) {
      const int plane = numQTiles * heads; // workgroups of a batch entry
      if (b * heads >= pairs) {
        readAhead<kThreads>(ahead, aheadBytes, b * plane + head * numQTiles + qTile - numQTiles * pairs,
                            int(gridDim.z) * plane - numQTiles * pairs, tid);
        return;
      }
    }
  }
  const int q0 = qTile * (QG * 32) + qg * 32;
  const int cuLo = cu[b], cuHi = cu[b + 1]; // consumed after the first loads are out
  __builtin_amdgcn_sched_barrier(0); // requested here, not where they are consumed

  const int64_t tokStride = int64_t(3) * heads * kHeadDim;
  const _Float16 *base = qkv + int64_t(b) * seq * tokStride;
  const _Float16 *qBase = base + head * kHeadDim;
  const _Float16 *kBase = base + (heads + head) * kHeadDim;
  const _Float16 *vBase = base + (2 * heads + head) * kHeadDim;
  const int64_t outStride = int64_t(heads) * kHeadDim;
  _Float16 *oBase = out + int64_t(b) * seq * outStride + head * kHeadDim;
  // Output columns 32 d + 8 g + 4 hb .. + 3 of this lane's query: oRow + d * oWide +
  // g * oEight (packedOut: fragment order).
  const int oWide = packedOut ? 512 : 32, oEight = packedOut ? 128 : 8;
  _Float16 *const oRow =
      (packedOut ? out + packedOffset(int64_t(b) * seq + q0 + l32, head * kHeadDim, outStride)
                 : oBase + int64_t(q0 + l32) * outStride) +
      hb * 4;

  // Key-split variant (short sequences, few workgroups: latency is what
  // counts): K and V rows of a 128-key chunk travel global -> registers -> LDS,
  // 16 bytes per vector.  The loads are unconditional (rows past the end of the tensor
  // are clamped, rows past the sequence end are zeroed on the way to LDS), so
  // the first chunk's loads and the Q loads are issued before the sequence
  // length has arrived.  The other variant serves long sequences with many
  // workgroups per CU, which cover each other's staging; there the early loads
  // are wasted on all-padding workgroups, and prefetching the next chunk into
  // registers measured 3-8 % slower than loading each chunk when it is due
  // (also with barriers that do not wait for the prefetch).
  // (D = 128: the prefetched rows would take 64 more registers than there are)
  // PACKED_IN: 8 values from column 8 * c8 of part `part` (0 Q, 1 K, 2 V) of token
  // row `row`, as an offset in halves
  const int wide = 3 * heads * (kHeadDim / 32); // 32-column blocks of QKV
  auto packedAt = [&](int row, int part, int c8) {
    const int t = b * seq + row;
    return (int64_t(t / 16) * wide + (part * heads + head) * (kHeadDim / 32) + c8 / 4) * 512 +
           (c8 % 4) * 128 + (t % 16) * 8;
  };
  constexpr bool kPrefetch = KS == 2 && D == 64 && !DMA;
  constexpr int VPT = kChunk * CPR / kThreads; // vectors of K (and of V) per thread
  half8 rk[VPT], rv[VPT];
  auto loadChunk = [&](int key0) {
#pragma unroll
    for (int i = 0; i < VPT; i++) {
      const int v = tid + i * kThreads;
      const int r = v / CPR, c = v % CPR;
      const int row = key0 + r < seq ? key0 + r : seq - 1;
      rk[i] = *reinterpret_cast<const half8 *>(
          PACKED_IN ? qkv + packedAt(row, 1, c) : kBase + int64_t(row) * tokStride + c * 8);
      rv[i] = *reinterpret_cast<const half8 *>(
          PACKED_IN ? qkv + packedAt(row, 2, c) : vBase + int64_t(row) * tokStride + c * 8);
    }
  };
  if (kPrefetch)
    loadChunk(0);
  // Q fragments (B operand of S^T = K Q^T): lane (q = l32, hb) holds
  // Q[q][kk*16 + hb*8 .. +8] for kk = 0..3, pre-multiplied by nothing: the scale
  // is applied to the fp32 scores.
  half8 fq[kHeadDim / 16];
  {
    // rows past the tensor are clamped: what they produce is never stored
    const int q = q0 + l32 < seq ? q0 + l32 : seq - 1;
#pragma unroll
    for (int kk = 0; kk < kHeadDim / 16; kk++)
      fq[kk] = *reinterpret_cast<const half8 *>(
          PACKED_IN ? qkv + packedAt(q, 0, kk * 2 + hb)
                    : qBase + int64_t(q) * tokStride + kk * 16 + hb * 8);
  }

  int len = cuHi - cuLo;
  len = len < 0 ? 0 : (len > seq ? seq : len);
  // A workgroup whose query rows are all padding has nothing to compute.  (Not
  // in the key-split variant: an early exit ahead of the first use of the
  // prefetched rows lets the compiler move their loads behind the test, i.e.
  // behind the arrival of the sequence length.  Such a workgroup walks one
  // empty chunk there and stores zeros at the end.)
  if ((KS == 1 || DMA) && qTile * (QG * 32) >= len) {
    const int q = q0 + l32;
    if (q < seq && kh == 0) {
      const u32x4 z = {};
#pragma unroll
      for (int c = 0; c < CPR; c += 2) // (the two lanes of a row take turns)
        storeVector(oRow - hb * 4 + c / 4 * oWide + (c % 4 + hb) * oEight, z);
    }
    return;
  }

  constexpr int DB = D / 32;
  float16v accO[DB]; // O^T: 32-wide d blocks
#pragma unroll
  for (int d = 0; d < DB; d++)
#pragma unroll
    for (int e = 0; e < 16; e++)
      accO[d][e] = 0.f;
  // rowMax: reference of the exponent, in raw (unscaled) score units
  float rowMax = -INFINITY, rowSum = 0.f;
  const float scaleLog2e = scale * 1.44269504088896340736f;

  // Per-lane constants of the fragment addresses.
  const int swzLane = swzK<D>(l32, 0);         // K: the row term for row = 32*x + l32
  const int trRow = (lane % 16) / 4;           // V: source row inside a run of 4 keys
  const int trCol = ((lane % 32) / 16) * 16 + (lane % 4) * 4;
  const int vSwz = swzV<D>(trRow, 0);          // key bases are multiples of 4

  // Staging without prefetch: thread t copies 16-byte vector t % 8 of rows
  // t / 8 + i * kThreads / 8.  Both swizzles depend on row bits that the
  // per-vector row step (a multiple of 16) leaves alone, so the LDS
  // destinations are one base plus immediates.
  // (Head sizes above 128: the row step is not a multiple of 16, or not a
  // whole number; those compute every vector's addresses, see below.)
  constexpr bool kFastStage = kThreads % CPR == 0 && (kThreads / CPR) % 16 == 0;
  static_assert(kFastStage || D > 128, "row step per vector must leave the swizzles alone");
  // (fragment order: 16 rows further on is one row of blocks further on; the
  // descriptors cannot end at row `len` there, so rows past it are aimed outside)
  const uint32_t rowBytes = PACKED_IN ? uint32_t(wide) * 64u : uint32_t(tokStride) * 2u;
  const uint32_t stageOff =
      PACKED_IN ? uint32_t(packedAt(tid / CPR, 1, tid % CPR)) * 2u
                : uint32_t(tid / CPR) * rowBytes + uint32_t(tid % CPR) * 16u;
  const uint32_t vFromK = PACKED_IN ? uint32_t(heads * (kHeadDim / 32)) * 1024u : 0u;
  const int stageK = (tid / CPR) * kRowB + swzK<D>(tid / CPR, tid % CPR) * 16;
  const int stageV = (tid / CPR) * kRowB + swzV<D>(tid / CPR, (tid % CPR) / 4) * 64 +
                     ((tid % CPR) % 4) * 16;
  const int32_t stageBytes = PACKED_IN ? int32_t(uint32_t((bs * seq + 15) / 16) *
                                                 uint32_t(wide) * 1024u)
                                       : int32_t(uint32_t(len) * rowBytes);
  const auto rsrcK = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<_Float16 *>(PACKED_IN ? qkv : kBase), 0, stageBytes, 0x00020000);
  const auto rsrcV = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<_Float16 *>(PACKED_IN ? qkv : vBase), 0, stageBytes, 0x00020000);

  // uniform over the workgroup; at least one round in the key-split variant,
  // whose first chunk is already on its way
  const int numChunks =
      KS == 2 && len <= kChunk ? 1 : (len + kChunk - 1) / kChunk;
  // DMA: chunk ch travels global -> LDS (buffer_load ... lds) into buffer ch % 2
  // while the chunk before it is worked on.  An instruction fills 1 KiB in lane
  // order, so the swizzles are applied on the source side: vector v of a tile
  // lies at byte 16 v, and the lane fetches the chunk that belongs there.  Rows past
  // the sequence end are outside the descriptors and arrive as zeros.
  uint32_t dmaK[DMA ? VPT : 1], dmaV[DMA ? VPT : 1];
  if constexpr (DMA) {
#pragma unroll
    for (int i = 0; i < VPT; i++) {
      const int v = tid + i * kThreads, r = v / CPR, pc = v % CPR;
      const int cK = swzK<D>(r, pc), cV = swzV<D>(r, pc / 4) * 4 + pc % 4;
      dmaK[i] = PACKED_IN ? uint32_t(packedAt(r, 1, cK)) * 2u
                          : uint32_t(r) * rowBytes + uint32_t(cK) * 16u;
      dmaV[i] = PACKED_IN ? uint32_t(packedAt(r, 2, cV)) * 2u
                          : uint32_t(r) * rowBytes + uint32_t(cV) * 16u;
    }
  }
  constexpr float kSumLimit = 4096.0f;
  auto requestTile = [&](auto valuesC, int ch) { // K or V rows of chunk ch
#if defined(__HIP_DEVICE_COMPILE__) // (the builtin's LDS pointer type exists only for the GPU target)
    if constexpr (DMA) {
      constexpr bool kValues = decltype(valuesC)::value;
      const uint32_t chunkOff = uint32_t(ch * kChunk) * rowBytes;
      unsigned char *dst =
          smem + (ch % 2) * (2 * kTileBytes) + (kValues ? kTileBytes : 0) + wave * 1024;
#pragma unroll
      for (int i = 0; i < VPT; i++) {
        const bool out = PACKED_IN && ch * kChunk + (tid + i * kThreads) / CPR >= len;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            kValues ? rsrcV : rsrcK, HOM_LDS_PTR(dst + i * (kThreads * 16)), 16,
            out ? 0x80000000u : (kValues ? dmaV[i] : dmaK[i]) + chunkOff, 0, 0, 0);
      }
    }
#endif
  };
  auto requestChunk = [&](int ch) {
    requestTile(std::false_type{}, ch);
    requestTile(std::true_type{}, ch);
  };
  // ---- O^T += V^T P^T: group g of 16 keys, whose probabilities are prob(g) ----
  auto weighValues = [&](const unsigned char *sV, int blk, auto &&prob) {
    // Transposing reads issued and waited for by hand: in front of its
    // own the compiler would wait for every copy into LDS
    // that is on its way, i.e. for the whole next chunk.
    // INVARIANT: what an asm read writes is not valid until the wait.  Every
    // destination is an in/out operand of a wait, so that no use of it can
    // move ahead of that one; that the register allocator does not copy or
    // spill one in between either is checked on the compiled kernels
    // (tests/test_attention_assembly.py).
    constexpr int kGroups = SBW * 2, kSets = D <= 128 ? 2 : 1;
    static_assert(DB % 2 == 0, "a wait takes the reads of two column blocks");
    const uint32_t vLane = uint32_t(uintptr_t(HOM_LDS_PTR(sV))) +
                           uint32_t((blk + 4 * hb + trRow) * kRowB + trCol * 2);
    short4v run[kSets][DB][2];
    auto readGroup = [&](auto gC) {
      constexpr int g = decltype(gC)::value;
#pragma unroll
      for (int d = 0; d < DB; d++) {
        const uint32_t at = vLane + uint32_t((d ^ vSwz) * 64);
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2"
                     : "=v"(run[g % kSets][d][0])
                     : "v"(at), "i"(g * 16 * kRowB));
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2"
                     : "=v"(run[g % kSets][d][1])
                     : "v"(at), "i"((g * 16 + 8) * kRowB));
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    __builtin_amdgcn_sched_barrier(0);
    readGroup(std::integral_constant<int, 0>{});
    priority(First{});
    auto pvGroup = [&](auto gC) {
      constexpr int g = decltype(gC)::value;
      constexpr bool kMore = g + 1 < kGroups;
      using Next = std::integral_constant<int, kMore ? g + 1 : 0>;
      const half8 fp = prob(gC);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (kMore && kSets == 2)
        readGroup(Next{});
#pragma unroll
      for (int d = 0; d < DB; d += 2) // (the first one waits for all of them)
        asm volatile("s_waitcnt lgkmcnt(%4)"
                     : "+v"(run[g % kSets][d][0]), "+v"(run[g % kSets][d][1]),
                       "+v"(run[g % kSets][d + 1][0]), "+v"(run[g % kSets][d + 1][1])
                     : "n"(kMore && kSets == 2 ? DB * 2 : 0)
                     : "memory");
#pragma unroll
      for (int d = 0; d < DB; d++) {
        const short4v lo = run[g % kSets][d][0], hi = run[g % kSets][d][1];
        short8v both;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          both[e] = lo[e];
          both[4 + e] = hi[e];
        }
        accO[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
            __builtin_bit_cast(half8, both), fp, accO[d], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (kMore && kSets == 1)
        readGroup(Next{});
    };
    pvGroup(std::integral_constant<int, 0>{});
    pvGroup(std::integral_constant<int, 1>{});
    if constexpr (kGroups == 4) {
      pvGroup(std::integral_constant<int, 2>{});
      pvGroup(std::integral_constant<int, 3>{});
    }
    priority(Even{});
  };
  if constexpr (PIPE) {
    // Chunk by chunk: the scores of the next one (matrix cores) between the
    // exponentials of this one (vector ALU), K a chunk further ahead than V.
    constexpr int kSteps = D / 16, NE = 16 * SBW, NM = kSteps * SBW;
    constexpr int kDeep = SBW == 1 && D <= 128 ? kSteps : kSteps >= 8 ? kSteps / 2 : kSteps;
    const int blk = kh * (SBW * 32); // this wavefront's keys of a chunk
    auto tileOf = [&](int ch) { return smem + (ch % 2) * (2 * kTileBytes); };
    float16v accS[SBW], accN[SBW];
    half8 fk[SBW][kDeep];
    auto readK = [&](const unsigned char *sK, int sb, int kk) {
      fk[sb][kk % kDeep] = *reinterpret_cast<const half8 *>(
          sK + (blk + sb * 32 + l32) * kRowB + ((kk * 2 + hb) ^ swzLane) * 16);
    };
    auto multiplyK = [&](const unsigned char *sK, int m) { // MFMA m of a block's scores
      const int kk = m / SBW, sb = m % SBW;
      accN[sb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
          fk[sb][kk % kDeep], fq[kk], kk == 0 ? float16v{} : accN[sb], 0, 0, 0);
      if (kk + kDeep < kSteps)
        readK(sK, sb, kk + kDeep);
    };
    auto firstReads = [&](const unsigned char *sK) {
#pragma unroll
      for (int kk = 0; kk < kDeep; kk++)
#pragma unroll
        for (int sb = 0; sb < SBW; sb++)
          readK(sK, sb, kk);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto hideKeys = [&](int key0) { // those past the sequence end
#pragma unroll
      for (int sb = 0; sb < SBW; sb++)
#pragma unroll
        for (int e = 0; e < 16; e++) {
          const int key = key0 + blk + sb * 32 + 8 * (e / 4) + 4 * hb + (e % 4);
          accN[sb][e] = key < len ? accN[sb][e] : -INFINITY;
        }
    };
    requestTile(std::false_type{}, 0);
    if (numChunks > 1) {
      requestTile(std::false_type{}, 1);
      requestTile(std::true_type{}, 0);
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * VPT) : "memory");
    } else {
      requestTile(std::true_type{}, 0);
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(VPT) : "memory");
    }
    if (blk < len) {
      firstReads(tileOf(0));
#pragma unroll
      for (int m = 0; m < NM; m++)
        multiplyK(tileOf(0), m);
      if (blk + SBW * 32 > len)
        hideKeys(0);
      float blockMax = -INFINITY;
#pragma unroll
      for (int sb = 0; sb < SBW; sb++)
#pragma unroll
        for (int e = 0; e < 16; e++)
          blockMax = fmaxf(blockMax, accN[sb][e]);
      rowMax = pairMax(blockMax);
    }
    auto step = [&](int ch, auto moreC) {
      constexpr bool MORE = decltype(moreC)::value;
      // the next chunk's K and this one's V have landed, and every wavefront is done
      // with this one's K and the previous one's V
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if constexpr (MORE) {
        if (ch + 2 < numChunks)
          requestTile(std::false_type{}, ch + 2);
        requestTile(std::true_type{}, ch + 1);
      }
      const unsigned char *sKn = tileOf(ch + 1);
      const int key0 = ch * kChunk;
      if constexpr (!MORE) {
        if (key0 + blk >= len)
          return; // (the last chunk ends before this wavefront's keys)
        if (ch > 0 && key0 + blk + SBW * 32 > len)
          hideKeys(key0);
      }
#pragma unroll
      for (int sb = 0; sb < SBW; sb++)
        accS[sb] = accN[sb];
      half8 p[SBW][2];
      float sum = 0.f;
      const float negMax = -rowMax * scaleLog2e;
      if constexpr (MORE)
        firstReads(sKn);
#pragma unroll
      for (int m = 0; m < NM; m++) {
#pragma unroll
        for (int x = m * NE / NM; x < (m + 1) * NE / NM; x++) {
          const int sb = x / 16, e = x % 16;
          const float pv = __builtin_amdgcn_exp2f(fmaf(accS[sb][e], scaleLog2e, negMax));
          sum += pv;
          p[sb][e / 8][e % 8] = _Float16(pv);
        }
        if constexpr (MORE) {
          __builtin_amdgcn_sched_barrier(0);
          multiplyK(sKn, m);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (__builtin_expect(__any(!(sum <= kSumLimit)), 0)) {
        float blockMax = -INFINITY;
#pragma unroll
        for (int sb = 0; sb < SBW; sb++)
#pragma unroll
          for (int e = 0; e < 16; e++)
            blockMax = fmaxf(blockMax, accS[sb][e]);
        const float newMax = fmaxf(rowMax, pairMax(blockMax));
        const float corr = __builtin_amdgcn_exp2f((rowMax - newMax) * scaleLog2e);
        rowSum *= corr;
        rowMax = newMax;
#pragma unroll
        for (int d = 0; d < DB; d++)
#pragma unroll
          for (int e = 0; e < 16; e++)
            accO[d][e] *= corr;
        sum = 0.f;
        const float toMax = -rowMax * scaleLog2e;
#pragma unroll
        for (int sb = 0; sb < SBW; sb++)
#pragma unroll
          for (int e = 0; e < 16; e++) {
            const float pv = __builtin_amdgcn_exp2f(fmaf(accS[sb][e], scaleLog2e, toMax));
            sum += pv;
            p[sb][e / 8][e % 8] = _Float16(pv);
          }
      }
      rowSum += sum;
      weighValues(tileOf(ch) + kTileBytes, blk, [&](auto gC) {
        constexpr int g = decltype(gC)::value;
        return p[g / 2][g % 2];
      });
    };
    int ch = 0;
    for (; ch + 1 < numChunks; ch++)
      step(ch, std::true_type{});
    step(ch, std::false_type{});
  } else {
  requestChunk(0);
  // (at least one round in either variant: a loop that may run zero times
  // would put a test of the sequence length ahead of the prefetched loads)
  int ch = 0;
  do {
    const int key0 = ch * kChunk;
    // keys of this chunk that any wavefront will touch, rounded up to a block
    constexpr int kRound = SBW * 32;
    const int live =
        len - key0 < kChunk ? ((len - key0 + kRound - 1) / kRound) * kRound : kChunk;
    if (ch > 0 && !DMA)
      __syncthreads(); // previous chunk fully consumed
    // ---- stage K and V rows [key0, key0 + live): 8 vectors of 16 bytes per row.
    // Rows past the sequence end are zero-filled: masked scores ignore K, but a
    // masked probability (0) times a non-finite V would poison the output.
    if constexpr (DMA) {
      // this chunk has landed and every wavefront is done with the one before it,
      // whose buffer takes the next
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (ch + 1 < numChunks)
        requestChunk(ch + 1);
      sK = smem + (ch % 2) * (2 * kTileBytes);
      sV = sK + kTileBytes;
    } else if (kPrefetch) {
#pragma unroll
      for (int i = 0; i < VPT; i++) {
        const int v = tid + i * kThreads;
        const int r = v / CPR, c = v % CPR;
        if (r < live) {
          half8 kv = rk[i], vv = rv[i];
          if (key0 + r >= len) {
#pragma unroll
            for (int e = 0; e < 8; e++)
              kv[e] = vv[e] = _Float16(0);
          }
          *reinterpret_cast<half8 *>(sK + r * kRowB + swzK<D>(r, c) * 16) = kv;
          *reinterpret_cast<half8 *>(sV + r * kRowB + swzV<D>(r, c / 4) * 64 + (c % 4) * 16) = vv;
        }
      }
    } else {
      // Whole chunk, no range tests: the descriptors end at row `len`, so rows
      // past the sequence read as zero without touching memory.  All loads go
      // out before the first LDS store; addresses are one add per vector.
      half8 kv[VPT], vv[VPT];
      if constexpr (kFastStage) {
        const uint32_t chunkOff = stageOff + uint32_t(key0) * rowBytes;
#pragma unroll
        for (int i = 0; i < VPT; i++) {
          uint32_t off = chunkOff + uint32_t(i * (kThreads / CPR)) * rowBytes;
          if (PACKED_IN && key0 + tid / CPR + i * (kThreads / CPR) >= len)
            off = 0x80000000u - vFromK;
          kv[i] = __builtin_bit_cast(
              half8, __builtin_amdgcn_raw_buffer_load_b128(rsrcK, off, 0, 0));
          vv[i] = __builtin_bit_cast(
              half8, __builtin_amdgcn_raw_buffer_load_b128(rsrcV, off + vFromK, 0, 0));
        }
#pragma unroll
        for (int i = 0; i < VPT; i++) {
          *reinterpret_cast<half8 *>(sK + stageK + i * (kThreads / CPR) * kRowB) = kv[i];
          *reinterpret_cast<half8 *>(sV + stageV + i * (kThreads / CPR) * kRowB) = vv[i];
        }
      } else {
        // vector v of the chunk = 16-byte chunk v % CPR of row v / CPR
        static_assert((kChunk * CPR) % kThreads == 0, "whole vectors per thread");
#pragma unroll
        for (int i = 0; i < VPT; i++) {
          const int v = tid + i * kThreads;
          const uint32_t off =
              uint32_t(key0 + v / CPR) * rowBytes + uint32_t(v % CPR) * 16u;
          kv[i] = __builtin_bit_cast(
              half8, __builtin_amdgcn_raw_buffer_load_b128(rsrcK, off, 0, 0));
          vv[i] = __builtin_bit_cast(
              half8, __builtin_amdgcn_raw_buffer_load_b128(rsrcV, off, 0, 0));
        }
#pragma unroll
        for (int i = 0; i < VPT; i++) {
          const int v = tid + i * kThreads;
          const int r = v / CPR, c = v % CPR;
          *reinterpret_cast<half8 *>(sK + r * kRowB + swzK<D>(r, c) * 16) = kv[i];
          *reinterpret_cast<half8 *>(sV + r * kRowB + swzV<D>(r, c / 4) * 64 +
                                     (c % 4) * 16) = vv[i];
        }
      }
    }
    if constexpr (!DMA) {
      if (kPrefetch && ch + 1 < numChunks)
        loadChunk(key0 + kChunk);
      __syncthreads();
    }

    for (int blk = kh * (SBW * 32); blk < live; blk += SBW * 32 * KS) {
      // ---- S^T = K Q^T for two 32-key sub-blocks ----
      // All eight K fragments are requested before the first MFMA: read one
      // at a time, each MFMA would wait out a full LDS round trip.
      // accS[sb][e] is the raw score (before scaling) of query l32 against key
      //   key0 + blk + sb*32 + 8*(e/4) + 4*hb + e%4.
      // Only a block that reaches past the sequence end pays for the key mask.
      float16v accS[SBW];
      auto scores = [&]() {
        constexpr int kSteps = kHeadDim / 16;
        constexpr int kBatch = D <= 128 ? kSteps : kSteps / 2; // fragments read at a time
#pragma unroll
        for (int sb = 0; sb < SBW; sb++)
#pragma unroll
          for (int e = 0; e < 16; e++)
            accS[sb][e] = 0.f;
#pragma unroll
        for (int k0 = 0; k0 < kSteps; k0 += kBatch) {
          half8 fk[SBW][kBatch];
#pragma unroll
          for (int sb = 0; sb < SBW; sb++)
#pragma unroll
            for (int kk = 0; kk < kBatch; kk++)
              fk[sb][kk] = *reinterpret_cast<const half8 *>(
                  sK + (blk + sb * 32 + l32) * kRowB + (((k0 + kk) * 2 + hb) ^ swzLane) * 16);
          __builtin_amdgcn_sched_barrier(0);
          priority(First{});
#pragma unroll
          for (int sb = 0; sb < SBW; sb++)
#pragma unroll
            for (int kk = 0; kk < kBatch; kk++)
              accS[sb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fk[sb][kk], fq[k0 + kk],
                                                                accS[sb], 0, 0, 0);
          priority(Even{});
        }
        if (key0 + blk + SBW * 32 > len) {
#pragma unroll
          for (int sb = 0; sb < SBW; sb++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
              const int key = key0 + blk + sb * 32 + 8 * (e / 4) + 4 * hb + (e % 4);
              accS[sb][e] = key < len ? accS[sb][e] : -INFINITY;
            }
        }
      };
      scores();
      // The softmax works on raw scores: with c = scale * log2(e) > 0,
      // exp(scale * (s - m)) = exp2(c * s - c * m), one FMA and one v_exp per
      // score; the reference m (rowMax, raw units) only has to keep p within
      // range, it need not be the true maximum, and the final O / rowSum cancels
      // whatever reference was used.  This part is VALU work the matrix core
      // cannot hide (16 MFMAs against a few hundred vector instructions per
      // block), so instruction count matters:
      //  - fast path (every block but a wavefront's first): p is computed
      //    against the reference as it stands, no maximum is taken at all, and
      //    the row sums that are needed anyway tell whether that was safe: if
      //    some lane's sum (its half of a row's keys; the halves meet behind the last
      //    block) exceeds kSumLimit (so a p could leave
      //    fp16's range; an overflowed exp2 gives inf and lands here too) the
      //    block's scores are recomputed from LDS and take the slow path;
      //  - slow path (the first block, and a block whose sums overflowed): the
      //    true block maximum, the reference moves to it, O and the running
      //    sum are rescaled (96 vector instructions on the accumulators).
      // With real score distributions the slow path runs once per wavefront.
      // Every block that is visited has at least one valid key, so blockMax
      // is finite and the differences below are never inf - inf.
      const bool first = ch == 0 && blk == kh * (SBW * 32);
      float blockSum = 0.f;
      bool slow = first;
      if (!first) {
        const float negMax = -rowMax * scaleLog2e;
#pragma unroll
        for (int sb = 0; sb < SBW; sb++)
#pragma unroll
          for (int e = 0; e < 16; e++) {
            const float pv =
                __builtin_amdgcn_exp2f(fmaf(accS[sb][e], scaleLog2e, negMax));
            accS[sb][e] = pv;
            blockSum += pv;
          }
        slow = __any(!(blockSum <= kSumLimit));
        if (slow)
          scores(); // the probabilities are discarded: raw scores again
      }
      if (slow) {
        float blockMax = -INFINITY;
#pragma unroll
        for (int sb = 0; sb < SBW; sb++)
#pragma unroll
          for (int e = 0; e < 16; e++)
            blockMax = fmaxf(blockMax, accS[sb][e]);
        blockMax = pairMax(blockMax);
        const float newMax = fmaxf(rowMax, blockMax);
        // (first block: rowMax = -inf, corr = 0 on accumulators that are 0)
        const float corr = __builtin_amdgcn_exp2f((rowMax - newMax) * scaleLog2e);
        rowSum *= corr;
        rowMax = newMax;
#pragma unroll
        for (int d = 0; d < DB; d++)
#pragma unroll
          for (int e = 0; e < 16; e++)
            accO[d][e] *= corr;
        const float negMax = -rowMax * scaleLog2e;
        blockSum = 0.f;
#pragma unroll
        for (int sb = 0; sb < SBW; sb++)
#pragma unroll
          for (int e = 0; e < 16; e++) {
            const float pv =
                __builtin_amdgcn_exp2f(fmaf(accS[sb][e], scaleLog2e, negMax));
            accS[sb][e] = pv;
            blockSum += pv;
          }
      }
      rowSum += blockSum;

      // ---- O^T += V^T P^T ----
      if constexpr (DMA) {
        weighValues(sV, blk, [&](auto gC) {
          constexpr int g = decltype(gC)::value;
          half8 fp;
#pragma unroll
          for (int e = 0; e < 8; e++)
            fp[e] = _Float16(accS[g / 2][8 * (g % 2) + e]);
          return fp;
        });
      } else {
#pragma unroll
      for (int sb = 0; sb < SBW; sb++) {
#pragma unroll
        for (int t = 0; t < 2; t++) {
          // B operand: P[q][key(hb, e)], key(hb, e) = sb*32 + 8*(2t + e/4) + 4*hb
          // + e%4, which is accumulators 8t .. 8t+7 of this lane.
          half8 fp;
#pragma unroll
          for (int e = 0; e < 8; e++)
            fp[e] = _Float16(accS[sb][8 * t + e]);
#pragma unroll
          for (int d = 0; d < DB; d++) {
            // A operand: V[key(hb, e)][d*32 + l32]: two runs of 4 consecutive
            // keys, each transposed out of 4 V rows x 16 columns by one read.
            short4v run[2];
#pragma unroll
            for (int g = 0; g < 2; g++) {
              const int keyLocal = blk + sb * 32 + 8 * (2 * t + g) + 4 * hb + trRow;
              run[g] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                  (__attribute__((address_space(3))) short4v *)(
                      sV + keyLocal * kRowB + (d ^ vSwz) * 64 + trCol * 2));
            }
            short8v both;
#pragma unroll
            for (int e = 0; e < 4; e++) {
              both[e] = run[0][e];
              both[4 + e] = run[1][e];
            }
            accO[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
                __builtin_bit_cast(half8, both), fp, accO[d], 0, 0, 0);
          }
        }
      }
      }
    }
  } while (++ch < numChunks);
  }
  rowSum = pairSum(rowSum); // (each lane has added up its own keys)

  // ---- merge the key shares ----
  // Share 1 hands (reference, sum, O) of its rows to share 0 through LDS, in
  // the layout [query group][value][lane]; lanes of the two wavefronts hold
  // the same (row, columns).  With references m0, m1 in raw score units and
  // m = max(m0, m1): O = O0 2^((m0-m)c) + O1 2^((m1-m)c), the same for the
  // sums.  A share that saw no valid key has m1 = -inf and weight 0; share 0
  // always owns the first block, which has one.
  if constexpr (KS == 2) {
    constexpr int XV = DB * 16; // accumulator values per lane
    static_assert(DMA || QG * (XV + 2) * kWave * 4 <= 2 * kTileBytes, "exchange fits the K/V tiles");
    float *xch = reinterpret_cast<float *>(smem) + qg * ((XV + 2) * kWave) + lane;
    __syncthreads(); // every wavefront is done with K and V
    if (kh == 1) {
#pragma unroll
      for (int d = 0; d < DB; d++)
#pragma unroll
        for (int e = 0; e < 16; e++)
          xch[(d * 16 + e) * kWave] = accO[d][e];
      xch[XV * kWave] = rowMax;
      xch[(XV + 1) * kWave] = rowSum;
    }
    __syncthreads();
    if (kh == 1)
      return;
    const float m1 = xch[XV * kWave], l1 = xch[(XV + 1) * kWave];
    const float m = fmaxf(rowMax, m1);
    const float c0 = __builtin_amdgcn_exp2f((rowMax - m) * scaleLog2e);
    const float c1 = __builtin_amdgcn_exp2f((m1 - m) * scaleLog2e);
    rowSum = rowSum * c0 + l1 * c1;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int e = 0; e < 16; e++)
        accO[d][e] = accO[d][e] * c0 + xch[(d * 16 + e) * kWave] * c1;
  }

  // ---- normalise and store ----
  // accO[d][e]: column dcol = d*32 + 8*(e/4) + 4*hb + e%4 of query row l32.
  const int q = q0 + l32;
  if (q < seq) {
    const bool valid = q < len;
    const float inv = valid ? 1.0f / rowSum : 0.f;
    // Lane and lane ^ 32 hold the halves of the same 16 bytes: they swap them, and a
    // lane stores those of the even or of the odd eight columns.  (8 bytes a lane
    // before: 8 x 384 x 16 heads of 128 17.7 -> 16.5 us, 32 x 512 x 16 of 64 41.7 -> 39.0,
    // 8 x 200 x 8 of 192 13.3 -> 11.9, 8 x 384 x 16 of 256 40.4 -> 37.1.)  In fragment
    // order the 8-byte stores of a wavefront are whole runs of 256 bytes as they are:
    // 32 x 46 x 12 4.37 us, with the swap 4.43.
    _Float16 *const o16 = oRow - hb * 4 + hb * oEight;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int g = 0; g < 4; g += 2) {
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
        half4 o[2];
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
          for (int e = 0; e < 4; e++)
            o[h][e] = valid ? _Float16(accO[d][(g + h) * 4 + e] * inv) : _Float16(0);
        if constexpr (PACKED_IN) {
          *reinterpret_cast<half4 *>(oRow + d * oWide + g * oEight) = o[0];
          *reinterpret_cast<half4 *>(oRow + d * oWide + (g + 1) * oEight) = o[1];
        } else {
          const u32x2 even = __builtin_bit_cast(u32x2, o[0]), odd = __builtin_bit_cast(u32x2, o[1]);
          storeVector(o16 + d * oWide + g * oEight, joinHalves(even[0], even[1], odd[0], odd[1]));
        }
      }
  }
}

struct Launch {
  const _Float16 *qkv;
  const int32_t *cu;
  _Float16 *out;
  int64_t bs, seq, heads;
  float scale;
  int packedOut;
  const char *ahead;
  int64_t aheadBytes;
  unsigned extra; // workgroups that read ahead
  hipStream_t stream;
};
template <int NW, int KS, int D, bool PACKED_IN, bool DMA, bool PIPE = false>
Status launchVariant(const Launch &l) {
  if constexpr (kPipe<D, KS, PACKED_IN, DMA> && !PIPE) {
    if (attentionOverlapsScores(D, l.seq))
      return launchVariant<NW, KS, D, PACKED_IN, DMA, true>(l);
  }
  constexpr int QG = NW / KS;
  constexpr int kTileBytes = (DMA ? 64 : Chunk<D>::value) * D * 2;
  constexpr int kExchange = KS == 2 ? QG * (D / 2 + 2) * kWave * 4 : 0;
  constexpr int kTiles = (DMA ? 4 : 2) * kTileBytes;
  constexpr int kLds = kTiles > kExchange ? kTiles : kExchange;
  auto kernel = bertAttentionKernel<NW, KS, D, PACKED_IN, DMA, PIPE>;
  if (kLds > 64 * 1024) {
    static bool done = false;
    if (!done)
      HOM_HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, kLds),
                  Status::kInternal);
    done = true;
  }
  const unsigned nq = unsigned((l.seq + QG * 32 - 1) / (QG * 32));
  const int64_t pairs = l.bs * l.heads;
  dim3 grid(unsigned(nq * pairs) + l.extra);
  if (KS == 2 && !DMA) {
    const unsigned plane = nq * unsigned(l.heads);
    grid = dim3(nq, unsigned(l.heads), unsigned(l.bs) + (l.extra + plane - 1) / plane);
  }
  const bool outside = kTilesOutside<NW, KS, D, DMA> && attentionTilesOutside(int(pairs), int(nq));
  kernel<<<grid, dim3(NW * kWave), kLds, l.stream>>>(l.qkv, l.cu, l.out, int(l.seq), int(l.heads),
                                                     int(nq), int(l.bs), l.scale, l.packedOut,
                                                     magicFor(outside ? uint32_t(pairs) : nq), magicFor(uint32_t(l.heads)),
                                                     l.ahead, l.aheadBytes);
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}

} // namespace

Status launchBertAttentionF16(const _Float16 *qkv, const int32_t *cuSeqlens,
                              _Float16 *out, int64_t bs, int64_t seq,
                              int64_t heads, int64_t headDim, float scale,
                              hipStream_t s, bool packedOut, bool packedIn,
                              const void *ahead, int64_t aheadBytes) {
  HOM_CHECK_RET(!packedIn || (headDim == 64 && ((bs * seq + 15) / 16) * 96 * heads * 64 <
                                                   (int64_t(1) << 30)),
                Status::kInvalidArgument,
                "attention: QKV in fragment order needs head size 64 and less than 1 GiB");
  // (the reference's contract is head size % 64 == 0, README.md:11; the
  // sizes with kernels here are 64, 128, 192 and 256)
  HOM_CHECK_RET(headDim == 64 || headDim == 128 || headDim == 192 || headDim == 256,
                Status::kInvalidArgument,
                "attention: head size %lld not supported (64, 128, 192 or 256)",
                (long long)headDim);
  // The softmax tracks the maximum of the unscaled scores, which is the
  // maximum of the scaled ones only for a positive scale (BERT: 1/sqrt(64)).
  HOM_CHECK_RET(scale > 0.f, Status::kInvalidArgument,
                "attention: scale must be positive (got %g)", double(scale));
  HOM_CHECK_RET(bs < 65536 && heads < 65536 && seq < (int64_t(1) << 24),
                Status::kInvalidArgument, "attention: shape out of range");
  // K/V staging addresses a batch entry with 32-bit byte offsets
  HOM_CHECK_RET(seq * 3 * heads * headDim * 2 < (int64_t(1) << 31),
                Status::kInvalidArgument,
                "attention: one batch entry of QKV must be smaller than 2 GiB");
  HOM_CHECK_RET((reinterpret_cast<uintptr_t>(qkv) & 15) == 0 &&
                    (reinterpret_cast<uintptr_t>(out) & 7) == 0,
                Status::kInvalidArgument, "attention: misaligned operands");
  if (bs == 0 || seq == 0 || heads == 0)
    return Status::kSuccess;
  const int cus = deviceInfo().computeUnits > 0 ? deviceInfo().computeUnits : 256;
  const int64_t pairs = bs * heads;
  HOM_CHECK_RET(pairs * ((seq + 63) / 64) < (int64_t(1) << 31),
                Status::kInvalidArgument, "attention: too many workgroups");
  // Workgroups that read weights ahead (readAhead() in packed_args.h), while the
  // attention itself leaves room: two workgroups of it per CU or fewer.
  const unsigned extra =
      ahead && pairs * ((seq + 127) / 128) <= 2 * cus ? aheadGroups<256>(aheadBytes, cus) : 0;
  const Launch l{qkv, cuSeqlens, out, bs, seq, heads, scale, packedOut,
                 static_cast<const char *>(ahead), aheadBytes, packedIn ? extra : 0, s};
  AttentionWay way = attentionWay(pairs, seq, headDim, packedIn, cus);
  // profiling knob: HOM_ATTENTION_VARIANT=wide | split
  if (const char *force = getenv("HOM_ATTENTION_VARIANT"))
    way = strcmp(force, "wide") != 0 ? AttentionWay::kDmaSplit
          : headDim == 256          ? AttentionWay::kWide
                                    : AttentionWay::kDma;
  switch (headDim) {
  case 64:
    switch (way) {
    case AttentionWay::kPrefetch:
      return packedIn ? launchVariant<4, 2, 64, true, false>(l)
                      : launchVariant<4, 2, 64, false, false>(l);
    case AttentionWay::kWide:
      return packedIn ? launchVariant<4, 1, 64, true, false>(l)
                      : launchVariant<4, 1, 64, false, false>(l);
    case AttentionWay::kDma:
      return packedIn ? launchVariant<4, 1, 64, true, true>(l)
                      : launchVariant<4, 1, 64, false, true>(l);
    default:
      return packedIn ? launchVariant<4, 2, 64, true, true>(l)
                      : launchVariant<4, 2, 64, false, true>(l);
    }
  case 128:
    return way == AttentionWay::kDma ? launchVariant<4, 1, 128, false, true>(l)
                                     : launchVariant<4, 2, 128, false, true, true>(l); // (beyond 64 tokens only)
  case 192:
    return way == AttentionWay::kDma ? launchVariant<8, 2, 192, false, true>(l)
                                     : launchVariant<4, 2, 192, false, true>(l);
  default:
    return way == AttentionWay::kWide ? launchVariant<4, 1, 256, false, false>(l)
                                      : launchVariant<4, 2, 256, false, true>(l);
  }
}

} // namespace hom

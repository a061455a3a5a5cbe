// GEMMs of a few dozen to a few hundred rows against weights laid out for them.
//
//   D = act(A . B) or act(LN(A) . B), linear results also + C or + LN(C)
//
// At these sizes a GEMM is a weight matrix passing once through the chip and a
// chain of latencies: launch, first load, K loop, epilogue.  The tiled kernels
// (gemm_pipe.h) walk K in slabs of 64 through LDS, 12 to 48 barriers one after
// the other; here the wavefronts of a workgroup split K between them, every
// wavefront requests all of its operands at once, straight into registers in
// the layout the MFMA takes them, and the partial sums meet in LDS once:
//   - B is packed when it is loaded: the fragment of 16 columns x 32 k that one
//     v_mfma_f32_16x16x32_f16 takes is 1 KiB in lane order, so a wavefront
//     streams its part of B with fully coalesced 16-byte loads, no LDS and no
//     transposition;
//   - A may come in the same order (packedOffset() in kernels.h), which is how
//     these kernels, the attention and the embedding kernel can leave their
//     results; from a row-major A a fragment load touches 16 half-used lines.
// A layer norm without affine parameters in front of the GEMM costs no kernel:
// the wavefronts have whole rows of A in registers between them, so they form
// sum and sum of squares on the way and the epilogue applies
//   LN(A) . B = rstd (A . B) - mu rstd colsum(B)
// with colsum(B) from packing time (rows whose mean is many times their spread get
// a second, centred pass, see meanDominates()); the statistics are written for the later
// GEMM whose residual source is the same tensor, LN(C) = rstd c - mu rstd,
// rounded to fp16 where the graph stores it: the residual is what carries rounding
// from layer to layer, and without that point 12 layers come out 1.74e-3 instead
// of 1.28e-3 (in norm) from a pipeline with separate layer norms (1.23e-3 apart
// from itself in another summation order; 1.41e-3 against 1.44e-3 from fp32).
#include "cross_lane.h"
#include "fast_div.h"
#include "packed_args.h"
#include "rectangles.h"
#include "store_policy.h"

#include <algorithm>

namespace hom {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWave = 64, kWaves = 8, kThreads = kWave * kWaves;
constexpr uint32_t kOob = 0x80000000u;

// MB x NB blocks of 16 x 16 per workgroup; CH k steps of a wavefront in flight
// at once (ONCE: that is all of them).  The leading scalars arrive
// in registers with the wavefront (kernel-argument preload, see the Makefile),
// so the operands are requested before anything is fetched; `rest` is read
// behind those requests.  1 x 1 x 3 is held to four workgroups to a CU, so that
// one that reads ahead fits beside three with a tile.
template <int MB, int NB, int CH, bool ONCE, bool NORM_A, bool A_PACKED>
__global__ __launch_bounds__(kThreads, A_PACKED && (MB + NB) * CH <= 6 ? 8 : (MB + NB) * CH <= 20 && (ONCE || !NORM_A) ? 4 : 2) void packedGemmKernel(
    const _Float16 *A, const _Float16 *B, int M, int N, int K, int steps, int perWave,
    int chunkM, uint32_t chunkMMagic, int chunkN, int xmLog, PackedArgs rest) {
  (void)rest; // (through the argument pointer, see below)
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int id = blockIdx.x;
  // XCD id % 8 owns a rectangle of chunkM x chunkN tiles (chooseRectangles()).
  const int xcd = id % 8, loc = id / 8, xm = xcd & ((1 << xmLog) - 1), xn = xcd >> xmLog;
  const int ln = int(divByMagic(uint32_t(loc), uint32_t(chunkM), chunkMMagic));
  const int tileM = xm * chunkM + loc - ln * chunkM, tileN = xn * chunkN + ln;
  const int m0 = tileM * (MB * 16), n0 = tileN * (NB * 16);
  const int stepBegin = wave * perWave;
  const int stepEnd = stepBegin + perWave < steps ? stepBegin + perWave : steps;
  auto clampBytes = [](int64_t b) -> int32_t {
    return b > 0x7fffffffLL ? 0x7fffffff : (b < 0 ? 0 : int32_t(b));
  };
  const bool isTile = ln < chunkN && m0 < M && n0 < N;
  const auto rsrcA = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<_Float16 *>(A) + int64_t(m0) * K, 0,
      isTile ? clampBytes(int64_t(A_PACKED ? (M - m0 + 15) / 16 * 16 : M - m0) * K * 2) : 0,
      0x00020000);
  const auto rsrcB = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<_Float16 *>(B) + int64_t(n0) * K, 0, isTile ? NB * 16 * K * 2 : 0,
      0x00020000);
  const uint32_t aLane = A_PACKED ? uint32_t(lane) * 16u
                                  : (uint32_t(lane % 16) * uint32_t(K) + uint32_t(lane / 16) * 8u) * 2u;
  const uint32_t aStep = A_PACKED ? 1024u : 64u;
  const uint32_t aBlock = 16u * uint32_t(K) * 2u;
  const uint32_t bBlock = uint32_t(steps) * 1024u;
  half8 fa[CH][MB], fb[CH][NB];
  // (steps past the wavefront's last one: an offset outside the descriptors
  // reads as zero without touching memory)
  auto requestStep = [&](int c, int s) {
    const bool in = s < stepEnd;
    const uint32_t step = uint32_t(s);
#pragma unroll
    for (int j = 0; j < NB; j++)
      fb[c][j] = __builtin_bit_cast(
          half8, __builtin_amdgcn_raw_buffer_load_b128(
                     rsrcB, in ? uint32_t(lane) * 16u + step * 1024u + uint32_t(j) * bBlock : kOob, 0, 0));
#pragma unroll
    for (int i = 0; i < MB; i++)
      fa[c][i] = __builtin_bit_cast(
          half8, __builtin_amdgcn_raw_buffer_load_b128(
                     rsrcA, in ? aLane + step * aStep + uint32_t(i) * aBlock : kOob, 0, 0));
  };
#pragma unroll
  for (int c = 0; c < CH; c++)
    requestStep(c, stepBegin + c);
  __builtin_amdgcn_sched_barrier(0);
  // (fetched where they are used: together, the two sides' fields would be waited
  // for one after the other)
  auto restArgs = [] {
    PackedArgs p = {};
#if defined(__HIP_DEVICE_COMPILE__) // (the host pass only needs the kernel's stub)
    typedef const __attribute__((address_space(4))) PackedArgs *RestPtr;
    constexpr int kRestOffset = 2 * 8 + 10 * 4; // bytes of the leading arguments
    static_assert(kRestOffset % alignof(PackedArgs) == 0, "argument layout");
    RestPtr late = (RestPtr)((const __attribute__((address_space(4))) char *)
                                 __builtin_amdgcn_kernarg_segment_ptr() +
                             kRestOffset);
    asm volatile("" : "+s"(late));
    p = *late;
#endif
    return p;
  };
  if (!isTile) {
    const int tiles = 8 * chunkM * chunkN;
    if (id >= tiles) {
      const PackedArgs p = restArgs();
      readAhead<kThreads>(p.ahead, p.aheadBytes, id - tiles, int(gridDim.x) - tiles, tid);
    }
    return;
  }
  const PackedArgs p = restArgs();
  // What the epilogue reads: wavefront w finishes 16 x 16 blocks w, w + 8, .. of
  // the tile, a lane 4 consecutive columns of one row of each.
  constexpr int OUTS = (MB * NB + kWaves - 1) / kWaves;
  half4 cv[OUTS] = {};
  float2v cStat[OUTS];
  float4v cSum[OUTS] = {};
  auto blockOf = [&](int q) { return wave + q * kWaves; }; // (mb, nb) = (/ NB, % NB)
  auto rowOf = [&](int q) { return m0 + blockOf(q) / NB * 16 + lane % 16; };
  auto colOf = [&](int q) { return n0 + blockOf(q) % NB * 16 + lane / 16 * 4; };
  auto mine = [&](int q) { return blockOf(q) < MB * NB && rowOf(q) < p.M; };
#pragma unroll
  for (int q = 0; q < OUTS; q++) {
    cStat[q] = float2v{1.f, 0.f};
    if (mine(q)) {
      const int m = rowOf(q), n = colOf(q);
      if (p.C)
        cv[q] = *reinterpret_cast<const half4 *>(
            p.C + (p.cPacked ? packedOffset(m, n, p.N) : int64_t(m) * p.N + n));
      if (p.statsIn)
        cStat[q] = *reinterpret_cast<const float2v *>(p.statsIn + int64_t(m) * 2);
      if (NORM_A)
        cSum[q] = *reinterpret_cast<const float4v *>(p.colSum + n);
    }
  }
  __builtin_amdgcn_sched_barrier(0);

  float4v acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; i++)
#pragma unroll
    for (int j = 0; j < NB; j++)
      acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
  float sum[MB], sq[MB];
#pragma unroll
  for (int i = 0; i < MB; i++)
    sum[i] = sq[i] = 0.f;
  auto multiply = [&](int c) {
#pragma unroll
    for (int i = 0; i < MB; i++) {
      if (NORM_A) {
        const half2v one = {_Float16(1), _Float16(1)};
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const half2v x = {fa[c][i][2 * e], fa[c][i][2 * e + 1]};
          sum[i] = __builtin_amdgcn_fdot2(x, one, sum[i], false);
          sq[i] = __builtin_amdgcn_fdot2(x, x, sq[i], false);
        }
      }
#pragma unroll
      for (int j = 0; j < NB; j++)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[c][j], fa[c][i], acc[i][j], 0, 0, 0);
      // (in the order of arrival: reordered, the operands of several steps
      // get second copies and the workgroup no longer fits a CU twice)
      if (NORM_A)
        __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Behind its MFMAs a step's registers are asked to hold the one CH further on.
  int s0 = stepBegin;
  if constexpr (!ONCE) {
#pragma unroll 1
    for (; s0 + CH < stepEnd; s0 += CH) {
#pragma unroll
      for (int c = 0; c < CH; c++) {
        multiply(c);
        __builtin_amdgcn_sched_barrier(0);
        requestStep(c, s0 + CH + c);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
#pragma unroll
  for (int c = 0; c < CH; c++)
    multiply(c);

  // The wavefronts' partial sums meet: [wave][block][lane] and, of the row
  // statistics, [wave][row].
  float4v *part = reinterpret_cast<float4v *>(smem);
  float2v *stat = reinterpret_cast<float2v *>(smem + kWaves * MB * NB * kWave * 16);
#pragma unroll
  for (int i = 0; i < MB; i++) {
#pragma unroll
    for (int j = 0; j < NB; j++)
      part[(wave * MB * NB + i * NB + j) * kWave + lane] = acc[i][j];
    if (NORM_A) {
      const float s = pairSum(rowPairSum(sum[i])), q = pairSum(rowPairSum(sq[i]));
      if (lane < 16)
        stat[wave * MB * 16 + i * 16 + lane] = float2v{s, q};
    }
  }
  __syncthreads();
  auto total = [&](int q) {
    float4v v = part[blockOf(q) * kWave + lane];
#pragma unroll
    for (int w = 1; w < kWaves; w++)
      v += part[(w * MB * NB + blockOf(q)) * kWave + lane];
    return v;
  };
  auto rowSums = [&](int q) {
    float2v st{0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kWaves; w++)
      st += stat[w * MB * 16 + (blockOf(q) / NB) * 16 + lane % 16];
    return st;
  };
  auto finish = [&](int q, float4v v, float mu, float var) {
    const int block = blockOf(q), m = rowOf(q), n = colOf(q);
    if (NORM_A) {
      const float rstd = 1.0f / sqrtf(var + p.eps);
      const float shift = -mu * rstd;
#pragma unroll
      for (int e = 0; e < 4; e++)
        v[e] = fmaf(rstd, v[e], shift * cSum[q][e]);
      if (p.statsOut && tileN == 0 && block % NB == 0 && lane < 16)
        storeWriteThrough(p.statsOut + int64_t(m) * 2, float2v{rstd, shift});
    }
    half4 o;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      float x = v[e];
      if (p.activation == 1)
        x = geluErf(x);
      else if (p.activation == 2)
        x = geluTanh(x);
      if (p.C)
        x += float(_Float16(fmaf(float(cv[q][e]), cStat[q][0], cStat[q][1])));
      o[e] = _Float16(x);
    }
    storeWriteThrough(p.D + (p.dPacked ? packedOffset(m, n, p.N) : int64_t(m) * p.N + n), o);
  };
  bool again[OUTS], any = false;
#pragma unroll
  for (int q = 0; q < OUTS; q++) {
    again[q] = false;
    if (!mine(q))
      continue;
    const float4v v = total(q);
    float mu = 0.f, var = 0.f;
    if (NORM_A) {
      const float2v st = rowSums(q);
      mu = st[0] * p.invK;
      // the difference cancels to a small negative number for near-constant
      // rows; clamped so that a tiny eps cannot turn it into a NaN
      var = fmaxf(st[1] * p.invK - mu * mu, 0.f);
      again[q] = meanDominates(mu, var);
      any = any || again[q];
    }
    finish(q, v, mu, var);
  }
  // Rows far from zero once more, centred.  (Behind the other rows' stores: in
  // front of them the test alone costs 0.1 us a launch.)
  if (NORM_A && __builtin_expect(__any(any), 0)) {
#pragma unroll
    for (int q = 0; q < OUTS; q++) {
      if (blockOf(q) >= MB * NB)
        continue; // (the same for the whole wavefront)
      const float mu = rowSums(q)[0] * p.invK;
      float d2 = 0.f;
#pragma unroll 2
      for (int s = 0; s < steps; s++) { // the block's rows as their fragments lie
        const half8 x = __builtin_bit_cast(
            half8, __builtin_amdgcn_raw_buffer_load_b128(
                       rsrcA, aLane + uint32_t(s) * aStep + uint32_t(blockOf(q) / NB) * aBlock, 0, 0));
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const float d = float(x[e]) - mu;
          d2 = fmaf(d, d, d2);
        }
      }
      d2 = pairSum(rowPairSum(d2));
      // (nothing shared with the stores above: what is would move in front of the
      // barrier, into every launch)
      asm volatile("" : "+v"(cv[q]), "+v"(cStat[q]), "+v"(cSum[q]));
      if (again[q])
        finish(q, total(q), mu, d2 * p.invK);
    }
  }
}

// Layer norm without affine parameters of rows in fragment order; the result in
// the same order (out may be in) or row-major.  A workgroup owns a block of 16
// rows, its wavefronts every eighth kilobyte of it, the row in registers for
// both passes: whole cache lines, where a wavefront per row would touch eight
// rows' lines for its own 16 bytes of each.
template <int VPW> // kilobytes per wavefront
__global__ __launch_bounds__(kThreads) void packedLayernormKernel(const _Float16 *in, _Float16 *out,
                                                                  int M, int N, bool outPacked,
                                                                  float eps) {
  __shared__ float part[2][kWaves][16];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int blocks = N / 32, r = lane % 16;
  const half8 *src = reinterpret_cast<const half8 *>(in) + int64_t(blockIdx.x) * blocks * kWave;
  half8 raw[VPW];
#pragma unroll
  for (int i = 0; i < VPW; i++) {
    const int j = i * kWaves + wave;
    raw[i] = src[(j < blocks ? j : 0) * kWave + lane];
  }
  __builtin_amdgcn_sched_barrier(0); // every request is out
  auto rowTotal = [&](float v, int which) { // over the row's lanes and wavefronts
    v = pairSum(rowPairSum(v));
    if (lane < 16)
      part[which][wave][lane] = v;
    __syncthreads();
    v = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; w++)
      v += part[which][w][r];
    return v;
  };
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < VPW; i++)
#pragma unroll
    for (int e = 0; e < 8; e++)
      sum += i * kWaves + wave < blocks ? float(raw[i][e]) : 0.f;
  const float invN = 1.0f / float(N);
  const float mean = rowTotal(sum, 0) * invN;
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < VPW; i++)
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float d = i * kWaves + wave < blocks ? float(raw[i][e]) - mean : 0.f;
      sq += d * d;
    }
  const float rstd = 1.0f / sqrtf(rowTotal(sq, 1) * invN + eps);
  const int64_t row = int64_t(blockIdx.x) * 16 + r;
#pragma unroll
  for (int i = 0; i < VPW; i++) {
    const int j = i * kWaves + wave;
    half8 o;
#pragma unroll
    for (int e = 0; e < 8; e++)
      o[e] = _Float16((float(raw[i][e]) - mean) * rstd);
    if (j < blocks && (outPacked || row < M))
      storeWriteThrough(outPacked ? out + (int64_t(blockIdx.x) * blocks + j) * 512 + lane * 8
                                  : out + row * N + j * 32 + (lane / 16) * 8,
                        o);
  }
}

// B [K, N] row-major -> fragments: block (column block j, k step s) is 1 KiB,
// lane l of it holds B[32 s + 8 (l / 16) + e][16 j + l % 16], e = 0..7.
__global__ __launch_bounds__(256) void packWeightKernel(const _Float16 *__restrict__ B,
                                                        _Float16 *__restrict__ out,
                                                        int K, int N) {
  const int64_t v = int64_t(blockIdx.x) * 256 + threadIdx.x; // 16-byte vector of the output
  const int steps = K / 32;
  if (v >= int64_t(N / 16) * steps * kWave)
    return;
  const int l = int(v % kWave);
  const int64_t block = v / kWave;
  const int s = int(block % steps), j = int(block / steps);
  half8 o;
#pragma unroll
  for (int e = 0; e < 8; e++)
    o[e] = B[int64_t(32 * s + 8 * (l / 16) + e) * N + 16 * j + l % 16];
  reinterpret_cast<half8 *>(out)[v] = o;
}

// The way back: fragments -> B [K, N] row-major.
__global__ __launch_bounds__(256) void unpackWeightKernel(const _Float16 *__restrict__ packed,
                                                          _Float16 *__restrict__ B, int K, int N) {
  const int64_t v = int64_t(blockIdx.x) * 256 + threadIdx.x; // 16-byte vector of the input
  const int steps = K / 32;
  if (v >= int64_t(N / 16) * steps * kWave)
    return;
  const int l = int(v % kWave);
  const int64_t block = v / kWave;
  const int s = int(block % steps), j = int(block / steps);
  const half8 x = reinterpret_cast<const half8 *>(packed)[v];
#pragma unroll
  for (int e = 0; e < 8; e++)
    B[int64_t(32 * s + 8 * (l / 16) + e) * N + 16 * j + l % 16] = x[e];
}

// Rows [M, C] row-major -> fragment order, zeros in the rows that fill the last
// block.  A copy, 16 bytes per thread: whole kilobytes out, 64 bytes of 16 rows in.
__global__ __launch_bounds__(256) void packRowsKernel(const _Float16 *__restrict__ in,
                                                      _Float16 *__restrict__ out, int64_t M, int C,
                                                      int64_t vecs) {
  const int64_t v = int64_t(blockIdx.x) * 256 + threadIdx.x; // 16-byte vector of the output
  if (v >= vecs)
    return;
  const int l = int(v % kWave), wide = C / 32;
  const int64_t block = v / kWave, row = block / wide * 16 + l % 16;
  const int col = int(block % wide) * 32 + l / 16 * 8;
  half8 x = {};
  if (row < M)
    x = *reinterpret_cast<const half8 *>(in + row * C + col);
  storeWriteThrough(out + v * 8, x);
}

template <int MB, int NB, int CH, bool ONCE>
Status launchVariant(const PackedGemm &g, const PackedArgs &p, const Rectangles &r,
                     int aheadGroups, hipStream_t s) {
  if (g.only) {
    *g.only = {false, MB * 16, NB * 16, CH * 32};
    return Status::kSuccess;
  }
  const int steps = int(g.K / 32), perWave = (steps + kWaves - 1) / kWaves;
  constexpr int kLds = kWaves * MB * NB * kWave * 16 + kWaves * MB * 16 * 8;
  const dim3 grid((unsigned)(8 * r.chunkM * r.chunkN + aheadGroups)), block(kThreads);
  constexpr bool kRowMajorA = MB * NB < 16; // (an A of so many rows arrives packed)
  auto kernel = g.aPacked || !kRowMajorA
                    ? (g.normA ? packedGemmKernel<MB, NB, CH, ONCE, true, true>
                               : packedGemmKernel<MB, NB, CH, ONCE, false, true>)
                    : (g.normA ? packedGemmKernel<MB, NB, CH, ONCE, true, !kRowMajorA>
                               : packedGemmKernel<MB, NB, CH, ONCE, false, !kRowMajorA>);
  if (kLds > 48 * 1024) {
    static bool done[4] = {};
    bool &set = done[2 * g.aPacked + g.normA];
    if (!set)
      HOM_HIP_RET(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, kLds),
                  Status::kInternal);
    set = true;
  }
  kernel<<<grid, block, kLds, s>>>(g.A, g.packedB, int(g.M), int(g.N), int(g.K), steps, perWave,
                                   r.chunkM, magicFor(uint32_t(r.chunkM)), r.chunkN, r.xmLog, p);
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}

} // namespace

Status launchPackWeight(const _Float16 *B, _Float16 *packed, int64_t K, int64_t N,
                        hipStream_t s) {
  const int64_t vecs = K * N / 8;
  packWeightKernel<<<dim3((unsigned)((vecs + 255) / 256)), dim3(256), 0, s>>>(B, packed, int(K),
                                                                              int(N));
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}

Status launchUnpackWeight(const _Float16 *packed, _Float16 *B, int64_t K, int64_t N,
                          hipStream_t s) {
  const int64_t vecs = K * N / 8;
  unpackWeightKernel<<<dim3((unsigned)((vecs + 255) / 256)), dim3(256), 0, s>>>(packed, B, int(K),
                                                                                int(N));
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}

Status launchPackRows(const _Float16 *in, _Float16 *out, int64_t M, int64_t C, hipStream_t s) {
  const int64_t vecs = (M + 15) / 16 * 16 * C / 8;
  packRowsKernel<<<dim3((unsigned)((vecs + 255) / 256)), dim3(256), 0, s>>>(in, out, M, int(C),
                                                                            vecs);
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}

Status launchPackedLayernorm(const _Float16 *in, _Float16 *out, int64_t M, int64_t N, float eps,
                             bool outPacked, hipStream_t s) {
  const dim3 grid((unsigned)((M + 15) / 16)), block(kThreads);
  const int perWave = int((N / 32 + kWaves - 1) / kWaves);
  auto kernel = perWave <= 3   ? packedLayernormKernel<3>
                : perWave <= 4 ? packedLayernormKernel<4>
                               : packedLayernormKernel<8>;
  kernel<<<grid, block, 0, s>>>(in, out, int(M), int(N), outPacked, eps);
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}

namespace {
// The steps in flight for a wavefront's share of K: all of it while that is 3 or 4
// steps (for one block of 16 x 16 up to 16), else a count that goes into it and
// fits the registers.
Status launchShape(int mb, int nb, int perWave, const PackedGemm &g, const PackedArgs &p,
                   const Rectangles &r, int groups, hipStream_t s) {
  const bool byThree = perWave % 3 == 0;
  switch (mb * 8 + nb) {
  case 1 * 8 + 1:
    return perWave <= 3    ? launchVariant<1, 1, 3, true>(g, p, r, groups, s)
           : perWave <= 4  ? launchVariant<1, 1, 4, true>(g, p, r, groups, s)
           : perWave <= 12 ? launchVariant<1, 1, 12, true>(g, p, r, groups, s)
           : perWave <= 16 ? launchVariant<1, 1, 16, true>(g, p, r, groups, s)
                           : launchVariant<1, 1, 12, false>(g, p, r, groups, s);
  case 2 * 8 + 1:
    return perWave <= 3   ? launchVariant<2, 1, 3, true>(g, p, r, groups, s)
           : perWave <= 4 ? launchVariant<2, 1, 4, true>(g, p, r, groups, s)
                          : launchVariant<2, 1, 6, false>(g, p, r, groups, s);
  case 2 * 8 + 2:
    return perWave <= 3   ? launchVariant<2, 2, 3, true>(g, p, r, groups, s)
           : perWave <= 4 ? launchVariant<2, 2, 4, true>(g, p, r, groups, s)
                          : launchVariant<2, 2, 4, false>(g, p, r, groups, s);
  case 4 * 8 + 1:
    return perWave <= 3   ? launchVariant<4, 1, 3, true>(g, p, r, groups, s)
           : perWave <= 4 ? launchVariant<4, 1, 4, true>(g, p, r, groups, s)
                          : launchVariant<4, 1, 4, false>(g, p, r, groups, s);
  case 4 * 8 + 2:
    return perWave <= 3   ? launchVariant<4, 2, 3, true>(g, p, r, groups, s)
           : perWave <= 4 ? launchVariant<4, 2, 4, true>(g, p, r, groups, s)
           : byThree      ? launchVariant<4, 2, 3, false>(g, p, r, groups, s)
                          : launchVariant<4, 2, 4, false>(g, p, r, groups, s);
  default:
    return perWave <= 3   ? launchVariant<4, 4, 3, true>(g, p, r, groups, s)
           : perWave <= 4 ? launchVariant<4, 4, 4, true>(g, p, r, groups, s)
           : byThree      ? launchVariant<4, 4, 3, false>(g, p, r, groups, s)
                          : launchVariant<4, 4, 4, false>(g, p, r, groups, s);
  }
}
} // namespace

Status launchPackedGemm(const PackedGemm &g, hipStream_t s) {
  PackedArgs p{};
  p.C = g.C;
  p.D = g.D;
  p.colSum = g.colSum;
  p.statsIn = g.statsIn;
  p.statsOut = g.statsOut;
  p.M = int(g.M);
  p.N = int(g.N);
  p.activation = g.activation;
  p.cPacked = g.cPacked;
  p.dPacked = g.dPacked;
  p.invK = 1.0f / float(g.K);
  p.eps = g.eps;
  p.ahead = static_cast<const char *>(g.ahead);
  p.aheadBytes = g.ahead ? g.aheadBytes : 0;
  const PackedTileChoice tiled = choosePackedTile(g);
  // k steps per wavefront, all in flight at once where the registers allow
  const int perWave = int((g.K / 32 + kWaves - 1) / kWaves);
  // The tile by a model of its time in a chain of launches, fitted to M = 16 ..
  // 2048 x the shapes of BERT-base and -large (6 % off in the mean, the choice within
  // 8 % of the best but for a few shapes): launch, latency and the meeting of
  // the partial sums; then what the fullest CU pulls through its L1, no faster
  // than its XCD fetches the rectangle's operands; and a chain of latencies more
  // for every round of workgroups that do not fit a CU together.  (Those of the
  // tile kernels that fill the chip do not read ahead, which is worth most of a
  // microsecond to the launch behind.)
  const int cus = deviceInfo().computeUnits > 0 ? deviceInfo().computeUnits : 256;
  struct Shape {
    int mb, nb, resident;
  };
  const Shape shapes[] = {{1, 1, perWave <= 4 ? 3 : 1},
                          {2, 1, 2},
                          {2, 2, 2},
                          {4, 1, 2},
                          {4, 2, perWave <= 3 || (perWave > 4 && perWave % 3 == 0) ? 2 : 1},
                          {4, 4, 1}};
  const Shape *best = nullptr;
  double bestCost = 1e300;
  Rectangles rect{};
  for (const Shape &t : shapes) {
    if (g.N % (t.nb * 16) != 0 || (t.mb * t.nb == 16 && !g.aPacked))
      continue;
    const Rectangles r = chooseRectangles((g.M + t.mb * 16 - 1) / (t.mb * 16),
                                          g.N / (t.nb * 16), t.mb, t.nb, g.K, cus);
    const double kb = double(t.mb + t.nb) * 16 * double(g.K) * 2 / 1024;
    const int64_t rounds = (r.perCu + t.resident - 1) / t.resident;
    // (a workgroup alone on its CU in the last round does not fetch twice as fast)
    const double load = perWave <= 4 || r.perCu == 1
                            ? double(r.perCu)
                            : 0.5 * double(r.perCu + rounds * t.resident);
    const double fetch =
        std::max((perWave <= 4 ? 0.00915 : 0.0077) * kb * load, r.fillBytes / 5.3e6);
    const double round = t.resident > 1 || t.mb == 1 ? 0.2 : perWave <= 4 ? 2.0 : 8.0;
    const double cost = 1.7 + 0.08 * t.mb * t.nb + fetch * (g.normA ? 1.25 : 1.0) +
                        round * double(rounds - 1);
    if (cost < bestCost) {
      bestCost = cost;
      best = &t;
      rect = r;
    }
  }
  if (tiled.us + (g.ahead ? 0.7 : 0.0) < bestCost)
    return launchPackedTile(tiled.tile, g, p, s);
  // (half the CUs read ahead when the tiles take all of them)
  const int groups = aheadGroups<kThreads>(p.aheadBytes, std::max<int64_t>(cus - int64_t(rect.chunkM) * rect.chunkN * 8, cus / 2));
  return launchShape(best->mb, best->nb, perWave, g, p, rect, groups, s);
}

} // namespace hom

// The layer-norm pair of the reference (cutlassGemmWithVarMeanF16 followed by
// cutlassLayernormGemmF16, include/NVGPUKernels/LayernormGemmRunner.h:17-361)
// with the normalisation folded into the two GEMMs' epilogues: the first GEMM's
// epilogue accumulates row statistics of the stored D, the second applies
// var/mean per row through the column sums of B.  Both use the register-staged
// pipeline kernels with the two extra epilogue codes.
#include "gemm_pipe.h"
#include "pair_tile.h"

namespace hom {
namespace {
using namespace gemmk;

// ------------------------------------------------------- layer-norm pair --
// Row-statistic partials [pieces][M] (sum, sum of squares) -> var / mean in the
// form the pair exchanges (Layernorm.h:166-192 of the reference: the second
// moment minus the squared mean, no shift).  A chain of latencies: a wavefront
// has 16 rows, four lanes each, 16 apart so that 16 neighbouring lanes read 16
// neighbouring rows; a lane asks for every fourth piece, eight at a time (32 pieces
// in one go), and a workgroup is one wavefront, so that all CUs take part.
__global__ __launch_bounds__(kWave) void rowStatsFinalizeKernel(
    const float *__restrict__ partials, int pieces, int M, int N, float eps,
    _Float16 *__restrict__ var, _Float16 *__restrict__ mean) {
  const int lane = threadIdx.x, q = lane / 16;
  const int m = blockIdx.x * 16 + lane % 16;
  const int mc = m < M ? m : M - 1;
  constexpr int kLoads = 8;
  float s = 0.f, sq = 0.f;
  for (int pc = q; pc < pieces; pc += 4 * kLoads) {
    float2v v[kLoads];
#pragma unroll
    for (int u = 0; u < kLoads; u++) {
      const int pu = pc + 4 * u;
      v[u] = pu < pieces ? *reinterpret_cast<const float2v *>(
                               partials + (int64_t(pu) * M + mc) * 2)
                         : float2v{0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < kLoads; u++) {
      s += v[u][0];
      sq += v[u][1];
    }
  }
  s = pairSum(rowPairSum(s));
  sq = pairSum(rowPairSum(sq));
  if (q == 0 && m < M) {
    const float mu = s / float(N);
    // the difference cancels to a small negative number for near-constant
    // rows; clamped so that a tiny eps cannot turn it into a NaN
    const float rstd = 1.0f / sqrtf(fmaxf(sq / float(N) - mu * mu, 0.f) + eps);
    var[m] = _Float16(rstd);
    mean[m] = _Float16(-mu * rstd);
  }
}

// Partial column sums of row-major B [K, N]: workgroup (x, y) sums rows
// [y * kPer, (y + 1) * kPer) of columns [64 x, 64 x + 64) into out[y][n]: whole
// cache lines, 8 columns of every 32nd row per thread, four rows asked for at a
// time; the row phases of a wavefront meet in registers, the wavefronts in LDS.
__global__ __launch_bounds__(256) void colSumKernel(
    const _Float16 *__restrict__ B, int64_t ldb, int K, int N, int kPer,
    float *__restrict__ out) {
  __shared__ float part[4][64];
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int cg = tid % 8, ph = tid / 8;
  const int n = blockIdx.x * 64 + cg * 8;
  const int kBegin = blockIdx.y * kPer;
  const int kEnd = kBegin + kPer < K ? kBegin + kPer : K;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (n < N) {
    for (int k = kBegin + ph; k < kEnd; k += 128) {
      half8 v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int ku = k + 32 * u;
        v[u] = *reinterpret_cast<const half8 *>(B + int64_t(ku < kEnd ? ku : k) * ldb + n);
      }
#pragma unroll
      for (int u = 0; u < 4; u++)
#pragma unroll
        for (int e = 0; e < 8; e++)
          acc[e] += k + 32 * u < kEnd ? float(v[u][e]) : 0.f;
    }
  }
  // (lanes 8 apart hold the same columns)
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const float s = pairSum(rowPairSum(acc[e] + __shfl_xor(acc[e], 8, kWave)));
    if (lane < 8)
      part[wave][lane * 8 + e] = s;
  }
  __syncthreads();
  if (tid < 64 && blockIdx.x * 64 + tid < N)
    out[int64_t(blockIdx.y) * N + blockIdx.x * 64 + tid] =
        (part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid]);
}

// Tiles the layer-norm pair kernels exist in (square, `edge` on a side, a
// wavefront covering `pieceWidth` columns); `likeKernel` picks the nearest.
struct FusedTile {
  int edge;
  int pieceWidth;
};
FusedTile fusedTileFor(int likeKernel) {
  const GemmKernelInfo &like = gemmKernelInfo(likeKernel);
  const int area = like.tileM * like.tileN;
  if (area >= 256 * 256)
    return {256, 64};
  if (area >= 128 * 128)
    return {128, 32};
  return {64, 32};
}
template <int EPI> Status launchFusedEdge(int edge, const GemmProblem &p, hipStream_t s) {
  // the folded-layer-norm epilogues run on the DMA-staged variants of the two
  // smaller tiles (the faster ones at the sizes those tiles serve)
  constexpr bool kDma = EPI >= kEpiFoldA;
  switch (edge) {
  case 256:
    return launchPipe<256, 256, 2, 4, 1, EPI, false>(p, s);
  case 128:
    return launchPipe<128, 128, 2, 4, kDma ? 3 : 2, EPI, false, kDma>(p, s);
  default:
    return launchPipe<64, 64, 2, 2, kDma ? 3 : 2, EPI, false, kDma>(p, s);
  }
}

// The pair's kernels with an epilogue of the folded layer norm: staged through
// registers, which is the same on every box (128 x 128 tiles staged by DMA: 8 % faster
// to 10 % slower).
template <int EPI> Status launchPairFolded(int edge, const GemmProblem &p, hipStream_t s) {
  if constexpr (EPI == kEpiRowAffineOwn) {
    // Without a source 256 x 256 tiles leave by lane exchanges, through LDS -> so, us: 4096 x 4096 x 1024 40.8 -> 38.5,
    // 8192 x 3072 x 1024 68.7 -> 65.8, 16384 x 768 x 768 27.6 -> 25.4, 16384 x 4096 x 1024 153 -> 148.
    // (Staged by DMA the same to 2 % slower; 128 x 128 tiles, 700 x 4096 x 1024: 11.8 -> 12.0.)
    if (edge == 256 && p.beta == 0.f)
      return launchPipe<256, 256, 2, 4, 1, kEpiRowAffineLanes, false>(p, s);
    if (edge == 256)
      return launchPipe<256, 256, 2, 4, 1, EPI, false>(p, s);
    if (edge == 64)
      return launchPipe<64, 64, 2, 2, 2, EPI, false>(p, s);
  }
  return launchPipe<128, 128, 2, 4, 2, EPI, false>(p, s);
}
template <int EPI>
Status launchFusedTile(int likeKernel, const GemmProblem &p, hipStream_t s) {
  return launchFusedEdge<EPI>(fusedTileFor(likeKernel).edge, p, s);
}
inline bool aligned16(const void *p) {
  return (reinterpret_cast<uintptr_t>(p) & 15) == 0;
}

// What the epilogues of the folded layer norm ask for beyond fusedGemmFits(): no
// source or a full matrix, 32-bit byte offsets inside a tile's rows.
bool foldFits(const GemmProblem &p) {
  return (p.beta == 0.f || (p.cRowPeriod >= p.M && p.ldc % 8 == 0 &&
                            int64_t(256) * p.ldc * 2 < (int64_t(1) << 31))) &&
         int64_t(256) * p.ldd * 2 < (int64_t(1) << 31);
}
// The pair's tile (second: of its second GEMM).
FusedTile pairTile(const GemmProblem &p, bool second) {
  const int cus = deviceInfo().computeUnits > 0 ? deviceInfo().computeUnits : 256;
  const PairSource source = p.beta == 0.f ? PairSource::kNone
                            : foldFits(p) ? PairSource::kMatrix
                                          : PairSource::kRow;
  const int edge = pairTileEdge(p.M, p.N, p.K, second, source, cus);
  return {edge, edge == 256 ? 64 : 32};
}

} // namespace

bool fusedGemmFits(const GemmProblem &p) {
  return !p.bIsNK && p.M > 0 && p.N > 0 && p.K > 0 &&
         p.M < (int64_t(1) << 31) && p.N < (int64_t(1) << 31) &&
         p.K < (int64_t(1) << 31) && p.K % 8 == 0 && p.N % 8 == 0 &&
         p.lda % 8 == 0 && p.ldb % 8 == 0 && p.ldd % 8 == 0 &&
         aligned16(p.A) && aligned16(p.B) && aligned16(p.D) &&
         (p.beta == 0.f || (p.C && p.ldc % 8 == 0 && aligned16(p.C)));
}

Status launchGemmRowStats(const GemmProblem &p, _Float16 *var, _Float16 *mean, float eps,
                          hipStream_t s) {
  HOM_CHECK_RET(fusedGemmFits(p), Status::kInvalidArgument,
                "gemm + row statistics: problem does not fit the fused kernels");
  // No source or a full matrix, on 128 x 128 tiles: the epilogue of the folded
  // layer norm with nothing folded in, which requests the source ahead of everything
  // and adds up a tile's columns before it writes them (with a source 1024 x 3072 x 768
  // 14.8 -> 12.7 us, 8192 x 768 x 768 25.0 -> 22.5, 4096 x 1024 x 1024 17.8 -> 16.8).  Others, a
  // bias row, small tiles (64 x 768 x 768 8.2 / 9.1) or 256 x 256 ones (whose registers do
  // not hold the source's vectors as well), write a partial sum per wavefront column,
  // also of those past N.
  const FusedTile t = pairTile(p, false);
  const bool whole = t.edge == 128 && foldFits(p);
  const int pieces = int((p.N + t.edge - 1) / t.edge) * (whole ? 1 : t.edge / t.pieceWidth);
  float *partials = static_cast<float *>(
      libraryScratch(kTemp, size_t(pieces) * size_t(p.M) * 2 * sizeof(float), false));
  if (!partials)
    return Status::kInternal;
  GemmProblem q = p;
  q.splitK = 1;
  q.rowStatPartials = partials;
  Status st = whole ? launchPairFolded<kEpiFoldCStats>(t.edge, q, s)
                    : launchFusedEdge<kEpiRowStats>(t.edge, q, s);
  if (st != Status::kSuccess)
    return st;
  rowStatsFinalizeKernel<<<dim3((unsigned)((p.M + 15) / 16)), dim3(kWave), 0,
                           s>>>(partials, pieces, int(p.M), int(p.N), eps, var,
                                mean);
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}

Status launchGemmRowAffine(const GemmProblem &p, const _Float16 *var, const _Float16 *mean,
                           hipStream_t s) {
  HOM_CHECK_RET(fusedGemmFits(p), Status::kInvalidArgument,
                "layernorm + gemm: problem does not fit the fused kernels");
  GemmProblem q = p;
  q.splitK = 1;
  q.rowScale = var;
  q.rowShift = mean;
  const int edge = pairTile(p, true).edge;
  // No source or a full matrix: the column sums are formed on the way, four dot
  // products per fragment of B in the shadow of its MFMAs; by a kernel of their own
  // they took 4.5 us of a launch.  With the pairs kept in LDS and the epilogue of
  // the folded layer norm, us: 64 x 768 x 768 9.2 -> 6.1, 1024 x 4096 x 1024 20.2 -> 14.5,
  // 4096 x 4096 x 1024 45.5 -> 41.6, 16384 x 4096 x 1024 165 -> 152.
  if (foldFits(p))
    return launchPairFolded<kEpiRowAffineOwn>(edge, q, s);
  // A source of another form: the column sums by a kernel of their own, 128 rows of
  // B per workgroup (four 16-byte loads per lane), at most 16 slices.
  int slices = int((p.K + 127) / 128);
  if (slices > 16)
    slices = 16;
  const int kPer = int((p.K + slices - 1) / slices);
  float *colSum = static_cast<float *>(
      libraryScratch(kTemp, size_t(slices) * size_t(p.N) * sizeof(float), false));
  if (!colSum)
    return Status::kInternal;
  colSumKernel<<<dim3((unsigned)((p.N + 63) / 64), (unsigned)slices), dim3(256),
                 0, s>>>(p.B, p.ldb, int(p.K), int(p.N), kPer, colSum);
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  q.colSum = colSum;
  q.colSumSlices = slices;
  return launchFusedEdge<kEpiRowAffine>(edge, q, s);
}

int foldedPieces(int likeKernel, int64_t N) {
  // one piece per tile column (the wavefront columns of a tile are added up
  // inside the workgroup)
  const FusedTile t = fusedTileFor(likeKernel);
  return int((N + t.edge - 1) / t.edge);
}

Status launchColumnSums(const _Float16 *B, int64_t ldb, int64_t K, int64_t N,
                        float *out, hipStream_t s) {
  HOM_CHECK_RET(K > 0 && N > 0 && K < (int64_t(1) << 31) &&
                    N < (int64_t(1) << 31) && N % 8 == 0 && ldb % 8 == 0 &&
                    aligned16(B),
                Status::kInvalidArgument,
                "column sums: N and the leading dimension must be multiples of 8");
  colSumKernel<<<dim3((unsigned)((N + 63) / 64), 1), dim3(256), 0, s>>>(
      B, ldb, int(K), int(N), int(K), out);
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}

Status launchGemmFolded(int likeKernel, const GemmProblem &p, int mode,
                        int activation, float *statsOut, hipStream_t s) {
  HOM_CHECK_RET(likeKernel >= 0 && likeKernel < gemmKernelCount() &&
                    fusedGemmFits(p) &&
                    (p.beta == 0.f || (p.cRowPeriod >= p.M && p.ldc % 8 == 0)),
                Status::kInvalidArgument,
                "folded layer norm + gemm: problem does not fit the fused kernels");
  HOM_CHECK_RET((mode == 1 && (activation == 0 || activation == 1) && !statsOut &&
                 (!p.foldStats || p.colSum)) ||
                    (mode == 2 && activation == 0 &&
                     (!p.foldStats || p.beta != 0.f)),
                Status::kInvalidArgument,
                "folded layer norm + gemm: mode %d / activation %d not supported",
                mode, activation);
  // 32-bit byte offsets inside a tile's rows
  HOM_CHECK_RET(int64_t(256) * p.ldd * 2 < (int64_t(1) << 31) &&
                    int64_t(256) * p.ldc * 2 < (int64_t(1) << 31),
                Status::kInvalidArgument,
                "folded layer norm + gemm: leading dimension too large");
  GemmProblem q = p;
  q.splitK = 1;
  q.colSumSlices = 1;
  q.rowStatPartials = statsOut;
  if (mode == 1)
    return activation == 1 ? launchFusedTile<kEpiFoldAGelu>(likeKernel, q, s)
                           : launchFusedTile<kEpiFoldA>(likeKernel, q, s);
  if (!statsOut) {
    // the kernel always writes its partial sums: give it somewhere to put them
    const size_t bytes =
        size_t(foldedPieces(likeKernel, p.N)) * size_t(p.M) * 2 * sizeof(float);
    q.rowStatPartials = static_cast<float *>(libraryScratch(kTemp, bytes, false));
    if (!q.rowStatPartials)
      return Status::kInternal;
  }
  return launchFusedTile<kEpiFoldCStats>(likeKernel, q, s);
}

} // namespace hom

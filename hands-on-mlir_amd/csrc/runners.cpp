#include "runners.h"

#include "hom_amdgpu_runner_utils.h"
#include "rectangles.h"

#include <cerrno>
#include <cmath>
#include <cstring>
#include <fstream>
#include <sstream>
#include <string>

namespace hom {

namespace {

Epilogue epilogueFor(int64_t activation, bool nvtePath) {
  if (activation == 2)
    return Epilogue::kGeluTanh;
  if (activation == 1)
    return nvtePath ? Epilogue::kGeluTanh : Epilogue::kGeluErf;
  return Epilogue::kLinear;
}

// Shape rules of GemmOperationRunner::construct_arguments
// (include/NVGPUKernels/GemmRunner.h:244-287), with two relaxations: C may be
// broadcast over the batch and/or row dimension (bias row / per-batch matrix),
// as the CPU matmulAddF32 allows, and C is not inspected when beta == 0.
struct GemmShapes {
  int64_t batch, Mp, N, K;
};

Status checkGemmOperands(const View<_Float16> &A, const View<_Float16> &B,
                         const View<_Float16> &C, const View<_Float16> &D,
                         bool bIsNK, float beta, GemmShapes *out,
                         GemmProblem *pr) {
  HOM_CHECK_RET(A.rank == 3 && B.rank == 3 && C.rank == 3 && D.rank == 3,
                Status::kInvalidArgument,
                "gemm: all operands must have rank 3 (got %lld %lld %lld %lld)",
                (long long)A.rank, (long long)B.rank, (long long)C.rank,
                (long long)D.rank);
  HOM_CHECK_RET(A.sizes && B.sizes && C.sizes && D.sizes,
                Status::kInvalidArgument, "gemm: null descriptor");
  const int64_t batch = A.sizes[0], Mp = A.sizes[1], K = A.sizes[2];
  const int64_t bK = bIsNK ? B.sizes[2] : B.sizes[1];
  const int64_t N = bIsNK ? B.sizes[1] : B.sizes[2];
  HOM_CHECK_RET(K == bK, Status::kInvalidArgument,
                "gemm: K mismatch, A is [..,%lld] but B contracts over %lld",
                (long long)K, (long long)bK);
  HOM_CHECK_RET(B.sizes[0] == 1 || B.sizes[0] == batch || batch == 1,
                Status::kInvalidArgument,
                "gemm: B batch %lld incompatible with A batch %lld",
                (long long)B.sizes[0], (long long)batch);
  HOM_CHECK_RET(D.sizes[0] == batch && D.sizes[1] == Mp && D.sizes[2] == N,
                Status::kInvalidArgument,
                "gemm: D is [%lld,%lld,%lld], expected [%lld,%lld,%lld]",
                (long long)D.sizes[0], (long long)D.sizes[1],
                (long long)D.sizes[2], (long long)batch, (long long)Mp,
                (long long)N);
  HOM_CHECK_RET(A.contiguous() && B.contiguous() && D.contiguous(),
                Status::kInvalidArgument,
                "gemm: operands must be contiguous row-major");
  pr->ldc = 0;
  pr->cRowPeriod = 1;
  pr->C = nullptr;
  if (beta != 0.f) {
    HOM_CHECK_RET(C.sizes[2] == N, Status::kInvalidArgument,
                  "gemm: C has %lld columns, expected %lld",
                  (long long)C.sizes[2], (long long)N);
    HOM_CHECK_RET((C.sizes[0] == batch || C.sizes[0] == 1) &&
                      (C.sizes[1] == Mp || C.sizes[1] == 1),
                  Status::kInvalidArgument,
                  "gemm: C is [%lld,%lld,%lld], not broadcastable to "
                  "[%lld,%lld,%lld]",
                  (long long)C.sizes[0], (long long)C.sizes[1],
                  (long long)C.sizes[2], (long long)batch, (long long)Mp,
                  (long long)N);
    HOM_CHECK_RET(C.contiguous(), Status::kInvalidArgument,
                  "gemm: C must be contiguous row-major");
    HOM_CHECK_RET(C.data != nullptr, Status::kInvalidArgument,
                  "gemm: beta != 0 with a null C");
    pr->C = C.data;
    const bool rowsFull = C.sizes[1] == Mp;
    const bool batchFull = C.sizes[0] == batch;
    pr->ldc = N;
    if (rowsFull && batchFull) {
      pr->cRowPeriod = batch * Mp; // a full [b, M', N] source
    } else if (rowsFull) {
      pr->cRowPeriod = Mp; // one [M', N] matrix shared by every batch
    } else {
      // a single bias row; one row per batch cannot be expressed as a period
      HOM_CHECK_RET(C.sizes[0] == 1 || batch == 1, Status::kInvalidArgument,
                    "gemm: C broadcast over rows but not over batch is not "
                    "supported");
      pr->cRowPeriod = 1;
    }
  }
  pr->A = A.data;
  pr->B = B.data;
  pr->D = D.data;
  pr->M = batch * Mp;
  pr->N = N;
  pr->K = K;
  pr->lda = K;
  pr->ldb = bIsNK ? K : N;
  pr->ldd = N;
  pr->bIsNK = bIsNK;
  if (pr->cRowPeriod < 1)
    pr->cRowPeriod = 1;
  out->batch = batch;
  out->Mp = Mp;
  out->N = N;
  out->K = K;
  return Status::kSuccess;
}

int findKernel(int tileM, int tileN, int tileK, Epilogue epi, int alignment) {
  for (int i = 0; i < gemmKernelCount(); i++) {
    const GemmKernelInfo &k = gemmKernelInfo(i);
    if (k.tileM == tileM && k.tileN == tileN && k.tileK == tileK &&
        k.epilogue == epi && k.alignment == alignment)
      return i;
  }
  return -1;
}

struct TunedEntry {
  int64_t M, N, K;
  int activation; // 0 linear, 1 gelu erf, 2 gelu tanh
  const char *kernel; // best kernel for row-major B ([K, N])
  int splitK;
  const char *nkKernel; // best kernel for B given as [N, K] (may be null)
  int nkSplitK;
  int preferNK; // 1: the [N, K] path (nvteGemmF16) is the faster of the two
};

// Produced on an MI355X by the autotuner (hands-on-mlir_amd/tune_gemm.py) for
// the GEMM shapes of BERT-base and BERT-large; replaces the role of the
// CUTLASS manifest generator's per-architecture tile lists
// (python/gemm_generator.py:237-278).
const TunedEntry kTuned[] = {
#include "gemm_tuned_table.inc"
    {0, 0, 0, 0, nullptr, 0, nullptr, 0, 0}};

const TunedEntry *findTuned(int64_t M, int64_t N, int64_t K, int64_t activation) {
  // HOM_GEMM_IGNORE_TUNED_TABLE=1 answers from the timing model only (to check
  // the model against the table it was fitted to).
  static const bool useTable = getenv("HOM_GEMM_IGNORE_TUNED_TABLE") == nullptr;
  if (!useTable || N % 8 != 0 || K % 8 != 0)
    return nullptr;
  for (const TunedEntry *t = kTuned; t->kernel; t++)
    if (t->M == M && t->N == N && t->K == K && t->activation == activation)
      return t;
  return nullptr;
}

int kernelByName(const char *name) {
  if (name)
    for (int i = 0; i < gemmKernelCount(); i++)
      if (strcmp(gemmKernelInfo(i).name, name) == 0)
        return i;
  return -1;
}

// 8: every operand 16-byte aligned with N, K multiples of 8; 2: K a multiple
// of 8 and the K-contiguous operands 16-byte aligned, but N (the row length of
// row-major B, C, D) only even; 1: anything else.
int alignmentClass(const GemmProblem &p) {
  auto al = [](const void *q, int bytes) {
    return (reinterpret_cast<uintptr_t>(q) & uintptr_t(bytes - 1)) == 0;
  };
  if (p.K % 8 != 0 || !al(p.A, 16))
    return 1;
  const bool c8 = p.N % 8 == 0 && al(p.B, 16) && al(p.D, 16) &&
                  (p.C == nullptr || al(p.C, 16));
  if (c8)
    return 8;
  const bool c2 = p.N % 2 == 0 && (p.bIsNK ? al(p.B, 16) : al(p.B, 4)) &&
                  al(p.D, 4) && (p.C == nullptr || al(p.C, 4)) &&
                  (p.C == nullptr || p.ldc % 2 == 0);
  return c2 ? 2 : 1;
}

// A vector-access kernel (alignment 8) serves the problem when the problem's
// class is 8, or 2 and the kernel tolerates 4-byte aligned rows.
bool kernelFits(const GemmKernelInfo &k, int cls) {
  if (k.alignment == 1)
    return true;
  return cls == 8 || (cls == 2 && k.alignmentN <= 2);
}

// The kernels of gemm_ksplit.h: one wavefront computes the whole tile.
bool wavesSplitK(const GemmKernelInfo &k) { return k.wavesM * k.wavesN == 1; }

GemmSource sourceOf(const GemmProblem &p) {
  return p.beta == 0.f        ? GemmSource::kNone
         : p.cRowPeriod == 1 ? GemmSource::kRow
                             : GemmSource::kMatrix;
}

// Kernel and split-K (stored into pr) the [N, K]-B path runs for a problem.
int chooseNvteKernel(GemmProblem *pr, int64_t activation);

// The class of a problem whose operands are all aligned as well as its sizes
// allow.
int naturalClass(int64_t N, int64_t K) {
  return K % 8 != 0 ? 1 : (N % 8 == 0 ? 8 : (N % 2 == 0 ? 2 : 1));
}

// One tile of the register-staged family as the model below sees it: the
// kernels per epilogue of the vector-aligned and the any-alignment form (-1:
// there is none).
struct TileModel {
  int tileM, tileN, wavesM, wavesN, depth;
  int aligned[3], any[3];
};
// (the manifest is looked through once per process, not once per call)
const std::vector<TileModel> &tileModels() {
  static const std::vector<TileModel> models = [] {
    std::vector<TileModel> v = {
        {64, 64, 2, 2, 2, {}, {}},   {128, 64, 2, 2, 2, {}, {}},
        {64, 128, 2, 2, 2, {}, {}},  {128, 128, 2, 4, 2, {}, {}},
        {128, 256, 2, 4, 2, {}, {}}, {256, 128, 4, 2, 2, {}, {}},
        {256, 256, 2, 4, 1, {}, {}},
    };
    static const char *const epiName[3] = {"linear", "gelu", "gelutanh"};
    for (TileModel &t : v)
      for (int e = 0; e < 3; e++)
        for (int any = 0; any < 2; any++) {
          char name[160];
          snprintf(name, sizeof(name),
                   "hom_gfx950_mfma_f16_s32x32x16gemm_f16_%dx%d_64x2%c%d_w%dx%d_"
                   "nn_align%d_%s",
                   t.tileM, t.tileN, any ? 'u' : 'r', t.depth, t.wavesM,
                   t.wavesN, any ? 1 : 8, epiName[e]);
          (any ? t.any : t.aligned)[e] = kernelByName(name);
        }
    return v;
  }();
  return models;
}

// More 64 x 64 tiles than CUs: K is not split, and the tiles differ by what a round
// of them costs beyond its slabs, above all where all CUs write (and read a full
// source) at once.  t = fixed + rounds (slab K / 64 + round + gelu + source) + out M N +
// outSource M N + traffic of all tiles, us; a round is a tile on every CU.  Fitted to
// 560 problems x 7 tiles, M = 400 .. 20000, N = 64 .. 4500, K = 8 .. 4500, three sets of
// operands in turn: 6 to 8 % off in the mean, the choice 1.3 % off the best, 18 % at
// worst, on short K (the model below: 5.0 % and 38 %; 15866 x 3288 x 328 with GELU 119.8 ->
// 87.9 us, 10289 x 912 x 1256 with GELU 1.31 x less, 8372 x 1936 x 904 with a source 1.12 x);
// and to 130 problems whose rows of C and D are not on 16 bytes, which cost the larger
// tiles more (0.7 % off the best, the model below 10.7 %; 4622 x 502 x 272 with a source 64 x 64
// 10.5 us, 64 x 128 13.3).
bool modelFullChip(int64_t M, int64_t N, int64_t K, Epilogue epi, int cls, GemmSource source,
                   int64_t *idx, int32_t *splitK) {
  struct Fit {
    double fixed, slab, round, gelu, source, out, outSource, traffic;
  };
  // in the order of tileModels(); rows on 16 bytes, and others
  static const Fit fits[2][7] = {{
      {1.87, 0.191, 0.518, 0.128, 0, 0.0454, 0.199, 0.0188},
      {2.63, 0.320, 0, 0.229, 0, 0.509, 0.213, 0.0180},
      {2.51, 0.278, 0.132, 0.282, 0, 0.414, 0.179, 0.0195},
      {1.37, 0.382, 2.32, 0.459, 0, 0.127, 0.201, 0.0301},
      {1.44, 0.577, 3.16, 1.45, 0, 0.0616, 0.293, 0.0357},
      {1.34, 0.697, 3.10, 1.50, 0, 0.0692, 0.307, 0.0312},
      {0.32, 0.999, 7.65, 3.14, 4.03, 0.239, 0.436, 0.0395},
  }, {
      {2.82, 0.182, 0.373, 0.215, 0.159, 0.313, 0.189, 0.0232},
      {4.18, 0.331, 0.195, 0.568, 0.484, 0.499, 0.339, 0.0147},
      {3.99, 0.273, 0.600, 0.515, 0.502, 0.360, 0.357, 0.0189},
      {3.23, 0.439, 1.24, 1.11, 1.41, 0.478, 0.209, 0.0231},
      {5.19, 0.581, 2.24, 2.08, 3.16, 0.322, 0.282, 0.0310},
      {5.66, 0.730, 1.89, 2.15, 3.30, 0.332, 0.247, 0.0173},
      {9.14, 0.929, 3.86, 4.23, 6.72, 0.295, 0.458, 0.0386},
  }};
  const int cus = deviceInfo().computeUnits > 0 ? deviceInfo().computeUnits : 256;
  if (cls == 1 || ((M + 63) / 64) * ((N + 63) / 64) <= cus)
    return false;
  const bool fullSource = source == GemmSource::kMatrix;
  double best = 1e300;
  const double outputs = double(M) * double(N) * 1e-6, slabs = double((K + 63) / 64);
  for (size_t t = 0; t < tileModels().size(); t++) {
    const TileModel &m = tileModels()[t];
    const Fit &f = fits[cls == 8 ? 0 : 1][t];
    const int kernel = m.aligned[int(epi)];
    if (kernel < 0)
      continue;
    const double tiles = double((M + m.tileM - 1) / m.tileM) * double((N + m.tileN - 1) / m.tileN);
    const double traffic = tiles * (m.tileM + m.tileN) * double(K) * 2e-6;
    const double cost =
        f.fixed +
        std::ceil(tiles / cus) * (f.slab * slabs + f.round + (epi == Epilogue::kLinear ? 0 : f.gelu) +
                                  (fullSource ? f.source : 0)) +
        (f.out + (fullSource ? f.outSource : 0)) * outputs + f.traffic * traffic;
    if (cost < best) {
      best = cost;
      *idx = kernel;
      *splitK = 1;
    }
  }
  return best < 1e300;
}

// Kernel and split-K for an untuned shape of alignment class cls, from a timing
// model of the register-staged kernels, fitted to measurements of every tile
// over BERT-base / BERT-large sized problems (it reproduces them within 10 %):
//   t = launch + max(slabs * floor, compute + traffic) + epilogue
// compute = 64-wide K slabs x workgroups on the fullest CU x tile area x
// kUsPerOutputSlab (matrix cores and LDS of a CU are shared by its
// workgroups); traffic = bytes all tiles pull from L2, tiles x (BM + BN) x K
// x 2, at kL2BytesPerUs; floor = the load -> LDS -> MFMA latency chain of a
// lone workgroup; the epilogue costs per output; split-K adds a second kernel
// that moves the fp32 partial tiles through memory.
double modelPipe(int64_t M, int64_t N, int64_t K, Epilogue epi, int cls,
                 int64_t *idx, int32_t *splitK) {
  const int cus = deviceInfo().computeUnits > 0 ? deviceInfo().computeUnits : 256;
  constexpr double kLaunchUs = 3.0, kReduceLaunchUs = 2.5, kInKernelSumUs = 1.0;
  constexpr double kUsPerOutputSlab = 2.234e-5;
  constexpr double kL2BytesPerUs = 24.0e6;
  constexpr double kSlabFloorUs = 0.17;
  constexpr double kReduceBytesPerUs = 3.0e6; // partial tiles, written + read
  constexpr double kInKernelBytesPerUs = 9.0e6; // the same, staying in one L2
  const double epiNsPerOutput = epi == Epilogue::kLinear ? 0.045 : 0.12;
  double bestCost = 1e300;
  *idx = findKernel(64, 64, 32, epi, 1); // (rows shorter than a vector)
  *splitK = 1;
  if (cls == 1 && (K < 8 || N < 8))
    return 0.0;
  const int slabs = int((K + 63) / 64);
  for (const TileModel &t : tileModels()) {
    const int kernel = (cls == 1 ? t.any : t.aligned)[int(epi)];
    if (kernel < 0)
      continue;
    const int64_t tiles =
        ((M + t.tileM - 1) / t.tileM) * ((N + t.tileN - 1) / t.tileN);
    const double area = double(t.tileM) * t.tileN;
    const double traffic = double(tiles) * (t.tileM + t.tileN) * double(K) *
                           2.0 / kL2BytesPerUs;
    const int maxSplit = std::max(1, std::min(16, int(K / 128)));
    for (int sp = 1; sp <= maxSplit; sp++) {
      const int perSlice = (slabs + sp - 1) / sp;
      if (sp > 1 && perSlice < 4)
        break;
      const double perCu = std::ceil(double(tiles) * sp / cus);
      const double compute = perSlice * perCu * area * kUsPerOutputSlab;
      double cost = kLaunchUs +
                    std::max(perSlice * kSlabFloorUs, compute + traffic) +
                    std::ceil(double(tiles) / cus) * area * epiNsPerOutput * 1e-3;
      if (sp > 1) {
        // (the in-kernel sum saves most of the second launch where the
        // launcher will take it: same conditions as launchPipe)
        const bool inKernel = splitKInKernelMode() != 0 && tiles % 8 == 0 &&
                              (splitKInKernelMode() != 3 ||
                               splitKInKernelPays(t.tileM * t.tileN, sp, tiles));
        cost += (inKernel ? kInKernelSumUs : kReduceLaunchUs) +
                double(tiles) * sp * area * 8.0 /
                    (inKernel ? kInKernelBytesPerUs : kReduceBytesPerUs);
      }
      if (cost < bestCost) {
        bestCost = cost;
        *idx = kernel;
        *splitK = sp;
      }
    }
  }
  return bestCost;
}

// The same for the kernels whose wavefronts split K (gemm_ksplit.h), as far as all
// workgroups are resident at once; more rounds of them are never the better
// choice.  t = first + n (slab + crowd x share of the CUs at work) + sum, n slabs
// per workgroup, sum only with slices across workgroups; no faster than the weights
// arrive, 57 GB/s for a CU and 6.5 TB/s for all.  Fitted to 670 timings, M = 16
// .. 1000 x 18 pairs of N and K from 256 to 4096, launches one after the
// other on three sets of operands in turn: 1.4 to 3.5 % off in the mean.
double modelKsplit(int64_t M, int64_t N, int64_t K, Epilogue epi, int cls,
                   int64_t *idx, int32_t *splitK) {
  struct Fit {
    double first[2], slab[2], crowd[2]; // tiles of 16 and of 32 rows
    double sum, sumPerSlice;
  };
  static const Fit kVec = {{3.54, 3.95}, {0.088, 0.114}, {0.036, 0.054}, 1.35, 0.147};
  static const Fit kDword = {{3.42, 3.55}, {0.094, 0.138}, {0.090, 0.136}, 1.05, 0.19};
  static const Fit kOdd = {{3.15, 3.29}, {0.140, 0.194}, {0.094, 0.121}, 1.40, 0.21};
  static const std::vector<int> kernels = [] { // (tile, alignment, epilogue)
    std::vector<int> k;
    for (int rows : {16, 32})
      for (int al : {8, 1})
        for (Epilogue e : {Epilogue::kLinear, Epilogue::kGeluErf, Epilogue::kGeluTanh})
          k.push_back(findKernel(rows, 64, 64, e, al));
    return k;
  }();
  double best = 1e300;
  if (K < 8 || N < 8 || (K + 63) / 64 * 64 * N * 2 >= (int64_t(1) << 31))
    return best;
  const bool oddK = cls == 1 && K % 2 != 0, oddN = cls == 1 && N % 2 != 0;
  const Fit &f = cls != 1 ? kVec : oddK || oddN ? kOdd : kDword;
  const int cus = deviceInfo().computeUnits > 0 ? deviceInfo().computeUnits : 256;
  const int64_t slabs = (K + (oddK ? 62 : 63)) / (oddK ? 63 : 64);
  const int64_t cols = oddN ? 63 : 64;
  for (int t = 0; t < 2; t++) {
    const Rectangles r = chooseRectangles((M + 16 * (t + 1) - 1) / (16 * (t + 1)),
                                          (N + cols - 1) / cols, t + 1, 4, K, cus);
    const int64_t perXcd = int64_t(r.chunkM) * r.chunkN;
    for (int64_t sp = 1; sp <= 16 && perXcd * sp <= cus / 8; sp++) {
      const int64_t n = (slabs + sp - 1) / sp;
      if (sp > 1 && n < 4)
        break;
      if ((slabs + n - 1) / n != sp)
        continue;
      const double share = double(perXcd * sp) / (cus / 8);
      const double fetch = double(K * N + M * K) * 2 / std::min(6.5e6, 57e3 * cus * share);
      const double cost = f.first[t] + std::max(double(n) * (f.slab[t] + f.crowd[t] * share), fetch) +
                          (sp > 1 ? f.sum + f.sumPerSlice * double(sp) : 0.0);
      if (cost < best) {
        best = cost;
        *idx = kernels[(t * 2 + (cls == 1)) * 3 + int(epi)];
        *splitK = int32_t(sp);
      }
    }
  }
  return best;
}

// (a round of the larger tile on every CU: what modelKsplit() looks at at most)
bool ksplitFits(int64_t M, int64_t N) {
  const int cus = deviceInfo().computeUnits > 0 ? deviceInfo().computeUnits : 256;
  return ((M + 31) / 32) * ((N + 63) / 64) <= cus;
}

// Which of the two: the timings of the slab pipelines in the same runs lay off
// their model (fitted to one set of operands, aligned rows) by the lines below.
// On few slabs they lie below those lines, with most of the wavefronts here idle: over
// 300 problems, this kernel / the pipelines by slabs of K, rows on 16 bytes 1: 1.16, 2:
// 1.09, 3: 1.06, 4: 1.01, 5: 1.06, 6: 1.02, 7: 0.98, 8: 0.96; rows of C and D off them,
// up to 16 rows 1: 1.05, 2: 1.06, 3: 1.03, 4: 0.95, more rows without a source 1: 1.00, 2:
// 1.00, 3: 0.96, with one 1: 0.93, 2: 0.83, 3: 0.83; any alignment, N a multiple of 8: 1:
// 1.07, 2: 1.01, 3: 0.94, else 1: 0.93.
bool ksplitPays(int64_t M, int64_t N, int64_t K, Epilogue epi, int cls, GemmSource source,
                double pipe, int32_t pipeSplitK, int64_t *idx, int32_t *splitK) {
  const int few = cls == 8   ? 6
                  : cls == 2 ? (M <= 16 ? 3 : source == GemmSource::kNone ? 2 : 0)
                             : (N % 8 == 0 ? 2 : 0);
  if (K <= 64 * few)
    return false;
  int64_t i = -1;
  int32_t sk = 1;
  const double ksplit = modelKsplit(M, N, K, epi, cls, &i, &sk);
  const double seen = cls != 1 ? (pipeSplitK == 1 ? 1.1 + 0.78 * pipe : 0.8 + pipe)
                               : (pipeSplitK == 1 ? 1.5 * pipe - 0.3 : 1.3 * pipe + 0.6);
  if (i < 0 || ksplit >= 0.97 * seen)
    return false;
  *idx = i;
  *splitK = sk;
  return true;
}

void modelGemm(int64_t M, int64_t N, int64_t K, Epilogue epi, int cls, GemmSource source,
               int64_t *idx, int32_t *splitK) {
  if (modelFullChip(M, N, K, epi, cls, source, idx, splitK))
    return;
  const double pipe = modelPipe(M, N, K, epi, cls, idx, splitK);
  if (ksplitFits(M, N))
    ksplitPays(M, N, K, epi, cls, source, pipe, *splitK, idx, splitK);
}

} // namespace

namespace {
// A split that the library chose needs scratch memory, which a stream under capture
// cannot allocate: in front of the first eager call, K is not split across
// workgroups there.
void unsplitWithoutScratch(int idx, GemmProblem *pr) {
  const GemmKernelInfo &ki = gemmKernelInfo(idx);
  if (pr->splitK <= 1 || pr->workspace || !wavesSplitK(ki))
    return;
  // (63 columns: see gemm_ksplit.h)
  const size_t tiles = size_t((pr->M + ki.tileM - 1) / ki.tileM) *
                       size_t((pr->N + ki.tileN - 2) / (ki.tileN - 1));
  if (!libraryScratchReady(kWorkspace, tiles * size_t(pr->splitK) * ki.tileM * ki.tileN * sizeof(float)))
    pr->splitK = 1;
}
} // namespace

bool gemmPrefersNvte(int64_t M, int64_t N, int64_t K, int64_t activation) {
  const TunedEntry *t = findTuned(M, N, K, activation);
  return t && t->preferNK && kernelByName(t->nkKernel) >= 0;
}

bool selectGemm(int64_t M, int64_t N, int64_t K, int64_t activation,
                int64_t *idx, int32_t *splitK, bool bIsNK, GemmSource source) {
  const Epilogue epi = epilogueFor(activation, false);
  if (const TunedEntry *t = findTuned(M, N, K, activation)) {
    const int nk = bIsNK ? kernelByName(t->nkKernel) : -1;
    const int i = nk >= 0 ? nk : kernelByName(t->kernel);
    if (i >= 0) {
      *idx = i;
      *splitK = nk >= 0 ? t->nkSplitK : t->splitK;
      return true;
    }
  }
  modelGemm(M, N, K, epi, naturalClass(N, K), source, idx, splitK);
  return false;
}

Status runGemmManifest(int64_t rankA, void *dstA, int64_t rankB, void *dstB,
                       int64_t rankC, void *dstC, int64_t rankD, void *dstD,
                       int64_t activation, float alpha, float beta,
                       int32_t gemmNum, int32_t splitK, bool noAlloc) {
  View<_Float16> A(rankA, dstA), B(rankB, dstB), C(rankC, dstC), D(rankD, dstD);
  GemmProblem pr{};
  GemmShapes sh{};
  Status st = checkGemmOperands(A, B, C, D, false, beta, &sh, &pr);
  if (st != Status::kSuccess)
    return st;
  if (noAlloc) {
    // split-K partial tiles go to the fixed device array; a problem that needs
    // more than it holds is rejected by the launch instead of allocating
    st = noAllocWorkspace(&pr.workspace, &pr.workspaceBytes);
    if (st != Status::kSuccess)
      return st;
  }
  pr.alpha = alpha;
  pr.beta = beta;
  int idx;
  if (gemmNum >= 1) {
    HOM_CHECK_RET(gemmNum <= gemmKernelCount(), Status::kInvalidArgument,
                  "gemm: kernel number %d outside the manifest (1..%d)",
                  gemmNum, gemmKernelCount());
    idx = gemmNum - 1;
    HOM_CHECK_RET(splitK >= 1, Status::kInvalidArgument,
                  "gemm: split-K factor must be >= 1 (got %d)", splitK);
    pr.splitK = splitK;
  } else {
    // The reference indexes manifest[-1] here (undefined); this library
    // treats 0 as "choose for me" using the activation argument.
    HOM_CHECK_RET(gemmNum == 0, Status::kInvalidArgument,
                  "gemm: negative kernel number %d", gemmNum);
    int64_t sel;
    int32_t sk;
    const GemmSource source = sourceOf(pr);
    selectGemm(pr.M, pr.N, pr.K, activation, &sel, &sk, false, source);
    const int cls = alignmentClass(pr);
    if (!kernelFits(gemmKernelInfo(int(sel)), cls))
      modelGemm(pr.M, pr.N, pr.K, gemmKernelInfo(int(sel)).epilogue, cls, source, &sel,
                &sk);
    idx = int(sel);
    pr.splitK = sk;
    if (noAlloc) {
      // The caller did not ask for split-K: a factor the library chose itself
      // shrinks until its partial tiles fit the fixed array (1 needs none).
      // An explicit gemmNum / splitK that does not fit is rejected by the launch.
      const GemmKernelInfo &ki = gemmKernelInfo(idx);
      const size_t perSlice = size_t((pr.M + ki.tileM - 1) / ki.tileM) *
                              size_t((pr.N + ki.tileN - 1) / ki.tileN) *
                              size_t(ki.tileM) * ki.tileN * sizeof(float);
      while (pr.splitK > 1 && perSlice * size_t(pr.splitK) > pr.workspaceBytes)
        pr.splitK--;
    }
  }
  if (gemmNum == 0)
    unsplitWithoutScratch(idx, &pr);
  return launchGemm(idx, pr, stream());
}

bool selectGemmNvte(int64_t M, int64_t N, int64_t K, int64_t activation,
                    int64_t *idx, int32_t *splitK, GemmSource source) {
  const Epilogue epi = epilogueFor(activation, true);
  return selectGemm(M, N, K, epi == Epilogue::kGeluTanh ? 2 : activation, idx,
                    splitK, true, source);
}

namespace {
int chooseNvteKernel(GemmProblem *pr, int64_t activation) {
  int64_t sel;
  int32_t sk;
  const Epilogue epi = epilogueFor(activation, true);
  const GemmSource source = sourceOf(*pr);
  selectGemmNvte(pr->M, pr->N, pr->K, activation, &sel, &sk, source);
  int idx = int(sel);
  pr->splitK = sk;
  // Profiling knob: HOM_NVTE_GEMM_KERNEL="<manifest name>[,<splitK>]" pins the
  // kernel used on this path (the epilogue must match the activation).
  if (const char *force = getenv("HOM_NVTE_GEMM_KERNEL")) {
    std::string f(force);
    const size_t comma = f.find(',');
    const std::string name = f.substr(0, comma);
    for (int i = 0; i < gemmKernelCount(); i++)
      if (name == gemmKernelInfo(i).name && gemmKernelInfo(i).epilogue == epi) {
        idx = i;
        pr->splitK = comma == std::string::npos ? 1 : atoi(f.c_str() + comma + 1);
      }
  }
  const int cls = alignmentClass(*pr);
  if (!kernelFits(gemmKernelInfo(idx), cls)) {
    modelGemm(pr->M, pr->N, pr->K, epi, cls, source, &sel, &sk);
    idx = int(sel);
    pr->splitK = sk;
  }
  return idx;
}
} // namespace

Status runGemmNvte(int64_t rankA, void *dstA, bool transa, int64_t rankB,
                   void *dstB, bool transb, int64_t rankC, void *dstC,
                   int64_t rankD, void *dstD, int64_t activation, float alpha,
                   float beta) {
  // Preconditions of GemmNVTERunner::construct_tensors (GemmRunner.h:342-381).
  HOM_CHECK_RET(transa == false, Status::kInvalidArgument,
                "nvte gemm: transa must be false");
  HOM_CHECK_RET(transb == true, Status::kInvalidArgument,
                "nvte gemm: transb must be true (B is [1, N, K])");
  HOM_CHECK_RET(alpha == 1.0f, Status::kInvalidArgument,
                "nvte gemm: alpha must be 1 (got %g)", double(alpha));
  HOM_CHECK_RET(beta == 0.0f || beta == 1.0f, Status::kInvalidArgument,
                "nvte gemm: beta must be 0 or 1 (got %g)", double(beta));
  HOM_CHECK_RET(activation >= 0 && activation <= 2, Status::kInvalidArgument,
                "nvte gemm: unknown activation %lld", (long long)activation);
  View<_Float16> A(rankA, dstA), B(rankB, dstB), C(rankC, dstC), D(rankD, dstD);
  GemmProblem pr{};
  GemmShapes sh{};
  Status st = checkGemmOperands(A, B, C, D, true, beta, &sh, &pr);
  if (st != Status::kSuccess)
    return st;
  HOM_CHECK_RET(B.sizes[0] == 1, Status::kInvalidArgument,
                "nvte gemm: B batch must be 1");
  if (beta != 0.f) {
    HOM_CHECK_RET(C.data == D.data, Status::kInvalidArgument,
                  "nvte gemm: beta == 1 accumulates in place, C must alias D");
  }
  pr.alpha = alpha;
  pr.beta = beta;
  const int idx = chooseNvteKernel(&pr, activation);
  unsplitWithoutScratch(idx, &pr);
  return launchGemm(idx, pr, stream());
}

// The two halves of the layer-norm pair (LayernormGemmRunner.h:17-361).  Both
// keep the normalisation out of memory when the problem is in the vector
// alignment class: the first GEMM's epilogue accumulates the row statistics
// of D, the second folds var/mean into its epilogue through the column sums of
// B.  Other shapes run the same arithmetic as separate kernels.
Status runGemmWithVarMean(int64_t rankA, void *dstA, int64_t rankB, void *dstB,
                          int64_t rankC, void *dstC, int64_t rankD, void *dstD,
                          int64_t rankVar, void *dstVar, int64_t rankMean,
                          void *dstMean, float alpha, float beta,
                          int64_t activation, float eps) {
  (void)activation; // linear epilogue only, as in the reference instance
  View<_Float16> A(rankA, dstA), B(rankB, dstB), C(rankC, dstC), D(rankD, dstD);
  View<_Float16> Var(rankVar, dstVar), Mean(rankMean, dstMean);
  GemmProblem pr{};
  GemmShapes sh{};
  Status st = checkGemmOperands(A, B, C, D, false, beta, &sh, &pr);
  if (st != Status::kSuccess)
    return st;
  const int64_t rows = pr.M, n = pr.N;
  HOM_CHECK_RET(Var.sizes && Mean.sizes && Var.numel() >= rows &&
                    Mean.numel() >= rows,
                Status::kInvalidArgument,
                "gemm+stats: Var/Mean need one element per output row (%lld)",
                (long long)rows);
  pr.alpha = alpha;
  pr.beta = beta;
  if (fusedGemmFits(pr)) {
    return launchGemmRowStats(pr, Var.data, Mean.data, eps, stream());
  }
  st = runGemmManifest(rankA, dstA, rankB, dstB, rankC, dstC, rankD, dstD, 0,
                       alpha, beta, 0, 1);
  if (st != Status::kSuccess)
    return st;
  HOM_CHECK_RET(D.contiguous(), Status::kInvalidArgument,
                "gemm+stats: D must be contiguous");
  return launchRowStatsF16(D.data, Var.data, Mean.data, rows, n, eps, stream());
}

namespace {
// The tile family member a folded GEMM imitates: the caller's manifest kernel
// (1-based) or the library's choice for the shape.
int foldedLikeKernel(const GemmProblem &pr, int64_t activation, int32_t likeGemmNum) {
  (void)activation;
  if (likeGemmNum >= 1 && likeGemmNum <= gemmKernelCount())
    return likeGemmNum - 1;
  // The folded kernels exist with 256 x 256, 128 x 128 and 64 x 64 tiles: the
  // largest that still gives most of the CUs a tile.
  auto tiles = [&](int64_t edge) {
    return ((pr.M + edge - 1) / edge) * ((pr.N + edge - 1) / edge);
  };
  const int cus = deviceInfo().computeUnits > 0 ? deviceInfo().computeUnits : 256;
  const int edge = tiles(256) * 5 >= int64_t(cus) * 4   ? 256
                   : tiles(128) * 2 >= int64_t(cus) ? 128
                                                    : 64;
  const int like = findKernel(edge, edge, 64, Epilogue::kLinear, 8);
  return like >= 0 ? like : 0;
}
} // namespace

Status runGemmFoldedLayernorm(int64_t rankA, void *dstA, int64_t rankB,
                              void *dstB, int64_t rankC, void *dstC,
                              int64_t rankD, void *dstD, int32_t mode,
                              int64_t activation, float alpha, float beta,
                              const float *statsIn, int32_t piecesIn, float eps,
                              const float *colSumB, float *statsOut,
                              int32_t likeGemmNum) {
  View<_Float16> A(rankA, dstA), B(rankB, dstB), C(rankC, dstC), D(rankD, dstD);
  GemmProblem pr{};
  GemmShapes sh{};
  Status st = checkGemmOperands(A, B, C, D, false, beta, &sh, &pr);
  if (st != Status::kSuccess)
    return st;
  HOM_CHECK_RET(mode == 1 || mode == 2, Status::kInvalidArgument,
                "folded layer norm: mode must be 1 (rows of A) or 2 (rows of C), got %d",
                mode);
  HOM_CHECK_RET(!statsIn || piecesIn >= 1, Status::kInvalidArgument,
                "folded layer norm: %d pieces of partial sums", piecesIn);
  pr.alpha = alpha;
  pr.beta = beta;
  pr.foldStats = statsIn;
  pr.foldPieces = piecesIn;
  pr.foldInvN = 1.0f / float(mode == 1 ? pr.K : pr.N);
  pr.foldEps = eps;
  pr.colSum = colSumB;
  if (pr.M == 0 || pr.N == 0)
    return Status::kSuccess;
  return launchGemmFolded(foldedLikeKernel(pr, activation, likeGemmNum), pr, mode,
                          int(activation), statsOut, stream());
}

int32_t foldedLayernormPieces(int64_t M, int64_t N, int64_t K, int64_t activation,
                              int32_t likeGemmNum) {
  GemmProblem pr{};
  pr.M = M;
  pr.N = N;
  pr.K = K;
  return foldedPieces(foldedLikeKernel(pr, activation, likeGemmNum), N);
}

Status runColumnSums(int64_t rankB, void *dstB, float *out) {
  View<_Float16> B(rankB, dstB);
  HOM_CHECK_RET(B.sizes && rankB == 3 && B.sizes[0] == 1 && B.strides[2] == 1,
                Status::kInvalidArgument,
                "column sums: B must be a [1, K, N] tensor with contiguous rows");
  return launchColumnSums(B.data, B.strides[1], B.sizes[1], B.sizes[2], out,
                          stream());
}

// B [1, K, N] as the packed form takes it, and where that lies
static Status checkPackWeight(const char *what, const View<_Float16> &B, const void *packed) {
  HOM_CHECK_RET(B.sizes && B.rank == 3 && B.sizes[0] == 1 && B.contiguous() &&
                    B.sizes[1] % 32 == 0 && B.sizes[2] % 16 == 0 &&
                    B.numel() * 2 < (int64_t(1) << 31),
                Status::kInvalidArgument,
                "%s: B must be a contiguous [1, K, N] tensor below 2 GiB "
                "with K a multiple of 32 and N of 16", what);
  HOM_CHECK_RET(packed && (reinterpret_cast<uintptr_t>(packed) & 15) == 0,
                Status::kInvalidArgument, "%s: misaligned packed weight", what);
  return Status::kSuccess;
}

Status runPackWeight(int64_t rankB, void *dstB, void *packed) {
  View<_Float16> B(rankB, dstB);
  const Status st = checkPackWeight("pack weight", B, packed);
  if (st != Status::kSuccess || B.numel() == 0)
    return st;
  return launchPackWeight(B.data, static_cast<_Float16 *>(packed), B.sizes[1],
                          B.sizes[2], stream());
}

Status runUnpackWeight(const void *packed, int64_t rankB, void *dstB) {
  View<_Float16> B(rankB, dstB);
  const Status st = checkPackWeight("unpack weight", B, packed);
  if (st != Status::kSuccess || B.numel() == 0)
    return st;
  return launchUnpackWeight(static_cast<const _Float16 *>(packed), B.data, B.sizes[1],
                            B.sizes[2], stream());
}

Status runPackRows(int64_t rankA, void *dstA, int64_t rankOut, void *dstOut) {
  View<_Float16> A(rankA, dstA), O(rankOut, dstOut);
  HOM_CHECK_RET(A.rank == 3 && O.rank == 3 && A.sizes && O.sizes &&
                    A.contiguous() && O.contiguous() &&
                    A.sizes[0] == O.sizes[0] && A.sizes[1] == O.sizes[1] &&
                    A.sizes[2] == O.sizes[2] && A.sizes[2] % 32 == 0 &&
                    A.data != O.data,
                Status::kInvalidArgument,
                "pack rows: A and Out must be two contiguous tensors of one "
                "[b, s, H] shape with H a multiple of 32");
  const int64_t M = A.sizes[0] * A.sizes[1], C = A.sizes[2];
  HOM_CHECK_RET(M < (int64_t(1) << 31) && (M + 15) / 16 * 16 * C < (int64_t(1) << 37),
                Status::kInvalidArgument, "pack rows: tensor too large");
  HOM_CHECK_RET(((reinterpret_cast<uintptr_t>(A.data) | reinterpret_cast<uintptr_t>(O.data)) & 15) == 0,
                Status::kInvalidArgument, "pack rows: misaligned operands");
  if (M == 0 || C == 0)
    return Status::kSuccess;
  return launchPackRows(A.data, O.data, M, C, stream());
}

Status runPackedLayernorm(int64_t rankA, void *dstA, int64_t rankOut, void *dstOut,
                          float eps, int32_t packing) {
  View<_Float16> A(rankA, dstA), O(rankOut, dstOut);
  HOM_CHECK_RET(A.rank == 3 && O.rank == 3 && A.sizes && O.sizes &&
                    A.contiguous() && O.contiguous() &&
                    A.sizes[0] == O.sizes[0] && A.sizes[1] == O.sizes[1] &&
                    A.sizes[2] == O.sizes[2],
                Status::kInvalidArgument,
                "packed layer norm: A and Out must be contiguous tensors of one "
                "[b, s, H] shape");
  const int64_t M = A.sizes[0] * A.sizes[1], N = A.sizes[2];
  HOM_CHECK_RET((packing & HOM_PACKED_A) && N % 32 == 0 && N <= 2048 &&
                    M < (int64_t(1) << 31) - 16,
                Status::kInvalidArgument,
                "packed layer norm: A must be in fragment order with H a multiple "
                "of 32, at most 2048");
  HOM_CHECK_RET(A.data != O.data || (packing & HOM_PACKED_D),
                Status::kInvalidArgument,
                "packed layer norm: a row-major result cannot replace A");
  if (M == 0 || N == 0)
    return Status::kSuccess;
  return launchPackedLayernorm(A.data, O.data, M, N, eps,
                               (packing & HOM_PACKED_D) != 0, stream());
}

Status runPackedGemm(int64_t rankA, void *dstA, const void *packedB, int64_t rankC,
                     void *dstC, int64_t rankD, void *dstD, int64_t activation,
                     int32_t normA, float eps, const float *colSumB,
                     const float *statsIn, float *statsOut, int32_t packing,
                     const void *ahead, int64_t aheadBytes) {
  View<_Float16> A(rankA, dstA), C(rankC, dstC), D(rankD, dstD);
  HOM_CHECK_RET(A.rank == 3 && D.rank == 3 && A.sizes && D.sizes &&
                    A.contiguous() && D.contiguous() &&
                    A.sizes[0] == D.sizes[0] && A.sizes[1] == D.sizes[1],
                Status::kInvalidArgument,
                "packed gemm: A and D must be contiguous [b, M', K] and [b, M', N]");
  PackedGemm g{};
  g.M = A.sizes[0] * A.sizes[1];
  g.K = A.sizes[2];
  g.N = D.sizes[2];
  HOM_CHECK_RET(g.K % 32 == 0 && g.N % 16 == 0 && g.K > 0 &&
                    g.M * std::max(g.K, g.N) < (int64_t(1) << 30) &&
                    g.K * g.N < (int64_t(1) << 30),
                Status::kInvalidArgument,
                "packed gemm: K must be a multiple of 32, N of 16, and the "
                "operands below 2 GiB (M=%lld N=%lld K=%lld)",
                (long long)g.M, (long long)g.N, (long long)g.K);
  g.aPacked = (packing & HOM_PACKED_A) != 0;
  g.cPacked = (packing & HOM_PACKED_C) != 0;
  g.dPacked = (packing & HOM_PACKED_D) != 0;
  HOM_CHECK_RET(g.N % 32 == 0 || !(g.cPacked || g.dPacked),
                Status::kInvalidArgument,
                "packed gemm: C or D in fragment order need N a multiple of 32");
  HOM_CHECK_RET(activation >= 0 && activation <= 2, Status::kInvalidArgument,
                "packed gemm: unknown activation %lld", (long long)activation);
  if (dstC) {
    HOM_CHECK_RET(C.rank == 3 && C.contiguous() && C.numel() == g.M * g.N &&
                      C.sizes[2] == g.N && activation == 0,
                  Status::kInvalidArgument,
                  "packed gemm: C must be a contiguous tensor of D's shape, and "
                  "the activation linear");
    g.C = C.data;
  }
  HOM_CHECK_RET(!normA || colSumB, Status::kInvalidArgument,
                "packed gemm: a normalised A needs the column sums of B");
  HOM_CHECK_RET(!statsOut || normA, Status::kInvalidArgument,
                "packed gemm: statistics are written for a normalised A only");
  HOM_CHECK_RET(!statsIn || dstC, Status::kInvalidArgument,
                "packed gemm: row statistics without a source");
  auto al16 = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  HOM_CHECK_RET(al16(A.data) && al16(packedB) && al16(D.data) && al16(g.C) &&
                    al16(colSumB) && al16(ahead),
                Status::kInvalidArgument, "packed gemm: misaligned operands");
  HOM_CHECK_RET(aheadBytes >= 0, Status::kInvalidArgument,
                "packed gemm: aheadBytes must not be negative (%lld)", (long long)aheadBytes);
  // D may take the place of C (same order: every value is read by the lane that
  // replaces it), of nothing else that other workgroups may still read
  auto overlaps = [&](const void *q, int64_t cols, bool packed) {
    auto rows = [&](bool whole) { return whole ? (g.M + 15) / 16 * 16 : g.M; };
    const uintptr_t d = reinterpret_cast<uintptr_t>(D.data), x = reinterpret_cast<uintptr_t>(q);
    return x < d + uintptr_t(rows(g.dPacked) * g.N * 2) && d < x + uintptr_t(rows(packed) * cols * 2);
  };
  HOM_CHECK_RET(!overlaps(A.data, g.K, g.aPacked), Status::kInvalidArgument,
                "packed gemm: D overlaps A");
  HOM_CHECK_RET(!dstC || (g.C == D.data && g.cPacked == g.dPacked) ||
                    !overlaps(g.C, g.N, g.cPacked),
                Status::kInvalidArgument,
                "packed gemm: D overlaps C in another place or order");
  if (g.M == 0 || g.N == 0)
    return Status::kSuccess;
  g.A = A.data;
  g.packedB = static_cast<const _Float16 *>(packedB);
  g.D = D.data;
  g.colSum = colSumB;
  g.statsIn = statsIn;
  g.statsOut = statsOut;
  g.activation = int(activation);
  g.normA = normA != 0;
  g.eps = eps;
  g.ahead = ahead;
  g.aheadBytes = aheadBytes & ~int64_t(15);
  return launchPackedGemm(g, stream());
}

bool selectPackedGemm(int64_t M, int64_t N, int64_t K, int64_t activation, int32_t normA,
                      int32_t source, int32_t packing, int32_t readsAhead, PackedKernel *out) {
  const bool wide = packing & (HOM_PACKED_C | HOM_PACKED_D);
  if (M < 1 || N < 1 || K < 1 || K % 32 != 0 || N % (wide ? 32 : 16) != 0 ||
      M * std::max(K, N) >= (int64_t(1) << 30) || K * N >= (int64_t(1) << 30) ||
      activation < 0 || activation > 2 || (source && activation))
    return false;
  // (operands are told apart by being there or not)
  static const _Float16 present = 0;
  PackedGemm g{};
  g.M = M;
  g.N = N;
  g.K = K;
  g.aPacked = (packing & HOM_PACKED_A) != 0;
  g.cPacked = (packing & HOM_PACKED_C) != 0;
  g.dPacked = (packing & HOM_PACKED_D) != 0;
  g.C = source ? &present : nullptr;
  g.ahead = readsAhead ? &present : nullptr;
  g.activation = int(activation);
  g.normA = normA != 0;
  g.only = out;
  return launchPackedGemm(g, nullptr) == Status::kSuccess;
}

Status runLayernormGemm(int64_t rankA, void *dstA, int64_t rankB, void *dstB,
                        int64_t rankC, void *dstC, int64_t rankD, void *dstD,
                        int64_t rankVar, void *dstVar, int64_t rankMean,
                        void *dstMean, float alpha, float beta,
                        int64_t activation) {
  (void)activation;
  View<_Float16> A(rankA, dstA), B(rankB, dstB), C(rankC, dstC), D(rankD, dstD);
  View<_Float16> Var(rankVar, dstVar), Mean(rankMean, dstMean);
  GemmProblem pr{};
  GemmShapes sh{};
  Status st = checkGemmOperands(A, B, C, D, false, beta, &sh, &pr);
  if (st != Status::kSuccess)
    return st;
  const int64_t rows = pr.M, k = pr.K;
  HOM_CHECK_RET(Var.sizes && Mean.sizes && Var.numel() >= rows &&
                    Mean.numel() >= rows,
                Status::kInvalidArgument,
                "layernorm-gemm: Var/Mean need one element per row (%lld)",
                (long long)rows);
  pr.alpha = alpha;
  pr.beta = beta;
  if (fusedGemmFits(pr)) {
    return launchGemmRowAffine(pr, Var.data, Mean.data, stream());
  }
  HOM_CHECK_RET(A.contiguous(), Status::kInvalidArgument,
                "layernorm-gemm: A must be a contiguous rank-3 tensor");
  _Float16 *tmp = static_cast<_Float16 *>(
      libraryScratch(kTemp, size_t(rows) * k * sizeof(_Float16), false));
  if (!tmp && rows * k > 0)
    return Status::kInternal;
  st = launchApplyRowStatsF16(A.data, Var.data, Mean.data, tmp, rows, k,
                              stream());
  if (st != Status::kSuccess)
    return st;
  // Same descriptor as A, pointing at the normalised copy.
  HomStridedMemRef3 normA;
  memcpy(&normA, dstA, sizeof(normA));
  normA.basePtr = normA.data = tmp;
  return runGemmManifest(3, &normA, rankB, dstB, rankC, dstC, rankD, dstD, 0,
                         alpha, beta, 0, 1);
}

// ---------------------------------------------------------------- profiler --
GemmProfiler::GemmProfiler(int64_t M, int64_t N, int64_t K, int64_t activation,
                           float alpha, float beta)
    : M_(M), N_(N), K_(K), activation_(activation), alpha_(alpha), beta_(beta) {
  if (hipEventCreate(&start_) != hipSuccess ||
      hipEventCreate(&stop_) != hipSuccess)
    recordError(__FILE__, __LINE__, "profiler: cannot create HIP events");
}

GemmProfiler::~GemmProfiler() {
  if (start_)
    (void)hipEventDestroy(start_);
  if (stop_)
    (void)hipEventDestroy(stop_);
  for (Buffer *b : {&a_, &b_, &c_})
    if (b->data)
      (void)hipFree(b->data);
}

bool GemmProfiler::ensure(Buffer &b, int64_t elems) {
  if (elems <= b.capacity)
    return true;
  if (b.data)
    (void)hipFree(b.data);
  b.data = nullptr;
  b.capacity = 0;
  void *p = nullptr;
  if (hipMalloc(&p, size_t(elems) * sizeof(_Float16)) != hipSuccess) {
    recordError(__FILE__, __LINE__, "profiler: hipMalloc of %lld halves failed",
                (long long)elems);
    return false;
  }
  // Random finite values: on this GPU the clock under MFMA load depends on how
  // much the operands toggle, so all-zero buffers would flatter every kernel.
  {
    std::vector<_Float16> host(static_cast<size_t>(elems));
    uint32_t x = 0x9E3779B9u ^ uint32_t(elems);
    for (auto &v : host) {
      x ^= x << 13;
      x ^= x >> 17;
      x ^= x << 5;
      v = _Float16((float(x & 0xffff) / 32768.0f - 1.0f) * 0.5f);
    }
    (void)hipMemcpy(p, host.data(), size_t(elems) * sizeof(_Float16),
                    hipMemcpyHostToDevice);
  }
  b.data = static_cast<_Float16 *>(p);
  b.capacity = elems;
  return true;
}

// Protocol of GemmProfiler::profileHelper (lib/NVGPUKernels/GemmProfiler.cu:
// 81-120): 10 warm-up launches, then batches of 100 between two events until
// 500 ms have been spent or the kernel is 1.2x slower than the best so far.
GemmProblem GemmProfiler::problem(bool bIsNK) const {
  GemmProblem pr{};
  pr.A = a_.data;
  pr.B = b_.data; // the same scratch values serve as [K, N] and as [N, K]
  pr.C = beta_ != 0.f ? c_.data : nullptr;
  pr.D = c_.data;
  pr.M = M_;
  pr.N = N_;
  pr.K = K_;
  pr.lda = K_;
  pr.ldb = bIsNK ? K_ : N_;
  pr.ldc = N_;
  pr.ldd = N_;
  pr.cRowPeriod = M_;
  pr.alpha = alpha_;
  pr.beta = beta_;
  pr.bIsNK = bIsNK;
  pr.splitK = 1;
  return pr;
}

float GemmProfiler::timeKernel(int idx, int splitK, float previousBest,
                               bool bIsNK) {
  GemmProblem pr = problem(bIsNK);
  pr.splitK = splitK;
  hipStream_t s = stream();
  if (hipStreamSynchronize(s) != hipSuccess)
    return INFINITY;
  // A kernel that cannot implement the problem (leading dimension or operand
  // too large for its 32-bit offsets, too many tiles, ...) is skipped, as the
  // reference skips kernels whose can_implement() fails: the first launch runs
  // with errors recorded silently instead of aborting the compiler process.
  {
    const int savedMode = errorMode();
    setErrorMode(2);
    const Status probe = launchGemm(idx, pr, s);
    setErrorMode(savedMode);
    if (probe != Status::kSuccess) {
      (void)takeLastError();
      return INFINITY;
    }
  }
  for (int i = 0; i < 9; i++)
    if (launchGemm(idx, pr, s) != Status::kSuccess)
      return INFINITY;
  // 500 ms per candidate is the reference's budget; HOM_PROFILE_BUDGET_MS
  // shortens it for table generation over many shapes.
  static const float budgetMs = [] {
    const char *v = getenv("HOM_PROFILE_BUDGET_MS");
    const float f = v ? float(atof(v)) : 500.f;
    return f > 1.f ? f : 500.f;
  }();
  float total = 0.f;
  int64_t iters = 0;
  while (total < budgetMs) {
    float batch = 0.f;
    (void)hipEventRecord(start_, s);
    for (int i = 0; i < 100; i++)
      (void)launchGemm(idx, pr, s);
    (void)hipEventRecord(stop_, s);
    if (hipEventSynchronize(stop_) != hipSuccess)
      return INFINITY;
    (void)hipEventElapsedTime(&batch, start_, stop_);
    total += batch;
    iters += 100;
    if (total / float(iters) / 1.2f > previousBest)
      break;
  }
  return total / float(iters);
}

// Every eligible manifest kernel x split-K factor for one B layout; a
// candidate has to beat (bestIdx, bestSplit, bestTime) as passed in.
void GemmProfiler::sweep(bool bIsNK, int64_t *bestIdx, int32_t *bestSplit,
                         float *bestTime) {
  const Epilogue epi = epilogueFor(activation_, false);
  // Alignment class (the reference walks {8,4,2,1} over M, N, K:
  // lib/NVGPUKernels/GemmProfiler.cu:170-180; here K must be a multiple of 8
  // for the vector kernels, N of 8 or 2, and the row count is free).
  const int cls = naturalClass(N_, K_);
  const int maxSplit = std::max(1, std::min<int>(16, int(K_ / 128)));
  const int cus = deviceInfo().computeUnits > 0 ? deviceInfo().computeUnits : 256;
  for (int idx = 0; idx < gemmKernelCount(); idx++) {
    const GemmKernelInfo &k = gemmKernelInfo(idx);
    if (k.epilogue != epi || !kernelFits(k, cls))
      continue;
    if (k.alignment == 1 && cls != 1)
      continue; // the scalar-access kernels never win on aligned problems
    const int64_t tiles = ((M_ + k.tileM - 1) / k.tileM) *
                          ((N_ + k.tileN - 1) / k.tileN);
    for (int s = 1; s <= maxSplit; s++) {
      // Slicing K further once the grid already covers the chip many times
      // only adds reduction traffic; skip those candidates.
      if (s > 1 && tiles * (s - 1) >= int64_t(cus) * 4)
        break;
      const float t = timeKernel(idx, s, *bestTime, bIsNK);
      if (t < *bestTime) {
        *bestTime = t;
        *bestIdx = idx;
        *bestSplit = s;
      }
    }
  }
}

// mode 0: the reference's protocol (GemmProfiler.cu:143-235): the path
// nvteGemmF16 takes -- B as [N, K], library-selected kernel -- is timed first
// and is the baseline; the answer is -1 unless a manifest kernel on row-major B
// beats it (the compiler then emits nvteGemmF16 for that matmul,
// HOMNVGPUAutotunePass.cpp:90 + HOMNVGPUToFunc.cpp:125-134).
// mode 1 / 2: best manifest kernel for row-major / [N, K] B, no baseline.
std::tuple<int64_t, int32_t> GemmProfiler::run(int mode) {
  const auto key = std::make_tuple(M_, N_, K_, activation_ * 4 + mode);
  auto it = cache_.find(key);
  if (it != cache_.end()) {
    bestTimeMs_ = std::get<2>(it->second);
    fprintf(stderr, "Cache hit, Idx = %lld, split k factor = %d\n",
            (long long)std::get<0>(it->second), std::get<1>(it->second));
    return {std::get<0>(it->second), std::get<1>(it->second)};
  }
  if (!ensure(a_, M_ * K_) || !ensure(b_, K_ * N_) || !ensure(c_, M_ * N_))
    return {-1, 1};
  int64_t bestIdx = -1;
  int32_t bestSplit = 1;
  float bestTime = INFINITY, baseTime = INFINITY;
  if (mode == 0) {
    GemmProblem pr = problem(true);
    const int nvteIdx = chooseNvteKernel(&pr, activation_);
    if (nvteIdx >= 0)
      baseTime = bestTime = timeKernel(nvteIdx, pr.splitK, INFINITY, true);
  }
  sweep(mode == 2, &bestIdx, &bestSplit, &bestTime);
  bestTimeMs_ = bestTime;
  fprintf(stderr,
          "Profile for %lld %lld %lld act: %lld done. Best kernel %s, best "
          "split k factor %d, best time %g ms (%.1f TFLOP/s)",
          (long long)M_, (long long)N_, (long long)K_, (long long)activation_,
          bestIdx >= 0 ? gemmKernelInfo(int(bestIdx)).name
                       : (mode == 0 && baseTime < INFINITY ? "nvte" : "none"),
          bestSplit, double(bestTime),
          2.0 * double(M_) * double(N_) * double(K_) / (double(bestTime) * 1e9));
  if (mode == 0)
    fprintf(stderr, ", speedup compared to nvte %g", double(baseTime / bestTime));
  fprintf(stderr, ".\n");
  cache_[key] = std::make_tuple(bestIdx, bestSplit, bestTime);
  return {bestIdx, bestSplit};
}

std::tuple<int64_t, int32_t> GemmProfiler::profile() { return run(0); }

std::tuple<int64_t, int32_t> GemmProfiler::profile(int64_t M, int64_t N,
                                                   int64_t K,
                                                   int64_t activation,
                                                   float alpha, float beta) {
  M_ = M;
  N_ = N;
  K_ = K;
  activation_ = activation;
  alpha_ = alpha;
  beta_ = beta;
  return run(0);
}

std::tuple<int64_t, int32_t>
GemmProfiler::profileLayout(int64_t M, int64_t N, int64_t K, int64_t activation,
                            float alpha, float beta, bool bIsNK) {
  M_ = M;
  N_ = N;
  K_ = K;
  activation_ = activation;
  alpha_ = alpha;
  beta_ = beta;
  return run(bIsNK ? 2 : 1);
}

// ------------------------------------------------------------- layer norm --
template <typename T>
Status runLayernorm(int64_t rankA, void *dstA, float eps) {
  View<T> A(rankA, dstA);
  // LayernormRunner::construct_tensors (Layernorm.h:619-624)
  HOM_CHECK_RET((A.rank == 3 || A.rank == 2) && A.sizes,
                Status::kInvalidArgument,
                "layernorm: rank must be 2 or 3 (got %lld)", (long long)A.rank);
  HOM_CHECK_RET(A.contiguous(), Status::kInvalidArgument,
                "layernorm: tensor must be contiguous row-major");
  const int64_t rows = A.rank == 3 ? A.sizes[0] * A.sizes[1] : A.sizes[0];
  const int64_t hidden = A.rank == 3 ? A.sizes[2] : A.sizes[1];
  return launchLayernorm<T>(A.data, nullptr, nullptr, nullptr, A.data, rows,
                            hidden, eps, stream());
}
template Status runLayernorm<_Float16>(int64_t, void *, float);
template Status runLayernorm<float>(int64_t, void *, float);

Status runAddLayernormF16(int64_t rankX, void *dstX, int64_t rankRes,
                          void *dstRes, int64_t rankGamma, void *dstGamma,
                          int64_t rankBeta, void *dstBeta, int64_t rankOut,
                          void *dstOut, float eps) {
  View<_Float16> X(rankX, dstX), R(rankRes, dstRes), G(rankGamma, dstGamma),
      Bt(rankBeta, dstBeta), O(rankOut, dstOut);
  HOM_CHECK_RET((X.rank == 3 || X.rank == 2) && X.sizes && O.sizes &&
                    O.rank == X.rank,
                Status::kInvalidArgument,
                "add+layernorm: X and Out must both have rank 2 or 3");
  for (int64_t i = 0; i < X.rank; i++)
    HOM_CHECK_RET(X.sizes[i] == O.sizes[i], Status::kInvalidArgument,
                  "add+layernorm: Out shape differs from X in dim %lld",
                  (long long)i);
  HOM_CHECK_RET(X.contiguous() && O.contiguous(), Status::kInvalidArgument,
                "add+layernorm: X and Out must be contiguous");
  const int64_t rows = X.rank == 3 ? X.sizes[0] * X.sizes[1] : X.sizes[0];
  const int64_t hidden = X.rank == 3 ? X.sizes[2] : X.sizes[1];
  if (dstRes) {
    HOM_CHECK_RET(R.rank == X.rank && R.contiguous(), Status::kInvalidArgument,
                  "add+layernorm: Res must match X");
    for (int64_t i = 0; i < X.rank; i++)
      HOM_CHECK_RET(X.sizes[i] == R.sizes[i], Status::kInvalidArgument,
                    "add+layernorm: Res shape differs from X in dim %lld",
                    (long long)i);
  }
  if (dstGamma)
    HOM_CHECK_RET(G.numel() == hidden && G.contiguous(),
                  Status::kInvalidArgument,
                  "add+layernorm: Gamma must hold %lld values",
                  (long long)hidden);
  if (dstBeta)
    HOM_CHECK_RET(Bt.numel() == hidden && Bt.contiguous(),
                  Status::kInvalidArgument,
                  "add+layernorm: Beta must hold %lld values",
                  (long long)hidden);
  return launchLayernorm<_Float16>(X.data, dstRes ? R.data : nullptr,
                                   dstGamma ? G.data : nullptr,
                                   dstBeta ? Bt.data : nullptr, O.data, rows,
                                   hidden, eps, stream());
}

// --------------------------------------------------------------- attention --
Status runBertAttentionF16(int64_t rankA, void *dstA, int64_t rankSeqlen,
                           void *dstSeqlen, int64_t rankOut, void *dstOut,
                           float scale, int64_t headNum, int32_t packing,
                           const void *ahead, int64_t aheadBytes) {
  View<_Float16> A(rankA, dstA), Out(rankOut, dstOut);
  View<int32_t> Seq(rankSeqlen, dstSeqlen);
  // BertAttentionRunner::construct_tensors (BertAttentionRunner.h:61-73)
  HOM_CHECK_RET(A.rank == 3 && A.sizes, Status::kInvalidArgument,
                "attention: QKV must have rank 3 (got %lld)",
                (long long)A.rank);
  HOM_CHECK_RET(headNum > 0 && A.sizes[2] % (headNum * 3) == 0,
                Status::kInvalidArgument,
                "attention: last dim %lld is not a multiple of 3 * heads (%lld)",
                (long long)A.sizes[2], (long long)headNum);
  HOM_CHECK_RET(Out.rank == 3 && Out.sizes, Status::kInvalidArgument,
                "attention: Out must have rank 3");
  HOM_CHECK_RET(Out.sizes[0] == A.sizes[0] && Out.sizes[1] == A.sizes[1] &&
                    Out.sizes[2] * 3 == A.sizes[2],
                Status::kInvalidArgument,
                "attention: Out is [%lld,%lld,%lld] for QKV [%lld,%lld,%lld]",
                (long long)Out.sizes[0], (long long)Out.sizes[1],
                (long long)Out.sizes[2], (long long)A.sizes[0],
                (long long)A.sizes[1], (long long)A.sizes[2]);
  const int64_t bs = A.sizes[0], seq = A.sizes[1];
  const int64_t headDim = A.sizes[2] / headNum / 3;
  HOM_CHECK_RET(Seq.rank == 1 && Seq.sizes && Seq.sizes[0] == bs + 1,
                Status::kInvalidArgument,
                "attention: cu_seqlens must be int32[%lld]", (long long)bs + 1);
  HOM_CHECK_RET(A.contiguous() && Out.contiguous(), Status::kInvalidArgument,
                "attention: tensors must be contiguous");
  HOM_CHECK_RET((reinterpret_cast<uintptr_t>(ahead) & 15) == 0,
                Status::kInvalidArgument, "attention: misaligned memory to read ahead");
  HOM_CHECK_RET(aheadBytes >= 0, Status::kInvalidArgument,
                "attention: aheadBytes must not be negative (%lld)", (long long)aheadBytes);
  return launchBertAttentionF16(A.data, Seq.data, Out.data, bs, seq, headNum,
                                headDim, scale, stream(),
                                (packing & HOM_PACKED_D) != 0,
                                (packing & HOM_PACKED_A) != 0, ahead, ahead ? aheadBytes & ~int64_t(15) : 0);
}

// ------------------------------------------------------------- elementwise --
template <typename T>
Status runElementwise(BinOp op, int64_t rankA, void *dstA, int64_t rankB,
                      void *dstB, int64_t rankOut, void *dstOut) {
  View<T> A(rankA, dstA), B(rankB, dstB), Out(rankOut, dstOut);
  // ElementwiseRunner::run (ElementwiseRunner.h:132-138)
  HOM_CHECK_RET(A.rank == B.rank && A.rank == Out.rank,
                Status::kInvalidArgument,
                "elementwise: ranks differ (%lld, %lld, %lld)",
                (long long)A.rank, (long long)B.rank, (long long)Out.rank);
  HOM_CHECK_RET(A.rank >= 0 && A.rank <= kMaxRank, Status::kInvalidArgument,
                "elementwise: rank %lld not supported (max %d)",
                (long long)A.rank, kMaxRank);
  HOM_CHECK_RET(A.rank == 0 || (A.sizes && B.sizes && Out.sizes),
                Status::kInvalidArgument, "elementwise: null descriptor");
  BroadcastDesc d{};
  d.rank = int(A.rank);
  for (int64_t i = 0; i < A.rank; i++) {
    HOM_CHECK_RET(A.sizes[i] == B.sizes[i] || B.sizes[i] == 1,
                  Status::kInvalidArgument,
                  "elementwise: only B can broadcast (dim %lld: A %lld, B %lld)",
                  (long long)i, (long long)A.sizes[i], (long long)B.sizes[i]);
    HOM_CHECK_RET(A.sizes[i] == Out.sizes[i], Status::kInvalidArgument,
                  "elementwise: Out differs from A in dim %lld", (long long)i);
  }
  HOM_CHECK_RET(A.contiguous() && Out.contiguous(), Status::kInvalidArgument,
                "elementwise: A and Out must be contiguous row-major");
  int64_t stride = 1;
  for (int64_t i = A.rank - 1; i >= 0; i--) {
    d.outSize[i] = A.sizes[i];
    d.outStride[i] = stride;
    stride *= A.sizes[i];
    d.bSize[i] = B.sizes[i];
    d.bStride[i] = B.sizes[i] == 1 ? 0 : B.strides[i];
  }
  return launchElementwise<T>(op, A.data, B.data, Out.data, A.numel(), d,
                              stream());
}
template Status runElementwise<_Float16>(BinOp, int64_t, void *, int64_t,
                                         void *, int64_t, void *);
template Status runElementwise<float>(BinOp, int64_t, void *, int64_t, void *,
                                      int64_t, void *);

template <typename T>
Status runGather(int64_t rankIdx, void *desIdx, int64_t rankValue,
                 void *desValue, int64_t rankOut, void *desOut) {
  View<int64_t> I(rankIdx, desIdx);
  View<T> V(rankValue, desValue), O(rankOut, desOut);
  // GatherRunner::run (GatherRunner.h:52-60)
  HOM_CHECK_RET(V.rank == 3 && V.sizes && V.sizes[0] == 1,
                Status::kInvalidArgument,
                "gather: value must be [1, V, H] (rank %lld)",
                (long long)V.rank);
  HOM_CHECK_RET(I.rank == 2 && I.sizes && O.sizes && O.rank == 3,
                Status::kInvalidArgument,
                "gather: indices must have rank 2 and out rank 3");
  HOM_CHECK_RET(O.sizes[2] == V.sizes[2] && I.sizes[0] == O.sizes[0] &&
                    I.sizes[1] == O.sizes[1],
                Status::kInvalidArgument, "gather: shape mismatch");
  HOM_CHECK_RET(I.contiguous() && V.contiguous() && O.contiguous(),
                Status::kInvalidArgument, "gather: tensors must be contiguous");
  return launchGather<T>(I.data, V.data, O.data, I.sizes[0] * I.sizes[1],
                         V.sizes[1], V.sizes[2], stream());
}
template Status runGather<_Float16>(int64_t, void *, int64_t, void *, int64_t,
                                    void *);
template Status runGather<float>(int64_t, void *, int64_t, void *, int64_t,
                                 void *);

template <typename InT>
Status runCuSeqLen(int64_t rankIn, void *desIn, int64_t rankOut, void *desOut) {
  View<InT> In(rankIn, desIn);
  View<int32_t> Out(rankOut, desOut);
  // CuSeqLenRunner::run (CuSeqLen.h:55-57)
  HOM_CHECK_RET(In.rank == 2 && In.sizes, Status::kInvalidArgument,
                "cu_seqlens: mask must have rank 2 (got %lld)",
                (long long)In.rank);
  HOM_CHECK_RET(Out.rank == 1 && Out.sizes, Status::kInvalidArgument,
                "cu_seqlens: out must have rank 1");
  HOM_CHECK_RET(In.sizes[0] + 1 == Out.sizes[0], Status::kInvalidArgument,
                "cu_seqlens: out has %lld entries, expected %lld",
                (long long)Out.sizes[0], (long long)In.sizes[0] + 1);
  HOM_CHECK_RET(In.contiguous(), Status::kInvalidArgument,
                "cu_seqlens: mask must be contiguous");
  return launchCuSeqLen<InT>(In.data, Out.data, In.sizes[0], In.sizes[1],
                             stream());
}
template Status runCuSeqLen<int64_t>(int64_t, void *, int64_t, void *);
template Status runCuSeqLen<int32_t>(int64_t, void *, int64_t, void *);

Status runEmbed(int64_t rankIds, void *desIds, int64_t rankMask, void *desMask,
                int64_t rankWord, void *desWord, int64_t rankPos, void *desPos,
                int64_t rankOut, void *desOut, int64_t rankCu, void *desCu,
                float eps, int32_t packing) {
  View<int64_t> I(rankIds, desIds), Mk(rankMask, desMask);
  View<_Float16> W(rankWord, desWord), P(rankPos, desPos), O(rankOut, desOut);
  View<int32_t> Cu(rankCu, desCu);
  HOM_CHECK_RET(I.rank == 2 && Mk.rank == 2 && I.sizes && Mk.sizes &&
                    I.sizes[0] == Mk.sizes[0] && I.sizes[1] == Mk.sizes[1],
                Status::kInvalidArgument,
                "embed: ids and mask must be [b, s] tensors of one shape");
  const int64_t bs = I.sizes[0], seq = I.sizes[1];
  HOM_CHECK_RET(W.rank == 3 && W.sizes && W.sizes[0] == 1 && P.rank == 3 &&
                    P.sizes && P.sizes[0] == 1 && P.sizes[1] == seq &&
                    P.sizes[2] == W.sizes[2],
                Status::kInvalidArgument,
                "embed: word must be [1, V, H] and positions [1, s, H]");
  const int64_t vocab = W.sizes[1], hidden = W.sizes[2];
  HOM_CHECK_RET(O.rank == 3 && O.sizes && O.sizes[0] == bs &&
                    O.sizes[1] == seq && O.sizes[2] == hidden,
                Status::kInvalidArgument, "embed: out must be [b, s, H]");
  HOM_CHECK_RET(Cu.rank == 1 && Cu.sizes && Cu.sizes[0] == bs + 1,
                Status::kInvalidArgument, "embed: cu_seqlens must be int32[%lld]",
                (long long)bs + 1);
  HOM_CHECK_RET(I.contiguous() && Mk.contiguous() && W.contiguous() &&
                    P.contiguous() && O.contiguous(),
                Status::kInvalidArgument, "embed: tensors must be contiguous");
  const bool packedOut = (packing & HOM_PACKED_D) != 0;
  HOM_CHECK_RET(!packedOut || hidden % 32 == 0, Status::kInvalidArgument,
                "embed: fragment order needs H a multiple of 32");
  if (embedFits(W.data, P.data, O.data, bs, seq, hidden, vocab))
    return launchEmbed(I.data, Mk.data, W.data, P.data, O.data, Cu.data, bs, seq,
                       hidden, vocab, eps, packedOut, stream());
  HOM_CHECK_RET(!packedOut, Status::kInvalidArgument,
                "embed: fragment order needs H of at most 2048");
  // rows off the vector width or beyond a wavefront's registers: step by step
  Status st = launchCuSeqLen<int64_t>(Mk.data, Cu.data, bs, seq, stream());
  if (st == Status::kSuccess)
    st = launchGather<_Float16>(I.data, W.data, O.data, bs * seq, vocab, hidden,
                                stream());
  BroadcastDesc d{};
  d.rank = 3;
  const int64_t size[3] = {bs, seq, hidden};
  for (int i = 2; i >= 0; i--) {
    d.outSize[i] = size[i];
    d.outStride[i] = i == 2 ? 1 : d.outStride[i + 1] * size[i + 1];
    d.bSize[i] = i == 0 ? 1 : size[i];
    d.bStride[i] = d.bSize[i] == 1 ? 0 : P.strides[i];
  }
  if (st == Status::kSuccess)
    st = launchElementwise<_Float16>(BinOp::kAdd, O.data, P.data, O.data,
                                     bs * seq * hidden, d, stream());
  if (st == Status::kSuccess)
    st = launchLayernorm<_Float16>(O.data, nullptr, nullptr, nullptr, O.data,
                                   bs * seq, hidden, eps, stream());
  return st;
}

Status runGeluF16(int64_t rankA, void *dstA, int64_t rankOut, void *dstOut,
                  int32_t form) {
  View<_Float16> A(rankA, dstA), O(rankOut, dstOut);
  HOM_CHECK_RET(A.sizes && O.sizes && A.rank == O.rank,
                Status::kInvalidArgument, "gelu: rank mismatch");
  HOM_CHECK_RET(A.numel() == O.numel() && A.contiguous() && O.contiguous(),
                Status::kInvalidArgument,
                "gelu: tensors must be contiguous and equally sized");
  HOM_CHECK_RET(form == 0 || form == 1, Status::kInvalidArgument,
                "gelu: form must be 0 (erf) or 1 (tanh)");
  return launchGeluF16(A.data, O.data, A.numel(), form, stream());
}

// ------------------------------------------------------------------ memory --
C_UnrankedMemRefType allocDevice(const std::vector<int64_t> &sizes,
                                 size_t elemBytes) {
  C_UnrankedMemRefType res{int64_t(sizes.size()), nullptr};
  const size_t rank = sizes.size();
  int64_t total = 1;
  for (int64_t s : sizes) {
    HOM_CHECK_RET(s >= 0, res, "alloc: negative extent %lld", (long long)s);
    total *= s;
  }
  const size_t descBytes = sizeof(HomMemRefHeader) + 2 * rank * sizeof(int64_t);
  void *desc = malloc(descBytes);
  HOM_CHECK_RET(desc != nullptr, res, "alloc: out of host memory");
  void *dev = nullptr;
  if (total > 0) {
    hipError_t e = hipMalloc(&dev, size_t(total) * elemBytes);
    if (e != hipSuccess) {
      free(desc);
      recordError(__FILE__, __LINE__, "alloc: hipMalloc of %zu bytes failed: %s",
                  size_t(total) * elemBytes, hipGetErrorString(e));
      return res;
    }
  }
  auto *h = static_cast<HomMemRefHeader *>(desc);
  h->basePtr = dev;
  h->data = dev;
  h->offset = 0;
  int64_t *sz = hom_memref_sizes(desc);
  int64_t *st = hom_memref_strides(desc, int64_t(rank));
  int64_t stride = 1;
  for (size_t i = 0; i < rank; i++) {
    sz[i] = sizes[i];
    st[rank - i - 1] = stride;
    stride *= sizes[rank - i - 1];
  }
  res.descriptor = desc;
  return res;
}

// Text format written by the reference's weight serialiser
// (lib/WeightsEngine/WeightsEngine.cpp:22-39) and read back by
// Binary constant file "<idx>.bin": the 40-byte little-endian header below
// (magic "HOMW", version 1, bytes per element: 2 = fp16 or 4 = fp32, rank 3, the
// three extents), then the values, row-major.  Values of the constant's own
// type are uploaded as they are; the other type is converted (fp32 -> fp16
// rounds to nearest even, like the text path).
struct ConstantHeader {
  char magic[4];
  uint32_t version;
  uint32_t elementBytes;
  uint32_t rank;
  int64_t extents[3];
};
static_assert(sizeof(ConstantHeader) == 40, "constant file header layout");

template <typename T>
bool loadBinaryConstant(const std::string &path, int32_t idx,
                        C_UnrankedMemRefType *res, bool *failed) {
  FILE *f = fopen(path.c_str(), "rb");
  if (!f)
    return false; // no binary file: the caller falls back to the text format
  *failed = true;
  ConstantHeader h{};
  const bool headOk = fread(&h, sizeof(h), 1, f) == 1 &&
                      memcmp(h.magic, "HOMW", 4) == 0 && h.version == 1 &&
                      h.rank == 3 && (h.elementBytes == 2 || h.elementBytes == 4);
  if (!headOk) {
    fclose(f);
    recordError(__FILE__, __LINE__, "constant %d: %s is not a HOMW v1 rank-3 file",
                idx, path.c_str());
    return true;
  }
  const int64_t total = h.extents[0] * h.extents[1] * h.extents[2];
  if (h.extents[0] < 0 || h.extents[1] < 0 || h.extents[2] < 0) {
    fclose(f);
    recordError(__FILE__, __LINE__, "constant %d: negative extent in %s", idx,
                path.c_str());
    return true;
  }
  std::vector<unsigned char> raw(size_t(total) * h.elementBytes);
  const size_t got = total ? fread(raw.data(), h.elementBytes, size_t(total), f) : 0;
  fclose(f);
  if (int64_t(got) != total) {
    recordError(__FILE__, __LINE__,
                "constant %d: %s holds %lld values, expected %lld", idx,
                path.c_str(), (long long)got, (long long)total);
    return true;
  }
  std::vector<T> conv;
  const void *src = raw.data();
  if (h.elementBytes != sizeof(T)) {
    conv.resize(size_t(total));
    for (int64_t i = 0; i < total; i++) {
      if (h.elementBytes == 4) {
        float v;
        memcpy(&v, raw.data() + size_t(i) * 4, 4);
        conv[size_t(i)] = T(v);
      } else {
        _Float16 v;
        memcpy(&v, raw.data() + size_t(i) * 2, 2);
        conv[size_t(i)] = T(v);
      }
    }
    src = conv.data();
  }
  *res = allocDevice({h.extents[0], h.extents[1], h.extents[2]}, sizeof(T));
  if (!res->descriptor)
    return true;
  if (total > 0) {
    hipError_t e = hipMemcpy(hom_memref_data(res->descriptor), src,
                             size_t(total) * sizeof(T), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
      recordError(__FILE__, __LINE__, "constant %d: upload failed: %s", idx,
                  hipGetErrorString(e));
      return true;
    }
  }
  *failed = false;
  return true;
}

// allocConstantNVGPU* (HandsOnNVGPURunnerUtils.cu:224-298): "<idx>.txt" holds
// the three extents on the first line, then the values as decimal text.  A
// "<idx>.bin" beside it (or instead of it) is preferred: parsing 110 M decimal
// weights takes minutes, reading them takes milliseconds.
template <typename T> C_UnrankedMemRefType allocConstant(int32_t idx) {
  C_UnrankedMemRefType res{3, nullptr};
  const char *dir = getenv("HOM_CONSTANT_DIR");
  const std::string stem =
      std::string(dir ? dir : ".") + "/" + std::to_string(idx);
  bool failed = false;
  if (loadBinaryConstant<T>(stem + ".bin", idx, &res, &failed))
    return res;
  std::string path = stem + ".txt";
  FILE *f = fopen(path.c_str(), "rb");
  HOM_CHECK_RET(f != nullptr, res, "constant %d: cannot open %s (%s)", idx,
                path.c_str(), strerror(errno));
  std::string text;
  {
    char buf[1 << 16];
    size_t n;
    while ((n = fread(buf, 1, sizeof(buf), f)) > 0)
      text.append(buf, n);
    fclose(f);
  }
  const size_t eol = text.find('\n');
  std::vector<int64_t> dims;
  {
    std::stringstream ss(text.substr(0, eol));
    int64_t v;
    while (ss >> v)
      dims.push_back(v);
  }
  HOM_CHECK_RET(dims.size() == 3, res,
                "constant %d: header of %s has %zu extents, expected 3", idx,
                path.c_str(), dims.size());
  int64_t total = dims[0] * dims[1] * dims[2];
  std::vector<T> host;
  host.resize(size_t(total));
  const char *p = eol == std::string::npos ? text.c_str() + text.size()
                                           : text.c_str() + eol + 1;
  for (int64_t i = 0; i < total; i++) {
    char *end = nullptr;
    const float v = strtof(p, &end);
    HOM_CHECK_RET(end != p, res,
                  "constant %d: %s holds %lld values, expected %lld", idx,
                  path.c_str(), (long long)i, (long long)total);
    host[size_t(i)] = T(v); // float -> half rounds to nearest even
    p = end;
  }
  res = allocDevice(dims, sizeof(T));
  if (!res.descriptor)
    return res;
  if (total > 0) {
    hipError_t e = hipMemcpy(hom_memref_data(res.descriptor), host.data(),
                             size_t(total) * sizeof(T), hipMemcpyHostToDevice);
    if (e != hipSuccess)
      recordError(__FILE__, __LINE__, "constant %d: upload failed: %s", idx,
                  hipGetErrorString(e));
  }
  return res;
}
template C_UnrankedMemRefType allocConstant<_Float16>(int32_t);
template C_UnrankedMemRefType allocConstant<float>(int32_t);

} // namespace hom

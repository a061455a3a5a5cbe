// Layer norm over the last dimension for gfx950.
//
// Semantics follow the reference's LayernormRunner (include/NVGPUKernels/
// Layernorm.h:584-694): statistics in fp32, biased variance, y = (x - mean) *
// rsqrt(var + eps); the reference form has no affine parameters and runs in
// place.  The optional residual / gamma / beta operands are a superset.
//
// The kernel is bandwidth bound: each row is read once with 128-bit loads and
// stays in registers for the two statistic passes; one 64-lane wavefront owns
// a row and reduces across lanes inside the vector ALU (no LDS); rows beyond
// 2048 fp16 values take the four wavefronts of a workgroup.
#include "cross_lane.h"
#include "kernels.h"
#include "store_policy.h"

namespace hom {
namespace {

constexpr int kWave = 64;

template <typename T> struct Vec16;
template <> struct Vec16<_Float16> {
  static constexpr int kN = 8;
  typedef _Float16 type __attribute__((ext_vector_type(8)));
};
template <> struct Vec16<float> {
  static constexpr int kN = 4;
  typedef float type __attribute__((ext_vector_type(4)));
};

// WPR wavefronts per row (1, or the 4 of a workgroup for long rows); VPL
// 16-byte vectors per lane.
//
// STREAM == false: tensors of a few megabytes, which the next kernel of the
// stream finds in the last-level cache (results written through, see
// store_policy.h).  STREAM == true: tensors beyond that cache; rows are read
// and written with the non-temporal hint, because nothing is touched twice and
// without the hint the written rows linger in the L2s and compete with the
// reads on their way out (16384 x 1024 in place, rotating over 800 MB so that
// every launch is cold: 4.5 TB/s with default accesses, 5.4 TB/s with the hint,
// 5.6 TB/s with the in-place form's stores also written through; a plain
// read-modify-write probe shows the same 4.65 -> 5.55 -> 5.72 TB/s.  With a
// residual operand, two read streams and a write stream, writing through costs
// 1 % instead: 17.4 against 17.5 us).
//
// The kernel is a chain of memory round trips (arguments, row, result) a few
// hundred nanoseconds each, so everything it will read is requested at once and
// nothing stands between the requests: a lane without a vector of its own
// (768 columns: lanes 32..63 of the second vector) and a wavefront past the
// last row load a valid address again and mask the values, instead of a branch
// around the load, which would make the second request wait for the first.
//
// Rows of any length and alignment: the hardware's 16-byte accesses take any
// element boundary, and the elements behind the last whole vector (TAIL:
// hidden % N of them) travel one per lane.  (Rows off the vector width used to
// take a workgroup-per-row kernel with scalar accesses and three passes over
// memory: 4096 x 1001 fp16 11.7 us, now 4.0, what 4096 x 1000 takes; 2000 x 6280
// with a residual 65 us, now 17.)
template <typename T, int WPR, int VPL, bool HAS_RES, bool HAS_AFFINE,
          bool STREAM, bool TAIL>
__global__ __launch_bounds__(256) void layernormRowKernel(
    const T *x, const T *res,
    const T *__restrict__ gamma, const T *__restrict__ beta, T *out,
    int64_t rows, int hidden, float eps) {
  using V = typename Vec16<T>::type;
  typedef V VAny __attribute__((aligned(sizeof(T))));
  constexpr int N = Vec16<T>::kN;
  constexpr int kRowsPerBlock = 256 / (kWave * WPR);
  constexpr int kLanes = kWave * WPR; // lanes of a row
  const int lane = threadIdx.x & (kLanes - 1);
  // the same for every lane of a wavefront: row addresses stay scalar
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
  const int64_t rowWant = int64_t(blockIdx.x) * kRowsPerBlock + group;
  const bool rowOk = rowWant < rows;
  const int64_t row = rowOk ? rowWant : rows - 1;
  const int nvec = hidden / N;
  const T *xr = x + row * hidden;
  const T *rr = HAS_RES ? res + row * hidden : nullptr;
  auto vec = [](const T *p, int at) {
    const VAny *q = reinterpret_cast<const VAny *>(p) + at;
    return V(STREAM ? __builtin_nontemporal_load(q) : *q);
  };

  V raw[VPL];
  V rawRes[VPL];
  V g[VPL], b[VPL];
  const bool hasG = HAS_AFFINE && gamma != nullptr;
  const bool hasB = HAS_AFFINE && beta != nullptr;
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    const int idx = lane + i * kLanes;
    const int at = idx < nvec ? idx : 0;
    raw[i] = vec(xr, at);
    if (HAS_RES)
      rawRes[i] = vec(rr, at);
    if (HAS_AFFINE) {
      // (null gamma / beta: wave-uniform branches, taken by nobody or everybody)
      if (hasG)
        g[i] = *(reinterpret_cast<const VAny *>(gamma) + at);
      if (hasB)
        b[i] = *(reinterpret_cast<const VAny *>(beta) + at);
    }
  }
  // the tail: element nvec * N + lane of the row
  const int tailAt = nvec * N + lane;
  const bool tailMine = TAIL && tailAt < hidden;
  T tRaw = T(0), tRes = T(0), tG = T(1), tB = T(0);
  if constexpr (TAIL) {
    const int at = tailMine ? tailAt : 0;
    tRaw = xr[at];
    if (HAS_RES)
      tRes = rr[at];
    if (HAS_AFFINE) {
      if (hasG)
        tG = gamma[at];
      if (hasB)
        tB = beta[at];
    }
  }
  // every request is out before the first value is touched
  __builtin_amdgcn_sched_barrier(0);
  // (the partial sums of a row's wavefronts meet in LDS)
  __shared__ float part[WPR > 1 ? 2 : 1][WPR > 1 ? WPR : 1];
  auto rowTotal = [&](float v, int which) {
    v = waveSum(v);
    if constexpr (WPR > 1) {
      if (lane % kWave == 0)
        part[which][lane / kWave] = v;
      __syncthreads();
      v = 0.f;
#pragma unroll
      for (int w = 0; w < WPR; w++)
        v += part[which][w];
    }
    return v;
  };
  float v[VPL][N];
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    const bool mine = lane + i * kLanes < nvec;
#pragma unroll
    for (int j = 0; j < N; j++) {
      float f = float(raw[i][j]);
      if (HAS_RES)
        f += float(rawRes[i][j]); // the sum stays in fp32
      f = mine ? f : 0.f;
      v[i][j] = f;
      sum += f;
    }
  }
  float vt = 0.f;
  if constexpr (TAIL) {
    vt = float(tRaw) + (HAS_RES ? float(tRes) : 0.f);
    sum += tailMine ? vt : 0.f;
  }
  const float invH = 1.0f / float(hidden);
  const float mean = rowTotal(sum, 0) * invH;
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    const bool mine = lane + i * kLanes < nvec;
#pragma unroll
    for (int j = 0; j < N; j++) {
      const float d = mine ? v[i][j] - mean : 0.f;
      sq += d * d;
    }
  }
  if constexpr (TAIL) {
    const float d = tailMine ? vt - mean : 0.f;
    sq += d * d;
  }
  const float var = rowTotal(sq, WPR > 1 ? 1 : 0) * invH;
  const float rstd = 1.0f / sqrtf(var + eps);

  T *orow = out + row * hidden;
#pragma unroll
  for (int i = 0; i < VPL; i++) {
    const int idx = lane + i * kLanes;
    V o;
#pragma unroll
    for (int j = 0; j < N; j++) {
      float y = (v[i][j] - mean) * rstd;
      if (hasG)
        y *= float(g[i][j]);
      if (hasB)
        y += float(b[i][j]);
      o[j] = T(y);
    }
    VAny *at = reinterpret_cast<VAny *>(orow) + idx;
    if (rowOk && idx < nvec) {
      if (STREAM && !HAS_RES)
        storeStreaming(at, o); // the in-place form: see store_policy.h
      else if (STREAM)
        __builtin_nontemporal_store(o, at);
      else
        storeWriteThrough(at, o);
    }
  }
  if constexpr (TAIL) {
    float y = (vt - mean) * rstd;
    if (hasG)
      y *= float(tG);
    if (hasB)
      y += float(tB);
    if (rowOk && tailMine)
      orow[tailAt] = T(y);
  }
}

__device__ __forceinline__ float blockSum(float v, float *lds) {
  v = waveSum(v);
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int nwaves = blockDim.x / kWave;
  __syncthreads(); // lds may still be read from a previous reduction
  if (lane == 0)
    lds[wave] = v;
  __syncthreads();
  float total = 0.f;
  for (int i = 0; i < nwaves; i++)
    total += lds[i];
  return total;
}

// One workgroup per row, for rows beyond the registers of the kernel above
// (16384 fp16 / 8192 fp32 values): scalar accesses, the row is read three times.
template <typename T>
__global__ __launch_bounds__(256) void layernormBlockKernel(
    const T *x, const T *res,
    const T *__restrict__ gamma, const T *__restrict__ beta, T *out,
    int64_t rows, int64_t hidden, float eps) {
  __shared__ float lds[8];
  const int64_t row = blockIdx.x;
  const T *xr = x + row * hidden;
  const T *rr = res ? res + row * hidden : nullptr;
  T *orow = out + row * hidden;
  auto load = [&](int64_t i) -> float {
    float f = float(xr[i]);
    if (rr)
      f += float(rr[i]);
    return f;
  };
  float sum = 0.f;
  for (int64_t i = threadIdx.x; i < hidden; i += blockDim.x)
    sum += load(i);
  const float mean = blockSum(sum, lds) / float(hidden);
  float sq = 0.f;
  for (int64_t i = threadIdx.x; i < hidden; i += blockDim.x) {
    const float d = load(i) - mean;
    sq += d * d;
  }
  const float var = blockSum(sq, lds) / float(hidden);
  const float rstd = 1.0f / sqrtf(var + eps);
  // All reads of this row are done (blockSum synchronised) before any write,
  // so out may alias x.
  for (int64_t i = threadIdx.x; i < hidden; i += blockDim.x) {
    float y = (load(i) - mean) * rstd;
    if (gamma)
      y *= float(gamma[i]);
    if (beta)
      y += float(beta[i]);
    orow[i] = T(y);
  }
}

// Results that the next kernel of the stream will find in the last-level cache
// (a few megabytes) are written through; larger tensors stream.
constexpr int64_t kSmallTensorBytes = int64_t(16) << 20;

template <typename T, int WPR, int VPL, bool STREAM, bool TAIL>
void launchRowVariant(const T *x, const T *res, const T *gamma, const T *beta,
                      T *out, int64_t rows, int hidden, float eps,
                      hipStream_t s) {
  constexpr int kRowsPerBlock = 256 / (kWave * WPR);
  const dim3 grid((unsigned)((rows + kRowsPerBlock - 1) / kRowsPerBlock)),
      block(256);
  // (the fp32 entry point is the in-place form only)
  if constexpr (sizeof(T) == 2) {
    const bool affine = gamma || beta;
    if (res && affine) {
      layernormRowKernel<T, WPR, VPL, true, true, STREAM, TAIL>
          <<<grid, block, 0, s>>>(x, res, gamma, beta, out, rows, hidden, eps);
      return;
    }
    if (res) {
      layernormRowKernel<T, WPR, VPL, true, false, STREAM, TAIL>
          <<<grid, block, 0, s>>>(x, res, gamma, beta, out, rows, hidden, eps);
      return;
    }
    if (affine) {
      layernormRowKernel<T, WPR, VPL, false, true, STREAM, TAIL>
          <<<grid, block, 0, s>>>(x, res, gamma, beta, out, rows, hidden, eps);
      return;
    }
  }
  layernormRowKernel<T, WPR, VPL, false, false, STREAM, TAIL>
      <<<grid, block, 0, s>>>(x, res, gamma, beta, out, rows, hidden, eps);
}

template <typename T, int WPR, int VPL>
void launchRow(const T *x, const T *res, const T *gamma, const T *beta, T *out,
               int64_t rows, int hidden, float eps, hipStream_t s) {
  const bool stream = rows * hidden * int64_t(sizeof(T)) > kSmallTensorBytes;
  const bool tail = hidden % Vec16<T>::kN != 0;
  // (streaming: a persistent variant whose wavefronts keep their next row in
  // flight while they reduce and store the current one measured the same
  // 12.3-12.6 us on 16384 x 1024 cold, at 2 to 8 workgroups per CU: the rate is
  // the memory system's for a read-modify-write stream of this size)
  if (stream && tail)
    launchRowVariant<T, WPR, VPL, true, true>(x, res, gamma, beta, out, rows, hidden, eps, s);
  else if (stream)
    launchRowVariant<T, WPR, VPL, true, false>(x, res, gamma, beta, out, rows, hidden, eps, s);
  else if (tail)
    launchRowVariant<T, WPR, VPL, false, true>(x, res, gamma, beta, out, rows, hidden, eps, s);
  else
    launchRowVariant<T, WPR, VPL, false, false>(x, res, gamma, beta, out, rows, hidden, eps, s);
}

} // namespace

template <typename T>
Status launchLayernorm(const T *x, const T *res, const T *gamma, const T *beta,
                       T *out, int64_t rows, int64_t hidden, float eps,
                       hipStream_t s) {
  if (rows == 0 || hidden == 0)
    return Status::kSuccess;
  HOM_CHECK_RET(rows < (int64_t(1) << 31), Status::kInvalidArgument,
                "layernorm: too many rows (%lld)", (long long)rows);
  const int64_t nvec = hidden / Vec16<T>::kN;
  HOM_CHECK_RET(sizeof(T) == 2 || (!res && !gamma && !beta),
                Status::kInvalidArgument,
                "layernorm: residual and affine operands are fp16 only");
  // One wavefront per row up to 4 vectors per lane (2048 fp16 values), beyond
  // that the workgroup's four: a lane's 8 vectors and more cost registers and
  // leave too few wavefronts in flight.  Rows shorter than a vector have only
  // the tail.
  if (nvec <= kWave * 32) {
    const int h = int(hidden);
    if (nvec >= 1 && nvec <= kWave)
      launchRow<T, 1, 1>(x, res, gamma, beta, out, rows, h, eps, s);
    else if (nvec >= 1 && nvec <= kWave * 2)
      launchRow<T, 1, 2>(x, res, gamma, beta, out, rows, h, eps, s);
    else if (nvec >= 1 && nvec <= kWave * 4)
      launchRow<T, 1, 4>(x, res, gamma, beta, out, rows, h, eps, s);
    else if (nvec >= 1 && nvec <= kWave * 8)
      launchRow<T, 4, 2>(x, res, gamma, beta, out, rows, h, eps, s);
    else if (nvec >= 1 && nvec <= kWave * 16)
      launchRow<T, 4, 4>(x, res, gamma, beta, out, rows, h, eps, s);
    else if (nvec >= 1)
      launchRow<T, 4, 8>(x, res, gamma, beta, out, rows, h, eps, s);
    else
      layernormBlockKernel<T><<<dim3((unsigned)rows), dim3(256), 0, s>>>(
          x, res, gamma, beta, out, rows, hidden, eps);
  } else {
    layernormBlockKernel<T><<<dim3((unsigned)rows), dim3(256), 0, s>>>(
        x, res, gamma, beta, out, rows, hidden, eps);
  }
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}

template Status launchLayernorm<_Float16>(const _Float16 *, const _Float16 *,
                                          const _Float16 *, const _Float16 *,
                                          _Float16 *, int64_t, int64_t, float,
                                          hipStream_t);
template Status launchLayernorm<float>(const float *, const float *,
                                       const float *, const float *, float *,
                                       int64_t, int64_t, float, hipStream_t);

} // namespace hom

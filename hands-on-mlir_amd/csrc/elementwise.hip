// Bandwidth-bound helper kernels for gfx950: broadcasting binary elementwise
// ops, embedding gather, cu_seqlens, GELU, and the row-statistic kernels of the
// LN-GEMM pair.  All use 128-bit accesses where shape and alignment allow.
//
// Reference semantics:
//   elementwise  include/NVGPUKernels/ElementwiseRunner.h:69-153
//   gather       include/NVGPUKernels/GatherRunner.h:32-77
//   cu_seqlens   include/NVGPUKernels/CuSeqLen.h:28-74
//   row stats    include/NVGPUKernels/Layernorm.h:33-195 (ApplyFinalReduction)
#include "cross_lane.h"
#include "fast_div.h"
#include "kernels.h"
#include "mask_sums.h"
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

inline bool aligned16(const void *p) {
  return (reinterpret_cast<uintptr_t>(p) & 15) == 0;
}

template <typename T> __device__ __forceinline__ T applyOp(int op, T a, T b) {
  switch (op) {
  case 0:
    return a + b;
  case 1:
    return a - b;
  case 2:
    return a * b;
  default:
    // fp16 division goes through fp32 (correctly rounded there, then rounded
    // to fp16), like a half division on the reference's hardware.
    return T(float(a) / float(b));
  }
}

// Tensors up to this size are written through (the next kernel of the stream
// finds them in the last-level cache and nothing dirty is left to write back
// in between); larger ones stream with the non-temporal hint.
constexpr int64_t kStreamingBytes = int64_t(16) << 20;

template <typename V, bool STREAM>
__device__ __forceinline__ void storeResult(V *p, const V &v) {
  if (STREAM)
    __builtin_nontemporal_store(v, p);
  else
    storeWriteThrough(p, v);
}

// How B is laid over A's elements once neighbouring dimensions that behave the
// same are merged: rows of `inner` elements of A, and row r of A meets row
//   (r / rowDiv) % rowMod
// of B, which is `inner` contiguous values (kRowOfB) or one value (!kRowOfB).
//   same shape         one row                     rowDiv 1, rowMod 1
//   [1, .., 1, n]      the same row every time     rowDiv 1, rowMod 1
//   [b, 1, n]          one row per rowDiv rows     rowDiv s, rowMod b
//   [b, s, 1]          one value per row           rowDiv 1, rowMod b*s
//   [1, s, 1]          values repeat every s rows  rowDiv 1, rowMod s
struct RowBroadcast {
  uint32_t inner, rowDiv, rowMod;
  uint32_t innerMagic, divMagic, modMagic; // see fast_div.h
  bool rowOfB;
};

// One 16-byte vector of the output per thread: every access of the launch is
// in flight at once and nothing is recomputed, so the kernel runs at the
// memory system's rate (16 x 200 x 768 fp32 times a [16, 200, 1] mask: 13.0 us
// with the generic index walk below, which pays a 64-bit division per
// dimension and element, 4.2 us this way).  Rows need not be whole vectors: a
// vector that crosses a row end (WHOLE false: inner not a multiple of the
// vector width) looks up B per element.
template <typename T, int OP, bool ROW_OF_B, bool WHOLE, bool STREAM>
__global__ __launch_bounds__(256) void elementwiseRowKernel(
    const T *a, const T *b, T *out, uint32_t total, RowBroadcast m) {
  using V = typename Vec16<T>::type;
  constexpr int N = Vec16<T>::kN;
  const uint32_t v = blockIdx.x * 256u + threadIdx.x;
  const uint32_t e0 = v * N;
  if (e0 >= total)
    return;
  uint32_t r = divByMagic(e0, m.inner, m.innerMagic);
  uint32_t c = e0 - r * m.inner;
  auto rowOf = [&](uint32_t row) {
    const uint32_t q = divByMagic(row, m.rowDiv, m.divMagic);
    return q - divByMagic(q, m.rowMod, m.modMagic) * m.rowMod;
  };
  if (WHOLE || e0 + N <= total) {
    const V *pa = reinterpret_cast<const V *>(a) + v;
    const V va = STREAM ? __builtin_nontemporal_load(pa) : *pa;
    V vb, vo;
    if (WHOLE && ROW_OF_B) {
      vb = *reinterpret_cast<const V *>(b + size_t(rowOf(r)) * m.inner + c);
    } else if (WHOLE) {
      const T x = b[rowOf(r)];
#pragma unroll
      for (int j = 0; j < N; j++)
        vb[j] = x;
    } else {
      uint32_t rb = rowOf(r);
#pragma unroll
      for (int j = 0; j < N; j++) {
        vb[j] = b[ROW_OF_B ? size_t(rb) * m.inner + c : size_t(rb)];
        if (++c == m.inner) {
          c = 0;
          rb = rowOf(++r);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < N; j++)
      vo[j] = applyOp<T>(OP, va[j], vb[j]);
    storeResult<V, STREAM>(reinterpret_cast<V *>(out) + v, vo);
  } else { // the last elements of a total that is not a multiple of the width
    for (uint32_t e = e0; e < total; e++) {
      const uint32_t rb = rowOf(r);
      out[e] = applyOp<T>(OP, a[e], b[ROW_OF_B ? size_t(rb) * m.inner + c : size_t(rb)]);
      if (++c == m.inner) {
        c = 0;
        r++;
      }
    }
  }
}

// Same-shape operands: no index arithmetic at all.
template <typename T, int OP, bool STREAM>
__global__ __launch_bounds__(256) void elementwiseSameKernel(
    const T *a, const T *b, T *out, int64_t total) {
  using V = typename Vec16<T>::type;
  constexpr int N = Vec16<T>::kN;
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i * N + N <= total) {
    const V *pa = reinterpret_cast<const V *>(a) + i;
    const V *pb = reinterpret_cast<const V *>(b) + i;
    const V va = STREAM ? __builtin_nontemporal_load(pa) : *pa;
    const V vb = STREAM ? __builtin_nontemporal_load(pb) : *pb;
    V vo;
#pragma unroll
    for (int j = 0; j < N; j++)
      vo[j] = applyOp<T>(OP, va[j], vb[j]);
    storeResult<V, STREAM>(reinterpret_cast<V *>(out) + i, vo);
  } else {
    for (int64_t e = i * N; e < total; e++)
      out[e] = applyOp<T>(OP, a[e], b[e]);
  }
}

// Any broadcast pattern, scalar accesses.  The index walk is the reference's:
// coordinate = x / stride, clamped to B's extent, times B's stride.
template <typename T, int OP>
__global__ __launch_bounds__(256) void elementwiseGenericKernel(
    const T *a, const T *b, T *out, int64_t total, BroadcastDesc d) {
  const int64_t step = int64_t(gridDim.x) * blockDim.x;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += step) {
    int64_t x = i, bIdx = 0;
    for (int k = 0; k < d.rank; k++) {
      const int64_t coord = x / d.outStride[k];
      x -= coord * d.outStride[k];
      bIdx += (coord < d.bSize[k] ? coord : d.bSize[k] - 1) * d.bStride[k];
    }
    out[i] = applyOp<T>(OP, a[i], b[bIdx]);
  }
}

// Merges dimensions and recognises the row forms above; false: a contiguous B
// of another pattern, or a strided B, which take the generic walk.
bool rowBroadcast(const BroadcastDesc &d, int64_t total, RowBroadcast *m) {
  // groups of neighbouring dimensions, innermost first: extent, and whether B
  // is full there (B must be dense over its full dimensions)
  int64_t extent[kMaxRank];
  bool full[kMaxRank];
  int groups = 0;
  int64_t dense = 1;
  for (int k = d.rank - 1; k >= 0; k--) {
    if (d.outSize[k] == 1)
      continue;
    const bool f = d.bSize[k] != 1;
    if (f && d.bStride[k] != dense)
      return false;
    if (f)
      dense *= d.outSize[k];
    if (groups > 0 && full[groups - 1] == f)
      extent[groups - 1] *= d.outSize[k];
    else {
      extent[groups] = d.outSize[k];
      full[groups++] = f;
    }
  }
  int64_t inner = 1, div = 1, mod = 1;
  bool rowOfB = true;
  if (groups > 3 || (groups == 3 && !full[1] && !full[2]))
    return false;
  if (groups >= 1) {
    inner = extent[0];
    rowOfB = full[0];
    if (full[0]) { // [.., n] with B repeating in front of it, or [b, 1, n]
      if (groups >= 2)
        div = groups == 3 ? extent[1] : 1;
      mod = groups == 3 ? extent[2] : 1;
    } else { // one value per row: [b, 1] or [1, s, 1]
      mod = groups >= 2 ? extent[1] : 1;
    }
  }
  if (total >= (int64_t(1) << 31))
    return false;
  m->inner = uint32_t(inner);
  m->rowDiv = uint32_t(div);
  m->rowMod = uint32_t(mod);
  m->innerMagic = magicFor(m->inner);
  m->divMagic = magicFor(m->rowDiv);
  m->modMagic = magicFor(m->rowMod);
  m->rowOfB = rowOfB;
  return true;
}

template <typename T, int OP, bool STREAM>
void launchRows(const T *a, const T *b, T *out, int64_t total,
                const RowBroadcast &m, bool whole, hipStream_t s) {
  constexpr int N = Vec16<T>::kN;
  const int64_t nvec = (total + N - 1) / N;
  const dim3 grid((unsigned)((nvec + 255) / 256)), block(256);
  if (m.rowOfB && whole)
    elementwiseRowKernel<T, OP, true, true, STREAM>
        <<<grid, block, 0, s>>>(a, b, out, uint32_t(total), m);
  else if (m.rowOfB)
    elementwiseRowKernel<T, OP, true, false, STREAM>
        <<<grid, block, 0, s>>>(a, b, out, uint32_t(total), m);
  else if (whole)
    elementwiseRowKernel<T, OP, false, true, STREAM>
        <<<grid, block, 0, s>>>(a, b, out, uint32_t(total), m);
  else
    elementwiseRowKernel<T, OP, false, false, STREAM>
        <<<grid, block, 0, s>>>(a, b, out, uint32_t(total), m);
}

template <typename T, int OP>
Status elementwiseDispatch(const T *a, const T *b, T *out, int64_t total,
                           const BroadcastDesc &d, hipStream_t s) {
  constexpr int N = Vec16<T>::kN;
  const bool stream = total * int64_t(sizeof(T)) > kStreamingBytes;
  const int64_t blocks = ((total + N - 1) / N + 255) / 256;
  const bool vec = aligned16(a) && aligned16(out);
  RowBroadcast m{};
  bool same = true; // B has A's shape and is dense
  for (int k = 0; k < d.rank; k++)
    same = same && d.bSize[k] == d.outSize[k] &&
           (d.outSize[k] == 1 || d.bStride[k] == d.outStride[k]);
  if (same && vec && aligned16(b) && blocks < (int64_t(1) << 31)) {
    const dim3 grid((unsigned)blocks), block(256);
    if (stream)
      elementwiseSameKernel<T, OP, true><<<grid, block, 0, s>>>(a, b, out, total);
    else
      elementwiseSameKernel<T, OP, false><<<grid, block, 0, s>>>(a, b, out, total);
  } else if (vec && rowBroadcast(d, total, &m)) {
    const bool whole = m.inner % N == 0 && (!m.rowOfB || aligned16(b));
    if (stream)
      launchRows<T, OP, true>(a, b, out, total, m, whole, s);
    else
      launchRows<T, OP, false>(a, b, out, total, m, whole, s);
  } else {
    const int cus = deviceInfo().computeUnits;
    int64_t generic = (total + 255) / 256;
    if (generic > int64_t(cus) * 32)
      generic = int64_t(cus) * 32;
    elementwiseGenericKernel<T, OP>
        <<<dim3((unsigned)generic), dim3(256), 0, s>>>(a, b, out, total, d);
  }
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}

// ---------------------------------------------------------------- gather --
// One 16-byte vector per thread, rowVecs of them per row.  Rows need not be
// whole vectors: they start at any element boundary (which the hardware's
// 16-byte accesses take), and the last vector of a row ends with the row,
// overlapping the one before it with the same values.
template <typename T>
__global__ __launch_bounds__(256) void gatherKernel(
    const int64_t *__restrict__ indices, const T *__restrict__ value,
    T *__restrict__ out, uint32_t total, int64_t vocab, uint32_t rowLength,
    uint32_t rowVecs, uint32_t rowMagic) {
  using V = typename Vec16<T>::type;
  typedef V VAny __attribute__((aligned(sizeof(T))));
  constexpr uint32_t N = Vec16<T>::kN;
  const uint32_t v = blockIdx.x * 256u + threadIdx.x;
  if (v >= total)
    return;
  const uint32_t r = divByMagic(v, rowVecs, rowMagic);
  uint32_t c = (v - r * rowVecs) * N;
  if (c + N > rowLength)
    c = rowLength - N;
  // An index outside the table would read foreign memory; clamp it.
  int64_t i = indices[r];
  i = i < 0 ? 0 : (i >= vocab ? vocab - 1 : i);
  const V got = *reinterpret_cast<const VAny *>(value + i * rowLength + c);
  storeWriteThrough(out + size_t(r) * rowLength + c, got);
}

// Rows shorter than a vector, outputs of 2^31 vectors and more.
template <typename T>
__global__ __launch_bounds__(256) void gatherScalarKernel(
    const int64_t *__restrict__ indices, const T *__restrict__ value,
    T *__restrict__ out, int64_t numIndices, int64_t vocab, int64_t rowLength) {
  const int64_t total = numIndices * rowLength;
  const int64_t step = int64_t(gridDim.x) * blockDim.x;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += step) {
    const int64_t r = i / rowLength;
    const int64_t c = i - r * rowLength;
    int64_t src = indices[r];
    src = src < 0 ? 0 : (src >= vocab ? vocab - 1 : src);
    out[i] = value[src * rowLength + c];
  }
}

// ------------------------------------------------------------ cu_seqlens --
// One workgroup, see mask_sums.h.
template <typename InT>
__global__ __launch_bounds__(1024) void cuSeqLenKernel(
    const InT *__restrict__ mask, int32_t *out, int64_t bs, int64_t seq) {
  __shared__ int32_t rowSum[256];
  sumMaskRows<InT, 16>(mask, out, bs, seq, rowSum);
}

// ------------------------------------------------------------------ gelu --
__device__ __forceinline__ float geluErf(float x) {
  return 0.5f * x * (1.0f + erff(x * 0.70710678118654752440f));
}
__device__ __forceinline__ float geluTanh(float x) {
  const float u = 0.7978845608028654f * (x + 0.044715f * x * x * x);
  return 0.5f * x * (1.0f + tanhf(u));
}

template <int FORM>
__global__ __launch_bounds__(256) void geluKernel(const _Float16 *in,
                                                  _Float16 *out,
                                                  int64_t total) {
  const int64_t step = int64_t(gridDim.x) * blockDim.x;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += step) {
    const float x = float(in[i]);
    out[i] = _Float16(FORM == 0 ? geluErf(x) : geluTanh(x));
  }
}

// ------------------------------------------------------------- row stats --
__global__ __launch_bounds__(256) void rowStatsKernel(
    const _Float16 *__restrict__ d, _Float16 *__restrict__ var,
    _Float16 *__restrict__ mean, int64_t rows, int64_t n, float eps) {
  const int lane = threadIdx.x % kWave;
  const int64_t row =
      int64_t(blockIdx.x) * (blockDim.x / kWave) + threadIdx.x / kWave;
  if (row >= rows)
    return;
  float s = 0.f, sq = 0.f;
  for (int64_t j = lane; j < n; j += kWave) {
    const float x = float(d[row * n + j]);
    s += x;
    sq += x * x;
  }
  s = waveSum(s);
  sq = waveSum(sq);
  if (lane == 0) {
    const float m = s / float(n);
    const float ms = sq / float(n);
    // E[x^2] - E[x]^2 cancels to a small negative number for near-constant
    // rows; clamped so that a tiny eps cannot turn it into a NaN
    const float rstd = 1.0f / sqrtf(fmaxf(ms - m * m, 0.f) + eps);
    var[row] = _Float16(rstd);
    mean[row] = _Float16(-m * rstd);
  }
}

__global__ __launch_bounds__(256) void applyRowStatsKernel(
    const _Float16 *__restrict__ a, const _Float16 *__restrict__ var,
    const _Float16 *__restrict__ mean, _Float16 *__restrict__ out,
    int64_t rows, int64_t k) {
  const int64_t total = rows * k;
  const int64_t step = int64_t(gridDim.x) * blockDim.x;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += step) {
    const int64_t r = i / k;
    out[i] = _Float16(float(a[i]) * float(var[r]) + float(mean[r]));
  }
}

inline unsigned cappedBlocks(int64_t work, int perBlock, int mult) {
  int64_t blocks = (work + perBlock - 1) / perBlock;
  const int64_t cap = int64_t(deviceInfo().computeUnits) * mult;
  if (blocks > cap)
    blocks = cap;
  if (blocks < 1)
    blocks = 1;
  return (unsigned)blocks;
}

} // namespace

template <typename T>
Status launchElementwise(BinOp op, const T *a, const T *b, T *out,
                         int64_t total, const BroadcastDesc &desc,
                         hipStream_t s) {
  if (total == 0)
    return Status::kSuccess;
  switch (op) {
  case BinOp::kAdd:
    return elementwiseDispatch<T, 0>(a, b, out, total, desc, s);
  case BinOp::kSub:
    return elementwiseDispatch<T, 1>(a, b, out, total, desc, s);
  case BinOp::kMul:
    return elementwiseDispatch<T, 2>(a, b, out, total, desc, s);
  case BinOp::kDiv:
    return elementwiseDispatch<T, 3>(a, b, out, total, desc, s);
  }
  return Status::kInvalidArgument;
}
template Status launchElementwise<_Float16>(BinOp, const _Float16 *,
                                            const _Float16 *, _Float16 *,
                                            int64_t, const BroadcastDesc &,
                                            hipStream_t);
template Status launchElementwise<float>(BinOp, const float *, const float *,
                                         float *, int64_t,
                                         const BroadcastDesc &, hipStream_t);

template <typename T>
Status launchGather(const int64_t *indices, const T *value, T *out,
                    int64_t numIndices, int64_t vocab, int64_t rowLength,
                    hipStream_t s) {
  if (numIndices == 0 || rowLength == 0)
    return Status::kSuccess;
  constexpr int N = Vec16<T>::kN;
  const int64_t rowVecs = (rowLength + N - 1) / N, total = numIndices * rowVecs;
  if (rowLength >= N && rowLength < (int64_t(1) << 31) &&
      total < (int64_t(1) << 31)) {
    const dim3 grid((unsigned)((total + 255) / 256));
    gatherKernel<T><<<grid, dim3(256), 0, s>>>(
        indices, value, out, uint32_t(total), vocab, uint32_t(rowLength),
        uint32_t(rowVecs), magicFor(uint32_t(rowVecs)));
  } else {
    gatherScalarKernel<T>
        <<<dim3(cappedBlocks(numIndices * rowLength, 256, 32)), dim3(256), 0,
           s>>>(indices, value, out, numIndices, vocab, rowLength);
  }
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}
template Status launchGather<_Float16>(const int64_t *, const _Float16 *,
                                       _Float16 *, int64_t, int64_t, int64_t,
                                       hipStream_t);
template Status launchGather<float>(const int64_t *, const float *, float *,
                                    int64_t, int64_t, int64_t, hipStream_t);

template <typename InT>
Status launchCuSeqLen(const InT *mask, int32_t *out, int64_t bs, int64_t seq,
                      hipStream_t s) {
  cuSeqLenKernel<InT><<<dim3(1), dim3(1024), 0, s>>>(mask, out, bs, seq);
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}
template Status launchCuSeqLen<int64_t>(const int64_t *, int32_t *, int64_t,
                                        int64_t, hipStream_t);
template Status launchCuSeqLen<int32_t>(const int32_t *, int32_t *, int64_t,
                                        int64_t, hipStream_t);

Status launchGeluF16(const _Float16 *in, _Float16 *out, int64_t total, int form,
                     hipStream_t s) {
  if (total == 0)
    return Status::kSuccess;
  const dim3 grid(cappedBlocks(total, 256, 32)), block(256);
  if (form == 0)
    geluKernel<0><<<grid, block, 0, s>>>(in, out, total);
  else
    geluKernel<1><<<grid, block, 0, s>>>(in, out, total);
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}

Status launchRowStatsF16(const _Float16 *d, _Float16 *var, _Float16 *mean,
                         int64_t rows, int64_t n, float eps, hipStream_t s) {
  if (rows == 0)
    return Status::kSuccess;
  rowStatsKernel<<<dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s>>>(
      d, var, mean, rows, n, eps);
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}

Status launchApplyRowStatsF16(const _Float16 *a, const _Float16 *var,
                              const _Float16 *mean, _Float16 *out, int64_t rows,
                              int64_t k, hipStream_t s) {
  if (rows == 0 || k == 0)
    return Status::kSuccess;
  applyRowStatsKernel<<<dim3(cappedBlocks(rows * k, 256, 32)), dim3(256), 0,
                        s>>>(a, var, mean, out, rows, k);
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}

} // namespace hom

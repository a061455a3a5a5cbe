// The embedding front of a lowered BERT graph in one kernel, for gfx950:
// cu_seqlens from the padding mask, word rows gathered by token id, position
// rows added, layer norm (no affine parameters).
//
// As four kernels (CuSeqLen.h:28-74, GatherRunner.h:32-77,
// ElementwiseRunner.h:69-153, Layernorm.h:584-694 of the reference's runners)
// this is four dependent launches of 2-4 us for a few hundred kilobytes.  Here
// workgroup 0 forms cu_seqlens while the others make the rows, a wavefront per
// row and the row in registers from the table to the normalised result.
// ids and mask are read once each and may therefore lie in pinned host memory:
// their 16 bytes per token then come over PCIe under the same latency a copy
// into device memory would add as a step of its own.
#include "cross_lane.h"
#include "fast_div.h"
#include "kernels.h"
#include "mask_sums.h"
#include "store_policy.h"

namespace hom {
namespace {

constexpr int kWave = 64;
typedef _Float16 half8 __attribute__((ext_vector_type(8)));

constexpr int kThreads = 1024, kWaves = kThreads / kWave;

// VPL: 16-byte vectors of a row per lane; kRows: token rows of a wavefront,
// consecutive, whose ids arrive with one request: 4 where there are enough rows
// to fill the chip, 1 where the chain of latencies (id, row, result) counts.
template <int VPL, int kRows>
__global__ __launch_bounds__(kThreads) void embedKernel(
    const int64_t *__restrict__ ids, const int64_t *__restrict__ mask,
    const _Float16 *__restrict__ word, const _Float16 *__restrict__ pos,
    _Float16 *__restrict__ out, int32_t *__restrict__ cu, int bs, int seq,
    int hidden, int vocab, uint32_t seqMagic, float eps, bool packedOut) {
  __shared__ int32_t rowSum[256];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  if (blockIdx.x == 0) {
    sumMaskRows<int64_t, kWaves>(mask, cu, bs, seq, rowSum);
    return;
  }
  const int rows = bs * seq;
  const int row0 = (int(blockIdx.x - 1) * kWaves + wave) * kRows;
  if (row0 >= rows)
    return;
  // Lane l < kRows holds the id of row row0 + l.  (The other lanes ask for
  // nothing: every lane's request of uncached host memory is one of its own.)
  int64_t idWant = 0;
  if (lane < kRows)
    idWant = ids[row0 + lane < rows ? row0 + lane : rows - 1];
  // An index outside the table would read foreign memory; clamp it.
  const int id = idWant < 0 ? 0 : (idWant >= vocab ? vocab - 1 : int(idWant));
  const int nvec = hidden / 8;
  half8 w[kRows][VPL], p[kRows][VPL];
#pragma unroll
  for (int r = 0; r < kRows; r++) {
    const int at = row0 + r < rows ? row0 + r : rows - 1;
    const int posRow = at - int(divByMagic(uint32_t(at), uint32_t(seq), seqMagic)) * seq;
    const int wordRow = __builtin_amdgcn_readlane(id, r);
#pragma unroll
    for (int i = 0; i < VPL; i++) {
      const int v = lane + i * kWave < nvec ? lane + i * kWave : 0;
      p[r][i] = reinterpret_cast<const half8 *>(pos + int64_t(posRow) * hidden)[v];
      w[r][i] = reinterpret_cast<const half8 *>(word + int64_t(wordRow) * hidden)[v];
    }
  }
  __builtin_amdgcn_sched_barrier(0); // every request is out
  const float invH = 1.0f / float(hidden);
#pragma unroll
  for (int r = 0; r < kRows; r++) {
    float v[VPL][8];
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; i++) {
      const bool mine = lane + i * kWave < nvec;
      // (the sum of the two rows is an fp16 tensor of the graph: rounded)
      const half8 x = w[r][i] + p[r][i];
#pragma unroll
      for (int e = 0; e < 8; e++) {
        v[i][e] = mine ? float(x[e]) : 0.f;
        sum += v[i][e];
      }
    }
    const float mean = waveSum(sum) * invH;
    float sq = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; i++)
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float d = lane + i * kWave < nvec ? v[i][e] - mean : 0.f;
        sq += d * d;
      }
    const float rstd = 1.0f / sqrtf(waveSum(sq) * invH + eps);
#pragma unroll
    for (int i = 0; i < VPL; i++) {
      half8 o;
#pragma unroll
      for (int e = 0; e < 8; e++)
        o[e] = _Float16((v[i][e] - mean) * rstd);
      if (row0 + r < rows && lane + i * kWave < nvec) {
        // (fragment order: 16 bytes of a line that the rows next to this one
        // complete, which is for the L2 to put together)
        if (packedOut)
          *reinterpret_cast<half8 *>(
              out + packedOffset(row0 + r, (lane + i * kWave) * 8, hidden)) = o;
        else
          storeWriteThrough(out + int64_t(row0 + r) * hidden + (lane + i * kWave) * 8, o);
      }
    }
  }
}

} // namespace

bool embedFits(const _Float16 *word, const _Float16 *pos, const _Float16 *out,
               int64_t bs, int64_t seq, int64_t hidden, int64_t vocab) {
  auto al16 = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  return hidden % 8 == 0 && hidden <= 4 * kWave * 8 && al16(word) && al16(pos) &&
         al16(out) && bs * seq < (int64_t(1) << 31) - kWaves * 4 &&
         vocab < (int64_t(1) << 31);
}

Status launchEmbed(const int64_t *ids, const int64_t *mask, const _Float16 *word,
                   const _Float16 *pos, _Float16 *out, int32_t *cu, int64_t bs,
                   int64_t seq, int64_t hidden, int64_t vocab, float eps,
                   bool packedOut, hipStream_t s) {
  const int64_t rows = bs * seq;
  const bool few = rows <= 4096;
  const int64_t perBlock = kWaves * (few ? 1 : 4);
  const dim3 grid((unsigned)(1 + (rows + perBlock - 1) / perBlock)), block(kThreads);
  const uint32_t magic = magicFor(uint32_t(seq));
  const int nvec = int(hidden / 8);
  auto kernel = nvec <= kWave       ? (few ? embedKernel<1, 1> : embedKernel<1, 4>)
                : nvec <= 2 * kWave ? (few ? embedKernel<2, 1> : embedKernel<2, 4>)
                                    : (few ? embedKernel<4, 1> : embedKernel<4, 4>);
  kernel<<<grid, block, 0, s>>>(ids, mask, word, pos, out, cu, int(bs), int(seq),
                                int(hidden), int(vocab), magic, eps, packedOut);
  HOM_HIP_RET(hipGetLastError(), Status::kInternal);
  return Status::kSuccess;
}

} // namespace hom

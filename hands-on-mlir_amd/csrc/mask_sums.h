// cu_seqlens of a padding mask: out[0] = 0, out[i + 1] = sum of mask rows 0 .. i
// (reference: include/NVGPUKernels/CuSeqLen.h:28-74).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hom {

// One workgroup of WAVES wavefronts: each sums rows of the mask, 8 loads in
// flight per lane, into LDS (rowSum: 256 words); the first wavefront then turns
// 64 row sums at a time into the running total with a prefix sum across its
// lanes.  A chain of memory round trips is all this is made of (a row at a time
// and a serial scan through memory by one thread: 7.4 us for 16 rows of 200,
// now 2.7).
template <typename InT, int WAVES>
__device__ __forceinline__ void sumMaskRows(const InT *__restrict__ mask,
                                            int32_t *out, int64_t bs,
                                            int64_t seq, int32_t *rowSum) {
  constexpr int kLanes = 64, kPass = 256; // rows per pass
  const int lane = threadIdx.x % kLanes;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kLanes);
  int32_t acc = 0; // total of all rows before this pass (first wavefront)
  if (threadIdx.x == 0)
    out[0] = 0;
  for (int64_t base = 0; base < bs; base += kPass) {
    const int rows = int(bs - base < kPass ? bs - base : kPass);
    for (int r = wave; r < rows; r += WAVES) {
      const InT *row = mask + (base + r) * seq;
      int32_t sum = 0;
      for (int64_t j = 0; j < seq; j += 8 * kLanes) {
        InT v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) { // (past the end: the last element again)
          const int64_t at = j + u * kLanes + lane;
          v[u] = row[at < seq ? at : seq - 1];
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
          sum += j + u * kLanes + lane < seq ? int32_t(v[u]) : 0;
      }
#pragma unroll
      for (int off = kLanes / 2; off > 0; off >>= 1)
        sum += __shfl_xor(sum, off, kLanes);
      if (lane == 0)
        rowSum[r] = sum;
    }
    __syncthreads();
    if (wave == 0) {
      for (int r = 0; r < rows; r += kLanes) {
        int32_t v = r + lane < rows ? rowSum[r + lane] : 0;
#pragma unroll
        for (int off = 1; off < kLanes; off <<= 1) {
          const int32_t below = __shfl_up(v, off, kLanes);
          v += lane >= off ? below : 0;
        }
        if (r + lane < rows)
          out[base + r + lane + 1] = acc + v;
        acc += __shfl(v, kLanes - 1, kLanes);
      }
    }
    __syncthreads();
  }
}

} // namespace hom

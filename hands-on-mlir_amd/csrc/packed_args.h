// What the two packed GEMM kernels (gemm_packed.hip, gemm_packed_tile.hip) share.
#pragma once

#include "gelu.h"
#include "kernels.h"

namespace hom {

struct PackedArgs {
  const _Float16 *C; // residual source [M, N] or null
  _Float16 *D;
  const float *colSum;  // [N], read when A is normalised
  const float *statsIn; // (rstd, -mu rstd) per row of C, or null: C as it is
  float *statsOut;      // (rstd, -mu rstd) per row of A, or null
  const char *ahead;    // weights of the kernels behind this one
  int64_t aheadBytes;
  int M, N;
  int activation;       // 0, 1 erf GELU, 2 tanh GELU
  int cPacked, dPacked; // in fragment order
  float invK, eps;
};

// A workgroup behind those with work of their own reads weights that the next
// kernels need, so that those find them in the last-level cache: a lone small
// kernel leaves CUs and most of the memory system idle.  Group `group` of
// `groups` takes its runs of kAheadBytes<THREADS>.
constexpr int kAheadLoads = 8;
template <int THREADS> constexpr int64_t kAheadBytes = int64_t(THREADS) * 16 * kAheadLoads;
template <int THREADS>
__device__ __forceinline__ void readAhead(const char *ahead, int64_t bytes, int group, int groups,
                                          int tid) {
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  for (int64_t at = group * kAheadBytes<THREADS>; at < bytes;
       at += groups * kAheadBytes<THREADS>) {
    u32x4 v[kAheadLoads];
#pragma unroll
    for (int i = 0; i < kAheadLoads; i++) {
      const int64_t o = at + (i * THREADS + tid) * 16;
      v[i] = *reinterpret_cast<const u32x4 *>(ahead + (o < bytes ? o : 0));
    }
#pragma unroll
    for (int i = 0; i < kAheadLoads; i++)
      asm volatile("" ::"v"(v[i])); // (nothing else uses the values)
  }
}
// Workgroups to add for that: one for each run, up to `most`.
template <int THREADS> inline int aheadGroups(int64_t bytes, int64_t most) {
  const int64_t runs = (bytes + kAheadBytes<THREADS> - 1) / kAheadBytes<THREADS>;
  return int(runs < most ? runs : most < 0 ? 0 : most);
}

// A folded layer norm takes its row statistics from sums that the GEMM can form on
// the way, and E[x^2] - mu^2 loses (mu / sigma)^2 units in the last place of sums
// of up to 256 terms in a row (1 / sigma off by 3e-4 at 60 sigma, 1.5e-2 at 300).
// Beyond 4 sigma, where that is 1e-5 at most, the rows are read a second time and
// centred, which gives 2e-7 at any mean.  That costs such rows what a layer norm
// costs, and no other row anything.
__device__ __forceinline__ bool meanDominates(float mu, float var) {
  return var * 16.0f < mu * mu;
}

// The tiled kernel (A packed); false: no tile of it suits the problem.
struct PackedTileChoice {
  int tile;
  double us; // modelled time
};
PackedTileChoice choosePackedTile(const PackedGemm &g);
Status launchPackedTile(int tile, const PackedGemm &g, const PackedArgs &p, hipStream_t s);

} // namespace hom

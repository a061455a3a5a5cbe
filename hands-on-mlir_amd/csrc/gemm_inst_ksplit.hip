// Instantiates the kernels whose wavefronts split K.
#include "gemm_ksplit.h"
#include "gemm_inst.h"

namespace hom {
namespace gemmk {
// (used by launchKsplitEntry, instantiated in gemm_inst_staged.hip)
#define HOM_KSPLIT_SHORT(E)                                                                        \
  extern template Status launchStaged<64, 64, 32, 2, 2, E, false, 1>(const GemmProblem &,          \
                                                                     hipStream_t);                 \
  extern template Status launchStaged<64, 64, 32, 2, 2, E, true, 1>(const GemmProblem &,           \
                                                                    hipStream_t);
HOM_KSPLIT_SHORT(0)
HOM_KSPLIT_SHORT(1)
HOM_KSPLIT_SHORT(2)
#undef HOM_KSPLIT_TILE
#define HOM_KSPLIT_TILE(BM, BN) HOM_INST_EPILOGUES(launchKsplitEntry, BM / 16, BN / 16)
#include "gemm_manifest.inc"
} // namespace gemmk
} // namespace hom

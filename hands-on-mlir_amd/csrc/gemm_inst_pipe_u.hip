// Instantiates the register-staged pipeline kernels for operands at any element
// alignment (group U of the manifest).
#include "gemm_pipe.h"
#include "gemm_inst.h"

namespace hom {
namespace gemmk {
#undef HOM_PIPE_TILE_U
#define HOM_PIPE_TILE_U(BM, BN, WM, WN, DIST)                                  \
  HOM_INST_EPILOGUES_ANY(launchPipe, BM, BN, WM, WN, DIST)
#include "gemm_manifest.inc"
} // namespace gemmk
} // namespace hom

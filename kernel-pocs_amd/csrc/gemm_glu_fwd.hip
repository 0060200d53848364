// Gate/up GEMMs with the SwiGLU / GeGLU forward epilogue: the gate and up weights
// are one dual B (both [N][K]), 256 x 256 tiles.
#include "gemm_launch.h"

namespace fgemm {

int launch_glu_fwd(int epi, int al, int bl, const GemmArgs& a, hipStream_t s) {
  if (al == ROW && bl == COL) switch (epi) {
      case EPI_SWIGLU_FWD: return launch_cfg<bf16_t, 256, 256, 2, 2, ROW, COL, B_DUAL, EPI_SWIGLU_FWD>(a, s);
      case EPI_GEGLU_TANH_FWD: return launch_cfg<bf16_t, 256, 256, 2, 2, ROW, COL, B_DUAL, EPI_GEGLU_TANH_FWD>(a, s);
      case EPI_GEGLU_ERF_FWD: return launch_cfg<bf16_t, 256, 256, 2, 2, ROW, COL, B_DUAL, EPI_GEGLU_ERF_FWD>(a, s);
    }
  return forge_set_error(FORGE_ERR_UNSUPPORTED, "gemm: epilogue %d with layouts (%d, %d)", epi, al, bl);
}

}  // namespace fgemm

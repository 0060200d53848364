// Down-projection backward GEMMs with the SwiGLU / GeGLU backward epilogue, 256 x 256
// tiles; W_down may be [K][N] or [N][K].
#include "gemm_launch.h"

namespace fgemm {

template <int EPI>
static int launch(int al, int bl, const GemmArgs& a, hipStream_t s) {
  if (al == ROW && bl == ROW) return launch_cfg<bf16_t, 256, 256, 2, 2, ROW, ROW, B_SINGLE, EPI>(a, s);
  if (al == ROW && bl == COL) return launch_cfg<bf16_t, 256, 256, 2, 2, ROW, COL, B_SINGLE, EPI>(a, s);
  return forge_set_error(FORGE_ERR_UNSUPPORTED, "gemm: epilogue %d with layouts (%d, %d)", EPI, al, bl);
}

int launch_glu_bwd(int epi, int al, int bl, const GemmArgs& a, hipStream_t s) {
  switch (epi) {
    case EPI_SWIGLU_BWD: return launch<EPI_SWIGLU_BWD>(al, bl, a, s);
    case EPI_GEGLU_TANH_BWD: return launch<EPI_GEGLU_TANH_BWD>(al, bl, a, s);
    case EPI_GEGLU_ERF_BWD: return launch<EPI_GEGLU_ERF_BWD>(al, bl, a, s);
  }
  return forge_set_error(FORGE_ERR_UNSUPPORTED, "gemm: epilogue %d with layouts (%d, %d)", epi, al, bl);
}

}  // namespace fgemm

// bf16 GEMMs that store an fp32 C (whole, beta-accumulated, or split-K partial slices).
#include "gemm_launch.h"

namespace fgemm {

int launch_store_f32(int cfg, int al, int bl, const GemmArgs& a, hipStream_t s) {
  return launch_epi<bf16_t, EPI_STORE_F32>(cfg, al, bl, a, s);
}

}  // namespace fgemm

// bf16 GEMMs that add into an fp32 C.
#include "gemm_launch.h"

namespace fgemm {

int launch_atomic_f32(int cfg, int al, int bl, const GemmArgs& a, hipStream_t s) {
  return launch_epi<bf16_t, EPI_ATOMIC_F32>(cfg, al, bl, a, s);
}

}  // namespace fgemm

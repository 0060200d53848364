// bf16 GEMMs that store a bf16 C.
#include "gemm_launch.h"

namespace fgemm {

int launch_store_bf16(int cfg, int al, int bl, const GemmArgs& a, hipStream_t s) {
  return launch_epi<bf16_t, EPI_STORE_BF16>(cfg, al, bl, a, s);
}

}  // namespace fgemm

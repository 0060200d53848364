// fp16 instantiations of the GEMM core: an fp16 or fp32 C (no fused epilogues).
#include "gemm_launch.h"

namespace fgemm {

int launch_f16(int epi, int cfg, int al, int bl, const GemmArgs& a, hipStream_t s) {
  switch (epi) {
    case EPI_STORE_BF16: return launch_epi<fp16_t, EPI_STORE_BF16>(cfg, al, bl, a, s);
    case EPI_STORE_F32: return launch_epi<fp16_t, EPI_STORE_F32>(cfg, al, bl, a, s);
  }
  return forge_set_error(FORGE_ERR_UNSUPPORTED, "gemm: epilogue %d with fp16 operands", epi);
}

}  // namespace fgemm

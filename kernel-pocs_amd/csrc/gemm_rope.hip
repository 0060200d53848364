// The LoRA-QKV GEMM with the RoPE epilogue (both operands K-contiguous, 256 x 256 tiles).
#include "gemm_launch.h"

namespace fgemm {

int launch_rope(const GemmArgs& a, hipStream_t s) {
  return launch_cfg<bf16_t, 256, 256, 2, 2, ROW, COL, B_SINGLE, EPI_ROPE>(a, s);
}

}  // namespace fgemm

// f32 GEMM on the matrix cores (gemm_tile.hpp).
#include "gemm_tile.inc.hpp"

namespace rstsr {
namespace hip {

void tile_gemm_f32(rstsr_hip_ctx* ctx, const GemmProblem& P, float alpha, float beta, bool beta_zero) {
    tile_gemm_run<float>(ctx, "s", P, alpha, beta, beta_zero, nullptr);
}

}  // namespace hip
}  // namespace rstsr

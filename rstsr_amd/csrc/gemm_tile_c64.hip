// c64 GEMM on the matrix cores (gemm_tile.hpp).
#include "gemm_tile.inc.hpp"

namespace rstsr {
namespace hip {

void tile_gemm_c64(rstsr_hip_ctx* ctx, const GemmProblem& P, c64 alpha, c64 beta, bool beta_zero) {
    tile_gemm_run<c64>(ctx, "c", P, alpha, beta, beta_zero, nullptr);
}

}  // namespace hip
}  // namespace rstsr

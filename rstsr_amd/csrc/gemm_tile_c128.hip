// c128 GEMM on the matrix cores (gemm_tile.hpp): single, batched and grouped.
#include "gemm_tile.inc.hpp"

namespace rstsr {
namespace hip {

void tile_gemm_c128(rstsr_hip_ctx* ctx, const GemmProblem& P, c128 alpha, c128 beta, bool beta_zero,
                   const int* run_if) {
    tile_gemm_run<c128>(ctx, "z2", P, alpha, beta, beta_zero, run_if);
}

void tile_grouped_c128(rstsr_hip_ctx* ctx, const std::vector<GemmProblem>& probs, c128 alpha, c128 beta,
                      bool beta_zero, const int* run_if) {
    tile_grouped_run<c128>(ctx, "z2", probs, alpha, beta, beta_zero, run_if);
}

}  // namespace hip
}  // namespace rstsr

// f64 GEMM on the matrix cores (gemm_tile.hpp): single, batched and grouped.
#include "gemm_tile.inc.hpp"

namespace rstsr {
namespace hip {

void tile_gemm_f64(rstsr_hip_ctx* ctx, const GemmProblem& P, double alpha, double beta, bool beta_zero,
                   const int* run_if) {
    tile_gemm_run<double>(ctx, "d2", P, alpha, beta, beta_zero, run_if);
}

void tile_grouped_f64(rstsr_hip_ctx* ctx, const std::vector<GemmProblem>& probs, double alpha, double beta,
                      bool beta_zero, const int* run_if) {
    tile_grouped_run<double>(ctx, "d2", probs, alpha, beta, beta_zero, run_if);
}

}  // namespace hip
}  // namespace rstsr

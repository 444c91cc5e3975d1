// gemm_f16.hip — the matrix-core GEMM (gemm_tile.h) over F16 weights.
#include "gemm_tile.h"

hipError_t gemm_f16_span(const GemmArgs& a, int tn, int stages, int grid, hipStream_t st) {
  return launch_span<GEMM_W_F16>(a, tn, stages, grid, st);
}

hipError_t gemm_f16_x3_span(const GemmArgs& a, int tn, int stages, int grid, hipStream_t st) {
  return launch_span<GEMM_W_F16_X3>(a, tn, stages, grid, st);
}

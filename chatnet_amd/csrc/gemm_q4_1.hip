// gemm_q4_1.hip — the matrix-core GEMM (gemm_tile.h) over Q4_1 weights.
#include "gemm_tile.h"

hipError_t gemm_q4_1_plane(const GemmArgs& a, int tn, int mt, int grid, hipStream_t st) {
  return launch_one_plane<GEMM_W_Q4_1>(a, tn, mt, grid, st);
}

hipError_t gemm_q4_1_span(const GemmArgs& a, int tn, int stages, int grid, hipStream_t st) {
  return launch_span<GEMM_W_Q4_1>(a, tn, stages, grid, st);
}

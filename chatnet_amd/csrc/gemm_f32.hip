// gemm_f32.hip — the matrix-core GEMM (gemm_tile.h) over F32 weights.
#include "gemm_tile.h"

hipError_t gemm_f32_span(const GemmArgs& a, int tn, int stages, int grid, hipStream_t st) {
  return launch_span<GEMM_W_F32>(a, tn, stages, grid, st);
}

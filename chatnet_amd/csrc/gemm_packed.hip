// gemm_packed.hip — the matrix-core GEMM (gemm_tile.h) over packed-unit weights.
#include "gemm_tile.h"

hipError_t gemm_packed_plane(const GemmArgs& a, int tn, int mt, int grid, hipStream_t st) {
  return launch_one_plane<GEMM_W_PACKED>(a, tn, mt, grid, st);
}

hipError_t gemm_packed_span(const GemmArgs& a, int tn, int stages, int grid, hipStream_t st) {
  return launch_span<GEMM_W_PACKED>(a, tn, stages, grid, st);
}

// gemm_iq4_xs.hip — the matrix-core GEMM (gemm_tile.h) over IQ4_XS weights.
#include "gemm_tile.h"

hipError_t gemm_iq4_xs_plane(const GemmArgs& a, int tn, int mt, int grid, hipStream_t st) {
  return launch_one_plane<GEMM_W_IQ4_XS>(a, tn, mt, grid, st);
}

hipError_t gemm_iq4_xs_span(const GemmArgs& a, int tn, int stages, int grid, hipStream_t st) {
  return launch_span<GEMM_W_IQ4_XS>(a, tn, stages, grid, st);
}

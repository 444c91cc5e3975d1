// gemm_iq4_nl.hip — the matrix-core GEMM (gemm_tile.h) over IQ4_NL weights.
#include "gemm_tile.h"

hipError_t gemm_iq4_nl_plane(const GemmArgs& a, int tn, int mt, int grid, hipStream_t st) {
  return launch_one_plane<GEMM_W_IQ4_NL>(a, tn, mt, grid, st);
}

hipError_t gemm_iq4_nl_span(const GemmArgs& a, int tn, int stages, int grid, hipStream_t st) {
  return launch_span<GEMM_W_IQ4_NL>(a, tn, stages, grid, st);
}

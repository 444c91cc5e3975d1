// gemm_q5_k.hip — the matrix-core GEMM (gemm_tile.h) over Q5_K weights.
#include "gemm_tile.h"

hipError_t gemm_q5_k_plane(const GemmArgs& a, int tn, int mt, int grid, hipStream_t st) {
  return launch_one_plane<GEMM_W_Q5_K>(a, tn, mt, grid, st);
}

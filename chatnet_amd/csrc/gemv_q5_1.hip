// gemv_q5_1.hip — the Q5_1 instances of the quantized GEMV (gemv_quant.h) and of
// the few-column products (gemv_xcols.h, gemv_mcol.h).
#include "gemv_mcol.h"
#include "gemv_xcols.h"

hipError_t gemv_q5_1_launch(int epi, const GemvArgs& a, int num_cus, hipStream_t st) {
  return launch_type<QT_Q5_1>(epi, a, num_cus, st);
}

hipError_t gemv_q5_1_cols_launch(const GemvArgs& a, int ncols, int num_cus, const McolPlan& p, hipStream_t st) {
  return p.fp32 ? launch_xcols<QT_Q5_1>(a, ncols, num_cus, st) : launch_mcol<QT_Q5_1>(a, ncols, num_cus, p, st);
}

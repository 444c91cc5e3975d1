// gemv_iq4_xs.hip — the IQ4_XS instances of the quantized GEMV (gemv_quant.h) and of
// the few-column products (gemv_xcols.h, gemv_mcol.h).
#include "gemv_mcol.h"
#include "gemv_xcols.h"

hipError_t gemv_iq4_xs_launch(int epi, const GemvArgs& a, int num_cus, hipStream_t st) {
  return launch_type<QT_IQ4_XS>(epi, a, num_cus, st);
}

hipError_t gemv_iq4_xs_cols_launch(const GemvArgs& a, int ncols, int num_cus, const McolPlan& p, hipStream_t st) {
  return p.fp32 ? launch_xcols<QT_IQ4_XS>(a, ncols, num_cus, st) : launch_mcol<QT_IQ4_XS>(a, ncols, num_cus, p, st);
}

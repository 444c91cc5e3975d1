// gemv.hip — fused dequant-GEMV for batch-1 decode on gfx950: the dispatch over
// weight types.  The kernels are gemv_quant.h, instantiated in gemv_*.hip.
//
// Replaces TensorMath.MatVecMulQ4_0 / MatVecMulQ6K / MatVecMulGeneric
// (src/ChatNet.Core/Tensors/TensorMath.cs:548-656) and the fused row dots
// DequantQ4_0.DotProduct (DequantQ4_0.cs:80-149), DequantQ4K.DotProduct
// (DequantQ4K.cs:89-163), DequantQ6K.DotProduct (DequantQ6K.cs:104-188),
// DequantQ8_0.DotProduct and DequantQ5K.DotProduct.
//
// Weights stay in their raw GGUF block layout in HBM.  One lane owns one
// "unit" of a row — two Q4_0 or Q8_0 blocks (64 weights, 36 / 68 B, dword
// aligned), or half a Q4_K / Q5_K / Q6_K super-block (128 weights plus the
// header or scales it needs; Q6_K realigned in registers) — and LPR lanes
// cover a row, so a wave reads each row as one contiguous stretch.  Every lane
// works on RPW rows at once so each x value it reads from LDS feeds RPW rows.
// The input vector is staged in LDS once per workgroup as integer digits (with
// RMSNorm's weight fused in when one is given, TensorMath.RmsNorm
// TensorMath.cs:97-165; the 1/rms factor is applied to the finished sums):
// x is scaled by a power of two per 32- or 16-element group to 19 significant
// bits and split into base-16 digits (Q4_0, short Q4_K rows: signed weight
// nibbles on v_dot8_i32_i4) or base-256 digits (Q8_0, Q5_K, Q6_K, long Q4_K
// rows: weight bytes on v_dot4_i32_i8).  Each group's dot is exact in int32;
// the per-group scales, offsets (q-8, q-32, dmin*m) and 2^-e are applied in
// fp32 once per group.  Q4_1, Q5_0, Q5_1, Q2_K, IQ4_NL and IQ4_XS keep x in fp32
// (products code * x on fmaf, the group's scale and offset after 16 of them).
// Partial row sums are reduced across the LPR lanes with
// cross-lane shuffles.
//
// Epilogues (fused into the lane that finishes a row pair):
//   STORE   y[r]  = dot                          (LM head, matmul API)
//   ADD     y[r] += dot                          (O / down + residual, TensorMath.Add :712-733)
//   QKV     RoPE on q/k pairs + K/V cache write  (TensorMath.ApplyRoPE :408-458, LlamaModel.cs:146-153)
//   SWIGLU  h[r] = silu(gate[r]) * up[r]         (TensorMath.SiluElementwiseMul :253-286)
#include <algorithm>
#include <cstring>

#include "kernels.h"

// The launch shapes cover rows of up to 256 lanes x units: K <= 16384.
bool gemv_supports(int qtype, int K) {
  switch (qtype) {
    case 0:  // F32 and F16 rows (gemv_float.hip): K floats of x in LDS
    case 1:
    case 2:
    case 8: return K > 0 && K % 64 == 0 && K <= 16384;
    case 11:
    case 12:
    case 13:
    case 14: return K > 0 && K % 256 == 0 && K <= 16384;
    case 3:   // Q4_1
    case 6:   // Q5_0
    case 7:   // Q5_1
    case 20: return K > 0 && K % 64 == 0 && K <= 16384;  // IQ4_NL
    case 10:  // Q2_K
    case 23: return K > 0 && K % 256 == 0 && K <= 16384;  // IQ4_XS
    // served as packed units (gemv_launch with kGemvPacked)
    case 15:  // Q8_K
    case 16:  // IQ2_XXS
    case 17:  // IQ2_XS
    case 18:  // IQ3_XXS
    case 19:  // IQ1_S
    case 21:  // IQ3_S
    case 22:  // IQ2_S
    case 29: return K > 0 && K % 256 == 0 && K <= 16384;  // IQ1_M
    default: return false;
  }
}

bool gemv_needs_pack(int qtype) { return qtype == 15 || (qtype >= 16 && qtype <= 19) || qtype == 21 || qtype == 22 || qtype == 29; }

hipError_t gemv_launch(int qtype, int epi, const GemvArgs& a, int num_cus, hipStream_t st) {
  if (epi == GEMV_EPI_ADD_MERGE &&
      (a.msplits < 2 || a.msplits > kFoldMaxSplits || a.mchunk < 1 || a.head_dim % 32 != 0))
    return hipErrorInvalidValue;
  if (qtype == 0 || qtype == 1 || qtype == kGemvPacked) return gemv_float_launch(qtype, epi, a, num_cus, st);
  const int e = epi == GEMV_EPI_ADD_MERGE ? gemv_merge_epi(a.msplits) : epi;
  switch (qtype) {  // the packed-unit types are launched as kGemvPacked
    case 2: return gemv_q4_0_launch(e, a, num_cus, st);
    case 3: return gemv_q4_1_launch(e, a, num_cus, st);
    case 6: return gemv_q5_0_launch(e, a, num_cus, st);
    case 7: return gemv_q5_1_launch(e, a, num_cus, st);
    case 8: return gemv_q8_0_launch(e, a, num_cus, st);
    case 10: return gemv_q2_k_launch(e, a, num_cus, st);
    case 11: return gemv_q3_k_launch(e, a, num_cus, st);
    case 12: return gemv_q4_k_launch(e, a, num_cus, st);
    case 13: return gemv_q5_k_launch(e, a, num_cus, st);
    case 14: return gemv_q6_k_launch(e, a, num_cus, st);
    case 20: return gemv_iq4_nl_launch(e, a, num_cus, st);
    case 23: return gemv_iq4_xs_launch(e, a, num_cus, st);
    default: return hipErrorInvalidValue;
  }
}

constexpr int kColsMax = 16;  // columns of one launch (gemv_mcol.h)

bool gemv_qcols_supports(int qtype) {
  return qtype == 3 || qtype == 6 || qtype == 7 || qtype == 8 || (qtype >= 10 && qtype <= 14) || qtype == 20 || qtype == 23;
}

// Few row groups and long rows (at most half a workgroup of 16 rows per CU, at
// least 24 steps of 128 weights): K shared out over up to 16 workgroups per row
// group, each wave keeping a step, and a launch that adds the shares: Q4_K 164 x
// 11008 at 6 columns 17.8 -> 8.8 us, 2048 x 11008 17.9 -> 15.3, 2048 x 4096 10.5 ->
// 8.2 (at 2 columns 5.5 -> 6.5).  At a workgroup per CU it lost (4096 x 4096 at 6
// columns 10.7 -> 11.2 us, at 12 12.3 -> 16.7).
// Otherwise staging x costs a workgroup about 20 VALU instructions an element,
// so from 32768 elements per CU on (columns x K, times the workgroups a CU runs)
// it is done once ahead, a launch of 3 us.  Every workgroup staging, and ahead:
// Q4_K 11008 x 4096 at 4 columns (22000) 14.4 and 16.0 us, 4096 x 4096 at 8 (32768)
// 10.8 and 10.8, 2048 x 2048 at 16 14.4 and 9.4, Q8_0 10.1 and 9.3, 32000 x 4096 at
// 4 36.9 and 38.1, Q4_K 4096 x 11008 at 4 (44000) 14.3 and 14.2, at 8 25.2 and 18.3.
static int mcol_shares(int M, int K, int num_cus) {
  const int groups = (M + 15) / 16, nsteps = (K + 127) / 128;
  if (nsteps < 24 || 2 * groups > num_cus) return 1;
  int s = num_cus / groups;
  if (s > nsteps / 8) s = nsteps / 8;
  return s > 16 ? 16 : s;
}

static bool mcol_ahead(int M, int K, int n, int num_cus) {
  const long long rows = M <= 16 * num_cus ? 16 : 32;
  const double wgs = (double)((M + rows - 1) / rows) / num_cus;
  return (double)n * K * (wgs < 1 ? 1 : wgs > 2 ? 2 : wgs) >= 32768.0;
}

// Types whose x stays in fp32 up to kFp32Cols columns, as the single column's does
// (a power of two shared by 32 elements costs a large element's neighbours their
// low bits).  More columns ran the GEMM on x rounded to fp16, which the digits of
// the matrix-core product are finer than.
static bool fp32_cols(int qtype, int N) {
  constexpr int kFp32Cols = 7;
  return N <= kFp32Cols && (qtype == 3 || qtype == 6 || qtype == 7 || qtype == 10 || qtype == 20 || qtype == 23);
}

// Columns of one fp32 launch: the records (gemv_quant.h, 68 floats per 64 elements
// or 140 per 128) of as many as 150 KB of LDS hold, two at K = 16384, 7 at 4096.
static int fp32_cols_max(int qtype, int K) {
  const size_t col = (qtype == 10 || qtype == 23 ? (size_t)K / 128 * 140 : (size_t)K / 64 * 68) * sizeof(float);
  return (int)std::min<size_t>(8, 150 * 1024 / col);
}

size_t gemv_qcols_workspace(int qtype, int M, int K, int N, int num_cus) {
  if (fp32_cols(qtype, N)) return 0;
  const int n = N < kColsMax ? N : kColsMax;
  const int shares = mcol_shares(M, K, num_cus);
  if (shares > 1) return (size_t)shares * n * M * sizeof(float);
  if (!mcol_ahead(M, K, n, num_cus)) return 0;
  const size_t tiles = (n + 3) / 4;
  return (size_t)((K + 127) / 128) * 4 * tiles * 560;  // the largest block (gemv_mcol.h)
}

hipError_t gemv_qcols_launch(int qtype, const void* w, const float* x, float* y, int M, int K, int N, int num_cus,
                             void* ws, hipStream_t st) {
  if (!gemv_qcols_supports(qtype) || !gemv_supports(qtype, K) || M <= 0 || N < 1 || !w || !x || !y)
    return hipErrorInvalidValue;
  McolPlan plan{fp32_cols(qtype, N), nullptr, 1, nullptr};
  const int g = plan.fp32 ? fp32_cols_max(qtype, K) : kColsMax;
  if (ws && !plan.fp32) {
    plan.shares = mcol_shares(M, K, num_cus);
    if (plan.shares > 1) plan.part = static_cast<float*>(ws);
    else plan.pre = static_cast<char*>(ws);
  }
  for (int c0 = 0; c0 < N;) {
    const int left = N - c0, groups = (left + g - 1) / g;
    const int nc = (left + groups - 1) / groups;  // even groups: 17 columns run as 9 + 8
    GemvArgs a;
    memset(&a, 0, sizeof(a));
    a.w[0] = a.w[1] = a.w[2] = static_cast<const uint8_t*>(w);
    a.seg_rows[0] = M;
    a.n_vrows = M;
    a.K = K;
    a.x = x + (size_t)c0 * K;
    a.out[0] = y + (size_t)c0 * M;
    hipError_t e;
    if (nc == 1) e = gemv_launch(qtype, GEMV_EPI_STORE, a, num_cus, st);
    else switch (qtype) {
      case 3: e = gemv_q4_1_cols_launch(a, nc, num_cus, plan, st); break;
      case 6: e = gemv_q5_0_cols_launch(a, nc, num_cus, plan, st); break;
      case 7: e = gemv_q5_1_cols_launch(a, nc, num_cus, plan, st); break;
      case 8: e = gemv_q8_0_cols_launch(a, nc, num_cus, plan, st); break;
      case 10: e = gemv_q2_k_cols_launch(a, nc, num_cus, plan, st); break;
      case 11: e = gemv_q3_k_cols_launch(a, nc, num_cus, plan, st); break;
      case 12: e = gemv_q4_k_cols_launch(a, nc, num_cus, plan, st); break;
      case 13: e = gemv_q5_k_cols_launch(a, nc, num_cus, plan, st); break;
      case 14: e = gemv_q6_k_cols_launch(a, nc, num_cus, plan, st); break;
      case 20: e = gemv_iq4_nl_cols_launch(a, nc, num_cus, plan, st); break;
      default: e = gemv_iq4_xs_cols_launch(a, nc, num_cus, plan, st); break;
    }
    if (e != hipSuccess) return e;
    c0 += nc;
  }
  return hipSuccess;
}

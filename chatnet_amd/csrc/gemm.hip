// gemm.hip — quantized-weight GEMM on the matrix cores of gfx950: x conversion,
// packing, K-split reduce, tile choice and the dispatch over weight formats (the
// kernels are gemm_tile.h, instantiated in gemm_*.hip).
//
// y[n][m] = sum_k W[m][k] * x[n][k] for a batch of N inputs: the batched form
// of TensorMath.MatVecMulQ4_0 (src/ChatNet.Core/Tensors/TensorMath.cs:548-578)
// that chatnet_matmul with many columns and a multi-token LlamaModel.Forward span
// (LlamaModel.cs:93-238) need.
//
// W is read as stored (gemm_stored_format) or as packed units (gemm_pack_kernel:
// Q3_K, Q6_K, Q8_K and seven IQ types re-encoded as u8 codes with an fp32 scale
// and offset per 16 weights); x arrives from the producer kernel in the cn_span_pos
// order, either as one fp16 plane scaled per column by a power of two
// (to_f16_scaled_kernel, chatnet_matmul) or, for the exact-weight variant the
// spans run, as fp16 hi + lo planes (conversion, RMSNorm, attention or the
// SwiGLU epilogue).  W bytes and x tiles stream through an LDS ring by direct
// global->LDS loads; each wave dequantizes its W rows into
// v_mfma_f32_32x32x16_f16 operands in registers (one rounded plane, or two
// exact planes) and accumulates in fp32.  When the tile grid leaves the chip
// under-filled the K range is split and gemm_reduce_kernel sums the partial
// tiles and applies the epilogue.  Epilogues: STORE y = acc, ADD y += acc
// (residual), SWIGLU (rows interleave gate/up; h = silu(gate)*up is written
// in the next GEMM's input format).
#include <algorithm>

#include "gemm_tile.h"

namespace {

// Sums the K-split partials [splits][N][M] and applies the epilogue; one
// thread per 4 consecutive rows of one column.
// COMP: the F16 product of chatnet_matmul (compensated, see gemm_s_kernel).
template <bool COMP>
__global__ __launch_bounds__(CN_BLOCK) void gemm_reduce_kernel(GemmArgs a) {
  const int m4 = (a.M + 3) / 4;
  const long long t = (long long)blockIdx.x * CN_BLOCK + threadIdx.x;
  if (t >= (long long)m4 * a.N) return;
  const int n = (int)(t / m4), m = (int)(t % m4) * 4;
  f32x4 s = {0.f, 0.f, 0.f, 0.f}, c = s;
  for (int k = 0; k < a.splits; k++) {
    const float* p = a.part + ((size_t)k * a.N + n) * a.M + m;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (m + 3 < a.M && (a.M & 3) == 0) {
      v = *reinterpret_cast<const f32x4*>(p);
    } else {
      for (int i = 0; i < 4 && m + i < a.M; i++) v[i] = p[i];
    }
    if constexpr (COMP) add_compensated(s, c, v);
    else s += v;
  }
  if constexpr (COMP) f16_dot_again(a, n, m, s);
  write_out4(a, a.epi, n, m, s);
}

// x [N][K] fp32 -> the one-plane kernel's input: per column n a power of two
// 2^e_n that brings max|x[n]| into [2^14, 2^15) (so every element stays
// inside fp16's range and as far above its subnormals as the column allows;
// e_n in [-125, 125]; 0 for a column that is all zero or holds an infinity),
// xh[n][cn_span_pos(k)] = fp16(x[n][k] * 2^e_n) (the scaling is exact, one
// rounding to nearest even) and xinv[n] = 2^-e_n.  One workgroup per column,
// the column held in registers between the max and the conversion.
template <int V>
__global__ __launch_bounds__(CN_BLOCK) void to_f16_scaled_kernel(const float* __restrict__ x,
                                                                uint16_t* __restrict__ xh,
                                                                float* __restrict__ xinv, int K) {
  __shared__ float red[4];
  const size_t n = blockIdx.x;
  const float* xr = x + n * K;
  f32x4 v[V];
  float mx = 0.f;
#pragma unroll
  for (int j = 0; j < V; j++) {
    const int i = (threadIdx.x + CN_BLOCK * j) * 4;
    v[j] = i < K ? *reinterpret_cast<const f32x4*>(xr + i) : f32x4{0.f, 0.f, 0.f, 0.f};
    mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[j][0]), fabsf(v[j][1])), fmaxf(fabsf(v[j][2]), fabsf(v[j][3]))));
  }
  mx = cn_block_max(mx, red);
  int e = 0;
  if (mx > 0.f && mx <= 3.402823466e38f) {
    int E;
    (void)frexpf(mx, &E);  // mx = f * 2^E, f in [0.5, 1)
    e = min(125, max(-125, 15 - E));
  }
  if (threadIdx.x == 0) xinv[n] = ldexpf(1.0f, -e);
  const float sc = ldexpf(1.0f, e);
  uint16_t* o = xh + n * K;
#pragma unroll
  for (int j = 0; j < V; j++) {
    const int i = (threadIdx.x + CN_BLOCK * j) * 4;
    if (i >= K) continue;
    const f32x4 y = v[j] * sc;  // 2^e is a normal float for e in [-125, 125]
    const cn_half2 a = __builtin_convertvector((cn_float2){y[0], y[1]}, cn_half2);
    const cn_half2 b = __builtin_convertvector((cn_float2){y[2], y[3]}, cn_half2);
    *reinterpret_cast<uint2*>(o + cn_span_pos(i)) =
        make_uint2(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b));
  }
}

// x [N][K] fp32 -> GEMM_W_F16_X3's planes with the per-column scaling of
// to_f16_scaled_kernel (the largest finite |x| in [2^14, 2^15)): y = x * 2^e, p0 =
// fp16(y), p1 = fp16((y - p0) 2^11), p2 = fp16((y - p0 - p1 2^-11) 2^22), both
// remainders exact in fp32 and below 2^15.
template <int V>
__global__ __launch_bounds__(CN_BLOCK) void to_f16_planes_kernel(const float* __restrict__ x,
                                                                uint16_t* __restrict__ xp, size_t plane,
                                                                float* __restrict__ xinv, int K) {
  __shared__ float red[4];
  const size_t n = blockIdx.x;
  const float* xr = x + n * K;
  f32x4 v[V];
  float mx = 0.f;
#pragma unroll
  for (int j = 0; j < V; j++) {
    const int i = (threadIdx.x + CN_BLOCK * j) * 4;
    v[j] = i < K ? *reinterpret_cast<const f32x4*>(xr + i) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const float m = fabsf(v[j][q]);
      mx = m <= 3.402823466e38f ? fmaxf(mx, m) : mx;  // finite elements only
    }
  }
  mx = cn_block_max(mx, red);
  int e = 0;
  if (mx > 0.f) {
    int E;
    (void)frexpf(mx, &E);  // mx = f * 2^E, f in [0.5, 1)
    e = min(125, max(-125, 15 - E));
  }
  if (threadIdx.x == 0) xinv[n] = ldexpf(1.0f, -e);
  const float sc = ldexpf(1.0f, e);
#pragma unroll
  for (int j = 0; j < V; j++) {
    const int i = (threadIdx.x + CN_BLOCK * j) * 4;
    if (i >= K) continue;
    const f32x4 y = v[j] * sc;  // 2^e is a normal float for e in [-125, 125]
    _Float16 pl[3][4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const bool fin = fabsf(y[q]) <= 3.402823466e38f;
      pl[0][q] = (_Float16)y[q];
      const float r = fin ? (y[q] - (float)pl[0][q]) * 2048.0f : 0.f;
      pl[1][q] = (_Float16)r;
      pl[2][q] = (_Float16)((r - (float)pl[1][q]) * 2048.0f);
    }
    const size_t o = n * K + cn_span_pos(i);  // four adjacent elements stay adjacent
#pragma unroll
    for (int p = 0; p < 3; p++)
      *reinterpret_cast<uint2*>(xp + p * plane + o) = make_uint2(__builtin_bit_cast(uint32_t, (cn_half2){pl[p][0], pl[p][1]}),
                                                                 __builtin_bit_cast(uint32_t, (cn_half2){pl[p][2], pl[p][3]}));
  }
}

// RMSNorm of each row (TensorMath.RmsNorm, TensorMath.cs:97-165) written as
// the next span GEMM's input: (x[r] * rms_r) * g as fp16 hi + lo planes
// (xb, xb_lo) in the cn_span_pos order.  One workgroup per row, the row held in registers between the sum of
// squares and the scaling (one pass over memory).  With `part` (splits > 0)
// the row is first completed as a residual add of the preceding GEMM's K-split
// partials [splits][rows][dim], summed in split order exactly as
// gemm_reduce_kernel does (x += ((0 + p0) + p1) + ...), and written back to x.
template <int V, int SPL>
__global__ __launch_bounds__(CN_BLOCK) void add_rmsnorm_span_kernel(float* __restrict__ x,
                                                                   const float* __restrict__ part, int splits,
                                                                   const float* __restrict__ g, float eps,
                                                                   uint16_t* __restrict__ xb,
                                                                   uint16_t* __restrict__ xb_lo, int rows, int dim) {
  __shared__ float red[4];
  const size_t row = blockIdx.x;
  float* xr = x + row * dim;
  f32x4 v[V];
#pragma unroll
  for (int j = 0; j < V; j++) {
    const int i = (threadIdx.x + CN_BLOCK * j) * 4;
    v[j] = i < dim ? *reinterpret_cast<const f32x4*>(xr + i) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if constexpr (SPL > 0) {
    // every partial's loads issued before the first add (SPL >= splits;
    // slots past splits are not read)
    f32x4 pv[SPL][V];
#pragma unroll
    for (int k = 0; k < SPL; k++) {
      const float* pr = part + ((size_t)(k < splits ? k : 0) * rows + row) * dim;
#pragma unroll
      for (int j = 0; j < V; j++) {
        const int i = (threadIdx.x + CN_BLOCK * j) * 4;
        pv[k][j] = (i < dim && k < splits) ? *reinterpret_cast<const f32x4*>(pr + i) : f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
    f32x4 sum[V];
#pragma unroll
    for (int j = 0; j < V; j++) sum[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < SPL; k++)
#pragma unroll
      for (int j = 0; j < V; j++)
        if (k < splits) sum[j] += pv[k][j];
#pragma unroll
    for (int j = 0; j < V; j++) {
      const int i = (threadIdx.x + CN_BLOCK * j) * 4;
      v[j] = v[j] + sum[j];
      if (i < dim) *reinterpret_cast<f32x4*>(xr + i) = v[j];
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < V; j++) ss += v[j][0] * v[j][0] + v[j][1] * v[j][1] + v[j][2] * v[j][2] + v[j][3] * v[j][3];
  ss = cn_block_sum(ss, red);
  const float rms = 1.0f / sqrtf(ss / (float)dim + eps);
  uint16_t* o = xb + row * dim;
#pragma unroll
  for (int j = 0; j < V; j++) {
    const int i = (threadIdx.x + CN_BLOCK * j) * 4;
    if (i >= dim) continue;
    const float4 w = *reinterpret_cast<const float4*>(g + i);
    const float y0 = v[j][0] * rms * w.x, y1 = v[j][1] * rms * w.y, y2 = v[j][2] * rms * w.z, y3 = v[j][3] * rms * w.w;
    // the four elements stay adjacent in the span order
    const int pos = cn_span_pos(i);
    uint2 hh, ll;
    cn_split_f16x2(y0, y1, hh.x, ll.x);
    cn_split_f16x2(y2, y3, hh.y, ll.y);
    *reinterpret_cast<uint2*>(o + pos) = hh;
    *reinterpret_cast<uint2*>(xb_lo + row * dim + pos) = ll;
  }
}

// ---------------------------------------------------------------------------
// Packing: one thread re-encodes the 64 weights of chunk c of row r as a
// 96-byte unit: 64 u8 codes in K order, then scale[4] and offset[4] (fp32,
// one pair per 16 weights).  Each block type's dequantized value is
// fmaf(code, scale, offset) with one rounding, as the reference rounds it:
//   Q4_0 (DequantQ4_0.cs)  code q,      scale d,        offset -8d
//   Q4_1 (DequantQ4_1.cs)  code q,      scale d,        offset m
//   Q5_0 (DequantQ5_0.cs)  code q5,     scale d,        offset -16d
//   Q5_1 (DequantQ5_1.cs)  code q5,     scale d,        offset m
//   Q8_0 (DequantQ8_0.cs)  code q+128,  scale d,        offset -128d
//   Q2_K (DequantQ2K.cs)   code q,      scale d*sc,     offset -(dmin*m)
//   Q3_K (DequantQ3K.cs)   code q3,     scale d*sc,     offset -4*d*sc
//   Q4_K (DequantQ4K.cs)   code q,      scale d*sc[s],  offset -(dmin*m[s])
//   Q5_K (DequantQ5K.cs)   code q5,     scale d*sc[s],  offset -(dmin*m[s])
//   Q6_K (DequantQ6K.cs)   code q+32,   scale d*sc[i],  offset -32*d*sc[i]
//   Q8_K (DequantQ8K.cs)   code q+128,  scale d (fp32), offset -128d
//   IQ4_NL, IQ4_XS (DequantIQ.cs)  code table[q]+128, scale d or d*sc, offset -128*scale
//   IQ3_S    code +-(sc*q3)+128, scale d, offset -128d (sc folded into the code)
//   IQ3_XXS  code q3, scale d, offset -4d
//   IQ2_XXS, IQ2_XS  code q, scale d or d*sc, offset -scale
//   IQ2_S    code +-q+128, scale d*sc, offset -128*scale
//   IQ1_S, IQ1_M  code 128+t (t in -1..1; IQ1_M 128+t*2 at full scale), scale d
//            (IQ1_M d/2), offset -128*scale
// (d*sc, dmin*m and the power-of-two multiples are exact in fp32, and so is
// code*scale for the fp16-scaled types, so their one rounding is the
// reference's final add (or none); Q6_K's (d*sc)*q and Q8_K's q*d are rounded
// once either way).  Q2_K and Q3_K elements follow the reference's layouts
// (DequantQ2K.cs:55-82: element 128g + 32t + 16h + l is bits 2t.. of qs[32g +
// 16h + l] with scale byte 8g + 2t + h; DequantQ3K.cs:52-63, :122-150).  Sub-block layouts: Q4_K / Q5_K sub-block s of a super-block
// holds its 32 weights in the reference's order (elements 0..15 are the
// low nibbles of qs[16s..16s+15], 16..31 the high ones), Q6_K as
// DequantQ6K.Dequantize (DequantQ6K.cs:37-88).
// ---------------------------------------------------------------------------
__device__ __forceinline__ float h2f_at(const uint8_t* p) { return cn_h2f((uint32_t)p[0] | ((uint32_t)p[1] << 8)); }

// Q4_K / Q5_K 6-bit scale and min of sub-block j (DequantQ4K.cs:218-264).
__device__ __forceinline__ void k4_scale_min(const uint8_t* q, int j, int& sc, int& mn) {
  if (j < 4) {
    sc = q[j] & 63;
    mn = q[j + 4] & 63;
  } else {
    sc = (q[j + 4] & 0xF) | ((q[j - 4] >> 6) << 4);
    mn = (q[j + 4] >> 4) | ((q[j] >> 6) << 4);
  }
}

// IQ4_NL's table (DequantIQ.IQ4NL_Table, DequantIQ.cs:29-33) plus 128: the
// packed code of each index.
__constant__ uint8_t cn_iq4nl_code[16] = {1, 24, 45, 63, 79, 93, 106, 118, 129, 141, 153, 166, 181, 197, 217, 241};

__global__ __launch_bounds__(CN_BLOCK) void gemm_pack_kernel(int qtype, const uint8_t* __restrict__ w,
                                                            size_t row_bytes, size_t w_bytes, int M, int nchunks,
                                                            uint8_t* __restrict__ dst) {
  const long long t = (long long)blockIdx.x * CN_BLOCK + threadIdx.x;
  if (t >= (long long)M * nchunks) return;
  const int r = (int)(t / nchunks), c = (int)(t % nchunks);
  const uint8_t* row = w + (size_t)r * row_bytes;
  uint32_t code[16];
  float sc[4], of[4];
  auto put = [&](int k, uint32_t v) {
    if ((k & 3) == 0) code[k >> 2] = 0;
    code[k >> 2] |= (v & 0xFFu) << (8 * (k & 3));
  };
  if (qtype == 2 || qtype == 8) {  // Q4_0 / Q8_0: blocks 2c and 2c+1 of 32
    const int bb = qtype == 2 ? 18 : 34;
#pragma unroll
    for (int b = 0; b < 2; b++) {
      const uint8_t* blk = row + (size_t)(2 * c + b) * bb;
      const float d = h2f_at(blk);
#pragma unroll
      for (int j = 0; j < 32; j++) {
        uint32_t v;
        if (qtype == 2) v = j < 16 ? (blk[2 + j] & 15u) : (uint32_t)(blk[2 + j - 16] >> 4);
        else v = (uint32_t)blk[2 + j] ^ 0x80u;
        put(32 * b + j, v);
      }
      sc[2 * b] = sc[2 * b + 1] = d;
      of[2 * b] = of[2 * b + 1] = (qtype == 2 ? -8.0f : -128.0f) * d;
    }
  } else if (qtype == 12 || qtype == 13) {  // Q4_K / Q5_K: sub-blocks 2(c%4), 2(c%4)+1
    const int sbb = qtype == 12 ? 144 : 176;
    const uint8_t* blk = row + (size_t)(c >> 2) * sbb;
    const float d = h2f_at(blk), dmin = h2f_at(blk + 2);
    const uint8_t* qs0 = blk + (qtype == 12 ? 16 : 48);
#pragma unroll
    for (int b = 0; b < 2; b++) {
      const int s = 2 * (c & 3) + b;
      int sv, mv;
      k4_scale_min(blk + 4, s, sv, mv);
      const uint8_t* qs = qs0 + 16 * s;
#pragma unroll
      for (int j = 0; j < 32; j++) {
        uint32_t v = j < 16 ? (qs[j] & 15u) : (uint32_t)(qs[j - 16] >> 4);
        if (qtype == 13) {
          const int e = 32 * s + j;
          v |= (uint32_t)((blk[16 + e / 8] >> (e % 8)) & 1) << 4;
        }
        put(32 * b + j, v);
      }
      sc[2 * b] = sc[2 * b + 1] = d * (float)sv;
      of[2 * b] = of[2 * b + 1] = -(dmin * (float)mv);
    }
  } else if (qtype == 3 || qtype == 6 || qtype == 7) {  // Q4_1 / Q5_0 / Q5_1: blocks 2c and 2c+1 of 32
    const int bb = qtype == 3 ? 20 : (qtype == 6 ? 22 : 24);
#pragma unroll
    for (int b = 0; b < 2; b++) {
      const uint8_t* blk = row + (size_t)(2 * c + b) * bb;
      const float d = h2f_at(blk);
      const uint8_t* qs = blk + bb - 16;
      uint32_t qh = 0;
      if (qtype != 3) {
        const uint8_t* h = blk + (qtype == 6 ? 2 : 4);
        qh = (uint32_t)h[0] | ((uint32_t)h[1] << 8) | ((uint32_t)h[2] << 16) | ((uint32_t)h[3] << 24);
      }
#pragma unroll
      for (int j = 0; j < 32; j++) {
        const uint32_t nib = j < 16 ? (qs[j] & 15u) : (uint32_t)(qs[j - 16] >> 4);
        put(32 * b + j, nib | (((qh >> j) & 1u) << 4));
      }
      sc[2 * b] = sc[2 * b + 1] = d;
      of[2 * b] = of[2 * b + 1] = qtype == 6 ? -16.0f * d : (qtype == 3 || qtype == 7 ? h2f_at(blk + 2) : 0.f);
    }
  } else if (qtype == 10) {  // Q2_K: elements 64(c%4) .. +63 of the super-block
    const uint8_t* blk = row + (size_t)(c >> 2) * 84;
    const float d = h2f_at(blk + 80), dmin = h2f_at(blk + 82);
#pragma unroll
    for (int j = 0; j < 64; j++) {
      const int e = 64 * (c & 3) + j, g = e >> 7, t = (e & 127) >> 5, h = (e & 31) >> 4, l = e & 15;
      put(j, (uint32_t)(blk[16 + 32 * g + 16 * h + l] >> (2 * t)) & 3u);
      if ((j & 15) == 0) {
        const uint8_t sb = blk[8 * g + 2 * t + h];
        sc[j >> 4] = d * (float)(sb & 15);
        of[j >> 4] = -(dmin * (float)(sb >> 4));
      }
    }
  } else if (qtype == 15) {  // Q8_K: elements 64(c%4) .. +63 of the super-block
    const uint8_t* blk = row + (size_t)(c >> 2) * 292;
    float d;
    __builtin_memcpy(&d, blk, 4);
#pragma unroll
    for (int j = 0; j < 64; j++) put(j, (uint32_t)blk[4 + 64 * (c & 3) + j] ^ 0x80u);
#pragma unroll
    for (int g = 0; g < 4; g++) {
      sc[g] = d;
      of[g] = -128.0f * d;
    }
  } else if (qtype == 20) {  // IQ4_NL: blocks 2c and 2c+1 of 32 (DequantIQ.cs:46-76)
#pragma unroll
    for (int b = 0; b < 2; b++) {
      const uint8_t* blk = row + (size_t)(2 * c + b) * 18;
      const float d = h2f_at(blk);
#pragma unroll
      for (int j = 0; j < 16; j++) {
        put(32 * b + j, cn_iq4nl_code[blk[2 + j] & 15]);
        put(32 * b + 16 + j, cn_iq4nl_code[blk[2 + j] >> 4]);
      }
      sc[2 * b] = sc[2 * b + 1] = d;
      of[2 * b] = of[2 * b + 1] = -128.0f * d;
    }
  } else if (qtype == 23) {  // IQ4_XS: sub-blocks 2(c%4), 2(c%4)+1 (DequantIQ.cs:139-176)
    const uint8_t* blk = row + (size_t)(c >> 2) * 136;
    const float d = h2f_at(blk);
    const int sh = blk[2] | (blk[3] << 8);
#pragma unroll
    for (int b = 0; b < 2; b++) {
      const int s = 2 * (c & 3) + b;
      // low scale bits from byte 4+s (bytes 8..11 are sub-block 0's first quants)
      const int scv = ((blk[4 + s] & 0x3F) | (((sh >> (2 * s)) & 3) << 6)) - 32;
      const uint8_t* qs = blk + 8 + 16 * s;
#pragma unroll
      for (int j = 0; j < 16; j++) {
        put(32 * b + j, cn_iq4nl_code[qs[j] & 15]);
        put(32 * b + 16 + j, cn_iq4nl_code[qs[j] >> 4]);
      }
      sc[2 * b] = sc[2 * b + 1] = d * (float)scv;
      of[2 * b] = of[2 * b + 1] = -128.0f * sc[2 * b];
    }
  } else if (qtype == 21) {  // IQ3_S: elements 64(c%4) .. +63 (DequantIQ.cs:244-290)
    // sign bytes 98..129 and scale bytes 130..137 reach up to 28 bytes into the
    // next block; past the end of w they read as zero (the tail a model's
    // upload pads with)
    const size_t base = (size_t)r * row_bytes + (size_t)(c >> 2) * 110;
    auto at = [&](int off) -> uint32_t { return base + off < w_bytes ? w[base + off] : 0u; };
    const float d = h2f_at(w + base);
#pragma unroll
    for (int j = 0; j < 64; j++) {
      const int idx = 64 * (c & 3) + j, sub = idx >> 3;
      const int q3 = (int)(((at(2 + idx / 4) >> (2 * (idx % 4))) & 3u) | (((at(66 + idx / 8) >> (idx % 8)) & 1u) << 2));
      const int scv = (int)((at(130 + sub / 4) >> (2 * (sub % 4))) & 3u) + 1;
      const int v = ((at(98 + sub) >> (idx & 7)) & 1u) ? -scv * q3 : scv * q3;
      put(j, (uint32_t)(v + 128));
    }
#pragma unroll
    for (int g = 0; g < 4; g++) {
      sc[g] = d;
      of[g] = -128.0f * d;
    }
  } else if (qtype == 18) {  // IQ3_XXS: d * (q3 - 4) (DequantIQ.cs:364-399)
    const uint8_t* blk = row + (size_t)(c >> 2) * 98;
    const float d = h2f_at(blk);
#pragma unroll
    for (int j = 0; j < 64; j++) {
      const int idx = 64 * (c & 3) + j;
      const uint8_t* p = blk + 2 + 3 * (idx >> 3);
      const uint32_t word = (uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16);
      put(j, (word >> (3 * (idx & 7))) & 7u);
    }
#pragma unroll
    for (int g = 0; g < 4; g++) {
      sc[g] = d;
      of[g] = -4.0f * d;
    }
  } else if (qtype == 16 || qtype == 17 || qtype == 22) {  // IQ2_XXS / IQ2_XS / IQ2_S: sub-blocks 4(c%4) ..
    const int bb = qtype == 16 ? 66 : (qtype == 17 ? 74 : 82);
    const uint8_t* blk = row + (size_t)(c >> 2) * bb;
    const float d = h2f_at(blk);
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const int sub = 4 * (c & 3) + g;
      const uint8_t* qs = blk + 2 + 4 * sub;
      if (qtype == 22) {  // (d * (low nibble + 1)) * q, elements 0..3 signed (DequantIQ.cs:656-696)
        const uint32_t qh = blk[66 + sub];
#pragma unroll
        for (int e = 0; e < 16; e++) {
          const int q = (qs[e >> 2] >> (2 * (e & 3))) & 3;
          const bool neg = e < 4 && ((qh >> (4 + e)) & 1u);
          put(16 * g + e, (uint32_t)((neg ? -q : q) + 128));
        }
        sc[g] = d * (float)((qh & 15u) + 1);
        of[g] = -128.0f * sc[g];
      } else {  // d * (q - 1) or (d * sc) * (q - 1), sc a signed nibble - 8 (DequantIQ.cs:456-598)
#pragma unroll
        for (int e = 0; e < 16; e++) put(16 * g + e, (qs[e >> 2] >> (2 * (e & 3))) & 3u);
        float dsc = d;
        if (qtype == 17) {
          const int raw = (int8_t)blk[66 + sub / 2];
          dsc = d * (float)(((sub & 1) ? (raw >> 4) & 15 : raw & 15) - 8);
        }
        sc[g] = dsc;
        of[g] = -dsc;
      }
    }
  } else if (qtype == 19 || qtype == 29) {  // IQ1_S / IQ1_M: ternary (DequantIQ.cs:767-805, :869-914)
    const int bb = qtype == 19 ? 50 : 56;
    const uint8_t* blk = row + (size_t)(c >> 2) * bb;
    const float d = h2f_at(blk);
#pragma unroll
    for (int j = 0; j < 64; j++) {
      const int idx = 64 * (c & 3) + j, sub = idx >> 3, e = idx & 7;
      const int tv = ((blk[2 + sub] >> e) & 1) ? 1 : (((blk[34 + sub / 2] >> ((sub & 1) * 4 + e / 2)) & 1) ? -1 : 0);
      // IQ1_M: d * sc with sc 1 or 0.5 (bit sub%8 of byte 50 + sub/8) as (d/2) * (2 or 1)
      const int m = qtype == 19 ? 1 : (((blk[50 + sub / 8] >> (sub & 7)) & 1) ? 2 : 1);
      put(j, (uint32_t)(128 + tv * m));
    }
    const float step = qtype == 19 ? d : 0.5f * d;
#pragma unroll
    for (int g = 0; g < 4; g++) {
      sc[g] = step;
      of[g] = -128.0f * step;
    }
  }
  uint4* o = reinterpret_cast<uint4*>(dst + ((size_t)r * nchunks + c) * kGemmPackUnit);
#pragma unroll
  for (int i = 0; i < 4; i++) o[i] = make_uint4(code[4 * i], code[4 * i + 1], code[4 * i + 2], code[4 * i + 3]);
  o[4] = make_uint4(__float_as_uint(sc[0]), __float_as_uint(sc[1]), __float_as_uint(sc[2]), __float_as_uint(sc[3]));
  o[5] = make_uint4(__float_as_uint(of[0]), __float_as_uint(of[1]), __float_as_uint(of[2]), __float_as_uint(of[3]));
}

// Q6_K and Q3_K, whose 210- and 110-byte super-blocks start on 2-byte boundaries:
// one thread per 16 weights instead of 64, dword reads instead of bytes (a group
// of either type takes whole dwords of its quants), four threads writing a unit.
// Bound by memory (the stored blocks read, 1.5 bytes a weight written) and the
// scattered reads: 4096 x 4096 Q6_K 16.1 -> 11.0 us, Q3_K 30.7 -> 11.7.
typedef uint32_t pk_u32a2 __attribute__((aligned(2)));
template <bool Q6>
__global__ __launch_bounds__(CN_BLOCK) void gemm_pack16_kernel(const uint8_t* __restrict__ w, size_t row_bytes, int M,
                                                              int nchunks, uint8_t* __restrict__ dst) {
  const long long t = (long long)blockIdx.x * CN_BLOCK + threadIdx.x;
  const long long unit = t >> 2;
  if (unit >= (long long)M * nchunks) return;
  const int g = (int)(t & 3);
  const int r = (int)(unit / nchunks), c = (int)(unit % nchunks);
  const int G = 4 * (c & 3) + g;  // group of the super-block
  uint32_t code[4];
  float sc, of;
  if constexpr (Q6) {
    const uint8_t* blk = w + (size_t)r * row_bytes + (size_t)(c >> 2) * 210;
    const int h = G >> 3, qq = (G >> 1) & 3, lb = G & 1;
    const uint8_t* ql = blk + 64 * h + 32 * (qq & 1) + 16 * lb;
    const uint8_t* qh = blk + 128 + 32 * h + 16 * lb;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t l = *reinterpret_cast<const pk_u32a2*>(ql + 4 * k), u = *reinterpret_cast<const pk_u32a2*>(qh + 4 * k);
      code[k] = ((l >> (4 * (qq >> 1))) & 0x0F0F0F0Fu) | (((u >> (2 * qq)) & 0x03030303u) << 4);
    }
    sc = h2f_at(blk + 208) * (float)(int8_t)blk[192 + G];
    of = -32.0f * sc;
  } else {
    const uint8_t* blk = w + (size_t)r * row_bytes + (size_t)(c >> 2) * 110;
    const uint32_t q = *reinterpret_cast<const pk_u32a2*>(blk + 32 + 4 * G);
    const uint32_t hm = *reinterpret_cast<const uint16_t*>(blk + 2 * G);
#pragma unroll
    for (int k = 0; k < 4; k++) {  // element 4k + i: bits 2i of byte k, mask bit 4k + i
      const uint32_t b = (q >> (8 * k)) & 0xFFu;
      code[k] = ((b | (b << 6) | (b << 12) | (b << 18)) & 0x03030303u) | (spread4(hm >> (4 * k)) << 2);
    }
    const uint8_t* s = blk + 96;
    const int lo = G < 8 ? (s[G] & 15) : (s[G - 8] >> 4);
    sc = h2f_at(blk + 108) * (float)((lo | (((s[8 + (G & 3)] >> (2 * (G >> 2))) & 3) << 4)) - 32);
    of = -4.0f * sc;
  }
  uint8_t* o = dst + (size_t)unit * kGemmPackUnit;
  *reinterpret_cast<uint4*>(o + 16 * g) = make_uint4(code[0], code[1], code[2], code[3]);
  *reinterpret_cast<float*>(o + 64 + 4 * g) = sc;
  *reinterpret_cast<float*>(o + 80 + 4 * g) = of;
}

// Column tile by batch size and kernel.  One-plane kernel: see pick_gemm
// (at least 8 chunks of 64 per split).  Span kernel: 32 or 64 columns; a tile grid of more than two workgroups per CU
// takes the 2-stage ring (44 KB for raw Q4_0 at 64 columns, three workgroups
// per CU; 56 KB for packed units and Q8_0, two), a smaller one the 3-stage ring
// (two per CU), unless three stages leave one workgroup per CU (F16 against three
// planes, at 32 columns too: 11008 x 4096 at 24 39.8 -> 29.5 us; packed units,
// Q8_0, F16: 7B-shaped Q4_K_M 2 layers, 333 tokens 1428 -> 1363 us; F16 200
// tokens 887 -> 818), and a K split into the largest count that keeps the grid
// within one round of resident workgroups with at least 8 chunks per split (a
// grid just over a round would run a second round on a few CUs).  Rows of less
// than 32 chunks whose grid leaves CUs idle go down to 2 chunks per split
// (Qwen2-0.5B-shaped Q8_0, 6 layers: 6 tokens at 700 592 -> 488 us, 100 tokens
// 624 -> 500; at K = 2048 and more 2 to 4 % slower).
struct GemmShape {
  int tn, splits, stages, mt = 1;
  int sk_wgs = 0, sk_dp = 0;  // one-plane kernel: stream-K workgroups (0: none), of them whole-tile ones
  long long tiles = 0;
};

constexpr int kStages = 3;

int span_ring_bytes(int tn, int stages, int wf) {
  switch (wf) {
    case GEMM_W_PACKED: return span_ring_bytes_t<GEMM_W_PACKED>(tn, stages);
    case GEMM_W_F16: return span_ring_bytes_t<GEMM_W_F16>(tn, stages);
    case GEMM_W_F16_X3: return span_ring_bytes_t<GEMM_W_F16_X3>(tn, stages);
    case GEMM_W_F32: return span_ring_bytes_t<GEMM_W_F32>(tn, stages);
    case GEMM_W_Q4_K: return span_ring_bytes_t<GEMM_W_Q4_K>(tn, stages);
    case GEMM_W_Q8_0: return span_ring_bytes_t<GEMM_W_Q8_0>(tn, stages);
    case GEMM_W_Q5_0: return span_ring_bytes_t<GEMM_W_Q5_0>(tn, stages);
    case GEMM_W_Q4_1: return span_ring_bytes_t<GEMM_W_Q4_1>(tn, stages);
    case GEMM_W_Q5_1: return span_ring_bytes_t<GEMM_W_Q5_1>(tn, stages);
    case GEMM_W_IQ4_NL: return span_ring_bytes_t<GEMM_W_IQ4_NL>(tn, stages);
    case GEMM_W_IQ4_XS: return span_ring_bytes_t<GEMM_W_IQ4_XS>(tn, stages);
    default: return span_ring_bytes_t<GEMM_W_Q4_0>(tn, stages);
  }
}

GemmShape pick_gemm(int M, int N, int K, int num_cus, bool precise, int wf, bool stream_k = false) {
  GemmShape s;
  const int nchunks = K / 64;
  s.splits = 1;
  s.stages = kStages;
  if (precise) {
    s.tn = N <= 32 ? 1 : 2;
    const long long tiles = (long long)((M + 127) / 128) * ((N + 32 * s.tn - 1) / (32 * s.tn));
    s.stages = tiles > 2LL * num_cus || ((s.tn == 2 || wf == GEMM_W_F16_X3) && span_ring_bytes(s.tn, 3, wf) > 80 * 1024) ? 2 : 3;
    const int per_cu = std::max(1, std::min(3, 160 * 1024 / span_ring_bytes(s.tn, s.stages, wf)));
    const long long slots = (long long)per_cu * num_cus;
    while (s.splits < 16 && tiles * (s.splits + 1) <= slots &&
           (nchunks / (s.splits + 1) >= 8 || (nchunks < 32 && tiles * (s.splits + 1) <= num_cus && nchunks / (s.splits + 1) >= 2)))
      s.splits++;
  } else {
    // 32, 64 or 128 columns per workgroup.  Tiles of 64 and 128 columns run
    // the 2-stage ring (44 KB of LDS for raw Q4_0 at 128 columns: three
    // workgroups per CU, which hide each other's waits better than a deeper
    // ring with fewer workgroups) and split K only while the tile grid is
    // smaller than the CU count (a split's partials cost a reduce pass over
    // N x M x splits floats); 32-column tiles (N <= 32, HBM-bound) run a
    // 4-stage ring (40 KB) under the same split rule.  Measured per call,
    // 11008 x 4096 at N = 512: 93.6 us with 3 stages and splits up to two
    // workgroups per CU, 81.4 us with this rule; at N = 8: 20.4 us with 3
    // stages and that wider split, 17.8 us with this rule (6 and 8 stages:
    // 18.4, 18.9).
    s.tn = N <= 32 ? 1 : (N <= 64 ? 2 : 4);
    s.stages = s.tn == 1 ? 4 : 2;
    // Two 32-row tiles per wave (256-row workgroups, each x fragment read
    // from LDS feeding two MFMAs) where that still leaves a tile per CU:
    // 32000 x 2048 at N = 512, 96.7 -> 85.3 us per call; 11008 x 4096 (172
    // such tiles) went 79.3 -> 88.3 us and keeps one.
    // Stream-K for a grid of 128-row tiles just over one per CU (a partial
    // second round: 11008 x 4096 at N = 512 has 344 tiles, and 88 CUs ran
    // two while the rest idled): one whole tile per CU, and a second
    // workgroup per CU takes an equal share (at least 8 chunks) of the
    // remaining tiles' chunks.  Measured per call (same box, alternating
    // builds): 11008 x 4096 N = 512 74.4 -> 71.2 us, N = 480 74.2 -> 70.6;
    // at 448 tiles (14336 x 4096) 82.1 -> 87.1, so only up to 1.4 tiles per
    // CU.  Sharing every tile of a smaller grid this way instead of splitting
    // K measured slower than the split and its reduce pass (4096 x 4096 N =
    // 512 41.5 -> 46.3 us, N = 8 11008 x 4096 18.7 -> 21.0): a shared tile's
    // parts cost device-scope round trips (store, arrival, reads).
    const long long tiles1 = (long long)((M + 127) / 128) * ((N + 32 * s.tn - 1) / (32 * s.tn));
    if (stream_k && tiles1 > num_cus && tiles1 <= kGemmTileCounters && tiles1 * 5 <= 7LL * num_cus &&
        (tiles1 - num_cus) * nchunks / num_cus >= 8) {
      s.tiles = tiles1;
      s.sk_dp = num_cus;
      s.sk_wgs = 2 * num_cus;
      return s;
    }
    if (s.tn == 4 && (long long)((M + 255) / 256) * ((N + 127) / 128) >= num_cus) s.mt = 2;
    const long long tiles = (long long)((M + 128 * s.mt - 1) / (128 * s.mt)) * ((N + 32 * s.tn - 1) / (32 * s.tn));
    s.tiles = tiles;
    const long long want = num_cus;
    while (tiles * s.splits < want && nchunks / (s.splits * 2) >= 8 && s.splits < 16) s.splits *= 2;
  }
  return s;
}

hipError_t launch_kernel(const GemmArgs& a, const GemmShape& s, bool precise, int grid, hipStream_t st) {
  switch (a.packed) {
    case GEMM_W_Q4_0: return precise ? gemm_q4_0_span(a, s.tn, s.stages, grid, st) : gemm_q4_0_plane(a, s.tn, s.mt, grid, st);
    case GEMM_W_PACKED: return precise ? gemm_packed_span(a, s.tn, s.stages, grid, st) : gemm_packed_plane(a, s.tn, s.mt, grid, st);
    case GEMM_W_F16: return precise ? gemm_f16_span(a, s.tn, s.stages, grid, st) : hipErrorInvalidValue;
    case GEMM_W_F16_X3: return precise ? gemm_f16_x3_span(a, s.tn, s.stages, grid, st) : hipErrorInvalidValue;
    case GEMM_W_F32: return precise ? gemm_f32_span(a, s.tn, s.stages, grid, st) : hipErrorInvalidValue;
    case GEMM_W_Q4_K: return precise ? gemm_q4_k_span(a, s.tn, s.stages, grid, st) : gemm_q4_k_plane(a, s.tn, s.mt, grid, st);
    case GEMM_W_Q8_0: return precise ? gemm_q8_0_span(a, s.tn, s.stages, grid, st) : gemm_q8_0_plane(a, s.tn, s.mt, grid, st);
    case GEMM_W_Q5_0: return precise ? gemm_q5_0_span(a, s.tn, s.stages, grid, st) : gemm_q5_0_plane(a, s.tn, s.mt, grid, st);
    case GEMM_W_Q4_1: return precise ? gemm_q4_1_span(a, s.tn, s.stages, grid, st) : gemm_q4_1_plane(a, s.tn, s.mt, grid, st);
    case GEMM_W_Q5_1: return precise ? gemm_q5_1_span(a, s.tn, s.stages, grid, st) : gemm_q5_1_plane(a, s.tn, s.mt, grid, st);
    case GEMM_W_IQ4_NL: return precise ? gemm_iq4_nl_span(a, s.tn, s.stages, grid, st) : gemm_iq4_nl_plane(a, s.tn, s.mt, grid, st);
    case GEMM_W_Q5_K: return precise ? hipErrorInvalidValue : gemm_q5_k_plane(a, s.tn, s.mt, grid, st);
    case GEMM_W_IQ4_XS: return precise ? gemm_iq4_xs_span(a, s.tn, s.stages, grid, st) : gemm_iq4_xs_plane(a, s.tn, s.mt, grid, st);
    case GEMM_W_Q2_K: return precise ? hipErrorInvalidValue : gemm_q2_k_plane(a, s.tn, s.mt, grid, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

int gemm_stored_format(int qtype, int K) {
  if (K <= 0 || K % 64) return -1;
  const bool sb = K % 256 == 0;
  switch (qtype) {
    case 0: return GEMM_W_F32;
    case 1: return GEMM_W_F16;
    case 2: return GEMM_W_Q4_0;
    case 3: return GEMM_W_Q4_1;
    case 6: return GEMM_W_Q5_0;
    case 7: return GEMM_W_Q5_1;
    case 8: return GEMM_W_Q8_0;
    case 10: return sb ? GEMM_W_Q2_K : -1;
    case 12: return sb ? GEMM_W_Q4_K : -1;
    case 13: return sb ? GEMM_W_Q5_K : -1;
    case 20: return GEMM_W_IQ4_NL;
    case 23: return sb ? GEMM_W_IQ4_XS : -1;
    default: return -1;
  }
}

// The span kernel is bound by VALU instructions, of which packed units take the
// fewest, and at 2.3 to 3.4 times the bytes the stored blocks win where those are
// cheap to unpack.  Q5_K and Q2_K are not (layers of a 7B shape, packed and stored,
// us: Q5_K 512 tokens 876 and 937, 64 230 and 238; of a 1.1B shape, 3 layers, 748 and
// 786, 64 294 and 341; Q2_K 857 and 986, 734 and 823); IQ4 is for rows of 4096 and
// more (IQ4_XS, 7B shape, 200 tokens 532 and 488, 16 185 and 176) and below 2048,
// where K splits go deeper (IQ4_NL, K = 896, 64 tokens 381 and 303), but not between
// (1.1B shape, 512 tokens 759 and 739, 64 292 and 311, 16 249 and 269).
int gemm_span_format(int qtype, int K) {
  if (qtype == 10 || qtype == 13) return -1;
  if ((qtype == 20 || qtype == 23) && K >= 2048 && K < 4096) return -1;
  return gemm_stored_format(qtype, K);
}

bool gemm_pack_supports(int qtype, int K) {
  if (K <= 0) return false;
  if (qtype == 2 || qtype == 3 || qtype == 6 || qtype == 7 || qtype == 8 || qtype == 20) return K % 64 == 0;
  if ((qtype >= 10 && qtype <= 19) || (qtype >= 21 && qtype <= 23) || qtype == 29) return K % 256 == 0;
  return false;
}

size_t gemm_pack_bytes(int M, int K) { return (size_t)M * (size_t)(K / 64) * kGemmPackUnit; }

hipError_t gemm_pack_launch(int qtype, const void* w, int M, int K, void* dst, hipStream_t st) {
  if (!gemm_pack_supports(qtype, K) || M <= 0 || !w || !dst) return hipErrorInvalidValue;
  size_t row_bytes;
  switch (qtype) {
    case 2: row_bytes = (size_t)K / 32 * 18; break;
    case 3: row_bytes = (size_t)K / 32 * 20; break;
    case 6: row_bytes = (size_t)K / 32 * 22; break;
    case 7: row_bytes = (size_t)K / 32 * 24; break;
    case 8: row_bytes = (size_t)K / 32 * 34; break;
    case 10: row_bytes = (size_t)K / 256 * 84; break;
    case 11: row_bytes = (size_t)K / 256 * 110; break;
    case 12: row_bytes = (size_t)K / 256 * 144; break;
    case 13: row_bytes = (size_t)K / 256 * 176; break;
    case 15: row_bytes = (size_t)K / 256 * 292; break;
    case 16: row_bytes = (size_t)K / 256 * 66; break;
    case 17: row_bytes = (size_t)K / 256 * 74; break;
    case 18: row_bytes = (size_t)K / 256 * 98; break;
    case 19: row_bytes = (size_t)K / 256 * 50; break;
    case 20: row_bytes = (size_t)K / 32 * 18; break;
    case 21: row_bytes = (size_t)K / 256 * 110; break;
    case 22: row_bytes = (size_t)K / 256 * 82; break;
    case 23: row_bytes = (size_t)K / 256 * 136; break;
    case 29: row_bytes = (size_t)K / 256 * 56; break;
    default: row_bytes = (size_t)K / 256 * 210; break;
  }
  const long long n = (long long)M * (K / 64);
  const long long blocks = (n + CN_BLOCK - 1) / CN_BLOCK;
  if (blocks > 0x7FFFFFFF) return hipErrorInvalidValue;
  if (qtype == 11 || qtype == 14) {
    if (4 * blocks > 0x7FFFFFFF) return hipErrorInvalidValue;  // 2^39 weights and more
    const dim3 grid((unsigned)((4 * n + CN_BLOCK - 1) / CN_BLOCK));
    const uint8_t* wb = static_cast<const uint8_t*>(w);
    uint8_t* to = static_cast<uint8_t*>(dst);
    if (qtype == 14) hipLaunchKernelGGL((gemm_pack16_kernel<true>), grid, dim3(CN_BLOCK), 0, st, wb, row_bytes, M, K / 64, to);
    else hipLaunchKernelGGL((gemm_pack16_kernel<false>), grid, dim3(CN_BLOCK), 0, st, wb, row_bytes, M, K / 64, to);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(gemm_pack_kernel, dim3((unsigned)blocks), dim3(CN_BLOCK), 0, st, qtype,
                     static_cast<const uint8_t*>(w), row_bytes, (size_t)M * row_bytes, M, K / 64,
                     static_cast<uint8_t*>(dst));
  return hipGetLastError();
}

size_t gemm_workspace_bytes(int M, int N, int K, int num_cus, bool precise, int wfmt, bool stream_k) {
  const GemmShape s = pick_gemm(M, N, K, num_cus, precise, wfmt, stream_k && !precise);
  if (s.sk_wgs > 0) return (size_t)2 * s.sk_wgs * (128 * s.mt) * (32 * s.tn) * sizeof(float);
  return s.splits > 1 ? (size_t)s.splits * N * M * sizeof(float) : 0;
}

hipError_t gemm_launch(const GemmArgs& a_in, int num_cus, hipStream_t st, int* splits_left) {
  if (a_in.packed < GEMM_W_Q4_0 || a_in.packed >= GEMM_W_COUNT) return hipErrorInvalidValue;
  if ((a_in.packed == GEMM_W_F16 || a_in.packed == GEMM_W_F16_X3 || a_in.packed == GEMM_W_F32) && !a_in.precise)
    return hipErrorInvalidValue;  // float rows only in the span kernel
  if (a_in.packed == GEMM_W_F16_X3 && (!a_in.xb_ll || !a_in.x32)) return hipErrorInvalidValue;
  const bool blocks = a_in.packed == GEMM_W_Q4_K || a_in.packed == GEMM_W_Q5_K || a_in.packed == GEMM_W_IQ4_XS ||
                      a_in.packed == GEMM_W_Q2_K;
  if (a_in.K <= 0 || a_in.K % (blocks ? 256 : 64) || a_in.M <= 0 || a_in.N <= 0) return hipErrorInvalidValue;
  const bool precise = a_in.precise != 0;
  if (precise && !a_in.xb_lo) return hipErrorInvalidValue;
  // partials can be left only for a store or a residual add (the folding
  // kernels apply no other epilogue)
  if (splits_left && a_in.epi != GEMV_EPI_STORE && a_in.epi != GEMV_EPI_ADD) return hipErrorInvalidValue;
  if (a_in.epi == GEMV_EPI_SWIGLU && (!a_in.hb || !a_in.hb_lo)) return hipErrorInvalidValue;
  const GemmShape s =
      pick_gemm(a_in.M, a_in.N, a_in.K, num_cus, precise, a_in.packed, a_in.tile_cnt != nullptr && !precise);
  GemmArgs a = a_in;
  a.splits = s.splits;
  a.sk_wgs = s.sk_wgs;
  a.sk_dp = s.sk_dp;
  a.sk_tiles = (int)s.tiles;
  if ((s.splits > 1 || s.sk_wgs > 0) && !a.part) return hipErrorInvalidValue;
  const long long grid = s.sk_wgs > 0 ? s.sk_wgs
                                      : (long long)((a.M + 128 * s.mt - 1) / (128 * s.mt)) *
                                            ((a.N + 32 * s.tn - 1) / (32 * s.tn)) * s.splits;
  if (grid > 0x7FFFFFFF) return hipErrorInvalidValue;
  hipError_t e = launch_kernel(a, s, precise, (int)grid, st);
  if (splits_left) *splits_left = 0;
  if (e != hipSuccess || s.splits == 1) return e;
  if (splits_left) {  // the caller folds the partials into its next kernel
    *splits_left = s.splits;
    return hipSuccess;
  }
  const long long work = (long long)((a.M + 3) / 4) * a.N;
  const dim3 rgrid((unsigned)((work + CN_BLOCK - 1) / CN_BLOCK));
  if (a.packed == GEMM_W_F16_X3) hipLaunchKernelGGL((gemm_reduce_kernel<true>), rgrid, dim3(CN_BLOCK), 0, st, a);
  else hipLaunchKernelGGL((gemm_reduce_kernel<false>), rgrid, dim3(CN_BLOCK), 0, st, a);
  return hipGetLastError();
}

hipError_t to_f16_scaled_launch(const float* x, uint16_t* xh, float* xinv, int N, int K, hipStream_t st) {
  if (N <= 0 || K <= 0 || K % 32 || K > 16384) return hipErrorInvalidValue;
  const int v = (K + 4 * CN_BLOCK - 1) / (4 * CN_BLOCK);  // float4 per thread
  const dim3 grid(N), block(CN_BLOCK);
  if (v <= 2) hipLaunchKernelGGL((to_f16_scaled_kernel<2>), grid, block, 0, st, x, xh, xinv, K);
  else if (v <= 4) hipLaunchKernelGGL((to_f16_scaled_kernel<4>), grid, block, 0, st, x, xh, xinv, K);
  else if (v <= 8) hipLaunchKernelGGL((to_f16_scaled_kernel<8>), grid, block, 0, st, x, xh, xinv, K);
  else hipLaunchKernelGGL((to_f16_scaled_kernel<16>), grid, block, 0, st, x, xh, xinv, K);
  return hipGetLastError();
}

hipError_t to_f16_planes_launch(const float* x, uint16_t* xp, size_t plane, float* xinv, int N, int K, hipStream_t st) {
  if (N <= 0 || K <= 0 || K % 32 || K > 16384) return hipErrorInvalidValue;
  const int v = (K + 4 * CN_BLOCK - 1) / (4 * CN_BLOCK);  // float4 per thread
  const dim3 grid(N), block(CN_BLOCK);
  if (v <= 2) hipLaunchKernelGGL((to_f16_planes_kernel<2>), grid, block, 0, st, x, xp, plane, xinv, K);
  else if (v <= 4) hipLaunchKernelGGL((to_f16_planes_kernel<4>), grid, block, 0, st, x, xp, plane, xinv, K);
  else if (v <= 8) hipLaunchKernelGGL((to_f16_planes_kernel<8>), grid, block, 0, st, x, xp, plane, xinv, K);
  else hipLaunchKernelGGL((to_f16_planes_kernel<16>), grid, block, 0, st, x, xp, plane, xinv, K);
  return hipGetLastError();
}

template <int V>
void add_rmsnorm_v(float* x, const float* part, int splits, const float* g, float eps, uint16_t* xb, uint16_t* xb_lo,
                   int rows, int dim, hipStream_t st) {
  const dim3 grid(rows), block(CN_BLOCK);
  if (V > 4 || splits <= 0) {  // wide rows: the norm alone (no partials folded)
    hipLaunchKernelGGL((add_rmsnorm_span_kernel<V, 0>), grid, block, 0, st, x, part, 0, g, eps, xb, xb_lo, rows, dim);
    return;
  }
  if constexpr (V <= 4) {
  if (splits <= 0) hipLaunchKernelGGL((add_rmsnorm_span_kernel<V, 0>), grid, block, 0, st, x, part, 0, g, eps, xb, xb_lo, rows, dim);
  else if (splits <= 2) hipLaunchKernelGGL((add_rmsnorm_span_kernel<V, 2>), grid, block, 0, st, x, part, splits, g, eps, xb, xb_lo, rows, dim);
  else if (splits <= 4) hipLaunchKernelGGL((add_rmsnorm_span_kernel<V, 4>), grid, block, 0, st, x, part, splits, g, eps, xb, xb_lo, rows, dim);
  else if (splits <= 8) hipLaunchKernelGGL((add_rmsnorm_span_kernel<V, 8>), grid, block, 0, st, x, part, splits, g, eps, xb, xb_lo, rows, dim);
  else hipLaunchKernelGGL((add_rmsnorm_span_kernel<V, 16>), grid, block, 0, st, x, part, splits, g, eps, xb, xb_lo, rows, dim);
  }
}

hipError_t add_rmsnorm_span_launch(float* x, const float* part, int splits, const float* g, float eps, uint16_t* xb,
                                   uint16_t* xb_lo, int rows, int dim, hipStream_t st) {
  if (dim % 4 || dim <= 0 || rows <= 0 || splits > 16 || (splits > 0 && !part)) return hipErrorInvalidValue;
  if (!xb || !xb_lo || dim % 32) return hipErrorInvalidValue;  // the span order permutes blocks of 32
  const int v = (dim + 4 * CN_BLOCK - 1) / (4 * CN_BLOCK);  // float4 per thread
  // at most 4 float4 per thread when partials are folded (the register budget of
  // 16 splits x 4 float4), 16 for the norm alone
  if (splits > 0 && v > 4) return hipErrorInvalidValue;
  if (v > 16) return hipErrorInvalidValue;
  if (v <= 2) add_rmsnorm_v<2>(x, part, splits, g, eps, xb, xb_lo, rows, dim, st);
  else if (v <= 4) add_rmsnorm_v<4>(x, part, splits, g, eps, xb, xb_lo, rows, dim, st);
  else if (v <= 8) add_rmsnorm_v<8>(x, part, 0, g, eps, xb, xb_lo, rows, dim, st);
  else add_rmsnorm_v<16>(x, part, 0, g, eps, xb, xb_lo, rows, dim, st);
  return hipGetLastError();
}


// gemv_mcol.h — a few columns of x (2 to 16) against the same quantized rows on
// the int8 matrix cores, instantiated per weight type by the gemv_*.hip files.
//
// x is held as base-256 digits: per 32-element block and column a power of two
// brings the largest |x| to 31 bits, X = D3 2^24 + D2 2^16 + D1 2^8 + D0 with signed
// bytes D.  Four digits of N columns are 4N rows of an int8 operand, so one
// v_mfma_i32_16x16x32_i8 multiplies a 32-element block of 16 weight rows (their
// codes as signed bytes) with four columns exactly.  The four int32 results of a
// lane are one column's digits of one weight row (the weight rows are the operand
// whose index the lane keeps, lane % 16): joined as (D3 2^8 + D2) + (D1 2^8 + D0)
// 2^-16 in fp32, they are scaled by the row's block scale, where its
// codes were unpacked, and the column's 2^-e.  31 bits of a block's largest are 12
// more than the single-column GEMV keeps of 16 elements' (three digits, 23 bits,
// fell short of it where the halves of a block differ by more than 16 times).
//
// What bounds it: joining, scaling and adding the digits (7 VALU instructions for 16
// rows x 32 weights x 4 columns); dot4 on packed digits took 21 per 16 weights and
// column, one launch per column the weight stream N times (per library call, calls
// back to back: 18.9 us at 5 columns of
// Q8_0 4864 x 896, here 5.3; the MFMA GEMM behind its packing pass 67.7 at 16 of Q4_K
// 11008 x 4096, here 24.5).  Three digits, whose
// results met a column at a time in fp32, took 12 for 5 columns: Q4_K 4096 x 4096 at
// 4 columns 9.5 -> 7.0 us, at 5 10.4 -> 8.7, at 16 14.6 -> 14.8, Q8_0 4864 x 896 at
// 5 6.6 -> 5.3, Q6_K 11008 x 4096 at 5 26.8 -> 30.8; error against float64 2.0e-7 ->
// 1.0e-7 (Q8_0).
#pragma once
#include "gemv_quant.h"

namespace {

typedef int mc_i32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t mc_u32a2 __attribute__((aligned(2)));  // a dword on a 2-byte boundary

// Types with a scale per 16 weights: each half of a block is a product of its own.
template <int QT>
constexpr bool mc_half_scales() { return QT == QT_Q2_K || QT == QT_Q3_K || QT == QT_Q6_K; }
// Dwords a lane loads per 128 weights of a row.
template <int QT>
constexpr int mc_raw() {
  return QT == QT_Q4_1 || QT == QT_IQ4_NL ? 5 : QT == QT_Q5_0 || QT == QT_Q5_1 ? 6 : QT == QT_Q8_0 ? 9
         : QT == QT_Q2_K ? 5 : QT == QT_Q3_K ? 16 : QT == QT_Q4_K ? 8 : QT == QT_Q5_K ? 9 : QT == QT_IQ4_XS ? 7 : 9;
}

// 4 x 4 transpose over the wave's rows of 16 lanes: lane group g holding dwords
// 0..3 of its own block ends with dword g of blocks 0..3.
__device__ __forceinline__ void mc_swap32(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
__device__ __forceinline__ void mc_swap16(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
__device__ __forceinline__ void mc_transpose(uint32_t& r0, uint32_t& r1, uint32_t& r2, uint32_t& r3) {
  mc_swap32(r0, r2);
  mc_swap32(r1, r3);
  mc_swap16(r0, r1);
  mc_swap16(r2, r3);
}
// out[g] = lane group g's v, in every group.
__device__ __forceinline__ void mc_spread(uint32_t v, uint32_t (&out)[4]) {
  uint32_t lo = v, hi = v;
  mc_swap32(lo, hi);  // groups 0 1 0 1 | groups 2 3 2 3
  out[0] = out[1] = lo;
  out[2] = out[3] = hi;
  mc_swap16(out[0], out[1]);
  mc_swap16(out[2], out[3]);
}

// What lane group p reads of weights 128s .. 128s+127 of a row, every load
// inside the row (blocks past its end re-read the last one).
//   32-weight types: block 4s + p whole, as the dword-aligned window that covers
//   it (18-, 22- and 34-byte blocks start on 2-byte boundaries when odd; a row
//   holds an even number of them, so an even block's window ends in the next).
//   Super-blocks: the half's header or scales, and a quarter of its quants.
template <int QT>
__device__ __forceinline__ void mc_load(const cn_gbyte* row, int s, int p, int K, uint32_t* r) {
  constexpr int NR = mc_raw<QT>();
  if constexpr (QTraits<QT>::BLOCK == 32) {
    const int b = min(4 * s + p, K / 32 - 1);
    constexpr int BB = QTraits<QT>::BLOCK_BYTES;
    const int off = b * BB - ((BB & 3) ? 2 * (b & 1) : 0);
    const CN_GLOBAL uint32_t* q = (const CN_GLOBAL uint32_t*)(row + off);
#pragma unroll
    for (int k = 0; k < NR; k++) r[k] = q[k];
  } else {
    const int h = s & 1;
    const cn_gbyte* sb = row + (size_t)(s >> 1) * QTraits<QT>::BLOCK_BYTES;
    auto dw = [&](int byte) { return *(const CN_GLOBAL uint32_t*)(sb + byte); };
    auto dw2 = [&](int byte) { return (uint32_t)*(const CN_GLOBAL mc_u32a2*)(sb + byte); };
    if constexpr (QT == QT_Q4_K || QT == QT_Q5_K) {
      load_u32x4(sb, r);
      load_u32x4(sb + (QT == QT_Q4_K ? 16 : 48) + 64 * h + 16 * p, r + 4);
      if constexpr (QT == QT_Q5_K) r[8] = dw(16 + 16 * h + 4 * p);
    } else if constexpr (QT == QT_IQ4_XS) {
#pragma unroll
      for (int k = 0; k < 3; k++) r[k] = dw(4 * k);
#pragma unroll
      for (int k = 0; k < 4; k++) r[3 + k] = dw(8 + 64 * h + 16 * p + 4 * k);
    } else if constexpr (QT == QT_Q2_K) {
      r[0] = dw(16 + 32 * h + 4 * p);
      r[1] = dw(32 + 32 * h + 4 * p);
      r[2] = dw(8 * h);
      r[3] = dw(8 * h + 4);
      r[4] = dw(80);
    } else if constexpr (QT == QT_Q6_K) {
#pragma unroll
      for (int k = 0; k < 4; k++) r[k] = dw2(64 * h + 16 * p + 4 * k);
      r[4] = dw2(128 + 32 * h + 4 * p);
      r[5] = dw2(144 + 32 * h + 4 * p);
      r[6] = dw2(192 + 8 * h);
      r[7] = dw2(196 + 8 * h);
      r[8] = *(const CN_GLOBAL uint16_t*)(sb + 208);
    } else {  // Q3_K: every lane group unpacks its two bits of the same dwords
#pragma unroll
      for (int k = 0; k < 8; k++) r[k] = dw2(32 + 32 * h + 4 * k);
#pragma unroll
      for (int k = 0; k < 4; k++) r[8 + k] = dw2(16 * h + 4 * k);
#pragma unroll
      for (int k = 0; k < 3; k++) r[12 + k] = dw2(96 + 4 * k);
      r[15] = *(const CN_GLOBAL uint16_t*)(sb + 108);
    }
  }
}

// Four blocks of 32 weights of the lane's row: q[b][0] the codes (signed bytes) of
// elements 4p .. 4p+3 of block b, q[b][1] those of 16+4p .. 16+4p+3 (Q3_K: of
// elements p, 4+p, 8+p, 12+p of each half), scale a and offset b per block, or
// per half where the type scales 16 weights.  Blocks past the row's end (nblk
// valid ones) get scale 0.
template <int QT>
__device__ __forceinline__ void mc_expand(uint32_t* r, int s, int p, int nblk, uint32_t (&q)[4][2], float (&a)[4][2],
                                          float (&b)[4][2]) {
  const int h = s & 1;
  constexpr uint32_t LO = 0x0F0F0F0Fu, S8 = 0x80808080u;
  if constexpr (QTraits<QT>::BLOCK == 32) {
    uint32_t sc[4];  // d, or d | m << 16, of each block
    uint32_t qs[8];
    uint32_t qh[4] = {0, 0, 0, 0};
    const uint32_t sh = 2 * (p & 1);  // block 4s + p: odd where p is (a clamped block has scale 0)
    if constexpr (QT == QT_Q4_1 || QT == QT_Q5_1) {
      mc_spread(r[0], sc);
      if constexpr (QT == QT_Q5_1) mc_spread(r[1], qh);
#pragma unroll
      for (int k = 0; k < 4; k++) qs[k] = r[k + (QT == QT_Q5_1 ? 2 : 1)];
    } else {
      // realigned: d in the first two bytes, the rest from byte 2
      uint32_t t[mc_raw<QT>()];
      constexpr int NR = mc_raw<QT>();
#pragma unroll
      for (int k = 0; k < NR; k++) t[k] = k + 1 < NR ? __builtin_amdgcn_alignbyte(r[k + 1], r[k], sh) : r[k] >> (8 * sh);
      mc_spread(t[0], sc);
#pragma unroll
      for (int k = 0; k + 1 < NR; k++) t[k] = __builtin_amdgcn_alignbyte(t[k + 1], t[k], 2);
      if constexpr (QT == QT_Q5_0) {
        mc_spread(t[0], qh);
#pragma unroll
        for (int k = 0; k < 4; k++) qs[k] = t[1 + k];
      } else {
#pragma unroll
        for (int k = 0; k < (QT == QT_Q8_0 ? 8 : 4); k++) qs[k] = t[k];
      }
    }
    mc_transpose(qs[0], qs[1], qs[2], qs[3]);
    if constexpr (QT == QT_Q8_0) mc_transpose(qs[4], qs[5], qs[6], qs[7]);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      if constexpr (QT == QT_Q8_0) {
        q[i][0] = qs[i];
        q[i][1] = qs[4 + i];
      } else {
        q[i][0] = qs[i] & LO;
        q[i][1] = (qs[i] >> 4) & LO;
        if constexpr (QT == QT_Q5_0 || QT == QT_Q5_1) {
          q[i][0] |= spread4(qh[i] >> (4 * p)) << 4;
          q[i][1] |= spread4(qh[i] >> (16 + 4 * p)) << 4;
        }
        if constexpr (QT == QT_Q5_0) {  // q5 - 16 as signed bytes
          q[i][0] = (q[i][0] + 0x70707070u) ^ S8;
          q[i][1] = (q[i][1] + 0x70707070u) ^ S8;
        }
        if constexpr (QT == QT_IQ4_NL) {
          q[i][0] = iq4_values(q[i][0]);
          q[i][1] = iq4_values(q[i][1]);
        }
      }
      const bool in = i < nblk;
      a[i][0] = in ? cn_h2f(sc[i]) : 0.f;
      b[i][0] = in ? cn_h2f(sc[i] >> 16) : 0.f;  // used by Q4_1 and Q5_1 only
    }
  } else if constexpr (QT == QT_Q4_K || QT == QT_Q5_K) {
    // the lane's own sub-block 4h + p: 6-bit scale and min (DequantQ4K.cs:218-241)
    const uint32_t b0 = r[1] >> (8 * p), b4 = r[2] >> (8 * p), b8 = r[3] >> (8 * p);
    const uint32_t sv = h ? (b8 & 0xFu) | ((b0 >> 2) & 0x30u) : b0 & 63u;
    const uint32_t mv = h ? ((b8 >> 4) & 0xFu) | ((b4 >> 2) & 0x30u) : b4 & 63u;
    uint32_t sm[4], qh[4];
    mc_spread(sv | (mv << 8), sm);
    if constexpr (QT == QT_Q5_K) mc_spread(r[8], qh);
    mc_transpose(r[4], r[5], r[6], r[7]);
    const float d = cn_h2f(r[0]), dmin = cn_h2f(r[0] >> 16);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      q[i][0] = r[4 + i] & LO;
      q[i][1] = (r[4 + i] >> 4) & LO;
      if constexpr (QT == QT_Q5_K) {
        q[i][0] |= spread4(qh[i] >> (4 * p)) << 4;
        q[i][1] |= spread4(qh[i] >> (16 + 4 * p)) << 4;
      }
      a[i][0] = d * cn_ubyte<0>(sm[i]);
      b[i][0] = -(dmin * cn_ubyte<1>(sm[i]));
    }
  } else if constexpr (QT == QT_IQ4_XS) {
    const uint32_t lo = ((h ? r[2] : r[1]) >> (8 * p)) & 0x3Fu, hi = (r[0] >> (16 + 8 * h + 2 * p)) & 3u;
    uint32_t sc[4];
    mc_spread(__float_as_uint(cn_h2f(r[0]) * (float)((int)(lo | (hi << 6)) - 32)), sc);
    mc_transpose(r[3], r[4], r[5], r[6]);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      q[i][0] = iq4_values(r[3 + i] & LO);
      q[i][1] = iq4_values((r[3 + i] >> 4) & LO);
      a[i][0] = __uint_as_float(sc[i]);
    }
  } else if constexpr (QT == QT_Q2_K) {  // block t: bits 2t; scale byte 2t + half
    const float d = cn_h2f(r[4]), dmin = cn_h2f(r[4] >> 16);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int k = 0; k < 2; k++) {
        q[i][k] = (r[k] >> (2 * i)) & 0x03030303u;
        const uint32_t sb = (r[2 + (i >> 1)] >> (16 * (i & 1) + 8 * k)) & 0xFFu;
        a[i][k] = d * (float)(sb & 15u);
        b[i][k] = -(dmin * (float)(sb >> 4));
      }
  } else if constexpr (QT == QT_Q6_K) {  // block qq: ql dwords p, 4 + p of its 32 bytes, qh bits 2qq
    mc_transpose(r[0], r[1], r[2], r[3]);  // ql dwords p, 4+p, 8+p, 12+p of the half
    const float d = cn_h2f(r[8]);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int k = 0; k < 2; k++) {
        const uint32_t ql = r[2 * (i & 1) + k], v = ((i < 2 ? ql : (ql >> 4)) & LO) | (((r[4 + k] >> (2 * i)) & 0x03030303u) << 4);
        q[i][k] = (v + 0x60606060u) ^ S8;  // q - 32
        a[i][k] = d * (float)(int8_t)((r[6 + (i >> 1)] >> (16 * (i & 1) + 8 * k)) & 0xFF);
      }
  } else {  // Q3_K: group 2i + k's dword, bits 2p: elements 4j + p in byte j
    const float d = cn_h2f(r[15]);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int k = 0; k < 2; k++) {
        const int g = 2 * i + k;
        uint32_t hs = (r[8 + (g >> 1)] >> (16 * (g & 1))) & 0xFFFFu;
        hs = (hs | (hs << 8)) & 0x00FF00FFu;
        hs = (hs | (hs << 4)) & LO;  // 4 mask bits per byte: element 4j + w at bit w of byte j
        const uint32_t v = ((r[g] >> (2 * p)) & 0x03030303u) | (((hs >> p) & 0x01010101u) << 2);
        q[i][k] = (v + 0x7C7C7C7Cu) ^ S8;  // q - 4
        const uint32_t lob = (r[12 + (g >> 2)] >> (8 * (g & 3))) >> (4 * h);
        const uint32_t hib = r[14] >> (8 * (g & 3) + 4 * h + 2 * (g >> 2));
        a[i][k] = d * (float)((int)((lob & 15u) | ((hib & 3u) << 4)) - 32);
      }
  }
}

constexpr int kMcTile = 4;  // columns of a tile of 16 digit rows

// LDS bytes of one staged 32-element block and tile: the digits in operand order,
// 2^(16 - e) per column, and for the types with an offset the sum of its x, per half
// where the scales are.
template <int QT>
constexpr int mc_block_bytes() { return 512 + 16 + (group_min<QT>() ? (mc_half_scales<QT>() ? 32 : 16) : 0); }

// Sixteen elements (half hb & 1 of block hb / 2) of column c into the staged
// blocks at `base`.  The block's two halves are on adjacent lanes.  A
// non-finite element makes the block's 2^-e NaN, and so the column's sums.
template <int QT, int CT>
__device__ __forceinline__ void mc_stage(const float (&v)[16], int c, int hb, char* base) {
  constexpr int BB = mc_block_bytes<QT>();
  constexpr bool HALF = mc_half_scales<QT>(), MIN = group_min<QT>(), TR = QT == QT_Q3_K;
  uint32_t mb = 0;  // magnitudes as bits: infinities and NaN compare above every number
#pragma unroll
  for (int j = 0; j < 16; j++) mb = max(mb, __float_as_uint(v[j]) & 0x7FFFFFFFu);
  mb = max(mb, (uint32_t)__shfl_xor((int)mb, 1, CN_WAVE));  // the block's other half
  const bool finite = mb < 0x7F800000u;
  int e = 0;
  const float f = frexpf(__uint_as_float(mb), &e);
  const int sc = mb == 0 || !finite ? 0 : (f > 0.996f ? 30 : 31) - e;  // |X| <= 0x7F7F7F7F, the digits' range
  uint32_t U[16];
#pragma unroll
  for (int j = 0; j < 16; j++)
    U[j] = (uint32_t)(int)rintf(finite ? ldexpf(v[j], sc) : 0.f) + 0x80808080u;  // its bytes are D + 128
  const int cc = c % kMcTile;
  char* blk = base + ((size_t)(hb >> 1) * CT + c / kMcTile) * BB;
#pragma unroll
  for (int g = 0; g < 4; g++) {  // lane group g's four elements of this half
    const uint32_t u0 = U[TR ? g : 4 * g], u1 = U[TR ? 4 + g : 4 * g + 1];
    const uint32_t u2 = U[TR ? 8 + g : 4 * g + 2], u3 = U[TR ? 12 + g : 4 * g + 3];
    const uint32_t a01 = __builtin_amdgcn_perm(u1, u0, 0x05010400u);  // u0.b0 u1.b0 u0.b1 u1.b1
    const uint32_t a23 = __builtin_amdgcn_perm(u3, u2, 0x05010400u);
    const uint32_t c01 = __builtin_amdgcn_perm(u1, u0, 0x07030602u);  // u0.b2 u1.b2 u0.b3 u1.b3
    const uint32_t c23 = __builtin_amdgcn_perm(u3, u2, 0x07030602u);
    const uint32_t D[4] = {__builtin_amdgcn_perm(a23, a01, 0x05040100u) ^ 0x80808080u,
                           __builtin_amdgcn_perm(a23, a01, 0x07060302u) ^ 0x80808080u,
                           __builtin_amdgcn_perm(c23, c01, 0x05040100u) ^ 0x80808080u,
                           __builtin_amdgcn_perm(c23, c01, 0x07060302u) ^ 0x80808080u};
#pragma unroll
    for (int d = 0; d < 4; d++)  // digit row 4 cc + d
      *reinterpret_cast<uint32_t*>(blk + 8 * (16 * g + 4 * cc + d) + 4 * (hb & 1)) = D[d];
  }
  float* sp = reinterpret_cast<float*>(blk + 512) + cc;
  if ((hb & 1) == 0) sp[0] = finite ? ldexpf(1.0f, 16 - sc) : NAN;
  if constexpr (MIN) {
    float s[8];
#pragma unroll
    for (int j = 0; j < 8; j++) s[j] = v[j] + v[j + 8];
    const float sum = ((s[0] + s[4]) + (s[1] + s[5])) + ((s[2] + s[6]) + (s[3] + s[7]));
    if constexpr (HALF) {
      sp[4 + 4 * (hb & 1)] = sum;
    } else {
      const float other = __shfl_xor(sum, 1, CN_WAVE);
      if ((hb & 1) == 0) sp[4] = sum + other;
    }
  }
}

__device__ __forceinline__ void mc_load16(const float* x, bool in, float (&v)[16]) {
#pragma unroll
  for (int j = 0; j < 4; j++) {
    float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
    if (in) f = *reinterpret_cast<const float4*>(x + 4 * j);
    v[4 * j] = f.x; v[4 * j + 1] = f.y; v[4 * j + 2] = f.z; v[4 * j + 3] = f.w;
  }
}

// 16 bytes from global memory straight into LDS: lane i of the wave writes
// base + 16 * i (the same base for the whole wave).
__device__ __forceinline__ void mc_dma16(const void* g, void* base) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t m =
      __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)base);
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "{m0}"(m) : "memory");
#endif
}

// x staged once for all workgroups: `halves` half-blocks (K padded to 128) of
// each column into dst.
template <int QT, int CT>
__global__ __launch_bounds__(CN_BLOCK) void mcol_prep_kernel(const float* __restrict__ x, int K, int halves, char* dst) {
  const int hb = blockIdx.x * CN_BLOCK + threadIdx.x, c = blockIdx.y;
  if (hb >= halves) return;  // halves is even: a block's two lanes leave together
  float v[16];
  mc_load16(x + (size_t)c * K + 16 * hb, 16 * hb < K, v);
  mc_stage<QT, CT>(v, c, hb, dst);
}

// CT: tiles of 16 digit rows (4 columns each), RT: tiles of 16 weight rows per wave.  The eight waves of a workgroup are rg row groups x 8 /
// rg interleaved shares of K.  kc elements of x at a time are staged in LDS, or
// with PRE copied from what mcol_prep_kernel staged (pre).
// With several workgroups along K (blockIdx.y, spb steps each) the sums go to
// part [blockIdx.y][column][row].
template <int QT, int CT, int RT, bool PRE>
__global__ __launch_bounds__(512) void gemv_mcol_kernel(GemvArgs a, int ncols, int kc, int rg, int spb, const char* pre,
                                                       float* part) {
  using T = QTraits<QT>;
  constexpr int NW = 8, NR = mc_raw<QT>(), BB = mc_block_bytes<QT>();
  constexpr bool HALF = mc_half_scales<QT>(), MIN = group_min<QT>();
  extern __shared__ __attribute__((aligned(16))) char mlds[];
  const int M = a.n_vrows;
  const int kb = blockIdx.y * spb * 128, K = min(a.K, kb + spb * 128);  // this workgroup's share
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int p = lane >> 4, li = lane & 15;
  const int nks = NW / rg, ks = wave % nks;
  const int row0 = (blockIdx.x * rg + wave / nks) * (16 * RT);
  const size_t bpr = (size_t)(a.K / T::BLOCK) * T::BLOCK_BYTES;
  const int nsteps = (K + 127) >> 7;  // end of the share

  const cn_gbyte* rp[RT];
#pragma unroll
  for (int t = 0; t < RT; t++) rp[t] = (const cn_gbyte*)a.w[0] + (size_t)min(row0 + 16 * t + li, M - 1) * bpr;
  uint32_t raw[RT][NR];
  auto load = [&](int s) {
#pragma unroll
    for (int t = 0; t < RT; t++) mc_load<QT>(rp[t], min(s, nsteps - 1), p, a.K, raw[t]);
  };
  load((kb >> 7) + ks);  // travels while x is staged

  float acc[RT][CT];  // weight row li of the tile, column p of the tile
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int c = 0; c < CT; c++) acc[t][c] = 0.f;

  for (int k0 = kb; k0 < K; k0 += kc) {
    const int kn = (min(kc, K - k0) + 127) & ~127;  // staged with zeros past K
    if (k0 > kb) __syncthreads();
    if constexpr (PRE) {  // a copy of the staged blocks
      const char* src = pre + (size_t)(k0 >> 5) * CT * BB;
      const int pieces = (kn >> 5) * CT * (BB / 16);
      for (int t = wave * CN_WAVE; t < pieces; t += 512) {
        const int i = t + lane;
        if (i < pieces) mc_dma16(src + (size_t)i * 16, mlds + (size_t)t * 16);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    } else {
      const int halves = kn >> 4;
      for (int t = threadIdx.x; t < ncols * halves; t += 512) {
        const int c = t / halves, hb = t - c * halves, k = k0 + 16 * hb;
        float v[16];
        mc_load16(a.x + (size_t)c * a.K + k, k < K, v);
        mc_stage<QT, CT>(v, c, hb, mlds);
      }
    }
    __syncthreads();
    // this wave's steps of 128 weights of the chunk (a multiple of the waves'
    // turns unless it is the whole row)
    const int s_end = (k0 + kn) >> 7;
    for (int s = (k0 >> 7) + ks; s < s_end; s += nks) {
      uint32_t q[RT][4][2];
      float sa[RT][4][2], sb[RT][4][2];
      const int nblk = T::BLOCK == 32 ? K / 32 - 4 * s : 4;
#pragma unroll
      for (int t = 0; t < RT; t++) mc_expand<QT>(raw[t], s, p, nblk, q[t], sa[t], sb[t]);
      if (s + nks < nsteps) load(s + nks);
#pragma unroll
      for (int b = 0; b < 4; b++) {
#pragma unroll
        for (int c = 0; c < CT; c++) {
          const char* blk = mlds + ((size_t)(4 * s + b - (k0 >> 5)) * CT + c) * BB;
          const long xf = *reinterpret_cast<const long*>(blk + 8 * lane);
          const float pe = *reinterpret_cast<const float*>(blk + 512 + 4 * p);
#pragma unroll
          for (int hv = 0; hv < (HALF ? 2 : 1); hv++) {
            float sx = 0.f;
            if constexpr (MIN) sx = *reinterpret_cast<const float*>(blk + 528 + 16 * hv + 4 * p);
#pragma unroll
            for (int t = 0; t < RT; t++) {
              const uint32_t w0 = HALF && hv == 1 ? 0u : q[t][b][0], w1 = HALF && hv == 0 ? 0u : q[t][b][1];
              const long wf = (long)(((uint64_t)w1 << 32) | w0);
              const mc_i32x4 r = __builtin_amdgcn_mfma_i32_16x16x32_i8(xf, wf, mc_i32x4{0, 0, 0, 0}, 0, 0, 0);
              // |r| <= 2^19: each pair joined in int32
              const float v = fmaf((float)(r[1] * 256 + r[0]), 0x1p-16f, (float)(r[3] * 256 + r[2]));
              if constexpr (MIN) acc[t][c] = fmaf(sb[t][b][hv], sx, acc[t][c]);
              acc[t][c] = fmaf(v * sa[t][b][hv], pe, acc[t][c]);
            }
          }
        }
      }
    }
  }
  // the waves' shares of K meet in LDS, summed in wave order
  __syncthreads();
  float* red = reinterpret_cast<float*>(mlds);
#pragma unroll
  for (int t = 0; t < RT; t++)
#pragma unroll
    for (int c = 0; c < CT; c++) red[((wave * RT + t) * CT + c) * 64 + lane] = acc[t][c];
  __syncthreads();
  for (int o = threadIdx.x; o < rg * RT * 16 * ncols; o += 512) {
    const int n = o & 15, t = (o >> 4) % RT, c = (o / (16 * RT)) % ncols, g = o / (16 * RT * ncols);
    const int row = (blockIdx.x * rg + g) * (16 * RT) + 16 * t + n;
    float v = 0.f;
    for (int k = 0; k < nks; k++)
      v += red[(((g * nks + k) * RT + t) * CT + c / kMcTile) * 64 + 16 * (c % kMcTile) + n];
    float* to = part ? part + (size_t)blockIdx.y * ncols * M : a.out[0];
    if (row < M) to[(size_t)c * M + row] = v;
  }
}

// y[i] = sum over the K shares, in order.
__global__ __launch_bounds__(CN_BLOCK) void mcol_reduce_kernel(const float* __restrict__ part, float* __restrict__ y,
                                                              int n, int shares) {
  const int i = blockIdx.x * CN_BLOCK + threadIdx.x;
  if (i >= n) return;
  float v = 0.f;
  for (int s = 0; s < shares; s++) v += part[(size_t)s * n + i];
  y[i] = v;
}

template <int QT, int CT, int RT, bool PRE>
hipError_t launch_mcol_one(const GemvArgs& a, int ncols, int num_cus, const char* pre, int shares, float* part,
                           hipStream_t st) {
  // staged x: at most 78 KB where two workgroups share a CU, else 156 KB; when
  // it takes several rounds, a multiple of the waves' turns
  constexpr int per_step = 4 * CT * mc_block_bytes<QT>();
  const int groups = (a.n_vrows + 16 * RT - 1) / (16 * RT);
  int rg = 1;
  while (rg < 8 && (groups + rg - 1) / rg > 2 * num_cus) rg *= 2;
  const int spb = ((a.K + 127) / 128 + shares - 1) / shares, nsteps = spb, turn = 8 / rg;
  int fit = (78 * 1024) / per_step;  // steps of 128
  if ((groups + rg - 1) / rg <= num_cus) fit = (156 * 1024) / per_step;
  const int steps = nsteps <= fit ? nsteps : fit / turn * turn;
  const size_t stage = (size_t)steps * per_step;
  const size_t red = (size_t)8 * RT * CT * 64 * sizeof(float);
  const size_t smem = stage > red ? stage : red;
  const auto kern = &gemv_mcol_kernel<QT, CT, RT, PRE>;
  if (smem > 64 * 1024) {
    static std::atomic<uint64_t> lds_done{0};
    const hipError_t e = allow_full_lds(reinterpret_cast<const void*>(kern), lds_done);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kern, dim3((groups + rg - 1) / rg, shares), dim3(512), smem, st, a, ncols, steps * 128, rg, spb, pre,
                     shares > 1 ? part : nullptr);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess || shares == 1) return e;
  const int n = ncols * a.n_vrows;
  hipLaunchKernelGGL(mcol_reduce_kernel, dim3((n + CN_BLOCK - 1) / CN_BLOCK), dim3(CN_BLOCK), 0, st, part, a.out[0], n,
                     shares);
  return hipGetLastError();
}

// One row tile per wave while that leaves at most a workgroup per CU, else two
// (each x fragment read then feeds two products).
template <int QT, int CT>
hipError_t launch_mcol_ct(const GemvArgs& a, int ncols, int num_cus, const McolPlan& p, hipStream_t st) {
  const bool one = CT > 2 || a.n_vrows <= 16 * num_cus;
  if (p.pre) {
    const int halves = (a.K + 127) / 128 * 8;
    hipLaunchKernelGGL((mcol_prep_kernel<QT, CT>), dim3((halves + CN_BLOCK - 1) / CN_BLOCK, ncols), dim3(CN_BLOCK), 0, st,
                       a.x, a.K, halves, p.pre);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if constexpr (CT <= 2) {
      if (!one) return launch_mcol_one<QT, CT, 2, true>(a, ncols, num_cus, p.pre, 1, nullptr, st);
    }
    return launch_mcol_one<QT, CT, 1, true>(a, ncols, num_cus, p.pre, 1, nullptr, st);
  }
  if constexpr (CT <= 2) {
    if (!one) return launch_mcol_one<QT, CT, 2, false>(a, ncols, num_cus, nullptr, 1, nullptr, st);
  }
  return launch_mcol_one<QT, CT, 1, false>(a, ncols, num_cus, nullptr, p.shares, p.part, st);
}

template <int QT>
hipError_t launch_mcol(const GemvArgs& a, int ncols, int num_cus, const McolPlan& p, hipStream_t st) {
  if (ncols <= 4) return launch_mcol_ct<QT, 1>(a, ncols, num_cus, p, st);
  if (ncols <= 8) return launch_mcol_ct<QT, 2>(a, ncols, num_cus, p, st);
  if (ncols <= 12) return launch_mcol_ct<QT, 3>(a, ncols, num_cus, p, st);
  return launch_mcol_ct<QT, 4>(a, ncols, num_cus, p, st);
}

}  // namespace

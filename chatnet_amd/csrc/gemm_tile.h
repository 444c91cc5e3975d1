// gemm_tile.h — the matrix-core GEMM kernels over weights as they are stored,
// instantiated per weight format by the gemm_*.hip files and dispatched by
// gemm.hip (whose header describes the whole).
#pragma once
#include <algorithm>

#include "device_common.h"
#include "kernels.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// s += v element by element, the rounding error of the sum so far carried in c.
template <class V>
__device__ __forceinline__ void add_compensated(V& s, V& c, const V& v) {
  const V y = v - c;
  const V t = s + y;
  c = (t - s) - y;
  s = t;
}

// W rows of the virtual row `vr`: single matrix, three concatenated (q|k|v)
// or two interleaved (gate even, up odd).
__device__ __forceinline__ const uint8_t* gemm_row_ptr(const GemmArgs& a, int vr, size_t row_bytes) {
  if (vr >= a.M) return nullptr;
  int seg = 0, r = vr;
  if (a.seg_mode == GEMM_SEG_INTERLEAVE) {
    seg = vr & 1;
    r = vr >> 1;
  } else if (a.seg_mode == GEMM_SEG_CONCAT) {
    if (r >= a.seg_rows[0]) {
      r -= a.seg_rows[0];
      seg = 1;
      if (r >= a.seg_rows[1]) {
        r -= a.seg_rows[1];
        seg = 2;
      }
    }
  }
  // a select, not a[seg]: indexing the argument array would copy it to scratch
  const uint8_t* w = seg == 0 ? a.w[0] : (seg == 1 ? a.w[1] : a.w[2]);
  return w + (size_t)r * row_bytes;
}

// silu(g) * u = g * u / (1 + e^-g) (TensorMath.SiluElementwiseMul,
// TensorMath.cs:253-286) with the hardware exp2 and reciprocal: about 1e-7
// relative, below the resolution of the fp16 hi + lo planes h is stored in
// (the span epilogue runs it for every h element of the tile).
__device__ __forceinline__ float silu_mul(float g, float u) {
  return g * u * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-g * 1.4426950408889634f));
}

// h[n][j] = silu(gate) * up as the next span GEMM's input: fp16 hi + lo
// planes in the span order (cn_span_pos).
__device__ __forceinline__ void write_h(const GemmArgs& a, int n, int j, float v) {
  const size_t i = (size_t)n * a.ldh + cn_span_pos(j);
  uint32_t hi, lo;
  cn_split_f16x2(v, 0.f, hi, lo);
  a.hb[i] = (uint16_t)hi;
  a.hb_lo[i] = (uint16_t)lo;
}

// Outputs of chatnet_matmul's F16 rows (rows m..m+3 of column n) that came out
// NaN, summed again from the fp32 x: in planes an infinite weight meets x's
// low parts too (inf * 0 or inf - inf), where the plain product is infinite.
// Never taken for finite operands.  Only the compensated instances call it (a
// loop in every instance's epilogue cost the others registers).
__device__ __forceinline__ void f16_dot_again(const GemmArgs& a, int n, int m, f32x4& v) {
  const float t = (v[0] + v[1]) + (v[2] + v[3]);
  if (t == t || n >= a.N) return;
  for (int i = 0; i < 4 && m + i < a.M; i++) {
    if (v[i] == v[i]) continue;
    const _Float16* w = reinterpret_cast<const _Float16*>(a.w[0]) + (size_t)(m + i) * a.K;
    const float* x = a.x32 + (size_t)n * a.K;
    float s = 0.f;
    for (int k = 0; k < a.K; k++) s = fmaf((float)w[k], x[k], s);
    v[i] = s;
  }
}

// Final write of 4 consecutive rows m..m+3 of column n.
__device__ __forceinline__ void write_out4(const GemmArgs& a, int epi, int n, int m, f32x4 v) {
  if (n >= a.N || m >= a.M) return;
  const bool full = (m + 3 < a.M) && ((a.ldy & 3) == 0);
  if (epi == GEMV_EPI_SWIGLU) {
    // rows (m, m+1) and (m+2, m+3) are (gate, up) pairs of h[m/2], h[m/2+1]
    // (m/2 even: the two stay adjacent in the span order too)
    if (m + 3 < a.M) {
      const float h0 = silu_mul(v[0], v[1]), h1 = silu_mul(v[2], v[3]);
      const size_t i = (size_t)n * a.ldh + cn_span_pos(m >> 1);
      uint32_t hi, lo;
      cn_split_f16x2(h0, h1, hi, lo);
      *reinterpret_cast<uint32_t*>(a.hb + i) = hi;
      *reinterpret_cast<uint32_t*>(a.hb_lo + i) = lo;
    } else {
      write_h(a, n, m >> 1, silu_mul(v[0], v[1]));
    }
    return;
  }
  float* y = a.y + (size_t)n * a.ldy + m;
  if (full) {
    f32x4* p = reinterpret_cast<f32x4*>(y);
    if (epi == GEMV_EPI_ADD) *p = *p + v;
    else *p = v;
  } else {
    for (int i = 0; i < 4 && m + i < a.M; i++) y[i] = (epi == GEMV_EPI_ADD) ? y[i] + v[i] : v[i];
  }
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x16 mma32(f16x8 a, f16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// Exact-weight (span) kernel, raw Q4_0, fp16 operands.  One MFMA step of a
// lane takes one qs dword of its block; wp holds its bytes in the order
// b0 b2 b1 b3, so that the elements (4s, 4s+1) sit in the low nibbles at bits
// 0-3 / 16-19, (4s+2, 4s+3) at bits 8-11 / 24-27, (16+4s, 16+4s+1) in the
// high nibbles at bits 4-7 / 20-23 and (16+4s+2, 16+4s+3) at 12-15 / 28-31:
// the element order cn_span_pos stores x in.  A pair (q_a, q_b) becomes two
// fp16 halves 0x6400 | q = 1024 + q (or 0x6400 | q << 4 = 1024 + 16q), and a
// packed fp16 add (fma) turns each into q - 8 exactly.  The weight d*(q-8)
// then splits exactly as Wa = (q-8)*dh + Wb = (q-8)*dl, dh = d with its three
// low mantissa bits cleared, dl = d - dh: (q-8) has at most 3 significant
// bits, dh at most 8 and dl at most 3, so both products are fp16 values for
// |d| < 4096 (fp16 subnormals included) and need no rounding.  `magic` holds
// 0x64006400 in a register (v_and_or_b32 takes no two literals).
__device__ __forceinline__ void dequant_q4_f16(uint32_t wp, uint32_t magic, cn_half2 dh, cn_half2 dl, f16x8& wa,
                                               f16x8& wb) {
  const uint32_t u = wp >> 8;
  const cn_half2 t0 = __builtin_bit_cast(cn_half2, (wp & 0x000F000Fu) | magic);
  const cn_half2 t1 = __builtin_bit_cast(cn_half2, (u & 0x000F000Fu) | magic);
  const cn_half2 t2 = __builtin_bit_cast(cn_half2, (wp & 0x00F000F0u) | magic);
  const cn_half2 t3 = __builtin_bit_cast(cn_half2, (u & 0x00F000F0u) | magic);
  const cn_half2 m1032 = {(_Float16)-1032.0f, (_Float16)-1032.0f};
  const cn_half2 s16 = {(_Float16)0.0625f, (_Float16)0.0625f};
  const cn_half2 m72 = {(_Float16)-72.0f, (_Float16)-72.0f};
  const cn_half2 p0 = t0 + m1032, p1 = t1 + m1032;
  const cn_half2 p2 = t2 * s16 + m72, p3 = t3 * s16 + m72;
  const cn_half2 a0 = p0 * dh, a1 = p1 * dh, a2 = p2 * dh, a3 = p3 * dh;
  const cn_half2 b0 = p0 * dl, b1 = p1 * dl, b2 = p2 * dl, b3 = p3 * dl;
  wa = (f16x8){a0[0], a0[1], a1[0], a1[1], a2[0], a2[1], a3[0], a3[1]};
  wb = (f16x8){b0[0], b0[1], b1[0], b1[1], b2[0], b2[1], b3[0], b3[1]};
}

// Exact-weight kernel, packed units: the 8 weights of one MFMA step, codes of
// ca with (sc0, of0) then codes of cb with (sc1, of1), as fp16 hi + lo
// (w = fmaf(code, sc, of) carries up to 24 bits; hi + lo keep ~22).
__device__ __forceinline__ void dequant_u8_f16(uint32_t ca, uint32_t cb, float sc0, float of0, float sc1, float of1,
                                               f16x8& wa, f16x8& wb) {
  float w[8];
  w[0] = fmaf(cn_ubyte<0>(ca), sc0, of0);
  w[1] = fmaf(cn_ubyte<1>(ca), sc0, of0);
  w[2] = fmaf(cn_ubyte<2>(ca), sc0, of0);
  w[3] = fmaf(cn_ubyte<3>(ca), sc0, of0);
  w[4] = fmaf(cn_ubyte<0>(cb), sc1, of1);
  w[5] = fmaf(cn_ubyte<1>(cb), sc1, of1);
  w[6] = fmaf(cn_ubyte<2>(cb), sc1, of1);
  w[7] = fmaf(cn_ubyte<3>(cb), sc1, of1);
  uint32_t hi[4], lo[4];
#pragma unroll
  for (int t = 0; t < 4; t++) cn_split_f16x2(w[2 * t], w[2 * t + 1], hi[t], lo[t]);
  wa = __builtin_bit_cast(f16x8, make_uint4(hi[0], hi[1], hi[2], hi[3]));
  wb = __builtin_bit_cast(f16x8, make_uint4(lo[0], lo[1], lo[2], lo[3]));
}

// One-plane kernel (chatnet_matmul), raw Q4_0: the 8 weights of one MFMA step
// as fp16(d * (q - 8)), one rounding each.  The nibble pairs of wp (bytes b0 b2
// b1 b3 of a qs dword, as dequant_q4_f16 takes them) become q - 8 exactly as
// there, and one packed fp16 multiply by d rounds each product once (|d| <
// 8188 keeps every product finite).
__device__ __forceinline__ f16x8 dequant_q4_h(uint32_t wp, uint32_t magic, cn_half2 d2) {
  const uint32_t u = wp >> 8;
  const cn_half2 t0 = __builtin_bit_cast(cn_half2, (wp & 0x000F000Fu) | magic);
  const cn_half2 t1 = __builtin_bit_cast(cn_half2, (u & 0x000F000Fu) | magic);
  const cn_half2 t2 = __builtin_bit_cast(cn_half2, (wp & 0x00F000F0u) | magic);
  const cn_half2 t3 = __builtin_bit_cast(cn_half2, (u & 0x00F000F0u) | magic);
  const cn_half2 m1032 = {(_Float16)-1032.0f, (_Float16)-1032.0f};
  const cn_half2 s16 = {(_Float16)0.0625f, (_Float16)0.0625f};
  const cn_half2 m72 = {(_Float16)-72.0f, (_Float16)-72.0f};
  const cn_half2 a0 = (t0 + m1032) * d2, a1 = (t1 + m1032) * d2;
  const cn_half2 a2 = (t2 * s16 + m72) * d2, a3 = (t3 * s16 + m72) * d2;
  return (f16x8){a0[0], a0[1], a1[0], a1[1], a2[0], a2[1], a3[0], a3[1]};
}

// One-plane kernel, packed units: the 8 weights of one MFMA step, codes of ca
// with (sc0, of0) then codes of cb with (sc1, of1), each fmaf(code, sc, of) in
// fp32 (the type's value) rounded once to fp16.
__device__ __forceinline__ f16x8 dequant_u8_h(uint32_t ca, uint32_t cb, float sc0, float of0, float sc1, float of1) {
  const cn_float2 w0 = {fmaf(cn_ubyte<0>(ca), sc0, of0), fmaf(cn_ubyte<1>(ca), sc0, of0)};
  const cn_float2 w1 = {fmaf(cn_ubyte<2>(ca), sc0, of0), fmaf(cn_ubyte<3>(ca), sc0, of0)};
  const cn_float2 w2 = {fmaf(cn_ubyte<0>(cb), sc1, of1), fmaf(cn_ubyte<1>(cb), sc1, of1)};
  const cn_float2 w3 = {fmaf(cn_ubyte<2>(cb), sc1, of1), fmaf(cn_ubyte<3>(cb), sc1, of1)};
  const cn_half2 h0 = __builtin_convertvector(w0, cn_half2), h1 = __builtin_convertvector(w1, cn_half2);
  const cn_half2 h2 = __builtin_convertvector(w2, cn_half2), h3 = __builtin_convertvector(w3, cn_half2);
  return (f16x8){h0[0], h0[1], h1[0], h1[1], h2[0], h2[1], h3[0], h3[1]};
}

// ---------------------------------------------------------------------------
// Pipelined 32x32 tile kernels (gemm_p_kernel, gemm_s_kernel): raw W bytes
// and the x tile stream into an LDS ring through direct global->LDS loads
// (global_load_lds_dwordx4, no registers held), so later chunks of 64 K are in
// flight while one is computed; a workgroup waits only for the chunk it needs
// (s_waitcnt vmcnt(n) + a bare s_barrier), not for the whole queue.
//
// Per chunk (one 36-byte Q4_0 unit per W row) lane half h of row li takes
// block h of the unit, and the x fragment of the same lane reads the same 8 k
// of every MFMA step, so the K order inside a chunk is permuted consistently
// for both operands (each kernel's comment gives its order).
// LDS layout per stage: x planes [BN rows][8 x 16 B] with the 16-byte chunk
// of logical index c of row r stored at c ^ ((r >> 1) & 7) (reads of 32 rows
// stay 2-way per bank), then W [128 rows][48 B] holding unit bytes [0,16),
// [16,32) and [20,36) (packed units: [128 rows][96 B]).
// A wave owns 32 W rows x 32*TN columns; the 4 waves stack along M and share
// the x tile.  Output layout of a 32x32 tile: lane l, accumulator v holds row
// 8*(v/4) + 4*(l/32) + v%4, column l%32.
// ---------------------------------------------------------------------------
// 16 bytes from global memory straight into LDS: lane i of the wave writes
// lds_wave_base + 16*i (lds_wave_base must be the same for the whole wave).
// Issued as inline assembly: the compiler treats its own LDS-DMA builtin as
// a write to all of LDS and waits for every load in flight (vmcnt(0)) before
// the next LDS read, which would drain the ring at every chunk; the kernels
// instead wait for the chunk they read with vm_wait and a barrier.  The
// compiler's own waits stay correct with these loads in flight (vector-memory
// counters retire in order, so a wait for one of its loads can only wait
// longer).
__device__ __forceinline__ void lds_dma16(const void* g, void* lds_wave_base) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t m = __builtin_amdgcn_readfirstlane(
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)lds_wave_base);
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "{m0}"(m) : "memory");
#endif
}

template <int N>
__device__ __forceinline__ void vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Waits until only the `later` chunks issued after the needed one (at most
// K, VPS vector-memory instructions each) may still be in flight.
template <int VPS, int K>
__device__ __forceinline__ void vm_wait_later(int later) {
  if constexpr (K == 0 || K * VPS > 63) {
    if constexpr (K == 0) vm_wait<0>();
    else vm_wait_later<VPS, K - 1>(later);
  } else {
    if (later >= K) vm_wait<K * VPS>();
    else vm_wait_later<VPS, K - 1>(later);
  }
}

__device__ __forceinline__ void wg_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// LDS reads issued as inline assembly, so that the compiler neither sinks them
// next to their first use nor waits for them itself: a chunk's reads are all
// issued at its start and each step waits (lds_wait) only for the reads it
// consumes.  LDS reads of one wave retire in order.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}
// OFF: a constant byte offset carried in the instruction's offset field (no
// address arithmetic for it).
template <int OFF = 0>
__device__ __forceinline__ cn_u32x4 lds_read128(uint32_t addr) {
  static_assert(OFF >= 0 && OFF < 65536, "ds offset field is 16 bits");
  cn_u32x4 v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF) : "memory");
  return v;
}
template <int OFF = 0>
__device__ __forceinline__ uint2 lds_read64(uint32_t addr) {
  static_assert(OFF >= 0 && OFF < 65536, "ds offset field is 16 bits");
  uint2 v;
  asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF) : "memory");
  return v;
}
template <int OFF = 0>
__device__ __forceinline__ uint32_t lds_read32(uint32_t addr) {
  static_assert(OFF >= 0 && OFF < 65536, "ds offset field is 16 bits");
  uint32_t v;
  asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF) : "memory");
  return v;
}
// The x fragments of one MFMA step for column tiles CC .. TN-1: tile cc lies
// 32 x-rows (4096 bytes) after tile cc-1, at the same swizzled chunk.
template <int CC, int TN>
__device__ __forceinline__ void lds_read_xtiles(uint32_t base, cn_u32x4 (&xr)[TN]) {
  if constexpr (CC < TN) {
    xr[CC] = lds_read128<CC * 4096>(base);
    lds_read_xtiles<CC + 1, TN>(base, xr);
  }
}
// Waits until at most N of this wave's LDS reads are outstanding.  A value
// read by lds_read* must pass through reg_fence after the wait that covers it,
// so that its uses stay behind that wait.
template <int N>
__device__ __forceinline__ void lds_wait() {
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
}
template <class T>
__device__ __forceinline__ void reg_fence(T& r) {
  asm volatile("" : "+v"(r));
}

// How a chunk of 64 weights of a row lies in global memory and in LDS, by weight
// format.  A row's chunk is moved as WP pieces of 16 bytes, every one inside the
// row: piece i from byte OFF[i] of the chunk's unit (UNIT bytes per chunk), or
// for the super-block types (SB bytes per four chunks) from byte OFF[i] + ((c &
// 3) * STEP[i] & MASK) of super-block c / 4.  Lane half h takes the unit's block
// h; the two-block types keep a window of its own for each half (aligned
// 16-byte LDS reads), the windows overlapping where a block starts inside a
// dword.
template <int WF>
struct WFmt;
template <> struct WFmt<GEMM_W_Q4_0> {  // two 18-byte blocks
  static constexpr int UNIT = 36, WP = 3, SB = 0, MASK = -1, WD = 5;
  static constexpr int OFF[WP] = {0, 16, 20}, STEP[WP] = {0, 0, 0};
};
template <> struct WFmt<GEMM_W_IQ4_NL> : WFmt<GEMM_W_Q4_0> {};
template <> struct WFmt<GEMM_W_PACKED> {  // gemm_pack_launch units
  static constexpr int UNIT = kGemmPackUnit, WP = 6, SB = 0, MASK = -1, WD = 12;
  static constexpr int OFF[WP] = {0, 16, 32, 48, 64, 80}, STEP[WP] = {0, 0, 0, 0, 0, 0};
};
template <> struct WFmt<GEMM_W_F16> {  // rows of the float type, pieces XOR-swizzled in LDS as the x rows are
  static constexpr int UNIT = 128, WP = 8, SB = 0, MASK = -1, WD = 16;
  static constexpr int OFF[WP] = {0, 16, 32, 48, 64, 80, 96, 112}, STEP[WP] = {};
};
template <> struct WFmt<GEMM_W_F16_X3> : WFmt<GEMM_W_F16> {};
template <> struct WFmt<GEMM_W_F32> {
  static constexpr int UNIT = 256, WP = 16, SB = 0, MASK = -1, WD = 32;
  static constexpr int OFF[WP] = {0, 16, 32, 48, 64, 80, 96, 112, 128, 144, 160, 176, 192, 208, 224, 240}, STEP[WP] = {};
};
template <> struct WFmt<GEMM_W_Q8_0> {  // two 34-byte blocks: windows at bytes 0 and 32
  static constexpr int UNIT = 68, WP = 6, SB = 0, MASK = -1, WD = 9;
  static constexpr int OFF[WP] = {0, 16, 20, 32, 48, 52}, STEP[WP] = {};
};
template <> struct WFmt<GEMM_W_Q5_0> {  // two 22-byte blocks: windows at bytes 0 and 20
  static constexpr int UNIT = 44, WP = 4, SB = 0, MASK = -1, WD = 6;
  static constexpr int OFF[WP] = {0, 8, 20, 28}, STEP[WP] = {};
};
template <> struct WFmt<GEMM_W_Q4_1> {  // two 20-byte blocks
  static constexpr int UNIT = 40, WP = 4, SB = 0, MASK = -1, WD = 5;
  static constexpr int OFF[WP] = {0, 4, 20, 24}, STEP[WP] = {};
};
template <> struct WFmt<GEMM_W_Q5_1> {  // two 24-byte blocks
  static constexpr int UNIT = 48, WP = 4, SB = 0, MASK = -1, WD = 6;
  static constexpr int OFF[WP] = {0, 8, 24, 32}, STEP[WP] = {};
};
template <> struct WFmt<GEMM_W_Q4_K> {  // the header, then the chunk's 32 qs bytes
  static constexpr int UNIT = 36, WP = 3, SB = 144, MASK = -1, WD = 8;
  static constexpr int OFF[WP] = {0, 16, 32}, STEP[WP] = {0, 32, 32};
};
template <> struct WFmt<GEMM_W_Q5_K> {  // the header, the 16 qh bytes that hold the chunk's 8, its 32 qs bytes
  static constexpr int UNIT = 44, WP = 4, SB = 176, MASK = ~15, WD = 9;
  static constexpr int OFF[WP] = {0, 16, 48, 64}, STEP[WP] = {0, 8, 32, 32};
};
template <> struct WFmt<GEMM_W_IQ4_XS> {  // bytes 0..15 (d and scales), the chunk's 32 qs bytes
  static constexpr int UNIT = 34, WP = 3, SB = 136, MASK = -1, WD = 8;
  static constexpr int OFF[WP] = {0, 8, 24}, STEP[WP] = {0, 32, 32};
};
template <> struct WFmt<GEMM_W_Q2_K> {  // the scales, the half's 32 qs bytes, d and dmin (bytes 80..83)
  static constexpr int UNIT = 21, WP = 4, SB = 84, MASK = ~31, WD = 13;
  static constexpr int OFF[WP] = {0, 16, 32, 68}, STEP[WP] = {0, 16, 16, 0};
};

// Formats read through u8 codes with an fp32 scale and offset per 16 weights,
// weight = fmaf(code, scale, offset): the values gemm_pack_kernel's units hold.
template <int WF>
constexpr bool float_format() { return WF == GEMM_W_F16 || WF == GEMM_W_F16_X3 || WF == GEMM_W_F32; }
template <int WF>
constexpr bool coded_format() { return WF != GEMM_W_Q4_0 && !float_format<WF>(); }

// The scales and offsets of a lane's 32 weights of chunk c (first and last 16), and
// their fifth bits.
struct WScale {
  float s0, o0, s1, o1;
  uint32_t qh;
};

// w: the lane's dwords (TileIO::wraw), h: its half of the chunk.
template <int WF, int WD>
__device__ __forceinline__ WScale w_scales(const uint32_t (&w)[WD], int h, int c) {
  WScale r{};
  const float d = cn_h2f(h ? w[0] >> 16 : w[0]);  // windows of a half that starts two bytes into the first dword
  if constexpr (WF == GEMM_W_PACKED) {
    r.s0 = __uint_as_float(w[8]), r.s1 = __uint_as_float(w[9]);
    r.o0 = __uint_as_float(w[10]), r.o1 = __uint_as_float(w[11]);
    return r;
  } else if constexpr (WF == GEMM_W_Q8_0) {
    r.s0 = d, r.o0 = -128.0f * d;
  } else if constexpr (WF == GEMM_W_Q5_0) {
    r.s0 = d, r.o0 = -16.0f * d;
    r.qh = __builtin_amdgcn_perm(w[1], w[0], h ? 0x07060504u : 0x05040302u);
  } else if constexpr (WF == GEMM_W_Q4_1 || WF == GEMM_W_Q5_1) {
    r.s0 = cn_h2f(w[0]), r.o0 = cn_h2f(w[0] >> 16);
    if constexpr (WF == GEMM_W_Q5_1) r.qh = w[1];
  } else if constexpr (WF == GEMM_W_IQ4_NL) {
    r.s0 = cn_h2f(h ? w[4] >> 16 : w[0]);
    r.o0 = -128.0f * r.s0;
  } else if constexpr (WF == GEMM_W_Q4_K || WF == GEMM_W_Q5_K) {
    // sub-block sb of the super-block (DequantQ4K.DecodeScales,
    // DequantQ4K.cs:218-264): its weights are d*sc*q - dmin*m, and both
    // products are exact in fp32 (11 x 6 bits)
    const int sb = 2 * (c & 3) + h;
    auto qb = [&](int i) { return (w[1 + (i >> 2)] >> (8 * (i & 3))) & 0xFFu; };
    uint32_t sc, mm;
    if (sb < 4) {
      sc = qb(sb) & 63u;
      mm = qb(sb + 4) & 63u;
    } else {
      sc = (qb(sb + 4) & 0xFu) | ((qb(sb - 4) >> 6) << 4);
      mm = (qb(sb + 4) >> 4) | ((qb(sb) >> 6) << 4);
    }
    r.s0 = cn_h2f(w[0]) * (float)sc;
    r.o0 = -(cn_h2f(w[0] >> 16) * (float)mm);
    if constexpr (WF == GEMM_W_Q5_K) r.qh = w[8];
  } else if constexpr (WF == GEMM_W_IQ4_XS) {
    const int sb = 2 * (c & 3) + h;
    const uint32_t lo = ((c & 2 ? w[2] : w[1]) >> (8 * (sb & 3))) & 0x3Fu, hi = (w[0] >> (16 + 2 * sb)) & 3u;
    r.s0 = cn_h2f(w[0]) * (float)((int)(lo | (hi << 6)) - 32);
    r.o0 = -128.0f * r.s0;
  } else {  // Q2_K: block t = 2 (c & 1) + h of half c >> 1, scale bytes 2t and 2t + 1 of the half
    static_assert(WF == GEMM_W_Q2_K, "no scales");
    const uint32_t b = (c & 2 ? (c & 1 ? w[3] : w[2]) : (c & 1 ? w[1] : w[0])) >> (16 * h);
    const float dd = cn_h2f(w[12]), dm = cn_h2f(w[12] >> 16);
    r.s0 = dd * (float)(b & 15u);
    r.o0 = -(dm * (float)((b >> 4) & 15u));
    r.s1 = dd * (float)((b >> 8) & 15u);
    r.o1 = -(dm * (float)((b >> 12) & 15u));
    return r;
  }
  r.s1 = r.s0, r.o1 = r.o0;
  return r;
}

// The codes of step s: elements 4s .. 4s+3 (ca) and 16+4s .. 16+4s+3 (cb) of the
// lane's 32 weights, the order x is stored in (packed units: of its first and
// last 16, the same elements).
template <int WF, int WD>
__device__ __forceinline__ void w_codes(const uint32_t (&w)[WD], const WScale& r, int h, int c, int s, uint32_t& ca,
                                        uint32_t& cb) {
  constexpr uint32_t LO = 0x0F0F0F0Fu, S8 = 0x80808080u;
  if constexpr (WF == GEMM_W_PACKED) {
    ca = w[s];
    cb = w[4 + s];
  } else if constexpr (WF == GEMM_W_Q8_0) {
    const uint32_t sel = h ? 0x07060504u : 0x05040302u;  // dword k of qs: bytes 4k + 2 .. (h = 0) or 4k + 4 .. of the window
    ca = __builtin_amdgcn_perm(w[s + 1], w[s], sel) ^ S8;
    cb = __builtin_amdgcn_perm(w[s + 5], w[s + 4], sel) ^ S8;
  } else if constexpr (WF == GEMM_W_Q2_K) {
    const int t = 2 * (2 * (c & 1) + h);
    ca = (w[4 + s] >> t) & 0x03030303u;
    cb = (w[8 + s] >> t) & 0x03030303u;
  } else {
    uint32_t q;  // qs dword s: low nibbles elements 4s.., high nibbles 16+4s..
    if constexpr (WF == GEMM_W_Q5_0) q = __builtin_amdgcn_perm(w[s + 2], w[s + 1], h ? 0x07060504u : 0x05040302u);
    else if constexpr (WF == GEMM_W_Q4_1) q = w[1 + s];
    else if constexpr (WF == GEMM_W_Q5_1) q = w[2 + s];
    else if constexpr (WF == GEMM_W_IQ4_NL) q = __builtin_amdgcn_perm(w[s + 1], w[s], h ? 0x03020100u : 0x05040302u);
    else q = w[4 + s];
    ca = q & LO;
    cb = (q >> 4) & LO;
    if constexpr (WF == GEMM_W_Q5_0 || WF == GEMM_W_Q5_1 || WF == GEMM_W_Q5_K) {
      ca |= spread4(r.qh >> (4 * s)) << 4;
      cb |= spread4(r.qh >> (16 + 4 * s)) << 4;
    }
    if constexpr (WF == GEMM_W_IQ4_NL || WF == GEMM_W_IQ4_XS) {
      ca = iq4_values(ca) ^ S8;
      cb = iq4_values(cb) ^ S8;
    }
  }
}

// MT: 32-row tiles per wave, TN: 32-column tiles per wave; each x fragment
// read from LDS feeds MT MFMAs, each dequantized W fragment TN.  WNC: waves
// along N (1: the four waves stack along M, BM = 128 * MT; 2: a 2 x 2 grid of
// waves, BM = 64 * MT, BN = 64 * TN, each wave reading half the x tile).
// WF: how W is stored (GemmArgs::packed, WFmt).
template <bool PRECISE, int TN, int S, int WF, int MT = 1, int WNC = 1>
struct PipeCfg {
  using F = WFmt<WF>;
  static constexpr int FMT = WF;
  static constexpr int PL = WF == GEMM_W_F16_X3 ? 3 : PRECISE ? 2 : 1;  // x planes
  static constexpr int MTILES = MT;
  static constexpr int WN = WNC, WM = 4 / WNC;  // waves along N and M
  static constexpr int BM = 32 * WM * MT, BN = 32 * TN * WN;
  static constexpr bool FLT = float_format<WF>();
  static constexpr int UNIT = F::UNIT;         // global bytes per row and chunk of 64
  static constexpr int WP = F::WP;             // 16-byte pieces per row and chunk
  static constexpr int WROW = 16 * WP;         // LDS bytes per row and chunk
  static constexpr int XB = BN * 128;          // bytes per x plane per stage
  static constexpr int WB = BM * WROW;         // bytes of W per stage
  static constexpr int STAGE = PL * XB + WB;
  static constexpr int LDS = S * STAGE;        // the ring
  static constexpr int XPW = BN * 8 / 4;       // x pieces (16 B) per wave per plane
  static constexpr int XI = XPW / 64;
  static constexpr int WPW = BM * WP / 4;      // W pieces per wave
  static constexpr int WI = (WPW + 63) / 64;
  static constexpr int VPS = PL * XI + WI;     // vector-memory instructions per stage per wave
  static constexpr int WD = F::WD;             // W dwords a lane reads per chunk
  static constexpr int TNW = TN;                // column tiles per wave
  static_assert(XPW % 64 == 0, "x pieces per wave must fill whole instructions");
};

// Tile coordinates, K range and stage loads of one workgroup (both kernels).
template <class C>
struct TileIO {
  int lane, wave, wm, wn, h, li, ks, m0, n0, c_begin, c_end;
  const uint16_t* xsrc[C::PL][C::XI];
  const char* wsrc[C::WI];
  int wstep[C::WI];  // bytes the piece moves per chunk within a super-block
  bool wact[C::WI];

  // The tile and K range of blockIdx.x (tile-major, K split innermost); a
  // stream-K launch (a.sk_wgs > 0) sets each of its segments with set_tile.
  __device__ __forceinline__ explicit TileIO(const GemmArgs& a) {
    lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    wm = wave % C::WM;
    wn = wave / C::WM;
    h = lane >> 5;
    li = lane & 31;
    ks = 0;
    if (a.sk_wgs > 0) return;  // stream-K launches do not split K (a.splits == 1)
    int bid = blockIdx.x;
    ks = bid % a.splits;
    bid /= a.splits;
    const int nchunks = a.K / 64;
    const int cps = (nchunks + a.splits - 1) / a.splits;
    set_tile(a, bid, ks * cps, min(nchunks, ks * cps + cps));
  }

  // Tile `tile` (row tile tile / n_nt, column tile tile % n_nt), chunks [cb, ce).
  __device__ __forceinline__ void set_tile(const GemmArgs& a, int tile, int cb, int ce) {
    const int n_nt = (a.N + C::BN - 1) / C::BN;
    m0 = (tile / n_nt) * C::BM;
    n0 = (tile % n_nt) * C::BN;
    c_begin = cb;
    c_end = ce;
    const size_t row_bytes = (size_t)(a.K / 64) * C::UNIT;
#pragma unroll
    for (int p = 0; p < C::PL; p++)
#pragma unroll
      for (int j = 0; j < C::XI; j++) {
        const int piece = wave * C::XPW + 64 * j + lane;
        const int row = piece >> 3, ch = piece & 7;
        const int n = min(n0 + row, a.N - 1);
        const int logical = ch ^ ((row >> 1) & 7);
        xsrc[p][j] = (p == 2 ? a.xb_ll : p ? a.xb_lo : a.xb) + (size_t)n * a.K + 8 * logical;
      }
#pragma unroll
    for (int j = 0; j < C::WI; j++) {
      const int q = 64 * j + lane;
      wact[j] = q < C::WPW;
      const int piece = wave * C::WPW + (wact[j] ? q : 0);
      const int row = piece / C::WP, part = piece % C::WP;
      const int vr = min(m0 + row, a.M - 1);
      // float rows: LDS slot `part` holds the row's piece part ^ ((row >> 1) & 7)
      int off = 0;
      wstep[j] = 0;
      if constexpr (C::FLT) {
        off = 16 * (part ^ ((row >> 1) & 7));
      } else {
#pragma unroll
        for (int i = 0; i < C::WP; i++) {
          off = part == i ? C::F::OFF[i] : off;
          wstep[j] = part == i ? C::F::STEP[i] : wstep[j];
        }
      }
      wsrc[j] = reinterpret_cast<const char*>(gemm_row_ptr(a, vr, row_bytes)) + off;
    }
  }

  // Chunk c's x planes and W rows into stage `st` (C::VPS vector-memory
  // instructions per wave).
  __device__ __forceinline__ void issue(int c, char* st) const {
#pragma unroll
    for (int p = 0; p < C::PL; p++)
#pragma unroll
      for (int j = 0; j < C::XI; j++)
        lds_dma16(xsrc[p][j] + c * 64, st + p * C::XB + (wave * C::XPW + 64 * j) * 16);
#pragma unroll
    for (int j = 0; j < C::WI; j++) {
      const char* src = C::F::SB ? wsrc[j] + (size_t)(c >> 2) * C::F::SB + (((c & 3) * wstep[j]) & C::F::MASK)
                                 : wsrc[j] + c * C::UNIT;
      if (wact[j]) lds_dma16(src, st + C::PL * C::XB + (wave * C::WPW + 64 * j) * 16);
    }
    asm volatile("" ::: "memory");
  }

  // The dwords of the lane's W slice of chunk c in stage `st` (w_scales and
  // w_codes take them).  Q4_0 (5 dwords): the stage holds unit bytes [0,16)
  // [16,32) [20,36): block A's d + qs at dwords 0..4, block B's d in the high
  // half of dword 4 and its qs at dwords 8..11.  Packed (12 dwords): codes
  // 32h..32h+31, then scales 2h, 2h+1 and offsets 2h, 2h+1.
  __device__ __forceinline__ void wraw(const char* st, uint32_t (&w)[C::WD], int c, int mt = 0) const {
    const uint32_t* wb =
        reinterpret_cast<const uint32_t*>(st + C::PL * C::XB + (wm * 32 * C::MTILES + 32 * mt + li) * C::WROW);
    auto run = [&](int to, int from, int n) {
      for (int i = 0; i < n; i++) w[to + i] = wb[from + i];
    };
    constexpr int WF = C::FMT;
    if constexpr (WF == GEMM_W_Q4_K || WF == GEMM_W_IQ4_XS) {
      run(0, 0, 4);
      run(4, 4 + 4 * h, 4);
    } else if constexpr (WF == GEMM_W_Q8_0) {
      run(0, 12 * h, 8);
      w[8] = wb[12 * h + 11];
    } else if constexpr (WF == GEMM_W_Q5_0 || WF == GEMM_W_Q5_1) {
      run(0, 8 * h, 4);
      run(4, 8 * h + 6, 2);
    } else if constexpr (WF == GEMM_W_Q4_1) {
      run(0, 8 * h, 4);
      w[4] = wb[8 * h + 7];
    } else if constexpr (C::FLT) {
      // the lane's block h: logical pieces P*h .. P*h+P-1 of the row (P = 4
      // for F16, 8 for F32), each in its swizzled slot
      constexpr int P = C::WP / 2;
      const int sw = (li >> 1) & 7;
#pragma unroll
      for (int q = 0; q < P; q++) {
        const uint32_t* pc = wb + 4 * ((P * h + q) ^ sw);
#pragma unroll
        for (int i = 0; i < 4; i++) w[4 * q + i] = pc[i];
      }
    } else if constexpr (WF == GEMM_W_PACKED) {
      run(0, 8 * h, 8);
      run(8, 16 + 2 * h, 2);
      run(10, 20 + 2 * h, 2);
    } else {
      static_assert(WF == GEMM_W_Q4_0 || WF == GEMM_W_IQ4_NL, "not a format of the span kernel");
      run(0, 8 * h, 4);
      w[4] = wb[4];
    }
  }

  // The same reads as inline assembly, all issued at once (gemm_p_kernel).
  __device__ __forceinline__ void wraw_issue(const char* st, uint32_t (&w)[C::WD], int c, int mt) const {
    constexpr int WF = C::FMT, WO = C::PL * C::XB;  // the W rows follow the x planes in the stage
    const uint32_t wb = lds_addr(st + (wm * 32 * C::MTILES + 32 * mt + li) * C::WROW);
    auto put4 = [&](int to, cn_u32x4 v) { w[to] = v[0], w[to + 1] = v[1], w[to + 2] = v[2], w[to + 3] = v[3]; };
    auto put2 = [&](int to, uint2 v) { w[to] = v.x, w[to + 1] = v.y; };
    if constexpr (WF == GEMM_W_PACKED) {
      put4(0, lds_read128<WO>(wb + 32 * h));
      put4(4, lds_read128<WO + 16>(wb + 32 * h));
      put2(8, lds_read64<WO + 64>(wb + 8 * h));
      put2(10, lds_read64<WO + 80>(wb + 8 * h));
    } else if constexpr (WF == GEMM_W_Q4_K || WF == GEMM_W_IQ4_XS) {
      put4(0, lds_read128<WO>(wb));
      put4(4, lds_read128<WO + 16>(wb + 16 * h));
    } else if constexpr (WF == GEMM_W_Q5_K) {
      put4(0, lds_read128<WO>(wb));
      put4(4, lds_read128<WO + 32>(wb + 16 * h));
      w[8] = lds_read32<WO + 16>(wb + 8 * (c & 1) + 4 * h);
    } else if constexpr (WF == GEMM_W_Q2_K) {
      put4(0, lds_read128<WO>(wb));
      put4(4, lds_read128<WO + 16>(wb));
      put4(8, lds_read128<WO + 32>(wb));
      w[12] = lds_read32<WO + 60>(wb);
    } else if constexpr (WF == GEMM_W_Q8_0) {
      put4(0, lds_read128<WO>(wb + 48 * h));
      put4(4, lds_read128<WO + 16>(wb + 48 * h));
      w[8] = lds_read32<WO + 44>(wb + 48 * h);
    } else if constexpr (WF == GEMM_W_Q5_0 || WF == GEMM_W_Q5_1) {
      put4(0, lds_read128<WO>(wb + 32 * h));
      put2(4, lds_read64<WO + 24>(wb + 32 * h));
    } else if constexpr (WF == GEMM_W_Q4_1) {
      put4(0, lds_read128<WO>(wb + 32 * h));
      w[4] = lds_read32<WO + 28>(wb + 32 * h);
    } else {
      static_assert(WF == GEMM_W_Q4_0 || WF == GEMM_W_IQ4_NL, "not a format of the one-plane kernel");
      put4(0, lds_read128<WO>(wb + 32 * h));
      w[4] = lds_read32<WO + 16>(wb);
    }
  }

  // Where the 16-byte x fragment of MFMA step s, column tile cc, plane p lies.
  __device__ __forceinline__ const char* xfrag_ptr(const char* st, int p, int s, int cc) const {
    const int xrow = wn * 32 * C::TNW + 32 * cc + li;
    const int phys = (4 * h + s) ^ ((xrow >> 1) & 7);
    return st + p * C::XB + xrow * 128 + phys * 16;
  }

  // The 16-byte x fragment of MFMA step s, column tile cc, plane p.
  __device__ __forceinline__ uint4 xfrag(const char* st, int p, int s, int cc) const {
    const int xrow = wn * 32 * C::TNW + 32 * cc + li;
    const int phys = (4 * h + s) ^ ((xrow >> 1) & 7);
    return *reinterpret_cast<const uint4*>(st + p * C::XB + xrow * 128 + phys * 16);
  }

  // The output scale of each of the lane's columns: the one-plane kernel's x
  // of column n was scaled by 1 / xinv[n] (a power of two); 1 otherwise.
  // Loaded at the kernel's start, so the epilogue does not wait for it.
  template <int TN>
  __device__ __forceinline__ void load_scales(const GemmArgs& a, float (&sc)[TN]) const {
#pragma unroll
    for (int cc = 0; cc < TN; cc++) {
      const int n = n0 + wn * 32 * C::TNW + 32 * cc + li;
      sc[cc] = a.xinv ? a.xinv[n < a.N ? n : a.N - 1] : 1.0f;
    }
  }

  // Final tiles: K-split partials [splits][N][M] or the epilogue.
  template <int TN>
  __device__ __forceinline__ void store(const GemmArgs& a, const f32x16 (&acc)[TN], const float (&scl)[TN],
                                        int mt = 0) const {
#pragma unroll
    for (int cc = 0; cc < TN; cc++) {
      const int n = n0 + wn * 32 * C::TNW + 32 * cc + li;
      const float sc = scl[cc];
#pragma unroll
      for (int v4 = 0; v4 < 4; v4++) {
        const int m = m0 + wm * 32 * C::MTILES + 32 * mt + 8 * v4 + 4 * h;
        f32x4 v = f32x4{acc[cc][4 * v4], acc[cc][4 * v4 + 1], acc[cc][4 * v4 + 2], acc[cc][4 * v4 + 3]} * sc;
        if (a.splits > 1) {
          if (n < a.N && m < a.M) {
            float* p = a.part + ((size_t)ks * a.N + n) * a.M + m;
            if (m + 3 < a.M && (a.M & 3) == 0) *reinterpret_cast<f32x4*>(p) = v;
            else
              for (int i = 0; i < 4 && m + i < a.M; i++) p[i] = v[i];
          }
        } else {
          if constexpr (C::FMT == GEMM_W_F16_X3) f16_dot_again(a, n, m, v);
          write_out4(a, a.epi, n, m, v);
        }
      }
    }
  }
};

// One-plane kernel (chatnet_matmul): x as one fp16 plane in the cn_span_pos
// order, each column scaled by a power of two (to_f16_scaled_launch) that
// store() undoes.  The ring and the step order are the span kernel's (below):
// at the start of chunk c every wave has landed its part of the chunk and
// finished chunk c-1, chunk c+S-1 is issued into the freed stage, and each
// step's 8 weights are dequantized into one fp16 operand just ahead of its
// TN MFMAs (one v_mfma_f32_32x32x16_f16 per column tile).  Step s of lane
// half h: Q4_0 qs dword s of block h; packed codes 32h + 4s .. +3 and
// 32h + 16 + 4s .. +3 with the scale/offset pairs 2h and 2h+1.
template <int TN, int S, int WF, int MT, int WNC, bool SK>
__global__ __launch_bounds__(CN_BLOCK) __attribute__((amdgpu_waves_per_eu(SK ? 2 : 1, 2))) void gemm_p_kernel(GemmArgs a) {
  using C = PipeCfg<false, TN, S, WF, MT, WNC>;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  __shared__ int sk_last;
  TileIO<C> io(a);
  const int h = io.h;
  const uint32_t psel = h ? 0x03010200u : 0x05030402u;
  uint32_t magic = 0x64006400u;
  asm volatile("" : "+v"(magic));

  // Stream-K (SK): the launch's tiles x chunks of 64 as one sequence
  // (tile-major).  Workgroups 0 .. D-1 take tiles 0 .. D-1 whole; the other
  // G2 share the remaining tiles' chunks in equal ranges, each covering the
  // end of one tile and the start of the next at most.  Otherwise one
  // segment: the tile and K range of blockIdx.x.
  const int nc = a.K / 64;
  const long long units = (long long)a.sk_tiles * nc;
  constexpr bool sk = SK;
  const int D = a.sk_dp, G2 = a.sk_wgs - a.sk_dp;
  const long long u0 = (long long)D * nc, units2 = units - u0;
  auto lo_of = [&](int g) -> long long { return g < D ? (long long)g * nc : u0 + units2 * (g - D) / G2; };
  long long u = sk ? lo_of(blockIdx.x) : 0;
  const long long u_end = sk ? lo_of(blockIdx.x + 1) : 1;
  for (bool first = true; u < u_end; first = false) {
    int tile = 0;
    if constexpr (sk) {
      tile = (int)(u / nc);
      const int cb = (int)(u % nc);
      const int ce = (int)min((long long)nc, cb + (u_end - u));
      io.set_tile(a, tile, cb, ce);
      u += ce - cb;
      if (!first) __syncthreads();  // every wave is done with the previous segment's ring
    } else {
      u = u_end;
    }
    float xsc[TN];
    io.template load_scales<TN>(a, xsc);

    f32x16 acc[MT][TN];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int cc = 0; cc < TN; cc++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[mt][cc][v] = 0.f;

    const int c_begin = io.c_begin, c_end = io.c_end;
    if (c_begin < c_end) {
      auto slot_of = [&](int c) { return lds + ((c - c_begin) % S) * C::STAGE; };
#pragma unroll
      for (int i = 0; i < S - 1; i++)
        if (c_begin + i < c_end) io.issue(c_begin + i, lds + i * C::STAGE);
      for (int c = c_begin; c < c_end; c++) {
        char* st = slot_of(c);
        // chunks c+1 .. c+S-2 may stay in flight
        vm_wait_later<C::VPS, S - 2>(min(S - 2, c_end - 1 - c));
        wg_barrier();
        if (c + S - 1 < c_end) io.issue(c + S - 1, slot_of(c + S - 1));
        // the lane's W dwords (as wraw), then every x fragment of the chunk, all
        // issued at once; step s waits for its own fragments only
        uint32_t w[MT][C::WD];
#pragma unroll
        for (int mt = 0; mt < MT; mt++) io.wraw_issue(st, w[mt], c, mt);
        cn_u32x4 xr[4][TN];
#pragma unroll
        for (int s = 0; s < 4; s++) lds_read_xtiles<0, TN>(lds_addr(io.xfrag_ptr(st, 0, s, 0)), xr[s]);
        // Step s's W operands are dequantized during step s-1 (step 0's before
        // the first MFMA) and interleaved with its MFMAs: one wave issues in
        // order, so VALU work placed after a run of MFMAs waits behind them
        // while the matrix pipe drains; between them it runs in their shadow.
        WScale ws[MT];
        auto dequant = [&](int s, int mt) -> f16x8 {
          if constexpr (coded_format<WF>()) {
            uint32_t ca, cb;
            w_codes<WF>(w[mt], ws[mt], h, c, s, ca, cb);
            return dequant_u8_h(ca, cb, ws[mt].s0, ws[mt].o0, ws[mt].s1, ws[mt].o1);
          } else {
            const _Float16 d = __builtin_bit_cast(_Float16, (uint16_t)(h ? (w[mt][4] >> 16) : (w[mt][0] & 0xFFFFu)));
            return dequant_q4_h(__builtin_amdgcn_perm(w[mt][s + 1], w[mt][s], psel), magic, (cn_half2){d, d});
          }
        };
        // the W dwords and step 0's fragments: reads issued after them are
        // those of steps 1 .. 3
        lds_wait<(3 * TN > 15 ? 15 : 3 * TN)>();
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
          for (int i = 0; i < C::WD; i++) reg_fence(w[mt][i]);
        if constexpr (coded_format<WF>()) {
#pragma unroll
          for (int mt = 0; mt < MT; mt++) ws[mt] = w_scales<WF>(w[mt], h, c);
        }
        f16x8 wa[MT];
#pragma unroll
        for (int mt = 0; mt < MT; mt++) wa[mt] = dequant(0, mt);
#pragma unroll
        for (int s = 0; s < 4; s++) {
          if (s == 1) lds_wait<2 * TN>();
          else if (s == 2) lds_wait<TN>();
          else if (s == 3) lds_wait<0>();
#pragma unroll
          for (int cc = 0; cc < TN; cc++) reg_fence(xr[s][cc]);
          f16x8 xh[TN];
#pragma unroll
          for (int cc = 0; cc < TN; cc++) xh[cc] = __builtin_bit_cast(f16x8, xr[s][cc]);
          f16x8 wn[MT];
#pragma unroll
          for (int mt = 0; mt < MT; mt++) {
#pragma unroll
            for (int cc = 0; cc < TN; cc++) acc[mt][cc] = mma32(wa[mt], xh[cc], acc[mt][cc]);
          }
          if (s < 3) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++) wn[mt] = dequant(s + 1, mt);
            // one MFMA, then a share of the next step's dequantization, ...
            // VALU instructions per dequantized operand
            constexpr int kDequantValu = WF == GEMM_W_Q4_0 ? 14 : (WF == GEMM_W_PACKED ? 24 : 32);
            constexpr int kPer = (kDequantValu * MT + MT * TN - 1) / (MT * TN);
#pragma unroll
            for (int i = 0; i < MT * TN; i++) {
              __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
              __builtin_amdgcn_sched_group_barrier(0x002, kPer, 0);
            }
#pragma unroll
            for (int mt = 0; mt < MT; mt++) wa[mt] = wn[mt];
          }
          __builtin_amdgcn_sched_barrier(0);  // the next step's wait stays behind these MFMAs
        }
      }
    }
    if (!sk || (io.c_begin == 0 && io.c_end == nc)) {
#pragma unroll
      for (int mt = 0; mt < MT; mt++) io.template store<TN>(a, acc[mt], xsc, mt);
      continue;
    }
    // A tile shared by the workgroups gf .. gl (K order).  Each writes its
    // scaled part to a slot of its own (2g for its range's first segment,
    // 2g + 1 for its last; float j of thread t at j * CN_BLOCK + t) with
    // device-scope stores, waits for them, then arrives on the tile's counter.
    // The last to arrive reads the parts back with device-scope loads (its
    // own too, so that no accumulator stays live), sums them in K order as
    // the K-split reduce does (((0 + p_gf) + ...) + p_gl, whatever the
    // arrival order), applies the epilogue and sets the counter back to zero
    // for the next launch.  Device-scope accesses go past the XCD's L2 copy
    // without the L2-wide writeback and invalidation of a device fence (which
    // would empty the L2 under every other workgroup of the XCD).  No
    // workgroup waits for another.
    if constexpr (SK) {
      constexpr int NF = MT * TN * 16;  // floats per thread
      auto wg_of = [&](long long unit) {  // the workgroup whose range holds chunk `unit`
        return unit < u0 ? (int)(unit / nc) : D + (int)(((unit - u0 + 1) * G2 - 1) / units2);
      };
      auto slot = [&](int g) {
        const bool first_seg = lo_of(g) >= (long long)tile * nc;
        return a.part + (size_t)(2 * g + (first_seg ? 0 : 1)) * NF * CN_BLOCK + threadIdx.x;
      };
      const int gf = wg_of((long long)tile * nc), gl = wg_of((long long)tile * nc + nc - 1);
      float* mine = slot(blockIdx.x);
#pragma unroll
      for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int cc = 0; cc < TN; cc++)
#pragma unroll
          for (int v = 0; v < 16; v++)
            __hip_atomic_store(mine + ((mt * TN + cc) * 16 + v) * CN_BLOCK, acc[mt][cc][v] * xsc[cc], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the part has reached device scope
      __syncthreads();
      if (threadIdx.x == 0) {
        const unsigned arrived = __hip_atomic_fetch_add(a.tile_cnt + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sk_last = arrived == (unsigned)(gl - gf);
        if (sk_last) __hip_atomic_store(a.tile_cnt + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __syncthreads();
      if (sk_last) {
        // B contributors' parts per batch, every load of a batch in flight
        // together (one device-scope round trip per batch), added in K order
        constexpr int B = NF >= 64 ? 1 : 64 / NF;
        float sum[NF];
#pragma unroll
        for (int j = 0; j < NF; j++) sum[j] = 0.f;
        for (int g0 = gf; g0 <= gl; g0 += B) {
          float v[B][NF];
#pragma unroll
          for (int b = 0; b < B; b++) {
            const float* p = slot(min(g0 + b, gl));
#pragma unroll
            for (int j = 0; j < NF; j++) v[b][j] = __hip_atomic_load(p + j * CN_BLOCK, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
#pragma unroll
          for (int b = 0; b < B; b++)
            if (g0 + b <= gl)
#pragma unroll
              for (int j = 0; j < NF; j++) sum[j] += v[b][j];
        }
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
          for (int cc = 0; cc < TN; cc++)
#pragma unroll
            for (int v4 = 0; v4 < 4; v4++) {
              const int j = (mt * TN + cc) * 16 + 4 * v4;
              write_out4(a, a.epi, io.n0 + io.wn * 32 * TN + 32 * cc + io.li,
                         io.m0 + io.wm * 32 * MT + 32 * mt + 8 * v4 + 4 * h,
                         f32x4{sum[j], sum[j + 1], sum[j + 2], sum[j + 3]});
            }
      }
    }
  }
}

// Span kernel (the exact-weight product of the forward pass's spans: fp16 x
// hi + lo planes in the cn_span_pos order).  An S-stage ring (S = 2 or 3): at
// the start of chunk c every wave has landed its part of the chunk and finished
// chunk c-1, chunk c+S-1 is issued into the freed stage, and chunk c's W is
// dequantized step by step just ahead of its MFMAs.  Two stages take 44 KB of
// LDS (raw Q4_0, 64 columns), so three workgroups share a CU and one's VALU
// work and waits overlap the others' MFMAs; three stages keep two chunks in
// flight for grids of at most two workgroups per CU.  Step s of lane half h:
// Q4_0 qs dword s of block h (dequant_q4_f16), packed codes 32h + 4s .. +3
// and 32h + 16 + 4s .. +3 with the scale/offset pairs 2h and 2h+1.  Three
// fp16 MFMAs per step: Wa*xh + Wa*xl + Wb*xh, W = Wa + Wb exact for Q4_0 (~22
// bits for packed units), x = xh + xl to ~2^-22; the dropped Wb*xl term is
// below 2^-19 relative.
//
// GEMM_W_F16_X3 (chatnet_matmul's F16 rows): x in three planes of 11 bits each, 2^11
// apart and each in fp16's normal range, so that the fp32 elements down to 2^-28 of
// their column's largest meet the weights exactly (the planes hold 24 bits down to
// 2^-38; the matrix cores' sums keep about 2^-52 of the largest element.  Two planes
// held 22 of the 24 bits, and 2^-39 of the largest at best).  Every chunk's MFMA steps start from zero, the lowest
// plane's first, and the chunk sums are added with a running compensation (Kahan),
// so the product rounds no worse than the fp32 GEMV whose place it takes (relative
// error against float64 at K = 4096: GEMV 1.0e-7, one accumulator 5.9e-7, this
// 0.86e-7).  The third plane's products and loads cost 2 us of 18 at 24 columns of
// 4096 x 4096, 65 -> 88 at 512.
template <int TN, int S, int WF>
__global__ __launch_bounds__(CN_BLOCK) void gemm_s_kernel(GemmArgs a) {
  using C = PipeCfg<true, TN, S, WF>;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const TileIO<C> io(a);
  const int h = io.h;

  f32x16 acc[TN];
#pragma unroll
  for (int cc = 0; cc < TN; cc++)
#pragma unroll
    for (int v = 0; v < 16; v++) acc[cc][v] = 0.f;
  constexpr bool COMP = WF == GEMM_W_F16_X3;
  f32x16 sum[COMP ? TN : 1], com[COMP ? TN : 1];
  if constexpr (COMP) {
#pragma unroll
    for (int cc = 0; cc < TN; cc++) sum[cc] = com[cc] = acc[cc];
  }

  // v_perm_b32 selectors: qs dword s of the lane's block (2 bytes into the
  // unit for block A) as bytes b0 b2 b1 b3; 0x64006400 kept in a register
  // so each nibble pair takes one v_and_or_b32
  const uint32_t psel = h ? 0x03010200u : 0x05030402u;
  uint32_t magic = 0x64006400u;
  asm volatile("" : "+v"(magic));

  const int c_begin = io.c_begin, c_end = io.c_end;
  if (c_begin < c_end) {
    auto slot_of = [&](int c) { return lds + ((c - c_begin) % S) * C::STAGE; };
#pragma unroll
    for (int i = 0; i < S - 1; i++)
      if (c_begin + i < c_end) io.issue(c_begin + i, lds + i * C::STAGE);
    for (int c = c_begin; c < c_end; c++) {
      char* st = slot_of(c);
      // this wave's part of chunk c (chunk c+1 may stay in flight with three stages)
      if (S >= 3 && c + 1 < c_end) vm_wait<C::VPS>();
      else vm_wait<0>();
      wg_barrier();  // every wave's part landed, every wave done with chunk c-1
      if (c + S - 1 < c_end) io.issue(c + S - 1, slot_of(c + S - 1));
      uint32_t w[C::WD];
      io.wraw(st, w, c);
      cn_half2 dh2 = {}, dl2 = {};
      WScale ws{};
      if constexpr (coded_format<WF>()) ws = w_scales<WF>(w, h, c);
      if constexpr (WF == GEMM_W_Q4_0) {
        // d = dh + dl: dh keeps the top 8 significant bits of the fp16 scale
        const uint32_t d16 = h ? (w[4] >> 16) : (w[0] & 0xFFFFu);
        const _Float16 d = __builtin_bit_cast(_Float16, (uint16_t)d16);
        const _Float16 dh = __builtin_bit_cast(_Float16, (uint16_t)(d16 & 0xFFF8u));
        const _Float16 dl = d - dh;
        dh2 = (cn_half2){dh, dh};
        dl2 = (cn_half2){dl, dl};
      }
      f16x8 xh[2][TN], xl[2][TN];
      auto load_x = [&](int s, int b) {
#pragma unroll
        for (int cc = 0; cc < TN; cc++) {
          xh[b][cc] = __builtin_bit_cast(f16x8, io.xfrag(st, 0, s, cc));
          xl[b][cc] = __builtin_bit_cast(f16x8, io.xfrag(st, 1, s, cc));
        }
      };
      if constexpr (COMP) {
        // the lower planes' products first, while the sum is still 2^-11 of the
        // next one's: their rounding then does not count
#pragma unroll
        for (int p = 2; p >= 0; p--) {
#pragma unroll
          for (int s = 0; s < 4; s++) {
            const f16x8 wa =
                __builtin_bit_cast(f16x8, (cn_u32x4){w[2 * s], w[2 * s + 1], w[8 + 2 * s], w[9 + 2 * s]});
#pragma unroll
            for (int cc = 0; cc < TN; cc++)
              acc[cc] = mma32(wa, __builtin_bit_cast(f16x8, io.xfrag(st, p, s, cc)), acc[cc]);
          }
          if (p > 0) {
#pragma unroll
            for (int cc = 0; cc < TN; cc++) acc[cc] *= 0x1p-11f;
          }
        }
#pragma unroll
        for (int cc = 0; cc < TN; cc++) {
          add_compensated(sum[cc], com[cc], acc[cc]);
          acc[cc] = f32x16{};
        }
        continue;
      }
      load_x(0, 0);
#pragma unroll
      for (int s = 0; s < 4; s++) {
        if (s < 3) load_x(s + 1, (s + 1) & 1);
        f16x8 wa, wb;
        if constexpr (WF == GEMM_W_F16) {
          // elements 4s..4s+3 and 16+4s..16+4s+3 of the lane's block, already
          // fp16: W * (xh + xl), exact products
          wa = __builtin_bit_cast(f16x8, (cn_u32x4){w[2 * s], w[2 * s + 1], w[8 + 2 * s], w[9 + 2 * s]});
        } else if constexpr (WF == GEMM_W_F32) {
          // the same elements as fp32, split as W = Wa + Wb in fp16 (one
          // rounding each, ~22 bits together)
          uint32_t hi[4], lo[4];
#pragma unroll
          for (int k = 0; k < 2; k++) {
            cn_split_f16x2(__uint_as_float(w[4 * s + 2 * k]), __uint_as_float(w[4 * s + 2 * k + 1]), hi[k], lo[k]);
            cn_split_f16x2(__uint_as_float(w[16 + 4 * s + 2 * k]), __uint_as_float(w[16 + 4 * s + 2 * k + 1]),
                           hi[2 + k], lo[2 + k]);
          }
          wa = __builtin_bit_cast(f16x8, (cn_u32x4){hi[0], hi[1], hi[2], hi[3]});
          wb = __builtin_bit_cast(f16x8, (cn_u32x4){lo[0], lo[1], lo[2], lo[3]});
        } else if constexpr (coded_format<WF>()) {
          uint32_t ca, cb;
          w_codes<WF>(w, ws, h, c, s, ca, cb);
          dequant_u8_f16(ca, cb, ws.s0, ws.o0, ws.s1, ws.o1, wa, wb);
        } else {
          dequant_q4_f16(__builtin_amdgcn_perm(w[s + 1], w[s], psel), magic, dh2, dl2, wa, wb);
        }
#pragma unroll
        for (int cc = 0; cc < TN; cc++) acc[cc] = mma32(wa, xh[s & 1][cc], acc[cc]);
#pragma unroll
        for (int cc = 0; cc < TN; cc++) acc[cc] = mma32(wa, xl[s & 1][cc], acc[cc]);
        if constexpr (WF != GEMM_W_F16) {
#pragma unroll
          for (int cc = 0; cc < TN; cc++) acc[cc] = mma32(wb, xh[s & 1][cc], acc[cc]);
        }
      }
    }
  }
  float sc[TN];
  io.template load_scales<TN>(a, sc);
  if constexpr (COMP) io.template store<TN>(a, sum, sc);
  else io.template store<TN>(a, acc, sc);
}

template <int TN, int S, int WF, int MT, bool SK = false>
hipError_t launch_p(const GemmArgs& a, int grid, hipStream_t st) {
  constexpr int lds = PipeCfg<false, TN, S, WF, MT, 1>::LDS;
  static_assert(lds <= 160 * 1024, "LDS ring exceeds the CU's 160 KB");
  static std::atomic<uint64_t> lds_done{0};
  if (lds > 64 * 1024) {
    const hipError_t e = allow_full_lds(reinterpret_cast<const void*>(&gemm_p_kernel<TN, S, WF, MT, 1, SK>), lds_done);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((gemm_p_kernel<TN, S, WF, MT, 1, SK>), dim3(grid), dim3(CN_BLOCK), lds, st, a);
  return hipGetLastError();
}

// Stream-K launches run one-row-tile (MT = 1) instances.
template <int TN, int WF>
hipError_t launch_p_ring(const GemmArgs& a, int mt, int grid, hipStream_t st) {
  constexpr int S = TN == 1 ? 4 : 2;
  if (a.sk_wgs > 0) return launch_p<TN, S, WF, 1, true>(a, grid, st);
  if constexpr (TN == 4) {
    if (mt == 2) return launch_p<TN, S, WF, 2>(a, grid, st);
  }
  return launch_p<TN, S, WF, 1>(a, grid, st);
}

template <int TN, int S, int WF>
hipError_t launch_s(const GemmArgs& a, int grid, hipStream_t st) {
  constexpr int lds = PipeCfg<true, TN, S, WF>::LDS;
  static_assert(lds <= 160 * 1024, "LDS ring exceeds the CU's 160 KB");
  static std::atomic<uint64_t> lds_done{0};
  if (lds > 64 * 1024) {
    const hipError_t e = allow_full_lds(reinterpret_cast<const void*>(&gemm_s_kernel<TN, S, WF>), lds_done);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((gemm_s_kernel<TN, S, WF>), dim3(grid), dim3(CN_BLOCK), lds, st, a);
  return hipGetLastError();
}

template <int TN, int WF>
hipError_t launch_s_ring(const GemmArgs& a, int stages, int grid, hipStream_t st) {
  return stages == 2 ? launch_s<TN, 2, WF>(a, grid, st) : launch_s<TN, 3, WF>(a, grid, st);
}

// One format's instances (gemm_<format>.hip): the one-plane kernel with tn
// column tiles per wave and mt row tiles, the span kernel with a ring of
// `stages`.
template <int WF>
hipError_t launch_one_plane(const GemmArgs& a, int tn, int mt, int grid, hipStream_t st) {
  if (tn == 1) return launch_p_ring<1, WF>(a, 1, grid, st);
  if (tn == 2) return launch_p_ring<2, WF>(a, 1, grid, st);
  return launch_p_ring<4, WF>(a, mt, grid, st);
}

template <int WF>
hipError_t launch_span(const GemmArgs& a, int tn, int stages, int grid, hipStream_t st) {
  return tn == 1 ? launch_s_ring<1, WF>(a, stages, grid, st) : launch_s_ring<2, WF>(a, stages, grid, st);
}

template <int WF>
int span_ring_bytes_t(int tn, int stages) {
  if (stages == 2) return tn == 1 ? PipeCfg<true, 1, 2, WF>::LDS : PipeCfg<true, 2, 2, WF>::LDS;
  return tn == 1 ? PipeCfg<true, 1, 3, WF>::LDS : PipeCfg<true, 2, 3, WF>::LDS;
}

}  // namespace

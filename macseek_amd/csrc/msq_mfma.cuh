// MFMA building blocks for the multi-token paths (small-N matvec_n, the prefill matmul and the prefill MoE GEMMs).
//
// v_mfma_f32_16x16x32_{f16,bf16}: D[16 x 16] += A[16 x 32] . B[32 x 16], one wave.
//   A operand: lane l holds row  (l % 16), eight K positions 8 * (l / 16) .. + 7   (activations: row = token)
//   B operand: lane l holds col  (l % 16), the same eight K positions               (weights: col = weight row)
//   D operand: lane l holds col  (l % 16), rows 4 * (l / 16) + i, i = 0..3          (token, weight row)
// A and B only have to agree on which matrix column each K position means, so every format is free to pick the
// column order that makes its fragment cheap to decode (Frag::col_of).
//
// A fragment decoder turns the bytes of 8 weights of one row into 8 exact fp16 (or bf16) payloads plus an fp32 scale
// that is applied to the MFMA result, so weights are never rounded: weight = scale * payload (+ add, Q5_K only, which
// multiplies the per-token sum of the K step's activations).
#pragma once
#include "msq_device.cuh"

namespace msq {

typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));

constexpr int kMvnSubSteps = 8;   // K steps a wave of the small-N matvec fetches and multiplies at a time

__device__ __forceinline__ f4_t mfma_f16(const uint32_t a[4], const uint32_t b[4], f4_t c) {
  typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
  const u4_t av = {a[0], a[1], a[2], a[3]}, bv = {b[0], b[1], b[2], b[3]};
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, av), __builtin_bit_cast(h8_t, bv), c, 0, 0, 0);
}
__device__ __forceinline__ f4_t mfma_bf16(const uint32_t a[4], const uint32_t b[4], f4_t c) {
  typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
  const u4_t av = {a[0], a[1], a[2], a[3]}, bv = {b[0], b[1], b[2], b[3]};
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8_t, av), __builtin_bit_cast(bf8_t, bv), c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t pk_add_f16(uint32_t a, uint32_t b) {
  const h2_t r = as_h2(a) + as_h2(b);
  return __builtin_bit_cast(uint32_t, r);
}
// float -> bf16 bits, round to nearest even (finite inputs)
__device__ __forceinline__ uint32_t bf16_rne(float f) {
  const uint32_t u = __builtin_bit_cast(uint32_t, f);
  return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

// fp16(scale * payload + add) for both halves of a payload word: fp32 arithmetic on the fp16 payloads, one rounding
// (v_fma_mixlo_f16 / v_fma_mixhi_f16. Left to the compiler: the second reads the half that the first wrote, which wants a
// wait state between them that it does not insert inside or around inline assembly)
__device__ __forceinline__ uint32_t scale_round_h2(uint32_t h, float scale, float add) {
  const h2_t p = as_h2(h);
  const h2_t r = {(_Float16)__builtin_fmaf((float)p.x, scale, add), (_Float16)__builtin_fmaf((float)p.y, scale, add)};
  return __builtin_bit_cast(uint32_t, r);
}

// ================================================================================================ fragments
// Interface of a fragment decoder F (one K step = 32 matrix columns, chunk q = l / 16 of the step, 8 positions p):
//   BF16_MATH          payloads are bf16 (activations are then split into two bf16 terms) instead of fp16
//   HAS_ADD            weight = scale * payload + add
//   LDS_WORDS, fill_lds
//   col_of(q, p)       column (0..31 inside the step) that position p of chunk q stands for
//   get(row, step, q, tbl)   payloads of the 8 weights of weight row `row` (pointer to its first byte); the block
//                            formats split it into load_raw (the lane's bytes: loads only) and finish (table lookups
//                            and arithmetic), so that a kernel can request a step's bytes ahead of its arithmetic
struct FragOut {
  uint32_t h[4];
  float scale, add;
};

struct FragIQ1S {
  static constexpr bool BF16_MATH = false, HAS_ADD = false;
  static constexpr int WS_BYTES = 50;  // bytes of a row per 256 columns
  static constexpr int LDS_WORDS = MSQ_IQ1S_GRID_N * 4;
  __device__ static void fill_lds(uint32_t* lds, int tid, int nt) { copy_words16(lds, g_tbl_iq1s.w, LDS_WORDS, tid, nt); }
  __device__ static uint32_t col_of(uint32_t q, uint32_t p) { return 8u * q + p; }
  struct Raw { uint32_t qh, qs, d; };
  template <class P>
  __device__ static Raw load_raw(P row, uint32_t step, uint32_t q) {
    const P b = row + (step >> 3) * 50u;
    const uint32_t ib = step & 7u;
    return {ld16(b + 34 + 2 * ib), ld8(b + 2 + 4 * ib + q), ld16(b)};
  }
  __device__ static FragOut finish(const Raw& r, uint32_t, uint32_t q, const uint32_t* tbl) {
    const uint32_t qh = r.qh;
    const uint32_t idx = r.qs | (((qh >> (3 * q)) & 7u) << 8);
    const uint4 g = ((const uint4*)tbl)[idx];
    const uint32_t delta2 = (qh & 0x8000u) ? 0xB000B000u : 0x30003000u;  // -0.125 / +0.125 in both halves
    FragOut o;
    o.h[0] = pk_add_f16(g.x, delta2); o.h[1] = pk_add_f16(g.y, delta2);  // grid + delta is exact in fp16
    o.h[2] = pk_add_f16(g.z, delta2); o.h[3] = pk_add_f16(g.w, delta2);
    o.scale = half_bits_to_float(r.d) * (float)(2u * ((qh >> 12) & 7u) + 1u);
    o.add = 0.f;
    return o;
  }
  template <class P>
  __device__ static FragOut get(P row, uint32_t step, uint32_t q, const uint32_t* tbl) { return finish(load_raw(row, step, q), step, q, tbl); }
};

struct FragIQ2XXS {
  static constexpr bool BF16_MATH = false, HAS_ADD = false;
  static constexpr int WS_BYTES = 66;  // bytes of a row per 256 columns
  static constexpr int LDS_WORDS = MSQ_IQ2XXS_GRID_N * 4 + 128 * 4;
  __device__ static void fill_lds(uint32_t* lds, int tid, int nt) { DecIQ2XXS::fill_lds(lds, tid, nt); }
  __device__ static uint32_t col_of(uint32_t q, uint32_t p) { return 8u * q + p; }
  template <class W32>
  struct Raw { W32 a1; uint32_t gi, d; };
  template <class P>
  __device__ static auto load_raw(P row, uint32_t step, uint32_t q) {
    const P b = row + (step >> 3) * 66u;
    const P a8 = b + 2 + 8 * (step & 7u);
    return Raw<decltype(ld32_raw(a8))>{ld32_raw(a8 + 4), ld8(a8 + q), ld16(b)};
  }
  template <class R>
  __device__ static FragOut finish(const R& r, uint32_t, uint32_t q, const uint32_t* tbl) {
    const uint32_t a1 = fix(r.a1);
    const uint4 g = ((const uint4*)tbl)[r.gi];
    const uint4 s = ((const uint4*)(tbl + MSQ_IQ2XXS_GRID_N * 4))[(a1 >> (7 * q)) & 127u];
    FragOut o;
    o.h[0] = g.x ^ s.x; o.h[1] = g.y ^ s.y; o.h[2] = g.z ^ s.z; o.h[3] = g.w ^ s.w;
    o.scale = half_bits_to_float(r.d) * (0.5f + (float)(a1 >> 28)) * 0.25f;
    o.add = 0.f;
    return o;
  }
  template <class P>
  __device__ static FragOut get(P row, uint32_t step, uint32_t q, const uint32_t* tbl) { return finish(load_raw(row, step, q), step, q, tbl); }
};

struct FragQ8_0 {
  static constexpr bool BF16_MATH = false, HAS_ADD = false;
  static constexpr int WS_BYTES = 272;  // bytes of a row per 256 columns
  static constexpr int LDS_WORDS = 0;
  __device__ static void fill_lds(uint32_t*, int, int) {}
  __device__ static uint32_t col_of(uint32_t q, uint32_t p) { return 8u * q + p; }
  template <class W64>
  struct Raw { W64 v; uint32_t d; };
  template <class P>
  __device__ static auto load_raw(P row, uint32_t step, uint32_t q) {
    const P b = row + step * 34u;
    return Raw<decltype(ld64_raw(b))>{ld64_raw(b + 2 + 8 * q), ld16(b)};
  }
  template <class P>
  __device__ static FragOut get(P row, uint32_t step, uint32_t q, const uint32_t* tbl) { return finish(load_raw(row, step, q), step, q, tbl); }
  template <class R>
  __device__ static FragOut finish(const R& r, uint32_t, uint32_t, const uint32_t*) {
    const u64_a2 v = fix(r.v);
    const uint32_t lo = v.x ^ 0x80808080u, hi = v.y ^ 0x80808080u;  // bytes become q + 128
    const uint32_t bias = 0xE480E480u;                              // -1152 in both halves
    FragOut o;
    o.h[0] = pk_add_f16(bytes01_to_h2_1024(lo), bias); o.h[1] = pk_add_f16(bytes23_to_h2_1024(lo), bias);
    o.h[2] = pk_add_f16(bytes01_to_h2_1024(hi), bias); o.h[3] = pk_add_f16(bytes23_to_h2_1024(hi), bias);
    o.scale = half_bits_to_float(r.d);
    o.add = 0.f;
    return o;
  }
};

// IQ4_NL: byte j of a block holds columns j (low nibble) and j + 16 (high nibble); chunk q takes bytes 4q .. 4q + 3, so
// its positions (2i, 2i + 1) stand for columns (4q + i, 4q + i + 16) and one table lookup per byte yields both.
struct FragIQ4NL {
  static constexpr bool BF16_MATH = false, HAS_ADD = false;
  static constexpr int WS_BYTES = 144;  // bytes of a row per 256 columns
  static constexpr int LDS_WORDS = 256;
  __device__ static void fill_lds(uint32_t* lds, int tid, int nt) { copy_words16(lds, g_tbl_iq4nl.w, 256, tid, nt); }
  __device__ static uint32_t col_of(uint32_t q, uint32_t p) { return 4u * q + (p >> 1) + 16u * (p & 1u); }
  __device__ static uint32_t pos_of(uint32_t c) { return 8u * ((c & 15u) >> 2) + 2u * (c & 3u) + (c >> 4); }  // inverse of col_of
  template <class W32>
  struct Raw { W32 v; uint32_t d; };
  template <class P>
  __device__ static auto load_raw(P row, uint32_t step, uint32_t q) {
    const P b = row + step * 18u;
    return Raw<decltype(ld32_raw(b))>{ld32_raw(b + 2 + 4 * q), ld16(b)};
  }
  template <class R>
  __device__ static FragOut finish(const R& r, uint32_t, uint32_t, const uint32_t* tbl) {
    const uint32_t v = fix(r.v);
    FragOut o;
    o.h[0] = tbl[v & 0xFFu]; o.h[1] = tbl[(v >> 8) & 0xFFu]; o.h[2] = tbl[(v >> 16) & 0xFFu]; o.h[3] = tbl[v >> 24];
    o.scale = half_bits_to_float(r.d);
    o.add = 0.f;
    return o;
  }
  template <class P>
  __device__ static FragOut get(P row, uint32_t step, uint32_t q, const uint32_t* tbl) { return finish(load_raw(row, step, q), step, q, tbl); }
};

// Q6_K: the 16-column scale groups are half a K step wide, so a step is issued as two MFMAs (chunks 0-1, chunks 2-3);
// get() returns the scale of the lane's own half and get_scales() both halves' scales of the lane's row.
struct FragQ6K {
  static constexpr bool BF16_MATH = false, HAS_ADD = false;
  static constexpr int WS_BYTES = 210;  // bytes of a row per 256 columns
  static constexpr int LDS_WORDS = 0;
  __device__ static void fill_lds(uint32_t*, int, int) {}
  __device__ static uint32_t col_of(uint32_t q, uint32_t p) { return 8u * q + p; }
  template <class P>
  __device__ static FragOut get(P row, uint32_t step, uint32_t q, const uint32_t*) {
    const P b = row + (step >> 3) * 210u;
    const uint32_t e0 = 32u * (step & 7u) + 8u * q, h = e0 >> 7, k = (e0 & 127u) >> 5, l0 = e0 & 31u;
    const u64_a2 ql = ld64(b + 64 * h + 32 * (k & 1u) + l0), qh = ld64(b + 128 + 32 * h + l0);
    const uint32_t sh4 = 4u * (k >> 1), sh2 = 2u * k;
    const uint32_t q0 = ((ql.x >> sh4) & 0x0F0F0F0Fu) | (((qh.x >> sh2) & 0x03030303u) << 4);
    const uint32_t q1 = ((ql.y >> sh4) & 0x0F0F0F0Fu) | (((qh.y >> sh2) & 0x03030303u) << 4);
    const uint32_t bias = 0xE420E420u;  // -1056 = -(1024 + 32) in both halves
    FragOut o;
    o.h[0] = pk_add_f16(bytes01_to_h2_1024(q0), bias); o.h[1] = pk_add_f16(bytes23_to_h2_1024(q0), bias);
    o.h[2] = pk_add_f16(bytes01_to_h2_1024(q1), bias); o.h[3] = pk_add_f16(bytes23_to_h2_1024(q1), bias);
    o.scale = 0.f;
    o.add = 0.f;
    return o;
  }
  template <class W64>
  struct Raw { W64 ql, qh; uint32_t sc, d; };
  template <class P>
  __device__ static auto load_raw(P row, uint32_t step, uint32_t q) {
    const P b = row + (step >> 3) * 210u;
    const uint32_t e0 = 32u * (step & 7u) + 8u * q, h = e0 >> 7, k = (e0 & 127u) >> 5, l0 = e0 & 31u;
    return Raw<decltype(ld64_raw(b))>{ld64_raw(b + 64 * h + 32 * (k & 1u) + l0), ld64_raw(b + 128 + 32 * h + l0),
                                      ld16(b + 192 + 8 * h + 2 * k), ld16(b + 208)};
  }
  // (the scale of the lane's own half of the step: chunks 0-1 the first 16 columns, chunks 2-3 the second)
  template <class R>
  __device__ static FragOut finish(const R& r, uint32_t step, uint32_t q, const uint32_t*) {
    const uint32_t k = step & 3u;
    const uint32_t sh4 = 4u * (k >> 1), sh2 = 2u * k;
    const u64_a2 ql = fix(r.ql), qh = fix(r.qh);
    const uint32_t q0 = ((ql.x >> sh4) & 0x0F0F0F0Fu) | (((qh.x >> sh2) & 0x03030303u) << 4);
    const uint32_t q1 = ((ql.y >> sh4) & 0x0F0F0F0Fu) | (((qh.y >> sh2) & 0x03030303u) << 4);
    const uint32_t bias = 0xE420E420u;  // -1056 = -(1024 + 32) in both halves
    FragOut o;
    o.h[0] = pk_add_f16(bytes01_to_h2_1024(q0), bias); o.h[1] = pk_add_f16(bytes23_to_h2_1024(q0), bias);
    o.h[2] = pk_add_f16(bytes01_to_h2_1024(q1), bias); o.h[3] = pk_add_f16(bytes23_to_h2_1024(q1), bias);
    o.scale = half_bits_to_float(r.d) * (float)(int)(int8_t)(q < 2 ? r.sc & 0xFFu : r.sc >> 8);
    o.add = 0.f;
    return o;
  }
  template <class P>
  __device__ static void get_scales(P row, uint32_t step, float& sa, float& sb) {
    const P b = row + (step >> 3) * 210u;
    const uint32_t e0 = 32u * (step & 7u), h = e0 >> 7, k = (e0 & 127u) >> 5;
    const uint32_t sc = ld16(b + 192 + 8 * h + 2 * k);
    const float d = half_bits_to_float(ld16(b + 208));
    sa = d * (float)(int)(int8_t)(sc & 0xFFu);
    sb = d * (float)(int)(int8_t)(sc >> 8);
  }
};

struct FragQ5K {
  static constexpr bool BF16_MATH = false, HAS_ADD = true;
  static constexpr int WS_BYTES = 176;  // bytes of a row per 256 columns
  static constexpr int LDS_WORDS = 0;
  __device__ static void fill_lds(uint32_t*, int, int) {}
  __device__ static uint32_t col_of(uint32_t q, uint32_t p) { return 8u * q + p; }
  template <class W64, class W128>
  struct Raw { W64 ql, qh; W128 hdr; };  // hdr: d | dmin, then the 12 scale bytes
  template <class P>
  __device__ static auto load_raw(P row, uint32_t step, uint32_t q) {
    const P b = row + (step >> 3) * 176u;
    const uint32_t g = (step & 7u) >> 1, l0 = 8u * q;
    return Raw<decltype(ld64_raw(b)), decltype(ld128_raw(b))>{ld64_raw(b + 48 + 32 * g + l0), ld64_raw(b + 16 + l0), ld128_raw(b)};
  }
  template <class P>
  __device__ static FragOut get(P row, uint32_t step, uint32_t q, const uint32_t* tbl) { return finish(load_raw(row, step, q), step, q, tbl); }
  template <class R>
  __device__ static FragOut finish(const R& r, uint32_t step, uint32_t, const uint32_t*) {
    const uint32_t is = step & 7u, run = is & 1u;
    const u64_a2 ql = fix(r.ql), qh = fix(r.qh);
    const u128_a2 hdr = fix(r.hdr);
    const uint32_t q0 = ((ql.x >> (4 * run)) & 0x0F0F0F0Fu) | (((qh.x >> is) & 0x01010101u) << 4);
    const uint32_t q1 = ((ql.y >> (4 * run)) & 0x0F0F0F0Fu) | (((qh.y >> is) & 0x01010101u) << 4);
    const uint32_t bias = 0xE400E400u;  // -1024 in both halves
    // (all 12 scale bytes were fetched: a load inside a branch makes the waits that follow conservative)
    const uint32_t s0 = hdr.y, s1 = hdr.z, s2 = hdr.w;
    auto byte = [&](uint32_t i) { const uint32_t w = i < 4 ? s0 : i < 8 ? s1 : s2; return (w >> (8 * (i & 3u))) & 0xFFu; };
    uint32_t sc, mn;
    if (is < 4) { sc = byte(is) & 63u; mn = byte(is + 4) & 63u; }
    else { sc = (byte(is + 4) & 0xFu) | ((byte(is - 4) >> 6) << 4); mn = (byte(is + 4) >> 4) | ((byte(is) >> 6) << 4); }
    const uint32_t dd = hdr.x;
    FragOut o;
    o.h[0] = pk_add_f16(bytes01_to_h2_1024(q0), bias); o.h[1] = pk_add_f16(bytes23_to_h2_1024(q0), bias);
    o.h[2] = pk_add_f16(bytes01_to_h2_1024(q1), bias); o.h[3] = pk_add_f16(bytes23_to_h2_1024(q1), bias);
    o.scale = half_bits_to_float(dd & 0xFFFFu) * (float)sc;
    o.add = -(half_bits_to_float(dd >> 16) * (float)mn);
    return o;
  }
};

template <int QT>  // MSQ_F16 or MSQ_BF16
struct FragDense16 {
  static constexpr bool BF16_MATH = QT == MSQ_BF16, HAS_ADD = false, PLAIN = true;  // PLAIN: the payload is the weight
  static constexpr int LDS_WORDS = 0;
  __device__ static void fill_lds(uint32_t*, int, int) {}
  __device__ static uint32_t col_of(uint32_t q, uint32_t p) { return 8u * q + p; }
  template <class P>
  __device__ static FragOut get(P row, uint32_t step, uint32_t q, const uint32_t*) {
    const u128_a2 v = ld128(row + 64u * step + 16u * q);
    FragOut o;
    o.h[0] = v.x; o.h[1] = v.y; o.h[2] = v.z; o.h[3] = v.w;
    o.scale = 1.f;
    o.add = 0.f;
    return o;
  }
};

// ================================================================================================ block fragments
// For the 256-weight codebook formats the large-token GEMM uses a second decomposition: the payload is the whole weight,
// scale included, as fp16 (the reference's prefill kernels feed their matrix units dequantized fp16 tiles too; they
// round d * scale * grid once, src/kernels/quant_moe_prefill.metal:137-167, where finish() below rounds twice: the
// sub-block scale to fp16, then its product with the grid value, 2^-11 relative per weight at worst instead of
// 2^-12; the scale in fp32 would cost a second multiply per register), so a wave accumulates
// all of K in the matrix cores without touching the accumulators in between. Lane (row n, chunk q) owns the sub-blocks 2 q and 2 q + 1 of its row's block
// (16 contiguous bytes of IQ2_XXS), so no lane loads a byte twice; step j (0..7) of a block therefore covers, for chunk
// q, the 8 columns 64 q + 32 (j / 4) + 8 (j % 4) .. + 7 of the block, and the activation operand is read with the same mapping.
//   Raw / load(at, slot, sel)       the lane's bytes of one block from LDS (PIECES, piece_at, at_of: how they lie there)
//   lane_low(lane % 16)             low byte of the lane's lookup addresses
//   lookup<j>(raw, low)             table reads of step j, issued ahead of their use (the table starts the workgroup's LDS)
//   scale(raw, sub)                 scale of the lane's sub-block sub (0, 1), in both halves
//   finish(scale, look, h)          payloads of a step
__device__ __forceinline__ uint32_t pk_mul_f16(uint32_t a, uint32_t b) {
  const h2_t r = as_h2(a) * as_h2(b);
  return __builtin_bit_cast(uint32_t, r);
}

// A table entry's LDS address is assembled from whole bytes: v_perm puts an index byte above the low byte that the caller
// prepared (one instruction instead of a shift, a mask and an addition). The low byte's bits must not be known to the
// compiler, which otherwise turns the assembly back into an addition to a base.
typedef __attribute__((address_space(3))) const uint8_t* lds_cptr_t;
template <int BYTE>
__device__ __forceinline__ uint32_t byte_over(uint32_t w, uint32_t low) {  // byte BYTE of w at bits 8..15, byte 0 of low below it
  return __builtin_amdgcn_perm(w, low, 0x0c0c0000u | ((4u + BYTE) << 8));
}
__device__ __forceinline__ uint32_t bits_from(uint32_t mask, uint32_t a, uint32_t b) { return (mask & a) | (~mask & b); }  // v_bfi
__device__ __forceinline__ uint32_t opaque(uint32_t v) { asm("" : "+v"(v)); return v; }
template <class T>
__device__ __forceinline__ T lds_at(uint32_t at, uint32_t off) {
  typedef const __attribute__((address_space(3))) T* p_t;
  return *(p_t)((lds_cptr_t)(uintptr_t)at + off);
}

// A row's block bytes in LDS: the whole dwords from the block's start, rounded down to a dword, on, in PIECES 16-byte pieces.
// A block starts in the first dword's low half or in its high half: SEL_LOW picks bytes that start two bytes into a pair of
// dwords, and ^ SEL_FLIP picks the second dword of the pair (blocks and rows are whole 16-bit words).
constexpr uint32_t SEL_LOW = 0x05040302u, SEL_FLIP = 0x02020606u;
__device__ __forceinline__ uint32_t halves_of(uint32_t lo, uint32_t hi, uint32_t sel) { return __builtin_amdgcn_perm(hi, lo, sel); }

// IQ2_XXS keeps 16 copies of its grid table in LDS, copy c in the 16-byte bank column c of each 256-byte row: a 16-lane
// group whose lanes read "their" column (c = lane % 16) touches every bank exactly once whatever the entries are, so the
// random lookups run at the conflict-free rate. So does the sign table (SIGNS = 16) where there is room for it; four copies
// leave about two lanes to a bank column.
template <int SIGNS>
struct BlkIQ2XXS {
  // the sign table comes first: both table bases then fit the 16-bit offset field of the LDS instructions, and a lookup
  // address is the entry index above the lane's column
  static constexpr uint32_t GRID_AT = 128u * 16u * SIGNS;
  static constexpr int LDS_WORDS = GRID_AT / 4 + MSQ_IQ2XXS_GRID_N * 16 * 4, BLOCK_BYTES = 66;
  __device__ static void fill_lds(uint32_t* lds, int tid, int nt) {
    const uint4* grid = (const uint4*)g_tbl_iq2xxs.w;
    const uint4* sign = (const uint4*)g_tbl_sign.w;
    uint4* dst = (uint4*)lds;
    for (int i = tid; i < 128 * SIGNS; i += nt) dst[i] = sign[i / SIGNS];
    dst += 128 * SIGNS;
    for (int i = tid; i < MSQ_IQ2XXS_GRID_N * 16; i += nt) dst[i] = grid[i / 16];
  }
  struct Raw { uint32_t w[4]; uint32_t d; };  // {a0, a1} of sub-block 2 q, then of 2 q + 1; fp16 bits of d in the high half
  // 17 dwords (BlkIQ1S says why through LDS). Rows 8-15 hold pieces 0-3 in the order 1, 0, 3, 2: a 16-byte read serves eight
  // rows of chunk q and the other eight of chunk q ^ 1 together
  static constexpr int PIECES = 5;
  __device__ static uint32_t piece_at(uint32_t row, uint32_t p) { return p < 4u ? p ^ (row >> 3) : 4u; }
  // LDS addresses, from the slot's start, of what the lane reads of its row
  struct At { uint32_t x, tail, d; };
  __device__ static At at_of(uint32_t row, uint32_t q) {
    const uint32_t b = row * (16u * PIECES);
    return {b + 16u * piece_at(row, q), b + 16u * piece_at(row, q + 1u), b + 16u * piece_at(row, 0u)};
  }
  __device__ static Raw load(const At& at, uint32_t slot, uint32_t sel) {
    const u32x4 x = lds_at<u32x4>(at.x, slot);
    const uint32_t tail = lds_at<uint32_t>(at.tail, slot), d = lds_at<uint32_t>(at.d, slot);
    Raw r;
#pragma unroll
    for (int i = 0; i < 4; i++) r.w[i] = halves_of(x[i], i < 3 ? x[i + 1] : tail, sel);
    r.d = halves_of(d, d, sel);
    return r;
  }
  struct Look { u32x4 g, s; };
  // low bytes of a lane's lookup addresses: its columns of the two tables' rows of copies
  struct Low { uint32_t g, s; };
  __device__ static Low lane_low(uint32_t col) {
    Low l;
    l.g = opaque(col << 4);
    l.s = SIGNS == 16 ? l.g : opaque((col % SIGNS) << 4);
    return l;
  }
  template <int J>
  __device__ static Look lookup(const Raw& r, Low low) {
    constexpr int l = J & 3, at = SIGNS == 16 ? 8 : 6;  // the sign index goes to bits at .. at + 6
    const uint32_t a0 = r.w[2 * (J >> 2)], a1 = r.w[2 * (J >> 2) + 1];
    const uint32_t s7 = 7 * l < at ? a1 << (7 * l < at ? at - 7 * l : 0) : a1 >> (7 * l < at ? 0 : 7 * l - at);
    return {lds_at<u32x4>(byte_over<l>(a0, low.g), GRID_AT), lds_at<u32x4>(bits_from(127u << at, s7, low.s), 0u)};
  }
  // weight = fp16(fp16(d (2 s + 1) / 8) * (+-grid)): the whole scale rides in the payload, rounded to fp16 before the
  // multiply (the reference's tile rounds the fp32 product once, src/kernels/quant_moe_prefill.metal:153-167)
  __device__ static uint32_t scale(const Raw& r, int sub) {
    const uint32_t a1 = r.w[2 * sub + 1];
    const float m = (half_bits_to_float(r.d >> 16) * 0.125f) * (float)(((a1 >> 27) & 0x1Eu) | 1u);
    return pack_h2(m, m);
  }
  __device__ static void finish(uint32_t m2, const Look& k, uint32_t (&h)[4]) {
#pragma unroll
    for (int i = 0; i < 4; i++) h[i] = pk_mul_f16(k.g[i] ^ k.s[i], m2);
  }
};

// grid + delta as fp8 (E4M3 holds +-1/8, +-7/8 and +-9/8 exactly), once with either delta: an entry of eight is two words,
// and a weight is one conversion and one multiplication per pair. Trits as fp4 (one word an entry, 8 KB instead of 32) want
// an addition as well: 37 tokens of IQ1_S experts 597 us instead of 522, 4096 tokens 3.86 ms instead of 3.73. Entries of
// fp16 (16 bytes) make every lookup a 16-byte read at a random place.
struct TblIQ1S8 { uint32_t w[2][MSQ_IQ1S_GRID_N][2]; };
constexpr TblIQ1S8 make_iq1s8() {
  TblIQ1S8 t{};
  constexpr uint32_t fp8[2][3] = {{0xB6, 0x20, 0x39}, {0xB9, 0xA0, 0x36}};  // sign, four exponent bits (bias 7), three mantissa bits
  for (int i = 0; i < MSQ_IQ1S_GRID_N; i++) {
    unsigned c = msq_iq1s_code[i];
    for (int j = 0; j < 8; j++, c /= 3)
      for (int s = 0; s < 2; s++) t.w[s][i][j / 4] |= fp8[s][c % 3] << (8 * (j % 4));
  }
  return t;
}
__device__ __attribute__((aligned(16))) const TblIQ1S8 g_tbl_iq1s8 = make_iq1s8();
template <bool HIGH>
__device__ __forceinline__ uint32_t fp8_pair_to_h2(uint32_t w) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8((int)w, 1.f, HIGH));
}

struct BlkIQ1S {
  // Entry (b = qs byte, h = 3 bits of qh, sign of delta) lives at LDS byte b << 8 | (copy << 7) | sign << 6 | h << 3: two
  // copies, since one entry set of 256-byte pitch would sit in half of the banks
  static constexpr int LDS_WORDS = 8 * MSQ_IQ1S_GRID_N, BLOCK_BYTES = 50;
  __device__ static void fill_lds(uint32_t* lds, int tid, int nt) {
    for (int i = tid; i < 2 * MSQ_IQ1S_GRID_N; i += nt) {  // item i: sign, then entry h << 8 | b
      const uint2 v = ((const uint2*)&g_tbl_iq1s8.w[0][0][0])[i];
      uint2* dst = (uint2*)((uint8_t*)lds + ((i & 255) << 8) + ((i >> 11) << 6) + (((i >> 8) & 7) << 3));
      dst[0] = v;
      dst[16] = v;
    }
  }
  struct Raw { uint32_t qs[2]; uint32_t qh; uint32_t d; };  // qs bytes 8 q .. 8 q + 7; qh[2 q] | qh[2 q + 1] << 16; d in the high half
  // The lane's bytes come through LDS. Fetched from memory in fragment order neighbouring lanes touch different rows: 290
  // vector cache lookups per 16 rows and block (58 a load), one in every cycle of a launch with few tokens per expert; by
  // pieces about 18 a load. 13 dwords of a row fit four pieces: one load per 16 rows. Piece p sits at place p ^ (row / 4) % 4.
  static constexpr int PIECES = 4;
  __device__ static uint32_t piece_at(uint32_t row, uint32_t p) { return p ^ ((row >> 2) & 3u); }
  struct At { uint32_t x, tail, h0, h1, d; };
  __device__ static At at_of(uint32_t row, uint32_t q) {
    auto dw = [&](uint32_t i) { return row * (16u * PIECES) + 16u * piece_at(row, i >> 2) + 4u * (i & 3u); };
    return {dw(2u * q), dw(2u * q + 2u), dw(8u + q), dw(9u + q), dw(0u)};
  }
  __device__ static Raw load(const At& at, uint32_t slot, uint32_t sel) {
    const u32x2 x = lds_at<u32x2>(at.x, slot);
    const uint32_t tail = lds_at<uint32_t>(at.tail, slot), h0 = lds_at<uint32_t>(at.h0, slot), h1 = lds_at<uint32_t>(at.h1, slot), d = lds_at<uint32_t>(at.d, slot);
    return {{halves_of(x[0], x[1], sel), halves_of(x[1], tail, sel)}, halves_of(h0, h1, sel), halves_of(d, d, sel)};
  }
  struct Look { u32x2 g; };
  using Low = uint32_t;
  __device__ static uint32_t lane_low(uint32_t col) { return opaque((col & 1u) << 7); }
  template <int J>
  __device__ static Look lookup(const Raw& r, uint32_t low) {
    constexpr int l = J & 3, sh = 3 * l + 16 * (J >> 2);  // the entry's three bits of qh start at bit sh
    const uint32_t sgn = bits_from(0x40u, r.qh >> (J < 4 ? 9 : 25), low);
    const uint32_t h8 = sh < 3 ? r.qh << (sh < 3 ? 3 - sh : 0) : r.qh >> (sh < 3 ? 0 : sh - 3);
    return {lds_at<u32x2>(byte_over<l>(r.qs[J >> 2], bits_from(0x38u, h8, sgn)), 0u)};
  }
  // weight = fp16(s2 * (grid + delta)) with s2 = fp16(d (2 s + 1)): scale and product are rounded once each (the reference's
  // tile rounds the fp32 product once, src/kernels/quant_moe_prefill.metal:137-147)
  __device__ static uint32_t scale(const Raw& r, int sub) {
    const uint32_t qh = sub ? r.qh >> 16 : r.qh & 0xFFFFu;
    const float m = half_bits_to_float(r.d >> 16) * (float)(((qh >> 11) & 0xEu) | 1u);
    return pack_h2(m, m);
  }
  __device__ static void finish(uint32_t m2, const Look& k, uint32_t (&h)[4]) {
    h[0] = pk_mul_f16(fp8_pair_to_h2<false>(k.g[0]), m2); h[1] = pk_mul_f16(fp8_pair_to_h2<true>(k.g[0]), m2);
    h[2] = pk_mul_f16(fp8_pair_to_h2<false>(k.g[1]), m2); h[3] = pk_mul_f16(fp8_pair_to_h2<true>(k.g[1]), m2);
  }
};

}  // namespace msq

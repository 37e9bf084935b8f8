// Whole-buffer dequantization to fp32, bit-exact with the reference CPU dequantizer: every expression keeps the
// operand order of tests/ref/dequant.cpp:34-120 and floating-point contraction is off, so no multiply-subtract fuses.
// One thread produces 8 consecutive elements, or twice 8 of the K-quants.
#pragma once
#include "msq_device.cuh"

namespace msq {

__device__ __forceinline__ float tbl_half(const uint32_t* w, int j) {  // element j of an 8-half table entry
  const uint32_t v = w[j >> 1];
  return half_bits_to_float((j & 1) ? (v >> 16) : (v & 0xFFFFu));
}

template <class OUT>
__device__ __forceinline__ void put8(OUT* dst, const float (&y)[8]) {
  if constexpr (sizeof(OUT) == 4) {
    float4* o = (float4*)dst;
    o[0] = make_float4(y[0], y[1], y[2], y[3]);
    o[1] = make_float4(y[4], y[5], y[6], y[7]);
  } else {
    *(uint4*)dst = uint4{pack_h2(y[0], y[1]), pack_h2(y[2], y[3]), pack_h2(y[4], y[5]), pack_h2(y[6], y[7])};
  }
}

// OUT = float: the bit-exact fp32 result. OUT = uint16_t: the same values rounded to fp16 (nearest even), the weight
// operand of the prefill matmul (reference: q_deq_f16, src/kernels/quant_mm.metal:143-154).
template <int QT, class OUT = float>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t* __restrict__ src, OUT* __restrict__ dst, int64_t nchunks) {
#pragma clang fp contract(off)
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nchunks) return;
  float y[8];
  if constexpr (QT == MSQ_F32) {
    for (int j = 0; j < 8; j++) y[j] = __builtin_bit_cast(float, ld32(src + 4 * (8 * c + j)));
  } else if constexpr (QT == MSQ_F16) {
    for (int j = 0; j < 8; j++) y[j] = half_bits_to_float(ld16(src + 2 * (8 * c + j)));
  } else if constexpr (QT == MSQ_BF16) {
    for (int j = 0; j < 8; j++) y[j] = bf16_bits_to_float(ld16(src + 2 * (8 * c + j)));
  } else if constexpr (QT == MSQ_Q8_0) {  // dequant.cpp:40-45
    const uint8_t* b = src + (c >> 2) * 34;
    const float d = half_bits_to_float(ld16(b));
    const uint8_t* q = b + 2 + 8 * (c & 3);
    for (int j = 0; j < 8; j++) y[j] = (float)(int8_t)q[j] * d;
  } else if constexpr (QT == MSQ_IQ4_NL) {  // dequant.cpp:107-112
    const uint8_t* b = src + (c >> 2) * 18;
    const float d = half_bits_to_float(ld16(b));
    const int part = (int)(c & 3);
    const uint8_t* q = b + 2 + 8 * (part & 1);
    for (int j = 0; j < 8; j++) {
      const int nib = part < 2 ? (q[j] & 0xF) : (q[j] >> 4);
      y[j] = d * half_bits_to_float(g_tbl_iq4nl.w[nib] & 0xFFFFu);  // low half of entry b = kv[b & 15]
    }
  } else if constexpr (QT == MSQ_IQ1_S) {  // dequant.cpp:77-91
    const uint8_t* b = src + (c >> 5) * 50;
    const int r = (int)(c & 31), ib = r >> 2, l = r & 3;
    const float d = half_bits_to_float(ld16(b));
    const uint32_t qh = ld16(b + 34 + 2 * ib);
    const float dl = d * (float)(2 * ((qh >> 12) & 7) + 1);
    const float delta = (qh & 0x8000) ? -0.125f : 0.125f;
    const uint32_t* g = g_tbl_iq1s.w + 4 * (b[2 + r] | (((qh >> (3 * l)) & 7) << 8));
    for (int j = 0; j < 8; j++) y[j] = dl * (tbl_half(g, j) + delta);
  } else if constexpr (QT == MSQ_IQ2_XXS) {  // dequant.cpp:92-106
    const uint8_t* b = src + (c >> 5) * 66;
    const int r = (int)(c & 31), ib = r >> 2, l = r & 3;
    const float d = half_bits_to_float(ld16(b));
    const uint8_t* a8 = b + 2 + 8 * ib;
    const uint32_t a1 = ld32(a8 + 4);
    const float db = d * (0.5f + (float)(a1 >> 28)) * 0.25f;
    const uint32_t* g = g_tbl_iq2xxs.w + 4 * a8[l];
    const uint32_t si = (a1 >> (7 * l)) & 127u;
    const uint32_t sg = si | ((__builtin_popcount(si) & 1u) << 7);
    for (int j = 0; j < 8; j++) y[j] = db * tbl_half(g, j) * ((sg >> j) & 1u ? -1.f : 1.f);
  }
  put8(dst + 8 * c, y);
}

// Q6_K, Q5_K: a thread takes eight low bytes and so 16 weights, eight from either nibble (64 and 32 elements apart: of fp16 eight
// threads store 128 consecutive bytes of Q6_K, four threads 64 of Q5_K), and works on words of four. Bound by memory as far as the
// launch is long: one nibble and a byte at a time (16 vector instructions a weight) took Q6_K 32768x1280 29.5 us, 1024x4096 7.7.
template <int QT, class OUT>
__global__ __launch_bounds__(256) void dequant_kq_kernel(const uint8_t* __restrict__ src, OUT* __restrict__ dst, int64_t nchunks) {
#pragma clang fp contract(off)
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nchunks) return;
  const uint32_t u = (uint32_t)c & 15u, l0 = 8u * (u & 3u);
  constexpr uint32_t BLOCK = QT == MSQ_Q6_K ? 210u : 176u;
  const uint8_t* b = src + (c >> 4) * BLOCK;
  OUT* o = dst + (c >> 4) * 256;
  float y[2][8];
  auto bytes = [](uint32_t w, float* f) {  // the four bytes of a word
    f[0] = (float)(w & 0xFFu); f[1] = (float)((w >> 8) & 0xFFu); f[2] = (float)((w >> 16) & 0xFFu); f[3] = (float)(w >> 24);
  };
  if constexpr (QT == MSQ_Q6_K) {  // dequant.cpp:60-76: elements 128 h + 32 k + l0 .. of runs k = kk and kk + 2
    const uint32_t h = u >> 3, kk = (u >> 2) & 1u;
    const u64_a2 ql = ld64(b + 64u * h + 32u * kk + l0), qh = ld64(b + 128u + 32u * h + l0);
    const uint8_t* s = b + 192u + 8u * h + (l0 >> 4) + 2u * kk;
    const float d = half_bits_to_float(ld16(b + 208));
#pragma unroll
    for (int r = 0; r < 2; r++) {
      const float ds = d * (float)(int)(int8_t)ld8(s + 4 * r);
      const uint32_t sh = 2u * kk + 4u * r;
      bytes(((ql.x >> (4 * r)) & 0x0F0F0F0Fu) | (((qh.x >> sh) & 0x03030303u) << 4), y[r]);
      bytes(((ql.y >> (4 * r)) & 0x0F0F0F0Fu) | (((qh.y >> sh) & 0x03030303u) << 4), y[r] + 4);
#pragma unroll
      for (int j = 0; j < 8; j++) y[r][j] = ds * (y[r][j] - 32.f);  // (q - 32 is exact)
    }
    o += 128u * h + 32u * kk + l0;
    put8(o, y[0]);
    put8(o + 64, y[1]);
  } else {  // dequant.cpp:46-59, scale unpack :29-32: elements 64 g + l0 .. of runs 2 g and 2 g + 1
    const uint32_t g = u >> 2;
    const u64_a2 ql = ld64(b + 48u + 32u * g + l0), qh = ld64(b + 16u + l0);
    const u128_a2 hdr = ld128(b);  // d, dmin, the twelve scale bytes s
    // s[i], s[i + 4], s[i + 8] of i = 2 g (mod 4) and the byte behind
    const uint32_t sh8 = 16u * (g & 1u), s0 = hdr.y >> sh8, s4 = hdr.z >> sh8, s8 = hdr.w >> sh8;
    const float d = half_bits_to_float(hdr.x & 0xFFFFu), mn = half_bits_to_float(hdr.x >> 16);
#pragma unroll
    for (int r = 0; r < 2; r++) {
      const uint32_t a = (s0 >> (8 * r)) & 0xFFu, e = (s4 >> (8 * r)) & 0xFFu, f = (s8 >> (8 * r)) & 0xFFu;
      const uint32_t sc = g < 2u ? a & 63u : (f & 0xFu) | ((a >> 6) << 4), m = g < 2u ? e & 63u : (f >> 4) | ((e >> 6) << 4);
      const float d1 = d * (float)sc, m1 = mn * (float)m;
      bytes(((ql.x >> (4 * r)) & 0x0F0F0F0Fu) | (((qh.x >> (2u * g + r)) & 0x01010101u) << 4), y[r]);
      bytes(((ql.y >> (4 * r)) & 0x0F0F0F0Fu) | (((qh.y >> (2u * g + r)) & 0x01010101u) << 4), y[r] + 4);
#pragma unroll
      for (int j = 0; j < 8; j++) y[r][j] = d1 * y[r][j] - m1;
    }
    o += 64u * g + l0;
    put8(o, y[0]);
    put8(o + 32, y[1]);
  }
}

// one launch over n_elems weights (whole blocks)
template <int QT, class OUT>
void launch_dequant(hipStream_t st, const uint8_t* src, OUT* dst, int64_t n_elems) {
  constexpr bool kq = QT == MSQ_Q6_K || QT == MSQ_Q5_K;
  const int64_t n = n_elems / (kq ? 16 : 8);
  const dim3 grid((unsigned)((n + 255) / 256)), block(256);
  if constexpr (kq) hipLaunchKernelGGL((dequant_kq_kernel<QT, OUT>), grid, block, 0, st, src, dst, n);
  else hipLaunchKernelGGL((dequant_kernel<QT, OUT>), grid, block, 0, st, src, dst, n);
}

}  // namespace msq

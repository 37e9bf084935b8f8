// Host side of the few-token product (msq_rows.cuh).
#include <algorithm>

#include "msq_host.h"
#include "msq_rows.cuh"

namespace msq {
namespace {

// workgroups: as many as are resident (four waves per SIMD, LDS), each a run of consecutive row tiles
template <class F>
size_t rows_lds(uint32_t waves, int S, int UT, int TT, bool gu = false) {
  return (size_t)F::LDS_WORDS * 4 + (size_t)rows_red_words(waves, UT, TT, gu) * 4 + (size_t)waves * rows_ring<F>(S);
}
uint32_t rows_tiles_per_wg(uint32_t ntiles, uint32_t waves, size_t lds, uint32_t blocks) {
  const uint32_t per_cu = std::max<uint32_t>(1, std::min<uint32_t>(16 / waves, (uint32_t)(kMaxLds / lds)));
  const uint32_t slots = std::max<uint32_t>(1, (uint32_t)device_info().cus * per_cu / blocks);
  return (ntiles + slots - 1) / slots;
}
template <class F, int BPW, int S, int NT, int UT, bool ROUND = false, bool XH = false, int TT = 1, bool GU = false>
int launch_nt(hipStream_t st, RowsArgs a, uint32_t waves) {
  const size_t lds = rows_lds<F>(waves, S, UT, TT, GU);
  if (lds > (size_t)kMaxLds) return MSQ_ERR_UNSUPPORTED;
  const int rc = allow_large_lds(mm_rows_kernel<F, BPW, S, NT, UT, ROUND, XH, TT, GU>, lds);
  if (rc != MSQ_OK) return rc;
  a.ntiles = (a.rows + 15) / 16;
  const uint32_t blocks = ROUND || XH ? (a.n + 16 * TT - 1) / (16 * TT) : 1;
  a.tiles_per_wg = rows_tiles_per_wg(a.ntiles, waves, lds, blocks);
  if (GU) { a.ntiles *= 2; a.tiles_per_wg *= 2; }
  if (a.rows_per_group != a.rows) {  // a workgroup's tiles belong to one group
    const uint32_t tg = a.rows_per_group / 16;
    while (tg % a.tiles_per_wg) a.tiles_per_wg--;
  }
  const uint32_t grid = (a.ntiles + a.tiles_per_wg - 1) / a.tiles_per_wg;
  hipLaunchKernelGGL((mm_rows_kernel<F, BPW, S, NT, UT, ROUND, XH, TT, GU>), dim3(grid, blocks), dim3(64 * waves), lds, st, a);
  MSQ_HIP(hipGetLastError());
  return MSQ_OK;
}
template <class F, int BPW, int S, int UT>
int launch(hipStream_t st, const RowsArgs& a, uint32_t waves) {
  return a.n <= 8 ? launch_nt<F, BPW, S, 8, UT>(st, a, waves) : launch_nt<F, BPW, S, 16, UT>(st, a, waves);
}
// one stage per wave up to 4096 columns, two stages up to 8192; rings of two stages, four of the small codebook blocks. Up to 2048
// columns, where there is LDS to spare, two tiles per meeting, but for workgroups of a single tile, which would carry an empty one
// through it (against two, 4000 random calls: up to eight tokens 1.00 to 1.10, more 1.01 to 1.15; IQ4_NL up to eight tokens 0.95 to 1.02;
// with two tiles and more 0.86 to 1.1), and of a single wave (1.01 to 1.28).
template <class F>
int launch_f(hipStream_t st, const RowsArgs& a) {
  constexpr int S = rows_slot<F>() <= 2048 ? 4 : 2;
  if (a.nws <= 8) {
    const bool one = rows_tiles_per_wg((a.rows + 15) / 16, a.nws, rows_lds<F>(a.nws, S, 2, 1), 1) == 1 && !(std::is_same_v<F, FragIQ4NL> && a.n <= 8);
    return one || a.nws == 1 ? launch<F, 1, S, 1>(st, a, a.nws) : launch<F, 1, S, 2>(st, a, a.nws);
  }
  if (a.nws <= 16) return launch<F, 1, S, 1>(st, a, a.nws);
  if (a.nws <= 32) return launch<F, 2, S, 1>(st, a, (a.nws + 1) / 2);
  return MSQ_ERR_UNSUPPORTED;
}

// Which calls of msq_matvec_n it serves, from what was measured against the dot-product kernel (few tokens) and the fused
// kernel of msq_matmul (nine and more) at 256 to 32768 rows x 768 to 8192 columns of every format; the lines lie where no
// shape on this side of them was more than 2 % behind. In brackets: the other kernel's time over this one's.
//  * nine tokens and more: up to 4096 columns everywhere (1.0 to 2.9), IQ4_NL, whose dot products are cheap, beyond 2048
//    columns from 1536 rows on (1536x4096 1.10; 512x3072 0.93). Two stages a wave (more than 4096 columns) want the row
//    tiles to fill half of the device, one workgroup a tile: Q5_K 1280x5120 0.93, 2048x5120 1.00, 2304x5120 1.07, Q6_K
//    1536x7168 0.97, 2048x7168 1.07, IQ4_NL 1536x8192 0.90, 2048x8192 1.14; the codebook formats from 1280 rows on (IQ1_S
//    1024x7168 0.96, 1280x7168 1.04, IQ2_XXS 1024x7680 0.89, 1280x7680 1.02);
//  * five to eight: up to 4096 columns, IQ4_NL and IQ2_XXS beyond 3072 in tall matrices only (IQ4_NL 1024x4096 0.93, 1280x4096
//    1.03, IQ2_XXS 512x3328 0.93, 512x4096 0.94, 1024x4096 1.00); beyond, from 1280 rows on (Q6_K 1024x7680 0.96, 1280x7680 1.07), IQ2_XXS
//    from 2048 past 6144 columns (1280x8192 0.91, 2048x8192 1.07), IQ4_NL from 3072 on (1.08 to 3.0);
//  * three and four: up to 4096 columns but for IQ4_NL (up to 2048) and IQ2_XXS (3072: 512x4096 0.92, 6144x4096 0.97, 8752x5376
//    0.93); the others in tall matrices beyond, Q6_K up to 6144 columns (6144x7168 0.98), Q5_K and IQ1_S up to 7168 (1.0 to 1.5),
//    where the row tiles fill the device's last round by more than half (Q6_K 4448x5888, 278 tiles on 256 CUs, 0.96);
//  * two: tall K-quant matrices of 256, 768 or 1280 columns, whose units neither fill the dot-product kernel's waves nor pair
//    up (Q6_K 20480x768 1.20, 24576x1280 1.12, 32768x1280 1.19; 18432x1280 0.95 to 0.99, 32768x1024 0.95, 32768x2048 0.97).
// A single stage (up to 256 columns) is a workgroup of one wave, which fills a codebook's table alone: IQ1_S 0.48 to 0.74,
// IQ2_XXS up to eight tokens from 1024 rows on (1.1 to 3.4; twelve tokens 0.76); the K-quants up to eight (1.4 to 2.7; fourteen
// 0.73), IQ4_NL beyond eight tokens from 1536 rows on (1024x256 0.94). IQ1_S of two stages wants 1536 rows
// (1024x512 0.95). Groups want 768 rows in all (IQ2_XXS 256x4096 in eight groups 0.82, IQ1_S 640x768 0.94), and the codebook
// formats with three or four tokens at most 16384 (a workgroup's tiles belong to one group: IQ1_S 27648x2816 0.83).
bool serves(int t, int rows, uint32_t nws, int cols, int n, int groups) {
  const bool iq4 = t == MSQ_IQ4_NL, iq2 = t == MSQ_IQ2_XXS, iq1 = t == MSQ_IQ1_S, kq = t == MSQ_Q6_K || t == MSQ_Q5_K;
  if (rows < (groups > 1 ? 768 : 256)) return false;
  if (nws == 1 && (iq1 || (iq4 && rows < 1536 && n >= 9) || (iq2 && (rows < 1024 || n >= 9)) || (kq && groups == 1 && n >= 9))) return false;
  if (iq1 && nws == 2 && rows < 1536) return false;
  if (groups > 1 && n < 5 && (iq1 || iq2) && rows > 16384) return false;
  if (n >= 9) return nws <= (iq4 ? 8u : 16u) || rows >= (nws <= 16 ? 1536 : kq || iq4 ? 2048 : 1280);
  if (nws <= 8 && n >= 3) return true;
  if (n >= 5) {
    if (nws <= 16) return iq4 ? nws <= 12 || rows >= 1280 : iq2 ? nws <= 12 || rows >= 1024 : true;
    return rows >= (iq4 ? 3072 : iq2 && nws > 24 ? 2048 : 1280);
  }
  if (n >= 3) {
    if (nws <= 16) return iq2 ? nws <= 12 : !iq4;
    const int tiles = (rows + 15) / 16, cus = device_info().cus;
    return !iq2 && !iq4 && rows >= 3072 && nws <= (t == MSQ_Q6_K ? 24u : 28u) && 5 * tiles >= 3 * cus * ((tiles + cus - 1) / cus);
  }
  return kq && nws <= 5 && cols % 512 && rows >= 20480;
}

// Blocks of sixteen or of 32 tokens (TT = 2: a decoded fragment feeds two matrix instructions, activations and partial tiles
// take twice the registers and LDS)? Row tiles per workgroup either way, t1 and t2, decide, since a launch takes about 5.7 +
// 2.9 t1 or 7.5 + 3.5 t2 us (IQ4_NL, 4096 columns). Measured over 20000 random calls that came here before, time with sixteen
// over time with 32, median (lowest of 100): up to 2048 columns, t1 over t2: 3 / 2 1.12 (0.98), 4 / 2 1.24, 5 / 3 1.14, 7 / 4 1.27; 4 / 3
// 0.98 (0.89), 2 / 2 0.90, 2 / 1 1.01 (0.89); beyond 2 / 1 1.10 (1.00), 3 / 2 1.08, 4 / 2 1.26, 5 / 3 1.20. Up to 512 rows, whose few
// tiles make t1 and t2 coarse, 0.8 to 1.2: sixteen. The sums are the same either way.
template <class F, bool XH>
int launch_mm(hipStream_t st, const RowsArgs& a) {
  constexpr int S = rows_slot<F>() <= 2048 ? 4 : 2;
  const uint32_t nt = (a.rows + 15) / 16, b1 = (a.n + 15) / 16, b2 = (a.n + 31) / 32;
  auto tiles = [&](int UT, int TT) { return rows_tiles_per_wg(nt, a.nws, rows_lds<F>(a.nws, S, UT, TT), TT == 1 ? b1 : b2); };
  if (a.nws <= 8) {
    const uint32_t t1 = tiles(2, 1), t2 = tiles(2, 2);
    if (a.rows > 512 && t1 >= 3 && 2 * t1 >= 3 * t2) return launch_nt<F, 1, S, 16, 2, true, XH, 2>(st, a, a.nws);
    return t1 == 1 ? launch_nt<F, 1, S, 16, 1, true, XH>(st, a, a.nws) : launch_nt<F, 1, S, 16, 2, true, XH>(st, a, a.nws);
  }
  const uint32_t t1 = tiles(1, 1), t2 = tiles(1, 2);
  if (a.rows > 512 && 5 * t1 >= 6 * t2 + 3) return launch_nt<F, 1, S, 16, 1, true, XH, 2>(st, a, a.nws);
  return launch_nt<F, 1, S, 16, 1, true, XH>(st, a, a.nws);
}
template <bool XH>
int launch_mm(hipStream_t st, int t, const RowsArgs& a) {
  switch (t) {
    case MSQ_Q6_K: return launch_mm<FragQ6K, XH>(st, a);
    case MSQ_Q5_K: return launch_mm<FragQ5K, XH>(st, a);
    case MSQ_IQ4_NL: return launch_mm<FragIQ4NL, XH>(st, a);
    case MSQ_IQ1_S: return launch_mm<FragIQ1S, XH>(st, a);
    case MSQ_IQ2_XXS: return launch_mm<FragIQ2XXS, XH>(st, a);
  }
  return MSQ_ERR_UNSUPPORTED;
}

}  // namespace

// The same for a call of msq_matmul over fp32 or fp16 activations: a workgroup a run of row tiles of one 16-token block, no
// K slices and so no second launch and no shared buffer. The weights are unpacked once per 16 tokens and the activations
// read once per workgroup, so it serves products of little work: more than 16 tokens (up to 16 msq_matvec_n is the call),
// up to 4096 columns (a stage per wave) and at most three weight stages (16 rows x 256 columns x 16 tokens) per wave of the
// device; four where the other route still unpacks in its product (up to 256 tokens, 2048 rows). Measured against the fused,
// the tile and the dequantize-then-GEMM route over every format, fp32 and fp16 activations, 64 to 8192 rows; in brackets the
// others' time over this one's. Three stages: 1.0 to 1.7; three to four beyond 256 tokens 0.78 (IQ1_S 768 columns) to 1.2.
//  * two stages a row (workgroups of two waves: the activations, and a codebook's table, are used by few): at most two per
//    wave of the device (IQ1_S 512 columns 1.04 to 1.3 there, at three 0.72 to 1.0) and 4096 rows (IQ1_S 8192x512 0.89);
//  * one stage a row: never (IQ1_S 1024x256 at 256 tokens 0.78, 2048x256 at 1024 0.72, Q5_K 6000x256 at 256 0.73);
//  * more than 4096 rows of five stages and more: up to 32 tokens (Q5_K 8192x1280 at 48 0.89, IQ1_S 8192x2048 at 48 0.93);
//    never more than 8192 (IQ1_S 16384x1536 at 17 0.86);
//  * two workgroups a token block at least, or a part of the device has none (IQ1_S 202x1536 at 2387, 150 blocks, 0.75).
//
// ... and in blocks of 32 tokens more work, up to 256 tokens (serves_32), `work` of it per wave of the device in units of 16 rows x
// 256 columns x 32 tokens. Measured over 28000 random calls against the route that each took before, median (lowest of 100):
//  * up to 64 tokens (not 33 to 39, whose second block is nearly empty) at 1280 to 4096 columns, work of at most five: IQ4_NL 1.59
//    (1.24), IQ2_XXS 1.55 (1.24), Q6_K 1.40 (1.11), IQ1_S 1.41 (1.10) but for more than 16384 rows (32768x1280 at 32 0.95) and 40 to 47
//    tokens (0.94 to 1.0), Q5_K 1.27 likewise (16427x1536 at 54 0.90, 10437x3840 at 42 0.96; fp16 activations, 48 to 55 tokens, 1.12
//    but 0.92 to 0.98 in one call of twenty, 10620x3328, 15500x2304);
//  * Q6_K of fp16 activations at 40 to 48 tokens over more than 16384 rows of 1280 or 1536 columns goes in steps, and so does the fused
//    kernel: not in the first half of every 4096 rows (0.88 to 1.09, mean 0.97; the other half 0.97 to 1.17); 1792 columns 0.89 to 0.96
//    at 14400 to 14900, 20800 to 21600 and 22700 rows, 1.03 to 1.3 between;
//  * in two launches of half the columns, 6144 to 8192: from 5120 rows on for the codebook formats and IQ4_NL (1.1 to 1.9; 3500 rows
//    0.87 to 1.2; IQ1_S from 40 tokens on and of fp32 activations, 0.9 with fp16), from 6144 rows on for the K-quants up to 32 tokens
//    (1.05 to 1.5; 5120 rows 0.86, more tokens 0.7 to 1.2); but not where the row tiles have just begun another round of the
//    workgroups and the fused kernel's slices come out even (two_launches_lose(); 0.92 to 1.09, median 0.99; the rest from 0.976 on);
//  * 65 to 128 tokens: IQ4_NL from 1536 columns on, work of at most seven (1.36, lowest 1.0; 20587x1536 at 102, 7.5, 0.94); Q6_K
//    from 3584 on, Q5_K 4096, at most eight (1.33; Q5_K 4500x3584 at 114 0.91); the codebook formats have the tile kernel;
//  * 129 to 256 tokens: 1152 to 2048 rows of 1536 columns and more, at most four (1.2 to 1.7).
bool two_launches_lose(int t, int rows, int cols, int n, bool x_half) {
  const bool narrow = cols > 6144 && cols <= 6656, iq2 = t == MSQ_IQ2_XXS, iq4 = t == MSQ_IQ4_NL;
  if (t == MSQ_Q5_K) return narrow && !x_half && rows <= 6512;
  if (n <= 32) return iq4 && cols >= 6400 && cols < 6656 && rows <= 5440;
  if (iq2 && cols > 7168 && cols <= 7424) return rows <= 5440;
  return narrow && (iq2 || iq4) && (rows <= 6144 ? n <= 48 && rows <= 5440 : rows <= 6512);
}
bool serves_32(int t, int rows, int cols, int n, bool x_half) {
  const size_t nws = ((size_t)cols + 255) / 256;
  const bool iq4 = t == MSQ_IQ4_NL, iq1 = t == MSQ_IQ1_S, q5 = t == MSQ_Q5_K, kq = q5 || t == MSQ_Q6_K;
  const size_t work = ((size_t)rows + 15) / 16 * nws * (((size_t)n + 31) / 32), waves = 16 * (size_t)device_info().cus;
  if (n <= 16 || nws > 32 || (n > 32 && n < 40)) return false;
  if (nws > 16)
    return n <= 64 && nws >= 24 && work <= 5 * waves && (kq ? n <= 32 && rows >= 6144 : rows >= 5120 && !(iq1 && (n <= 32 || x_half))) &&
           !two_launches_lose(t, rows, cols, n, x_half);
  if (t == MSQ_Q6_K && x_half && n > 32 && n <= 48 && nws <= 6 && rows > 16384) {
    const size_t cus = (size_t)device_info().cus;
    if (2 * ((((size_t)rows + 15) / 16 - 1) % cus) < cus) return false;
  }
  if (n <= 32) return nws >= 5 && work <= 5 * waves && !(iq1 && rows > 16384);
  if (n <= 64) return nws >= 5 && work <= 5 * waves && !((iq1 || q5) && (rows > 16384 || n < 48));
  if (n <= 128) return iq4 ? nws >= 6 && work <= 7 * waves : kq && nws >= (q5 ? 16u : 14u) && work <= 8 * waves;
  return n <= 256 && nws >= 6 && rows >= 1152 && rows <= 2048 && work <= 4 * waves;
}
bool matmul_rows_serves(int t, int rows, int cols, int n, const void* X, bool x_half, size_t x_stride) {
  switch (t) {
    case MSQ_Q6_K: case MSQ_Q5_K: case MSQ_IQ4_NL: case MSQ_IQ1_S: case MSQ_IQ2_XXS: break;
    default: return false;
  }
  const size_t nws = ((size_t)cols + 255) / 256, waves = 16 * (size_t)device_info().cus;
  if (cols % 128 || ((uintptr_t)X & (x_half ? 7 : 15)) || x_stride % 4 || x_stride > 0xFFFFFFFFull) return false;
  if (serves_32(t, rows, cols, n, x_half)) return true;
  const size_t stages = ((size_t)rows + 15) / 16 * nws * (((size_t)n + 15) / 16);
  if (n <= 16 || nws < 2 || nws > 16 || rows > 8192 || 2 * (((size_t)n + 15) / 16) > (size_t)device_info().cus) return false;
  if ((nws == 2 && rows > 4096) || (nws > 4 && rows > 4096 && n > 32)) return false;
  return stages <= waves * (nws == 2 ? 2 : n <= 256 && rows <= 2048 ? 4 : 3);
}
int matmul_rows(hipStream_t st, int t, const uint8_t* W, int rows, int cols, const void* X, bool x_half, size_t x_stride, float* Y, int n,
                int accumulate) {
  RowsArgs a{};
  a.W = W; a.X = X; a.Y = Y;
  a.n = (uint32_t)n; a.rows = (uint32_t)rows; a.cols = (uint32_t)cols; a.x_stride = (uint32_t)x_stride;
  a.row_bytes = (uint32_t)msq_type_row_bytes(t, cols); a.accumulate = accumulate ? 1u : 0u;
  a.rows_per_group = (uint32_t)rows; a.x_group_stride = 0; a.nws = ((uint32_t)cols + 255) / 256;
  // rows of more than sixteen weight stages in pieces of equal length, each a launch of its own that adds to the one before
  const uint32_t pieces = (a.nws + 15) / 16, per = (a.nws + pieces - 1) / pieces, ws = (uint32_t)msq_type_row_bytes(t, 256);
  for (uint32_t s0 = 0; s0 < a.nws; s0 += per) {
    RowsArgs b = a;
    b.W = a.W + (size_t)s0 * ws;
    b.X = (const uint8_t*)X + (size_t)s0 * 256 * (x_half ? 2 : 4);
    b.nws = std::min(per, a.nws - s0); b.cols = std::min(per * 256, a.cols - s0 * 256);
    b.w_bytes = a.rows * a.row_bytes - s0 * ws;
    if (s0) b.accumulate = 1u;
    const int rc = x_half ? launch_mm<true>(st, t, b) : launch_mm<false>(st, t, b);
    if (rc != MSQ_OK) return rc;
  }
  return MSQ_OK;
}

// A shared expert of a K-quant / Q8_0 type over few tokens (fp16 activations, fp32 scales as in the small-N product): gate, up and
// SwiGLU in one launch, or the down product.
namespace {
template <class F>
bool shared_fits(uint32_t nws_gu, uint32_t nws_dn) {  // a workgroup's waves and their LDS
  const uint32_t gu = (nws_gu + 1) / 2, dn = nws_dn <= 16 ? nws_dn : (nws_dn + 1) / 2;
  return gu <= 16 && dn <= 16 && rows_lds<F>(gu, 2, 2, 1, true) <= (size_t)kMaxLds && rows_lds<F>(dn, 2, 1, 1) <= (size_t)kMaxLds;
}
template <class F>
int launch_shared(hipStream_t st, const RowsArgs& a, bool gu) {
  if (gu) return launch_nt<F, 2, 2, 16, 2, false, true, 1, true>(st, a, (a.nws + 1) / 2);
  return a.nws <= 16 ? launch_nt<F, 1, 2, 16, 1, false, true>(st, a, a.nws) : launch_nt<F, 2, 2, 16, 1, false, true>(st, a, (a.nws + 1) / 2);
}
}  // namespace
bool shared_rows_serves(int t, int dim, int inter) {
  const uint32_t g = (uint32_t)dim / 256, d = (uint32_t)inter / 256;
  return t == MSQ_Q6_K ? shared_fits<FragQ6KG>(g, d) : t == MSQ_Q8_0 && shared_fits<FragQ8_0>(g, d);
}
int shared_rows(hipStream_t st, int t, const uint8_t* W, const uint8_t* up, int rows, int cols, const uint16_t* X, uint16_t* H, float* Z, int n) {
  RowsArgs a{};
  a.W = W; a.W1 = up; a.X = X; a.Y = Z; a.H = H;
  a.n = (uint32_t)n; a.rows = (uint32_t)rows; a.cols = (uint32_t)cols; a.x_stride = (uint32_t)cols;
  a.row_bytes = (uint32_t)msq_type_row_bytes(t, cols); a.rows_per_group = (uint32_t)rows; a.nws = (uint32_t)cols / 256;
  a.w_bytes = a.rows * a.row_bytes;
  return t == MSQ_Q6_K ? launch_shared<FragQ6KG>(st, a, up != nullptr) : launch_shared<FragQ8_0>(st, a, up != nullptr);
}

bool matvec_rows_serves(int t, int rows, int cols, int n, int groups, const void* X) {
  switch (t) {
    case MSQ_Q6_K: case MSQ_Q5_K: case MSQ_IQ4_NL: case MSQ_IQ1_S: case MSQ_IQ2_XXS: break;
    default: return false;
  }
  const uint32_t nws = ((uint32_t)cols + 255) / 256;
  return cols % 128 == 0 && nws <= 32 && (groups == 1 || rows / groups % 16 == 0) && !((uintptr_t)X & 15) &&
         msq_type_row_bytes(t, cols) * (size_t)rows <= 0xFFFFFF00ull && serves(t, rows, nws, cols, n, groups);
}
int matvec_rows(hipStream_t st, int t, const uint8_t* W, int rows, int cols, const float* X, float* Y, int n, int accumulate, int groups) {
  RowsArgs a{};
  a.W = W; a.X = X; a.Y = Y;
  a.n = (uint32_t)n; a.rows = (uint32_t)rows; a.cols = (uint32_t)cols; a.x_stride = (uint32_t)cols * (uint32_t)groups;
  a.row_bytes = (uint32_t)msq_type_row_bytes(t, cols); a.accumulate = accumulate ? 1u : 0u;
  a.rows_per_group = (uint32_t)(rows / groups); a.x_group_stride = (uint32_t)cols; a.nws = ((uint32_t)cols + 255) / 256;
  a.w_bytes = a.rows * a.row_bytes;
  switch (t) {
    case MSQ_Q6_K: return launch_f<FragQ6KG>(st, a);
    case MSQ_Q5_K: return launch_f<FragQ5K>(st, a);
    case MSQ_IQ4_NL: return launch_f<FragIQ4NL>(st, a);
    case MSQ_IQ1_S: return launch_f<FragIQ1S>(st, a);
    case MSQ_IQ2_XXS: return launch_f<FragIQ2XXS>(st, a);
  }
  return MSQ_ERR_UNSUPPORTED;
}

}  // namespace msq

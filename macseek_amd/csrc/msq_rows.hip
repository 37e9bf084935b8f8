// Host side of the few-token product (msq_rows.cuh).
#include <algorithm>

#include "msq_host.h"
#include "msq_rows.cuh"

namespace msq {
namespace {

// workgroups: as many as are resident (four waves per SIMD, LDS), each a run of consecutive row tiles
template <class F, int BPW, int S, int NT, int UT, bool ROUND = false, bool XH = false>
int launch_nt(hipStream_t st, RowsArgs a, uint32_t waves) {
  const size_t lds = (size_t)F::LDS_WORDS * 4 + (size_t)waves * (2 * UT * 16 * 16 * 4 + rows_ring<F>(S));
  if (lds > (size_t)kMaxLds) return MSQ_ERR_UNSUPPORTED;
  const int rc = allow_large_lds(mm_rows_kernel<F, BPW, S, NT, UT, ROUND, XH>, lds);
  if (rc != MSQ_OK) return rc;
  a.ntiles = (a.rows + 15) / 16;
  const uint32_t per_cu = std::max<uint32_t>(1, std::min<uint32_t>(16 / waves, (uint32_t)(kMaxLds / lds)));
  const uint32_t blocks = ROUND ? (a.n + 15) / 16 : 1;
  const uint32_t slots = std::max<uint32_t>(1, (uint32_t)device_info().cus * per_cu / blocks);
  a.tiles_per_wg = (a.ntiles + slots - 1) / slots;
  if (a.rows_per_group != a.rows) {  // a workgroup's tiles belong to one group
    const uint32_t tg = a.rows_per_group / 16;
    while (tg % a.tiles_per_wg) a.tiles_per_wg--;
  }
  const uint32_t grid = (a.ntiles + a.tiles_per_wg - 1) / a.tiles_per_wg;
  hipLaunchKernelGGL((mm_rows_kernel<F, BPW, S, NT, UT, ROUND, XH>), dim3(grid, blocks), dim3(64 * waves), lds, st, a);
  MSQ_HIP(hipGetLastError());
  return MSQ_OK;
}
template <class F, int BPW, int S, int UT>
int launch(hipStream_t st, const RowsArgs& a, uint32_t waves) {
  return a.n <= 8 ? launch_nt<F, BPW, S, 8, UT>(st, a, waves) : launch_nt<F, BPW, S, 16, UT>(st, a, waves);
}
// one stage per wave up to 4096 columns (with LDS to spare up to 2048: two tiles per meeting), two stages up to 8192; rings
// of two stages, four of the small codebook blocks
template <class F>
int launch_f(hipStream_t st, const RowsArgs& a) {
  constexpr int S = rows_slot<F>() <= 2048 ? 4 : 2;
  if (a.nws <= 8) return launch<F, 1, S, 2>(st, a, a.nws);
  if (a.nws <= 16) return launch<F, 1, S, 1>(st, a, a.nws);
  if (a.nws <= 32) return launch<F, 2, S, 1>(st, a, (a.nws + 1) / 2);
  return MSQ_ERR_UNSUPPORTED;
}

// Which calls it serves, from what was measured against the dot-product kernel (few tokens) and the fused kernel of
// msq_matmul (nine and more) at 512 to 32768 rows x 1024 to 8192 columns of every format:
//  * nine tokens and more: everywhere (1.1x to 2.7x) but for matrices of few rows and many columns, whose handful of row
//    tiles leaves most CUs idle while one workgroup decodes all of K (Q6_K 512x6144 at 16: 9.5 us against 7.9; IQ4_NL,
//    whose dot products are cheap, 512x3072: 6.3 against 5.8);
//  * three to eight: up to 2048 columns everywhere (Q6_K 512x1024 at 4: 3.7 against 5.3), up to 4096 for IQ4_NL from five
//    tokens on (7168x4096 at 4: 11.3 against 10.6, at 6: 11.6 against 14.1), beyond 4096 with the rows to fill the chip
//    (Q6_K 1536x6144 at 4 / 8: 8.2 / 8.3 against 8.1 / 9.9, 3072x6144: 9.3 / 9.7 against 10.4 / 13.6);
//  * two: only tall K-quant matrices (Q6_K 32768x1280: 12.3 against 13.9; 6144x3072: 8.4 against 7.3).
bool serves(int t, int rows, uint32_t nws, int n) {
  const bool iq4 = t == MSQ_IQ4_NL;
  if (rows < 256) return false;
  if (n >= 9) return nws <= (iq4 ? 8u : 16u) || rows >= (iq4 ? 1536 : 1024);
  if (n >= 3) {
    if (nws <= 8) return true;
    if (nws <= 16) return !iq4 || n >= 5;
    return n >= 5 ? rows >= (iq4 ? 3072 : 1024) : !iq4 && nws <= 28 && rows >= 3072;
  }
  return (t == MSQ_Q6_K || t == MSQ_Q5_K) && nws <= 8 && rows >= 16384;
}

template <class F, bool XH>
int launch_mm(hipStream_t st, const RowsArgs& a) {
  constexpr int S = rows_slot<F>() <= 2048 ? 4 : 2;
  if (a.nws <= 8) return launch_nt<F, 1, S, 16, 2, true, XH>(st, a, a.nws);
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
// read once per workgroup, so it serves products of little work: more than 16 tokens (up to 16 msq_matvec_n is the call)
// and at most four weight stages (16 rows x 256 columns x 16 tokens) per wave of the device, three from 2049 rows on,
// where a workgroup's activations are used for fewer tiles; up to 4096 columns (a stage per wave). Measured against the
// fused, the tile and the dequantize-then-GEMM route (us, these first): IQ4_NL 1024x2048 at 17 / 100 / 512 tokens 8.0 / 12.9 / 31.2
// -> 5.6 / 7.1 / 18.1, at 768 (six) 28.5 against 28.0; Q6_K 577x4096 at 100 12.6 -> 10.6, 4096x1536 at 128 (three) 19.2 -> 16.0, at 192
// (four and a half) 21.5 against 25.7; 1024x4096 at 256 (four) 19.5 -> 17.5, at 384 (six) 27.1 against 30.1; IQ1_S 512x1024
// at 256 11.0 -> 6.6, 16384x1536 at 17 (three) 14.6 against 17.0: not beyond 8192 rows.
int matmul_rows(hipStream_t st, int t, const uint8_t* W, int rows, int cols, const void* X, bool x_half, size_t x_stride, float* Y, int n,
                int accumulate) {
  const size_t rb = msq_type_row_bytes(t, cols);
  const uint32_t nws = ((uint32_t)cols + 255) / 256;
  const size_t stages = ((size_t)rows + 15) / 16 * nws * (((size_t)n + 15) / 16);
  if (cols % 128 || nws > 16 || n <= 16 || rows > 8192 || stages > (rows <= 2048 ? 16384u : 12288u) || ((uintptr_t)X & (x_half ? 7 : 15)) ||
      x_stride % 4 || x_stride > 0xFFFFFFFFull)
    return MSQ_ERR_UNSUPPORTED;
  RowsArgs a{};
  a.W = W; a.X = X; a.Y = Y;
  a.n = (uint32_t)n; a.rows = (uint32_t)rows; a.cols = (uint32_t)cols; a.x_stride = (uint32_t)x_stride;
  a.row_bytes = (uint32_t)rb; a.accumulate = accumulate ? 1u : 0u;
  a.rows_per_group = (uint32_t)rows; a.x_group_stride = 0; a.nws = nws;
  return x_half ? launch_mm<true>(st, t, a) : launch_mm<false>(st, t, a);
}

// MSQ_ERR_UNSUPPORTED, without a message, when the call is another kernel's
int matvec_rows(hipStream_t st, int t, const uint8_t* W, int rows, int cols, const float* X, float* Y, int n, int accumulate, int groups) {
  const int rpg = rows / groups;
  const size_t rb = msq_type_row_bytes(t, cols);
  const uint32_t nws = ((uint32_t)cols + 255) / 256;
  if (cols % 128 || (groups > 1 && rpg % 16) || ((uintptr_t)X & 15) || rb * (size_t)rows > 0xFFFFFF00ull || !serves(t, rows, nws, n))
    return MSQ_ERR_UNSUPPORTED;
  RowsArgs a{};
  a.W = W; a.X = X; a.Y = Y;
  a.n = (uint32_t)n; a.rows = (uint32_t)rows; a.cols = (uint32_t)cols; a.x_stride = (uint32_t)cols * (uint32_t)groups;
  a.row_bytes = (uint32_t)rb; a.accumulate = accumulate ? 1u : 0u;
  a.rows_per_group = (uint32_t)rpg; a.x_group_stride = (uint32_t)cols; a.nws = nws;
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

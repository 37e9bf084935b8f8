// Host side of the few-token product (msq_rows.cuh).
#include <algorithm>

#include "msq_host.h"
#include "msq_rows.cuh"

namespace msq {
namespace {

// workgroups: as many as are resident (four waves per SIMD, LDS), each a run of consecutive row tiles
template <class F, int BPW, int S, int NT, int UT>
int launch_nt(hipStream_t st, RowsArgs a, uint32_t waves) {
  const size_t lds = (size_t)F::LDS_WORDS * 4 + (size_t)waves * (2 * UT * 16 * 16 * 4 + rows_ring<F>(S));
  if (lds > (size_t)kMaxLds) return MSQ_ERR_UNSUPPORTED;
  const int rc = allow_large_lds(mm_rows_kernel<F, BPW, S, NT, UT>, lds);
  if (rc != MSQ_OK) return rc;
  a.ntiles = (a.rows + 15) / 16;
  const uint32_t per_cu = std::max<uint32_t>(1, std::min<uint32_t>(16 / waves, (uint32_t)(kMaxLds / lds)));
  const uint32_t slots = (uint32_t)device_info().cus * per_cu;
  a.tiles_per_wg = (a.ntiles + slots - 1) / slots;
  if (a.rows_per_group != a.rows) {  // a workgroup's tiles belong to one group
    const uint32_t tg = a.rows_per_group / 16;
    while (tg % a.tiles_per_wg) a.tiles_per_wg--;
  }
  const uint32_t grid = (a.ntiles + a.tiles_per_wg - 1) / a.tiles_per_wg;
  hipLaunchKernelGGL((mm_rows_kernel<F, BPW, S, NT, UT>), dim3(grid), dim3(64 * waves), lds, st, a);
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

}  // namespace

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

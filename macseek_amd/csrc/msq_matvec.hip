// C ABI: library bring-up, geometry queries, decode matvec and dequantization (see include/msq.h).
#include <algorithm>
#include <map>
#include <mutex>
#include <utility>

#include "msq_deq.cuh"
#include "msq_host.h"
#include "msq_mv.cuh"
#include "msq_mvq.cuh"

namespace msq {

thread_local char g_err[512] = "";

const DeviceInfo& device_info() {
  static const DeviceInfo info = [] {
    DeviceInfo d{0, 256};
    int dev = 0;
    hipDeviceProp_t p;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&p, dev) == hipSuccess) {
      d.cus = p.multiProcessorCount > 0 ? p.multiProcessorCount : 256;
      d.ok = strncmp(p.gcnArchName, "gfx950", 6) == 0;
    }
    return d;
  }();
  return info;
}

int grant_large_lds(const void* kernel, size_t lds) {
  static std::mutex mu;
  static std::map<std::pair<const void*, int>, size_t> granted;
  int dev = 0;
  MSQ_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  size_t& g = granted[{kernel, dev}];
  if (lds > g) {
    MSQ_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    g = lds;
  }
  return MSQ_OK;
}

// Plain streaming read: every workgroup walks contiguous 16 KiB chunks grid-stride, one 128-bit load per lane per step.
__global__ __launch_bounds__(1024) void bw_probe_kernel(const uint4* __restrict__ src, size_t n16, uint32_t* __restrict__ sink) {
  uint4 acc = {0, 0, 0, 0};
  const size_t chunk = 1024;  // uint4 per workgroup step
  for (size_t base = (size_t)blockIdx.x * chunk; base < n16; base += (size_t)gridDim.x * chunk) {
    const size_t i = base + threadIdx.x;
    if (i < n16) { const uint4 v = src[i]; acc.x ^= v.x; acc.y ^= v.y; acc.z ^= v.z; acc.w ^= v.w; }
  }
  const uint32_t r = acc.x ^ acc.y ^ acc.z ^ acc.w;
  if (r == 0x9E3779B9u) sink[blockIdx.x & 1023] = r;  // practically never true: keeps the loads alive without a store stream
}

namespace {

// Launch shape of the decode matvec. units = cols / UNIT columns-slices per row; a wave covers 64 * iters of them.
// per_cu: persistent workgroups per CU (own_per_cu: not imposed by MSQ_MV_WGS), stage_w: weight rows through LDS (mv_tok_kernel), free_shape:
// no part of the shape was imposed by the caller
struct MvShape { int iters, ks, rw, rpw, unit; int per_cu = 1; bool stage_w = false, free_shape = false, own_per_cu = true; };

int mv_unit(int t) { return msq_type_block_elems(t) == 1 ? 8 : 32; }

bool mv_shape(int t, int rows, int cols, int groups, const MsqMvCfg* cfg, MvShape* s) {
  const int unit = mv_unit(t);
  const int units = cols / unit;
  int iters = 1;
  while (iters < 4 && units > 64 * 16 * iters) iters *= 2;
  int ks = (units + 64 * iters - 1) / (64 * iters);
  if (cfg && cfg->ks > 0) {  // a wider K split than needed only adds idle waves; a narrower one needs more iters
    ks = cfg->ks;
    while (iters < 4 && units > 64 * ks * iters) iters *= 2;
  }
  if (ks > 16 || units > 64 * ks * iters) return false;
  // the codebook formats stage a table of up to 32 KB per workgroup: one 16-wave workgroup per CU, each wave a run of
  // rows long enough for its register ring; the others run several small workgroups per CU
  const bool table = t == MSQ_IQ1_S || t == MSQ_IQ2_XXS;
  int rw = std::max(1, (table ? 16 : 8) / ks);
  if (cfg && cfg->rsg > 0) rw = cfg->rsg;
  if (rw * ks > 16) rw = std::max(1, 16 / ks);
  const int rpg = rows / groups;
  int rpw;
  if (table) {  // about one tile per CU
    const long per_cu = ((long)rows + device_info().cus - 1) / device_info().cus;
    rpw = (int)std::min<long>(64, std::max<long>(1, (per_cu + rw - 1) / rw));
  } else {  // rows per wave per tile: enough tiles to fill the chip a few times over, at most 8 rows per wave
    rpw = 8;
    while (rpw > 1 && (long)rows / (rw * rpw) < 2048) rpw /= 2;
  }
  if (cfg && cfg->nr > 0) rpw = std::min(cfg->nr, 64);
  if (groups > 1) {  // every tile must stay inside one block-diagonal group
    while (rpw > 1 && rpg % (rw * rpw)) rpw /= 2;
    while (rw > 1 && rpg % (rw * rpw)) rw /= 2;
    if (rpg % (rw * rpw)) return false;
  }
  *s = {iters, ks, rw, rpw, unit};
  return true;
}

// static LDS of the matvec kernels of decoder D: the codebook table (an array of at least four words)
template <class D>
constexpr size_t kStaticLds = (D::LDS_WORDS > 0 ? D::LDS_WORDS : 4) * 4 + 64;

// LDS layout behind the partial sums: the four partial sums of a fused norm, then the padded activation
// rows the workgroup stages, `tokens` of them, when all of it fits under `limit` bytes (else the activations are read
// straight from device memory; refused with a fused norm or when the kernel has no such path).
bool place_x_row(MvArgs& a, size_t& lds, int tokens = 1, size_t limit = 64 * 1024, bool required = false) {
  size_t at = (lds + 15) / 16 * 16;
  if (a.norm_w) { a.norm_off = (uint32_t)(at / 4); at += 16; }
  a.xs_off = (uint32_t)(at / 4);
  const size_t end = at + (size_t)xlds_words(a.cols) * 4 * tokens;
  a.stage_x = end <= limit ? 1u : 0u;
  if (a.stage_x) lds = end;
  return a.stage_x || !(a.norm_w || required);
}

// Which prologue of a fused norm (msq_mv.cuh) a launch takes. One trip to memory needs more registers and code and makes the
// norm's weights wait behind the first weight rows: two trips are ahead where a row is short, one trip where it is long or
// the matrix large. Measured with an input row of its own for every launch, as layers have (a row that stays in the caches
// makes two trips look better by 5 to 10 %); in brackets two trips' time over one trip's.
//  * mv_tok_kernel, block formats: from 4608 columns on (Q5_K 4096x4096 0.96, x4608 1.04, IQ4_NL 1100x5120 1.09), and 40 MB and
//    more of more than 2048 columns (Q6_K 16384x3072 1.04; IQ4_NL 32768x2048 0.98); Q8_0, whose activations stay fp32, from 3072
//    (2048x2560 0.98, x3072 1.00, 4096x4096 1.03), from 16 MB of more than 2048 (8192x2304 1.05) and from 30 MB (16384x2048 1.04,
//    8192x2048 0.98); F32 always (0.98 to 1.3); fp16 types up to 1024 columns (2048x1024 1.06), beyond 2048 (1100x2560 1.06, 4096x2304
//    0.98, x3072 1.05) and from 32 MB (8192x2048 1.02, 1100x2048 0.96).
//  * mv_kernel, sums from registers, lowest, median and highest of 8000 random matrices: block formats from 2304 columns on, Q8_0 from
//    2560 (up to 4096 0.99, 1.05, 1.2, beyond 0.99, 1.3, 1.45; 2048 columns 0.92, 0.97, 1.0); dense types from 2304 on where they are
//    alone on a CU (1.07, 1.24, 1.35), else, since the registers cut the overlap of workgroups, up to 4096 (0.99, 1.03, 1.18; beyond
//    0.88, 1.00, 1.04).
//  * mv_kernel, sums from LDS: dense types of more than 4096 columns with more than one workgroup per CU (two trips 0.79 to 0.92 of its
//    speed at 4352 to 10240), but rows over more than twelve waves: of 80 registers a CU holds 24 waves, so these would run one by one
//    (F32 512x7168 0.87); F32 of less than 3072 columns (sums from registers 0.96 to 1.03 of its speed at 2304, 0.93 to 1.05 at 1280).
template <class D>
Norm norm_of_tok(uint32_t cols, double bytes) {
  if constexpr (D::UNIT == 8) return std::is_same_v<D, DecDense<MSQ_F32>> || cols > 2048 || cols <= 1024 || bytes >= 32e6 ? kNormOneTrip : kNormTwoTrips;
  else if constexpr (std::is_same_v<D, DecQ8_0>) return cols >= 3072 || bytes >= (cols > 2048 ? 16e6 : 30e6) ? kNormOneTrip : kNormTwoTrips;
  else return cols >= 4608 || (cols > 2048 && bytes >= 40e6) ? kNormOneTrip : kNormTwoTrips;
}
template <class D>
Norm norm_of_mv(uint32_t cols, int grid, int threads) {
  if constexpr (D::UNIT == 8) {
    constexpr bool f32 = std::is_same_v<D, DecDense<MSQ_F32>>;
    const bool crowded = grid > device_info().cus;
    if (cols >= (f32 ? 3072 : 2304)) return !crowded || cols <= 4096 ? kNormOneTripRegs : threads <= 768 ? kNormOneTrip : kNormTwoTrips;
    return f32 ? kNormOneTrip : kNormTwoTrips;
  } else {
    return cols >= (std::is_same_v<D, DecQ8_0> ? 2560u : 2304u) ? kNormOneTripRegs : kNormTwoTrips;
  }
}

template <class D>
int launch_mv(hipStream_t st, const MvShape& s, MvArgs& a) {
  const int threads = 64 * s.rw * s.ks;
  const int tile_rows = s.rw * s.rpw;
  a.units = a.cols / D::UNIT;
  a.ks = s.ks;
  a.rpw = s.rpw;
  a.ntiles = (a.rows + tile_rows - 1) / tile_rows;
  size_t lds = (size_t)tile_rows * s.ks * 4;  // dynamic LDS: partial sums, staged activations (the table is static)
  if ((D::STAGE_X || a.norm_w) && !place_x_row(a, lds, 1, 64 * 1024 - kStaticLds<D>)) return MSQ_ERR_UNSUPPORTED;
  // persistent workgroups: as many as can be resident, never more than there are tiles
  const int wg_per_cu = std::max(1, std::min(2048 / threads, (int)((size_t)kMaxLds / (lds + kStaticLds<D>))));
  const int grid = (int)std::min<long>(a.ntiles, (long)device_info().cus * wg_per_cu);
  if (a.norm_w) {
    if constexpr (requires { D::STAGES; }) return MSQ_ERR_UNSUPPORTED;  // codebook formats: as in the reference (quant.mm:110)
    else {
      auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), lds, st, a); };
      const Norm norm = norm_of_mv<D>(a.cols, grid, threads);
      auto by_norm = [&]<int ITERS>() {
        if (norm == kNormTwoTrips) return launch(mv_kernel<D, ITERS, kNormTwoTrips>);
        if constexpr (D::UNIT == 8) { if (norm == kNormOneTrip) return launch(mv_kernel<D, ITERS, kNormOneTrip>); }
        launch(mv_kernel<D, ITERS, kNormOneTripRegs>);
      };
      switch (s.iters) {
        case 1: by_norm.template operator()<1>(); break;
        case 2: by_norm.template operator()<2>(); break;
        default: by_norm.template operator()<4>(); break;
      }
      MSQ_HIP(hipGetLastError());
      return MSQ_OK;
    }
  }
  if constexpr (requires { D::STAGES; }) {  // codebook formats: ring kernel (one unit per lane, matrix below 4 GiB)
    if (s.iters == 1 && (uint64_t)a.rows * a.row_bytes < (1ull << 32)) {
      hipLaunchKernelGGL((mv_ring_kernel<D>), dim3(grid), dim3(threads), lds, st, a);
      MSQ_HIP(hipGetLastError());
      return MSQ_OK;
    }
  }
  switch (s.iters) {
    case 1: hipLaunchKernelGGL((mv_kernel<D, 1>), dim3(grid), dim3(threads), lds, st, a); break;
    case 2: hipLaunchKernelGGL((mv_kernel<D, 2>), dim3(grid), dim3(threads), lds, st, a); break;
    default: hipLaunchKernelGGL((mv_kernel<D, 4>), dim3(grid), dim3(threads), lds, st, a); break;
  }
  MSQ_HIP(hipGetLastError());
  return MSQ_OK;
}

int env_knob_early(const char* name, int dflt) {
  const char* v = getenv(name);
  return v && *v ? atoi(v) : dflt;
}
// Launch shape of the small-N matvec: workgroups of at most 8 waves (the kernel keeps T activation slices per lane
// and is built for 512 threads), one or two units per lane.
bool mv_tok_shape(int t, int rows, int cols, int groups, int n, int token_groups, const MsqMvCfg* cfg, MvShape* s) {
  const int unit = mv_unit(t);
  const int units = cols / unit;
  int iters = 1;
  while (iters < 2 && units > 64 * 8 * iters) iters *= 2;
  int ks = (units + 64 * iters - 1) / (64 * iters);
  if (cfg && cfg->ks > 0) {
    ks = cfg->ks;
    iters = units > 64 * ks ? 2 : 1;
  }
  if (ks > 8 || units > 64 * ks * iters) return false;
  int rw = std::max(1, 8 / ks);
  if (cfg && cfg->rsg > 0) rw = cfg->rsg;
  if (rw * ks > 8) return false;
  // rows per wave per tile: one workgroup per CU, one tile each, is what measures fastest (a wave prefetches along its
  // run of rows; every tile ends in a workgroup-wide reduction)
  // One token, a matrix without a codebook table that is large (48 MB: the launch is bound by the bytes a CU keeps in
  // flight, and a wave still walks a long run of rows) or dense and at least 8 MB (nothing to decode): two workgroups
  // per CU. Measured, one / two workgroups: Q6_K 129280x5120 165 / 132 us, Q6_K 25600x6144 43.6 / 29.9, F16 5120x5120
  // 13.7 / 11.2, BF16 4096x1280 6.75 / 5.2; the block formats between 5 and 35 MB lose up to 1.5 us with two.
  const bool table = t == MSQ_IQ1_S || t == MSQ_IQ2_XXS;
  static const int env_wgs = env_knob_early("MSQ_MV_WGS", 0);  // imposes the number for every call of one token
  const bool free_shape = !(cfg && (cfg->nr > 0 || cfg->rsg > 0 || cfg->ks > 0));
  const double bytes = (double)msq_type_row_bytes(t, cols) * rows;
  const bool two = !table && (bytes >= 48e6 || (unit == 8 && bytes >= 8e6));
  const int per_cu = (n == 1 && free_shape) ? (env_wgs > 0 ? env_wgs : two ? 2 : 1) : 1;
  const long wgs = std::max(1, per_cu * device_info().cus / token_groups);
  int rpw = (int)std::min<long>(32, std::max<long>(1, (rows + wgs * rw - 1) / (wgs * rw)));
  if (cfg && cfg->nr > 0) rpw = std::min(cfg->nr, 64);
  const int rpg = rows / groups;
  if (groups > 1) {  // every tile must stay inside one block-diagonal group
    while (rpw > 1 && rpg % (rw * rpw)) rpw--;
    while (rw > 1 && rpg % (rw * rpw)) rw /= 2;
    if (rpg % (rw * rpw)) return false;
  }
  // Weight rows through LDS (mv_tok_kernel) where it measures faster: Q6_K (five loads per lane and row otherwise) from
  // 12 MB, Q8_0 (three) from 40 MB -- ring / through LDS: Q6_K 8192x5120 12.3 / 12.0 us, 65536x5120 71.9 / 57.0, Q8_0
  // 8192x5120 12.9 / 12.2, 65536x5120 82.4 / 67.5. Q5_K and IQ4_NL, whose 16-byte reads from LDS cost five words and four
  // shifts each, lose 10 to 17 %; the codebook formats are bound by their table lookups. MSQ_MV_STAGEW = 0 / 1 imposes
  // the choice.
  static const int env_sw = env_knob_early("MSQ_MV_STAGEW", -1);
  const bool stage_w = n == 1 && free_shape &&
                       (env_sw >= 0 ? env_sw > 0 : (t == MSQ_Q6_K && bytes >= 12e6) || (t == MSQ_Q8_0 && bytes >= 40e6));
  *s = {iters, ks, rw, rpw, unit, per_cu, stage_w, free_shape, env_wgs <= 0};
  return true;
}

// n = 1: the prefetching kernel pays from two full rows per wave and CU on (below that mv_kernel does the same with
// less ceremony). Large codebook matrices are bound by decode arithmetic and do better in the 16-wave ring kernel
// (measured: IQ1_S 4096x7168 7.5 against 8.6 us, 8192 rows 9.9 against 10.1 us, 16384 rows 20.3 against 14.7 us).
// An imposed shape with nr >= 2 and at most 8 waves names the prefetching kernel outright.
bool tok_serves_single(int t, int rows, int cols, const MvShape& s, const MsqMvCfg* cfg) {
  if (cfg && cfg->nr > 0) return s.rpw >= 2;
  const bool table = t == MSQ_IQ1_S || t == MSQ_IQ2_XXS;
  if (table && (double)msq_type_row_bytes(t, cols) * rows > 10e6) return false;
  return s.rpw >= 2 && (long)rows >= 2L * device_info().cus * s.rw;
}

// Rows whose units do not fill whole waves: two, four or eight rows are launched as one (mv_tok_kernel, PACK), as few as leave
// the fewest waves per row. One group, a number of rows that divides, a row's units a multiple of 8 (several tokens: two rows, 16).
// Measured with weights beyond the caches, rows one by one / packed: Q6_K 32768 rows of 256 columns 10.8 / 5.4 us, 512 10.3 / 6.2 (in pairs
// 7.6), 768 10.4 / 7.5, 1280 11.9 / 10.6, 1536 12.0 / 11.5, 129280x5120 108.3 / 99.1, 1536x7168 6.27 / 5.94; Q8_0 32768x512 9.1 / 7.2,
// 2304x5120 6.37 / 6.29; against pairs at most over 19000 random matrices of the K-quants, Q8_0, BF16 and F32 0.96 to 2.1, below 0.975 in
// one of a thousand (under a norm Q6_K 2304x11000 and 2816x7500, Q5_K 1536x15000, and Q6_K pairs of 512 columns from the caches). More than two
// rows for an eighth fewer waves or less gain nothing (3328 columns 0.96 to 1.06), nor do five waves a workgroup where there are
// not four packed rows for each (2304x2304 0.95), nor rows of 2304 columns below 6 MB (0.94 to 0.97), nor four short rows of Q8_0 where
// they make the waves' runs two long and pairs would make them three (512 columns, 8193 to 12288 rows 0.95 to 0.97, on either side 1.01 to
// 1.03); the codebook formats, bound by their lookups, lose 1 % and keep the one-row form. MSQ_MV_PAIR = 0 / 2: never / every format.
// Under a fused norm likewise, but for Q8_0 below 20 MB (2560, 4608, 5120 and 7168 columns, one by one over in pairs: 6 to 18 MB
// 0.97 to 1.02 and once 1.07, 22 to 45 MB 1.00 to 1.04) and Q5_K rows of 2304 and 2816 columns below 12 MB (0.95 to 0.98). A row's bits are
// the same packed or not, so the rule is free to differ.
//
// Five waves a workgroup leave the SIMDs unequal work: K-quants take two of them per CU from 16 MB on (2560 and 5120 columns, one / two:
// 12 MB 0.95 to 1.03, 16 MB 1.02 to 1.06, 26 MB 1.10 to 1.17, 44 MB 1.17 to 1.24), under a norm of two trips from 26 MB on (1.03 to
// 1.12; Q6_K 20 MB 0.93); Q8_0 does not (0.69 to 0.92 up to 34 MB). Unless MSQ_MV_WGS names a number.
template <class D, int T>
int packed_rows(const MvArgs& a, MvShape& s) {
  static const int env_pair = env_knob_early("MSQ_MV_PAIR", -1);
  const double bytes = (double)a.rows * a.row_bytes;
  const int u = (int)(a.cols / D::UNIT), cus = device_info().cus;
  constexpr bool q8 = std::is_same_v<D, DecQ8_0>, kq = std::is_same_v<D, DecQ6KQ> || std::is_same_v<D, DecQ5KQ>;
  auto waves = [&](int p) { return (p * u + 63) / 64; };
  const double bytes8 = q8 ? 20e6 : u < 64 ? 0. : a.norm_w && std::is_same_v<D, DecQ5KQ> ? 12e6 : 6e6;  // sums of eight lanes from here on
  int pack = 1;
  if (s.iters == 1 && s.free_shape && (D::LDS_WORDS == 0 || env_pair == 2) && env_pair != 0 && a.rows_per_group >= a.rows &&
      !(a.norm_w && q8 && bytes < 20e6) && u % (T == 1 && D::LDS_WORDS == 0 ? 8 : 16) == 0)
    for (int p = 2; p <= (T == 1 ? 8 : 2); p *= 2) {
      if (q8 && p == 4 && waves(4) == 1 && (long)a.rows > 32L * cus && (long)a.rows <= 48L * cus) break;  // (eight waves a workgroup, one a CU)
      if (a.rows % p == 0 && waves(p) <= 8 && (u % 16 == 0 || bytes >= bytes8) && waves(p) * pack < waves(pack) * p &&
          (p == 2 || (8 * waves(p) < 7 * p * waves(1) && (waves(p) != 5 || (long)a.rows >= 4L * p * cus))))
        pack = p;
    }
  if (kq && s.own_per_cu && pack > 1 && waves(pack) == 5 && bytes >= (a.norm_w ? 26e6 : 16e6) &&
      !(a.norm_w && norm_of_tok<D>(a.cols, bytes) == kNormOneTrip))
    s.per_cu = 2;
  return pack;
}

template <class D, int T>
int launch_mv_tok(hipStream_t st, const MvShape& s_, const MvTokArgs& ta_) {
  MvTokArgs ta = ta_;  // (the launch may reshape rows into pairs: the caller's arguments stay as they are)
  MvArgs& a = ta.m;
  MvShape s = s_;
  const double bytes = (double)a.rows * a.row_bytes;
  const int pack = packed_rows<D, T>(a, s), u = (int)(a.cols / D::UNIT);
  if (pack > 1) {
    a.rows /= pack;
    a.rows_per_group = a.rows;
    a.row_bytes *= pack;
    s.ks = (pack * u + 63) / 64;
    s.rw = std::max(1, 8 / s.ks);
    const long wgs = std::max<long>(1, s.per_cu * device_info().cus / (((long)ta.n + T - 1) / T));
    s.rpw = (int)std::min<long>(32, std::max<long>(1, (a.rows + wgs * s.rw - 1) / (wgs * s.rw)));
  }
  const bool sums8 = pack > 1 && u % 16;
  const int threads = 64 * s.rw * s.ks;
  const int tile_rows = s.rw * s.rpw;
  a.units = pack * (a.cols / D::UNIT);
  a.ks = s.ks;
  a.rpw = s.rpw;
  a.ntiles = (a.rows + tile_rows - 1) / tile_rows;
  size_t lds = (size_t)tile_rows * s.ks * (sums8 ? 8 : 4) * T * 4;  // dynamic LDS: partial sums, staged activations (the table is static)
  const int gy = ((int)ta.n + T - 1) / T;
  if (tok_stages_x<D, T>() || a.norm_w) {
    // one workgroup per CU: all of its LDS (decoders that stage only in the four-token kernel read directly when a round does not fit)
    if (!place_x_row(a, lds, tok_round<D, T>(), kMaxLds - kStaticLds<D>, D::STAGE_X)) return MSQ_ERR_UNSUPPORTED;
  }
  // Weight rows through LDS: where the waves' buffers, four slots each, find room behind the staged activations (Q8_0 rows of more
  // than 14336 columns, eight waves of three pieces a slot, leave none), ...
  const size_t w_at = (lds + 15) / 16 * 16, w_end = w_at + (size_t)(threads / 64) * 4 * wspan_loads<D>() * 1024;
  const int w_per_cu = (w_end + kStaticLds<D>) * s.per_cu <= (size_t)kMaxLds ? s.per_cu : 1;
  // ... and under a fused norm, for Q6_K, where a CU then holds six waves and more and the matrix has 17 MB, or 26 where the rows
  // take the norm in one trip. Time without / with them, matrices and rows rotated beyond the caches:
  //   2048 to 4352 columns (six to eight waves) 17.5 MB 1.00 to 1.06, 26 MB 1.03 to 1.08;
  //   5632, 6144, 7168, 8192, 12288 columns (six to eight waves) 17.5 MB 0.98 to 1.00, 23 MB 0.99 to 1.00, 26 MB 1.01, 47 MB 1.02 to 1.05;
  //   4608, 5120, 9216, 10240 columns (five waves) 17.5 MB 0.95 to 0.97, 30 MB 0.98 to 1.00, 47 MB 1.00 to 1.01; the first two with a
  //   second workgroup (from 48 MB) 1.15 to 1.19, the other two, which have no room for it, 0.97 to 0.99;
  //   2048, 4096, 6144, 8192 columns 210 MB 1.12 to 1.21 (one such matrix alone, which stays in the 256 MB cache, 0.91 to 1.00).
  const bool norm_sw = std::is_same_v<D, DecQ8_0> || (threads / 64 * w_per_cu >= 6 && bytes >= (a.cols < 4608 ? 17e6 : 26e6));
  const bool sw = tok_stages_w<D, 1, T>() && s.iters == 1 && s.stage_w && (!a.norm_w || norm_sw) && w_end + kStaticLds<D> <= (size_t)kMaxLds;
  if (sw) {
    a.w_off = (uint32_t)(w_at / 4);
    lds = w_end;
  }
  auto launch = [&](auto kernel, dim3 grid) {
    allow_large_lds(kernel, lds);
    hipLaunchKernelGGL(kernel, grid, dim3(threads), lds, st, a.W, a.rows, a.row_bytes, a.units, a.ks, a.rpw, a.ntiles, a.rows_per_group, a.x, a.cols, (uint32_t)threads, ta);
  };
  // persistent workgroups, one per CU over all token groups (two for a large matrix: MvShape::per_cu)
  // A fused norm's prologue of one trip leaves Q5_K, Q6_K rows in registers (144) and two units of F32 no room for a second one:
  // they would run one by one (Q5_K 16384x7168 0.89 of the speed, F32 768x5120 0.79; IQ4_NL, Q8_0 and the fp16 types gain 3 to 25 %).
  const bool one_trip = a.norm_w && norm_of_tok<D>(a.cols, bytes) == kNormOneTrip;
  constexpr bool wide = std::is_same_v<D, DecQ5KQ> || std::is_same_v<D, DecQ6KQ>;
  const bool alone = one_trip && ((wide && !sw) || (std::is_same_v<D, DecDense<MSQ_F32>> && s.iters > 1));
  const int per_cu = (T == 1 && !alone && (lds + kStaticLds<D>) * s.per_cu <= (size_t)kMaxLds) ? s.per_cu : 1;
  const int gx = (int)std::min<long>(a.ntiles, std::max(1, per_cu * device_info().cus / gy));
  const dim3 grid((unsigned)gx, (unsigned)gy);
  if (a.norm_w) {  // fused input norm (single token)
    if constexpr (T != 1 || requires { D::STAGES; }) return MSQ_ERR_UNSUPPORTED;
    else {
      auto by_norm = [&]<int ITERS, bool SW, int PACK>() {
        one_trip ? launch(mv_tok_kernel<D, ITERS, 1, kNormOneTrip, SW, PACK>, grid) : launch(mv_tok_kernel<D, ITERS, 1, kNormTwoTrips, SW, PACK>, grid);
      };
      auto by_pack = [&]<int ITERS, bool SW>() {
        pack == 1 ? by_norm.template operator()<ITERS, SW, 0>() : sums8 ? by_norm.template operator()<ITERS, SW, 8>() : by_norm.template operator()<ITERS, SW, 16>();
      };
      if (sw) {
        if constexpr (tok_stages_w<D, 1, 1>()) by_pack.template operator()<1, true>();
      } else if (s.iters == 1) {
        by_pack.template operator()<1, false>();
      } else if constexpr (D::UNIT == 8) by_norm.template operator()<2, false, 0>();
      else return MSQ_ERR_UNSUPPORTED;
      MSQ_HIP(hipGetLastError());
      return MSQ_OK;
    }
  }
  auto by_pack = [&]<bool SW>() {
    if (pack == 1) return launch(mv_tok_kernel<D, 1, T, kNormNone, SW>, grid);
    if constexpr (T == 1 && D::LDS_WORDS == 0) { if (sums8) return launch(mv_tok_kernel<D, 1, T, kNormNone, SW, 8>, grid); }
    launch(mv_tok_kernel<D, 1, T, kNormNone, SW, 16>, grid);
  };
  if (sw) {
    if constexpr (tok_stages_w<D, 1, T>()) by_pack.template operator()<true>();
  } else if (s.iters == 1) {
    by_pack.template operator()<false>();
  } else if constexpr (D::UNIT == 8) launch(mv_tok_kernel<D, 2, T>, grid);
  else return MSQ_ERR_UNSUPPORTED;  // two block-format units per lane and T activation slices do not fit the registers
  MSQ_HIP(hipGetLastError());
  return MSQ_OK;
}

template <int T>
int launch_mv_tok_t(hipStream_t st, int t, const MvShape& s, MvTokArgs& ta) {
  if constexpr (T == 1) {  // one token: the block formats' integer decoders (msq_mvq.cuh)
    switch (t) {
      case MSQ_IQ1_S: return launch_mv_tok<DecIQ1SM, 1>(st, s, ta);
      case MSQ_IQ2_XXS: return launch_mv_tok<DecIQ2XXSM, 1>(st, s, ta);
      case MSQ_IQ4_NL: return launch_mv_tok<DecIQ4NLQ, 1>(st, s, ta);
      case MSQ_Q6_K: return launch_mv_tok<DecQ6KQ, 1>(st, s, ta);
      case MSQ_Q5_K: return launch_mv_tok<DecQ5KQ, 1>(st, s, ta);
    }
  }
  switch (t) {
    case MSQ_IQ1_S: return launch_mv_tok<DecIQ1S, T>(st, s, ta);
    case MSQ_IQ2_XXS: return launch_mv_tok<DecIQ2XXS, T>(st, s, ta);
    case MSQ_IQ4_NL: return launch_mv_tok<DecIQ4NL, T>(st, s, ta);
    case MSQ_Q6_K: return launch_mv_tok<DecQ6K, T>(st, s, ta);
    case MSQ_Q5_K: return launch_mv_tok<DecQ5K, T>(st, s, ta);
    case MSQ_F32: return launch_mv_tok<DecDense<MSQ_F32>, T>(st, s, ta);
    case MSQ_F16: return launch_mv_tok<DecDense<MSQ_F16>, T>(st, s, ta);
    case MSQ_BF16: return launch_mv_tok<DecDense<MSQ_BF16>, T>(st, s, ta);
  }
  return MSQ_ERR_UNSUPPORTED;
}

// rows launched as one and workgroups per CU of a one-token call (0: not through mv_tok_kernel)
template <class D>
int tok_launch_of(int t, int rows, int cols, bool norm, int* per_cu) {
  MvShape s;
  if (!mv_tok_shape(t, rows, cols, 1, 1, 1, nullptr, &s) || !tok_serves_single(t, rows, cols, s, nullptr)) return 0;
  const float w = 0.f;
  MvArgs a{};
  a.rows = a.rows_per_group = (uint32_t)rows; a.cols = (uint32_t)cols; a.row_bytes = (uint32_t)msq_type_row_bytes(t, cols);
  a.norm_w = norm ? &w : nullptr;
  const int pack = packed_rows<D, 1>(a, s);
  *per_cu = s.per_cu;
  return pack;
}

bool mv_type_ok(int t) {
  switch (t) {
    case MSQ_F32: case MSQ_F16: case MSQ_BF16: case MSQ_Q8_0: case MSQ_Q5_K: case MSQ_Q6_K: case MSQ_IQ1_S:
    case MSQ_IQ2_XXS: case MSQ_IQ4_NL: return true;
    default: return false;
  }
}
// Launch-shape overrides from the environment, on top of the caller's MsqMvCfg (reference: MACSEEK_MV_NR / _RSG / _KS,
// quant.mm:78-83, and MACSEEK_MVN_NR / _SG for the small-N form, quant.mm:141): MSQ_MV_NR / MSQ_MV_RSG / MSQ_MV_KS for
// one token, MSQ_MVN_NR / MSQ_MVN_RSG / MSQ_MVN_KS for several. Returns null when nothing is imposed.
int env_knob(const char* name) {
  const char* v = getenv(name);
  return v && *v ? atoi(v) : 0;
}
const MsqMvCfg* effective_cfg(const MsqMvCfg* cfg, bool several, MsqMvCfg* store) {
  static const int e1[3] = {env_knob("MSQ_MV_NR"), env_knob("MSQ_MV_RSG"), env_knob("MSQ_MV_KS")};
  static const int en[3] = {env_knob("MSQ_MVN_NR"), env_knob("MSQ_MVN_RSG"), env_knob("MSQ_MVN_KS")};
  const int* e = several ? en : e1;
  *store = cfg ? *cfg : MsqMvCfg{0, 0, 0};
  if (e[0] > 0) store->nr = e[0];
  if (e[1] > 0) store->rsg = e[1];
  if (e[2] > 0) store->ks = e[2];
  return (store->nr > 0 || store->rsg > 0 || store->ks > 0) ? store : nullptr;
}
// column granularity the kernels need: dense types use a virtual 256 block like the reference (quant.mm:31-32)
int mv_col_multiple(int t) { return msq_type_block_elems(t) == 1 ? 256 : msq_type_block_elems(t); }

}  // namespace
}  // namespace msq

namespace msq {

// Small-N matvec through the dot-product kernels. Returns MSQ_ERR_UNSUPPORTED without an error message when the shape
// does not fit them (the caller then takes another path). Arguments are already validated.
int matvec_tok(hipStream_t st, int t, const uint8_t* W, int rows, int cols, const float* X, float* Y, int n, int accumulate,
               int groups, const MsqMvCfg* cfg, const float* norm_w, float eps) {
  MsqMvCfg several;
  if (n > 1) cfg = effective_cfg(cfg, true, &several);
  // tokens per pass over the weights: one, two, four or eight (Q8_0 keeps fp32 activations, 32 registers per token: four at most)
  // ... and groups of four also for more tokens over a small matrix (below 8 MB): every workgroup then fetches four
  // tokens' activations instead of eight, and the second group finds the weights in the caches (Q5_K 512x7168 at 8 / 16
  // tokens: 10.4 / 11.1 -> 7.3 / 8.8 us; BF16 384x7168 6.1 / 6.7 -> 5.2 / 6.2; the 9 MB and 16 MB matrices lose at 16)
  static const int env_t = env_knob("MSQ_MVN_T");
  const bool small = (double)msq_type_row_bytes(t, cols) * rows < 8e6;
  const int T = n <= 2 ? n : (t == MSQ_Q8_0 || n <= 4 || env_t == 4 || (small && env_t != 8)) ? 4 : 8;
  MvShape s;
  if (!mv_tok_shape(t, rows, cols, groups, n, (n + T - 1) / T, cfg, &s)) return MSQ_ERR_UNSUPPORTED;
  if (n == 1 && !tok_serves_single(t, rows, cols, s, cfg)) return MSQ_ERR_UNSUPPORTED;
  MvTokArgs ta{};
  MvArgs& a = ta.m;
  a.W = W; a.x = X; a.y = Y;
  a.rows = (uint32_t)rows; a.cols = (uint32_t)cols; a.row_bytes = (uint32_t)msq_type_row_bytes(t, cols);
  a.rows_per_group = (uint32_t)(rows / groups); a.x_group_stride = (uint32_t)cols; a.accumulate = accumulate ? 1u : 0u;
  ta.n = (uint32_t)n; ta.x_stride = (uint32_t)((size_t)cols * groups); ta.y_stride = (uint32_t)rows;
  a.norm_w = norm_w; a.eps = eps;
  if (n == 1) return t == MSQ_Q8_0 ? launch_mv_tok<DecQ8_0, 1>(st, s, ta) : launch_mv_tok_t<1>(st, t, s, ta);
  if (t == MSQ_Q8_0) return T == 2 ? launch_mv_tok<DecQ8_0, 2>(st, s, ta) : launch_mv_tok<DecQ8_0, 4>(st, s, ta);
  return T == 2 ? launch_mv_tok_t<2>(st, t, s, ta) : T == 4 ? launch_mv_tok_t<4>(st, t, s, ta) : launch_mv_tok_t<8>(st, t, s, ta);
}

}  // namespace msq

using namespace msq;

extern "C" {

int msq_init(void) {
  g_err[0] = 0;
  const DeviceInfo& d = device_info();
  if (!d.ok) return fail(MSQ_ERR_HIP, "macseek quant: no gfx950 device is current");
  prefill_side_stream_setup();
  matmul_partials_setup();
  return static_scratch_setup(nullptr);
}
const char* msq_last_error(void) { return g_err; }
int msq_device_ok(void) { return device_info().ok; }

int msq_block_elems(int t) { return msq_type_block_elems(t); }
size_t msq_block_bytes(int t) { return msq_type_block_bytes(t); }
size_t msq_row_bytes(int t, int64_t cols) { return msq_type_row_bytes(t, cols); }
const char* msq_type_name(int t) { return msq_type_name_of(t); }

int msq_matvec_supported(int t) { return mv_type_ok(t) ? 1 : 0; }

int msq_matvec_cfg(int t, int rows, int cols, MsqMvCfg* out) {
  MvShape s;
  if (!out) return fail(MSQ_ERR_ARGUMENT, "macseek quant: matvec_cfg: null output");
  if (!mv_type_ok(t) || rows < 1 || cols < 1 || cols % mv_col_multiple(t)) return unsupported("matvec_cfg", t, rows, cols);
  MsqMvCfg env;
  const MsqMvCfg* cfg = effective_cfg(nullptr, false, &env);
  const bool tok = mv_tok_shape(t, rows, cols, 1, 1, 1, cfg, &s) && tok_serves_single(t, rows, cols, s, cfg);  // as msq_matvec decides
  if (!tok && !mv_shape(t, rows, cols, 1, cfg, &s)) return unsupported("matvec_cfg", t, rows, cols);
  out->nr = s.rpw; out->rsg = s.rw; out->ks = s.ks;
  return MSQ_OK;
}

// for tests: what tok_launch_of says of the types whose rows are packed
int msq_test_matvec_pack(int t, int rows, int cols, int norm, int* per_cu) {
  switch (t) {
    case MSQ_Q6_K: return tok_launch_of<DecQ6KQ>(t, rows, cols, norm != 0, per_cu);
    case MSQ_Q5_K: return tok_launch_of<DecQ5KQ>(t, rows, cols, norm != 0, per_cu);
    case MSQ_Q8_0: return tok_launch_of<DecQ8_0>(t, rows, cols, norm != 0, per_cu);
    case MSQ_BF16: return tok_launch_of<DecDense<MSQ_BF16>>(t, rows, cols, norm != 0, per_cu);
    default: return 0;
  }
}

// msq_matvec and msq_matvec_rmsnorm (norm_w != nullptr: the activations are normalized on the way in; the kernel is the
// one msq_matvec picks for the matrix, so the two agree bit for bit on a pre-normalized input)
static int matvec_impl(void* stream, const char* what, int t, const MsqBuffer* W, int rows, int cols, const MsqBuffer* x,
                       const MsqBuffer* y, int accumulate, int groups, const MsqMvCfg* cfg, const float* norm_w, float eps) {
  const size_t rb = msq_type_row_bytes(t, cols);
  if (!buf_ok(W, rb * (size_t)rows) || !buf_ok(x, (size_t)cols * groups * 4) || !buf_ok(y, (size_t)rows * 4))
    return fail(MSQ_ERR_ARGUMENT, "macseek quant: %s: buffer missing or too small (type %s rows %d cols %d)", what,
                msq_type_name_of(t), rows, cols);
  hipStream_t st = (hipStream_t)stream;
  MsqMvCfg imposed;
  cfg = effective_cfg(cfg, false, &imposed);
  {  // shapes with several rows per wave (chosen for matrices of more than a row per wave and CU, or imposed by cfg) go
     // through the prefetching kernel; a shape names its kernel, so row chunks launched with the shape of the whole
     // matrix repeat its bits
    const int rc = matvec_tok(st, t, bptr(W), rows, cols, (const float*)bptr(x), (float*)bptr_mut(y), 1, accumulate, groups, cfg,
                              norm_w, eps);
    if (rc != MSQ_ERR_UNSUPPORTED) return rc;
  }
  MvShape s;
  if (!mv_shape(t, rows, cols, groups, cfg, &s)) return unsupported("matvec launch shape", t, rows, cols);
  MvArgs a{};
  a.W = bptr(W); a.x = (const float*)bptr(x); a.y = (float*)bptr_mut(y);
  a.rows = (uint32_t)rows; a.cols = (uint32_t)cols; a.row_bytes = (uint32_t)rb;
  a.rows_per_group = (uint32_t)(rows / groups); a.x_group_stride = (uint32_t)cols; a.accumulate = accumulate ? 1u : 0u;
  a.norm_w = norm_w; a.eps = eps;
  int rc = MSQ_ERR_UNSUPPORTED;
  switch (t) {
    case MSQ_IQ1_S: rc = launch_mv<DecIQ1SM>(st, s, a); break;
    case MSQ_IQ2_XXS: rc = launch_mv<DecIQ2XXSM>(st, s, a); break;
    case MSQ_Q8_0: rc = launch_mv<DecQ8_0>(st, s, a); break;
    case MSQ_IQ4_NL: rc = launch_mv<DecIQ4NLQ>(st, s, a); break;
    case MSQ_Q6_K: rc = launch_mv<DecQ6KQ>(st, s, a); break;
    case MSQ_Q5_K: rc = launch_mv<DecQ5KQ>(st, s, a); break;
    case MSQ_F32: rc = launch_mv<DecDense<MSQ_F32>>(st, s, a); break;
    case MSQ_F16: rc = launch_mv<DecDense<MSQ_F16>>(st, s, a); break;
    case MSQ_BF16: rc = launch_mv<DecDense<MSQ_BF16>>(st, s, a); break;
  }
  return rc == MSQ_ERR_UNSUPPORTED ? unsupported(what, t, rows, cols) : rc;
}

int msq_matvec(void* stream, int t, const MsqBuffer* W, int rows, int cols, const MsqBuffer* x, const MsqBuffer* y,
               int accumulate, int groups, const MsqMvCfg* cfg) {
  if (!mv_type_ok(t) || rows < 1 || cols < 1 || cols % mv_col_multiple(t) || groups < 1 || rows % groups)
    return unsupported("matvec", t, rows, cols);
  return matvec_impl(stream, "matvec", t, W, rows, cols, x, y, accumulate, groups, cfg, nullptr, 0.f);
}

int msq_matvec_rmsnorm(void* stream, int t, const MsqBuffer* W, int rows, int cols, const MsqBuffer* x, const MsqBuffer* norm_w,
                       float eps, const MsqBuffer* y, int tiles_per_tg) {
  (void)tiles_per_tg;  // the reference's amortisation knob for the norm prologue; workgroups here are persistent
  if (!mv_type_ok(t) || t == MSQ_IQ1_S || t == MSQ_IQ2_XXS || rows < 1 || cols < 1 || cols % mv_col_multiple(t))
    return unsupported("matvec_rmsnorm", t, rows, cols);
  if (!buf_ok(norm_w, (size_t)cols * 4))
    return fail(MSQ_ERR_ARGUMENT, "macseek quant: matvec_rmsnorm: norm weights missing or too small (cols %d)", cols);
  return matvec_impl(stream, "matvec_rmsnorm", t, W, rows, cols, x, y, 0, 1, nullptr, (const float*)bptr(norm_w), eps);
}

int msq_rmsnorm(void* stream, const MsqBuffer* x, const MsqBuffer* w, const MsqBuffer* y, int rows, int dim, float eps,
                int in_stride, int out_stride) {
  if (rows < 0 || dim < 1 || (in_stride && in_stride < dim) || (out_stride && out_stride < dim))
    return unsupported("rmsnorm", MSQ_F32, rows, dim);
  if (rows == 0) return MSQ_OK;
  const int is = in_stride ? in_stride : dim, os = out_stride ? out_stride : dim;
  const bool has_w = w && w->dev;
  if (!buf_ok(x, ((size_t)(rows - 1) * is + dim) * 4) || !buf_ok(y, ((size_t)(rows - 1) * os + dim) * 4) ||
      (has_w && !buf_ok(w, (size_t)dim * 4)))
    return fail(MSQ_ERR_ARGUMENT, "macseek quant: rmsnorm: buffer missing or too small (rows %d dim %d)", rows, dim);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)rows), dim3(256), 0, (hipStream_t)stream, (const float*)bptr(x),
                       has_w ? (const float*)bptr(w) : nullptr, (float*)bptr_mut(y), (uint32_t)dim, eps, (uint32_t)is, (uint32_t)os);
  };
  switch ((dim + 1023) / 1024) {  // 1024 elements: four per thread
    case 1: launch(rmsnorm_kernel<4>); break;
    case 2: launch(rmsnorm_kernel<8>); break;
    case 3: launch(rmsnorm_kernel<12>); break;
    case 4: launch(rmsnorm_kernel<16>); break;
    case 5: launch(rmsnorm_kernel<20>); break;
    case 6: launch(rmsnorm_kernel<24>); break;
    case 7: launch(rmsnorm_kernel<28>); break;
    case 8: launch(rmsnorm_kernel<32>); break;
    default: launch(rmsnorm_kernel<0>);
  }
  MSQ_HIP(hipGetLastError());
  return MSQ_OK;
}

int msq_bw_probe(void* stream, const MsqBuffer* src, size_t bytes, const MsqBuffer* sink) {
  if (!buf_ok(src, bytes) || !buf_ok(sink, 4096) || bytes % 16 || ((uintptr_t)bptr(src) & 15))
    return fail(MSQ_ERR_ARGUMENT, "macseek quant: bw_probe: buffer missing, too small or misaligned");
  if (bytes == 0) return MSQ_OK;
  const size_t n16 = bytes / 16;
  const long grid = std::min<long>((long)((n16 + 1023) / 1024), (long)device_info().cus * 2);
  hipLaunchKernelGGL(bw_probe_kernel, dim3((unsigned)grid), dim3(1024), 0, (hipStream_t)stream, (const uint4*)bptr(src), n16,
                     (uint32_t*)bptr_mut(sink));
  MSQ_HIP(hipGetLastError());
  return MSQ_OK;
}

int msq_dequant(void* stream, int t, const MsqBuffer* W, int64_t n, const MsqBuffer* out) {
  const int be = msq_type_block_elems(t);
  if (!be || n < 0 || n % be || n % 8) return unsupported("dequant", t, 0, (int)n);
  if (n == 0) return MSQ_OK;
  if (!buf_ok(W, msq_type_row_bytes(t, n)) || !buf_ok(out, (size_t)n * 4))
    return fail(MSQ_ERR_ARGUMENT, "macseek quant: dequant: buffer missing or too small");
  const uint8_t* src = bptr(W);
  float* dst = (float*)bptr_mut(out);
  hipStream_t st = (hipStream_t)stream;
  switch (t) {
#define MSQ_DEQ(T) case T: launch_dequant<T>(st, src, dst, n); break;
    MSQ_DEQ(MSQ_F32) MSQ_DEQ(MSQ_F16) MSQ_DEQ(MSQ_BF16) MSQ_DEQ(MSQ_Q8_0) MSQ_DEQ(MSQ_IQ4_NL) MSQ_DEQ(MSQ_IQ1_S)
    MSQ_DEQ(MSQ_IQ2_XXS) MSQ_DEQ(MSQ_Q6_K) MSQ_DEQ(MSQ_Q5_K)
#undef MSQ_DEQ
    default: return unsupported("dequant", t, 0, (int)n);
  }
  MSQ_HIP(hipGetLastError());
  return MSQ_OK;
}

}  // extern "C"

// Few-token product over block formats: Y[t][r] (+)= W[r] . X[t] for 2 <= n <= 16 tokens (reference operator:
// ms::q::encode_matvec_n, src/kernels/quant.mm:129-156), exact payloads times fp16 activations, scales in fp32; and, ROUND,
// any number of tokens in blocks of sixteen with weights rounded to fp16 (ms::q::encode_matmul, quant.mm:193-248).
//
// The product is a stream of weights: one 16-token tile, so every weight byte is used by one matrix instruction. A
// persistent workgroup's waves split K: a wave owns BPW weight stages (256 columns each) of every row, holds the
// activations of its columns as fragments in registers for the whole launch, and walks the 16-row tiles of the workgroup.
// Its raw weight bytes come by loads that write LDS directly, as consecutive aligned 16-byte pieces of its rows, into a
// ring of its own, the next stages while one is being decoded; nothing else is fetched in the loop, so the waits are
// exact. The waves' partial tiles meet in LDS every UT tiles (two buffers, one barrier per meeting) and are added in wave
// order: no second launch, no buffer outside the call.
//
// Why this split: fetched lane by lane in fragment order a weight load touches sixteen rows and the vector cache, not
// memory, sets the pace; and activations fetched per row tile instead of once per launch are several times the weight
// bytes (16 tokens x 8192 columns in fp32: 512 KB). What bounds it now: a wave of Q6_K
// 32768x1280 at 16 tokens spends 19 % of its cycles issuing vector instructions (46 a fragment with the activations; 38 % of
// the launch's issue slots), waits on counters 43 % -- first trip to memory, activations, meeting, the fragments' latency
// chains -- and for its turn 28 %. Measured (MI355X, weights from HBM,
// before -> after, us): Q6_K 32768x1280 at 4 / 8 / 16 tokens 18.7 / 28.4 / 22.8 -> 12.6 / 13.0 / 14.8, 5120x8192 at 16
// 28.8 -> 20.8, IQ4_NL 16384x1536 at 16 22.5 -> 10.4, IQ1_S 7168x4096 at 4 / 16 9.9 / 20.7 -> 8.6 / 9.9.
#pragma once
#include <type_traits>

#include "msq_mfma.cuh"

namespace msq {

struct RowsArgs {
  const uint8_t* W;  // raw block rows, below 4 GiB in all
  const void* X;     // [n][x_stride]: fp32 on 16-byte boundaries, or fp16 on 8-byte ones
  float* Y;          // [n][rows]
  uint32_t n, rows, cols, x_stride, row_bytes, accumulate;
  uint32_t rows_per_group, x_group_stride;  // block-diagonal: rows per group (whole tiles), elements between the groups' inputs
  uint32_t nws;             // weight stages of a row
  uint32_t w_bytes;         // bytes from W to the matrix's end
  uint32_t tiles_per_wg;    // consecutive row tiles of a workgroup (of one group)
  uint32_t ntiles;
  const uint8_t* W1;        // GU: the up matrix (W: gate), of the same shape
  uint16_t* H;              // GU: output [n][rows]
};

constexpr int kRowsXPitch = 128 * 2 + 16;           // activations pass through LDS 128 columns at a time, fp16
constexpr int kRowsXBytes = 16 * kRowsXPitch;
template <class F> constexpr int rows_pieces() { return ((F::WS_BYTES + 14 + 15) / 16) | 1; }  // see mm_tile_kernel
template <class F> constexpr int rows_slot() { return 16 * rows_pieces<F>() * 16; }            // bytes of a stage of 16 rows
// slots requested ahead of the activations, which pass through the rest of the ring
template <class F> constexpr int rows_early(int S) { return rows_slot<F>() < 2048 ? 1 : S - 1; }
// words of the waves' partial tiles
__host__ __device__ constexpr uint32_t rows_red_words(uint32_t waves, int UT, int TT, bool gu = false) { return (TT == 1 && !gu ? 2u : TT) * waves * 256u * UT; }
template <class F> constexpr int rows_ring(int S) {
  const int x = rows_early<F>(S) * rows_slot<F>() + kRowsXBytes;
  return S * rows_slot<F>() > x ? S * rows_slot<F>() : x;
}

// Q6_K with the two 16-column scale groups of a step in different matrix instructions (K = 16 each): chunk q holds columns
// 4 q .. 4 q + 3 of either group
struct FragQ6KG {
  static constexpr int WS_BYTES = 210, LDS_WORDS = 0;
  static constexpr bool HAS_ADD = false, GROUPS = true;
  __device__ static void fill_lds(uint32_t*, int, int) {}
  struct Out { uint32_t h[4]; float sa, sb; };
  __device__ static Out get(const LdsRow& b, int js, uint32_t q, const uint32_t*) {
    const int h = js >> 2, k = js & 3;
    const uint32_t la = ld32(b + 64u * h + 32u * (k & 1) + 4u * q), lb = ld32(b + 64u * h + 32u * (k & 1) + 16u + 4u * q);
    const uint32_t ha = ld32(b + 128u + 32u * h + 4u * q), hb = ld32(b + 128u + 32u * h + 16u + 4u * q);
    const uint32_t sc = ld16(b + 192u + 8u * h + 2u * k);
    const float d = half_bits_to_float(ld16(b + 208u));
    const uint32_t qa = ((la >> (4 * (k >> 1))) & 0x0F0F0F0Fu) | (((ha >> (2 * k)) & 0x03030303u) << 4);
    const uint32_t qb = ((lb >> (4 * (k >> 1))) & 0x0F0F0F0Fu) | (((hb >> (2 * k)) & 0x03030303u) << 4);
    const uint32_t bias = 0xE420E420u;  // -1056 = -(1024 + 32) in both halves
    Out o;
    o.h[0] = pk_add_f16(bytes01_to_h2_1024(qa), bias); o.h[1] = pk_add_f16(bytes23_to_h2_1024(qa), bias);
    o.h[2] = pk_add_f16(bytes01_to_h2_1024(qb), bias); o.h[3] = pk_add_f16(bytes23_to_h2_1024(qb), bias);
    o.sa = d * (float)(int)(int8_t)(sc & 0xFFu);
    o.sb = d * (float)(int)(int8_t)(sc >> 8);
    return o;
  }
};

__device__ __forceinline__ f4_t mfma_f16_k16(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1, f4_t c) {
  typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
  typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
  const u2_t av = {a0, a1}, bv = {b0, b1};
  return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(h4_t, av), __builtin_bit_cast(h4_t, bv), c, 0, 0, 0);
}
__device__ __forceinline__ f4_t fma4(float s, f4_t p, f4_t c) {
  return f4_t{__builtin_fmaf(s, p[0], c[0]), __builtin_fmaf(s, p[1], c[1]), __builtin_fmaf(s, p[2], c[2]), __builtin_fmaf(s, p[3], c[3])};
}

// ROUND: the arithmetic of msq_matmul -- scale times payload rounded to fp16, summed in the matrix cores -- over any number
// of tokens, 16 TT per workgroup (blockIdx.y). XH: activations in memory are fp16. Decoding bounds the larger of these products
// (about 37 vector instructions a fragment, which one matrix instruction uses), hence TT = 2: 8192x4096 at 64 tokens against
// the routes of msq_matmul that slice K over workgroups: IQ4_NL 38.2 -> 22.0 us, Q6_K 30.8 -> 22.5, IQ2_XXS 38.1 -> 21.3; 1536x4096 of
// IQ1_S at 200 32.1 -> 17.2. Three tiles' activations do not fit the registers of four waves a SIMD.
// GU (the prefill MoE layer's shared expert, few tokens): row tiles 2 k and 2 k + 1 are tile k of the gate and of the up matrix, which
// meet together and leave silu(min(gate, 10)) * clamp(up, -10, 10) in fp16.
template <class F, int BPW, int S, int NT, int UT, bool ROUND = false, bool XH = false, int TT = 1, bool GU = false>
__global__ __launch_bounds__(1024) void mm_rows_kernel(const RowsArgs a) {
  constexpr int P = rows_pieces<F>(), PIECES = 16 * P, NPI = (PIECES + 63) / 64, SLOT = rows_slot<F>();
  constexpr bool GROUPS = requires { F::GROUPS; };
  constexpr bool PAIR = requires { F::pos_of(0u); };
  extern __shared__ __attribute__((aligned(16))) uint32_t smem[];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, nthreads = blockDim.x, nwaves = nthreads >> 6;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t n16 = lane & 15u, q = lane >> 4;
  uint32_t* tbl = smem;
  float* red = (float*)(smem + F::LDS_WORDS);                    // [2][wave][tile][token][16]
  static_assert(!GU || (UT == 2 && TT == 1));
  uint8_t* mine = (uint8_t*)(red + rows_red_words(nwaves, UT, TT, GU)) + wave * (uint32_t)rows_ring<F>(S);

  constexpr bool BLOCKS = ROUND || XH;  // any number of tokens
  const uint32_t m0 = BLOCKS ? blockIdx.y * (16u * TT) : 0u, ntok = BLOCKS ? min(a.n - m0, 16u * TT) : a.n;
  const uint32_t tile0 = blockIdx.x * a.tiles_per_wg, ntile = min(a.tiles_per_wg, a.ntiles - tile0);  // (grid: tile0 < ntiles)
  const uint32_t group = (tile0 * 16u) / a.rows_per_group;
  const uint32_t ws0 = wave * BPW;

  struct Matrix { rsrc_t rs; uint32_t mis, bytes, end; };
  auto matrix = [&](const uint8_t* w) {
    const uintptr_t wa = (uintptr_t)w;
    const uint32_t mis = (uint32_t)wa & 15u, bytes = (mis + a.w_bytes + 15u) & ~15u;  // whole aligned pieces: no piece straddles the end
    return Matrix{make_rsrc((const void*)(wa - mis), bytes), mis, bytes, mis + a.w_bytes};
  };
  const Matrix w0 = matrix(a.W), w1 = GU ? matrix(a.W1) : w0;
  auto of_tile = [&](uint32_t tile) -> const Matrix& { return GU && (tile & 1u) ? w1 : w0; };
  auto row_tile = [&](uint32_t tile) { return GU ? tile >> 1 : tile; };
  // stage i of the wave's walk: tile i / BPW, weight stage ws0 + i % BPW
  uint32_t rowoff[NPI], pc[NPI];  // per piece: row inside the tile (in bytes), 16-byte piece of the row
#pragma unroll
  for (int k = 0; k < NPI; k++) {
    const uint32_t p = (uint32_t)k * 64u + lane;
    rowoff[k] = (p / P) * a.row_bytes; pc[k] = 16u * (p % P);
  }
  auto request = [&](uint32_t tile, int b, uint32_t slot) {
    const Matrix& w = of_tile(tile);
    const uint32_t at = w.mis + (row_tile(tile) * 16u) * a.row_bytes + min(ws0 + b, a.nws - 1u) * (uint32_t)F::WS_BYTES;  // (a stage past the row's end: bytes nobody reads)
#pragma unroll
    for (int k = 0; k < NPI; k++) {
      const uint32_t v = at + rowoff[k];
      if (PIECES % 64 == 0 || k + 1 < NPI || (uint32_t)k * 64u + lane < (uint32_t)PIECES)
        lds_dma16(w.rs, mine + slot * SLOT + k * 1024, v < w.end ? (v & ~15u) + pc[k] : w.bytes, 0u);  // rows past the end: no traffic
    }
  };

  const uint32_t total = ntile * BPW;
#pragma unroll
  for (int i = 0; i < rows_early<F>(S); i++)
    if ((uint32_t)i < total) request(tile0 + i / BPW, i % BPW, (uint32_t)i);
  F::fill_lds(tbl, (int)tid, (int)nthreads);
  // ---- activations of the wave's columns, through LDS: rows are read along the columns (lane by lane in fragment order
  // every load would touch sixteen rows), rounded to fp16, and read back as fragments
  uint32_t xr[TT][BPW * 8][4];
  {
    uint8_t* xs = mine + rows_early<F>(S) * SLOT;
    using XT = std::conditional_t<XH, uint16_t, float>;
    using XV = std::conditional_t<XH, uint2, f4_t>;  // four activations
    const XT* xg = (const XT*)a.X + (size_t)group * a.x_group_stride + (size_t)m0 * a.x_stride;
    // (all of them requested at once where the registers hold them)
    constexpr int NK = NT / 2, NH = 2 * BPW, NB = TT * NH, AHEAD = NB * NK <= 16 ? NB : 2;
    XV raw[AHEAD][NK];
    auto fetch = [&](int i, XV (&r)[NK]) {  // half stage i % NH (128 columns) of token tile i / NH; lanes 0-31 even tokens, 32-63 odd ones
      const uint32_t col = min((ws0 * 2u + i % NH) * 128u, a.cols - 128u) + 4u * (lane & 31u);
#pragma unroll
      for (int k = 0; k < NK; k++) r[k] = *(const XV*)(xg + (size_t)min(16u * (i / NH) + 2u * k + (lane >> 5), ntok - 1u) * a.x_stride + col);  // tokens past n repeat the last
    };
#pragma unroll
    for (int i = 0; i < AHEAD; i++) fetch(i, raw[i]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NB; i++) {
      const int hb = i % NH;
      XV(&r)[NK] = raw[i % AHEAD];
#pragma unroll
      for (int k = 0; k < NK; k++) {
        uint2 v;
        if constexpr (XH) v = r[k];
        else v = uint2{pack_h2(r[k][0], r[k][1]), pack_h2(r[k][2], r[k][3])};
        *(uint2*)(xs + (2u * k + (lane >> 5)) * kRowsXPitch + 8u * (lane & 31u)) = v;
      }
      asm volatile("" ::: "memory");  // (written and read through different types)
      if (i + AHEAD < NB) fetch(i + AHEAD, raw[i % AHEAD]);
#pragma unroll
      for (int js = 0; js < 4; js++) {
        const uint8_t* p = xs + (n16 & (NT - 1u)) * kRowsXPitch + 64u * js;
        uint32_t(&x)[4] = xr[i / NH][hb * 4 + js];
        if constexpr (PAIR || GROUPS) {
          const uint2 lo = *(const uint2*)(p + 8u * q), hi = *(const uint2*)(p + 32u + 8u * q);
          if constexpr (PAIR) {
            x[0] = __builtin_amdgcn_perm(hi.x, lo.x, 0x05040100u); x[1] = __builtin_amdgcn_perm(hi.x, lo.x, 0x07060302u);
            x[2] = __builtin_amdgcn_perm(hi.y, lo.y, 0x05040100u); x[3] = __builtin_amdgcn_perm(hi.y, lo.y, 0x07060302u);
          } else {
            x[0] = lo.x; x[1] = lo.y; x[2] = hi.x; x[3] = hi.y;
          }
        } else {
          const uint4 v = *(const uint4*)(p + 16u * q);
          x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
        }
        // columns past the row's end (a row may end with half a stage, the last wave with a whole one): zero activations
        if ((ws0 * 2u + hb) * 128u >= a.cols) x[0] = x[1] = x[2] = x[3] = 0u;
      }
      asm volatile("" ::: "memory");
    }
  }
  wait_lgkm0();  // the staging area is read: ring slots from here on
#pragma unroll
  for (int i = rows_early<F>(S); i < S; i++)
    if ((uint32_t)i < total) request(tile0 + i / BPW, i % BPW, (uint32_t)i);
  if (F::LDS_WORDS) __syncthreads();

  const f4_t zero = {0.f, 0.f, 0.f, 0.f};
  const uint32_t ones[4] = {0x3C003C00u, 0x3C003C00u, 0x3C003C00u, 0x3C003C00u};
  uint32_t i = 0, slot = 0;
  for (uint32_t tl = 0; tl < ntile; tl += UT) {
    f4_t acc[UT][TT];
#pragma unroll
    for (int u = 0; u < UT; u++) {
#pragma unroll
      for (int t = 0; t < TT; t++) acc[u][t] = zero;
      if (tl + u >= ntile) continue;
      const uint32_t row = min(row_tile(tile0 + tl + u) * 16u + n16, a.rows - 1u), wmis = of_tile(tile0 + tl + u).mis;
#pragma unroll
      for (int b = 0; b < BPW; b++, i++) {
        if (i + S <= total) wait_vm<NPI*(S - 1)>();  // S - 1 younger stages may stay in flight
        else wait_vm<0>();
        const LdsRow lrow = LdsRow::of(mine + slot * SLOT + n16 * (uint32_t)(P * 16),
                                       (wmis + row * a.row_bytes + min(ws0 + b, a.nws - 1u) * (uint32_t)F::WS_BYTES) & 15u);
        if (ws0 + b < a.nws) {
#pragma unroll
          for (int js = 0; js < 8; js++) {
            const uint32_t(&x)[4] = xr[0][b * 8 + js];
            f4_t& sum = acc[u][0];
            if constexpr (GROUPS) {
              const auto f = F::get(lrow, js, q, tbl);
              sum = fma4(f.sa, mfma_f16_k16(x[0], x[1], f.h[0], f.h[1], zero), sum);
              sum = fma4(f.sb, mfma_f16_k16(x[2], x[3], f.h[2], f.h[3], zero), sum);
            } else {
              const FragOut f = F::finish(F::load_raw(lrow, (uint32_t)js, q), (uint32_t)js, q, tbl);
              // (formats of 32-weight blocks: past a row that ends with half a stage the bytes are no blocks)
              const float sc = !PAIR || (ws0 + b) * 256u + 32u * js < a.cols ? f.scale : 0.f;
              if constexpr (ROUND) {
                uint32_t h[4];
#pragma unroll
                for (int p = 0; p < 4; p++) h[p] = scale_round_h2(f.h[p], sc, F::HAS_ADD ? f.add : 0.f);
#pragma unroll
                for (int t = 0; t < TT; t++) acc[u][t] = mfma_f16(xr[t][b * 8 + js], h, acc[u][t]);
              } else {
                sum = fma4(sc, mfma_f16(x, f.h, zero), sum);
                if constexpr (F::HAS_ADD) sum = fma4(f.add, mfma_f16(x, ones, zero), sum);
              }
            }
          }
        }
        wait_lgkm0();  // the slot is read: refill it
        if (i + S < total) request(tile0 + (i + S) / BPW, (int)((i + S) % BPW), slot);
        slot = slot + 1 == S ? 0u : slot + 1;
      }
    }
    // [wave][row tile][token tile][token][row]; two buffers, so that one barrier separates the meetings, or (TT > 1, GU: LDS) one
    // that everyone has read when the next partial tiles come
    float* rb = red + (TT == 1 && !GU ? (tl / UT) & 1u : 0u) * (nwaves * (256u * UT));
    if ((TT > 1 || GU) && tl > 0) __syncthreads();
#pragma unroll
    for (int u = 0; u < UT; u++)
#pragma unroll
      for (int t = 0; t < TT; t++)
#pragma unroll
        for (int k = 0; k < 4; k++) rb[(((wave * UT + u) * TT + t) * 16u + 4u * q + k) * 16u + n16] = acc[u][t][k];
    __syncthreads();  // (everyone read this buffer's last contents before the barrier between)
    auto sum = [&](uint32_t t, uint32_t u, uint32_t r) {
      float s = 0.f;
      for (uint32_t w0 = 0; w0 < nwaves; w0 += 8u) {  // eight partials requested before the first is added
        float v[8];
#pragma unroll
        for (uint32_t k = 0; k < 8u; k++) v[k] = rb[((min(w0 + k, nwaves - 1u) * UT + u) * (16u * TT) + t) * 16u + r];
#pragma unroll
        for (uint32_t k = 0; k < 8u; k++) s += w0 + k < nwaves ? v[k] : 0.f;
      }
      return s;
    };
    if constexpr (GU) {
      for (uint32_t idx = tid; idx < 16u * ntok; idx += nthreads) {
        const uint32_t t = idx >> 4, orow = row_tile(tile0 + tl) * 16u + (idx & 15u);
        if (orow >= a.rows) continue;
        const float g = fminf(sum(t, 0u, idx & 15u), 10.f), u = fminf(fmaxf(sum(t, 1u, idx & 15u), -10.f), 10.f);
        a.H[(size_t)(m0 + t) * a.rows + orow] = __builtin_bit_cast(uint16_t, (_Float16)(g / (1.f + expf(-g)) * u));
      }
    } else
    for (uint32_t idx = tid; idx < 16u * UT * ntok; idx += nthreads) {
      const uint32_t t = idx / (16u * UT), r = idx % (16u * UT), u = r >> 4, orow = (tile0 + tl) * 16u + r;
      if (tl + u >= ntile || orow >= a.rows) continue;
      const float s = sum(t, u, r & 15u);
      float* y = a.Y + (size_t)(m0 + t) * a.rows + orow;
      *y = a.accumulate ? *y + s : s;
    }
  }
}

}  // namespace msq

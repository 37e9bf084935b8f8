// Prefill MoE, shared expert of a K-quant / Q8_0 type (few tokens: msq_rows.cuh): dense gate/up and down products over all tokens of the call
// (reference: the shared expert's part of ms::q::encode_moe_prefill, src/kernels/quant.mm:433-612).
//
// A workgroup of eight waves owns 128 weight rows x 128 tokens and walks K in stages of 64 columns, both operands in LDS
// as fp16 rows of 128 bytes (two buffers each). The activations of the next stage come by loads that write LDS
// themselves; the weights of the next stage are decoded by all threads, a quarter of a row each, from bytes requested
// a stage or more ahead, so a weight is unpacked once per 128 tokens and no lane loads a byte twice.
// A wave multiplies two token tiles by four row tiles: six fragment reads per eight matrix instructions.
// Weights stay exact: payloads are integers in fp16, and the fp32 scale of a group (32 columns of Q8_0, 16 of Q6_K, whose
// steps are therefore issued as two matrix instructions of K = 16) is applied to the group's product. Those multiply-adds,
// four per matrix instruction, bound the kernel with many tokens (512 of the 850 vector instructions that a wave issues per
// block of Q6_K), which is why two workgroups
// share a CU (128 registers, 68 KB). Measured: Q6_K, 4096 tokens, dim 5120, inter 2304: gate/up 421 us, down 215 us = 455
// TFLOP/s, against 4.83 and 1.77 ms of a kernel that decoded every weight once per sixteen tokens.
#pragma once
#include "msq_rows.cuh"

namespace msq {

struct PfTileArgs {
  const uint16_t* A;     // fp16 activations [cnt][K] (of the shared expert's entries)
  const uint8_t* W[2];   // gate, up; or down
  uint16_t* H;           // gate/up output [cnt][N] fp16
  float* Z;              // down output [cnt][N]
  uint32_t cnt, K, N, row_bytes;
  uint32_t row_chunks, token_blocks;
};

constexpr int kPfTileThreads = 512, kPfTileTok = 128, kPfTileRows = 128;
constexpr int kPfTileBuf = 128 * 128;  // bytes of one operand's stage: 128 rows of 64 halves

// Where 16-byte chunk c of row r sits in a staged operand: rows are 128 bytes apart, so the row's low three bits go into
// the chunk's place (a 16-byte read serves groups of eight rows of one chunk and eight of its neighbour)
__device__ __forceinline__ uint32_t pf_tile_at(uint32_t r, uint32_t c) { return r * 128u + 16u * (c ^ (r & 7u)); }

// the four dwords at a 2-byte-aligned offset, as aligned loads plus the word that follows (never past the bytes asked for)
struct Raw4 { u32x4 v; uint32_t tail, odd; };
__device__ __forceinline__ Raw4 pf_ld4(rsrc_t rs, uint32_t at) {
  const uint32_t odd = at & 2u, o = at - odd;
  const u128_a2 v = buf_ld128(rs, o, 0u);
  return {u32x4{v.x, v.y, v.z, v.w}, buf_ld32(rs, o + (odd ? 16u : 12u), 0u), odd};
}
__device__ __forceinline__ void pf_fix4(const Raw4& r, uint32_t (&w)[4]) {
#pragma unroll
  for (int i = 0; i < 4; i++) w[i] = __builtin_amdgcn_alignbit(i < 3 ? r.v[i + 1] : r.tail, r.v[i], r.odd * 8u);
}

// A decoder's thread (row, quarter q) turns its bytes of a 256-column block into the 16 weights it owns of each of the
// block's four stages.
//   acol(c), STAGE_COLS  column of chunk c of the activations in stage 0, and how far the next stage is on
//   decode(raw, s, q)    stage s: payload halves; put() stores them where the fragments are read, and the scale
struct TileQ6K {
  static constexpr int BLOCK_BYTES = 210, GROUPS = 4, STAGE_COLS = 32;  // GROUPS: scales per row and stage
  // thread q owns the group of 16 columns 128 (q / 2) + 32 s + 16 (q % 2) of stage s: its bytes are contiguous
  __device__ static uint32_t acol(uint32_t c) { return 128u * (c >> 2) + 16u * ((c >> 1) & 1u) + 8u * (c & 1u); }
  struct Raw { Raw4 l0, l1, h; uint32_t s0, s1, st, d, odd; };
  __device__ static Raw load(rsrc_t rs, uint32_t at, uint32_t q) {
    const uint32_t h = q >> 1, l0 = 16u * (q & 1u);
    Raw r;
    r.l0 = pf_ld4(rs, at + 64u * h + l0);
    r.l1 = pf_ld4(rs, at + 64u * h + 32u + l0);
    r.h = pf_ld4(rs, at + 128u + 32u * h + l0);
    const uint32_t sa = at + 192u + 8u * h;
    r.odd = sa & 2u;
    const u64_a2 s = buf_ld64(rs, sa - r.odd, 0u);
    r.s0 = s.x; r.s1 = s.y;
    r.st = buf_ld32(rs, sa - r.odd + (r.odd ? 8u : 4u), 0u);
    r.d = buf_ld16(rs, at + 208u, 0u);
    return r;
  }
  __device__ static void stage(const Raw& r, int s, uint32_t q, uint32_t row, uint8_t* b, float* sc) {
    uint32_t l[4], h[4];
    pf_fix4((s & 1) ? r.l1 : r.l0, l);
    pf_fix4(r.h, h);
    const uint32_t bias = 0xE420E420u;  // -1056 = -(1024 + 32) in both halves
#pragma unroll
    for (int i = 0; i < 4; i++) {  // columns 4 i .. 4 i + 3 of the group: half q % 2 of chunk i of step q / 2
      const uint32_t v = ((l[i] >> (4 * (s >> 1))) & 0x0F0F0F0Fu) | (((h[i] >> (2 * s)) & 0x03030303u) << 4);
      *(uint2*)(b + pf_tile_at(row, 4u * (q >> 1) + i) + 8u * (q & 1u)) =
          uint2{pk_add_f16(bytes01_to_h2_1024(v), bias), pk_add_f16(bytes23_to_h2_1024(v), bias)};
    }
    // scale bytes 8 (q / 2) + 2 s + q % 2 of the block, s = 0 .. 3
    const uint32_t w = s < 2 ? __builtin_amdgcn_alignbit(r.s1, r.s0, r.odd * 8u) : __builtin_amdgcn_alignbit(r.st, r.s1, r.odd * 8u);
    const int k = (int)(int8_t)((w >> (16 * (s & 1) + 8u * (q & 1u))) & 0xFFu);
    sc[4u * row + q] = half_bits_to_float(r.d) * (float)k;
  }
};
struct TileQ8_0 {
  static constexpr int BLOCK_BYTES = 272, GROUPS = 2, STAGE_COLS = 64;
  __device__ static uint32_t acol(uint32_t c) { return 8u * c; }
  struct Raw { Raw4 v[4]; uint32_t d[4]; };
  // thread q owns columns 16 q .. 16 q + 15 of every stage: half q % 2 of 32-weight block q / 2 of the stage's two
  __device__ static Raw load(rsrc_t rs, uint32_t at, uint32_t q) {
    Raw r;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const uint32_t b = at + 34u * (2u * s + (q >> 1));
      r.v[s] = pf_ld4(rs, b + 2u + 16u * (q & 1u));
      r.d[s] = buf_ld16(rs, b, 0u);
    }
    return r;
  }
  __device__ static void stage(const Raw& r, int s, uint32_t q, uint32_t row, uint8_t* b, float* sc) {
    uint32_t v[4];
    pf_fix4(r.v[s], v);
    const uint32_t bias = 0xE480E480u;  // -1152 in both halves (bytes become q + 128)
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const uint32_t lo = v[2 * i] ^ 0x80808080u, hi = v[2 * i + 1] ^ 0x80808080u;
      *(uint4*)(b + pf_tile_at(row, 2u * q + i)) =
          uint4{pk_add_f16(bytes01_to_h2_1024(lo), bias), pk_add_f16(bytes23_to_h2_1024(lo), bias),
                pk_add_f16(bytes01_to_h2_1024(hi), bias), pk_add_f16(bytes23_to_h2_1024(hi), bias)};
    }
    sc[2u * row + (q >> 1)] = half_bits_to_float(r.d[s]);  // (two threads, one value: no branch)
  }
};

template <class D, bool GU>
__global__ __launch_bounds__(kPfTileThreads, 4) void moe_pf_tile_kernel(const PfTileArgs a) {
  constexpr int NM = GU ? 2 : 1, G = D::GROUPS;
  constexpr bool K16 = G == 4;  // a step holds two scale groups
  extern __shared__ __attribute__((aligned(16))) uint32_t smem[];
  uint8_t* abuf = (uint8_t*)smem;                       // [2][128 tokens][64]
  uint8_t* bbuf = abuf + 2 * kPfTileBuf;                // [2][128 rows][64]
  float* sbuf = (float*)(bbuf + 2 * kPfTileBuf);        // [2][128 rows][G]
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t n16 = lane & 15u, q = lane >> 4;
  const uint32_t wm = wave & 3u, wn = wave >> 2;  // the wave's token tiles wm, wm + 4 and its half of the rows
  const uint32_t rc = blockIdx.x % a.row_chunks, m0 = (blockIdx.x / a.row_chunks) * kPfTileTok;
  const uint32_t cnt = min((uint32_t)kPfTileTok, a.cnt - m0);

  // staged row r: gate/up -- each half of the rows is 32 gate rows, then the same 32 up rows
  auto weight_row = [&](uint32_t r) { return GU ? rc * 64u + (r >> 6) * 32u + (r & 31u) : rc * 128u + r; };
  const uint32_t drow = tid >> 2, dq = tid & 3u;
  const uintptr_t wa = (uintptr_t)(GU && (drow & 32u) ? a.W[1] : a.W[0]);
  // (one descriptor per lane would not be uniform: gate and up rows are decoded by different waves -- rows 0-31 and
  // 64-95 are gate, 32-63 and 96-127 up, sixteen rows a wave)
  const uintptr_t wbase = ((uintptr_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)wa >> 32)) << 32) |
                          (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)wa);
  const uint32_t wmis = (uint32_t)wbase & 3u;  // whole aligned words
  const rsrc_t wrs = make_rsrc((const void*)(wbase - wmis), (wmis + a.N * a.row_bytes + 3u) & ~3u);
  const uint32_t woff = wmis + min(weight_row(drow), a.N - 1u) * a.row_bytes;

  const rsrc_t ars = make_rsrc(a.A + (size_t)m0 * a.K, ((cnt - 1u) * a.K + a.K) * 2u);
  uint32_t aoff[2];
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const uint32_t i = (uint32_t)k * kPfTileThreads + tid, t = i >> 3;
    aoff[k] = (min(t, cnt - 1u) * a.K + D::acol((i & 7u) ^ (t & 7u))) * 2u;  // tokens past the last repeat it
  }
  auto a_request = [&](uint32_t st, uint32_t buf) {
    const uint32_t so = ((st >> 2) * 256u + (st & 3u) * (uint32_t)D::STAGE_COLS) * 2u;
#pragma unroll
    for (int k = 0; k < 2; k++) lds_dma16(ars, abuf + buf * kPfTileBuf + ((uint32_t)k * kPfTileThreads + wave * 64u) * 16u, aoff[k], so);
  };

  // where the wave's fragments start: token tile t and row tile r are 64 and 16 rows further on
  uint32_t xat[2][2], wat[2];
#pragma unroll
  for (int js = 0; js < 2; js++) {
    const uint32_t tr = wm * 16u + n16;
    xat[js][0] = K16 ? pf_tile_at(tr, 4u * js + (q >> 1)) + 8u * (q & 1u) : pf_tile_at(tr, 4u * js + q);
    xat[js][1] = K16 ? pf_tile_at(tr, 4u * js + 2u + (q >> 1)) + 8u * (q & 1u) : 0u;
    wat[js] = pf_tile_at(wn * 64u + n16, 4u * js + q);
  }
  f4_t acc[2][4];
#pragma unroll
  for (int t = 0; t < 2; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) acc[t][r] = f4_t{0.f, 0.f, 0.f, 0.f};
  const f4_t zero = {0.f, 0.f, 0.f, 0.f};
  const uint32_t nblk = a.K / 256u, nst = 4u * nblk;

  typename D::Raw raw = D::load(wrs, woff, dq);
  a_request(0, 0);
  D::stage(raw, 0, dq, drow, bbuf, sbuf);
  wait_vm<0>();
  __syncthreads();

  for (uint32_t blk = 0; blk < nblk; blk++) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const uint32_t st = 4u * blk + s;
      const int buf = s & 1;  // (four stages a block: a stage's buffers are known at compile time)
      // the other buffers were last read one stage ago, before the barrier; the last stage requests itself again
      a_request(min(st + 1u, nst - 1u), buf ^ 1);
      __builtin_amdgcn_sched_barrier(0);
      const uint8_t* ab = abuf + buf * kPfTileBuf;
      const uint8_t* bb = bbuf + buf * kPfTileBuf;
      const float* sb = sbuf + buf * (128 * G) + G * (wn * 64u + n16);
#pragma unroll
      for (int js = 0; js < 2; js++) {
        uint32_t x[2][4];
#pragma unroll
        for (int t = 0; t < 2; t++) {
          if constexpr (K16) {
            const uint2 lo = *(const uint2*)(ab + xat[js][0] + t * 8192), hi = *(const uint2*)(ab + xat[js][1] + t * 8192);
            x[t][0] = lo.x; x[t][1] = lo.y; x[t][2] = hi.x; x[t][3] = hi.y;
          } else {
            const uint4 v = *(const uint4*)(ab + xat[js][0] + t * 8192);
            x[t][0] = v.x; x[t][1] = v.y; x[t][2] = v.z; x[t][3] = v.w;
          }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const uint4 v = *(const uint4*)(bb + wat[js] + r * 2048);
          if constexpr (K16) {
            const float2 sc = *(const float2*)(sb + 64 * r + 2 * js);
#pragma unroll
            for (int t = 0; t < 2; t++) {
              acc[t][r] = fma4(sc.x, mfma_f16_k16(x[t][0], x[t][1], v.x, v.y, zero), acc[t][r]);
              acc[t][r] = fma4(sc.y, mfma_f16_k16(x[t][2], x[t][3], v.z, v.w, zero), acc[t][r]);
            }
          } else {
            const float sc = sb[32 * r + js];
            const uint32_t h[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int t = 0; t < 2; t++) acc[t][r] = fma4(sc, mfma_f16(x[t], h, zero), acc[t][r]);
          }
        }
      }
      D::stage(raw, (s + 1) & 3, dq, drow, bbuf + (buf ^ 1) * kPfTileBuf, sbuf + (buf ^ 1) * (128 * G));
      // the next stage's activations, requested a stage of products ago. (Waited for ahead of the loads of the next block's
      // bytes: behind them it would take a count of loads, which the compiler is free to merge.)
      if (s == 2) {  // the block's last stage is decoded: the next block's bytes, in flight over the next stage's products
        wait_vm<0>();
        __builtin_amdgcn_sched_barrier(0);
        raw = D::load(wrs, woff + min(blk + 1u, nblk - 1u) * (uint32_t)D::BLOCK_BYTES, dq);
        __builtin_amdgcn_sched_barrier(0);
        wait_vm<63>();  // waits for nothing: without it the Q8_0 variant keeps 44 registers in scratch memory
      }
      else wait_vm<0>();
      __syncthreads();
    }
  }

  // D: lane holds weight row n16 of a tile, tokens 4 q + i
#pragma unroll
  for (int t = 0; t < 2; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t tok = (wm + 4u * t) * 16u + 4u * q + i;
      if (tok >= cnt) continue;
      const size_t orow = (size_t)(m0 + tok) * a.N;
#pragma unroll
      for (int r = 0; r < 4 / NM; r++) {
        const uint32_t row = weight_row(wn * 64u + 16u * r + n16);
        if (row >= a.N) continue;
        if constexpr (GU) {
          const float g = fminf(acc[t][r][i], 10.f), u = fminf(fmaxf(acc[t][r + 2][i], -10.f), 10.f);
          a.H[orow + row] = __builtin_bit_cast(uint16_t, (_Float16)(g / (1.f + expf(-g)) * u));
        } else {
          a.Z[orow + row] = acc[t][r][i];
        }
      }
    }
}

}  // namespace msq

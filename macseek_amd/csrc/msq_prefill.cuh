// Prefill MoE: grouped GEMM over experts on the matrix cores (reference operator: ms::q::encode_moe_prefill,
// src/kernels/quant.mm:433-612; reference kernels q_moe_gather / q_moe_rgu / q_moe_rdown / q_moe_reduce,
// src/kernels/quant_moe_prefill.metal:22-29,190-239,275-303,330-344).
//
//   convert: Xg[total + t] = fp16(X[t]); an entry's row is its token's (or gather: Xg[i] = fp16(X[tok[i]]), see the host)
//   gate/up: H[i][r] = fp16(silu(min(Xg_e[i].Wg[r], 10)) * clamp(Xg_e[i].Wu[r], -10, 10) * wt[i])
//   down   : Z[i][c] = H_e[i] . Wd[c]   (fp32, one row per entry)
//   reduce : Y[t] += Z[total + t] + sum_k Z[slot_of[t][k]]   in that fixed order
//
// The routed experts and a shared expert of a codebook type go through the block GEMM below, a K-quant / Q8_0 shared
// expert through the dense tile kernel of msq_prefill_tile.cuh.
#pragma once
#include <algorithm>
#include <type_traits>
#include <utility>

#include "msq_mfma.cuh"

namespace msq {

// ------------------------------------------------------------------------------------------------ block GEMM
// Grouped GEMM for the 256-weight codebook formats (block fragments, see msq_mfma.cuh). A work item is one expert's
// block of entries (T token tiles of 16) times a chunk of weight rows; the item's waves own different
// weight-row tiles and walk K block by block (256 columns): the activation block is staged in LDS for
// all waves, every wave decodes the fragments of its own rows once per block and reuses each of them for all T token
// tiles, and accumulates in the matrix cores; the scale rides in the fragments. Weights are decoded exactly
// once per (item, row), no lane loads a weight byte twice, and the next block's bytes are in flight during a block.
// What bounds it. Small items (T <= 3): vector issue (14 instructions per eight weights of a lane, 62 % of the cycles), LDS (51 %)
// and the texture addresser (53 %) beside each other, four waves per SIMD; a unit's first trip to memory and its end are 10 %
// (gate/up) to 25 % (down). Larger blocks: see pf_big_body. Against a variant that fetched IQ2_XXS rows lane by lane (three loads
// a row, 50 vector cache lookups each), staged activations through registers and tested the tile count in every step
// (27 instructions per eight weights), launched a workgroup per unit and gathered a copy of the entries' rows: 2048 tokens,
// 384 IQ2_XXS experts of 7168x2048: gate/up 644 -> 537 us (T > 3) and 1080 -> 1009, down 348 -> 308 and 569 -> 565, the call
// 2735 -> 2501; IQ1_S 5120x2304: 37 tokens 515 -> 451, 4096 tokens 3693 -> 3141.
struct PfBlkArgs {
  const uint16_t* A;        // fp16 activations [entries][K], or (tok) [tokens][K]
  const int* tok;           // per entry: its row of A; null: the entry itself
  uint32_t a_bytes;         // (tok) bytes of A
  const uint64_t* ptrs;     // per expert: gate, up, down addresses
  const uint32_t* items;    // per item: expert, first entry of the block, entries in the block
  const float* wt;          // per routed entry: routing weight
  uint16_t* H;              // gate/up output [entries][N] fp16
  float* Z;                 // down output [entries][N] fp32
  uint32_t nitems, total;
  uint32_t K, N, row_bytes, nblocks;
  uint32_t row_chunks;      // chunks of pf_blk_rows() weight rows
  uint32_t chunks_per_wg;   // consecutive row chunks one workgroup takes, one after the other
  uint32_t row_groups;      // units of work per item: row_chunks / chunks_per_wg, rounded up
  uint32_t per_xcd;         // units of an XCD (see PfUnit)
  uint32_t* queue;          // eight counters, one per XCD: units taken beyond those that the workgroups start with; or null
};

// A unit of work is one item's row chunks of one workgroup. Unit 8 s + x belongs to XCD x: the units of one item stay on one
// XCD (shared L2 for its activations), and items are dealt round-robin over the XCDs; consecutive workgroups land on
// different XCDs. There is a workgroup for every unit, or (QUEUE) as many as the chip holds: a workgroup then takes units of
// its XCD until they are used up, the first by its number, the others from the XCD's counter. The tables are in LDS once, and a
// unit does not wait for the workgroup before it to be taken down and its own to be set up (4096 tokens of IQ1_S: blocks of
// the first product 942 -> 859 us, calls 3349 -> 3160; 2048 of IQ2_XXS 2500 -> 2470). The rule is at the launch.
// (The tables are read as constants, which they are while the kernel runs: scalar loads.)
struct PfUnit {
  uint32_t cnt, base;  // the item's entries (none: the last items of eight may be missing), the first one
  uint32_t group;
  uint64_t w[2];       // the expert's matrices: gate and up, or down
  template <bool GU>
  __device__ __forceinline__ static PfUnit of(const PfBlkArgs& a, uint32_t s) {
    const uint32_t item = (s / a.row_groups) * 8u + (blockIdx.x & 7u);
    if (item >= a.nitems) return PfUnit{};
    const auto items = (const __attribute__((address_space(4))) uint32_t*)(uintptr_t)(a.items + 3 * (size_t)item);
    const uint32_t e = items[0], base = items[1];
    const auto ptrs = (const __attribute__((address_space(4))) uint64_t*)(uintptr_t)(a.ptrs + 3 * (size_t)e);
    return {items[2], base, s % a.row_groups, {ptrs[GU ? 0 : 2], ptrs[GU ? 1 : 2]}};
  }
};

constexpr int kPfBigTokens = 112, kPfBigTiles = kPfBigTokens / 16;
// waves per workgroup by token tiles per item: four per SIMD for up to three tiles, three for more (registers)
constexpr int pf_blk_waves(int T) { return T > 3 ? 12 : 16; }
// weight-row tiles per wave: two fragments per K step (gate + up of one tile, or two tiles of the down matrix) keep the
// register count low enough for three or four waves per SIMD, which is what overlaps decode, matrix and LDS work
constexpr int pf_blk_rt(bool gu, int) { return gu ? 1 : 2; }
constexpr int pf_blk_rows(bool gu, int T) { return pf_blk_waves(T) * pf_blk_rt(gu, T) * 16; }  // weight rows per work item
// Weight bytes come through LDS: a wave's block bytes of 16 rows (its two fragments: twice that), PIECES 16-byte pieces a
// row, by loads that write LDS themselves
template <class B>
constexpr size_t pf_blk_raw_lds(int T) { return pf_blk_waves(T) * 2 * (16 * 16 * B::PIECES); }
// Activations are staged by halves of a block: the columns of steps 0-3 and those of steps 4-7, in two planes each (chunks 0
// and 2, chunks 1 and 3) of 128-byte rows. Unit 4 (q / 2) + j % 4 of a row sits at place unit ^ (row / 2) % 8. A 16-byte LDS
// read serves the lanes in four groups of sixteen -- {0-7, 24-31}, {8-15, 16-23}, {32-39, 56-63}, {40-47, 48-55}, measured
// -- so a group holds tokens 0-7 of one chunk and tokens 8-15 of its neighbour (lane = 16 q + token): sixteen different
// bank groups. Two whole blocks (one barrier a block) where they fit, else one block, whose halves are refilled in turn.
constexpr int pf_half_bytes(int T) { return 16 * T * 256; }
constexpr size_t kPfLds = 160 * 1024;
template <class B>
constexpr bool pf_two_blocks(int T) { return T <= 3 && (size_t)B::LDS_WORDS * 4 + pf_blk_raw_lds<B>(T) + 4 * pf_half_bytes(T) <= kPfLds; }
template <class B>
constexpr size_t pf_act_lds(int T) { return (pf_two_blocks<B>(T) ? 4 : 2) * (size_t)pf_half_bytes(T); }
// ... of a launch: T = 3 holds items of one to three tiles, T = 7 of four to seven
template <class B>
constexpr size_t pf_act_lds_of_launch(int T) { return T > 3 ? pf_act_lds<B>(T) : std::max({pf_act_lds<B>(1), pf_act_lds<B>(2), pf_act_lds<B>(3)}); }
template <class B>
constexpr size_t pf_blk_lds(int T) { return (size_t)B::LDS_WORDS * 4 + pf_act_lds_of_launch<B>(T) + pf_blk_raw_lds<B>(T); }

template <int N, class F>
__device__ __forceinline__ void static_for(F f) {
  [&]<int... I>(std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }(std::make_integer_sequence<int, N>{});
}

// An expert's matrix: a descriptor over the whole aligned 16-byte pieces that hold it, and where in the first it starts.
// (A matrix is far below 4 GiB; a weight row is then a 32-bit offset per lane and the block's a scalar one.)
struct PfMatrix {
  rsrc_t rs;
  uint32_t mis, bytes;
  __device__ __forceinline__ static PfMatrix of(const PfBlkArgs& a, uint64_t at) {
    // (uniform, which an inline assembly operand has to be shown)
    const uintptr_t base = ((uintptr_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(at >> 32)) << 32) |
                           (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)at);
    const uint32_t mis = (uint32_t)base & 15u, bytes = (mis + a.N * a.row_bytes + 15u) & ~15u;
    return {make_rsrc((const void*)(base - mis), bytes), mis, bytes};
  }
};
// The weight bytes of a wave's fragments: the block at scalar byte `at` of 16 rows, into an LDS slot of the wave's own. Lane l
// of load k fetches the piece at place 64 k + l. (Dwords past the matrix's end lie past its descriptor's: zeros, no traffic.)
template <class B>
struct PfRows {
  static constexpr int LOADS = (16 * B::PIECES + 63) / 64;
  static constexpr uint32_t SLOT = 16 * 16 * B::PIECES;
  uint32_t from[LOADS];  // where the lane's piece lies behind the first row's block
  uint32_t sel;          // the lane's row: which half of a dword a block starts in when the first row's starts in the low one
  __device__ __forceinline__ void init(uint32_t row_bytes, uint32_t lane) {
#pragma unroll
    for (int k = 0; k < LOADS; k++) {
      const uint32_t l = 64u * k + lane, row = min(l / B::PIECES, 15u), place = l % B::PIECES;
      from[k] = row * row_bytes + 16u * B::piece_at(row, place);  // (piece_at is its own inverse)
    }
    sel = ((lane & 15u) * row_bytes) & 2u ? SEL_LOW ^ SEL_FLIP : SEL_LOW;
  }
  __device__ __forceinline__ void request(const PfMatrix& w, uint8_t* slot, uint32_t at, uint32_t lane) const {
#pragma unroll
    for (int k = 0; k < LOADS; k++)
      if (64 * (k + 1) <= 16 * B::PIECES || 64u * k + lane < 16u * B::PIECES) lds_dma16(w.rs, slot + 1024 * k, (from[k] + at) & ~3u, 0u);
  }
  __device__ __forceinline__ typename B::Raw fetched(const typename B::At& lane_at, const uint8_t* slot, uint32_t at) const {
    return B::load(lane_at, (uint32_t)(uintptr_t)(lds_cptr_t)slot, sel ^ (at & 2u ? SEL_FLIP : 0u));
  }
};

// Results of an item's rows: SwiGLU and routing weight to H, or the plain sums to Z
template <bool GU, int T, int RT>
__device__ __forceinline__ void pf_epilogue(const PfBlkArgs& a, const f4_t (&acc)[T][GU ? 2 * RT : RT], uint32_t base, uint32_t cnt, uint32_t q,
                                            const uint32_t (&row_of)[RT]) {
  float wts[T][4];  // routing weights of the lane's entries, fetched together ahead of the epilogue's math
#pragma unroll
  for (int t = 0; t < T; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t entry = base + min(16u * t + 4u * q + i, cnt - 1);
      wts[t][i] = GU && entry < a.total ? a.wt[entry] : 1.f;
    }
  __builtin_amdgcn_sched_barrier(0);  // all requests first: sunk to their uses they would be waited for one by one
#pragma unroll
  for (int t = 0; t < T; t++) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t tok = 16u * t + 4u * q + i;
      if (tok >= cnt) continue;
      const uint32_t entry = base + tok;
#pragma unroll
      for (int jt = 0; jt < RT; jt++) {
        if (row_of[jt] >= a.N) continue;
        if constexpr (GU) {
          const float g = fminf(acc[t][2 * jt][i], 10.f), u = fminf(fmaxf(acc[t][2 * jt + 1][i], -10.f), 10.f);
          const float hv = g / (1.f + expf(-g)) * u * wts[t][i];
          a.H[(size_t)entry * a.N + row_of[jt]] = __builtin_bit_cast(uint16_t, (_Float16)hv);
        } else {
          a.Z[(size_t)entry * a.N + row_of[jt]] = acc[t][jt][i];
        }
      }
    }
  }
}

// The activations of an item's entries: consecutive rows of A, or (the first product) the rows that the entries' tokens name.
// A gathered copy costs a write and a read of every entry's row; the list costs one word a lane, beside the item's addresses
// in the same trip (4096 tokens, 36864 rows of 7168: copy 123 us, conversion of the tokens' own rows 22).
template <bool GU>
__device__ __forceinline__ rsrc_t pf_act_rows(const PfBlkArgs& a, const PfUnit& unit) {
  if (GU && a.tok) return make_rsrc(a.A, a.a_bytes);
  return make_rsrc(a.A + (size_t)unit.base * a.K, unit.cnt * a.K * 2u);
}
template <bool GU>
__device__ __forceinline__ uint32_t pf_act_row(const PfBlkArgs& a, uint32_t base, uint32_t row) {
  return GU && a.tok ? (uint32_t)a.tok[base + row] : row;
}

template <class B, bool GU, int T>
__device__ __forceinline__ void pf_block_body(const PfBlkArgs& a, PfUnit unit, bool first) {
  constexpr int WAVES = pf_blk_waves(T), NT = 64 * WAVES;
  constexpr int NM = GU ? 2 : 1, RT = pf_blk_rt(GU, T), R = RT * NM;
  constexpr int HALF = pf_half_bytes(T), PLANE = HALF / 2;
  constexpr bool TWO = pf_two_blocks<B>(T);
  static_assert(R == 2 && T <= 3, "fragments are processed in pairs; more token tiles: pf_big_body");
  extern __shared__ __attribute__((aligned(16))) uint32_t smem[];
  uint8_t* abuf = (uint8_t*)(smem + B::LDS_WORDS);  // [TWO: 2][2 halves][2 planes][T * 16 tokens][128 bytes]
  uint32_t tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // (kept from one unit to the next, what follows from it would cost registers)
  const uint32_t lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t n16 = lane & 15u, q = lane >> 4;
  const typename B::Low low = B::lane_low(n16);

  const uint32_t cnt = unit.cnt, base = unit.base, rc0 = unit.group * a.chunks_per_wg;
  // A workgroup takes chunks_per_wg consecutive row chunks of its item, one after the other: the first trip to memory
  // (about 4.5 us before the first block can be multiplied, 17 % of a down-projection workgroup's life) is paid once, and
  // the next chunk's first block is requested during the last block of the one before, where a single chunk would
  // fetch its last block again
  // (built into the down projection of the small items only: the other variants have no registers to spare for it)
  constexpr bool MULTI = !GU;
  const uint32_t nch = MULTI ? min(a.chunks_per_wg, a.row_chunks - rc0) : 1u;

  PfMatrix wm[NM];
  uint32_t row_of[RT];
#pragma unroll
  for (int m = 0; m < NM; m++) wm[m] = PfMatrix::of(a, unit.w[m]);
#pragma unroll
  for (int jt = 0; jt < RT; jt++) row_of[jt] = ((rc0 * WAVES + wave) * RT + jt) * 16u + n16;
  PfRows<B> rows;
  rows.init(a.row_bytes, lane);
  auto block_at = [&](int r, uint32_t off) { return wm[r % NM].mis + ((rc0 * WAVES + wave) * RT + r / NM) * 16u * a.row_bytes + off; };
  const typename B::At at_row = B::at_of(n16, q);
  uint8_t* const raw_lds = abuf + pf_act_lds_of_launch<B>(3) + wave * (R * PfRows<B>::SLOT);
  auto request = [&](int r, uint32_t off) { rows.request(wm[r % NM], raw_lds + r * PfRows<B>::SLOT, block_at(r, off), lane); };
  auto fetched = [&](int r, uint32_t off) { return rows.fetched(at_row, raw_lds + r * PfRows<B>::SLOT, block_at(r, off)); };

  // activation loader. Piece g of a block (TWO) or of half h: row g / 32 (g / 16), then (half,) plane and unit.
  constexpr int PB = TWO ? 5 : 4, AG = ((T << (4 + PB)) + NT - 1) / NT;
  static_assert(TWO || AG == 1);
  const rsrc_t ars = pf_act_rows<GU>(a, unit);
  uint32_t aoff[AG];
  uint8_t* adst[AG];
#pragma unroll
  for (int i = 0; i < AG; i++) {
    // rows past the block's last entry repeat it (their products are never stored): no branch around the load, so
    // the number of loads in flight stays known to every wait that follows
    const uint32_t g = min(tid + i * NT, (16u * T << PB) - 1u), row = g >> PB, h = TWO ? (g >> 4) & 1u : 0u, plane = (g >> 3) & 1u, unit = g & 7u;
    aoff[i] = pf_act_row<GU>(a, base, min(row, cnt - 1u)) * (a.K * 2u) + (64u * (2u * (unit >> 2) + plane) + 32u * h + 8u * (unit & 3u)) * 2u;
    adst[i] = abuf + h * HALF + plane * PLANE + row * 128u + 16u * (unit ^ ((row >> 1) & 7u));
  }
  if constexpr (GU)
#pragma unroll
    for (int i = 0; i < AG; i++) asm volatile("" : "+v"(aoff[i]));  // (waited for here, not behind the weights that are asked for next)
  u32x4 pa[TWO ? 1 : 2][AG];  // (a plain vector type: the HIP struct type keeps the array in scratch memory)
  auto a_issue = [&](int h, uint32_t kc) {
#pragma unroll
    for (int i = 0; i < AG; i++) pa[h][i] = buf_ld128v(ars, aoff[i], kc * 512u + 64u * h);
  };
  auto a_store = [&](int h, uint32_t at) {
#pragma unroll
    for (int i = 0; i < AG; i++)
      if (tid + i * NT < (16u * T << PB)) *(u32x4*)(adst[i] + at) = pa[h][i];
  };
  const uint32_t afrag = (uint32_t)(uintptr_t)(lds_cptr_t)abuf + (q & 1u) * PLANE + n16 * 128u + 16u * ((4u * (q >> 1)) ^ (n16 >> 1));
  auto next_k = [&](uint32_t kc) { return kc + 1u < a.nblocks ? kc + 1u : 0u; };  // (past a workgroup's last block: the first again)

  typename B::Raw cur[R];
#pragma unroll
  for (int r = 0; r < R; r++) request(r, 0u);
  a_issue(0, 0);
  if constexpr (!TWO) a_issue(1, 0);
  if (first) B::fill_lds(smem, (int)tid, NT);
  a_store(0, 0);
  if constexpr (!TWO) a_issue(0, next_k(0));
  wait_vm<0>();
#pragma unroll
  for (int r = 0; r < R; r++) cur[r] = fetched(r, 0u);
  __syncthreads();

  constexpr bool A2 = T < 3, LA = GU || T < 3;  // activations, table entries read a step ahead (three tiles: registers)
  typename B::Look lk[2][2];
  if constexpr (LA) {
    lk[0][0] = B::template lookup<0>(cur[0], low);
    lk[0][1] = B::template lookup<0>(cur[1], low);
  }
  u32x4 af[A2 ? 2 : 1][T];
  uint32_t sc[R];
  uint32_t kb = 0;  // blocks done so far (double buffering: block kb sits in buffer kb % 2)
  for (uint32_t c = 0; c < nch; c++) {
  const bool more = c + 1 < nch;
  f4_t acc[T][R];
#pragma unroll
  for (int t = 0; t < T; t++)
#pragma unroll
    for (int r = 0; r < R; r++) acc[t][r] = f4_t{0.f, 0.f, 0.f, 0.f};

  for (uint32_t kc = 0; kc < a.nblocks; kc++, kb++) {
    // the block requested during this one: the chunk's next, or the first of the workgroup's next chunk, or (nothing left)
    // this one again: no branch around the loads
    const bool lastb = kc + 1 == a.nblocks;
    const uint32_t kn = !lastb ? kc + 1 : more ? 0u : kc;
    // (the host lets a workgroup take several chunks only when all chunks are whole: the next chunk's rows are then the
    // same number of bytes further for every lane)
    const uint32_t wn = kn * (uint32_t)B::BLOCK_BYTES + (c + (lastb && more ? 1u : 0u)) * ((uint32_t)(WAVES * RT * 16) * a.row_bytes);
    const uint32_t at = afrag + (TWO ? (kb & 1u) * (2u * HALF) : 0u), ka = next_k(kc);
    static_for<8>([&](auto j_) __attribute__((always_inline)) {
      constexpr int j = j_;
      constexpr bool fresh = !A2 || j == 0 || (!TWO && j == 4);  // behind a barrier: nothing could be read ahead of it
      auto a_read = [&](int i) {  // activations of step i, read with the fragments' column mapping
#pragma unroll
        for (int t = 0; t < T; t++) af[A2 ? i & 1 : 0][t] = lds_at<u32x4>(at ^ (16u * (i & 3)), (i >> 2) * HALF + t * 2048);
      };
      // The reads of step j + 1 are issued ahead of the arithmetic of step j (the scheduler would sink them to their use, and
      // the waves of a workgroup, in step behind every barrier, then take the LDS and the vector unit in turns)
      __builtin_amdgcn_sched_barrier(0);
      // the next block's bytes are requested a few at a time between the steps: requested all at once by
      // all waves right after the barrier, they queue up in the texture addresser and hold the waves at issue
      if constexpr (j < 2) request(j, wn);  // (the slots are read: the barrier has waited for that)
      if constexpr (TWO && j == 3) a_issue(0, ka);
      if constexpr (!TWO && j == 4) {
        // one block staged: its second half arrives, into the buffer that the block before has left
        a_store(1, HALF);
        __syncthreads();
        a_issue(1, ka);
      }
      if constexpr (fresh) a_read(j);
      if constexpr (!LA || j < 7) {
        constexpr int jl = LA ? j + 1 : j;
        lk[jl & 1][0] = B::template lookup<jl & 7>(cur[0], low);
        lk[jl & 1][1] = B::template lookup<jl & 7>(cur[1], low);
      }
      if constexpr (A2 && j < 7 && (TWO || j != 3)) a_read(j + 1);
      if constexpr (j == 7) {  // the block's own bytes are used up
        wait_vm<0>();
#pragma unroll
        for (int r = 0; r < R; r++) cur[r] = fetched(r, wn);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (j % 4 == 0) {
#pragma unroll
        for (int r = 0; r < R; r++) sc[r] = B::scale(cur[r], j / 4);
      }
      uint32_t h[2][4];
      B::finish(sc[0], lk[j & 1][0], h[0]);
      B::finish(sc[1], lk[j & 1][1], h[1]);
#pragma unroll
      for (int t = 0; t < T; t++) {
        const u32x4 v = af[A2 ? j & 1 : 0][t];
        const uint32_t x[4] = {v[0], v[1], v[2], v[3]};
        acc[t][0] = mfma_f16(x, h[0], acc[t][0]);
        acc[t][1] = mfma_f16(x, h[1], acc[t][1]);
      }
    });
    __builtin_amdgcn_sched_barrier(0);
    // the other buffer was last read one block ago (or, one block staged, ahead of the barrier between the halves)
    a_store(0, TWO ? ((kb & 1u) ^ 1u) * (2u * HALF) : 0u);
    if constexpr (LA) {
      lk[0][0] = B::template lookup<0>(cur[0], low);
      lk[0][1] = B::template lookup<0>(cur[1], low);
    }
    __syncthreads();
    if constexpr (!TWO) a_issue(0, next_k(ka));
  }

  pf_epilogue<GU, T, RT>(a, acc, base, cnt, q, row_of);
  // the next chunk: its first block is in `cur` and in LDS already
#pragma unroll
  for (int jt = 0; jt < RT; jt++) row_of[jt] += WAVES * RT * 16;
  }
}

// The blocks of 49 to 112 entries (T = 4 .. 7 token tiles, each with a body of its own: a test per tile and step splits
// the loop into blocks that nothing is scheduled across). The matrix cores' T instructions per fragment should hide the
// fourteen vector instructions of decoding; what keeps them at about half of that is three waves per SIMD in step:
//   * the activations are staged by halves of a block (the columns of steps 0-3 and 4-7), one buffer each: while a half is
//     multiplied the other one's buffer is refilled by loads that write LDS themselves, so the two barriers of a block stand
//     between steps and not around a copy;
//   * the fragments of step j + 1 are looked up at the start of step j and finished between its matrix instructions.
template <class B, bool GU, int T>
__device__ __forceinline__ void pf_big_body(const PfBlkArgs& a, PfUnit unit, bool first) {
  constexpr int WAVES = pf_blk_waves(kPfBigTiles), NT = 64 * WAVES;
  constexpr int NM = GU ? 2 : 1, RT = pf_blk_rt(GU, T), R = RT * NM;
  constexpr int HALF = pf_half_bytes(T), PLANE = HALF / 2;
  static_assert(R == 2 && T > 3 && T <= kPfBigTiles);
  extern __shared__ __attribute__((aligned(16))) uint32_t smem[];
  uint8_t* abuf = (uint8_t*)(smem + B::LDS_WORDS);  // [2 halves][2 planes][112 tokens][128 bytes]
  uint32_t tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // (as in pf_block_body)
  const uint32_t lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t n16 = lane & 15u, q = lane >> 4;
  const typename B::Low low = B::lane_low(n16);

  const uint32_t cnt = unit.cnt, base = unit.base, rc = unit.group;

  PfMatrix wm[NM];
  uint32_t row_of[RT];
#pragma unroll
  for (int m = 0; m < NM; m++) wm[m] = PfMatrix::of(a, unit.w[m]);
#pragma unroll
  for (int jt = 0; jt < RT; jt++) row_of[jt] = ((rc * WAVES + wave) * RT + jt) * 16u + n16;
  PfRows<B> rows;
  rows.init(a.row_bytes, lane);
  auto block_at = [&](int r, uint32_t off) { return wm[r % NM].mis + ((rc * WAVES + wave) * RT + r / NM) * 16u * a.row_bytes + off; };
  const typename B::At at_row = B::at_of(n16, q);
  typename B::Raw cur[R];
  uint8_t* const raw_lds = abuf + pf_act_lds_of_launch<B>(kPfBigTiles) + wave * (R * PfRows<B>::SLOT);
  auto request = [&](int r, uint32_t off) { rows.request(wm[r % NM], raw_lds + r * PfRows<B>::SLOT, block_at(r, off), lane); };
  auto fetched = [&](int r, uint32_t off) { return rows.fetched(at_row, raw_lds + r * PfRows<B>::SLOT, block_at(r, off)); };

  // activation loader: a half of a block is 4 T kilobytes, a load (eight rows of a plane) each; wave w's are w, w + 12, ...
  constexpr int AL = 4 * T, AMIN = AL / WAVES, AMAX = (AL + WAVES - 1) / WAVES;
  const rsrc_t ars = pf_act_rows<GU>(a, unit);
  uint32_t aoff[AMAX];
#pragma unroll
  for (int i = 0; i < AMAX; i++) {  // rows past the block's last entry repeat it (their products are never stored)
    const uint32_t l = wave + i * WAVES, plane = l >= 2u * T ? 1u : 0u, row = 8u * (l - plane * 2u * T) + (lane >> 3), unit = (lane & 7u) ^ ((row >> 1) & 7u);
    aoff[i] = pf_act_row<GU>(a, base, min(row, cnt - 1u)) * (a.K * 2u) + (64u * (2u * (unit >> 2) + plane) + 8u * (unit & 3u)) * 2u;
  }
  if constexpr (GU)
#pragma unroll
    for (int i = 0; i < AMAX; i++) asm volatile("" : "+v"(aoff[i]));  // (as in pf_block_body)
  const bool amore = wave + AMIN * WAVES < AL;  // (uniform) one load more than the waves that have the fewest
  auto a_request = [&](int h, uint32_t kc) {
#pragma unroll
    for (int i = 0; i < AMAX; i++)
      if (i < AMIN || amore) lds_dma16(ars, abuf + h * HALF + (wave + i * WAVES) * 1024u, aoff[i], kc * 512u + 64u * h);
  };
  constexpr int WLOADS = R * PfRows<B>::LOADS;
  // where the lane's fragments of step 0 start (tile t: 2048 bytes further; step j: the place's low bits the other way)
  uint32_t afrag = (uint32_t)(uintptr_t)(lds_cptr_t)abuf + (q & 1u) * PLANE + n16 * 128u + 16u * ((4u * (q >> 1)) ^ (n16 >> 1));

#pragma unroll
  for (int r = 0; r < R; r++) request(r, 0u);
  a_request(0, 0);
  if (first) B::fill_lds(smem, (int)tid, NT);
  wait_vm<0>();
#pragma unroll
  for (int r = 0; r < R; r++) cur[r] = fetched(r, 0u);
  __syncthreads();

  f4_t acc[T][R];
#pragma unroll
  for (int t = 0; t < T; t++)
#pragma unroll
    for (int r = 0; r < R; r++) acc[t][r] = f4_t{0.f, 0.f, 0.f, 0.f};
  uint32_t h[2][R][4], sc[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    sc[r] = B::scale(cur[r], 0);
    B::finish(sc[r], B::template lookup<0>(cur[r], low), h[0][r]);
  }
  // activation fragments are read AHEAD tiles before their use, across the ends of steps
  constexpr int AHEAD = 3, RING = 4;
  uint32_t af[RING][4];
  auto a_read = [&](int i) {  // i: step T + tile of the block
    const int j = i / T & 7, t = i % T;
    const u32x4 av = lds_at<u32x4>(afrag ^ (16u * (j & 3)), (j >> 2) * HALF + t * 2048);
#pragma unroll
    for (int k = 0; k < 4; k++) af[i % RING][k] = av[k];
  };
  // (8 T is a multiple of the ring's four places: a block's first tile is always in the same one)
#pragma unroll
  for (int i = 0; i < AHEAD; i++) a_read(i);

  for (uint32_t kc = 0; kc < a.nblocks; kc++) {
    const uint32_t kn = min(kc + 1u, a.nblocks - 1u), wn = kn * (uint32_t)B::BLOCK_BYTES;  // (the last block is fetched again)
    typename B::Look lk;
    afrag = opaque(afrag);  // (one register: the steps' places are not worth keeping)
    static_for<8 * T>([&](auto i_) __attribute__((always_inline)) {
      constexpr int i = i_, j = i / T, t = i % T, jn = (j + 1) & 7;
      // The order below is the order of issue (the scheduler would sink every read to its use)
      __builtin_amdgcn_sched_barrier(0);
      // Loads complete in order, and nothing but these is in flight, so a wait names the loads behind what it waits for.
      // Half 1 of this block, into the buffer that the block before has left; the next block's weight bytes (the slots are
      // read: the barrier has waited for that), a few at a time: all at once they queue up in the texture addresser.
      if constexpr (i == 0) a_request(1, kc);
      if constexpr (i == 1 || i == 3) request(i / 2, wn);
      // the last reads of a half are issued: what follows comes from the other buffer
      if constexpr (j == 3 && t == T - AHEAD) {
        wait_vm<WLOADS>();
        __syncthreads();
        a_request(0, kn);
      }
      if constexpr (j == 7 && t == 0) {  // the block's own bytes are used up
        if (amore) wait_vm<AMIN + 1>(); else wait_vm<AMIN>();
#pragma unroll
        for (int r = 0; r < R; r++) cur[r] = fetched(r, wn);
      }
      if constexpr (j == 7 && t == T - AHEAD) {
        wait_vm<0>();
        __syncthreads();
      }
      a_read(i + AHEAD);
      // the next step's fragments, one after the other
      if constexpr (t == 0) lk = B::template lookup<jn>(cur[0], low);
      if constexpr (t == T / 2) {
        if constexpr ((jn & 3) == 0) sc[0] = B::scale(cur[0], jn / 4);
        B::finish(sc[0], lk, h[jn & 1][0]);
        lk = B::template lookup<jn>(cur[1], low);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < R; r++) acc[t][r] = mfma_f16(af[i % RING], h[j & 1][r], acc[t][r]);
      if constexpr (t == T - 1) {
        __builtin_amdgcn_sched_barrier(0);
        if constexpr ((jn & 3) == 0) sc[1] = B::scale(cur[1], jn / 4);
        B::finish(sc[1], lk, h[jn & 1][1]);
      }
    });
  }
  pf_epilogue<GU, T, RT>(a, acc, base, cnt, q, row_of);
}

// Kernel variants: T = 3 takes the items of up to three token tiles in one launch, largest first (each runs the body
// built for its tile count; one launch has one tail of half-idle CUs); T = 7 the blocks of 49 to 112 entries that the
// popular experts are cut into (their weights are then decoded once per 112 entries; 12 waves, one activation buffer).
template <class B, bool GU, int T>
__device__ __forceinline__ void pf_unit(const PfBlkArgs& a, const PfUnit& unit, bool first) {
  const uint32_t cnt = unit.cnt;
  if constexpr (T > 3) {
    if (cnt > 96) pf_big_body<B, GU, 7>(a, unit, first);
    else if (cnt > 80) pf_big_body<B, GU, 6>(a, unit, first);
    else if (cnt > 64) pf_big_body<B, GU, 5>(a, unit, first);
    else pf_big_body<B, GU, 4>(a, unit, first);
  } else {
    if (cnt > 32) pf_block_body<B, GU, 3>(a, unit, first);
    else if (cnt > 16) pf_block_body<B, GU, 2>(a, unit, first);
    else pf_block_body<B, GU, 1>(a, unit, first);
  }
}
template <class B, bool GU, int T, bool QUEUE>
__global__ __launch_bounds__(64 * pf_blk_waves(T)) void moe_pf_block_kernel(const PfBlkArgs a) {
  uint32_t s = blockIdx.x >> 3;
  if constexpr (!QUEUE) {
    const PfUnit unit = PfUnit::of<GU>(a, s);
    if (unit.cnt) pf_unit<B, GU, T>(a, unit, true);
  } else {
    extern __shared__ __attribute__((aligned(16))) uint32_t smem[];
    uint32_t* const next_unit = smem + B::LDS_WORDS;  // (in the activation buffers, between two units)
    for (bool first = true; s < a.per_xcd;) {
      uint32_t next = 0;  // (asked for beside the item's words; a lane register held over the unit would be one too many)
      if (threadIdx.x == 0) next = atomicAdd(a.queue + (blockIdx.x & 7u), 1u);
      const PfUnit unit = PfUnit::of<GU>(a, s);
      next = (gridDim.x >> 3) + (uint32_t)__builtin_amdgcn_readfirstlane((int)next);
      if (unit.cnt) {
        pf_unit<B, GU, T>(a, unit, first);
        first = false;
      }
      wait_vm<0>();  // (requests past the unit's last block still write the buffers)
      __syncthreads();
      if (threadIdx.x == 0) *next_unit = next;
      __syncthreads();
      s = (uint32_t)__builtin_amdgcn_readfirstlane((int)*next_unit);
      __syncthreads();
    }
  }
}

// ------------------------------------------------------------------------------------------------ scratch header
// The header of the prefill scratch (expert addresses, the work items of the block GEMM) is built on the device. What only the
// host knows travels in kernel arguments: a raw image
//   word 0 n_exp | 1 has_shared | 2 n_tokens | 3 total | 4, 5 base address | 6 address mode | 7 unused
//   words 8 .. 8 + n_exp: entry offsets offs[0 .. n_exp]
//   then 3 addresses per expert (gate, up, down; the shared expert last): mode 0 one word each, (address - base) / 4;
//   mode 1 two words each
// cut into pieces of kHdrChunkWords (the argument block holds 4 KB). Every launch stores its piece behind the header;
// the last one then expands the image: addresses as the GEMM kernels read them, and the work items --
// an expert of m entries gives m / 112 blocks of 112 entries and one of m % 112 -- grouped by the token tiles a block
// fills, seven-tile blocks first, one-tile blocks last, inside a group in expert order (a counting sort over seven
// buckets: nothing in it depends on timing, so the table is the same on every run).
constexpr int kHdrChunkWords = 960, kHdrRawHead = 8, kHdrThreads = 1024;
constexpr uint32_t kPfCounters = 32;  // four launches of the routed experts' block GEMM (two projections, two sizes of items)
struct HdrChunk { uint32_t w[kHdrChunkWords]; };
struct HdrBuild {
  uint32_t* raw;        // the image, behind the header
  uint64_t* ptrs;       // (n_exp + 1) x {gate, up, down}
  uint32_t* items;      // routed items, then the shared expert's
  uint32_t build;       // 1: this launch holds the image's last piece and expands it
};
__host__ __device__ constexpr uint32_t pf_item_bucket(uint32_t cnt) { return 7u - (cnt + 15u) / 16u; }  // cnt in 1..112

// Where a thread's items of each of the seven buckets start: the buckets one behind the other, in each the threads' in order.
// All seven go through the two steps (inside a wave, over the waves) together: the kernel is one workgroup's chain of
// latencies, and a bucket at a time, three barriers and 16 serial additions each, took it 8.9 us (now 7.2; the 37 tokens of the performance cases).
struct HdrScan { uint32_t wave[kHdrThreads / 64][8], all[8]; };
__device__ __forceinline__ uint32_t hdr_scan(uint32_t (&v)[7], HdrScan& m, uint32_t tid) {
  const uint32_t lane = tid & 63u, wave = tid >> 6;
  uint32_t inc[7];
#pragma unroll
  for (int k = 0; k < 7; k++) {
    inc[k] = v[k];
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t t = (uint32_t)__shfl_up((int)inc[k], d, 64);
      if (lane >= (uint32_t)d) inc[k] += t;
    }
    if (lane == 63u) m.wave[wave][k] = inc[k];
  }
  __syncthreads();
  if (tid < 8u) {
    uint32_t run = 0;
#pragma unroll
    for (int w = 0; w < kHdrThreads / 64; w++) { const uint32_t t = tid < 7u ? m.wave[w][tid] : 0u; m.wave[w][tid] = run; run += t; }
    m.all[tid] = run;
  }
  __syncthreads();
  uint32_t first = 0;
#pragma unroll
  for (int k = 0; k < 7; k++) {
    v[k] = first + m.wave[wave][k] + inc[k] - v[k];
    first += m.all[k];
  }
  return first;  // all items
}

__global__ __launch_bounds__(kHdrThreads) void moe_pf_header_kernel(const HdrBuild b, const HdrChunk c, uint32_t word0, uint32_t nwords) {
  __shared__ HdrScan scan;
  __shared__ uint32_t whole[kHdrChunkWords];
  const uint32_t tid = threadIdx.x;
  // (an image of one piece stays in LDS: no trip to memory and back)
  uint32_t* const image = b.build && word0 == 0 ? whole : b.raw;
  for (uint32_t i = tid; i < nwords; i += kHdrThreads) image[word0 + i] = c.w[i];
  if (!b.build) return;
  __syncthreads();  // the image's earlier pieces were stored by earlier launches, the last one just now
  const uint32_t* raw = image;
  const uint32_t ne = raw[0], has_shared = raw[1], n = raw[2], total = raw[3], mode = raw[6];
  const uint64_t base = (uint64_t)raw[4] | ((uint64_t)raw[5] << 32);
  const uint32_t* roffs = raw + kHdrRawHead;
  const uint32_t* rp = roffs + ne + 1;
  for (uint32_t i = tid; i < 3u * (ne + has_shared); i += kHdrThreads)
    b.ptrs[i] = mode ? ((uint64_t)rp[2 * i] | ((uint64_t)rp[2 * i + 1] << 32)) : base + 4ull * rp[i];
  // routed items: this thread's experts [j0, j1)
  const uint32_t per = (ne + kHdrThreads - 1) / kHdrThreads, j0 = min(ne, tid * per), j1 = min(ne, j0 + per);
  uint32_t at[7] = {0, 0, 0, 0, 0, 0, 0};  // items of each bucket, then where they start
  for (uint32_t j = j0; j < j1; j++) {
    const uint32_t m = roffs[j + 1] - roffs[j], r = m % 112u;
    at[0] += m / 112u;
    if (r) {
      const uint32_t bk = pf_item_bucket(r);
#pragma unroll
      for (int k = 0; k < 7; k++) at[k] += bk == (uint32_t)k;
    }
  }
  const uint32_t first = hdr_scan(at, scan, tid);
  for (uint32_t j = j0; j < j1; j++) {
    const uint32_t m = roffs[j + 1] - roffs[j], q = m / 112u, r = m % 112u;
    for (uint32_t k = 0; k < q; k++) {
      uint32_t* it = b.items + 3 * (size_t)at[0]++;
      it[0] = j; it[1] = roffs[j] + 112u * k; it[2] = 112u;
    }
    if (r) {
      const uint32_t bk = pf_item_bucket(r);
      uint32_t pos = 0;
#pragma unroll
      for (int k = 0; k < 7; k++)
        if (bk == (uint32_t)k) pos = at[k]++;
      uint32_t* it = b.items + 3 * (size_t)pos;
      it[0] = j; it[1] = roffs[j] + 112u * q; it[2] = r;
    }
  }
  // the shared expert's items follow: blocks of 112 tokens, then the rest
  if (has_shared) {
    const uint32_t q = n / 112u, r = n % 112u;
    for (uint32_t k = tid; k < q + (r ? 1u : 0u); k += kHdrThreads) {
      uint32_t* it = b.items + 3 * (size_t)(first + k);
      it[0] = ne; it[1] = total + 112u * k; it[2] = k < q ? 112u : r;
    }
  }
}

// Xg[i] = fp16(X[src(i)]): i < total gathers token tok[i]; rows total .. total + n - 1 are the tokens themselves. One
// workgroup per row, eight elements (one 16-byte store) per thread and pass. The first workgroup also clears the block GEMM's
// counters (null: it has none).
template <bool X_BF16>
__global__ __launch_bounds__(256) void moe_pf_gather_kernel(const void* __restrict__ X, uint16_t* __restrict__ Xg,
                                                            const int* __restrict__ tok, uint32_t total, uint32_t nrows,
                                                            uint32_t dim, uint32_t* __restrict__ counters) {
  const uint32_t i = blockIdx.x;
  if (i >= nrows) return;
  if (counters && i == 0 && threadIdx.x < kPfCounters) counters[threadIdx.x] = 0u;
  const uint32_t src = i < total ? (uint32_t)tok[i] : i - total;
  auto f = [](uint32_t w) { return __builtin_bit_cast(float, w); };
  for (uint32_t c8 = threadIdx.x; c8 < dim / 8; c8 += blockDim.x) {
    u32x4 o;
    if constexpr (X_BF16) {
      const u32x4 b = ((const u32x4*)((const uint16_t*)X + (size_t)src * dim))[c8];
      o = u32x4{pack_h2(f(b.x << 16), f(b.x & 0xFFFF0000u)), pack_h2(f(b.y << 16), f(b.y & 0xFFFF0000u)),
                pack_h2(f(b.z << 16), f(b.z & 0xFFFF0000u)), pack_h2(f(b.w << 16), f(b.w & 0xFFFF0000u))};
    } else {
      const u32x4* p = (const u32x4*)((const float*)X + (size_t)src * dim) + 2 * (size_t)c8;
      const u32x4 lo = p[0], hi = p[1];
      o = u32x4{pack_h2(f(lo.x), f(lo.y)), pack_h2(f(lo.z), f(lo.w)), pack_h2(f(hi.x), f(hi.y)), pack_h2(f(hi.z), f(hi.w))};
    }
    ((u32x4*)(Xg + (size_t)i * dim))[c8] = o;
  }
}

// Y[t] += Z[total + t] (shared) + sum_k Z[slot_of[t][k]] in fixed k order; tokens without any entry are left alone
__global__ __launch_bounds__(256) void moe_pf_reduce_kernel(const float* __restrict__ Z, float* __restrict__ Y,
                                                            const int* __restrict__ slot_of, uint32_t n, uint32_t total,
                                                            uint32_t dim, uint32_t k_per_token, uint32_t has_shared) {
  const uint32_t t = blockIdx.y;
  if (t >= n) return;
  for (uint32_t c4 = blockIdx.x * blockDim.x + threadIdx.x; c4 < dim / 4; c4 += gridDim.x * blockDim.x) {
    float4 s = has_shared ? ((const float4*)(Z + (size_t)(total + t) * dim))[c4] : make_float4(0.f, 0.f, 0.f, 0.f);
    bool any = has_shared != 0;
    for (uint32_t k = 0; k < k_per_token; k++) {
      const int i = slot_of[t * k_per_token + k];
      if (i >= 0) {
        const float4 z = ((const float4*)(Z + (size_t)i * dim))[c4];
        s.x += z.x; s.y += z.y; s.z += z.z; s.w += z.w;
        any = true;
      }
    }
    if (!any) continue;
    float4* y = (float4*)(Y + (size_t)t * dim) + c4;
    float4 o = *y;
    o.x += s.x; o.y += s.y; o.z += s.z; o.w += s.w;
    *y = o;
  }
}

}  // namespace msq

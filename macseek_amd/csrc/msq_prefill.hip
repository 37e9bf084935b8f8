// C ABI: prefill MoE (see include/msq.h; reference host code src/kernels/quant.mm:372-612).
#include <algorithm>
#include <array>
#include <cstdlib>
#include <cstring>
#include <vector>

#include <mutex>

#include "msq_host.h"
#include "msq_prefill.cuh"
#include "msq_prefill_tile.cuh"

namespace msq {
namespace {

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }
// header: addresses | n_exp + 2 words that nothing uses (callers keep the scratch size) | work items | raw image (see moe_pf_header_kernel)
struct HdrLayout { size_t ptrs, items, raw, bytes; };
HdrLayout header_layout(int total, int n, int n_exp) {
  HdrLayout h;
  const size_t items = 2 * ((size_t)n_exp + 1) + (size_t)total / kPfBigTokens + (size_t)n / kPfBigTokens;  // m / 112 blocks + a rest per expert
  const size_t raw_words = kHdrRawHead + ((size_t)n_exp + 1) + 6 * ((size_t)n_exp + 1);
  h.ptrs = 0;
  h.items = 24 * (size_t)(n_exp + 1) + 4 * (size_t)(n_exp + 2);
  h.raw = h.items + 12 * items;
  h.bytes = align256(h.raw + 4 * raw_words);
  return h;
}
size_t header_bytes(int total, int n, int n_exp) { return header_layout(total, n, n_exp).bytes; }
bool routed_ok(int t) { return t == MSQ_IQ1_S || t == MSQ_IQ2_XXS; }
bool shared_ok(int t) { return t == MSQ_Q6_K || t == MSQ_Q8_0 || t == MSQ_IQ2_XXS || t == MSQ_IQ1_S; }

template <class D, bool GU>
int launch_tile_t(hipStream_t st, PfTileArgs a) {
  const size_t lds = 4 * (size_t)kPfTileBuf + 2 * (size_t)kPfTileRows * D::GROUPS * 4;
  const int rc = allow_large_lds(moe_pf_tile_kernel<D, GU>, lds);
  if (rc != MSQ_OK) return rc;
  a.row_chunks = a.N / (GU ? kPfTileRows / 2 : kPfTileRows);  // (N is a multiple of 256)
  a.token_blocks = (a.cnt + kPfTileTok - 1) / kPfTileTok;
  hipLaunchKernelGGL((moe_pf_tile_kernel<D, GU>), dim3(a.row_chunks * a.token_blocks), dim3(kPfTileThreads), lds, st, a);
  MSQ_HIP(hipGetLastError());
  return MSQ_OK;
}
template <bool GU>
int launch_tile(int t, hipStream_t st, const PfTileArgs& a) {
  return t == MSQ_Q6_K ? launch_tile_t<TileQ6K, GU>(st, a) : launch_tile_t<TileQ8_0, GU>(st, a);
}
template <class B, bool GU, int T, bool QUEUE>
int launch_block_q(hipStream_t st, uint32_t grid, const PfBlkArgs& a) {
  static bool attr_set = false;  // per instantiation: allow more than 64 KiB of dynamic LDS
  if (!attr_set) {
    MSQ_HIP(hipFuncSetAttribute((const void*)moe_pf_block_kernel<B, GU, T, QUEUE>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
    attr_set = true;
  }
  hipLaunchKernelGGL((moe_pf_block_kernel<B, GU, T, QUEUE>), dim3(grid), dim3(64 * pf_blk_waves(T)), pf_blk_lds<B>(T), st, a);
  MSQ_HIP(hipGetLastError());
  return MSQ_OK;
}
template <class B, bool GU, int T>
int launch_block_tt(hipStream_t st, PfBlkArgs a) {
  if (!a.nitems) return MSQ_OK;
  const uint32_t rows_per_item = pf_blk_rows(GU, T);
  a.row_chunks = (a.N + rows_per_item - 1) / rows_per_item;
  // two row chunks per workgroup while that leaves three workgroups and more per CU (MSQ_MOEP_CHUNKS imposes a count)
  static const int env_ch = [] { const char* e = getenv("MSQ_MOEP_CHUNKS"); return e && *e ? atoi(e) : 0; }();
  const uint32_t items8 = ((a.nitems + 7) / 8) * 8;
  uint32_t ch = env_ch > 0 ? (uint32_t)env_ch : ((size_t)items8 * ((a.row_chunks + 1) / 2) >= (size_t)3 * device_info().cus ? 2u : 1u);
  ch = std::max(1u, std::min(ch, a.row_chunks));
  if (a.N % rows_per_item || GU || T > 3) ch = 1;  // (a ragged last chunk clamps its rows: the chunks are then not a fixed stride apart)
  a.chunks_per_wg = ch;
  a.row_groups = (a.row_chunks + ch - 1) / ch;
  a.per_xcd = items8 / 8 * a.row_groups;
  // workgroups that stay (see PfUnit) once there are more units than the chip holds workgroups
  const uint32_t held = (uint32_t)device_info().cus / 8 * (160 * 1024 / (uint32_t)pf_blk_lds<B>(T));
  return a.queue && a.per_xcd > held ? launch_block_q<B, GU, T, true>(st, 8 * held, a) : launch_block_q<B, GU, T, false>(st, 8 * a.per_xcd, a);
}
// A second stream of the library's own, per device, and the two events that fork work onto it and join it back: the
// shared expert's two products run beside the routed experts', which they only meet in the reduction. With few tokens
// the shared expert has too few workgroups to fill the chip and its K loop is a chain of latencies (37 tokens, dim 5120:
// 115 us that are hidden, the call 774 -> 659 us); with many it changes nothing. (The popular experts' blocks and the small
// items stay on one stream: each takes a whole CU's LDS, side by side they measured 2.73 ms against 2.70 in turn.)
// Fork and join are event dependencies, so a stream capture records them like any other (the objects are created
// outside of captures: by msq_init() or by the first call that is not being captured; until then calls stay on one stream).
struct SideStream { hipStream_t stream = nullptr; hipEvent_t fork = nullptr, join = nullptr; bool ok = false; };
std::mutex g_side_mu;
SideStream g_side[16];
// The device's side stream, or null when this call has to stay on the caller's stream: the fork is switched off, the
// objects do not exist yet and `st` is being captured, or the side stream still belongs to a stream capture that `st`
// is not part of (work forked from a capturing stream pulls the side stream into that capture until the capture ends;
// an eager call, or a call under another capture, must not enqueue into it). Call with g_side_mu held.
SideStream* side_stream(hipStream_t st) {
  static const bool off = [] { const char* e = getenv("MSQ_MOEP_ONE_STREAM"); return e && *e && atoi(e) != 0; }();
  int dev = 0;
  if (off || hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return nullptr;
  SideStream& s = g_side[dev];
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  unsigned long long cid = 0;
  if (st && hipStreamGetCaptureInfo(st, &cs, &cid) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
  if (!s.ok) {
    if (cs != hipStreamCaptureStatusNone) return nullptr;
    if (hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&s.fork, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&s.join, hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
    s.ok = true;
  }
  hipStreamCaptureStatus ss = hipStreamCaptureStatusNone;
  unsigned long long sid = 0;
  if (hipStreamGetCaptureInfo(s.stream, &ss, &sid) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
  if (ss != hipStreamCaptureStatusNone && !(cs == hipStreamCaptureStatusActive && ss == hipStreamCaptureStatusActive && cid == sid))
    return nullptr;
  return &s;
}

// items are sorted by size, largest first: n6 blocks of more than 48 entries, n3 items of three token tiles, n2 of two,
// then the one-tile items: the blocks in one launch, everything up to three tiles in another (one tail of half-idle CUs
// instead of two); skip: profiling mask (see msq_moe_prefill)
template <class BIG, class B, bool GU>
int launch_block_t(hipStream_t st, PfBlkArgs a, uint32_t n6, uint32_t n3, uint32_t n2, int skip) {
  const uint32_t* items = a.items;
  const uint32_t n = a.nitems;
  int rc;
  uint32_t* const queue = a.queue;
  a.items = items; a.nitems = n6;
  if (!(skip & 256) && (rc = launch_block_tt<BIG, GU, kPfBigTiles>(st, a))) return rc;
  const uint32_t lo = (skip & 128) ? n6 + n3 + n2 : n6, hi = (skip & 64) ? n6 + n3 + n2 : n;
  a.items = items + 3 * (size_t)lo; a.nitems = hi > lo ? hi - lo : 0u;
  a.queue = queue ? queue + 8 : nullptr;
  return launch_block_tt<B, GU, 3>(st, a);
}
// With the shared expert's products on the side stream, workgroups that stay pay from this many tokens on. They leave no room
// for the shared expert's second product until the routed experts' first has ended, which costs while the shared expert's chain
// is as long as theirs. Time of a workgroup per unit over workgroups that stay, one stream:
// 0.98 to 1.10 (mean 1.02) at any number of tokens. Two streams, 104 calls of all types, 128 and 384 experts, back to back
// (in brackets each alone): 7 to 60 tokens 0.88 to 1.05 (0.90 to 1.17), 100 and 140 0.96 to 1.10 (1.01 to 1.13), 178 to 212 0.99 to
// 1.11 (1.01 to 1.11), 224 to 420 0.98 to 1.10 (1.01 to 1.10). Where the loss ends lies between 100 and 178 tokens and differs from
// layer to layer; the line is drawn above all of it.
constexpr int kPfQueueTokens = 2 * kPfBigTokens;
// The shared expert of a K-quant / Q8_0 type through the few-token kernel (msq_rows.cuh), on the caller's stream? The tile kernel's 128 x 128
// tiles are a chain of 150 us however few the tokens, and the fork to a second stream costs 14 us by itself; but they run beside the routed
// experts, and the few-token kernel's launches (36 us at 37 tokens) come behind them. Time before / after, Q6_K and Q8_0 alike, 384 IQ1_S
// experts: 5120x2304 at 2 tokens 186 / 119, 16 307 / 280, 37 517 / 502, 64 650 / 606, 100 761 / 761, 150 (the tile kernel ahead) 992 / 978;
// Q6_K 7168x2048 at 64 703 / 694, 100 918 / 889, 150 1171 / 1190 (Q8_0 of 7168 columns does not fit the LDS); 2560x1024 at 100 252 / 229, 150
// 347 / 338. 94 to 242 experts in use 0.98 to 1.3 times the former speed at 37 to 112 tokens. Fewer of them leave compute units to the tile
// kernel: 49 to 64 in use 1.02 to 1.5 at up to 48 tokens and, as long as no expert has more than 48 entries (the routed experts are one
// launch then), 1.02 to 1.46 up to 112 (in a graph, where the fork is cheaper, 0.92 to 1.25); with such an expert, 9 to 64 in use, 0.86 to
// 0.98 at 64 to 112 tokens of 5120x2304 and 4096x1536 (7168x2048 0.87 to 1.08, 2560x1024 0.98 to 1.08): the tile kernel has these.
bool shared_few(int n, int used, bool crowded) { return n <= 112 && (!crowded || used >= 94); }
bool block_path(int t) { return t == MSQ_IQ1_S || t == MSQ_IQ2_XXS; }
template <bool GU>
int launch_block(int t, hipStream_t st, const PfBlkArgs& a, uint32_t n6, uint32_t n3, uint32_t n2, int skip) {
  return t == MSQ_IQ1_S ? launch_block_t<BlkIQ1S, BlkIQ1S, GU>(st, a, n6, n3, n2, skip)
                        : launch_block_t<BlkIQ2XXS<4>, BlkIQ2XXS<16>, GU>(st, a, n6, n3, n2, skip);
}

}  // namespace

void prefill_side_stream_setup() {
  std::lock_guard<std::mutex> lock(g_side_mu);
  (void)side_stream(nullptr);
}

}  // namespace msq

using namespace msq;

extern "C" {

size_t msq_moe_prefill_scratch_bytes(int total, int n, int n_exp, int dim, int inter) {
  if (dim <= 0) dim = MSQ_EXPERT_DIM;
  if (inter <= 0) inter = MSQ_EXPERT_INTER;
  const size_t rows = (size_t)std::max(total, 0) + (size_t)std::max(n, 0);
  return header_bytes(std::max(total, 0), std::max(n, 0), std::max(n_exp, 0)) + align256(rows * dim * 2) +
         align256(rows * inter * 2) + align256(rows * dim * 4);
}

// whether a shared expert goes to the few-token kernel, without the LDS it needs (for tests)
int msq_test_prefill_shared_few(int n, int used, int crowded) { return shared_few(n, used, crowded != 0) ? 1 : 0; }

int msq_moe_prefill(void* stream, const MsqMoePrefillArgs* p) {
  if (!p) return fail(MSQ_ERR_ARGUMENT, "macseek quant: moe_prefill: null arguments");
  const int n = p->n_tokens, ne = p->n_exp;
  if (n <= 0) return MSQ_OK;
  const int dim = p->dim ? p->dim : MSQ_EXPERT_DIM, inter = p->inter ? p->inter : MSQ_EXPERT_INTER;
  if (ne < 0 || (ne > 0 && (!p->slots || !p->offs))) return fail(MSQ_ERR_ARGUMENT, "macseek quant: moe_prefill: slots / offs missing");
  const int total = ne > 0 ? p->offs[ne] : 0;
  if (!routed_ok(p->t_gate_up) || !routed_ok(p->t_down) || (p->has_shared && !shared_ok(p->t_shared)))
    return unsupported("moe_prefill types", p->t_gate_up, 0, 0);
  if (dim < 256 || inter < 256 || dim % 256 || inter % 256 || dim > 8192 || inter > 8192)
    return unsupported("moe_prefill expert shape", p->t_gate_up, inter, dim);
  if (total < 0 || p->k_per_token < 0) return fail(MSQ_ERR_ARGUMENT, "macseek quant: moe_prefill: negative counts");
  for (int j = 0; j < ne; j++)
    if (p->offs[j + 1] < p->offs[j] || p->offs[0] != 0) return fail(MSQ_ERR_ARGUMENT, "macseek quant: moe_prefill: offs not ascending from 0");
  if (!buf_ok(&p->scratch, msq_moe_prefill_scratch_bytes(total, n, ne, dim, inter)))
    return fail(MSQ_ERR_SCRATCH, "macseek quant: moe_prefill scratch too small unsupported (type %s rows %d cols %d)",
                msq_type_name_of(p->t_gate_up), total, n);
  const size_t xbytes = (size_t)n * dim * (p->x_is_bf16 ? 2 : 4);
  if (!buf_ok(&p->X, xbytes) || !buf_ok(&p->Y, (size_t)n * dim * 4))
    return fail(MSQ_ERR_ARGUMENT, "macseek quant: moe_prefill: X / Y missing or too small");
  if (((uintptr_t)bptr(&p->X) & 15) || ((uintptr_t)bptr(&p->Y) & 15) || ((uintptr_t)bptr(&p->scratch) & 255))
    return fail(MSQ_ERR_ARGUMENT, "macseek quant: moe_prefill: X / Y not 16-byte aligned or scratch not 256-byte aligned");
  if (total > 0 && (!buf_ok(&p->tok, (size_t)total * 4) || !buf_ok(&p->wt, (size_t)total * 4)))
    return fail(MSQ_ERR_ARGUMENT, "macseek quant: moe_prefill: tok / wt missing or too small");
  if (p->k_per_token > 0 && !buf_ok(&p->slot_of, (size_t)n * p->k_per_token * 4))
    return fail(MSQ_ERR_ARGUMENT, "macseek quant: moe_prefill: slot_of missing or too small");
  const size_t rb_gu = msq_type_row_bytes(p->t_gate_up, dim), rb_d = msq_type_row_bytes(p->t_down, inter);
  const size_t rb_sgu = msq_type_row_bytes(p->t_shared, dim), rb_sd = msq_type_row_bytes(p->t_shared, inter);
  for (int j = 0; j < ne; j++) {
    const MsqExpertSlot& s = p->slots[j];
    if (!buf_ok(&s.gate, rb_gu * inter) || !buf_ok(&s.up, rb_gu * inter) || !buf_ok(&s.down, rb_d * dim))
      return fail(MSQ_ERR_ARGUMENT, "macseek quant: moe_prefill: expert slot %d missing or too small", j);
  }
  if (p->has_shared && (!buf_ok(&p->shared.gate, rb_sgu * inter) || !buf_ok(&p->shared.up, rb_sgu * inter) ||
                        !buf_ok(&p->shared.down, rb_sd * dim)))
    return fail(MSQ_ERR_ARGUMENT, "macseek quant: moe_prefill: shared expert missing or too small");

  hipStream_t st = (hipStream_t)stream;
  // PROFILING ONLY (wrong output): MSQ_MOEP_SKIP bit mask 1 gather, 2 routed gate/up, 4 shared gate/up, 8 routed down,
  // 16 shared down, 32 reduce; of the block GEMMs' work 64 the one-tile items, 128 the two- and three-tile
  // items, 256 the blocks of the popular experts -- read on every call (reference: MACSEEK_MOEP_SKIP,
  // src/kernels/quant.mm:520-522)
  const char* skip_env = getenv("MSQ_MOEP_SKIP");
  const int skip = skip_env && *skip_env ? atoi(skip_env) : 0;
  // ---- header. The host only counts the work items per class (the launches' grids); the tables themselves are built
  // on the device from a raw image that travels in kernel arguments (moe_pf_header_kernel): nothing is read from host
  // memory after this call returns, the call never waits for the stream, and a stream capture records the values.
  const HdrLayout hl = header_layout(total, n, ne);
  uint32_t ni_routed = 0, ni_shared = 0;
  uint32_t nc_routed[3] = {0, 0, 0}, nc_shared[3] = {0, 0, 0};  // items of more than 48 entries / three tiles / two tiles
  auto count = [](int m, uint32_t& ni, uint32_t* nc) {  // an expert of m entries: m / 112 blocks of 112 and one of m % 112
    const uint32_t q = (uint32_t)(m / kPfBigTokens), r = (uint32_t)(m % kPfBigTokens);
    ni += q + (r ? 1u : 0u);
    nc[0] += q + (r > 48 ? 1u : 0u); nc[1] += r > 32 && r <= 48; nc[2] += r > 16 && r <= 32;
  };
  int used = 0;  // experts with entries
  for (int j = 0; j < ne; j++) {
    count(p->offs[j + 1] - p->offs[j], ni_routed, nc_routed);
    used += p->offs[j + 1] > p->offs[j];
  }
  if (p->has_shared) count(n, ni_shared, nc_shared);
  uint8_t* sc = bptr_mut(&p->scratch);
  // the block GEMM's counters take the place of the raw image, which is used up by then (a header of one or two experts may be too short)
  uint32_t* const counters = hl.bytes - hl.raw >= 4 * kPfCounters ? (uint32_t*)(sc + hl.raw) : nullptr;
  {
    const int nptr = 3 * (ne + (p->has_shared ? 1 : 0));
    std::vector<uint64_t> ptrs((size_t)nptr);
    for (int j = 0; j < ne; j++) {
      ptrs[3 * j] = (uint64_t)(uintptr_t)bptr(&p->slots[j].gate);
      ptrs[3 * j + 1] = (uint64_t)(uintptr_t)bptr(&p->slots[j].up);
      ptrs[3 * j + 2] = (uint64_t)(uintptr_t)bptr(&p->slots[j].down);
    }
    if (p->has_shared) {
      ptrs[3 * ne] = (uint64_t)(uintptr_t)bptr(&p->shared.gate);
      ptrs[3 * ne + 1] = (uint64_t)(uintptr_t)bptr(&p->shared.up);
      ptrs[3 * ne + 2] = (uint64_t)(uintptr_t)bptr(&p->shared.down);
    }
    // addresses as one word each, (address - lowest address) / 4, when they all lie within 16 GiB of the lowest and
    // are 4 bytes apart (expert matrices are 4-byte aligned); else in full
    uint64_t base = nptr ? *std::min_element(ptrs.begin(), ptrs.end()) : 0;
    bool rel = true;
    for (uint64_t v : ptrs) rel = rel && !((v - base) & 3) && ((v - base) >> 2) <= 0xFFFFFFFFull;
    std::vector<uint32_t> raw;
    raw.reserve(kHdrRawHead + (size_t)ne + 1 + (rel ? 1 : 2) * (size_t)nptr);
    raw.insert(raw.end(), {(uint32_t)ne, p->has_shared ? 1u : 0u, (uint32_t)n, (uint32_t)total, (uint32_t)base, (uint32_t)(base >> 32),
                           rel ? 0u : 1u, 0u});
    for (int j = 0; j < ne; j++) raw.push_back((uint32_t)p->offs[j]);
    raw.push_back((uint32_t)total);
    for (uint64_t v : ptrs) {
      if (rel) raw.push_back((uint32_t)((v - base) >> 2));
      else { raw.push_back((uint32_t)v); raw.push_back((uint32_t)(v >> 32)); }
    }
    HdrBuild hb{};
    hb.raw = (uint32_t*)(sc + hl.raw); hb.ptrs = (uint64_t*)(sc + hl.ptrs);
    hb.items = (uint32_t*)(sc + hl.items);
    for (size_t w0 = 0; w0 < raw.size(); w0 += kHdrChunkWords) {
      HdrChunk c;
      const uint32_t nw = (uint32_t)std::min<size_t>(kHdrChunkWords, raw.size() - w0);
      memcpy(c.w, raw.data() + w0, 4 * (size_t)nw);
      hb.build = w0 + nw == raw.size() ? 1u : 0u;
      hipLaunchKernelGGL(moe_pf_header_kernel, dim3(1), dim3(kHdrThreads), 0, st, hb, c, (uint32_t)w0, nw);
    }
    MSQ_HIP(hipGetLastError());
  }
  const size_t hbytes = hl.bytes;
  const size_t rows = (size_t)total + n;
  uint16_t* Xg = (uint16_t*)(sc + hbytes);
  uint16_t* H = (uint16_t*)((uint8_t*)Xg + align256(rows * dim * 2));
  float* Z = (float*)((uint8_t*)H + align256(rows * inter * 2));
  const uint64_t* d_ptrs = (const uint64_t*)(sc + hl.ptrs);
  const uint32_t* d_items = (const uint32_t*)(sc + hl.items);
  const bool any_routed = total > 0;

  // 1) gather + convert
  // The block GEMM finds an entry's row by its token, and only the tokens' own rows are converted, where these are wanted anyway
  // (shared expert) or no more than the entries, and within what one descriptor reaches; else the entries' rows are gathered.
  const bool by_token = any_routed && (p->has_shared || n <= total) && (size_t)n * dim * 2 < 0xFFFFFFF0ull;
  const uint32_t gathered = by_token ? 0u : (uint32_t)total, grows = gathered + (uint32_t)(p->has_shared || by_token ? n : 0);
  uint16_t* const Xt = Xg + (size_t)total * dim;  // the tokens' own rows
  const int* tok = any_routed ? (const int*)bptr(&p->tok) : nullptr;
  if (grows > 0) {
    const dim3 grid(skip & 1 ? 1u : grows), block(256);  // (skipped: one row is left, with the counters)
    uint16_t* to = gathered ? Xg : Xt;
    if (p->x_is_bf16) hipLaunchKernelGGL((moe_pf_gather_kernel<true>), grid, block, 0, st, (const void*)bptr(&p->X), to, tok, gathered, grows, (uint32_t)dim, counters);
    else hipLaunchKernelGGL((moe_pf_gather_kernel<false>), grid, block, 0, st, (const void*)bptr(&p->X), to, tok, gathered, grows, (uint32_t)dim, counters);
    MSQ_HIP(hipGetLastError());
  }
  PfBlkArgs b{};
  b.H = H; b.Z = Z; b.wt = total > 0 ? (const float*)bptr(&p->wt) : nullptr;
  b.ptrs = d_ptrs; b.total = (uint32_t)total;
  // one product over the routed experts' items
  bool forked = false;
  auto routed = [&](auto gu_tag, hipStream_t gs) -> int {
    constexpr bool GU = decltype(gu_tag)::value;
    b.A = !GU ? H : by_token ? Xt : Xg; b.tok = GU && by_token ? tok : nullptr; b.a_bytes = (uint32_t)((size_t)n * dim * 2);
    b.K = (uint32_t)(GU ? dim : inter); b.N = (uint32_t)(GU ? inter : dim);
    b.nblocks = b.K / 256; b.row_bytes = (uint32_t)(GU ? rb_gu : rb_d);
    b.items = d_items; b.nitems = ni_routed;
    b.queue = counters && (!forked || n >= kPfQueueTokens) ? counters + (GU ? 0 : 16) : nullptr;
    return launch_block<GU>(GU ? p->t_gate_up : p->t_down, gs, b, nc_routed[0], nc_routed[1], nc_routed[2], skip);
  };
  // ... and one over all tokens with the shared expert's weights
  const bool few = p->has_shared && shared_few(n, used, nc_routed[0] > 0) && shared_rows_serves(p->t_shared, dim, inter);
  auto shared = [&](auto gu_tag, hipStream_t gs) -> int {
    constexpr bool GU = decltype(gu_tag)::value;
    const uint32_t K = (uint32_t)(GU ? dim : inter), N = (uint32_t)(GU ? inter : dim), rb = (uint32_t)(GU ? rb_sgu : rb_sd);
    if (block_path(p->t_shared)) {
      b.A = GU ? Xg : H; b.tok = nullptr; b.K = K; b.N = N; b.nblocks = K / 256; b.row_bytes = rb;
      b.items = d_items + 3 * (size_t)ni_routed; b.nitems = ni_shared; b.queue = nullptr;
      return launch_block<GU>(p->t_shared, gs, b, nc_shared[0], nc_shared[1], nc_shared[2], skip);
    }
    if (few)
      return GU ? shared_rows(gs, p->t_shared, bptr(&p->shared.gate), bptr(&p->shared.up), inter, dim, Xt, H + (size_t)total * inter, nullptr, n)
                : shared_rows(gs, p->t_shared, bptr(&p->shared.down), nullptr, dim, inter, H + (size_t)total * inter, nullptr, Z + (size_t)total * dim, n);
    PfTileArgs t{};
    t.A = (GU ? Xg : H) + (size_t)total * K;
    t.H = H + (size_t)total * inter; t.Z = Z + (size_t)total * dim;
    t.W[0] = bptr(GU ? &p->shared.gate : &p->shared.down); t.W[1] = GU ? bptr(&p->shared.up) : nullptr;
    t.cnt = (uint32_t)n; t.K = K; t.N = N; t.row_bytes = rb;
    return launch_tile<GU>(p->t_shared, gs, t);
  };
  int rc = MSQ_OK;
  using GuT = std::true_type; using DnT = std::false_type;
  const bool routed_gu = any_routed && !(skip & 2), routed_dn = any_routed && !(skip & 8);
  const bool shared_gu = p->has_shared && !(skip & 4), shared_dn = p->has_shared && !(skip & 16);
  // The shared expert and the routed experts only meet in the reduction: two pipelines on two streams (see SideStream)
  if (p->has_shared && any_routed && !few) {
    std::lock_guard<std::mutex> lock(g_side_mu);
    SideStream* s = side_stream(st);
    if (s && hipEventRecord(s->fork, st) == hipSuccess && hipStreamWaitEvent(s->stream, s->fork, 0) == hipSuccess) {
      forked = true;
      if (shared_gu) rc = shared(GuT{}, s->stream);
      if (rc == MSQ_OK && shared_dn) rc = shared(DnT{}, s->stream);
      const hipError_t ej = hipEventRecord(s->join, s->stream);
      if (rc == MSQ_OK && routed_gu) rc = routed(GuT{}, st);
      if (rc == MSQ_OK && routed_dn) rc = routed(DnT{}, st);
      // whatever happened above, the side stream is joined back: a caller's capture is never left with an unjoined stream
      const hipError_t ew = ej == hipSuccess ? hipStreamWaitEvent(st, s->join, 0) : ej;
      if (rc == MSQ_OK && ew != hipSuccess) rc = hip_fail(ew, "joining the side stream");
      if (rc != MSQ_OK) return rc;
    } else {
      (void)hipGetLastError();
    }
  }
  if (!forked) {
    // 2) gate + up + SwiGLU -> H
    if (routed_gu && (rc = routed(GuT{}, st))) return rc;
    if (shared_gu && (rc = shared(GuT{}, st))) return rc;
    // 3) down -> Z
    if (routed_dn && (rc = routed(DnT{}, st))) return rc;
    if (shared_dn && (rc = shared(DnT{}, st))) return rc;
  }
  // 4) ordered reduction into Y
  if ((any_routed || p->has_shared) && !(skip & 32)) {
    const dim3 grid((dim / 4 + 255) / 256, (unsigned)n), block(256);
    hipLaunchKernelGGL(moe_pf_reduce_kernel, grid, block, 0, st, (const float*)Z, (float*)bptr_mut(&p->Y),
                       p->k_per_token > 0 ? (const int*)bptr(&p->slot_of) : nullptr, (uint32_t)n, (uint32_t)total, (uint32_t)dim,
                       (uint32_t)(any_routed ? p->k_per_token : 0), (uint32_t)(p->has_shared ? 1 : 0));
    MSQ_HIP(hipGetLastError());
  }
  return MSQ_OK;
}

}  // extern "C"

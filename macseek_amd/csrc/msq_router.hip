// C ABI: MoE router (top-6 selection) and the expert-sorted routing lists the prefill grouped GEMM consumes
// (see include/msq.h; reference host code src/kernels/arch.hpp:79-97, kernels src/kernels/arch_router.metal:26-183,
// CPU twin tests/ref/arch_ref.cpp:97-130).
//
// score = sqrt(softplus(logit)), key = score + bias, the six experts with the largest keys (ties: lowest id), weight =
// score / (sum of the six scores + 1e-20) * route_scale. The scores are computed in double precision and rounded where
// the reference's CPU twin rounds (fp64 runs at a quarter of the fp32 rate on this device and a token has 384 experts),
// so expert ids and weights repeat that twin's bits rather than being close to them.
#include <algorithm>

#include "msq_device.cuh"
#include "msq_host.h"

namespace msq {
namespace {

constexpr int kTopK = MSQ_MAX_ROUTED;
constexpr int kMaxEpl = 8;  // experts per lane: n_exp <= 512

// Wave-wide maximum / minimum, returned in every lane: the DPP steps of wave_sum with the lane's own value standing in
// where a step has no source lane.
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ float dpp_fmax(float v) {
  const int b = __builtin_bit_cast(int, v);
  return fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(b, b, CTRL, ROW_MASK, 0xF, false)));
}
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ int dpp_imin(int v) {
  return min(v, __builtin_amdgcn_update_dpp(v, v, CTRL, ROW_MASK, 0xF, false));
}
__device__ __forceinline__ float wave_max_f(float v) {
  v = dpp_fmax<0xB1>(v); v = dpp_fmax<0x4E>(v); v = dpp_fmax<0x141>(v); v = dpp_fmax<0x140>(v);
  v = dpp_fmax<0x142, 0xA>(v); v = dpp_fmax<0x143, 0xC>(v);
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
__device__ __forceinline__ int wave_min_i(int v) {
  v = dpp_imin<0xB1>(v); v = dpp_imin<0x4E>(v); v = dpp_imin<0x141>(v); v = dpp_imin<0x140>(v);
  v = dpp_imin<0x142, 0xA>(v); v = dpp_imin<0x143, 0xC>(v);
  return __builtin_amdgcn_readlane(v, 63);
}

// score and key of one expert, rounded where the reference's CPU twin rounds (tests/ref/arch_ref.cpp:100-105)
__device__ __forceinline__ void score_key(float logit, float bias, double& sc, float& key) {
  const double x = (double)logit;
  const double sp = x > 20.0 ? x : log1p(exp(x));
  sc = sqrt(sp);
  key = (float)sc + bias;
}

// One wave selects the top six experts of one token from the keys and scores its lanes hold (lane l: experts l + 64 i)
// and writes ids / weights.
__device__ __forceinline__ void select6(float (&key)[kMaxEpl], const double (&sc)[kMaxEpl], uint32_t epl, float route_scale,
                                        uint32_t lane, int* __restrict__ ids, float* __restrict__ wts) {
  int sel_e[kTopK];
  double sel_s[kTopK];
  double sum = 0.0;  // the six scores are added in selection order, as the reference adds them
#pragma unroll
  for (int k = 0; k < kTopK; k++) {
    float bk = -INFINITY;
    double bs = 0.0;
    int be = 0x7fffffff;
#pragma unroll
    for (uint32_t i = 0; i < kMaxEpl; i++)  // ascending expert id, strict comparison: the lane's lowest id among equals
      if (i < epl && key[i] > bk) { bk = key[i]; bs = sc[i]; be = (int)(lane + 64u * i); }
    const float m = wave_max_f(bk);
    const int win = wave_min_i(bk == m ? be : 0x7fffffff);
    if (win == 0x7fffffff) {  // fewer than six comparable keys (NaN logits): expert 0 with weight 0
      sel_e[k] = 0;
      sel_s[k] = 0.0;
      continue;
    }
#pragma unroll
    for (uint32_t i = 0; i < kMaxEpl; i++)
      if ((int)(lane + 64u * i) == win) key[i] = -INFINITY;
    const int src = __builtin_amdgcn_readfirstlane(win) & 63;  // the winner's lane holds its score in bs
    const uint64_t bits = __builtin_bit_cast(uint64_t, bs);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)bits, src);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(bits >> 32), src);
    sel_e[k] = win;
    sel_s[k] = __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
    sum += sel_s[k];
  }
  if (lane < (uint32_t)kTopK) {
#pragma unroll
    for (int k = 0; k < kTopK; k++)
      if (lane == (uint32_t)k) { ids[k] = sel_e[k]; wts[k] = (float)(sel_s[k] / (sum + 1e-20) * (double)route_scale); }
  }
}

// A workgroup of `waves` waves, up to eight, selects the top six of one token, one expert a thread (key -inf: none, or not comparable) and writes ids
// and weights; after(): by one thread, behind the barrier.
// Selection in two levels: each wave picks the six best of its 64 experts, one a lane, and leaves them in LDS; wave 0 picks
// the six best of those 48. The six best overall are among the six best of their waves, and "greater key, then lower expert
// id" is a total order: experts, and the candidates that a wave leaves, stand in the lanes in the order of their ids where keys
// are equal, so the first lane with the greatest key is the choice. NaN and -inf are never chosen.
template <class After>
__device__ __forceinline__ void select6_of_block(float key, double sc, uint32_t tid, uint32_t waves, float route_scale, int* __restrict__ ids,
                                               float* __restrict__ wts, After after) {
  constexpr uint32_t WAVES = 8;
  __shared__ float c_key[WAVES * kTopK];
  __shared__ int c_id[WAVES * kTopK];
  __shared__ double c_sc[WAVES * kTopK];
  const uint32_t lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
#pragma unroll
  for (int k = 0; k < kTopK; k++) {
    const float m = wave_max_f(key);
    const uint64_t best = __builtin_amdgcn_ballot_w64(key == m && m > -INFINITY);
    const bool won = best ? (uint32_t)__builtin_ctzll(best) == lane : lane == 0;
    if (won) {
      c_key[wave * kTopK + k] = m;
      c_id[wave * kTopK + k] = (int)tid;
      c_sc[wave * kTopK + k] = sc;
      key = -INFINITY;
    }
  }
  __syncthreads();
  if (wave != 0) return;
  if (lane == 0) after();
  const uint32_t candidates = waves * kTopK;
  float ck = lane < candidates ? c_key[lane] : -INFINITY;
  const int ce = lane < candidates ? c_id[lane] : 0;
  const uint64_t cs = lane < candidates ? __builtin_bit_cast(uint64_t, c_sc[lane]) : 0;
  int sel_e[kTopK];
  double sel_s[kTopK];
  double sum = 0.0;  // the six scores are added in selection order, as the reference adds them
#pragma unroll
  for (int k = 0; k < kTopK; k++) {
    const float m = wave_max_f(ck);
    const uint64_t best = __builtin_amdgcn_ballot_w64(ck == m && m > -INFINITY);
    if (!best) {  // fewer than six comparable keys (NaN logits): expert 0 with weight 0
      sel_e[k] = 0;
      sel_s[k] = 0.0;
      continue;
    }
    const int src = (int)__builtin_ctzll(best);
    if (lane == (uint32_t)src) ck = -INFINITY;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)cs, src);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(cs >> 32), src);
    sel_e[k] = __builtin_amdgcn_readlane(ce, src);
    sel_s[k] = __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
    sum += sel_s[k];
  }
  if (lane < (uint32_t)kTopK) {
#pragma unroll
    for (int k = 0; k < kTopK; k++)
      if (lane == (uint32_t)k) { ids[k] = sel_e[k]; wts[k] = (float)(sel_s[k] / (sum + 1e-20) * (double)route_scale); }
  }
}

// logits [n][n_exp] -> ids [n][6], weights [n][6]; one wave per token, four per workgroup.
__global__ __launch_bounds__(256) void router_topk_kernel(const float* __restrict__ logits, const float* __restrict__ bias,
                                                          int* __restrict__ ids, float* __restrict__ wts, uint32_t n_tokens,
                                                          uint32_t n_exp, float route_scale) {
  const uint32_t lane = threadIdx.x & 63u, t = blockIdx.x * 4u + (threadIdx.x >> 6);
  if (t >= n_tokens) return;  // whole waves leave; no barrier follows
  const float* row = logits + (size_t)t * n_exp;
  const uint32_t epl = n_exp >> 6;
  double sc[kMaxEpl];
  float key[kMaxEpl];
#pragma unroll
  for (uint32_t i = 0; i < kMaxEpl; i++) {
    sc[i] = 0.0;
    key[i] = -INFINITY;
    if (i < epl) score_key(row[lane + 64u * i], bias[lane + 64u * i], sc[i], key[i]);
  }
  select6(key, sc, epl, route_scale, lane, ids + (size_t)t * kTopK, wts + (size_t)t * kTopK);
}

// The same, a workgroup per token and an expert a thread: the double-precision chain of one expert instead of up to eight.
__global__ __launch_bounds__(512) void router_topk_wide_kernel(const float* __restrict__ logits, const float* __restrict__ bias, int* __restrict__ ids,
                                                               float* __restrict__ wts, uint32_t n_exp, float route_scale) {
  const uint32_t tid = threadIdx.x, t = blockIdx.x;
  float key = -INFINITY;
  double sc = 0.0;
  if (tid < n_exp) {
    score_key(logits[(size_t)t * n_exp + tid], bias[tid], sc, key);
    if (!(key > -INFINITY)) key = -INFINITY;
  }
  select6_of_block(key, sc, tid, (n_exp + 63u) >> 6, route_scale, ids + (size_t)t * kTopK, wts + (size_t)t * kTopK, [] {});
}

// Decode: logits = W[n_exp][dim] . x[dim] and the selection in one launch. A workgroup is eight waves, four to an expert's row,
// so that a row of up to 8192 columns is one trip to memory; the launch's last workgroup has no rows and selects.
//
// What bounds it is a chain of latencies: launch, one trip to memory, the hand-over of the logits between workgroups, the
// scores' double-precision arithmetic, the selection. The hand-over is a record per expert: the logit and the number of the
// call in one 64-bit device-scope store, and the selecting workgroup, one expert a thread, reads its record until it holds
// this call's number. Against workgroups that waited for their stores, counted themselves in and left the selection to the last
// one, with a wave a row (14 vectors a lane in two trips) and two reductions per choice: 384x7168 of BF16 10.9 -> 7.7 us,
// 384x5120 10.1 -> 7.2, 64x2048 8.3 -> 5.4, F32 384x7168 12.4 -> 8.6 (calls back to back, weights from HBM).
// The call's number stands behind the records; the selecting workgroup counts it up at its end, when every other workgroup
// has read it (it has their records). Every wait ends: the other workgroups wait for nothing, and the selecting one, the last
// of the launch, gives up after `polls` reads (kRouterPolls: seconds). Then a workgroup may still be to come that reads the number
// only after it has been counted up, and its record would pass for one of the next call. So a call that gave up leaves
// kRouterGaveUp in place of its number: records written under it name no call (0), and this call and all that follow return six NaN
// weights, until the scratch is zeroed. (Should six keys of +inf stand ahead of the missing ones, the choice does not depend on these.)
constexpr uint32_t kRouterPolls = 1u << 22;
constexpr uint32_t kRouterGaveUp = 0xFFFFFFFFu;  // (as a number, the last before counting starts again at 1: never left by a call that ended well)
template <int QT, uint32_t U>
__global__ __launch_bounds__(512) void router_fused_kernel(const float* __restrict__ x, const void* __restrict__ W, uint32_t dim,
                                                           uint32_t n_exp, const float* __restrict__ bias, float* logits,
                                                           uint64_t* recs, uint32_t* call, int* __restrict__ ids,
                                                           float* __restrict__ wts, float route_scale, uint32_t polls) {
  constexpr uint32_t WAVES = 8, SPLIT = 4;
  __shared__ float part[WAVES];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  const uint32_t number = *call + 1u;  // 0: an earlier call gave up
  if (blockIdx.x + 1u < gridDim.x) {
    const uint32_t e = blockIdx.x * (WAVES / SPLIT) + wave / SPLIT, first = 64u * (wave % SPLIT) + lane;
    constexpr uint32_t STEP = 64u * SPLIT;
    float acc = 0.f;
    if constexpr (QT == MSQ_F32) {
      const float4* wr = (const float4*)((const float*)W + (size_t)e * dim);
      const float4* xv = (const float4*)x;
      const uint32_t nv = dim / 4u;
      for (uint32_t c0 = first; c0 < nv; c0 += STEP * U) {
        float4 a[U], b[U];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) { const uint32_t c = min(c0 + STEP * u, nv - 1u); a[u] = wr[c]; b[u] = xv[c]; }
#pragma unroll
        for (uint32_t u = 0; u < U; u++)
          if (c0 + STEP * u < nv) acc += a[u].x * b[u].x + a[u].y * b[u].y + a[u].z * b[u].z + a[u].w * b[u].w;
      }
    } else {
      const uint4* wr = (const uint4*)((const uint16_t*)W + (size_t)e * dim);
      const float4* xv = (const float4*)x;
      const uint32_t nv = dim / 8u;
      for (uint32_t c0 = first; c0 < nv; c0 += STEP * U) {
        uint4 a[U];
        float4 b0[U], b1[U];
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
          const uint32_t c = min(c0 + STEP * u, nv - 1u);
          a[u] = wr[c]; b0[u] = xv[2 * c]; b1[u] = xv[2 * c + 1];
        }
#pragma unroll
        for (uint32_t u = 0; u < U; u++)
          if (c0 + STEP * u < nv)
            acc += __builtin_bit_cast(float, a[u].x << 16) * b0[u].x + __builtin_bit_cast(float, a[u].x & 0xFFFF0000u) * b0[u].y +
                   __builtin_bit_cast(float, a[u].y << 16) * b0[u].z + __builtin_bit_cast(float, a[u].y & 0xFFFF0000u) * b0[u].w +
                   __builtin_bit_cast(float, a[u].z << 16) * b1[u].x + __builtin_bit_cast(float, a[u].z & 0xFFFF0000u) * b1[u].y +
                   __builtin_bit_cast(float, a[u].w << 16) * b1[u].z + __builtin_bit_cast(float, a[u].w & 0xFFFF0000u) * b1[u].w;
      }
    }
    const float v = wave_sum(acc);
    if (lane == 0) part[wave] = v;
    __syncthreads();
    if (wave % SPLIT == 0 && lane == 0) {
      const float logit = (part[wave] + part[wave + 1]) + (part[wave + 2] + part[wave + 3]);
      __hip_atomic_store(recs + e, (uint64_t)__builtin_bit_cast(uint32_t, logit) | ((uint64_t)number << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      logits[e] = logit;
    }
    return;
  }
  float key = -INFINITY;
  double sc = 0.0;
  if (tid < n_exp) {
    const float b = bias[tid];
    uint64_t r = 0;
    for (uint32_t k = 0; k < polls; k++) {
      r = __hip_atomic_load(recs + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if ((uint32_t)(r >> 32) == number) break;
    }
    score_key(__builtin_bit_cast(float, (uint32_t)r), b, sc, key);
    if (!(key > -INFINITY)) key = -INFINITY;
    if ((uint32_t)(r >> 32) != number || number == 0u) {  // no logit: ahead of every other key, with a score that makes all six weights NaN
      key = INFINITY;
      sc = __builtin_nan("");
      __hip_atomic_store(call, kRouterGaveUp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // ahead of the barrier, and so of the number
    }
  }
  select6_of_block(key, sc, tid, WAVES, route_scale, ids, wts, [&] {  // (the mark is the greatest number: it stays)
    if (number != kRouterGaveUp) __hip_atomic_fetch_max(call, number, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else atomicCAS(call, number - 1u, 0u);
  });
}

// Routing lists: one workgroup per expert e, its waves on consecutive slices of the entries. A first pass over the ids
// counts the entries of lower experts (the expert's offset) and its own; a second pass writes its entries in entry order,
// positions from ballots behind what the waves before count. No atomics: the lists are the same on every run, sorted by
// (expert, entry index). Bound by the latency of a wave's loads, hence the waves: with one per expert 4096 tokens of 384
// experts took 41 us, now 14. SPLIT = false, entries that one wave fetches in one round: a wave per expert, four to a
// workgroup, no meeting (1 to 128 tokens 3 to 4 % less than a workgroup of one wave per expert).
template <bool SPLIT>
__global__ __launch_bounds__(1024) void route_lists_kernel(const int* __restrict__ ids, const float* __restrict__ w,
                                                          uint32_t n_entries, uint32_t n_exp, uint32_t* __restrict__ counts,
                                                          uint32_t* __restrict__ offsets, uint32_t* __restrict__ entry,
                                                          uint32_t* __restrict__ tok, float* __restrict__ lw,
                                                          uint32_t* __restrict__ slot_of) {
  const uint32_t lane = threadIdx.x & 63u, wave = SPLIT ? threadIdx.x >> 6 : 0u, nwaves = SPLIT ? blockDim.x >> 6 : 1u;
  const int e = SPLIT ? (int)blockIdx.x : (int)(blockIdx.x * 4u + (threadIdx.x >> 6));
  if (e >= (int)n_exp) return;  // whole waves leave, and only where no barrier follows
  const uint32_t per = ((n_entries + nwaves - 1u) / nwaves + 63u) & ~63u;  // (entries: below 2^31)
  const uint32_t first = min(wave * per, n_entries), end = min(first + per, n_entries);
  constexpr uint32_t U = 16;  // ids fetched per lane before they are used: the loop is bound by load latency otherwise
  uint32_t lt = 0, eq = 0;
  for (uint32_t i0 = first; i0 < end; i0 += 64u * U) {
    int id[U];
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
      const uint32_t i = i0 + 64u * u + lane;
      id[u] = ids[min(i, end - 1u)];
      if (i >= end) id[u] = -1;
    }
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
      lt += (id[u] >= 0 && id[u] < e) ? 1u : 0u;
      eq += id[u] == e ? 1u : 0u;
    }
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) { lt += __shfl_xor(lt, m, 64); eq += __shfl_xor(eq, m, 64); }
  const uint32_t mine = eq;
  uint32_t before = 0;
  if constexpr (SPLIT) {
    __shared__ uint32_t s_lt[16], s_eq[16];
    if (lane == 0) { s_lt[wave] = lt; s_eq[wave] = eq; }
    __syncthreads();
    lt = 0; eq = 0;
    for (uint32_t w0 = 0; w0 < nwaves; w0++) {
      lt += s_lt[w0];
      if (w0 < wave) before += s_eq[w0];
      eq += s_eq[w0];
    }
  }
  if (lane == 0 && wave == 0) {
    counts[e] = eq;
    offsets[e] = lt;
    if (e == (int)n_exp - 1) offsets[n_exp] = lt + eq;
  }
  if (mine == 0) return;
  uint32_t base = lt + before;
  const uint64_t below = (1ull << lane) - 1ull;
  for (uint32_t i0 = first; i0 < end; i0 += 64u * U) {
    int id[U];
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
      const uint32_t i = i0 + 64u * u + lane;
      id[u] = ids[min(i, end - 1u)];
      if (i >= end) id[u] = -1;
    }
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
      const uint32_t i = i0 + 64u * u + lane;
      const bool m = id[u] == e;
      const uint64_t bits = __ballot(m);
      if (m) {
        const uint32_t pos = base + (uint32_t)__popcll(bits & below);
        entry[pos] = i;
        tok[pos] = i / (uint32_t)kTopK;
        lw[pos] = w[i];
        slot_of[i] = pos;
      }
      base += (uint32_t)__popcll(bits);
    }
  }
}

// Up to 1024 tokens the chain of a wave bounds the launch: an expert a thread. Beyond, the double-precision arithmetic of all of
// them, and a wave per token has fewer reductions, but 64 experts are one wave either way. A wave per token / an expert a thread,
// us: 384 experts, 2 tokens 8.0 / 4.4, 37 8.6 / 4.6, 512 8.9 / 6.1, 1024 9.2 / 7.8, 2048 11.5 / 13.0; 128, 37 tokens 5.8 / 4.3, 4096 9.9 / 9.7,
// 6000 13.0 / 13.7, 16384 27.5 / 29.5; 64, 4096 tokens 8.4 / 7.8, 262144 298 / 254. (A launch holds fewer than 2^32 threads: 64 a token of
// either form here, where 128 would halve the tokens that a call can have.)
bool topk_wide(int n_tokens, int n_exp) { return n_tokens <= 1024 || n_exp <= 64 || (n_exp <= 128 && n_tokens <= 4096); }
bool exp_ok(int n_exp) { return n_exp >= 64 && n_exp <= 64 * kMaxEpl && n_exp % 64 == 0; }

}  // namespace
}  // namespace msq

using namespace msq;

extern "C" {

// which of its two forms msq_router_topk takes (for tests)
int msq_test_router_topk_wide(int n_tokens, int n_exp) { return topk_wide(n_tokens, n_exp) ? 1 : 0; }

int msq_router_topk(void* stream, const MsqBuffer* logits, const MsqBuffer* bias, const MsqBuffer* ids, const MsqBuffer* w,
                    int n_tokens, int n_exp, float route_scale) {
  if (!exp_ok(n_exp) || n_tokens < 0) return unsupported("router_topk", MSQ_F32, n_tokens, n_exp);
  if (n_tokens == 0) return MSQ_OK;
  if (!buf_ok(logits, (size_t)n_tokens * n_exp * 4) || !buf_ok(bias, (size_t)n_exp * 4) ||
      !buf_ok(ids, (size_t)n_tokens * kTopK * 4) || !buf_ok(w, (size_t)n_tokens * kTopK * 4))
    return fail(MSQ_ERR_ARGUMENT, "macseek quant: router_topk: buffer missing or too small (tokens %d experts %d)", n_tokens, n_exp);
  if (topk_wide(n_tokens, n_exp))
    hipLaunchKernelGGL(router_topk_wide_kernel, dim3((unsigned)n_tokens), dim3((unsigned)n_exp), 0, (hipStream_t)stream, (const float*)bptr(logits),
                       (const float*)bptr(bias), (int*)bptr_mut(ids), (float*)bptr_mut(w), (uint32_t)n_exp, route_scale);
  else hipLaunchKernelGGL(router_topk_kernel, dim3((unsigned)((n_tokens + 3) / 4)), dim3(256), 0, (hipStream_t)stream,
                     (const float*)bptr(logits), (const float*)bptr(bias), (int*)bptr_mut(ids), (float*)bptr_mut(w),
                     (uint32_t)n_tokens, (uint32_t)n_exp, route_scale);
  MSQ_HIP(hipGetLastError());
  return MSQ_OK;
}

// scratch: logits f32 [n_exp] (padded to 256 bytes), records {logit f32, number of the call u32} [n_exp] in the first half of 16
// bytes an expert (callers keep the scratch size), then the number of the last call in a 256-byte line of its own
size_t msq_router_scratch_bytes(int n_exp) { return ((size_t)n_exp * 4 + 255) / 256 * 256 + (size_t)n_exp * 16 + 256; }

static int router_fused_impl(void* stream, int wtype, const MsqBuffer* x, const MsqBuffer* W, const MsqBuffer* bias, const MsqBuffer* scratch,
                             const MsqBuffer* ids, const MsqBuffer* w, int dim, int n_exp, float route_scale, uint32_t polls) {
  if (!exp_ok(n_exp) || dim < 8 || dim % 8 || (wtype != MSQ_F32 && wtype != MSQ_BF16)) return unsupported("router_fused", wtype, n_exp, dim);
  const size_t esz = wtype == MSQ_F32 ? 4 : 2;
  if (!buf_ok(x, (size_t)dim * 4) || !buf_ok(W, (size_t)n_exp * dim * esz) || !buf_ok(bias, (size_t)n_exp * 4) ||
      !buf_ok(ids, kTopK * 4) || !buf_ok(w, kTopK * 4) || ((uintptr_t)bptr(x) & 15) || ((uintptr_t)bptr(W) & 15))
    return fail(MSQ_ERR_ARGUMENT, "macseek quant: router_fused: buffer missing, too small or not 16-byte aligned (experts %d dim %d)", n_exp, dim);
  if (!buf_ok(scratch, msq_router_scratch_bytes(n_exp)) || ((uintptr_t)bptr(scratch) & 15))
    return fail(MSQ_ERR_SCRATCH, "macseek quant: router_fused scratch too small unsupported (type %s rows %d cols %d)",
                msq_type_name_of(wtype), n_exp, dim);
  float* logits = (float*)bptr_mut(scratch);
  uint64_t* recs = (uint64_t*)(bptr_mut(scratch) + ((size_t)n_exp * 4 + 255) / 256 * 256);
  uint32_t* call = (uint32_t*)(bptr_mut(scratch) + msq_router_scratch_bytes(n_exp) - 256);
  const dim3 grid((unsigned)(n_exp / 2 + 1)), block(512);  // two rows a workgroup, and the selecting one
  hipStream_t st = (hipStream_t)stream;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, block, 0, st, (const float*)bptr(x), (const void*)bptr(W), (uint32_t)dim, (uint32_t)n_exp,
                       (const float*)bptr(bias), logits, recs, call, (int*)bptr_mut(ids), (float*)bptr_mut(w), route_scale, polls);
  };
  // vectors a lane of the four waves that share a row: one trip to memory up to 8192 columns
  const int per_lane = (dim / (wtype == MSQ_F32 ? 4 : 8) + 255) / 256;
  auto by_u = [&]<int QT>() {
    if (per_lane <= 2) return launch(router_fused_kernel<QT, 2>);
    if constexpr (QT == MSQ_F32) {
      if (per_lane > 4) return launch(router_fused_kernel<QT, 8>);
    }
    launch(router_fused_kernel<QT, 4>);
  };
  if (wtype == MSQ_F32) by_u.template operator()<MSQ_F32>();
  else by_u.template operator()<MSQ_BF16>();
  MSQ_HIP(hipGetLastError());
  return MSQ_OK;
}

int msq_router_fused(void* stream, int wtype, const MsqBuffer* x, const MsqBuffer* W, const MsqBuffer* bias, const MsqBuffer* scratch,
                     const MsqBuffer* ids, const MsqBuffer* w, int dim, int n_exp, float route_scale) {
  return router_fused_impl(stream, wtype, x, W, bias, scratch, ids, w, dim, n_exp, route_scale, kRouterPolls);
}
// the same with a limit of its own on the selecting workgroup's wait (for tests)
int msq_test_router_fused_polls(void* stream, int wtype, const MsqBuffer* x, const MsqBuffer* W, const MsqBuffer* bias, const MsqBuffer* scratch,
                                const MsqBuffer* ids, const MsqBuffer* w, int dim, int n_exp, float route_scale, uint32_t polls) {
  return router_fused_impl(stream, wtype, x, W, bias, scratch, ids, w, dim, n_exp, route_scale, polls);
}

int msq_route_lists(void* stream, const MsqBuffer* ids, const MsqBuffer* w, int n_tokens, int n_exp, const MsqRouteLists* L) {
  if (n_exp < 1 || n_tokens < 0 || !L) return unsupported("route_lists", MSQ_F32, n_tokens, n_exp);
  const size_t n_entries = (size_t)n_tokens * kTopK;
  if (n_tokens > L->max_tokens || n_entries >= (1ull << 31))
    return fail(MSQ_ERR_ARGUMENT, "macseek quant: route_lists: %d tokens exceed the lists' capacity of %d", n_tokens, L->max_tokens);
  if (!buf_ok(&L->counts, (size_t)n_exp * 4) || !buf_ok(&L->offsets, (size_t)(n_exp + 1) * 4))
    return fail(MSQ_ERR_ARGUMENT, "macseek quant: route_lists: counts / offsets missing or too small (experts %d)", n_exp);
  if (n_tokens > 0 && (!buf_ok(ids, n_entries * 4) || !buf_ok(w, n_entries * 4) || !buf_ok(&L->entry, n_entries * 4) ||
                       !buf_ok(&L->tok, n_entries * 4) || !buf_ok(&L->w, n_entries * 4) || !buf_ok(&L->slot_of, n_entries * 4)))
    return fail(MSQ_ERR_ARGUMENT, "macseek quant: route_lists: buffer missing or too small (tokens %d)", n_tokens);
  // a wave per 1024 entries (one round of its loads), at most sixteen
  const unsigned waves = (unsigned)std::min<size_t>(16, (n_entries + 1023) / 1024);
  hipLaunchKernelGGL(waves > 1 ? route_lists_kernel<true> : route_lists_kernel<false>, dim3((unsigned)(waves > 1 ? n_exp : (n_exp + 3) / 4)),
                     dim3(waves > 1 ? 64 * waves : 256), 0, (hipStream_t)stream,
                     n_tokens ? (const int*)bptr(ids) : nullptr, n_tokens ? (const float*)bptr(w) : nullptr, (uint32_t)n_entries,
                     (uint32_t)n_exp, (uint32_t*)bptr_mut(&L->counts), (uint32_t*)bptr_mut(&L->offsets),
                     n_tokens ? (uint32_t*)bptr_mut(&L->entry) : nullptr, n_tokens ? (uint32_t*)bptr_mut(&L->tok) : nullptr,
                     n_tokens ? (float*)bptr_mut(&L->w) : nullptr, n_tokens ? (uint32_t*)bptr_mut(&L->slot_of) : nullptr);
  MSQ_HIP(hipGetLastError());
  return MSQ_OK;
}

}  // extern "C"

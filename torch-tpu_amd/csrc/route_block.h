// Routing of ONE token by a whole 256-thread workgroup (E <= 256), for batches so small that the
// time of a launch is the length of its longest dependent chain, not its instruction count.
//
// Thread e owns expert e.  Instead of K arg-max rounds in sequence, every thread counts the
// experts that come before its own in "greater score, then lower index" order, first in its part of the row, then
// among the best of all parts: that count is the expert's position in the sorted row, so the K picks are those whose
// count is below K, and they come out in descending order.  The order is one unsigned 64-bit compare per pair: the
// score mapped to an unsigned integer of the same order in the high half, "lower index first" in
// the low half (compare masks combined on the scalar side cost several times as much).  The group limit works the same way: position inside the
// group (0 and 1 make the group's score), then position of the group among the groups.  All reads
// of the score table are LDS broadcasts.  Orders, sums and divisions are those of the
// one-wavefront-per-token kernel, so both give the same ids and the same weights, bit for bit.
#pragma once
#include "moe_common.h"
#include "../../include/moe_hip.h"

namespace moe {

constexpr int kRouteBlock = 256;

struct RouteBlockSmem {
  uint64_t key[kRouteBlock];   // order key of every expert's selection score (0 beyond E: after everything)
  uint64_t cand[kRouteBlock];  // order keys of the experts that are still in question (0: none)
  float raw[kRouteBlock];      // what the weights are made of
  float gtop[64][2];           // best two selection scores of every group
  uint64_t gkey[64];           // order key of every group's score
  float wmax[kRouteBlock / 64];
  float wsel[64];              // weight source of pick k
  int isel[64];                // expert of pick k
  int above[kRouteBlock / 64], level[kRouteBlock / 64];   // experts better than -inf under the group limit, and at -inf, per wavefront
};

// (score a, index ai) comes before (b, bi) - greater score, then lower index - exactly when
// order_key(a, ai) > order_key(b, bi).  Adding +0 first makes -0 and +0 the same key, as they compare equal; NaN comes first.
__device__ __forceinline__ uint64_t order_key(float v, int idx) {
  uint32_t u = __float_as_uint(v + 0.0f);
  u = v != v ? 0xffffffffu : (u >> 31) ? ~u : (u | 0x80000000u);
  return ((uint64_t)u << 32) | (uint32_t)(0x7fffffff - idx);
}

__device__ __forceinline__ void route_block(RouteBlockSmem &sm, const void *logits_row, int logits_bf16,
                                            const float *__restrict__ bias, int E, int K, int mode, int n_groups,
                                            int topk_groups, int renorm, float scale, float *weights_row,
                                            int32_t *ids_row, float *scores_row) {
  const int e = threadIdx.x, lane = e & 63, wave = e >> 6;
  const bool live = e < E;
  float x = -INFINITY;
  if (live) x = logits_bf16 ? bf16_to_f32(((const uint16_t *)logits_row)[e]) : ((const float *)logits_row)[e];
  if (mode == MOE_ROUTE_SIGMOID && live) x = 1.0f / (1.0f + expf(-x));
  const bool logit_bias = mode == MOE_ROUTE_SOFTMAX_LOGIT_BIAS;     // the bias is part of the logits
  if (logit_bias) {
    mode = MOE_ROUTE_SOFTMAX;
    if (bias != nullptr && live) x += bias[e];
    bias = nullptr;
  }
  float raw = x;                                          // what the weight is made of (no bias)
  float v = (bias != nullptr && live) ? x + bias[e] : x;  // what the selection looks at
  if (scores_row != nullptr && live && mode != MOE_ROUTE_SOFTMAX) scores_row[e] = x;
  if (e < 64) { sm.isel[e] = -1; sm.wsel[e] = 0.f; }
  sm.cand[e] = 0;
  float denom_all = 0.f;
  if (mode == MOE_ROUTE_SOFTMAX) {
    float m = x;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    if (lane == 0) sm.wmax[wave] = m;
    __syncthreads();
    m = fmaxf(fmaxf(sm.wmax[0], sm.wmax[1]), fmaxf(sm.wmax[2], sm.wmax[3]));
    raw = live ? expf(x - m) : 0.f;
    sm.raw[e] = raw;
    __syncthreads();
    // the sum in the order the per-wavefront kernel uses: lane l adds elements l, l+64, l+128, l+192, then a butterfly
    float part = 0.f;
#pragma unroll
    for (int j = 0; j < kRouteBlock / 64; j++) part += sm.raw[lane + 64 * j];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) part += __shfl_xor(part, off, 64);
    denom_all = part;
    if (scores_row != nullptr && live) scores_row[e] = raw / denom_all;
  }
  uint64_t key = live ? order_key(v, e) : 0;
  sm.key[e] = key;
  sm.raw[e] = raw;
  __syncthreads();

  // First the position inside a part of the row - the expert's group, or the 64 experts of its wavefront: a pick is among
  // the K best of its part, so only those are compared with one another afterwards.  Against one pass over the whole
  // table that is 32 + 32 compares instead of 32 + 256 for the DeepSeek-V3 router, 64 + 16 for 128 experts.  A launch of one
  // token, one pass -> parts, in us: 256 experts in 8 groups, 8 picks 5.8 -> 3.7 (with fewer than 8 finite scores in the kept
  // groups 5.9 -> 3.8), 32 picks 5.8 -> 4.5; 256 experts without groups, 8 / 32 picks 4.8 -> 3.7 / 4.5; 128 experts 4.6 -> 3.5;
  // 8 experts 4.7 -> 2.7.
  const bool grouped = n_groups > 1 && topk_groups < n_groups;       // (a limit that keeps every group is none)
  const int per = grouped ? E / n_groups : 64;
  const int part = live ? (grouped ? e / per : wave) : 0, first = part * per, last = min(first + per, E);
  int pos = 0;                                            // position in the part
  if (live) {
#pragma unroll 8
    for (int j = first; j < last; j++) pos += sm.key[j] > key;
  }
  int n_parts = (E + 63) / 64, place = part;              // parts still in question, and which of them this one is
  bool low = false;                                       // -inf, as it came or by the limit
  uint64_t lows = 0;
  if (grouped) {
    if (live && pos < 2) sm.gtop[part][pos] = v;
    __syncthreads();
    if (e < n_groups) sm.gkey[e] = order_key(sm.gtop[e][0] + sm.gtop[e][1], e);
    __syncthreads();
    place = 0;
    if (live) {
      const uint64_t gk = sm.gkey[part];
#pragma unroll 8
      for (int h = 0; h < n_groups; h++) place += sm.gkey[h] > gk;
    }
    n_parts = topk_groups;
    // Experts of dropped groups stay candidates with -inf, as a masked_fill would leave them.  Nothing sorts below that, so
    // such an expert's position in the row is the number of better ones plus the number of its like before it.
    low = live && (place >= topk_groups || key <= order_key(-INFINITY, 0));
    lows = __ballot(low);
    const uint64_t better = __ballot(live && !low);
    if (lane == 0) {
      sm.above[wave] = __popcll(better);
      sm.level[wave] = __popcll(lows);
    }
  }
  const int kept = min(K, per), n_cand = n_parts * kept;  // at least K (the caller has checked topk_groups * per >= K)
  if (live && !low && place < n_parts && pos < kept) sm.cand[place * kept + pos] = key;
  __syncthreads();
  if (low) {
    int r = __popcll(lows & ((1ull << lane) - 1));
#pragma unroll
    for (int w = 0; w < kRouteBlock / 64; w++) r += sm.above[w] + (w < wave ? sm.level[w] : 0);
    if (r < K) { sm.isel[r] = e; sm.wsel[r] = raw; }
  }
  const uint64_t mine = sm.cand[e];
  if (mine != 0) {
    int r = 0;
    // sixteen at a time (0 beyond the candidates), all reads before the first comparison: left to itself the compiler
    // waits for every read in turn in some of the kernels
#pragma unroll 1
    for (int j0 = 0; j0 < n_cand; j0 += 16) {
      uint64_t other[16];
#pragma unroll
      for (int j = 0; j < 16; j++) other[j] = sm.cand[j0 + j];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 16; j++) r += other[j] > mine;
    }
    if (r < K) {
      const int who = 0x7fffffff - (int)(uint32_t)mine;
      sm.isel[r] = who;
      sm.wsel[r] = sm.raw[who];
    }
  }
  __syncthreads();
  if (wave == 0) {
    float w = lane < K ? sm.wsel[lane] : 0.f;
    const int idx = lane < K ? sm.isel[lane] : -1;
    if (mode == MOE_ROUTE_SOFTMAX && !renorm) w = w / denom_all;
    if (renorm) {
      float s = w;
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
      w = w / s;
    }
    if (lane < K) {
      weights_row[lane] = w * scale;
      ids_row[lane] = idx;
    }
  }
}

}  // namespace moe

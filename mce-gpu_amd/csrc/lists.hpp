// Out-lists of oriented vertices searched for the members of a vertex set, a
// wave at a time (subproblem set-up and the cost model's features).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "wave.hpp"

namespace mce {

// ---- out-lists against a subproblem's members ------------------------------
// Which arcs of some vertices' out-lists lead into S (p members, ascending).
// A step takes four arcs a lane; its chain is one load of arcs and one search
// of log2 p steps, both for all four at once. (A list after the other with an
// arc a lane waited for its offsets, its arcs and a search of its own: 2.6 us
// a list, which was 50 to 90 % of the enumeration of graphs with up to some
// 100 members a subproblem.) Enumeration in ms before and after: G(50,000, deg
// 90) 3.26 -> 1.74, 100 block-model graphs of 500..900 3.16 -> 1.84, 301 of
// 400..500 2.74 -> 1.72, 64 of 64..2,000 15.7 -> 11.6, 64 of 200..4,096 309 ->
// 297, R-MAT 12 arcs 3.1 -> 2.35, R-MAT 14 21.0 -> 18.5.
enum : int { kInGlb = 0, kInLds = 1, kAnywhere = 2 };
template <int kS>
__device__ __forceinline__ uint32_t ld_s(const uint32_t *p, uint32_t i) {
  if constexpr (kS == kAnywhere) return p[i];
  else if constexpr (kS == kInLds) return ((const __attribute__((address_space(3))) uint32_t *)p)[i];
  else return ((const __attribute__((address_space(1))) uint32_t *)p)[i];
}
constexpr uint32_t kArcs = 4;
// Places in S of the heads of list[k], list[k + step], ... (below n_arcs), or
// kNone.
template <int kS>
__device__ __forceinline__ void find_arcs(const uint32_t *S, uint32_t p, const uint32_t *list, uint32_t k, uint32_t step,
                                          uint32_t n_arcs, uint32_t (&j)[kArcs]) {
  uint32_t y[kArcs];
#pragma unroll
  for (uint32_t m = 0; m < kArcs; ++m) {
    y[m] = k + step * m < n_arcs ? list[k + step * m] : kNone;
    j[m] = 0;
  }
  for (uint32_t st = 1u << (31 - __builtin_clz(p)); st; st >>= 1) {
#pragma unroll
    for (uint32_t m = 0; m < kArcs; ++m) {
      const uint32_t t = j[m] + st;
      const uint32_t v = ld_s<kS>(S, min(t, p) - 1u);
      j[m] = t <= p && v < y[m] ? t : j[m];
    }
  }
#pragma unroll
  for (uint32_t m = 0; m < kArcs; ++m) {
    const uint32_t v = ld_s<kS>(S, min(j[m], p - 1u));
    j[m] = y[m] != kNone && v == y[m] ? j[m] : kNone;
  }
}
// All arcs of n <= 64 lists (lane r < n: list [b, b + len)): hit gets a list's
// number and the places of four of its arcs, lane by lane. Lists no longer
// than they are many go a lane each, four arcs at a time (as many steps as
// the longest has fours; a step of 16 lanes a list would leave most of them
// idle: R-MAT 12 (ef 8) 0.54 -> 0.36 ms), lists of more than kLongList arcs one by one on the whole wave (one
// on 16 lanes would keep the other three groups waiting; R-MAT 14 in ms: from
// 64 arcs on 22.0, 128 19.8, 256 19.5, never 20.9), all others four at a time
// on 16 lanes.
constexpr uint32_t kLongList = 256;
template <int kS, typename Hit>
__device__ __forceinline__ void walk_lists(const uint32_t *oc, const uint32_t *S, uint32_t p, uint32_t n, uint64_t b,
                                           uint32_t len, Hit hit) {
  const uint32_t L = lane_id();
  if (L >= n) len = 0;
  const uint32_t most = wave_max(len);
  uint32_t j[kArcs];
  if (most <= n) {
    for (uint32_t k0 = 0; k0 < most; k0 += kArcs) {
      find_arcs<kS>(S, p, oc + b, k0, 1, len, j);
      hit(L, j);
    }
    return;
  }
  const uint32_t gl = L & 15u, g = L >> 4, shorts = len <= kLongList ? len : 0u;
  for (uint32_t r0 = 0; r0 < n; r0 += 4) {
    const uint32_t r = r0 + g, at = 4 * (r & 63u);
    const uint32_t bl = (uint32_t)__builtin_amdgcn_ds_bpermute((int)at, (int)(uint32_t)b);
    const uint32_t bh = (uint32_t)__builtin_amdgcn_ds_bpermute((int)at, (int)(uint32_t)(b >> 32));
    const uint32_t nr = (uint32_t)__builtin_amdgcn_ds_bpermute((int)at, (int)shorts), lr = r < n ? nr : 0u;
    const uint32_t *list = oc + ((uint64_t)bh << 32 | bl);
    for (uint32_t k0 = 0; ballot(k0 < lr) != 0; k0 += 16 * kArcs) {
      find_arcs<kS>(S, p, list, k0 + gl, 16, lr, j);
      hit(r, j);
    }
  }
  for (uint64_t m = ballot(len > kLongList); m; m &= m - 1) {
    const uint32_t r = ctz64(m), lr = rdlane(len, r);
    const uint32_t *list = oc + rdlane64(b, r);
    for (uint32_t k0 = 0; k0 < lr; k0 += kWave * kArcs) {
      find_arcs<kS>(S, p, list, k0 + L, kWave, lr, j);
      hit(r, j);
    }
  }
}

}  // namespace mce

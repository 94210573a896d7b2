// Preprocessing on the GPU: degeneracy ordering by batched k-core peeling,
// orientation of the CSR, and the heaviest-first first-level work list.
//
// Peeling follows the reference's round semantics (include/kcore.cuh:80-143,
// :233-316): a round removes the whole frontier (alive vertices of degree <=
// level) and gives it the round index as priority; neighbours whose degree
// falls to `level` during the round form the next frontier; when a round
// comes up empty the level rises. The design differs: a round is a chain of
// dependent memory accesses over few vertices (at R-MAT 14, 300 rounds of 55
// vertices), so what bounds the peel is latency and launches, not bandwidth.
// A small graph, and the densest part of a larger one, is peeled by one
// workgroup with its degrees in LDS, in one launch; above that each level
// step and each large round is one launch of the grid whose last workgroup
// advances the device-resident state and runs the small rounds that follow.
// The host only polls a done flag every 16..128 launches. Against three
// launches a round (select, peel, advance), same card: R-MAT 14 5.1 -> 0.68
// ms, R-MAT 18 11 -> 6.1 ms, Chung-Lu 2^18 15.2 -> 5.6 ms, ER 4096 0.67 ->
// 0.15 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "engine.hpp"
#include "internal.hpp"
#include "wave.hpp"

namespace mce {

namespace {

enum : uint32_t { kModeLevel = 0, kModePeel = 1, kModeDone = 2 };

struct PeelState {
  int32_t level;
  uint32_t round;
  uint32_t mode;
  uint32_t cur;
  uint32_t fcnt, ncnt;
  uint32_t alive_cur, acnt, acnt2;
  uint32_t degeneracy;
  uint32_t arrived;  // workgroups of the running launch that have finished
  unsigned long long arcs, arcs2;  // arcs between the alive vertices at the last level step
  uint32_t taken;  // arc slots handed out by kc_number
};

// Device arrays of one peel.
struct PeelBufs {
  PeelState *st;
  const uint64_t *rp;
  const uint32_t *ci;
  int32_t *deg;
  uint32_t *prio, *core;
  uint32_t *alive0, *alive1, *front0, *front1;
  uint32_t *loc;   // tail: vertex -> its index in the alive list (kNone: removed)
  uint32_t *trow;  // tail: first arc and arc count of each list entry
  uint16_t *tarc;  // tail: the arcs between alive vertices, as indices
  uint32_t n;
};

constexpr uint32_t kBlock = 256;
constexpr uint32_t kPeelBlock = 1024;
// One workgroup takes the whole peel of a graph of at most kTailMax vertices
// and kTailArcsEarly arcs, and the rest of a larger graph's peel once the alive
// vertices and the arcs between them are as few: its round costs 2 to 3 us
// against 6 us for a launch of the grid, but one CU takes only about 0.4 arcs
// a nanosecond (measured on Chung-Lu 2^18: 3.3 ms against 10.8 ms a tail of
// 32,768 vertices with no bound on its arcs).
constexpr uint32_t kTailMax = 32768;
// Arcs of a tail (16-bit indices, 4 MiB), and those of a tail or a whole graph
// before kTailRounds rounds: a peel that took many rounds has many small ones
// left, which launches cost more than the one CU's 0.4 arcs a nanosecond (2^20
// and 2^21 arcs in ms: R-MAT 18 6.4 and 5.1, Chung-Lu 2^18 5.7 and 5.0), one
// that took few goes in large rounds (G(20,000, 600,000) 0.76 and 0.93).
constexpr uint32_t kTailArcs = 1u << 21, kTailArcsEarly = 1u << 20, kTailRounds = 64;
// With at most this many vertices, row offsets share the LDS with degrees.
constexpr uint32_t kTailRowsMax = 16384;
// A larger graph's rounds run on one workgroup while they hold about this
// many arcs.
constexpr uint32_t kFrontArcs = 8192;
// Workgroups of a grid step: enough for the vertices, at most one per CU (the
// last-to-finish count takes 11 ns of each).
constexpr uint32_t kPeelGridMin = 32, kPeelGridMax = 256, kPeelGridVerts = 2048;
// Frontier entries kept in LDS by the one-workgroup rounds; the rest of a
// longer frontier is in the frontier array.
constexpr uint32_t kFrontLds = 1536;
// Rows above this many neighbours are left to the whole workgroup, which
// takes them one at a time; at most kLongMax of them a round (LDS list).
constexpr uint32_t kLongRow = 512, kLongMax = 512;
// Sentinel degree of a removed vertex in LDS: more than any degree and any
// number of later decrements can bring to a level.
constexpr int32_t kGone = 0x40000000;

struct PeelLds {
  uint32_t front[2][kFrontLds];
  uint32_t longs[kLongMax];
  uint32_t ncnt, nlong, left, min_deg, last;
  uint32_t wsel[kPeelBlock / kWave], wkeep[kPeelBlock / kWave];  // level step: per wave
  uint32_t bsel, bkeep;
  unsigned long long arcs;
};
constexpr size_t kPeelLds = sizeof(PeelLds), kTailLds = sizeof(PeelLds) + 4 * (size_t)kTailMax + 16;
static_assert(2 * kTailRowsMax == kTailMax, "degrees and row offsets share kTailLds");

__device__ __forceinline__ uint32_t ld_dev(const uint32_t *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void st_dev(uint32_t *p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ void kc_init(PeelBufs b) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < b.n; v += stride) {
    b.deg[v] = (int32_t)(b.rp[v + 1] - b.rp[v]);
    b.prio[v] = kNone;
    b.alive0[v] = (uint32_t)v;
    b.loc[v] = kNone;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    PeelState *st = b.st;
    st->level = -1;
    st->round = 0;
    st->mode = kModeLevel;
    st->cur = 0;
    st->fcnt = st->ncnt = 0;
    st->alive_cur = 0;
    st->acnt = b.n;
    st->acnt2 = 0;
    st->degeneracy = 0;
    st->arrived = 0;
    st->arcs = b.rp[b.n];
    st->arcs2 = 0;
    st->taken = 0;
  }
}

// One frontier vertex's neighbour w loses a neighbour. Its degree is lowered
// whether or not it is still there: a removed vertex's degree is at most the
// level it was removed at, so it never falls from level + 1 again. Returns
// true when w falls to the level: it joins the next round.
__device__ __forceinline__ bool lower_dev(int32_t *deg, uint32_t w, int32_t level) {
  return atomicSub(&deg[w], 1) == level + 1;
}

// ---- rounds by one workgroup ----------------------------------------------
// Where the vertices' rows and degrees are: kDev, both in device memory;
// kWhole, degrees in LDS; kWholeRows, row offsets too; kCore, degrees in LDS
// and rows in the tail's compacted arcs. Frontier entries are vertex ids, in
// kCore tail indices.
enum Where : int { kDev, kWhole, kWholeRows, kCore };

template <int kAt>
struct Rounds {
  const PeelBufs &b;
  PeelLds &sh;
  int32_t *dl;          // LDS degrees
  const uint32_t *rows;  // kWholeRows: LDS row offsets
  const uint32_t *ids;   // kCore: vertex ids of the tail indices

  __device__ __forceinline__ uint32_t front(uint32_t c, uint32_t i) const {
    return i < kFrontLds ? sh.front[c][i] : ld_dev(&(c ? b.front1 : b.front0)[i]);
  }
  __device__ __forceinline__ void push(uint32_t c, uint32_t v) const {
    const uint32_t i = atomicAdd(&sh.ncnt, 1u);
    if (i < kFrontLds) sh.front[c][i] = v;
    else st_dev(&(c ? b.front1 : b.front0)[i], v);
  }
  __device__ __forceinline__ void row_of(uint32_t v, uint64_t &k, uint64_t &e) const {
    if constexpr (kAt == kWholeRows) {
      k = rows[v];
      e = rows[v + 1];
    } else if constexpr (kAt == kCore) {
      k = b.trow[2 * v];
      e = k + b.trow[2 * v + 1];
    } else {
      k = b.rp[v];
      e = b.rp[v + 1];
    }
  }
  __device__ __forceinline__ uint32_t arc(uint64_t k) const {
    if constexpr (kAt == kCore) return b.tarc[k];
    else return b.ci[k];
  }
  __device__ __forceinline__ void settled(uint32_t v, int32_t level, uint32_t pri) const {
    const uint32_t id = kAt == kCore ? ids[v] : v;
    b.prio[id] = pri;
    b.core[id] = (uint32_t)level;
  }
  // Takes a neighbour of w away; a vertex that falls to the level is appended
  // to frontier c with priority `pri`.
  __device__ __forceinline__ void lower(uint32_t w, int32_t level, uint32_t pri, uint32_t c) const {
    bool add;
    if constexpr (kAt == kDev) {
      add = lower_dev(b.deg, w, level);
    } else {
      add = atomicSub(&dl[w], 1) == level + 1;
      if (add) dl[w] = kGone;
    }
    if (add) {
      settled(w, level, pri);
      push(c, w);
    }
  }
  // The length of the frontier just appended to, once every wave's entries
  // can be read (those past the LDS part are in device memory).
  __device__ __forceinline__ uint32_t settle() const {
    __syncthreads();
    const uint32_t n = sh.ncnt;
    if (n > kFrontLds) __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    return n;
  }
  // One round over the fcnt vertices of frontier c; fills frontier c ^ 1 and
  // returns its length. Groups of 16 lanes take four rows at a time (the
  // chain of loads of a row, offsets -> neighbours -> degree, is what a round
  // waits for), long rows go to the whole workgroup.
  __device__ __forceinline__ uint32_t round(uint32_t fcnt, uint32_t c, int32_t level, uint32_t pri) const {
    constexpr uint32_t kGroups = kPeelBlock / 16, kRows = 4;
    const uint32_t t = threadIdx.x, gl = t & 15u, gid = t >> 4;
    if (t == 0) sh.ncnt = sh.nlong = 0;
    __syncthreads();
    for (uint32_t i0 = gid; i0 < fcnt; i0 += kGroups * kRows) {
      uint64_t k[kRows], e[kRows];
      uint32_t w[kRows];
#pragma unroll
      for (uint32_t j = 0; j < kRows; ++j) {
        const uint32_t i = i0 + j * kGroups;
        k[j] = e[j] = 0;
        if (i < fcnt) {
          const uint32_t v = front(c, i);
          row_of(v, k[j], e[j]);
          if (e[j] - k[j] > kLongRow) {
            uint32_t at = 0;
            if (gl == 0) at = atomicAdd(&sh.nlong, 1u);
            at = (uint32_t)__shfl((int)at, 0, 16);
            if (at < kLongMax) {
              if (gl == 0) sh.longs[at] = v;
              e[j] = k[j];
            }
          }
          k[j] += gl;
        }
      }
#pragma unroll
      for (uint32_t j = 0; j < kRows; ++j)
        if (k[j] < e[j]) w[j] = arc(k[j]);
#pragma unroll
      for (uint32_t j = 0; j < kRows; ++j)
        if (k[j] < e[j]) lower(w[j], level, pri, c ^ 1u);
#pragma unroll
      for (uint32_t j = 0; j < kRows; ++j) {
        uint64_t q = k[j] + 16;
        for (; q + 48 < e[j]; q += 64) {
          const uint32_t w0 = arc(q), w1 = arc(q + 16), w2 = arc(q + 32), w3 = arc(q + 48);
          lower(w0, level, pri, c ^ 1u);
          lower(w1, level, pri, c ^ 1u);
          lower(w2, level, pri, c ^ 1u);
          lower(w3, level, pri, c ^ 1u);
        }
        for (; q < e[j]; q += 16) lower(arc(q), level, pri, c ^ 1u);
      }
    }
    __syncthreads();
    const uint32_t nl = min(sh.nlong, kLongMax);
    for (uint32_t i = 0; i < nl; ++i) {
      uint64_t q, e;
      row_of(sh.longs[i], q, e);
      for (q += t; q < e; q += kPeelBlock) lower(arc(q), level, pri, c ^ 1u);
    }
    return settle();
  }
  // The peel from a level step on, of `left` vertices among the cnt of dl.
  // A level's frontier comes from a scan of the LDS degrees; a level without
  // one has no round, so the next level is then the smallest degree left.
  __device__ __forceinline__ void levels(uint32_t cnt, uint32_t left, int32_t level, uint32_t pri,
                                         uint32_t degen) const {
    const uint32_t t = threadIdx.x;
    while (left) {
      ++level;
      if (t == 0) {
        sh.ncnt = 0;
        sh.min_deg = 0xFFFFFFFFu;
      }
      __syncthreads();
      uint32_t mn = 0xFFFFFFFFu;
      for (uint32_t i = t; i < cnt; i += kPeelBlock) {
        const int32_t d = dl[i];
        if (d <= level) {
          dl[i] = kGone;
          settled(i, level, pri);
          push(0, i);
        } else {
          mn = min(mn, (uint32_t)d);
        }
      }
      mn = wave_min(mn);
      if (lane_id() == 0) atomicMin(&sh.min_deg, mn);
      uint32_t fcnt = settle(), c = 0;
      if (!fcnt) {
        level = (int32_t)sh.min_deg - 1;
        __syncthreads();
        continue;
      }
      degen = (uint32_t)level;
      while (fcnt) {
        left -= fcnt;
        fcnt = round(fcnt, c, level, ++pri);
        c ^= 1u;
      }
    }
    if (t == 0) {
      b.st->level = level;
      b.st->round = pri;
      b.st->degeneracy = degen;
      b.st->mode = kModeDone;
    }
  }
};

// The whole peel of a graph of at most kTailMax vertices and kTailArcsEarly arcs
// (kAt kWholeRows: at most kTailRowsMax vertices).
template <int kAt>
__global__ __launch_bounds__(kPeelBlock) void kc_small(PeelBufs b) {
  extern __shared__ __align__(16) uint8_t smem[];
  PeelLds &sh = *(PeelLds *)smem;
  int32_t *dl = (int32_t *)(smem + sizeof(PeelLds));
  uint32_t *rows = (uint32_t *)(dl + kTailRowsMax);
  for (uint32_t i = threadIdx.x; i < b.n; i += kPeelBlock) {
    const uint64_t r0 = b.rp[i], r1 = b.rp[i + 1];
    dl[i] = (int32_t)(r1 - r0);
    if (kAt == kWholeRows) {
      rows[i] = (uint32_t)r0;
      if (i == b.n - 1) rows[b.n] = (uint32_t)r1;
    }
  }
  __syncthreads();
  Rounds<kAt>{b, sh, dl, rows, nullptr}.levels(b.n, b.n, -1, 0, 0);
}

// Before kc_tail, once few enough vertices and arcs are left at a level step
// (launches before that, and after the tail, do nothing): numbers the alive
// vertices, then lays the arcs between them out as 16-bit indices.
__device__ __forceinline__ bool tail_due(const PeelState *st) {
  return st->mode == kModeLevel && st->acnt <= kTailMax &&
         st->arcs <= (st->round < kTailRounds ? kTailArcsEarly : kTailArcs);
}
__global__ __launch_bounds__(kBlock) void kc_number(PeelBufs b) {
  if (!tail_due(b.st)) return;
  __shared__ uint32_t wsum[kBlock / kWave], base;
  const uint32_t *alive = b.st->alive_cur ? b.alive1 : b.alive0;
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x, wig = threadIdx.x / kWave;  // the grid covers kTailMax
  const bool valid = i < b.st->acnt;
  uint32_t d = 0;
  if (valid) {
    const uint32_t v = alive[i];
    // (the rounds since the level step may have removed it); an alive vertex's
    // degree is the number of its alive neighbours
    if (b.prio[v] == kNone) {
      b.loc[v] = i;
      d = (uint32_t)b.deg[v];
    }
  }
  uint32_t incl = d;
  for (uint32_t o = 1; o < kWave; o <<= 1) {
    const uint32_t y = (uint32_t)__shfl_up((int)incl, o);
    if (lane_id() >= o) incl += y;
  }
  if (lane_id() == kWave - 1) wsum[wig] = incl;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t acc = 0;
    for (uint32_t w = 0; w < kBlock / kWave; ++w) {
      const uint32_t x = wsum[w];
      wsum[w] = acc;
      acc += x;
    }
    base = acc ? atomicAdd(&b.st->taken, acc) : 0;
  }
  __syncthreads();
  if (valid) {
    b.trow[2 * i] = base + wsum[wig] + incl - d;
    b.trow[2 * i + 1] = d;
  }
}
__global__ __launch_bounds__(kBlock) void kc_compact(PeelBufs b) {
  PeelState *st = b.st;
  if (!tail_due(st)) return;
  const uint32_t *alive = st->alive_cur ? b.alive1 : b.alive0;
  const uint32_t waves = gridDim.x * (kBlock / kWave);
  for (uint32_t i = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave; i < st->acnt; i += waves) {
    if (b.trow[2 * i + 1] == 0) continue;
    const uint32_t v = alive[i];
    uint32_t at = b.trow[2 * i];
    const uint64_t r1 = b.rp[v + 1];
    for (uint64_t k0 = b.rp[v]; k0 < r1; k0 += kWave) {
      const uint64_t k = k0 + lane_id();
      const uint32_t l = k < r1 ? b.loc[b.ci[k]] : kNone;
      const uint64_t m = ballot(l != kNone);
      if (l != kNone) b.tarc[at + mbcnt(m)] = (uint16_t)l;
      at += popc64(m);
    }
  }
}

// The rest of the peel in one workgroup.
__global__ __launch_bounds__(kPeelBlock) void kc_tail(PeelBufs b) {
  extern __shared__ __align__(16) uint8_t smem[];
  PeelState *st = b.st;
  if (!tail_due(st)) return;
  PeelLds &sh = *(PeelLds *)smem;
  int32_t *dl = (int32_t *)(smem + sizeof(PeelLds));
  const uint32_t *alive = st->alive_cur ? b.alive1 : b.alive0;
  const uint32_t cnt = st->acnt, t = threadIdx.x;
  if (t == 0) sh.left = 0;
  __syncthreads();
  uint32_t mine = 0;
  for (uint32_t i = t; i < cnt; i += kPeelBlock) {
    const uint32_t v = alive[i];
    const bool in = b.prio[v] == kNone;
    dl[i] = in ? b.deg[v] : kGone;
    mine += in;
  }
  if (mine) atomicAdd(&sh.left, mine);
  __syncthreads();
  Rounds<kCore>{b, sh, dl, nullptr, alive}.levels(cnt, sh.left, st->level, st->round, st->degeneracy);
}

// One step of the peel of a large graph: the grid selects a level's frontier
// (and compacts the alive list) or runs one round with a large frontier; the
// last workgroup to finish advances the state and goes on alone with the
// level's rounds while their frontiers are small. Once the tail is due the
// launches leave the level step to kc_tail.
__global__ __launch_bounds__(kPeelBlock) void kc_iterate(PeelBufs b, uint32_t row) {
  extern __shared__ __align__(16) uint8_t smem[];
  PeelLds &sh = *(PeelLds *)smem;
  PeelState *st = b.st;
  const uint32_t mode = st->mode, round = st->round;
  if (mode == kModeDone || tail_due(st)) return;
  const uint32_t cur = st->cur, cnt = mode == kModeLevel ? st->acnt : st->fcnt;
  const int32_t L = mode == kModeLevel ? st->level + 1 : st->level;
  if (mode == kModeLevel) {
    const uint32_t ac = st->alive_cur;
    const uint32_t *src = ac ? b.alive1 : b.alive0;
    uint32_t *dst = ac ? b.alive0 : b.alive1;
    uint32_t *F = cur ? b.front1 : b.front0;
    const uint32_t stride = gridDim.x * blockDim.x, wig = threadIdx.x / kWave;
    unsigned long long arcs = 0;
    if (threadIdx.x == 0) sh.arcs = 0;
    // every lane of a workgroup runs the same number of iterations; one
    // append per list and iteration for the whole workgroup (appends of all
    // waves to two counters of one line took 11 ns each)
    for (uint32_t o = blockIdx.x * blockDim.x; o < cnt; o += stride) {
      const uint32_t i = o + threadIdx.x;
      uint32_t v = 0;
      bool alive = false, sel = false;
      if (i < cnt) {
        v = src[i];
        alive = b.prio[v] == kNone;
        const int32_t d = b.deg[v];
        sel = alive && d <= L;
        if (alive && !sel) arcs += (uint32_t)d;
      }
      const uint64_t ms = ballot(sel), mk = ballot(alive && !sel);
      if (lane_id() == 0) {
        sh.wsel[wig] = popc64(ms);
        sh.wkeep[wig] = popc64(mk);
      }
      __syncthreads();
      if (threadIdx.x == 0) {
        uint32_t s0 = 0, s1 = 0;
        for (uint32_t w = 0; w < kPeelBlock / kWave; ++w) {
          const uint32_t x = sh.wsel[w], y = sh.wkeep[w];
          sh.wsel[w] = s0;
          sh.wkeep[w] = s1;
          s0 += x;
          s1 += y;
        }
        sh.bsel = s0 ? atomicAdd(&st->fcnt, s0) : 0;
        sh.bkeep = s1 ? atomicAdd(&st->acnt2, s1) : 0;
      }
      __syncthreads();
      if (sel) {
        b.prio[v] = round;
        b.core[v] = (uint32_t)L;
        st_dev(&F[sh.bsel + sh.wsel[wig] + mbcnt(ms)], v);
      }
      if (alive && !sel) dst[sh.bkeep + sh.wkeep[wig] + mbcnt(mk)] = v;
      __syncthreads();
    }
    // (each lane's share cut to more than kTailArcs: the sum only has to show
    // whether it is above)
    const uint32_t wa = wave_sum((uint32_t)min(arcs, 2ull * kTailArcs));
    if (lane_id() == 0 && wa) atomicAdd(&sh.arcs, (unsigned long long)wa);
    __syncthreads();
    if (threadIdx.x == 0 && sh.arcs) atomicAdd(&st->arcs2, sh.arcs);
  } else {
    // appended vertices gather in LDS and leave with one append a workgroup
    const uint32_t *F = cur ? b.front1 : b.front0;
    uint32_t *N = cur ? b.front0 : b.front1;
    const uint32_t waves = gridDim.x * (blockDim.x / kWave);
    const uint32_t wid = blockIdx.x + gridDim.x * (threadIdx.x / kWave);
    if (threadIdx.x == 0) sh.ncnt = 0;
    __syncthreads();
    for (uint32_t i = wid; i < cnt; i += waves) {
      const uint32_t v = F[i];
      const uint64_t r1 = b.rp[v + 1];
      for (uint64_t k = b.rp[v] + lane_id(); k < r1; k += kWave) {
        const uint32_t w = b.ci[k];
        if (lower_dev(b.deg, w, L)) {
          b.prio[w] = round + 1;
          b.core[w] = (uint32_t)L;
          const uint32_t at = atomicAdd(&sh.ncnt, 1u);
          if (at < kFrontLds) sh.front[0][at] = w;
          else st_dev(&N[atomicAdd(&st->ncnt, 1u)], w);
        }
      }
    }
    __syncthreads();
    const uint32_t mine = min(sh.ncnt, kFrontLds);
    if (threadIdx.x == 0) sh.bsel = mine ? atomicAdd(&st->ncnt, mine) : 0;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < mine; i += kPeelBlock) st_dev(&N[sh.bsel + i], sh.front[0][i]);
  }
  // the last workgroup to finish goes on with what the others left: counters
  // (atomics) and the frontier, written and read with agent-scope stores and
  // loads that have completed here (a release fence instead would write the
  // L2 back, 40 us a launch with one from every wave)
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) sh.last = atomicAdd(&st->arrived, 1u) == gridDim.x - 1;
  __syncthreads();
  if (!sh.last) return;
  uint32_t r = round, c = cur, acnt = st->acnt, fcnt, degen = st->degeneracy;
  unsigned long long arcs = 0;
  if (mode == kModeLevel) {
    acnt = ld_dev(&st->acnt2);
    fcnt = ld_dev(&st->fcnt);
    if (fcnt) degen = (uint32_t)L;
    arcs = __hip_atomic_load(&st->arcs2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  } else {
    r += 1;
    c ^= 1u;
    fcnt = ld_dev(&st->ncnt);
  }
  // frontier vertices have about L alive neighbours each; rows of average
  // length stand for the removed ones
  const uint32_t fmax = min(kFrontLds, kFrontArcs / (L + row));
  const Rounds<kDev> R{b, sh, nullptr, nullptr, nullptr};
  if (fcnt && fcnt <= fmax) {
    const uint32_t *f0 = c ? b.front1 : b.front0;
    for (uint32_t i = threadIdx.x; i < fcnt; i += kPeelBlock) sh.front[c][i] = ld_dev(&f0[i]);
    __syncthreads();
    while (fcnt && fcnt <= fmax) {
      fcnt = R.round(fcnt, c, L, ++r);
      c ^= 1u;
    }
    // a frontier that grew goes back to the grid whole
    uint32_t *f1 = c ? b.front1 : b.front0;
    for (uint32_t i = threadIdx.x; i < min(fcnt, kFrontLds); i += kPeelBlock) f1[i] = sh.front[c][i];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (mode == kModeLevel) {
      st->level = L;
      st->alive_cur ^= 1u;
      st->acnt = acnt;
      st->acnt2 = 0;
      st->degeneracy = degen;
      st->arcs = arcs;
      st->arcs2 = 0;
    }
    st->round = r;
    st->cur = c;
    st->fcnt = fcnt;
    st->ncnt = 0;
    st->mode = fcnt ? kModePeel : acnt ? kModeLevel : kModeDone;
    st->arrived = 0;
  }
}

// Orientation: one wave per row, stable split into [earlier | later].
__global__ __launch_bounds__(kBlock) void orient_kernel(uint32_t n, const uint64_t *__restrict__ rp,
                                                        const uint32_t *__restrict__ ci,
                                                        const uint32_t *__restrict__ prio,
                                                        uint32_t *__restrict__ oc, uint64_t *__restrict__ split,
                                                        uint32_t *__restrict__ dplus, uint32_t *maxima) {
  const uint32_t waves = gridDim.x * (blockDim.x / kWave);
  const uint32_t wid = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
  uint32_t mdeg = 0, mout = 0, min_ = 0;
  for (uint32_t u = wid; u < n; u += waves) {
    const uint64_t b = rp[u], e = rp[u + 1];
    const uint32_t pu = prio[u];
    // rows of more than a wave's arcs: four a lane at a time, as a step waits
    // for the chain arc -> priority and a hub's row is thousands of arcs on
    // one wave (R-MAT 18, one and four arcs a lane: 1.04 and 0.75 ms)
    uint64_t sp;
    auto place = [&](auto arcs) {
      constexpr uint32_t kU = decltype(arcs)::value;
      uint32_t w[kU];
      bool later[kU];
      auto look = [&](uint64_t k0) {
#pragma unroll
        for (uint32_t m = 0; m < kU; ++m) {
          const uint64_t k = k0 + m * kWave + lane_id();
          w[m] = k < e ? ci[k] : u;
        }
#pragma unroll
        for (uint32_t m = 0; m < kU; ++m) {
          const uint32_t pw = prio[w[m]];
          later[m] = pw > pu || (pw == pu && w[m] > u);
        }
      };
      uint32_t late = 0;
      for (uint64_t k0 = b; k0 < e; k0 += kU * kWave) {
        look(k0);
#pragma unroll
        for (uint32_t m = 0; m < kU; ++m) late += popc64(ballot(later[m]));
      }
      sp = e - late;
      uint64_t we = b, wl = sp;
      for (uint64_t k0 = b; k0 < e; k0 += kU * kWave) {
        if (e - b > kU * kWave) look(k0);  // (else still there)
#pragma unroll
        for (uint32_t m = 0; m < kU; ++m) {
          const bool valid = k0 + m * kWave + lane_id() < e;
          const uint64_t be = ballot(valid && !later[m]), bl = ballot(later[m]);
          if (valid) {
            if (later[m]) oc[wl + mbcnt(bl)] = w[m];
            else oc[we + mbcnt(be)] = w[m];
          }
          we += popc64(be);
          wl += popc64(bl);
        }
      }
    };
    if (e - b > kWave) place(std::integral_constant<uint32_t, 4>{});
    else place(std::integral_constant<uint32_t, 1>{});
    const uint32_t early = (uint32_t)(sp - b);
    if (lane_id() == 0) {
      split[u] = sp;
      dplus[u] = (uint32_t)(e - sp);
    }
    mdeg = max(mdeg, (uint32_t)(e - b));
    mout = max(mout, (uint32_t)(e - sp));
    min_ = max(min_, early);
  }
  // one update per workgroup, and only of a maximum that it raises (an
  // update by every wave took 11 ns each on the one line)
  __shared__ uint32_t mx[3];
  if (threadIdx.x < 3) mx[threadIdx.x] = 0;
  __syncthreads();
  if (lane_id() == 0) {
    atomicMax(&mx[0], mdeg);
    atomicMax(&mx[1], mout);
    atomicMax(&mx[2], min_);
  }
  __syncthreads();
  if (threadIdx.x < 3 && mx[threadIdx.x] > ld_dev(&maxima[threadIdx.x])) atomicMax(&maxima[threadIdx.x], mx[threadIdx.x]);
}

// ---- heaviest-first counting sort of vertices with out-degree >= 1 --------
constexpr uint32_t kTile = 4096;

__global__ __launch_bounds__(kBlock) void sched_count(uint32_t n, const uint32_t *__restrict__ dplus,
                                                      const uint32_t *__restrict__ key, uint32_t kmax,
                                                      uint32_t *counts) {
  extern __shared__ uint32_t lh[];
  for (uint32_t i = threadIdx.x; i <= kmax; i += blockDim.x) lh[i] = 0;
  __syncthreads();
  const uint32_t t0 = blockIdx.x * kTile;
  for (uint32_t v = t0 + threadIdx.x; v < min(n, t0 + kTile); v += blockDim.x)
    if (dplus[v]) atomicAdd(&lh[min(key[v], kmax)], 1u);
  __syncthreads();
  for (uint32_t i = threadIdx.x; i <= kmax; i += blockDim.x)
    if (lh[i]) atomicAdd(&counts[i], lh[i]);
}

// start[k] = number of vertices with a larger key (descending order). One
// workgroup: thread t sums a run of keys, the runs' sums are scanned, and the
// run is walked again (one thread alone took 0.5 ms for the 4,096 keys of the
// learned schedule, a dependent load each).
constexpr uint32_t kScanThreads = 1024;
__global__ __launch_bounds__(kScanThreads) void sched_scan(uint32_t kmax, const uint32_t *__restrict__ counts,
                                                           uint32_t *__restrict__ start, uint32_t *total) {
  __shared__ uint32_t wsum[kScanThreads / kWave];
  const uint32_t kb = kmax + 1, run = (kb + kScanThreads - 1) / kScanThreads;
  // thread t walks positions [t * run, t * run + run) of the descending keys
  const uint32_t i0 = min(threadIdx.x * run, kb), i1 = min(i0 + run, kb);
  uint32_t own = 0;
  for (uint32_t i = i0; i < i1; ++i) own += counts[kmax - i];
  uint32_t incl = own;
  for (uint32_t d = 1; d < kWave; d <<= 1) {
    const uint32_t y = (uint32_t)__shfl_up((int)incl, d);
    if (lane_id() >= d) incl += y;
  }
  const uint32_t w = threadIdx.x / kWave;
  if (lane_id() == kWave - 1) wsum[w] = incl;
  __syncthreads();
  uint32_t acc = incl - own;
  for (uint32_t j = 0; j < w; ++j) acc += wsum[j];
  for (uint32_t i = i0; i < i1; ++i) {
    const uint32_t c = counts[kmax - i];
    start[kmax - i] = acc;
    acc += c;
  }
  if (threadIdx.x == kScanThreads - 1) *total = acc;
}

__global__ __launch_bounds__(kBlock) void sched_scatter(uint32_t n, const uint32_t *__restrict__ dplus,
                                                        const uint32_t *__restrict__ key, uint32_t kmax,
                                                        uint32_t *cursor, uint32_t *__restrict__ order) {
  extern __shared__ uint32_t lh[];
  uint32_t *base = lh + (kmax + 1);
  for (uint32_t i = threadIdx.x; i <= kmax; i += blockDim.x) lh[i] = 0;
  __syncthreads();
  const uint32_t t0 = blockIdx.x * kTile;
  for (uint32_t v = t0 + threadIdx.x; v < min(n, t0 + kTile); v += blockDim.x)
    if (dplus[v]) atomicAdd(&lh[min(key[v], kmax)], 1u);
  __syncthreads();
  for (uint32_t i = threadIdx.x; i <= kmax; i += blockDim.x) {
    base[i] = lh[i] ? atomicAdd(&cursor[i], lh[i]) : 0;
    lh[i] = 0;
  }
  __syncthreads();
  for (uint32_t v = t0 + threadIdx.x; v < min(n, t0 + kTile); v += blockDim.x)
    if (dplus[v]) {
      const uint32_t k = min(key[v], kmax);
      order[base[k] + atomicAdd(&lh[k], 1u)] = v;
    }
}

// ---- arc list for level-2 subproblems ------------------------------------
constexpr uint32_t kScanTile = 1024;

// Items per ordered vertex: its out-degree (one arc item per out-neighbour)
// when it is split (all vertices when `split_flag` is null), else one.
__global__ __launch_bounds__(kScanTile) void scan_tiles(uint32_t len, const uint32_t *__restrict__ order,
                                                        const uint32_t *__restrict__ dplus,
                                                        const uint8_t *__restrict__ split_flag, uint64_t *off,
                                                        uint64_t *tile_sums) {
  __shared__ uint64_t s[kScanTile];
  const uint32_t i = blockIdx.x * kScanTile + threadIdx.x;
  uint64_t x = 0;
  if (i < len) {
    const uint32_t v = order[i];
    x = (!split_flag || split_flag[v]) ? dplus[v] : 1;
  }
  s[threadIdx.x] = x;
  __syncthreads();
  for (uint32_t d = 1; d < kScanTile; d <<= 1) {
    const uint64_t y = threadIdx.x >= d ? s[threadIdx.x - d] : 0;
    __syncthreads();
    s[threadIdx.x] += y;
    __syncthreads();
  }
  if (i < len) off[i] = s[threadIdx.x] - x;  // exclusive within the tile
  if (threadIdx.x == kScanTile - 1) tile_sums[blockIdx.x] = s[threadIdx.x];
}

__global__ void scan_sums(uint32_t tiles, uint64_t *tile_sums, uint64_t *total) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  uint64_t acc = 0;
  for (uint32_t t = 0; t < tiles; ++t) {
    const uint64_t x = tile_sums[t];
    tile_sums[t] = acc;
    acc += x;
  }
  *total = acc;
}

__global__ __launch_bounds__(kBlock) void write_arcs(uint32_t len, const uint32_t *__restrict__ order,
                                                     const uint64_t *__restrict__ off,
                                                     const uint64_t *__restrict__ tile_sums,
                                                     const uint8_t *__restrict__ split_flag,
                                                     const uint64_t *__restrict__ split,
                                                     const uint64_t *__restrict__ rp,
                                                     const uint32_t *__restrict__ oc, uint2 *__restrict__ arcs) {
  const uint32_t waves = gridDim.x * (blockDim.x / kWave);
  const uint32_t wid = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
  for (uint32_t i = wid; i < len; i += waves) {
    const uint32_t u = order[i];
    const uint64_t o = off[i] + tile_sums[i / kScanTile];
    if (split_flag && !split_flag[u]) {
      if (lane_id() == 0) arcs[o] = make_uint2(u, 0xFFFFFFFFu);  // the whole vertex subproblem
      continue;
    }
    const uint64_t b = split[u], e = rp[u + 1];
    for (uint64_t k = b + lane_id(); k < e; k += kWave) arcs[o + (k - b)] = make_uint2(u, oc[k]);
  }
}

uint32_t grid_for(uint64_t work, uint32_t per_block, uint32_t cap) {
  const uint64_t g = (work + per_block - 1) / per_block;
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(g, cap));
}

}  // namespace

int hip_fail(hipError_t e, const char *what) {
  if (e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation)
    return set_error(MCE_ENOMEM, "%s: %s", what, hipGetErrorString(e));
  return set_error(MCE_EDEVICE, "%s: %s", what, hipGetErrorString(e));
}

int peel(const DevGraph &g, hipStream_t s, OrderInfo *info) {
  const uint32_t n = g.n;
  if (n == 0) {
    info->degeneracy = 0;
    info->rounds = 0;
    return MCE_OK;
  }
  PeelBufs b{};
  const bool small = n <= kTailMax && g.m <= kTailArcsEarly;
  const uint32_t row = (uint32_t)std::min<uint64_t>(std::max<uint64_t>(g.m / n, 1), 1u << 20);
  // frontiers, and for a large graph degrees, alive lists and tail numbering
  uint32_t *buf = nullptr;
  // (plain host memory: pinning and unpinning it is 65 us, its few copies are
  // 100 bytes)
  PeelState hst0{}, *hst = &hst0;
  int rc = MCE_OK;
  auto cleanup = [&]() {
    hipFree(buf);
  };
  const uint64_t words = (small ? 2ull * n : 6ull * n + 2 * kTailMax + kTailArcs / 2) + (sizeof(PeelState) + 15) / 16 * 4;
  if (hipMalloc(&buf, sizeof(uint32_t) * words) != hipSuccess) {
    cleanup();
    return set_error(MCE_ENOMEM, "peel: device allocation failed (n=%u)", n);
  }
  b.st = (PeelState *)buf;
  uint32_t *at = buf + (sizeof(PeelState) + 15) / 16 * 4;
  b.front0 = at;
  b.front1 = at + n;
  if (!small) {
    b.alive0 = at + 2ull * n;
    b.alive1 = at + 3ull * n;
    b.loc = at + 4ull * n;
    b.deg = (int32_t *)(at + 5ull * n);
    b.trow = at + 6ull * n;
    b.tarc = (uint16_t *)(b.trow + 2 * kTailMax);
  }
  b.rp = g.rp;
  b.ci = g.ci;
  b.prio = g.prio;
  b.core = g.core;
  b.n = n;
  auto *whole = n <= kTailRowsMax ? kc_small<kWholeRows> : kc_small<kWhole>;
  hipError_t e = hipFuncSetAttribute((const void *)(small ? whole : kc_tail), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)kTailLds);
  if (e == hipSuccess) {
    if (small) hipLaunchKernelGGL(whole, dim3(1), dim3(kPeelBlock), kTailLds, s, b);
    else kc_init<<<grid_for(n, kBlock, 4096), kBlock, 0, s>>>(b);
    const uint32_t grid = std::max(kPeelGridMin, grid_for(n, kPeelGridVerts, kPeelGridMax));
    uint32_t batch = 16;
    for (uint64_t it = 0;; it += batch) {
      if (!small) {
        for (uint32_t k = 0; k < batch; ++k) kc_iterate<<<grid, kPeelBlock, kPeelLds, s>>>(b, row);
        kc_number<<<kTailMax / kBlock, kBlock, 0, s>>>(b);
        kc_compact<<<1024, kBlock, 0, s>>>(b);
        kc_tail<<<1, kPeelBlock, kTailLds, s>>>(b);
      }
      e = hipMemcpyAsync(hst, b.st, sizeof(PeelState), hipMemcpyDeviceToHost, s);
      if (e == hipSuccess) e = hipStreamSynchronize(s);
      if (e != hipSuccess || hst->mode == kModeDone) break;
      if (small || it > 4ull * n + 64) {
        rc = set_error(MCE_EINTERNAL, "peel did not terminate");
        break;
      }
      batch = std::min<uint32_t>(batch * 2, 128);
    }
  }
  if (e != hipSuccess) {
    cleanup();
    return hip_fail(e, "peel");
  }
  info->degeneracy = hst->degeneracy;
  info->rounds = hst->round;
  info->n_rounds = hst->round;
  cleanup();
  return rc;
}

int orient(DevGraph &g, hipStream_t s, OrderInfo *info) {
  uint32_t *maxima = nullptr;
  MCE_HIP(hipMalloc(&maxima, 3 * sizeof(uint32_t)));
  MCE_HIP(hipMemsetAsync(maxima, 0, 3 * sizeof(uint32_t), s));
  if (g.n) {
    const uint32_t grid = grid_for((uint64_t)g.n * kWave, kBlock, 8192);
    orient_kernel<<<grid, kBlock, 0, s>>>(g.n, g.rp, g.ci, g.prio, g.oc, g.split, g.dplus, maxima);
  }
  uint32_t h[3];
  MCE_HIP(hipMemcpyAsync(h, maxima, sizeof(h), hipMemcpyDeviceToHost, s));
  MCE_HIP(hipStreamSynchronize(s));
  hipFree(maxima);
  info->max_degree = h[0];
  info->max_out_degree = h[1];
  info->max_in_degree = h[2];
  return MCE_OK;
}

int schedule_by_key(const DevGraph &g, const uint32_t *key, uint32_t key_max, uint32_t *order,
                    uint32_t *len_out, hipStream_t s, Scratch *sc) {
  *len_out = 0;
  if (g.n == 0) return MCE_OK;
  uint32_t *buf = nullptr;
  const uint32_t kb = key_max + 1;
  if (sc) {
    buf = (uint32_t *)sc->take(sizeof(uint32_t) * (2 * kb + 1));
    if (!buf) return set_error(MCE_ELIMIT, "scratch too small for the schedule's %u key bins", kb);
  } else {
    MCE_HIP(hipMalloc(&buf, sizeof(uint32_t) * (2 * kb + 1)));
  }
  uint32_t *counts = buf, *cursor = buf + kb, *total = buf + 2 * kb;
  MCE_HIP(hipMemsetAsync(buf, 0, sizeof(uint32_t) * (2 * kb + 1), s));
  const uint32_t tiles = (g.n + kTile - 1) / kTile;
  const size_t lds1 = sizeof(uint32_t) * kb, lds2 = 2 * lds1;
  sched_count<<<tiles, kBlock, lds1, s>>>(g.n, g.dplus, key, key_max, counts);
  sched_scan<<<1, kScanThreads, 0, s>>>(key_max, counts, cursor, total);
  sched_scatter<<<tiles, kBlock, lds2, s>>>(g.n, g.dplus, key, key_max, cursor, order);
  MCE_HIP(hipMemcpyAsync(len_out, total, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
  MCE_HIP(hipStreamSynchronize(s));
  if (!sc) hipFree(buf);
  return MCE_OK;
}

int arcs_from_order(const DevGraph &g, const uint32_t *order, uint32_t len, const uint8_t *split_flag,
                    uint2 **arcs_out, uint64_t *n_arcs, hipStream_t s) {
  *arcs_out = nullptr;
  *n_arcs = 0;
  if (len == 0) return MCE_OK;
  const uint32_t tiles = (len + kScanTile - 1) / kScanTile;
  uint64_t *off = nullptr, *sums = nullptr;
  MCE_HIP(hipMalloc(&off, sizeof(uint64_t) * len));
  MCE_HIP(hipMalloc(&sums, sizeof(uint64_t) * (tiles + 1)));
  scan_tiles<<<tiles, kScanTile, 0, s>>>(len, order, g.dplus, split_flag, off, sums);
  scan_sums<<<1, 1, 0, s>>>(tiles, sums, sums + tiles);
  uint64_t total = 0;
  MCE_HIP(hipMemcpyAsync(&total, sums + tiles, sizeof(uint64_t), hipMemcpyDeviceToHost, s));
  MCE_HIP(hipStreamSynchronize(s));
  uint2 *arcs = nullptr;
  if (total) {
    MCE_HIP(hipMalloc(&arcs, sizeof(uint2) * total));
    write_arcs<<<grid_for((uint64_t)len * kWave, kBlock, 8192), kBlock, 0, s>>>(len, order, off, sums, split_flag,
                                                                                   g.split, g.rp, g.oc, arcs);
  }
  MCE_HIP(hipStreamSynchronize(s));
  hipFree(off);
  hipFree(sums);
  *arcs_out = arcs;
  *n_arcs = total;
  return MCE_OK;
}

}  // namespace mce

// Bron-Kerbosch with pivoting on gfx950: one wave64 per subproblem, with an
// optional worker list that moves subtrees from busy waves to idle ones.
//
// Semantics follow the reference (yen-hsiang-chang/mce-gpu):
//   L1 subproblem of vertex v: R = {v}, P = N+(v), X = N-(v)
//       (mce/mce_kernel_nowl.cuh:45-108, setup mce/mce_utils.cuh:565-611);
//   L2 subproblem of arc u->w: R = {u, w}, P = N+(u) & N+(w), X = N(u) & N-(w);
//       an arc with P and X empty is a maximal clique (nowl.cuh:250-307);
//   pivot = argmax |P & N(u)| over u in P, the X vertices inside the induced
//   subgraph and (IPX) the X rows outside it; an X vertex that covers P ends
//   the branch (mce/mce_utils.cuh:338-472); a leaf with P and X empty is a
//   maximal clique (mce/mce_utils.cuh:507-524); IP tests outside-X vertices
//   by binary search of N-(c) (mce/mce_utils.cuh:265-292), IPX by a bit of
//   their bitmap row (mce/mce_utils.cuh:294-319);
//   worker list: idle workers receive subtrees from busy ones once the
//   first-level work is gone (mce/mce_utils.cuh:241-263, :861-1217).
//
// Design (not the reference's): the induced subgraph over a sorted vertex set
// S is a |S| x W bit matrix of 64-bit words (W = ceil(|S|/64)); the sets P, X
// and the branch mask live one word per lane (lane k holds word k) in
// registers, so intersections, emptiness tests and next-candidate search are
// single wave instructions plus a ballot, with no workgroup barriers on the
// hot loop. Pivot scores run one candidate row per lane. A subproblem's arena
// (S, the matrix, the outside-X rows and lists, the hash terms, the first
// stack frames) comes from its workgroup's LDS pool when the pool has room and
// from the wave's HBM arena otherwise; deeper frames spill to HBM. Tie-breaks
// are deterministic (lowest index, outside-X rows by vertex id), so the tree
// is reproducible, matches the CPU oracle node for node, and a donated
// subtree expands exactly as it would have in the donor.
//
// Worker list: an idle wave puts its id on a bounded lock-free queue in HBM
// (per-slot sequence numbers; what one wave hands another, on any XCD, goes
// through agent-scope stores and loads, never through fences) and waits on
// its own mailbox line.
// A busy wave whose task has run long enough takes an idle wave off the queue
// and writes into that wave's task slot the next candidate of its shallowest
// frame (the largest remaining subtree): its P and X words, the donor's vertex
// set and bit matrix, and the outside-X rows that survive. The receiver
// copies them into its own arena and continues in the donor's index space, so
// no arena is ever shared and nothing is rebuilt. A counter of outstanding
// work (tickets + handed-over tasks) ends the kernel exactly; a realtime
// watchdog turns any termination bug into an error flag instead of a hang.
#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <chrono>
#include <thread>
#include <vector>

#include "engine.hpp"
#include "internal.hpp"
#include "layout.hpp"
#include "lists.hpp"
#include "rng.hpp"
#include "wave.hpp"

namespace mce {

namespace {

enum Acc : uint32_t {
  kAccCount = 0,
  kAccHash,
  kAccNodes,
  kAccDonations,
  kAccOverflow,
  kAccMaxSize,
  kAccError,
  kAccN
};

// Kernel instances: no statistics, the three eval variants, and no
// statistics with the lane solver compiled in (kept out of the other
// instances, whose register allocation it would otherwise share).
enum Stat : int { kStatNone = 0, kStatLb = 1, kStatDonor = 2, kStatBd = 3, kStatLane = 4 };
// Kernel instances that solve in functions of their own (see "functions of
// their own" below): those of the bitmap path without statistics. The IP
// instances only have the list path, whose code stays in the kernel.
constexpr bool fn_of(bool ipx, int stat) { return ipx && (stat == kStatNone || stat == kStatLane); }
constexpr bool lane_of(int stat) { return stat == kStatLane; }
enum Bd : int { kBdOther = 0, kBdInduced, kBdQueue, kBdPivot, kBdSetOps, kBdMaximal, kBdBranch };

// One idle queue per XCD (its head and tail each on a line of their own from
// word kCtlQueues + 16q), so that donors and idle waves of different XCDs do
// not contend for one line.
constexpr uint32_t kQueues = 8;
// Word kCtlProgress (a line of its own) counts heartbeats of busy waves.
constexpr unsigned long long kMboxTask = 1, kMboxDone = 2;
constexpr uint32_t kCtlProgress = 0, kCtlOutstanding = 16, kCtlQueues = 32, kCtlWords = kCtlQueues + 16 * kQueues;
// Mailbox words of the waves, each on its own 128-byte line.
constexpr uint32_t kMboxStride = 16;
constexpr unsigned long long kNoSlot = ~0ull;
constexpr uint32_t kSlotHeader = 64;  // bytes
// Launch shape of the enumeration kernel: at most 12 waves per workgroup, 4
// waves per SIMD (128 VGPRs), for every variant. Measured alternatives for the
// worker-list variants, which spill at 128 VGPRs: 2 waves per SIMD (256
// VGPRs, no spill) took Chung-Lu 2^18 from 353 to 207 ms but 2^20 from 15.2
// to 22.2 s, 3 waves per SIMD gave 250 ms and 17.2 s; on heavy tails the
// number of waves that can take donated work counts for more than their speed.
constexpr uint32_t max_wpg_of(bool) { return 12u; }
constexpr uint32_t waves_per_simd_of(bool) { return 4u; }
enum TaskKind : uint32_t { kTaskList = 0, kTaskBits = 1 };
// Idle waves watch for global progress (a change of the outstanding-work
// count or of the busy waves' heartbeat counter); after this many 100 MHz
// realtime ticks without any they report a termination failure and exit
// (default 120 s; BkParams::watchdog_ticks overrides it). A busy wave beats
// once per kBeatNodes tree nodes.
// HBM arena a wave up to which arenas are sized by the degree maxima
constexpr uint64_t kSmallNeed = 16 << 10;
constexpr uint64_t kWatchdogTicks = 12000000000ull;
constexpr uint64_t kBeatNodes = 1u << 16;

struct BkParams {
  const uint64_t *rp;
  const uint32_t *ci;
  const uint32_t *oc;
  const uint64_t *split;
  const void *items;
  uint64_t n_items;
  uint32_t *ticket;
  uint64_t t1;     // tickets below t1 carry one item each
  uint32_t chunk;  // later tickets carry `chunk` items
  uint32_t level;
  uint32_t pool_bytes;  // LDS pool shared by the waves of a workgroup
  uint32_t stack_lds;   // most BK frames kept in LDS (0 = as many as fit)
  uint32_t want_levels; // frame levels a subproblem asks the pool for
  uint8_t *hbm;        // per-wave HBM arenas
  uint64_t hbm_bytes;
  unsigned long long *acc;
  unsigned long long *hist;
  uint32_t hist_len;
  uint32_t hist_lds;  // histogram bins cached in LDS per workgroup
  unsigned long long *sub_nodes;
  unsigned long long *sub_cliques;
  uint64_t *overflow;  // items that need a larger arena
  uint64_t overflow_cap;
  unsigned long long *wave_val;  // per-wave statistic
  uint32_t *wave_cu;
  unsigned long long *wave_bd;  // 7 cycle counters per wave
  uint32_t wpg;                 // waves per workgroup
  // worker list
  unsigned long long *ctl;
  unsigned long long *seq;
  uint8_t *ring;           // task slots, one per wave
  uint32_t ring_cap;       // idle-queue capacity (= waves)
  uint32_t *idle_ids;      // idle queue entries: wave ids
  unsigned long long *mbox;  // per-wave mailbox: kMboxTask once a task is in the wave's slot, kMboxDone at the end
  uint64_t slot_bytes;       // task slot per wave (pr.ring + wave * slot_bytes)
  uint32_t slot_pmax;  // largest donor |S|
  uint32_t slot_wmax;
  uint32_t slot_xcap;  // largest outside-X list carried
  uint32_t slot_oP, slot_oS, slot_oA, slot_oXI, slot_oXR;  // byte offsets in a slot
  uint32_t donate_min_p;
  uint32_t donate_check;
  uint64_t donate_age;  // 100 MHz realtime ticks a task runs before it may donate
  uint64_t poll_ticks;  // realtime ticks between looks at the idle queues
  uint32_t small_max;   // nodes with P + X + outside rows <= this go to the small-universe solver
  uint32_t small_pmax;  // ... and, with the worker list, |P| <= this
  uint64_t watchdog_ticks;  // idle time without global progress before the kernel gives up
  // pinned host words the kernel mirrors its progress into while it runs
  // (word 0: a recent ticket claimed, word 1: heartbeats); nullable
  unsigned long long *host_progress;
  // lane solver (ls_max = 0: off): largest member count, the waves' regions
  uint32_t ls_max;
  uint32_t ls_off;  // byte offsets of the waves' LDS parts: found cliques, hand-over blocks
  uint32_t io_off;
  uint8_t *ls;
  uint64_t *cover;  // hub row filter: 64 words per wave
};

// The workgroup's histogram bins in LDS, typed as such.
typedef __attribute__((address_space(3))) unsigned long long lds_ull;

// Posts a progress value to pinned host memory (a system-scope vector store;
// the host polls it while the persistent launch holds every CU, when a copy
// from device memory could not be scheduled).
__device__ __forceinline__ void post_progress(unsigned long long *p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

struct Sub {
  uint32_t *S;
  uint64_t *A;
  uint64_t *XR;
  uint64_t *H;  // bitmap path: splitmix64(S[i]), the clique-hash term of S[i]
  uint32_t *XL;
  uint32_t *XA;
  uint32_t *XV;  // IPX: vertex id of each outside-X row
  uint8_t *fr_lds;
  uint8_t *fr_hbm;
  uint32_t lds_levels;
  uint32_t FS;
  uint32_t p, W, q, xe0;
  uint32_t WX;  // bitmap path: words of the outside-X row bitmap
  uint32_t where;  // bitmap path: bit 0 S and A in LDS, bit 1 outside rows in LDS
  uint32_t rsize;
  uint32_t root;  // first-level vertex the subproblem belongs to
  uint64_t rmix;
  const uint32_t *oc;
  const uint64_t *rp;
  const uint64_t *split;
  uint64_t *cover;  // hub row filter: the wave's 64 union words (device memory)
  uint64_t t0;      // realtime at which the subproblem was taken up
};

struct WaveAcc {
  uint64_t count = 0, hash = 0, nodes = 0, donations = 0;
  uint32_t max_size = 0;
  uint64_t sub_cliques = 0;
  int32_t budget = 0;
  uint64_t last_poll = 0;  // nodes at the last poll
  uint64_t next_poll = 0;  // realtime before which the idle queues are not looked at
  uint64_t poll_wait = 1;
  uint64_t last_beat = 0;  // tree nodes (lane solver's included) at the last heartbeat
  uint32_t xq = 0;      // this wave's idle queue (its XCD)
  uint32_t peek = 0;    // another queue sampled at the next poll
  uint64_t t_task = 0;  // realtime at the start of the current task
  // lane solver: queued subtrees, the most P and X members among them, this
  // wave's region; what its runs found (their labels go to the subtrees'
  // roots, so they stay out of the running subproblem's counts)
  uint32_t ls_n = 0, ls_p = 0, ls_x = 0, ls_lds = 0;
  uint32_t io = 0;  // LDS address of the wave's hand-over block
  uint8_t *ls = nullptr;
  uint64_t ls_nodes = 0, ls_count = 0;
};

typedef const __attribute__((address_space(4))) BkParams ConstParams;
template <int kStat>
struct Clock {
  uint64_t acc[7];
  uint64_t last;
  int cur;
  __device__ __forceinline__ void start() {
    if constexpr (kStat == kStatBd) {
      for (int i = 0; i < 7; ++i) acc[i] = 0;
      last = __builtin_amdgcn_s_memtime();
      cur = kBdOther;
    }
  }
  __device__ __forceinline__ void to(int c) {
    if constexpr (kStat == kStatBd) {
      const uint64_t t = __builtin_amdgcn_s_memtime();
      acc[cur] += t - last;
      last = t;
      cur = c;
    }
  }
};


// All-ones P over the first p bits (lane k holds word k).
__device__ __forceinline__ uint64_t full_word(uint32_t p) {
  const uint32_t L = lane_id(), W = (p + 63) / 64;
  if (L >= W) return 0;
  return (L == W - 1 && (p & 63)) ? ((1ull << (p & 63)) - 1) : ~0ull;
}

// Words handed from one wave to another, on any XCD: agent-scope stores and
// loads, which go past the caches that are not shared, so that no fence is
// needed around them. An agent-scope release writes the whole L2 of the XCD
// back and an acquire empties the caches under the waves still at work: with
// them a hand-over cost 1.7 us of the whole launch (R-MAT 13, IP, donating at
// 10 us: 69,000 donations in 130 ms). Without them, default settings: R-MAT 13
// IP 13.3 -> 6.9 ms, Chung-Lu 30,011 11.1 -> 4.1, R-MAT 14 40.8 -> 29.6,
// Chung-Lu 2^18 121 -> 111.
template <class T>
__device__ __forceinline__ void st_shared(T *p, T v) {
  __hip_atomic_store((__attribute__((address_space(1))) T *)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ T ld_shared(const T *p) {
  return __hip_atomic_load((__attribute__((address_space(1))) T *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// This wave's earlier stores have reached their scope and its loads have
// returned; the compiler moves no access across.
__device__ __forceinline__ void drain() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Forward wave copies, four loads in flight per lane; each chunk of 256
// elements is read before it is written, so a destination below an
// overlapping source is safe. kOut / kIn: the destination / source is a task
// slot (st_shared, ld_shared).
template <class T, bool kOut, bool kIn>
__device__ __forceinline__ void wave_copy_t(T *dst, const T *src, uint64_t n) {
  const uint32_t L = lane_id();
  auto get = [&](uint64_t i) -> T {
    if constexpr (kIn) return i < n ? ld_shared(src + i) : T(0);
    else return i < n ? src[i] : T(0);
  };
  auto put = [&](uint64_t i, T x) {
    if (i >= n) return;
    if constexpr (kOut) st_shared(dst + i, x);
    else dst[i] = x;
  };
  for (uint64_t b = 0; b < n; b += 4 * kWave) {
    const uint64_t i0 = b + L, i1 = i0 + kWave, i2 = i1 + kWave, i3 = i2 + kWave;
    const T x0 = get(i0), x1 = get(i1), x2 = get(i2), x3 = get(i3);
    put(i0, x0);
    put(i1, x1);
    put(i2, x2);
    put(i3, x3);
  }
}
template <bool kOut = false, bool kIn = false>
__device__ __forceinline__ void wave_copy(uint32_t *dst, const uint32_t *src, uint32_t n) {
  wave_copy_t<uint32_t, kOut, kIn>(dst, src, n);
}
template <bool kOut = false, bool kIn = false>
__device__ __forceinline__ void copy64(uint64_t *dst, const uint64_t *src, uint64_t n) {
  wave_copy_t<uint64_t, kOut, kIn>(dst, src, n);
}

// Typed arena accesses: kL picks LDS (ds_*) over global memory (global_*).
// Arena pointers are generic because a subproblem's placement is chosen at
// run time; the bitmap solver is instantiated per placement so that its hot
// loop issues the instruction of the memory it touches instead of flat_*
// (which waits on both the LDS and the vector-memory counters).
typedef __attribute__((address_space(3))) uint64_t lds_u64;
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(1))) unsigned long long glb_ull;
typedef __attribute__((address_space(1))) uint64_t glb_u64;
typedef __attribute__((address_space(1))) uint32_t glb_u32;

template <bool kL>
__device__ __forceinline__ uint64_t ld64(const uint64_t *p, uint64_t i) {
  if constexpr (kL) return ((const lds_u64 *)p)[i];
  else return ((const glb_u64 *)p)[i];
}
template <bool kL>
__device__ __forceinline__ uint32_t ld32(const uint32_t *p, uint64_t i) {
  if constexpr (kL) return ((const lds_u32 *)p)[i];
  else return ((const glb_u32 *)p)[i];
}
template <bool kL>
__device__ __forceinline__ void or64(uint64_t *p, uint64_t i, uint64_t v) {
  if constexpr (kL) __hip_atomic_fetch_or((lds_ull *)p + i, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  else __hip_atomic_fetch_or((glb_ull *)p + i, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool kL>
__device__ __forceinline__ void st64(uint64_t *p, uint64_t i, uint64_t v) {
  if constexpr (kL) ((lds_u64 *)p)[i] = v;
  else ((glb_u64 *)p)[i] = v;
}
template <bool kL>
__device__ __forceinline__ void st32(uint32_t *p, uint64_t i, uint32_t v) {
  if constexpr (kL) ((lds_u32 *)p)[i] = v;
  else ((glb_u32 *)p)[i] = v;
}

__device__ __forceinline__ uint8_t *frame_at(const Sub &s, uint32_t d) {
  return d < s.lds_levels ? s.fr_lds + (uint64_t)d * s.FS : s.fr_hbm + (uint64_t)(d - s.lds_levels) * s.FS;
}

// Lays out the list-path arena for bounds (p, q, W) over an LDS region and
// the wave's HBM arena. Returns false when the HBM arena is too small.
__device__ __forceinline__ bool place(Sub &s, uint32_t p, uint32_t q, uint32_t W, bool ipx, uint8_t *lds, uint32_t lds_bytes,
                      uint8_t *hbm, uint64_t hbm_bytes, uint32_t stack_lds = 0) {
  uint32_t levels = 0;
  bool in_lds = false;
  if (list_hbm_need(p, q, W, ipx, lds_bytes, stack_lds, &levels, &in_lds) > hbm_bytes) return false;
  const uint64_t fixed = fixed_bytes(p, q, W, ipx);
  uint8_t *base = in_lds ? lds : hbm;
  s.fr_lds = in_lds ? lds + fixed : lds;
  s.fr_hbm = in_lds ? hbm : hbm + fixed;
  s.lds_levels = levels;
  s.FS = list_fs(W);
  uint64_t o = 0;
  s.S = (uint32_t *)(base + o);
  o += align8(4ull * p);
  s.A = (uint64_t *)(base + o);
  o += 8ull * p * W;
  s.XR = (uint64_t *)(base + o);
  if (ipx) o += 8ull * q * W;
  s.XV = (uint32_t *)(base + o);
  if (ipx) o += align8(4ull * q);
  s.XL = (uint32_t *)(base + o);
  o += align8(4ull * q);
  s.XA = (uint32_t *)(base + o);
  return true;
}

// Workgroup LDS pool: granules of kGranule bytes handed to waves for the
// lifetime of one subproblem, first fit, under a workgroup spin lock held by
// lane 0 of the asking wave. A wave never waits for LDS while holding any, so
// the lock is the only wait and every holder runs to release.
constexpr uint32_t kGranule = 512;
constexpr uint32_t kPoolWords = 5;  // up to 320 granules (160 KiB)
constexpr uint32_t kPoolHeader = 64;

struct Pool {
  uint64_t *mask;  // bit set: granule taken (bits past ngran stay set)
  uint32_t *lock;
  uint8_t *base;
  uint32_t ngran;
};

struct Region {
  uint8_t *ptr;
  uint32_t bytes;
  uint32_t g0, gk;
};

__device__ __forceinline__ void pool_lock(uint32_t *lock) {
  while (true) {
    uint32_t e = 0;
    if (__hip_atomic_compare_exchange_strong(lock, &e, 1u, __ATOMIC_ACQUIRE, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_WORKGROUP))
      return;
    __builtin_amdgcn_s_sleep(1);
  }
}

__device__ __forceinline__ void pool_unlock(uint32_t *lock) {
  __hip_atomic_store(lock, 0u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// First run of k clear bits, or kNone.
__device__ __forceinline__ uint32_t pool_find(const Pool &pl, uint32_t k) {
  if (k == 0 || k > pl.ngran) return kNone;
  uint32_t i = 0;
  while (i + k <= pl.ngran) {
    uint32_t w = i >> 6;
    uint64_t x = ~pl.mask[w] & (~0ull << (i & 63));
    while (!x) {
      if (++w >= kPoolWords) return kNone;
      x = ~pl.mask[w];
    }
    i = w * 64 + ctz64(x);
    if (i + k > pl.ngran) return kNone;
    uint64_t y = pl.mask[w] & (~0ull << (i & 63));
    while (!y && ++w < kPoolWords) y = pl.mask[w];
    const uint32_t j = y ? w * 64 + ctz64(y) : kPoolWords * 64;
    if (j - i >= k) return i;
    i = j;
  }
  return kNone;
}

__device__ __forceinline__ void pool_mark(const Pool &pl, uint32_t i, uint32_t k, bool set) {
  while (k) {
    const uint32_t w = i >> 6, b = i & 63, n = min(k, 64u - b);
    const uint64_t m = (n == 64 ? ~0ull : ((1ull << n) - 1)) << b;
    pl.mask[w] = set ? (pl.mask[w] | m) : (pl.mask[w] & ~m);
    i += n;
    k -= n;
  }
}

// The largest of want, mid, low (bytes, tried in that order) that fits now;
// an empty region when none does.
__device__ __forceinline__ Region pool_take(const Pool &pl, uint32_t want, uint32_t mid, uint32_t low) {
  uint32_t g0 = kNone, gk = 0;
  if (lane_id() == 0) {
    pool_lock(pl.lock);
    const uint32_t k1 = (uint32_t)min<uint64_t>(((uint64_t)want + kGranule - 1) / kGranule, 0xFFFFu);
    const uint32_t k2 = (uint32_t)min<uint64_t>(((uint64_t)mid + kGranule - 1) / kGranule, 0xFFFFu);
    const uint32_t k3 = (uint32_t)min<uint64_t>(((uint64_t)low + kGranule - 1) / kGranule, 0xFFFFu);
    uint32_t g = kNone, k = 0;
    if (k1) g = pool_find(pl, k = k1);
    if (g == kNone && k2) g = pool_find(pl, k = k2);
    if (g == kNone && k3) g = pool_find(pl, k = k3);
    if (g != kNone) {
      pool_mark(pl, g, k, true);
      g0 = g;
      gk = k;
    }
    pool_unlock(pl.lock);
  }
  Region r;
  r.g0 = uniform(g0);
  r.gk = uniform(gk);
  r.ptr = pl.base + (r.gk ? (uint64_t)r.g0 * kGranule : 0);
  r.bytes = r.gk * kGranule;
  return r;
}

__device__ __forceinline__ void pool_give(const Pool &pl, const Region &r) {
  if (r.gk && lane_id() == 0) {
    pool_lock(pl.lock);
    pool_mark(pl, r.g0, r.gk, false);
    pool_unlock(pl.lock);
  }
}

// pool_take that waits (up to about a millisecond) for at least `need` bytes
// when the pool could hold them: a subproblem run from HBM costs far more
// than the wait, and the waves holding LDS never wait, so space comes free.
__device__ __forceinline__ Region pool_take_wait_in(const Pool &pl, uint32_t want, uint32_t mid, uint32_t low,
                                                 uint32_t need) {
  Region r = pool_take(pl, want, mid, low);
  if (r.bytes >= need || need > pl.ngran * kGranule) return r;
  uint32_t backoff = 1;
  for (uint32_t t = 0; t < 24; ++t) {
    pool_give(pl, r);
    for (uint32_t z = 0; z < backoff; ++z) __builtin_amdgcn_s_sleep(32);
    backoff = min(backoff * 2, 32u);
    r = pool_take(pl, want, mid, low);
    if (r.bytes >= need) return r;
  }
  return r;
}
// Both also as functions, for the kernel's many places (the search for a run
// of free granules alone is inlined six times in a taking); mask: the LDS
// address of the pool's words.
typedef __attribute__((address_space(3))) uint8_t lds_u8;
__device__ __forceinline__ Pool pool_at(uint32_t mask, uint32_t ngran) {
  uint8_t *at = (uint8_t *)(lds_u8 *)(uintptr_t)uniform(mask);
  Pool pl;
  pl.mask = (uint64_t *)at;
  pl.lock = (uint32_t *)(at + 8 * kPoolWords);
  pl.base = at + kPoolHeader;
  pl.ngran = uniform(ngran);
  return pl;
}
__device__ __noinline__ __attribute__((not_tail_called)) uint64_t pool_take_fn(uint32_t mask, uint32_t ngran, uint32_t want,
                                                                               uint32_t mid, uint32_t low, uint32_t need) {
  const Region r =
      pool_take_wait_in(pool_at(mask, ngran), uniform(want), uniform(mid), uniform(low), uniform(need));
  return (uint64_t)r.gk << 32 | r.g0;
}
__device__ __noinline__ __attribute__((not_tail_called)) void pool_put_fn(uint32_t mask, uint32_t ngran, uint32_t g0,
                                                                          uint32_t gk) {
  pool_give(pool_at(mask, ngran), Region{nullptr, 0, uniform(g0), uniform(gk)});
}
template <bool kFn>
__device__ __forceinline__ Region pool_take_wait(const Pool &pl, uint32_t want, uint32_t mid, uint32_t low,
                                                 uint32_t need) {
  if constexpr (!kFn) return pool_take_wait_in(pl, want, mid, low, need);
  const uint64_t got = uniform64(pool_take_fn((uint32_t)(uintptr_t)pl.mask, pl.ngran, want, mid, low, need));
  Region r;
  r.g0 = (uint32_t)got;
  r.gk = (uint32_t)(got >> 32);
  r.ptr = pl.base + (r.gk ? (uint64_t)r.g0 * kGranule : 0);
  r.bytes = r.gk * kGranule;
  return r;
}
template <bool kFn>
__device__ __forceinline__ void pool_put(const Pool &pl, const Region &r) {
  if constexpr (!kFn) pool_give(pl, r);
  else if (r.gk) pool_put_fn((uint32_t)(uintptr_t)pl.mask, pl.ngran, r.g0, r.gk);
}

__device__ __forceinline__ const uint64_t *row_of(const Sub &s, uint32_t piv) {
  return piv < s.p ? s.A + (uint64_t)piv * s.W : s.XR + (uint64_t)(piv - s.p) * s.W;
}

// Pivot: max |P & N(u)| over u in P|X (bit order), then outside-X rows (IPX).
// Ties go to the lowest index, and every inside vertex precedes every outside
// row; outside rows tie-break by vertex id. Uniform outputs.
template <bool kIPX>
__device__ __forceinline__ void pick_pivot(const Sub &s, uint64_t Pw, uint64_t Xw, uint32_t xe_len, uint32_t &piv,
                                           uint32_t &best) {
  const uint32_t L = lane_id(), W = s.W;
  uint32_t bs = 0, bk = kNone, brow = 0;
  const uint64_t C = Pw | Xw;
  for (uint32_t k = 0; k < W; ++k) {
    const uint64_t ck = rdlane64(C, k);
    if (ck == 0) continue;
    if ((ck >> L) & 1ull) {
      const uint32_t u = k * 64 + L;
      const uint64_t *row = s.A + (uint64_t)u * W;
      uint32_t sc = 0;
      for (uint32_t j = 0; j < W; ++j) sc += popc64(rdlane64(Pw, j) & row[j]);
      if (bk == kNone || sc > bs) {
        bs = sc;
        bk = u;
      }
    }
  }
  if (kIPX) {
    for (uint32_t b = 0; b < xe_len; b += kWave) {
      const uint32_t i = b + L;
      if (i < xe_len) {
        const uint32_t e = s.XL[i];
        const uint64_t *row = s.XR + (uint64_t)e * W;
        uint32_t sc = 0;
        for (uint32_t j = 0; j < W; ++j) sc += popc64(rdlane64(Pw, j) & row[j]);
        const uint32_t key = 0x80000000u | s.XV[e];
        if (bk == kNone || sc > bs || (sc == bs && key < bk)) {
          bs = sc;
          bk = key;
          brow = e;
        }
      }
    }
  }
  const uint32_t mx = wave_max(bk == kNone ? 0u : bs + 1u);
  const uint32_t kmin = wave_min((bk != kNone && bs + 1u == mx) ? bk : kNone);
  best = mx - 1u;
  if (kmin == kNone) {
    piv = kNone;
  } else if (kmin & 0x80000000u) {
    const uint32_t who = ctz64(ballot(bk == kmin));
    piv = s.p + rdlane(brow, who);
  } else {
    piv = kmin;
  }
}

// Is outside-X entry e adjacent to S[c]? IPX: bit c of its row. IP: e is a
// vertex id, searched in N-(S[c]) (every outside vertex precedes all of S).
template <bool kIPX>
__device__ __forceinline__ bool xe_adj(const Sub &s, uint32_t e, uint32_t c, const uint32_t *nb, uint32_t nlen) {
  if (kIPX) return (s.XR[(uint64_t)e * s.W + (c >> 6)] >> (c & 63)) & 1ull;
  const uint32_t pos = lower_bound_u32(nb, nlen, e);
  return pos < nlen && nb[pos] == e;
}

template <bool kIPX>
__device__ __forceinline__ void in_nbrs(const Sub &s, uint32_t c, const uint32_t *&nb, uint32_t &nlen) {
  nb = nullptr;
  nlen = 0;
  if (!kIPX) {
    const uint32_t cv = s.S[c];
    const uint64_t b = s.rp[cv];
    nb = s.oc + b;
    nlen = (uint32_t)(s.split[cv] - b);
  }
}

template <bool kIPX>
__device__ __forceinline__ bool xe_any(const Sub &s, uint32_t len, uint32_t c) {
  const uint32_t *nb;
  uint32_t nlen;
  in_nbrs<kIPX>(s, c, nb, nlen);
  for (uint32_t b = 0; b < len; b += kWave) {
    const uint32_t i = b + lane_id();
    const bool t = i < len && xe_adj<kIPX>(s, s.XL[i], c, nb, nlen);
    if (ballot(t)) return true;
  }
  return false;
}

// Stable partition of XL[0, len) into [adjacent to S[c] | the rest]; returns
// the adjacent count. The prefix keeps the same set, so the parent's list is
// intact after the child returns.
template <bool kIPX>
__device__ __forceinline__ uint32_t xe_partition(const Sub &s, uint32_t len, uint32_t c) {
  const uint32_t *nb;
  uint32_t nlen;
  in_nbrs<kIPX>(s, c, nb, nlen);
  const uint32_t L = lane_id();
  uint32_t kept = 0, drop = 0;
  for (uint32_t b = 0; b < len; b += kWave) {
    const uint32_t i = b + L;
    const bool valid = i < len;
    const uint32_t e = valid ? s.XL[i] : 0;
    const bool t = valid && xe_adj<kIPX>(s, e, c, nb, nlen);
    const uint64_t km = ballot(t), dm = ballot(valid && !t);
    if (t) s.XL[kept + mbcnt(km)] = e;
    if (valid && !t) s.XA[drop + mbcnt(dm)] = e;
    kept += popc64(km);
    drop += popc64(dm);
  }
  if (kept && drop)
    for (uint32_t i = L; i < drop; i += kWave) s.XL[kept + i] = s.XA[i];
  return kept;
}

__device__ __forceinline__ void report(const BkParams &pr, lds_ull *hist_lds, WaveAcc &wa, uint32_t size,
                                       uint64_t mix) {
  wa.count++;
  wa.sub_cliques++;
  wa.hash += clique_hash(mix, size);
  wa.max_size = max(wa.max_size, size);
  if (lane_id() == 0) {
    if (size < pr.hist_lds) __hip_atomic_fetch_add(&hist_lds[size], 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else atomicAdd(&pr.hist[min(size, pr.hist_len - 1)], 1ull);
  }
}

__device__ __forceinline__ void zero_words(uint64_t *a, uint64_t n) {
  for (uint64_t i = lane_id(); i < n; i += kWave) a[i] = 0;
}

// Builds the induced bit matrix over S and (IPX) the outside-X rows; fills
// s.xe0. XL holds the outside-X vertex ids on entry; with IPX it holds row
// indices on exit and XV keeps the ids.
template <bool kIPX>
__device__ __forceinline__ void build(const BkParams &pr, Sub &s) {
  const uint32_t L = lane_id(), p = s.p, W = s.W;
  zero_words(s.A, (uint64_t)p * W);
  if (kIPX) zero_words(s.XR, (uint64_t)s.q * W);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  for (uint32_t i = 0; i < p; ++i) {
    const uint32_t u = s.S[i];
    const uint64_t b = pr.split[u], e = pr.rp[u + 1];
    for (uint64_t k0 = b; k0 < e; k0 += kWave) {
      const uint64_t k = k0 + L;
      if (k < e) {
        const uint32_t y = pr.oc[k];
        const uint32_t j = lower_bound_u32(s.S, p, y);
        if (j < p && s.S[j] == y) {
          atomicOr((unsigned long long *)&s.A[(uint64_t)i * W + (j >> 6)], 1ull << (j & 63));
          atomicOr((unsigned long long *)&s.A[(uint64_t)j * W + (i >> 6)], 1ull << (i & 63));
        }
      }
    }
  }
  if (kIPX) {
    // one lane per outside vertex; rows with no neighbour in S are skipped
    uint32_t nz = 0;
    for (uint32_t b = 0; b < s.q; b += kWave) {
      const uint32_t i = b + L;
      bool any = false;
      if (i < s.q) {
        const uint32_t x = s.XL[i];
        s.XV[i] = x;
        uint64_t *row = s.XR + (uint64_t)i * W;
        for (uint64_t k = pr.split[x]; k < pr.rp[x + 1]; ++k) {
          const uint32_t y = pr.oc[k];
          const uint32_t j = lower_bound_u32(s.S, p, y);
          if (j < p && s.S[j] == y) {
            row[j >> 6] |= 1ull << (j & 63);
            any = true;
          }
        }
      }
      const uint64_t m = ballot(any);
      if (any) s.XL[nz + mbcnt(m)] = i;
      nz += popc64(m);
    }
    s.xe0 = nz;
  } else {
    s.xe0 = s.q;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
}

// ---- worker list: idle-wave queue and mailboxes ---------------------------

__device__ __forceinline__ unsigned long long ld_relaxed(unsigned long long *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Claims a queue position to publish into (lane 0 only). kNoSlot when full or
// contended.
__device__ __forceinline__ unsigned long long ring_claim_push(const BkParams &pr, uint32_t q) {
  unsigned long long *tail = pr.ctl + kCtlQueues + 16 * q + 8;
  unsigned long long *seq = pr.seq + (uint64_t)q * pr.ring_cap;
  unsigned long long pos = ld_relaxed(tail);
  for (int it = 0; it < 8; ++it) {
    const unsigned long long sq = ld_relaxed(&seq[pos % pr.ring_cap]);
    const long long dif = (long long)(sq - pos);
    if (dif == 0) {
      if (__hip_atomic_compare_exchange_weak(tail, &pos, pos + 1, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT))
        return pos;
    } else if (dif < 0) {
      return kNoSlot;
    } else {
      pos = ld_relaxed(tail);
    }
  }
  return kNoSlot;
}

// Claims a published queue position to consume (lane 0 only). kNoSlot when
// empty or contended.
__device__ __forceinline__ unsigned long long ring_claim_pop(const BkParams &pr, uint32_t q) {
  unsigned long long *head = pr.ctl + kCtlQueues + 16 * q;
  unsigned long long *seq = pr.seq + (uint64_t)q * pr.ring_cap;
  unsigned long long pos = ld_relaxed(head);
  for (int it = 0; it < 8; ++it) {
    const unsigned long long sq = ld_relaxed(&seq[pos % pr.ring_cap]);
    const long long dif = (long long)(sq - (pos + 1));
    if (dif == 0) {
      if (__hip_atomic_compare_exchange_weak(head, &pos, pos + 1, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT))
        return pos;
    } else if (dif < 0) {
      return kNoSlot;
    } else {
      pos = ld_relaxed(head);
    }
  }
  return kNoSlot;
}

__device__ __forceinline__ uint32_t queue_len(const BkParams &pr, uint32_t q) {
  const unsigned long long h = ld_relaxed(pr.ctl + kCtlQueues + 16 * q),
                           t = ld_relaxed(pr.ctl + kCtlQueues + 16 * q + 8);
  return t > h ? (uint32_t)min(t - h, 0x7fffffffull) : 0u;
}

// Progress signal of a busy wave for the idle waves' watchdog.
__device__ __forceinline__ void heartbeat(const BkParams &pr, WaveAcc &wa) {
  if (wa.nodes + wa.ls_nodes - wa.last_beat >= kBeatNodes) {
    wa.last_beat = wa.nodes + wa.ls_nodes;
    if (lane_id() == 0) {
      const unsigned long long b = atomicAdd(pr.ctl + kCtlProgress, 1ull);
      if (pr.host_progress) post_progress(pr.host_progress + 1, b + 1);
    }
  }
}

// Idle waves waiting for work: the length of this wave's queue plus one
// other queue, visited in turn (lane 0 samples).
__device__ __forceinline__ int32_t donation_budget(const BkParams &pr, WaveAcc &wa) {
  int32_t b = 0;
  wa.peek = (wa.peek + 1) % kQueues;
  if (lane_id() == 0) {
    b = (int32_t)queue_len(pr, wa.xq);
    if (wa.peek != wa.xq) b += (int32_t)queue_len(pr, wa.peek);
  }
  return (int32_t)uniform((uint32_t)b);
}

// A busy wave's poll, every donate_check nodes: its heartbeat, and from
// donate_age on, at most once every poll_ticks, a look at the idle queues
// (loads past the L2, some microseconds).
__device__ __forceinline__ void poll_idle(const BkParams &pr, WaveAcc &wa) {
  const uint64_t nodes = wa.nodes + wa.ls_nodes;
  if (nodes - wa.last_poll < pr.donate_check) return;
  wa.last_poll = nodes;
  heartbeat(pr, wa);
  const uint64_t now = __builtin_amdgcn_s_memrealtime();
  wa.budget = 0;
  if (now - wa.t_task < pr.donate_age || now < wa.next_poll) return;
  wa.budget = donation_budget(pr, wa);
  // nobody idle: look half as often each time, down to every 32 poll_ticks
  // (thousands of busy waves on the queues' 16 lines keep the idle ones from
  // getting on them)
  wa.poll_wait = wa.budget ? pr.poll_ticks : min(2 * wa.poll_wait, 32 * pr.poll_ticks);
  wa.next_poll = now + wa.poll_wait;
}
// No child to give, or nobody left to take it: the next look waits longer.
__device__ __forceinline__ void no_donation(const BkParams &pr, WaveAcc &wa) {
  wa.budget = 0;
  wa.next_poll += 3 * pr.poll_ticks;
}

// Takes an idle wave off the two queues last looked at (this XCD's first) for a donation
// and counts the task as outstanding; returns that wave's id (its slot
// receives the task) or kNone.
__device__ __forceinline__ uint32_t claim_receiver(const BkParams &pr, const WaveAcc &wa) {
  uint32_t r = kNone;
  if (lane_id() == 0) {
    for (uint32_t i = 0; i < 2 && r == kNone; ++i) {
      const uint32_t q = i ? wa.peek : wa.xq;
      if (i && q == wa.xq) break;
      const unsigned long long pos = ring_claim_pop(pr, q);
      if (pos != kNoSlot) {
        const uint64_t at = (uint64_t)q * pr.ring_cap + pos % pr.ring_cap;
        r = ld_shared(&pr.idle_ids[at]);
        drain();  // the id is read before its queue entry is free again
        st_shared(&pr.seq[at], pos + pr.ring_cap);
        atomicAdd(pr.ctl + kCtlOutstanding, 1ull);
      }
    }
  }
  return uniform(r);
}

// A task's header, written by lane 0 as 64-bit words: {root, |R|}, {|S|, W},
// {outside rows or ids, kind}, R's hash sum.
__device__ __forceinline__ void put_header(uint8_t *slot, uint32_t root, uint32_t rsize, uint32_t p, uint32_t W,
                                           uint32_t nx, uint32_t kind, uint64_t mix) {
  if (lane_id() == 0) {
    uint64_t *h = (uint64_t *)slot;
    st_shared(h, (uint64_t)rsize << 32 | root);
    st_shared(h + 1, (uint64_t)W << 32 | p);
    st_shared(h + 2, (uint64_t)kind << 32 | nx);
    st_shared(h + 3, mix);
  }
}

// Hands the task written into receiver r's slot over to it.
__device__ __forceinline__ void publish_task(const BkParams &pr, uint32_t r) {
  drain();  // the slot is written
  if (lane_id() == 0) st_shared(&pr.mbox[(uint64_t)r * kMboxStride], kMboxTask);
}

// Puts this idle wave on its XCD's idle queue (its mailbox is empty); false when the queue's tail was too contended this time.
__device__ __forceinline__ bool register_idle(const BkParams &pr, uint32_t gw, uint32_t xq) {
  unsigned long long pos = kNoSlot;
  if (lane_id() == 0) {
    pos = ring_claim_push(pr, xq);
    if (pos != kNoSlot) {
      const uint64_t at = (uint64_t)xq * pr.ring_cap + pos % pr.ring_cap;
      st_shared(&pr.idle_ids[at], gw);
      drain();  // the id is written before the entry is published
      st_shared(&pr.seq[at], pos + 1);
    }
  }
  return uniform64(pos) != kNoSlot;
}

// Takes n tasks off the outstanding count. The wave that takes the last one
// tells all others through their mailboxes: on their own they look at the
// count every 16th poll only, some 0.2 ms apart once they have waited long
// (worker-list launches in ms: 301 block-model graphs 1.77 -> 1.23, R-MAT 12
// (ef 8) 1.53 -> 1.13, G(4,096, deg 20) 0.44 -> 0.34).
__device__ __forceinline__ void tasks_done(const BkParams &pr, uint32_t n) {
  unsigned long long left = 1;
  if (lane_id() == 0) left = atomicSub(pr.ctl + kCtlOutstanding, (unsigned long long)n) - n;
  if (uniform64(left) != 0) return;
  for (uint32_t i = lane_id(); i < pr.ring_cap; i += kWave) st_shared(&pr.mbox[(uint64_t)i * kMboxStride], kMboxDone);
}

// Publishes the next child of the shallowest frame that still has one, when
// that child is large enough. The task carries the donor's induced bit matrix
// (same index space), the child's P and X words and its outside-X entries
// (ids, and rows with IPX), so the receiver copies instead of rebuilding.
// The frame is updated as if the child had been explored. Returns true on a
// donation.
template <bool kIPX>
__device__ __forceinline__ bool donate_shallowest(const BkParams &pr, Sub &s, uint32_t d, uint64_t &cP, uint64_t &cX, uint32_t cpiv,
                                  uint32_t cxe, uint64_t cmix, WaveAcc &wa) {
  const uint32_t L = lane_id(), W = s.W;
  const bool act = L < W;
  if (s.p > pr.slot_pmax) return false;
  for (uint32_t j = 0; j <= d; ++j) {
    uint64_t Pj = cP, Xj = cX, mixj = cmix;
    uint32_t pivj = cpiv, xej = cxe;
    uint8_t *f = nullptr;
    if (j < d) {
      f = frame_at(s, j);
      if (act) {
        Pj = ((const uint64_t *)f)[L];
        Xj = ((const uint64_t *)f)[W + L];
      } else {
        Pj = Xj = 0;
      }
      const uint32_t *meta = (const uint32_t *)(f + 16 * W);
      pivj = uniform(meta[0]);
      xej = uniform(meta[1]);
      mixj = uniform64(*(const uint64_t *)(f + 16 * W + 8));
    }
    const uint64_t Nj = act ? row_of(s, pivj)[L] : 0;
    const uint64_t B = Pj & ~Nj;
    const uint64_t bm = ballot(B != 0);
    if (bm == 0) continue;
    const uint32_t k0 = ctz64(bm);
    const uint32_t bit = ctz64(rdlane64(B, k0));
    const uint32_t c = k0 * 64 + bit;
    const uint64_t Ac = act ? s.A[(uint64_t)c * W + L] : 0;
    const uint64_t Pn = Pj & Ac, Xn = Xj & Ac;
    if (wave_sum(popc64(Pn)) < pr.donate_min_p) continue;
    // outside X of the child: entries of the frame's list adjacent to S[c]
    const uint32_t *nb;
    uint32_t nlen;
    in_nbrs<kIPX>(s, c, nb, nlen);
    uint32_t nx = 0;
    for (uint32_t b = 0; b < xej; b += kWave) {
      const uint32_t i = b + L;
      nx += popc64(ballot(i < xej && xe_adj<kIPX>(s, s.XL[i], c, nb, nlen)));
    }
    if (nx > pr.slot_xcap || hbm_need(s.p, nx, kIPX) > pr.hbm_bytes) continue;
    const uint32_t rcv = claim_receiver(pr, wa);
    if (rcv == kNone) return false;
    uint8_t *slot = pr.ring + (uint64_t)rcv * pr.slot_bytes;
    put_header(slot, s.root, s.rsize + j + 1, s.p, W, nx, kTaskList, mixj + splitmix64(s.S[c]));
    uint64_t *sp = (uint64_t *)(slot + pr.slot_oP);
    if (act) {
      st_shared(sp + L, Pn);
      st_shared(sp + pr.slot_wmax + L, Xn);
    }
    wave_copy<true>((uint32_t *)(slot + pr.slot_oS), s.S, s.p);
    copy64<true>((uint64_t *)(slot + pr.slot_oA), s.A, (uint64_t)s.p * W);
    uint32_t *sXI = (uint32_t *)(slot + pr.slot_oXI);
    uint64_t *sXR = (uint64_t *)(slot + pr.slot_oXR);
    uint32_t w = 0;
    for (uint32_t b = 0; b < xej; b += kWave) {
      const uint32_t i = b + L;
      uint32_t e = 0;
      bool t = false;
      if (i < xej) {
        e = s.XL[i];
        t = xe_adj<kIPX>(s, e, c, nb, nlen);
      }
      const uint64_t m = ballot(t);
      if (t) {
        const uint32_t k = w + mbcnt(m);
        if (kIPX) {
          st_shared(sXI + k, s.XV[e]);
          for (uint32_t x = 0; x < W; ++x) st_shared(sXR + (uint64_t)k * W + x, s.XR[(uint64_t)e * W + x]);
        } else {
          st_shared(sXI + k, e);
        }
      }
      w += popc64(m);
    }
    publish_task(pr, rcv);
    // the donor treats c as explored: P -> X in frame j
    const uint64_t m = 1ull << bit;
    if (j == d) {
      if (L == k0) {
        cP &= ~m;
        cX |= m;
      }
    } else if (L == k0) {
      ((uint64_t *)f)[L] = Pj & ~m;
      ((uint64_t *)f)[W + L] = Xj | m;
    }
    wa.nodes++;
    wa.donations++;
    return true;
  }
  return false;
}

// Runs BK from the root state (P, X) of an arena that `build` has filled.
template <bool kIPX, bool kWL, int kStat>
__device__ __forceinline__ void bk_solve(const BkParams &pr, Sub &s, uint64_t cP, uint64_t cX, lds_ull *hist_lds,
                         WaveAcc &wa, Clock<kStat> &clk) {
  const uint32_t L = lane_id(), W = s.W;
  const bool act = L < W;
  uint32_t xe = s.xe0;
  uint32_t piv, best;
  clk.to(kBdPivot);
  pick_pivot<kIPX>(s, cP, cX, xe, piv, best);
  if (piv == kNone || best == wave_sum(popc64(cP))) return;  // an X vertex covers all of P
  uint64_t cN = act ? row_of(s, piv)[L] : 0;
  uint64_t mix = s.rmix;
  uint32_t d = 0;
  while (true) {
    if constexpr (kWL) {
      clk.to(kBdQueue);
      poll_idle(pr, wa);
      if (wa.budget > 0) {
        if (donate_shallowest<kIPX>(pr, s, d, cP, cX, piv, xe, mix, wa)) wa.budget--;
        else no_donation(pr, wa);
      }
    }
    clk.to(kBdSetOps);
    const uint64_t B = cP & ~cN;
    const uint64_t bm = ballot(B != 0);
    if (bm == 0) {
      if (d == 0) break;
      clk.to(kBdBranch);
      --d;
      const uint8_t *f = frame_at(s, d);
      if (act) {
        cP = ((const uint64_t *)f)[L];
        cX = ((const uint64_t *)f)[W + L];
      }
      const uint32_t *meta = (const uint32_t *)(f + 16 * W);
      piv = uniform(meta[0]);
      xe = uniform(meta[1]);
      mix = uniform64(*(const uint64_t *)(f + 16 * W + 8));
      cN = act ? row_of(s, piv)[L] : 0;
      continue;
    }
    const uint32_t k0 = ctz64(bm);
    const uint32_t bit = ctz64(rdlane64(B, k0));
    const uint32_t c = k0 * 64 + bit;
    {
      const uint64_t m = L == k0 ? (1ull << bit) : 0ull;
      cP ^= m;
      cX |= m;
    }
    const uint64_t Ac = act ? s.A[(uint64_t)c * W + L] : 0;
    const uint64_t Pn = cP & Ac, Xn = cX & Ac;
    wa.nodes++;
    const uint64_t cmix = mix + splitmix64(uniform(s.S[c]));
    if (ballot(Pn != 0) == 0) {
      clk.to(kBdMaximal);
      if (ballot(Xn != 0) == 0 && (xe == 0 || !xe_any<kIPX>(s, xe, c))) report(pr, hist_lds, wa, s.rsize + d + 1, cmix);
      continue;
    }
    const uint32_t xn = xe ? xe_partition<kIPX>(s, xe, c) : 0;
    uint32_t npiv, nbest;
    clk.to(kBdPivot);
    pick_pivot<kIPX>(s, Pn, Xn, xn, npiv, nbest);
    // (a pivot from X covering P needs no test here: the child level finds
    // P & ~N(pivot) empty at once and backtracks, counting no node)
    if (npiv == kNone) continue;
    clk.to(kBdBranch);
    uint8_t *f = frame_at(s, d);
    if (act) {
      ((uint64_t *)f)[L] = cP;
      ((uint64_t *)f)[W + L] = cX;
    }
    uint32_t *meta = (uint32_t *)(f + 16 * W);
    meta[0] = piv;
    meta[1] = xe;
    *(uint64_t *)(f + 16 * W + 8) = mix;
    ++d;
    cP = Pn;
    cX = Xn;
    piv = npiv;
    xe = xn;
    mix = cmix;
    cN = act ? row_of(s, piv)[L] : 0;
  }
}

// ---- bitmap path: outside X as a set of row indices ----------------------
//
// Arena: S (p ids) | A (p x W) | XR (q x W rows of the outside-X vertices,
// in vertex-id order, zero rows kept) | frames. A frame holds P, X (W words),
// E (WX words) and {pivot, mix}. Row index order is vertex-id order, so the
// lowest-index tie-break equals the list path's id tie-break.

// Lays out a bitmap subproblem over an LDS region of lds_bytes (taken from
// the workgroup pool) and the wave's HBM arena, as bits_plan decides: all of
// S, A, the outside rows and the first frames in LDS; S, A and the first
// frames in LDS with the outside rows in HBM; everything but the frames the
// region holds in HBM. Frames past the LDS levels continue in HBM. The order
// S | A | rows | H keeps a level-2 staging list that starts right after the
// rows intact while the rows are built (H is written last).
__device__ __forceinline__ bool place_bits(Sub &s, uint32_t p, uint32_t q, uint32_t W, uint8_t *lds, uint32_t lds_bytes,
                                           uint8_t *hbm, uint64_t hbm_bytes, uint32_t stack_lds = 0) {
  const BitsPlan b = bits_plan(p, q, W, lds_bytes, stack_lds);
  if (b.hbm > hbm_bytes) return false;
  const uint64_t sa = align8(4ull * p) + 8ull * p * W, xr = 8ull * q * W;
  uint8_t *base, *xbase, *hbase;
  if (b.where == 3) {
    base = lds;
    xbase = lds + sa;
    hbase = lds + sa + xr;
    s.fr_hbm = hbm;
  } else if (b.where == 1) {
    base = lds;
    hbase = lds + sa;
    xbase = hbm;
    s.fr_hbm = hbm + xr;
  } else {
    base = hbm;
    xbase = hbm + sa;
    hbase = hbm + sa + xr;
    s.fr_hbm = hbm + sa + xr + 8ull * p;
  }
  s.where = b.where;
  s.fr_lds = lds + b.in_lds;
  s.lds_levels = b.lds_levels;
  s.FS = bits_fs(W, words_of(q));
  s.WX = words_of(q);
  s.S = (uint32_t *)base;
  s.A = (uint64_t *)(base + align8(4ull * p));
  s.XR = (uint64_t *)xbase;
  s.H = (uint64_t *)hbase;
  s.XL = nullptr;
  s.XA = nullptr;
  s.XV = nullptr;
  return true;
}

// H[i] = splitmix64(S[i]) for the subproblem's p vertices.
__device__ __forceinline__ void fill_hash_terms(const Sub &s) {
  for (uint32_t i = lane_id(); i < s.p; i += kWave) s.H[i] = splitmix64(s.S[i]);
}

// Builds A over S and the outside-X rows of the q vertices in `ids`; returns
// the initial outside-X bitmap word of this lane (rows with a neighbour in S).
// The outside rows worth keeping: those of the q vertices in `ids` with a
// neighbour in S (sorted, p ids; rows are N+(x) & S since S lies later than
// every x). Lane k returns the keep mask of rows 64k..64k+63 (q <= 4096);
// nkeep is their count. Rows with no bit are never candidates, so dropping
// them (in order) changes nothing but the memory a subproblem needs.
// Rows kept from the chunk ids[b, b + 64) of a long outside list (more than
// 64 x 64 rows): every row with two or more neighbours in S, and a row with
// exactly one, S[j], only if no earlier kept row contains j. Such a row never
// decides anything: whenever it is live the earlier row is too (it holds the
// row's only member), on every pivot score the earlier row scores at least as
// much and wins a tie (lower row first), and it covers every node the row
// covers. cover (64 words in device memory, the wave's own, zeroed by the
// caller) holds the union of the rows kept so far; the chunk's singles are
// decided in row order, each also against the chunk's earlier multi-member
// rows, then those rows join the union.
__device__ __forceinline__ uint64_t keep_chunk(const BkParams &pr, const uint32_t *S, uint32_t p, const uint32_t *ids,
                                               uint32_t q, uint32_t b, uint64_t *cover) {
  const uint32_t L = lane_id(), i = b + L;
  uint32_t hits = 0, j = 0, x = 0;
  uint64_t t0 = 0, t1 = 0;
  if (i < q) {
    x = ids[i];
    t0 = pr.split[x];
    t1 = pr.rp[x + 1];
    for (uint64_t t = t0; t < t1 && hits < 2; ++t) {
      const uint32_t y = pr.oc[t];
      const uint32_t k = lower_bound_u32(S, p, y);
      if (k < p && S[k] == y) {
        if (hits == 0) j = k;
        ++hits;
      }
    }
  }
  const bool multi = hits >= 2;
  uint64_t km = ballot(multi);
  for (uint64_t pend = ballot(hits == 1); pend; pend &= pend - 1) {
    const uint32_t l = ctz64(pend), jl = rdlane(j, l), yj = S[jl];
    bool cov = (__hip_atomic_load(&cover[jl >> 6], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >> (jl & 63)) & 1ull;
    if (!cov) {
      bool has = false;
      if (L < l && multi) {
        const uint64_t len = t1 - t0;
        const uint32_t k = lower_bound_u32(pr.oc + t0, (uint32_t)len, yj);
        has = k < len && pr.oc[t0 + k] == yj;
      }
      cov = ballot(has) != 0;
    }
    if (!cov) {
      km |= 1ull << l;
      if (L == 0) atomicOr((unsigned long long *)&cover[jl >> 6], 1ull << (jl & 63));
      __builtin_amdgcn_s_waitcnt(0);
    }
  }
  if (multi)
    for (uint64_t t = t0; t < t1; ++t) {
      const uint32_t y = pr.oc[t];
      const uint32_t k = lower_bound_u32(S, p, y);
      if (k < p && S[k] == y) atomicOr((unsigned long long *)&cover[k >> 6], 1ull << (k & 63));
    }
  __builtin_amdgcn_s_waitcnt(0);
  return km;
}

// Clears the wave's cover words.
__device__ __forceinline__ void clear_cover(uint64_t *cover) {
  __hip_atomic_store(&cover[lane_id()], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __builtin_amdgcn_s_waitcnt(0);
}

// Number of rows keep_chunk keeps from the q vertices in ids, for any q.
__device__ __noinline__ __attribute__((not_tail_called)) uint32_t live_count_fn(ConstParams *kargs, const uint32_t *S,
                                                                                uint32_t p, const uint32_t *ids, uint32_t q,
                                                                                uint64_t *cover) {
  const BkParams &pr = *(const BkParams *)(ConstParams *)uniform64((uint64_t)kargs);
  p = uniform(p);
  q = uniform(q);
  uint32_t n = 0;
  clear_cover(cover);
  for (uint32_t b = 0; b < q; b += kWave) n += popc64(keep_chunk(pr, S, p, ids, q, b, cover));
  return n;
}

template <int kS>
__device__ __noinline__ __attribute__((not_tail_called)) uint64_t live_rows_fn(ConstParams *kargs, const uint32_t *S,
                                                                               uint32_t p, const uint32_t *ids, uint32_t q) {
  const BkParams &pr = *(const BkParams *)(ConstParams *)uniform64((uint64_t)kargs);
  p = uniform(p);
  q = uniform(q);
  const uint32_t L = lane_id();
  uint64_t keep = 0;
  for (uint32_t b = 0, k = 0; b < q; b += kWave, ++k) {
    const uint32_t n = min(q - b, (uint32_t)kWave);
    uint64_t t0 = 0;
    uint32_t len = 0;
    if (L < n) {
      const uint32_t x = ids[b + L];
      t0 = pr.split[x];
      len = (uint32_t)(pr.rp[x + 1] - t0);
    }
    // a lane a list: most have a hit among their first arcs
    bool any = false;
    for (uint32_t k0 = 0; ballot(!any && k0 < len) != 0; k0 += kArcs) {
      uint32_t j[kArcs];
      find_arcs<kS>(S, p, pr.oc + t0, k0, 1, any ? 0u : len, j);
      any = any || (j[0] & j[1] & j[2] & j[3]) != kNone;
    }
    const uint64_t mask = ballot(any);
    if (L == k) keep = mask;
  }
  return keep;
}

__device__ __forceinline__ uint32_t live_count(const uint32_t *S, uint32_t p, const uint32_t *ids, uint32_t q,
                                               uint64_t *cover) {
  return uniform(live_count_fn((ConstParams *)__builtin_amdgcn_kernarg_segment_ptr(), S, p, ids, q, cover));
}
template <int kS>
__device__ __forceinline__ uint64_t live_rows(const uint32_t *S, uint32_t p, const uint32_t *ids, uint32_t q,
                                              uint32_t &nkeep) {
  const uint64_t keep = live_rows_fn<kS>((ConstParams *)__builtin_amdgcn_kernarg_segment_ptr(), S, p, ids, q);
  nkeep = wave_sum(popc64(keep));
  return keep;
}

// Keep mask of all q rows (lane k: rows 64k..64k+63).
__device__ __forceinline__ uint64_t all_rows(uint32_t q) { return full_word(q); }

// ---- functions of their own -----------------------------------------------
// The kernel's places that set a subproblem up and solve it call functions:
// with everything inlined a kernel was 119,000 instructions, the solver
// shared its registers with all that surrounds it, and what bounded a small
// subproblem was the scratch memory its registers were spilled to (500 bytes
// a lane, 32 KB a wave and subproblem). `kargs` is the kernel's argument
// segment, whose first argument is pr; s goes through the wave's hand-over
// block in LDS (address wa.io) once a subproblem, the wave's totals stay
// there, and both are read back as uniform values. not_tail_called lets the
// compiler see which registers a function leaves alone (otherwise each call
// saved and restored 54 of them). Enumeration in ms, everything inlined but
// the solvers -> now: G(4,096, deg 20) 0.175 -> 0.10, G(50,000, deg 40) 1.56
// -> 1.14, 301 block-model graphs of 64..300 1.22 -> 0.79, of 400..500 4.26
// -> 2.73, R-MAT 12 (ef 8) 0.53 -> 0.48.
struct Handover {
  Sub s;
  WaveAcc w;
};
typedef __attribute__((address_space(3))) Handover LdsHandover;
constexpr uint32_t kHandoverBytes = (sizeof(Handover) + 15) / 16 * 16;
__device__ __forceinline__ LdsHandover *handover(uint32_t io) { return (LdsHandover *)(uintptr_t)io; }
// Word copies between registers and the block (all lanes hold and write the
// same values).
template <class T>
__device__ __forceinline__ void lds_put(__attribute__((address_space(3))) T *to, const T &v) {
  static_assert(sizeof(T) % 8 == 0, "whole words");
  uint64_t t[sizeof(T) / 8];
  __builtin_memcpy(t, &v, sizeof(T));
#pragma unroll
  for (uint32_t i = 0; i < sizeof(T) / 8; ++i) ((lds_u64 *)to)[i] = t[i];
}
// (read back as uniform values)
template <class T>
__device__ __forceinline__ T lds_get(const __attribute__((address_space(3))) T *from) {
  uint64_t t[sizeof(T) / 8];
#pragma unroll
  for (uint32_t i = 0; i < sizeof(T) / 8; ++i) t[i] = uniform64(((const lds_u64 *)from)[i]);
  T v;
  __builtin_memcpy(&v, t, sizeof(T));
  return v;
}
// Builds A over S and the kept outside rows (keep: mask from live_rows over
// the q0 vertices in `ids`; s.q = their count), numbered in order; returns
// this lane's word of the initial outside-row set (all kept rows).
// filter: q0 may exceed 64 x 64 and the kept rows are found chunk by chunk
// (keep_chunk) instead of from keep; their count, s.q, was taken by
// live_count.
template <bool kLA, bool kLX>
__device__ __forceinline__ uint64_t build_bits(const BkParams &pr, const Sub &s, const uint32_t *ids, uint32_t q0,
                                               uint64_t keep, bool filter) {
  const uint32_t L = lane_id(), p = s.p, W = s.W, q = s.q;
  zero_words(s.A, (uint64_t)p * W);
  zero_words(s.XR, (uint64_t)q * W);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  for (uint32_t i0 = 0; i0 < p; i0 += kWave) {
    const uint32_t n = min(p - i0, (uint32_t)kWave);
    uint64_t b = 0;
    uint32_t len = 0;
    if (L < n) {
      const uint32_t u = ld32<kLA>(s.S, i0 + L);
      b = pr.split[u];
      len = (uint32_t)(pr.rp[u + 1] - b);
    }
    walk_lists<kLA ? kInLds : kInGlb>(pr.oc, s.S, p, n, b, len, [&](uint32_t r, const uint32_t (&j)[kArcs]) {
      const uint32_t i = i0 + r;
#pragma unroll
      for (uint32_t m = 0; m < kArcs; ++m)
        if (j[m] != kNone) {
          or64<kLA>(s.A, (uint64_t)i * W + (j[m] >> 6), 1ull << (j[m] & 63));
          or64<kLA>(s.A, (uint64_t)j[m] * W + (i >> 6), 1ull << (i & 63));
        }
    });
  }
  uint32_t base = 0;
  if (filter) clear_cover(s.cover);
  for (uint32_t b = 0, k = 0; b < q0; b += kWave, ++k) {
    const uint64_t km = filter ? keep_chunk(pr, s.S, p, ids, q0, b, s.cover) : rdlane64(keep, k);
    const uint32_t n = popc64(km);
    if (n == 0) continue;
    // the kept vertices, in order, to lanes 0.. (the others behind them)
    const uint32_t x0 = b + L < q0 ? ids[b + L] : 0u;
    const uint32_t dst = lane_in(km) ? mbcnt(km) : n + (L - mbcnt(km));
    const uint32_t x = (uint32_t)__builtin_amdgcn_ds_permute((int)(dst * 4), (int)x0);
    uint64_t t0 = 0;
    uint32_t len = 0;
    if (L < n) {
      t0 = pr.split[x];
      len = (uint32_t)(pr.rp[x + 1] - t0);
    }
    walk_lists<kLA ? kInLds : kInGlb>(pr.oc, s.S, p, n, t0, len, [&](uint32_t r, const uint32_t (&j)[kArcs]) {
#pragma unroll
      for (uint32_t m = 0; m < kArcs; ++m)
        if (j[m] != kNone) or64<kLX>(s.XR, (uint64_t)(base + r) * W + (j[m] >> 6), 1ull << (j[m] & 63));
    });
    base += n;
  }
  fill_hash_terms(s);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  return full_word(q);
}

template <bool kLA, bool kLX>
__device__ __noinline__ __attribute__((not_tail_called)) uint64_t build_bits_fn(ConstParams *kargs, uint32_t io,
                                                                                const uint32_t *ids, uint32_t q0,
                                                                                uint64_t keep, uint32_t filter) {
  const BkParams &pr = *(const BkParams *)(ConstParams *)uniform64((uint64_t)kargs);
  const Sub s = lds_get(&handover(uniform(io))->s);
  return build_bits<kLA, kLX>(pr, s, (const uint32_t *)uniform64((uint64_t)ids), uniform(q0), keep, uniform(filter) != 0);
}

// Pivot over P|X (index order) then the outside rows in E (row order): the
// largest |P & N(u)|, ties to the lowest index u, outside row e indexed p + e.
// Each lane scores the candidates of its bit position in every nonzero word;
// one reduction over key = (score + 1) << 13 | (8191 - index) picks the
// winner (p <= 4096 and q <= 4096 keep index < 8192).
template <bool kLA, bool kLX>
__device__ __forceinline__ void pick_pivot_bits(const Sub &s, uint64_t Pw, uint64_t Xw, uint64_t Ew, uint32_t &piv,
                                                uint32_t &best) {
  const uint32_t L = lane_id(), W = s.W;
  const uint64_t C = Pw | Xw;
  const uint64_t pm = ballot(Pw != 0);
  uint32_t key = 0;
  for (uint64_t cm = ballot(C != 0); cm; cm &= cm - 1) {
    const uint32_t k = ctz64(cm);
    if ((rdlane64(C, k) >> L) & 1ull) {
      const uint32_t u = k * 64 + L;
      const uint64_t r0 = (uint64_t)u * W;
      uint32_t sc = 0;
      for (uint64_t m = pm; m; m &= m - 1) {
        const uint32_t j = ctz64(m);
        sc += popc64(rdlane64(Pw, j) & ld64<kLA>(s.A, r0 + j));
      }
      key = max(key, ((sc + 1u) << 13) | (8191u - u));
    }
  }
  for (uint64_t em = ballot(Ew != 0); em; em &= em - 1) {
    const uint32_t k = ctz64(em);
    if ((rdlane64(Ew, k) >> L) & 1ull) {
      const uint32_t e = k * 64 + L;
      const uint64_t r0 = (uint64_t)e * W;
      uint32_t sc = 0;
      for (uint64_t m = pm; m; m &= m - 1) {
        const uint32_t j = ctz64(m);
        sc += popc64(rdlane64(Pw, j) & ld64<kLX>(s.XR, r0 + j));
      }
      key = max(key, ((sc + 1u) << 13) | (8191u - (s.p + e)));
    }
  }
  const uint32_t mx = wave_max(key);
  piv = mx ? 8191u - (mx & 8191u) : kNone;
  best = mx ? (mx >> 13) - 1u : 0u;
}

// Outside rows of E adjacent to S[c] (this lane's word of the result).
template <bool kLX>
__device__ __forceinline__ uint64_t filter_rows(const Sub &s, uint64_t Ew, uint32_t c) {
  const uint32_t L = lane_id(), W = s.W, cw = c >> 6, cb = c & 63;
  uint64_t out = 0;
  for (uint64_t em = ballot(Ew != 0); em; em &= em - 1) {
    const uint32_t k = ctz64(em);
    const uint64_t ek = rdlane64(Ew, k);
    const bool t = ((ek >> L) & 1ull) && ((ld64<kLX>(s.XR, (uint64_t)(k * 64 + L) * W + cw) >> cb) & 1ull);
    const uint64_t m = ballot(t);
    if (L == k) out = m;
  }
  return out;
}

// Does any outside row of E touch S[c]?
template <bool kLX>
__device__ __forceinline__ bool rows_any(const Sub &s, uint64_t Ew, uint32_t c) {
  const uint32_t L = lane_id(), W = s.W, cw = c >> 6, cb = c & 63;
  for (uint64_t em = ballot(Ew != 0); em; em &= em - 1) {
    const uint32_t k = ctz64(em);
    const uint64_t ek = rdlane64(Ew, k);
    if (ballot(((ek >> L) & 1ull) && ((ld64<kLX>(s.XR, (uint64_t)(k * 64 + L) * W + cw) >> cb) & 1ull))) return true;
  }
  return false;
}

// One frame of the bitmap solver: P, X, E words, then the pivot and R's hash.
template <bool kL>
__device__ __forceinline__ void frame_put(uint8_t *f, uint32_t W, uint32_t WX, uint64_t P, uint64_t X, uint64_t E,
                                          uint32_t piv, uint64_t mix) {
  const uint32_t L = lane_id();
  uint64_t *fw = (uint64_t *)f;
  if (L < W) {
    st64<kL>(fw, L, P);
    st64<kL>(fw, W + L, X);
  }
  if (L < WX) st64<kL>(fw, 2 * W + L, E);
  if (L == 0) {
    st32<kL>((uint32_t *)(f + 8 * (2 * W + WX)), 0, piv);
    st64<kL>((uint64_t *)(f + 8 * (2 * W + WX) + 8), 0, mix);
  }
}

template <bool kL>
__device__ __forceinline__ void frame_get(const uint8_t *f, uint32_t W, uint32_t WX, uint64_t &P, uint64_t &X,
                                          uint64_t &E, uint32_t &piv, uint64_t &mix) {
  const uint32_t L = lane_id();
  const uint64_t *fw = (const uint64_t *)f;
  if (L < W) {
    P = ld64<kL>(fw, L);
    X = ld64<kL>(fw, W + L);
  }
  E = L < WX ? ld64<kL>(fw, 2 * W + L) : 0;
  piv = uniform(ld32<kL>((const uint32_t *)(f + 8 * (2 * W + WX)), 0));
  mix = uniform64(ld64<kL>((const uint64_t *)(f + 8 * (2 * W + WX) + 8), 0));
}

// This lane's word of the pivot's row: an inside vertex's row of A or an
// outside row.
template <bool kLA, bool kLX>
__device__ __forceinline__ uint64_t pivot_word(const Sub &s, uint32_t piv) {
  const uint32_t L = lane_id();
  if (L >= s.W) return 0;
  return piv < s.p ? ld64<kLA>(s.A, (uint64_t)piv * s.W + L) : ld64<kLX>(s.XR, (uint64_t)(piv - s.p) * s.W + L);
}

// Hands the node (P, X, E) with |R| = rsize and R's hash sum rmix to an idle
// wave (bitmap path): the donor's S and A, the node's P and X words, and the
// outside rows live in E packed in row order (which keeps the pivot's tie
// rule), renumbered 0..q'-1. False when no wave is idle.
template <bool kLX>
__device__ __forceinline__ bool send_bits(const BkParams &pr, const Sub &s, uint32_t rsize, uint64_t rmix,
                                          uint64_t Pn, uint64_t Xn, uint64_t En, WaveAcc &wa) {
  const uint32_t L = lane_id(), W = s.W;
  const uint32_t rcv = claim_receiver(pr, wa);
  if (rcv == kNone) return false;
  uint8_t *slot = pr.ring + (uint64_t)rcv * pr.slot_bytes;
  uint64_t *sp = (uint64_t *)(slot + pr.slot_oP);
  if (L < W) {
    st_shared(sp + L, Pn);
    st_shared(sp + pr.slot_wmax + L, Xn);
  }
  wave_copy<true>((uint32_t *)(slot + pr.slot_oS), s.S, s.p);
  copy64<true>((uint64_t *)(slot + pr.slot_oA), s.A, (uint64_t)s.p * W);
  uint64_t *sXR = (uint64_t *)(slot + pr.slot_oXR);
  uint32_t qn = 0;
  for (uint64_t em = ballot(En != 0); em; em &= em - 1) {
    const uint32_t k = ctz64(em);
    const uint64_t ek = rdlane64(En, k);
    if ((ek >> L) & 1ull) {
      const uint64_t src = (uint64_t)(k * 64 + L) * W, dst = (uint64_t)(qn + mbcnt(ek)) * W;
      for (uint32_t w = 0; w < W; ++w) st_shared(sXR + dst + w, ld64<kLX>(s.XR, src + w));
    }
    qn += popc64(ek);
  }
  if (L < (qn + 63) / 64) st_shared(sp + 2 * pr.slot_wmax + L, full_word(qn));
  put_header(slot, s.root, rsize, s.p, W, qn, kTaskBits, rmix);
  publish_task(pr, rcv);
  return true;
}

// Publishes the next child of the shallowest frame with a large enough child
// (bitmap path): the donor's S, A and outside rows plus the child's P, X, E.
template <bool kLA, bool kLX>
__device__ __forceinline__ bool donate_bits(const BkParams &pr, const Sub &s, uint32_t d, uint64_t &cP, uint64_t &cX, uint64_t cE,
                            uint32_t cpiv, uint64_t cmix, WaveAcc &wa) {
  const uint32_t L = lane_id(), W = s.W, WX = s.WX;
  const bool act = L < W;
  // a receiver may get no LDS from its pool: it must fit the HBM arena alone
  if (s.p > pr.slot_pmax || s.q > pr.slot_xcap || bits_need(s.p, s.q) > pr.hbm_bytes) return false;
  for (uint32_t j = 0; j <= d; ++j) {
    uint64_t Pj = cP, Xj = cX, Ej = cE, mixj = cmix;
    uint32_t pivj = cpiv;
    uint8_t *f = nullptr;
    const bool fl = j < s.lds_levels;
    if (j < d) {
      f = frame_at(s, j);
      Pj = Xj = 0;
      if (fl) frame_get<true>(f, W, WX, Pj, Xj, Ej, pivj, mixj);
      else frame_get<false>(f, W, WX, Pj, Xj, Ej, pivj, mixj);
    }
    const uint64_t Nj = pivot_word<kLA, kLX>(s, pivj);
    const uint64_t B = Pj & ~Nj;
    const uint64_t bm = ballot(B != 0);
    if (bm == 0) continue;
    const uint32_t k0 = ctz64(bm);
    const uint32_t bit = ctz64(rdlane64(B, k0));
    const uint32_t c = k0 * 64 + bit;
    const uint64_t Ac = act ? ld64<kLA>(s.A, (uint64_t)c * W + L) : 0;
    const uint64_t Pn = Pj & Ac, Xn = Xj & Ac;
    if (wave_sum(popc64(Pn)) < pr.donate_min_p) continue;
    const uint64_t En = filter_rows<kLX>(s, Ej, c);
    if (!send_bits<kLX>(pr, s, s.rsize + j + 1, mixj + s.H[c], Pn, Xn, En, wa)) return false;
    const uint64_t m = 1ull << bit;
    if (j == d) {
      if (L == k0) {
        cP &= ~m;
        cX |= m;
      }
    } else if (L == k0) {
      if (fl) {
        st64<true>((uint64_t *)f, L, Pj & ~m);
        st64<true>((uint64_t *)f, W + L, Xj | m);
      } else {
        st64<false>((uint64_t *)f, L, Pj & ~m);
        st64<false>((uint64_t *)f, W + L, Xj | m);
      }
    }
    wa.nodes++;
    wa.donations++;
    return true;
  }
  return false;
}

// Member codes of the small-universe solver: bits 0..12 the position (S
// index, or outside row with kMemOut), kMemP for a member of P.
constexpr uint32_t kMemOut = 1u << 14, kMemP = 1u << 15;
// Largest P + X + outside rows the small-universe solver takes (one lane per
// member).
constexpr uint32_t kSmallMax = 64;

// Solves the whole subtree under one node whose P, X and outside rows E number
// at most 64 in total. The members are renumbered in the order the bitmap
// solver breaks ties in (S indices ascending, then outside rows ascending):
// lane i holds member i's adjacency row over the members and, for an S
// member, its hash term. P and X (which takes in the outside rows) become
// wave-uniform 64-bit masks, a child is one lane read and two scalar ANDs,
// the pivot one AND + popcount per lane and one reduction, and the frames sit
// in lane d of seven registers. Pivot (largest |P & N(u)|, ties to the lowest
// member) and child order (lowest member first) are the bitmap solver's, so
// the same nodes are visited. rbase = |R| at the node; mix = R's hash sum.
// Maximal cliques found by the small-universe solver, buffered one per lane
// (R's hash sum and size) so that the 64-bit hash mixing and the histogram
// updates run on the vector unit 64 cliques at a time; hacc keeps each lane's
// running sum of hash terms.
struct CliqueBuf {
  uint64_t mix = 0, hacc = 0;
  uint32_t size = 0, n = 0;
};

__device__ __forceinline__ void flush_cliques(const BkParams &pr, lds_ull *hist_lds, CliqueBuf &cb) {
  if (lane_id() < cb.n) {
    cb.hacc += clique_hash(cb.mix, cb.size);
    if (cb.size < pr.hist_lds) __hip_atomic_fetch_add(&hist_lds[cb.size], 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else atomicAdd(&pr.hist[min(cb.size, pr.hist_len - 1)], 1ull);
  }
  cb.n = 0;
}

// (the caller flushes before the buffer can overflow)
__device__ __forceinline__ void keep_clique(const BkParams &pr, lds_ull *hist_lds, WaveAcc &t,
                                            CliqueBuf &cb, uint32_t size, uint64_t mix) {
  cb.mix = wrlane64(cb.mix, cb.n, mix);
  cb.size = wrlane(cb.size, cb.n, size);
  t.count++;
  t.max_size = max(t.max_size, size);
  cb.n++;
}

// Sum of a 64-bit value over the wave (uniform result).
__device__ __forceinline__ uint64_t wave_add64(uint64_t v) {
  for (int off = 1; off < (int)kWave; off <<= 1) {
    const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)v, off), hi = (uint32_t)__shfl_xor((int)(v >> 32), off);
    v += ((uint64_t)hi << 32) | lo;
  }
  return uniform64(v);
}

// Does a node go to the small-universe solver? P + X + outside rows within
// the threshold; with the worker list also |P| <= kSmallMaxPWl, since a
// small-universe subtree is never split between waves and its size is
// bounded by |P| (at most 3^(|P|/3) maximal cliques). 32 measured best of
// 16..40 on R-MAT 14, Chung-Lu 2^19 and a 32-graph SBM batch.
constexpr uint32_t kSmallMaxPWl = 32;
template <bool kWL>
__device__ __forceinline__ bool small_ok(const BkParams &pr, uint64_t P, uint64_t X, uint64_t E, uint32_t &np,
                                         uint32_t &nx) {
  // both counts in one reduction (each is at most 64 x 192 < 2^16)
  const uint32_t n = wave_sum(popc64(P) | (popc64(X) + popc64(E)) << 16);
  np = n & 0xFFFFu;
  nx = n >> 16;
  return np + nx <= pr.small_max && (!kWL || np <= pr.small_pmax);
}

// Mask width of the small-universe solver's loop: a universe of at most 32
// members runs with 32-bit masks and rows (one register and one lane read per
// row, one AND and one POPCNT per pivot key, two frame fields fewer), a
// larger one with 64-bit masks. Members, pivots and child order are the same
// either way.
template <typename Mk>
struct MaskOps;
template <>
struct MaskOps<uint32_t> {
  __device__ static uint32_t popc(uint32_t x) { return (uint32_t)__builtin_popcount(x); }
  __device__ static uint32_t ctz(uint32_t x) { return (uint32_t)__builtin_ctz(x); }
  __device__ static uint32_t rd(uint32_t v, uint32_t l) { return rdlane(v, l); }
  // as a lane mask: lanes 32..63 hold no member
  __device__ static uint64_t lanes(uint32_t m) { return m; }
  __device__ static uint32_t wr(uint32_t f, uint32_t l, uint32_t v) { return wrlane(f, l, v); }
  __device__ static uint32_t permute(uint32_t to, uint32_t v) { return (uint32_t)__builtin_amdgcn_ds_permute((int)to, (int)v); }
};
template <>
struct MaskOps<uint64_t> {
  __device__ static uint32_t popc(uint64_t x) { return popc64(x); }
  __device__ static uint32_t ctz(uint64_t x) { return ctz64(x); }
  __device__ static uint64_t rd(uint64_t v, uint32_t l) { return rdlane64(v, l); }
  __device__ static uint64_t lanes(uint64_t m) { return m; }
  __device__ static uint64_t wr(uint64_t f, uint32_t l, uint64_t v) { return wrlane64(f, l, v); }
  __device__ static uint64_t permute(uint32_t to, uint64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_permute((int)to, (int)(uint32_t)v);
    return (uint64_t)(uint32_t)__builtin_amdgcn_ds_permute((int)to, (int)(v >> 32)) << 32 | lo;
  }
};

// ---------------------------------------------------------------------------
// Lane solver: subtrees with at most kLsP members in P and kLsX in X run one
// per lane, kLsSlots at a time. The small-universe solver queues such a
// subtree (ls_put), whole if its root fits, instead of working it off on the
// wave; a full queue and the end of a wave's work run the queue (ls_run), so
// that subtrees of many small subproblems share a run.
//
// What bounds the wave-wide loop is instructions: about 120 a node, for the
// 24 members an average block-model universe has on 64 lanes. Here a step,
// one node on every busy lane, is about 300 instructions. A node is decided
// by which members each member of P sees: column r, of P's member r, holds a
// bit for every member, P's at bits 0..15 and X's from bit 16 on (two words,
// the second for X's members 16..47). A child's P' and X' are one AND with
// its column. The pivot scores |P' & N(u)| of all members at once are a sum
// of the columns of P' in bit-sliced counters (four words of sum bits; 9
// instructions for three columns), and the best pivot falls out of them from
// the top bit down. The columns and the frames of the first kLsRegs levels
// are registers; a clique found is one word in LDS (the members chosen since
// the subtree's root), hashed and counted later by full waves: with hash sums
// carried from node to node and frames in memory, a step waited for loads
// that missed the L2.
//
// Enumeration in ms, without it -> with it (donating alike): Chung-Lu 2^17
// 21.5 -> 15.4, R-MAT 14 25 -> 21.4, R-MAT 12 5.4 -> 3.0; against subtrees of
// at most 16 members, one 32-bit column each: R-MAT 14 29.6 -> 21.4, a batch
// of 2.8 G nodes 617 -> 405 (whole call). About 29 of the 64 lanes are busy in
// a step; the rest have run out of work in their subtree.
//
// Members keep their order (S indices, then outside rows) within P and
// within X; byte r of `xb` says how many X members come before P member r,
// which decides a tie between the two. Pivots (largest |P & N(u)|, ties to
// the lowest member) and child order are those of the small-universe solver,
// so the same nodes are visited.
constexpr uint32_t kLsP = 15, kLsX = 48, kLsSlots = 64;
// A wave's region in device memory: a slot per subtree ({column words 0, 1}
// of 16 P members, 16 bytes xb, {p | x << 8 | |R| << 16}, root, R's hash
// sum), the hash terms of its P members, and the frames past kLsRegs levels
// {P | X of P's members << 16, X (two words), the pivot's row | chosen members
// << 16}, level-major. A pushed level has |P| >= 3 and each level at least
// one member fewer than its parent's. In LDS: the cliques found and not
// counted yet, {chosen members | slot << 16}.
constexpr uint32_t kLsLevels = kLsP - 3, kLsRegs = 4;
constexpr uint32_t kLsXbAt = 128, kLsHeadAt = 144, kLsSlotBytes = 160, kLsHOff = kLsSlots * kLsSlotBytes,
                   kLsFrOff = kLsHOff + kLsSlots * 16 * 8, kLsBytes = kLsFrOff + (kLsLevels - kLsRegs) * kLsSlots * 16;
constexpr uint32_t kLsFound = 512, kLsLds = kLsFound * 4;
// busy lanes at which the wave takes over the rest of their subtrees
constexpr uint32_t kLsDrain = 4;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(1))) uint8_t glb_u8;
typedef __attribute__((address_space(1))) u32x2 glb_u32x2;
typedef __attribute__((address_space(1))) u32x4 glb_u32x4;

struct LsOut {
  uint64_t count, nodes, hash;
  uint32_t max_size;
};

__device__ __forceinline__ bool ls_fits(const BkParams &pr, uint32_t p, uint32_t x) {
  return p + x <= pr.ls_max && p <= kLsP && x <= kLsX;
}

// Queues a subtree of p members of P and x of X (a free slot is the caller's).
// Lane r < p holds the column of P member r (c0, c1), its hash term and the
// number of X members before it; rb = |R|, mix = R's hash sum.
__device__ __forceinline__ void ls_put(WaveAcc &wa, uint32_t p, uint32_t x, uint32_t c0, uint32_t c1, uint64_t hs,
                                       uint32_t xb, uint32_t rb, uint32_t root, uint64_t mix) {
  const uint32_t j = wa.ls_n, L = lane_id();
  uint8_t *slot = wa.ls + j * kLsSlotBytes;
  if (L < p) {
    ((glb_u32x2 *)slot)[L] = u32x2{c0, c1};
    ((glb_u8 *)(slot + kLsXbAt))[L] = (uint8_t)xb;
    ((glb_u64 *)(wa.ls + kLsHOff))[j * 16 + L] = hs;
  }
  if (L == 0) *(glb_u32x4 *)(slot + kLsHeadAt) = u32x4{p | x << 8 | rb << 16, root, (uint32_t)mix, (uint32_t)(mix >> 32)};
  wa.ls_n = j + 1;
  wa.ls_p = max(wa.ls_p, p);
  wa.ls_x = max(wa.ls_x, x);
}

// The small-universe solver's loop over a renumbered universe: lane i holds
// member i's row M over the members and its hash term hs; lP / lX are the
// root's P and X over the members. Of a member that is in X from the start
// only the row's bits of P's members are used. kResume: the root is a node
// whose pivot row Np0 is known (its remaining children are solved).
template <int kStat>
__device__ __forceinline__ void ls_flush(const BkParams &pr, lds_ull *hist_lds, WaveAcc &wa);

template <typename Mk, int kStat, bool kResume = false>
__device__ __forceinline__ void small_loop(const BkParams &pr, Mk M, uint64_t hs, Mk lP, Mk lX, uint64_t mix,
                                           uint32_t rbase, uint32_t root, lds_ull *hist_lds, WaveAcc &wa,
                                           Clock<kStat> &clk, Mk Np0 = 0) {
  using O = MaskOps<Mk>;
  // pivot over P | X (the lowest member among the best scores): false when
  // it covers P (no child)
  auto pick = [&](Mk P, Mk X, uint32_t &pv) -> bool {
    const uint32_t key = lane_in(O::lanes(P | X)) ? O::popc(M & P) + 1u : 0u;
    const uint32_t mx = wave_max(key);
    pv = ctz64(ballot(key == mx));
    return mx != 0 && mx - 1u != O::popc(P);
  };
  clk.to(kBdPivot);
  Mk P = lP, X = lX, Np = Np0;
  if constexpr (!kResume) {
    uint32_t piv;
    if (!pick(P, X, piv)) return;
    Np = O::rd(M, piv);
  }
  uint32_t d = 0;
  // frames: lane d of each register holds level d
  Mk fP = 0, fX = 0, fN = 0;
  uint32_t fMl = 0, fMh = 0;
  // tallies of this subtree, added to the wave's totals at the end; the
  // cliques' hash terms and histogram bins are taken 64 at a time
  WaveAcc t{};
  uint64_t &nodes = t.nodes;
  CliqueBuf kb;
  while (true) {
    // an iteration keeps at most two cliques
    if (kb.n > kWave - 2) flush_cliques(pr, hist_lds, kb);
    clk.to(kBdSetOps);
    const Mk B = P & ~Np;
    if (B == 0) {
      if (d == 0) break;
      clk.to(kBdBranch);
      --d;
      P = O::rd(fP, d);
      X = O::rd(fX, d);
      mix = ((uint64_t)rdlane(fMh, d) << 32) | rdlane(fMl, d);
      Np = O::rd(fN, d);
      continue;
    }
    const Mk cb = B & (~B + 1);
    P ^= cb;
    X |= cb;
    const uint32_t c = O::ctz(cb);
    const Mk Mc = O::rd(M, c);
    const Mk Pn = P & Mc, Xn = X & Mc;
    ++nodes;
    const uint64_t cmix = mix + rdlane64(hs, c);
    if (Pn == 0) {
      clk.to(kBdMaximal);
      if (Xn == 0) keep_clique(pr, hist_lds, t, kb, rbase + d + 1, cmix);
      continue;
    }
    const uint32_t np = O::popc(Pn);
    if (np <= 2) {
      // |P| <= 2 decided without a pivot scan, node for node as the scan
      // would go (see the word-per-lane solver)
      clk.to(kBdMaximal);
      const uint32_t a = O::ctz(Pn);
      const Mk Ma = O::rd(M, a);
      const uint64_t ha = rdlane64(hs, a);
      if (np == 1) {
        if ((Xn & Ma) == 0) {
          ++nodes;
          keep_clique(pr, hist_lds, t, kb, rbase + d + 2, cmix + ha);
        }
        continue;
      }
      const uint32_t b = O::ctz(Pn & (Pn - 1));
      const Mk Mb = O::rd(M, b);
      const uint64_t hb = rdlane64(hs, b);
      if (Xn & Ma & Mb) continue;  // an X member covers P
      if ((Ma >> b) & 1u) {
        nodes += 2;
        keep_clique(pr, hist_lds, t, kb, rbase + d + 3, cmix + ha + hb);
        continue;
      }
      const Mk xs = Xn & (Ma | Mb);
      if (xs == 0) {
        nodes += 2;
        keep_clique(pr, hist_lds, t, kb, rbase + d + 2, cmix + ha);
        keep_clique(pr, hist_lds, t, kb, rbase + d + 2, cmix + hb);
        continue;
      }
      // the pivot is the lowest X member adjacent to one of a, b; the child
      // is the other one
      const bool piv_a = (Ma >> O::ctz(xs)) & 1u;
      ++nodes;
      if ((Xn & (piv_a ? Mb : Ma)) == 0) keep_clique(pr, hist_lds, t, kb, rbase + d + 2, cmix + (piv_a ? hb : ha));
      continue;
    }
    if constexpr (lane_of(kStat)) {
      if (ls_fits(pr, np, O::popc(Xn))) {
        if (wa.ls_n == kLsSlots) ls_flush<kStat>(pr, hist_lds, wa);
        // members move to their lanes in a queued subtree, P's to 0.., X's to
        // 16.. (all others to lane 15, which no member has)
        const uint64_t mP = O::lanes(Pn), mX = O::lanes(Xn);
        const bool inP = lane_in(mP), inX = lane_in(mX);
        const uint32_t r = mbcnt(mP), x = mbcnt(mX), dst = 4 * (inP ? r : inX ? 16 + x : 15u);
        const Mk Mq = O::permute(dst, M);
        const uint64_t hq = MaskOps<uint64_t>::permute(dst, hs);
        const uint32_t xbq = (uint32_t)__builtin_amdgcn_ds_permute((int)dst, (int)x);
        const uint32_t nx = O::popc(Xn), L = lane_id();
        const bool on = L < np || (L >= 16 && L < 16 + nx);
        uint32_t c0 = 0, c1 = 0, k = 0;
        for (Mk m = Pn; m; m &= m - 1, ++k) {
          const uint64_t col = ballot(on && ((Mq >> O::ctz(m)) & 1u));
          c0 = wrlane(c0, k, (uint32_t)col);
          c1 = wrlane(c1, k, (uint32_t)(col >> 32));
        }
        ls_put(wa, np, nx, c0, c1, hq, xbq, rbase + d + 1, root, cmix);
        continue;
      }
    }
    clk.to(kBdPivot);
    uint32_t npiv;
    if (!pick(Pn, Xn, npiv)) continue;
    clk.to(kBdBranch);
    fP = O::wr(fP, d, P);
    fX = O::wr(fX, d, X);
    fMl = wrlane(fMl, d, (uint32_t)mix);
    fMh = wrlane(fMh, d, (uint32_t)(mix >> 32));
    fN = O::wr(fN, d, Np);
    ++d;
    P = Pn;
    X = Xn;
    mix = cmix;
    Np = O::rd(M, npiv);
  }
  if (kb.n) flush_cliques(pr, hist_lds, kb);
  wa.nodes += t.nodes;
  wa.count += t.count;
  wa.sub_cliques += t.count;
  wa.hash += wave_add64(kb.hacc);
  wa.max_size = max(wa.max_size, t.max_size);
}

// A word of the 16 picked by a lane's index. (Vectors, not arrays: an array
// indexed so goes to memory.)
__device__ __forceinline__ uint32_t ls_pick16(u32x16 w, uint32_t i) {
  const u32x8 a = (i & 8u) ? w.hi : w.lo;
  const u32x4 b = (i & 4u) ? a.hi : a.lo;
  const uint32_t c0 = (i & 2u) ? b[2] : b[0], c1 = (i & 2u) ? b[3] : b[1];
  return (i & 1u) ? c1 : c0;
}

// Does P member r come after X member x in the members' order (xb)?
__device__ __forceinline__ bool ls_after(u32x4 xb, uint32_t r, uint32_t x) {
  const uint32_t t01 = (r & 4u) ? xb[1] : xb[0], t23 = (r & 4u) ? xb[3] : xb[2];
  return ((((r & 8u) ? t23 : t01) >> (8 * (r & 3u))) & 0xFFu) > x;
}

// Bit-sliced counters: bit u of s[3..0] is the count of member u, at most 15.
struct LsCount {
  uint32_t s0 = 0, s1 = 0, s2 = 0, s3 = 0;
  // adds three words
  __device__ __forceinline__ void add3(uint32_t a, uint32_t b, uint32_t c) {
    const uint32_t x = a ^ b ^ c, y = (a & b) | (c & (a ^ b));
    const uint32_t c0 = s0 & x;
    s0 ^= x;
    const uint32_t z = (y & c0) | (s1 & (y ^ c0));
    s1 ^= y ^ c0;
    const uint32_t c2 = s2 & z;
    s2 ^= z;
    s3 |= c2;
  }
};

// Runs the n queued subtrees, lane j the subtree of slot j. A step takes one
// child of a lane's node (after one pop, if its node has none left) and
// decides it: leaf, at most two vertices left (decided without a child, as in
// the wave-wide loop), covered, or a new node. maxp / maxx: the most members
// of P and X among the subtrees. Once at most kLsDrain lanes are still busy,
// the wave takes over: each such lane's remaining work (the open children of
// its current node and of every frame below it) runs through the
// small-universe solver's loop, so that one large subtree does not hold the
// other lanes idle. Returns the totals; the subtrees' own counts go to their
// roots' labels.
__device__ __noinline__ __attribute__((not_tail_called)) LsOut ls_run(uint32_t n, uint32_t maxp, uint32_t maxx, uint8_t *ls, uint32_t ls_lds,
                                     uint32_t hist_lds_addr, uint32_t hist_lds_n, unsigned long long *hist,
                                     uint32_t hist_len, unsigned long long *sub_nodes,
                                     unsigned long long *sub_cliques) {
  n = uniform(n);
  maxp = uniform(maxp);
  maxx = uniform(maxx);
  ls_lds = uniform(ls_lds);
  hist_lds_addr = uniform(hist_lds_addr);
  hist_lds_n = uniform(hist_lds_n);
  hist_len = uniform(hist_len);
  ls = (uint8_t *)uniform64((uint64_t)(uintptr_t)ls);
  hist = (unsigned long long *)uniform64((uint64_t)(uintptr_t)hist);
  const uint32_t L = lane_id();
  // the queue's writes precede these reads
  drain();
  lds_ull *hist_lds = (lds_ull *)(uintptr_t)hist_lds_addr;
  lds_u32 *found = (lds_u32 *)(uintptr_t)ls_lds;
  const glb_u64 *H = (const glb_u64 *)(ls + kLsHOff);
  glb_u32x4 *fr = (glb_u32x4 *)(ls + kLsFrOff) + L;
  const bool wide = maxx > 16;  // some subtree has X members past the first word
  u32x16 A = 0, B = 0;          // columns: words 0 and 1
  u32x4 xb = 0;
  // the lane's node: P and X over P's members (PX = P | X << 16), X's members
  // (X0 << 16: the first 16 as in A; X1), the pivot's row | members chosen
  // since the subtree's root << 16, depth
  uint32_t PX = 0, X0 = 0, X1 = 0, NR = 0, d = 0;
  uint32_t fP[kLsRegs], fX0[kLsRegs], fX1[kLsRegs], fN[kLsRegs];
#pragma unroll
  for (uint32_t k = 0; k < kLsRegs; ++k) fP[k] = fX0[k] = fX1[k] = fN[k] = 0;
  bool act = L < n, fresh = true;  // fresh: the subtree's root, not decided yet
  if (act) {
    const glb_u32x4 *sl = (const glb_u32x4 *)(ls + L * kLsSlotBytes);
    const uint32_t head = ((const glb_u32 *)(ls + L * kLsSlotBytes + kLsHeadAt))[0];
    xb = sl[kLsXbAt / 16];
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
      const u32x4 q = sl[k];
      A[2 * k] = q[0];
      B[2 * k] = q[1];
      A[2 * k + 1] = q[2];
      B[2 * k + 1] = q[3];
    }
    const uint32_t p = head & 0xFFu, x = (head >> 8) & 0xFFu;
    PX = (1u << p) - 1u;
    X0 = x < 16 ? ((1u << x) - 1u) << 16 : 0xFFFF0000u;
    X1 = x > 16 ? 0xFFFFFFFFu >> (48u - x) : 0u;
  }
  uint32_t cnt = 0, nodes = 0, nf = 0;  // the lane's cliques and nodes; cliques in `found`
  LsOut o{};
  uint64_t hacc = 0;
  uint32_t maxs = 0;
  // hashes and counts the cliques in `found`, one per lane
  auto count_found = [&]() {
    for (uint32_t b = 0; b < nf; b += kWave) {
      if (b + L < nf) {
        const uint32_t rec = found[b + L], j = rec >> 16;
        const u32x4 hd = *(const glb_u32x4 *)(ls + j * kLsSlotBytes + kLsHeadAt);
        uint64_t m = (uint64_t)hd[2] | (uint64_t)hd[3] << 32;
        const uint32_t sel = rec & 0xFFFFu, size = (hd[0] >> 16) + (uint32_t)__builtin_popcount(sel);
        for (uint32_t q = sel; q; q &= q - 1) m += H[j * 16 + (uint32_t)__builtin_ctz(q)];
        hacc += clique_hash(m, size);
        maxs = max(maxs, size);
        if (size < hist_lds_n) __hip_atomic_fetch_add(&hist_lds[size], 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        else atomicAdd(&hist[min(size, hist_len - 1)], 1ull);
      }
    }
    nf = 0;
  };
  while (true) {
    if (popc64(ballot(act)) <= kLsDrain) break;
    if (nf > kLsFound - 2 * kWave) count_found();  // a step finds at most two cliques a lane
    uint32_t e1 = 0, e2 = 0;  // members of the cliques the lane finds
    if (act) {
      // pop one level if the node has no child left
      uint32_t ch = PX & ~NR & 0xFFFFu;
      if (ch == 0 && !fresh) {
        act = d != 0;
        if (act) {
          --d;
          if (d >= kLsRegs) {
            const u32x4 f = fr[(d - kLsRegs) * kLsSlots];
            PX = f[0];
            X0 = f[1];
            X1 = f[2];
            NR = f[3];
          } else {
#pragma unroll
            for (uint32_t k = 0; k < kLsRegs; ++k) {
              PX = d == k ? fP[k] : PX;
              X0 = d == k ? fX0[k] : X0;
              X1 = d == k ? fX1[k] : X1;
              NR = d == k ? fN[k] : NR;
            }
          }
          ch = PX & ~NR & 0xFFFFu;
        }
      }
      // the node to decide: a child of the lane's node, or the root itself
      const bool go = fresh || ch != 0;
      const uint32_t c = fresh || !go ? 0u : (uint32_t)__builtin_ctz(ch);
      const uint32_t ca = fresh ? ~0u : ls_pick16(A, c);
      if (go && !fresh) {
        PX ^= 0x10001u << c;  // c leaves P for X
        ++nodes;
      }
      const uint32_t sel = fresh ? 0u : (NR >> 16) | 1u << c;
      const uint32_t Pn = PX & ca & 0xFFFFu, Qn = (PX >> 16) & ca, Xa = X0 & ca;
      const uint32_t Ca = Pn | Qn | Xa;  // pivot candidates
      uint32_t Cb = 0;
      if (wide) Cb = X1 & (fresh ? ~0u : ls_pick16(B, c));
      // scores of all members: the sum of the columns of P'
      LsCount sa, sb;
      auto col = [&](u32x16 w, uint32_t r) -> uint32_t {
        return w[r] & (uint32_t)__builtin_amdgcn_sbfe((int)Pn, r, 1);
      };
#pragma unroll
      for (uint32_t r = 0; r < kLsP; r += 3)
        if (r == 0 || r < maxp) {
          sa.add3(col(A, r), col(A, r + 1), col(A, r + 2));
          if (wide) sb.add3(col(B, r), col(B, r + 1), col(B, r + 2));
        }
      // the candidates with the best score, from its top bit down
      uint32_t Ka = Ca, Kb = Cb, best = 0;
      auto top = [&](uint32_t pa, uint32_t pb, uint32_t bit) {
        const uint32_t ta = Ka & pa, tb = wide ? Kb & pb : 0u;
        const bool any = (ta | tb) != 0;
        Ka = any ? ta : Ka;
        if (wide) Kb = any ? tb : Kb;
        best |= any ? bit : 0u;
      };
      top(sa.s3, sb.s3, 8);
      top(sa.s2, sb.s2, 4);
      top(sa.s1, sb.s1, 2);
      top(sa.s0, sb.s0, 1);
      // the pivot: the lowest of them in the members' order (xb)
      const uint32_t kp = Ka & 0xFFFFu, kx = Ka >> 16;
      const uint32_t pr = kp ? (uint32_t)__builtin_ctz(kp) : 0u;
      const uint32_t px = kx ? (uint32_t)__builtin_ctz(kx) : 16u + (Kb ? (uint32_t)__builtin_ctz(Kb) : 0u);
      const bool isx = kp == 0 || ((kx | Kb) != 0 && ls_after(xb, pr, px));
      // its row: its bit of every column
      const uint32_t at = isx ? px + 16u : pr;
      uint32_t piv = 0;
#pragma unroll
      for (uint32_t r = 0; r < kLsP; r += 3)
        if (r == 0 || r < maxp) {
#pragma unroll
          for (uint32_t k = r; k < r + 3; ++k) {
            const uint32_t w = wide && at >= 32 ? B[k] : A[k];
            piv |= ((w >> (at & 31u)) & 1u) << k;
          }
        }
      const uint32_t np = (uint32_t)__builtin_popcount(Pn);
      if (go && np >= 3 && best < np) {
        // a node of its own
        if (!fresh) {
          if (d >= kLsRegs) {
            fr[(d - kLsRegs) * kLsSlots] = u32x4{PX, X0, X1, NR};
          } else {
#pragma unroll
            for (uint32_t k = 0; k < kLsRegs; ++k) {
              fP[k] = d == k ? PX : fP[k];
              fX0[k] = d == k ? X0 : fX0[k];
              fX1[k] = d == k ? X1 : fX1[k];
              fN[k] = d == k ? NR : fN[k];
            }
          }
          ++d;
        }
        PX = Pn | Qn << 16;
        X0 = Xa;
        X1 = Cb;
        NR = piv | sel << 16;
        fresh = false;
      } else if (go) {
        act = !fresh;  // a root decided here has no node of its own
        if (np == 0) {
          e1 = (Ca | Cb) == 0 ? sel : 0u;
        } else if (np == 1) {
          nodes += best == 0;
          e1 = best == 0 ? sel | Pn : 0u;
        } else if (np == 2 && best < 2) {  // at 2 an X member covers P
          const uint32_t a = (uint32_t)__builtin_ctz(Pn), b = 31u - (uint32_t)__builtin_clz(Pn);
          if ((sa.s0 >> a) & 1u) {  // a sees b
            nodes += 2;
            e1 = sel | Pn;
          } else if (best == 0) {
            nodes += 2;
            e1 = sel | 1u << a;
            e2 = sel | 1u << b;
          } else {
            // the pivot is an X member adjacent to one of a, b (a and b see
            // neither); the child is the other, maximal if no X member sees it
            const uint32_t o1 = (piv >> a) & 1u ? b : a;
            ++nodes;
            uint32_t cov = Ca & ls_pick16(A, o1);
            if (wide) cov |= Cb & ls_pick16(B, o1);
            e1 = cov == 0 ? sel | 1u << o1 : 0u;
          }
        }
      }
    }
    const uint64_t m1 = ballot(e1 != 0), m2 = ballot(e2 != 0);
    if (e1) found[nf + mbcnt(m1)] = e1 | L << 16;
    nf += popc64(m1);
    if (m2) {
      if (e2) found[nf + mbcnt(m2)] = e2 | L << 16;
      nf += popc64(m2);
    }
    cnt += (e1 != 0) + (e2 != 0);
  }
  count_found();
  o.hash = wave_add64(hacc);
  o.max_size = wave_max(maxs);
  // the busy lanes' remaining work, on the whole wave
  BkParams q{};
  q.hist = hist;
  q.hist_len = hist_len;
  q.hist_lds = hist_lds_n;
  Clock<kStatNone> clk;
  for (uint64_t left = ballot(act); left; left &= left - 1) {
    const uint32_t j = ctz64(left);
    // the members of slot j in their order, one per lane: P member r at
    // position r + xb[r]
    const uint8_t *slot = ls + j * kLsSlotBytes;
    const u32x4 hd = *(const glb_u32x4 *)(slot + kLsHeadAt);
    const uint32_t h0 = uniform(hd[0]);
    const uint32_t p = h0 & 0xFFu, nm = p + ((h0 >> 8) & 0xFFu), rbj = h0 >> 16;
    const uint64_t mixj = uniform64((uint64_t)hd[2] | (uint64_t)hd[3] << 32);
    const uint32_t pos = L < p ? L + ((const glb_u8 *)(slot + kLsXbAt))[L] : 0u;
    const u32x2 cw = L < p ? ((const glb_u32x2 *)slot)[L] : u32x2{0u, 0u};
    uint64_t mP = 0;
    for (uint32_t r = 0; r < p; ++r) mP |= 1ull << rdlane(pos, r);
    const uint32_t r = mbcnt(mP);
    const bool inP = lane_in(mP), in = L < nm;
    const uint32_t ix = inP ? r : 16u + (L - r);  // the lane's member's bit in a column
    const uint64_t hs = inP ? H[j * 16 + r] : 0ull;
    // rows over the members: a P member's is its column, of an X member only
    // the bits of P's members
    uint64_t M = 0;
    for (uint32_t k = 0; k < p; ++k) {
      const uint32_t to = rdlane(pos, k);
      const uint64_t ck = (uint64_t)rdlane(cw[1], k) << 32 | rdlane(cw[0], k);
      const bool t = in && ((ck >> (ix & 63u)) & 1ull);
      const uint64_t cb = ballot(t);
      if (L == to) M = cb;
      else if (!inP && t) M |= 1ull << to;
    }
    WaveAcc t{};
    uint32_t PXk = rdlane(PX, j), X0k = rdlane(X0, j), X1k = rdlane(X1, j), Nk = rdlane(NR, j);
    const uint32_t dj = rdlane(d, j);
    const bool fj = (ballot(fresh) >> j) & 1ull;
    for (uint32_t k = dj + 1; k-- > 0;) {
      if (k < dj) {
        if (k >= kLsRegs) {
          const u32x4 f = ((const glb_u32x4 *)(ls + kLsFrOff))[(k - kLsRegs) * kLsSlots + j];
          PXk = uniform(f[0]);
          X0k = uniform(f[1]);
          X1k = uniform(f[2]);
          Nk = uniform(f[3]);
        } else {
#pragma unroll
          for (uint32_t i = 0; i < kLsRegs; ++i)
            if (i == k) {
              PXk = rdlane(fP[i], j);
              X0k = rdlane(fX0[i], j);
              X1k = rdlane(fX1[i], j);
              Nk = rdlane(fN[i], j);
            }
        }
      }
      // the node's sets over the members; R: the slot's R and those chosen since
      const uint64_t xk = (uint64_t)X1k << 32 | X0k;
      const uint64_t Pk = ballot(inP && ((PXk >> r) & 1u));
      const uint64_t Qk = ballot(in && (inP ? (PXk >> (16 + r)) & 1u : (uint32_t)(xk >> (ix & 63u)) & 1u));
      const uint64_t Nm = ballot(inP && ((Nk >> r) & 1u));
      uint64_t mk = mixj;
      for (uint64_t m = ballot(inP && ((Nk >> (16 + r)) & 1u)); m; m &= m - 1) mk += rdlane64(hs, ctz64(m));
      if (fj)
        small_loop<uint64_t, kStatNone>(q, M, hs, Pk, Qk, mk, rbj, 0, hist_lds, t, clk);
      else
        small_loop<uint64_t, kStatNone, true>(q, M, hs, Pk, Qk, mk, rbj + k, 0, hist_lds, t, clk,
                                              Nm);
    }
    if (L == j) {
      cnt += (uint32_t)t.count;
      nodes += (uint32_t)t.nodes;
    }
    o.hash += t.hash;
    o.max_size = max(o.max_size, t.max_size);
  }
  // per-root labels: one update when the whole run belongs to one root
  const uint32_t ncnt = wave_sum(cnt), nnodes = wave_sum(nodes);
  if (sub_nodes || sub_cliques) {
    const uint32_t root = L < n ? ((const glb_u32 *)(ls + L * kLsSlotBytes + kLsHeadAt))[1] : 0u, r0 = uniform(root);
    const bool one = ballot(L < n && root != r0) == 0;
    const bool on = one ? L == 0 : L < n;
    if (on && sub_nodes) atomicAdd(&sub_nodes[root], (unsigned long long)(one ? nnodes : nodes));
    if (on && sub_cliques) atomicAdd(&sub_cliques[root], (unsigned long long)(one ? ncnt : cnt));
  }
  o.count = ncnt;
  o.nodes = nnodes;
  return o;
}

// Runs the wave's queue, if any, and adds its totals to the wave's.
template <int kStat>
__device__ __forceinline__ void ls_flush(const BkParams &pr, lds_ull *hist_lds, WaveAcc &wa) {
  if constexpr (lane_of(kStat)) {
    if (wa.ls_n == 0) return;
    const LsOut o = ls_run(wa.ls_n, wa.ls_p, wa.ls_x, wa.ls, wa.ls_lds, (uint32_t)(uintptr_t)hist_lds, pr.hist_lds, pr.hist,
                           pr.hist_len, pr.sub_nodes, pr.sub_cliques);
    // (the results of a call are uniform, but only this says so)
    wa.ls_count += uniform64(o.count);
    wa.ls_nodes += uniform64(o.nodes);
    wa.hash += uniform64(o.hash);
    wa.max_size = max(wa.max_size, uniform(o.max_size));
    wa.ls_n = wa.ls_p = wa.ls_x = 0;
  }
}

// Solves the subtree of a node whose P, X and outside rows E number at most
// 64: numbers the members, one per lane, and queues the subtree for the lane
// solver or works it off in the wave-wide loop.
template <bool kWL, int kStat, bool kLA, bool kLX>
__device__ __forceinline__ void solve_small(const BkParams &pr, const Sub &s, uint64_t Pw, uint64_t Xw, uint64_t Ew,
                                            uint32_t p, uint32_t x, uint64_t mix, uint32_t rbase, lds_ull *hist_lds, WaveAcc &wa,
                                            Clock<kStat> &clk) {
  const uint32_t L = lane_id(), W = s.W;
  clk.to(kBdInduced);
  const uint64_t Cw = Pw | Xw;
  // a lane's word k of its member's row over S (mem: the member's code)
  auto row_word = [&](uint32_t mem, bool valid, uint32_t k) -> uint64_t {
    const uint64_t at = (uint64_t)(mem & 8191u) * W + k;
    if (!valid) return 0;
    return (mem & kMemOut) ? ld64<kLX>(s.XR, at) : ld64<kLA>(s.A, at);
  };
  if constexpr (lane_of(kStat)) {
    // (a full queue is run from the loop below, which then meets this subtree)
    if (wa.ls_n < kLsSlots && ls_fits(pr, p, x)) {
      // members go to lanes, P's to 0.., X's to 16.., with the number of X
      // members before them (each nonzero word pushes its set bits; lanes
      // without a bit push to lane 15, which no member has)
      uint32_t mem = 0, bp = 0, bx = 0;
      for (uint64_t cm = ballot(Cw != 0); cm; cm &= cm - 1) {
        const uint32_t k = ctz64(cm);
        const uint64_t pw = rdlane64(Pw, k), xw = rdlane64(Xw, k);
        const uint32_t rx = bx + mbcnt(xw), np = popc64(pw), nx = popc64(xw);
        const uint32_t dst = lane_in(pw) ? bp + mbcnt(pw) : lane_in(xw) ? 16 + rx : 15u;
        const uint32_t got = (uint32_t)__builtin_amdgcn_ds_permute((int)(dst * 4), (int)((k * 64 + L) | rx << 16));
        if (L - bp < np || L - 16 - bx < nx) mem = got;
        bp += np;
        bx += nx;
      }
      for (uint64_t em = ballot(Ew != 0); em; em &= em - 1) {
        const uint32_t k = ctz64(em);
        const uint64_t w = rdlane64(Ew, k);
        const uint32_t ne = popc64(w), dst = lane_in(w) ? 16 + bx + mbcnt(w) : 15u;
        const uint32_t got = (uint32_t)__builtin_amdgcn_ds_permute((int)(dst * 4), (int)((k * 64 + L) | kMemOut));
        if (L - 16 - bx < ne) mem = got;
        bx += ne;
      }
      const bool on = L < p || (L >= 16 && L < 16 + x);
      const uint64_t hs = L < p ? ld64<kLA>(s.H, mem & 8191u) : 0ull;
      // column of P member r: the lanes whose row has its bit
      uint32_t c0 = 0, c1 = 0, r = 0;
      for (uint64_t pm = ballot(Pw != 0); pm; pm &= pm - 1) {
        const uint32_t k = ctz64(pm);
        const uint64_t pw = rdlane64(Pw, k), rw = row_word(mem, on, k);
        for (uint32_t h = 0; h < 2; ++h) {
          const uint32_t rh = (uint32_t)(rw >> (32 * h));
          for (uint32_t m = (uint32_t)(pw >> (32 * h)); m; m &= m - 1, ++r) {
            const uint64_t col = ballot((rh & m & (0u - m)) != 0);
            c0 = wrlane(c0, r, (uint32_t)col);
            c1 = wrlane(c1, r, (uint32_t)(col >> 32));
          }
        }
      }
      ls_put(wa, p, x, c0, c1, hs, (mem >> 16) & 0xFFu, rbase, s.root, mix);
      return;
    }
  }
  // lane i <- code of member i: each nonzero word pushes its set bits to
  // consecutive lanes (lanes without a bit push to a lane outside the range)
  uint32_t mem = 0, base = 0;
  for (uint64_t cm = ballot(Cw != 0); cm; cm &= cm - 1) {
    const uint32_t k = ctz64(cm);
    const uint64_t w = rdlane64(Cw, k), pw = rdlane64(Pw, k);
    const uint32_t cnt = popc64(w);
    const bool in = lane_in(w);
    const uint32_t dst = in ? base + mbcnt(w) : (base + cnt) & 63u;
    const uint32_t code = (k * 64 + L) | (lane_in(pw) ? kMemP : 0u);
    const uint32_t got = (uint32_t)__builtin_amdgcn_ds_permute((int)(dst * 4), (int)code);
    if (L - base < cnt) mem = got;
    base += cnt;
  }
  for (uint64_t em = ballot(Ew != 0); em; em &= em - 1) {
    const uint32_t k = ctz64(em);
    const uint64_t w = rdlane64(Ew, k);
    const uint32_t cnt = popc64(w);
    const bool in = lane_in(w);
    const uint32_t dst = in ? base + mbcnt(w) : (base + cnt) & 63u;
    const uint32_t got = (uint32_t)__builtin_amdgcn_ds_permute((int)(dst * 4), (int)((k * 64 + L) | kMemOut));
    if (L - base < cnt) mem = got;
    base += cnt;
  }
  const uint32_t nm = base;
  const bool valid = L < nm;
  const uint64_t lP = ballot(valid && (mem & kMemP)), lX = ballot(valid && !(mem & kMemP));
  const uint64_t hs = lane_in(lP) ? ld64<kLA>(s.H, mem & 8191u) : 0ull;
  // rows over the members: only the bits of P's members are looked up; a P
  // member's own row over all members is its column of them
  uint64_t M = 0, left = lP;
  for (uint64_t pm = ballot(Pw != 0); pm; pm &= pm - 1) {
    const uint32_t k = ctz64(pm);
    const uint64_t pw = rdlane64(Pw, k), rw = row_word(mem, valid, k);
    for (uint32_t h = 0; h < 2; ++h) {
      const uint32_t rh = (uint32_t)(rw >> (32 * h));
      for (uint32_t m = (uint32_t)(pw >> (32 * h)); m; m &= m - 1, left &= left - 1) {
        const uint32_t at = uniform(ctz64(left));
        const uint32_t t = (rh >> __builtin_ctz(m)) & 1u;
        const uint64_t col = ballot(t != 0);
        M |= lane_in(lP) ? 0ull : (uint64_t)t << at;
        M = wrlane64(M, at, col);
      }
    }
  }
  // (the lane-solver instances keep one copy of the loop: most of what it
  // would solve with 32-bit masks is queued)
  if (!lane_of(kStat) && nm <= 32)
    small_loop<uint32_t, kStat>(pr, (uint32_t)M, hs, (uint32_t)lP, (uint32_t)lX, mix, rbase, s.root, hist_lds, wa, clk);
  else
    small_loop<uint64_t, kStat>(pr, M, hs, lP, lX, mix, rbase, s.root, hist_lds, wa, clk);
}

// Runs BK from (P, X, E) on an arena that build_bits (or a received task)
// has filled; kLA / kLX: S and A / the outside rows are in LDS.
template <bool kWL, int kStat, bool kLA, bool kLX>
__device__ __forceinline__ void solve_bits_t(const BkParams &pr, const Sub &s, uint64_t cP, uint64_t cX, uint64_t cE,
                                             lds_ull *hist_lds, WaveAcc &wa, Clock<kStat> &clk) {
  const uint32_t L = lane_id(), W = s.W, WX = s.WX;
  const bool act = L < W;
  uint32_t piv = 0;
  uint64_t cN = 0, mix = s.rmix;
  int32_t d = -1;  // -1: the root itself is the node to decide
  while (true) {
    uint64_t Pn = cP, Xn = cX, En = cE, cmix = mix;
    if (d >= 0) {
      if constexpr (kWL) {
        clk.to(kBdQueue);
        poll_idle(pr, wa);
        if (wa.budget > 0) {
          if (donate_bits<kLA, kLX>(pr, s, (uint32_t)d, cP, cX, cE, piv, mix, wa)) wa.budget--;
          else no_donation(pr, wa);
        }
      }
      clk.to(kBdSetOps);
      const uint64_t B = cP & ~cN;
      const uint64_t bm = ballot(B != 0);
      if (bm == 0) {
        if (d == 0) break;
        clk.to(kBdBranch);
        --d;
        if ((uint32_t)d < s.lds_levels) frame_get<true>(s.fr_lds + (uint64_t)d * s.FS, W, WX, cP, cX, cE, piv, mix);
        else frame_get<false>(s.fr_hbm + (uint64_t)(d - s.lds_levels) * s.FS, W, WX, cP, cX, cE, piv, mix);
        cN = pivot_word<kLA, kLX>(s, piv);
        continue;
      }
      const uint32_t k0 = ctz64(bm);
      const uint32_t bit = ctz64(rdlane64(B, k0));
      const uint32_t c = k0 * 64 + bit;
      {
        // c leaves P for X: one lane-select of the bit, then XOR (the bit is
        // set in P) and OR
        const uint64_t m = L == k0 ? (1ull << bit) : 0ull;
        cP ^= m;
        cX |= m;
      }
      const uint64_t Ac = act ? ld64<kLA>(s.A, (uint64_t)c * W + L) : 0;
      Pn = cP & Ac;
      Xn = cX & Ac;
      wa.nodes++;
      cmix = mix + uniform64(ld64<kLA>(s.H, c));
      const uint64_t pnz = ballot(Pn != 0);
      if (pnz == 0) {
        clk.to(kBdMaximal);
        if (ballot(Xn != 0) == 0 && !rows_any<kLX>(s, cE, c)) report(pr, hist_lds, wa, s.rsize + d + 1, cmix);
        continue;
      }
      En = filter_rows<kLX>(s, cE, c);
      const uint64_t pnz2 = pnz & (pnz - 1);
      if ((pnz2 & (pnz2 - 1)) == 0) {
        // |P| <= 2 decided without the pivot scan, node for node as the scan
        // would go (a pivot from X covering P leaves no child; ties go to the
        // lowest index, inside X before outside rows)
        const uint32_t k1 = ctz64(pnz);
        const uint64_t w1 = rdlane64(Pn, k1);
        const uint64_t w2 = pnz2 ? rdlane64(Pn, ctz64(pnz2)) : 0ull;
        const uint32_t np = popc64(w1) + popc64(w2);
        if (np == 1) {
          // P = {a}: either an X vertex or outside row adjacent to a is the
          // pivot and covers P, or a is the one child and a maximal clique
          clk.to(kBdMaximal);
          const uint32_t na = k1 * 64 + ctz64(w1);
          const uint64_t Aa = act ? ld64<kLA>(s.A, (uint64_t)na * W + L) : 0;
          if (ballot((Xn & Aa) != 0) == 0 && !rows_any<kLX>(s, En, na)) {
            wa.nodes++;
            report(pr, hist_lds, wa, s.rsize + d + 2, cmix + uniform64(ld64<kLA>(s.H, na)));
          }
          continue;
        }
        if (np == 2) {
          clk.to(kBdMaximal);
          const uint32_t na = k1 * 64 + ctz64(w1);
          const uint32_t nb = w2 ? (uint32_t)ctz64(pnz2) * 64 + ctz64(w2) : k1 * 64 + ctz64(w1 & (w1 - 1));
          const uint64_t Aa = act ? ld64<kLA>(s.A, (uint64_t)na * W + L) : 0;
          const uint64_t Ab = act ? ld64<kLA>(s.A, (uint64_t)nb * W + L) : 0;
          const uint64_t Ea = filter_rows<kLX>(s, En, na), Eb = filter_rows<kLX>(s, En, nb);
          const uint64_t Xa = Xn & Aa, Xb = Xn & Ab;
          if (ballot(((Xa & Xb) | (Ea & Eb)) != 0)) continue;  // a pivot covers P
          const uint64_t ha = uniform64(ld64<kLA>(s.H, na)), hb = uniform64(ld64<kLA>(s.H, nb));
          if ((rdlane64(Aa, nb >> 6) >> (nb & 63)) & 1ull) {
            // a ~ b: whichever pivot, the path is a then b (or b then a)
            wa.nodes += 2;
            report(pr, hist_lds, wa, s.rsize + d + 3, cmix + ha + hb);
            continue;
          }
          const uint64_t xs = Xa | Xb, es = Ea | Eb;
          const uint64_t xm = ballot(xs != 0), em = ballot(es != 0);
          if (xm == 0 && em == 0) {
            // all scores 0: children a and b, each a maximal clique
            wa.nodes += 2;
            report(pr, hist_lds, wa, s.rsize + d + 2, cmix + ha);
            report(pr, hist_lds, wa, s.rsize + d + 2, cmix + hb);
            continue;
          }
          // the pivot is the lowest X vertex (else outside row) adjacent to
          // exactly one of a, b; the child is the other, maximal iff nothing
          // in X or outside touches it
          bool piv_a;
          if (xm) {
            const uint32_t k = ctz64(xm);
            piv_a = (rdlane64(Xa, k) >> ctz64(rdlane64(xs, k))) & 1ull;
          } else {
            const uint32_t k = ctz64(em);
            piv_a = (rdlane64(Ea, k) >> ctz64(rdlane64(es, k))) & 1ull;
          }
          wa.nodes++;
          const uint64_t Xc = piv_a ? Xb : Xa, Ec = piv_a ? Eb : Ea;
          if (ballot((Xc | Ec) != 0) == 0) report(pr, hist_lds, wa, s.rsize + d + 2, cmix + (piv_a ? hb : ha));
          continue;
        }
      }
    }
    uint32_t np, nx;
    if (small_ok<kWL>(pr, Pn, Xn, En, np, nx)) {
      solve_small<kWL, kStat, kLA, kLX>(pr, s, Pn, Xn, En, np, nx, cmix, s.rsize + d + 1, hist_lds, wa, clk);
      if (d < 0) break;
      continue;
    }
    uint32_t npiv, nbest;
    clk.to(kBdPivot);
    pick_pivot_bits<kLA, kLX>(s, Pn, Xn, En, npiv, nbest);
    if (npiv == kNone || nbest == np) {  // nothing left, or a pivot that covers P
      if (d < 0) break;
      continue;
    }
    clk.to(kBdBranch);
    if (d >= 0) {
      if ((uint32_t)d < s.lds_levels) frame_put<true>(s.fr_lds + (uint64_t)d * s.FS, W, WX, cP, cX, cE, piv, mix);
      else frame_put<false>(s.fr_hbm + (uint64_t)(d - s.lds_levels) * s.FS, W, WX, cP, cX, cE, piv, mix);
    }
    ++d;
    cP = Pn;
    cX = Xn;
    cE = En;
    piv = npiv;
    mix = cmix;
    cN = pivot_word<kLA, kLX>(s, piv);
  }
}

// A subproblem's own labels: tree nodes and cliques from here to end_task.
__device__ __forceinline__ uint64_t begin_task(const Sub &s, WaveAcc &wa) {
  wa.sub_cliques = 0;
  wa.t_task = s.t0;
  return wa.nodes;
}
__device__ __forceinline__ void end_task(const BkParams &pr, const Sub &s, const WaveAcc &wa, uint64_t nodes0) {
  if (lane_id() == 0) {
    if (pr.sub_nodes) atomicAdd(&pr.sub_nodes[s.root], (unsigned long long)(wa.nodes - nodes0));
    if (pr.sub_cliques && wa.sub_cliques) atomicAdd(&pr.sub_cliques[s.root], (unsigned long long)wa.sub_cliques);
  }
}

// solve_bits_t as a function of its own, one per placement.
template <bool kWL, int kStat, bool kLA, bool kLX>
__device__ __noinline__ __attribute__((not_tail_called)) void solve_bits_fn(ConstParams *kargs, uint32_t io, uint64_t cP, uint64_t cX,
                                           uint64_t cE, uint32_t hist_lds_addr) {
  const BkParams &pr = *(const BkParams *)(ConstParams *)uniform64((uint64_t)kargs);
  LdsHandover *ho = handover(uniform(io));
  const Sub s = lds_get(&ho->s);
  WaveAcc wa = lds_get(&ho->w);
  Clock<kStat> clk;
  const uint64_t nodes0 = begin_task(s, wa);
  solve_bits_t<kWL, kStat, kLA, kLX>(pr, s, cP, cX, cE,
                                     (lds_ull *)(uintptr_t)uniform(hist_lds_addr), wa, clk);
  end_task(pr, s, wa, nodes0);
  lds_put(&ho->w, wa);
}

// (s is in the hand-over block already where the kernel uses functions)
template <bool kWL, int kStat>
__device__ __forceinline__ void solve_bits(const BkParams &pr, Sub &s, uint64_t cP, uint64_t cX, uint64_t cE,
                                           lds_ull *hist_lds, WaveAcc &wa, Clock<kStat> &clk) {
  if constexpr (fn_of(true, kStat)) {
    ConstParams *ka = (ConstParams *)__builtin_amdgcn_kernarg_segment_ptr();
    const uint32_t ha = (uint32_t)(uintptr_t)hist_lds;
    if (s.where == 3) solve_bits_fn<kWL, kStat, true, true>(ka, wa.io, cP, cX, cE, ha);
    else if (s.where == 1) solve_bits_fn<kWL, kStat, true, false>(ka, wa.io, cP, cX, cE, ha);
    else solve_bits_fn<kWL, kStat, false, false>(ka, wa.io, cP, cX, cE, ha);
    return;
  }
  const uint64_t nodes0 = begin_task(s, wa);
  if (s.where == 3) solve_bits_t<kWL, kStat, true, true>(pr, s, cP, cX, cE, hist_lds, wa, clk);
  else if (s.where == 1) solve_bits_t<kWL, kStat, true, false>(pr, s, cP, cX, cE, hist_lds, wa, clk);
  else solve_bits_t<kWL, kStat, false, false>(pr, s, cP, cX, cE, hist_lds, wa, clk);
  clk.to(kBdOther);
  end_task(pr, s, wa, nodes0);
}

// Intersection of ascending a[0,na) and b[0,nb) written to out (ascending);
// iterates the shorter list and binary-searches the longer.
__device__ __forceinline__ uint32_t intersect_in(const uint32_t *a, uint32_t na, const uint32_t *b, uint32_t nb, uint32_t *out) {
  if (na > nb) {
    const uint32_t *t = a;
    a = b;
    b = t;
    const uint32_t tn = na;
    na = nb;
    nb = tn;
  }
  uint32_t w = 0;
  for (uint32_t k0 = 0; k0 < na; k0 += kWave) {
    const uint32_t k = k0 + lane_id();
    bool hit = false;
    uint32_t y = 0;
    if (k < na) {
      y = a[k];
      const uint32_t j = lower_bound_u32(b, nb, y);
      hit = j < nb && b[j] == y;
    }
    const uint64_t m = ballot(hit);
    if (hit) out[w + mbcnt(m)] = y;
    w += popc64(m);
  }
  return w;
}
__device__ __noinline__ __attribute__((not_tail_called)) uint32_t intersect_fn(const uint32_t *a, uint32_t na,
                                                                               const uint32_t *b, uint32_t nb,
                                                                               uint32_t *out) {
  return intersect_in((const uint32_t *)uniform64((uint64_t)a), uniform(na), (const uint32_t *)uniform64((uint64_t)b),
                      uniform(nb), out);
}
template <bool kFn>
__device__ __forceinline__ uint32_t intersect_into(const uint32_t *a, uint32_t na, const uint32_t *b, uint32_t nb, uint32_t *out) {
  if constexpr (!kFn) return intersect_in(a, na, b, nb, out);
  return uniform(intersect_fn(a, na, b, nb, out));
}


__device__ __forceinline__ uint32_t hw_cu_id() {
  // HW_ID (hwreg 4): CU_ID [11:8], SH_ID [12], SE_ID [15:13]; XCC_ID (hwreg 20) [3:0]
  const uint32_t hw = __builtin_amdgcn_s_getreg((4) | (0 << 6) | (31 << 11));
  const uint32_t xcc = __builtin_amdgcn_s_getreg((20) | (0 << 6) | (3 << 11));
  const uint32_t cu = ((hw >> 8) & 0xF) | (((hw >> 12) & 1) << 4) | (((hw >> 13) & 7) << 5);
  return (xcc << 8) | cu;
}

// Records an item whose arena does not fit, for the large-arena pass. The
// slot is counted even past the capacity so the host can see an overrun.
__device__ __forceinline__ void defer(const BkParams &pr, uint64_t it) {
  if (lane_id() == 0) {
    const unsigned long long slot = atomicAdd(&pr.acc[kAccOverflow], 1ull);
    if (slot < pr.overflow_cap) pr.overflow[slot] = it;
  }
}


// The list path: builds the rows (a received task has them) and solves.
template <bool kIPX, bool kWL, int kStat, bool kBuild>
__device__ __noinline__ __attribute__((not_tail_called)) void solve_list_fn(ConstParams *kargs, uint32_t io, uint64_t cP, uint64_t cX,
                                           uint32_t hist_lds_addr) {
  const BkParams &pr = *(const BkParams *)(ConstParams *)uniform64((uint64_t)kargs);
  LdsHandover *ho = handover(uniform(io));
  Sub s = lds_get(&ho->s);
  WaveAcc wa = lds_get(&ho->w);
  Clock<kStat> clk;
  const uint64_t nodes0 = begin_task(s, wa);
  if constexpr (kBuild) build<kIPX>(pr, s);
  bk_solve<kIPX, kWL, kStat>(pr, s, cP, cX, (lds_ull *)(uintptr_t)uniform(hist_lds_addr), wa, clk);
  end_task(pr, s, wa, nodes0);
  lds_put(&ho->w, wa);
}
template <bool kIPX, bool kWL, int kStat, bool kBuild>
__device__ __forceinline__ void solve_list(const BkParams &pr, Sub &s, uint64_t cP, uint64_t cX,
                                           lds_ull *hist_lds, WaveAcc &wa, Clock<kStat> &clk) {
  if constexpr (fn_of(kIPX, kStat)) {
    lds_put(&handover(wa.io)->s, s);
    solve_list_fn<kIPX, kWL, kStat, kBuild>((ConstParams *)__builtin_amdgcn_kernarg_segment_ptr(), wa.io, cP, cX,
                                            (uint32_t)(uintptr_t)hist_lds);
    return;
  }
  const uint64_t nodes0 = begin_task(s, wa);
  clk.to(kBdInduced);
  if constexpr (kBuild) build<kIPX>(pr, s);
  bk_solve<kIPX, kWL, kStat>(pr, s, cP, cX, hist_lds, wa, clk);
  clk.to(kBdOther);
  end_task(pr, s, wa, nodes0);
}

template <bool kWL, int kStat>
__device__ __forceinline__ void finish_bits(const BkParams &pr, Sub &s, const uint32_t *ids, uint32_t q0, bool filter,
                                            uint64_t keep, lds_ull *hist_lds, WaveAcc &wa,
                                            Clock<kStat> &clk) {
  clk.to(kBdInduced);
  lds_put(&handover(wa.io)->s, s);
  ConstParams *ka = (ConstParams *)__builtin_amdgcn_kernarg_segment_ptr();
  const uint64_t E0 = s.where == 3   ? build_bits_fn<true, true>(ka, wa.io, ids, q0, keep, filter)
                      : s.where == 1 ? build_bits_fn<true, false>(ka, wa.io, ids, q0, keep, filter)
                                     : build_bits_fn<false, false>(ka, wa.io, ids, q0, keep, filter);
  solve_bits<kWL, kStat>(pr, s, full_word(s.p), 0, E0, hist_lds, wa, clk);
}

// The kernel's arguments, read again: values read before are not carried over
// the calls in between (which use all registers, so that they were stored to
// scratch memory and read back, 100 registers a subproblem).
template <bool kFn>
__device__ __forceinline__ const BkParams &fresh_params(const BkParams &args) {
  if constexpr (!kFn) return args;
  ConstParams *k = (ConstParams *)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(k));
  return *(const BkParams *)k;
}
// A subproblem of wave gw with nothing but the graph set.
__device__ __forceinline__ Sub fresh_sub(const BkParams &pr, uint32_t gw) {
  Sub s{};
  s.oc = pr.oc;
  s.rp = pr.rp;
  s.split = pr.split;
  s.cover = pr.cover + (uint64_t)gw * kWave;
  return s;
}

// Runs what is left in the wave's lane queue.
template <int kStat>
__device__ __noinline__ __attribute__((not_tail_called)) void ls_flush_fn(ConstParams *kargs, uint32_t io,
                                                                          uint32_t hist_lds_addr) {
  const BkParams &pr = *(const BkParams *)(ConstParams *)uniform64((uint64_t)kargs);
  LdsHandover *ho = handover(uniform(io));
  WaveAcc wa = lds_get(&ho->w);
  ls_flush<kStat>(pr, (lds_ull *)(uintptr_t)uniform(hist_lds_addr), wa);
  lds_put(&ho->w, wa);
}
template <int kStat>
__device__ __forceinline__ void finish_lanes(lds_ull *hist_lds, const WaveAcc &wa) {
  if constexpr (lane_of(kStat))
    ls_flush_fn<kStat>((ConstParams *)__builtin_amdgcn_kernarg_segment_ptr(), wa.io, (uint32_t)(uintptr_t)hist_lds);
}

template <bool kIPX, bool kWL, int kStat>
// At least four waves per SIMD (<= 128 VGPRs): occupancy hides the LDS and
// memory latency of the set operations better than registers would.
__global__ __launch_bounds__(max_wpg_of(kWL) * kWave, waves_per_simd_of(kWL)) void bk_kernel(BkParams args) {
  constexpr bool kFn = fn_of(kIPX, kStat);
  const BkParams &pr = args;
  extern __shared__ __align__(16) uint8_t smem[];
  lds_ull *hist_lds = (lds_ull *)smem;
  const uint32_t wig = threadIdx.x / kWave, L = lane_id();
  const uint32_t hb = (uint32_t)align8(8ull * pr.hist_lds);
  Pool pl;
  pl.mask = (uint64_t *)(smem + hb);
  pl.lock = (uint32_t *)(smem + hb + 8 * kPoolWords);
  pl.base = smem + hb + kPoolHeader;
  pl.ngran = pr.pool_bytes / kGranule;
  for (uint32_t i = threadIdx.x; i < pr.hist_lds; i += blockDim.x) hist_lds[i] = 0;
  if (threadIdx.x < kPoolWords) {
    const uint32_t lo = threadIdx.x * 64;
    pl.mask[threadIdx.x] = lo >= pl.ngran ? ~0ull : (lo + 64 <= pl.ngran ? 0ull : (~0ull << (pl.ngran - lo)));
  }
  if (threadIdx.x == 0) *pl.lock = 0;
  __syncthreads();
  const uint32_t lv = pr.want_levels;
  const uint32_t gw = blockIdx.x * pr.wpg + wig;
  uint8_t *hbm = pr.hbm + (uint64_t)gw * pr.hbm_bytes;
  WaveAcc wa;
  wa.io = (uint32_t)(uintptr_t)(smem + pr.io_off + wig * kHandoverBytes);
  if (lane_of(kStat)) {
    wa.ls = pr.ls + (uint64_t)gw * kLsBytes;
    wa.ls_lds = (uint32_t)(uintptr_t)(smem + pr.ls_off + wig * kLsLds);
  }
  wa.xq = (hw_cu_id() >> 8) % kQueues;
  wa.peek = wa.xq;
  Clock<kStat> clk;
  clk.start();
  // the totals live in the hand-over block while functions solve; of `wa`,
  // only io and xq are then used between here and the end
  if constexpr (kFn) lds_put(&handover(wa.io)->w, wa);
  // phase 1: first-level subproblems by ticket. A wave's first ticket is its
  // position in the grid (neighbouring tickets, the heaviest, on different
  // workgroups, so that they do not share a CU's LDS pool), the next ones
  // come from the counter: 11 ns each on its line, 45 us a launch of 4096
  // waves when their first ones came from it too.
  const uint32_t nwaves = gridDim.x * pr.wpg;
  uint32_t tickets = 0;
  while (true) {
    const BkParams &pr = fresh_params<kFn>(args);
    clk.to(kBdQueue);
    uint32_t t = wig * gridDim.x + blockIdx.x;
    if (tickets) {
      if (pr.n_items <= pr.t1 && pr.n_items <= nwaves) break;  // one each and no more
      if (L == 0) {
        t = nwaves + atomicAdd(pr.ticket, 1u);
        if (pr.host_progress && (t & 1023u) == 0) post_progress(pr.host_progress, t);
      }
      t = uniform(t);
    }
    uint64_t lo, hi;
    if (t < pr.t1) {
      lo = t;
      hi = t + 1;
    } else {
      lo = pr.t1 + (uint64_t)(t - pr.t1) * pr.chunk;
      hi = lo + pr.chunk;
    }
    if (lo >= pr.n_items) break;
    lo = uniform64(lo);
    hi = uniform64(min(hi, pr.n_items));
    ++tickets;
    clk.to(kBdInduced);
    for (uint64_t it = lo; it < hi; ++it) {
      const BkParams &pr = fresh_params<kFn>(args);
      const uint32_t *items1 = (const uint32_t *)pr.items;
      const uint2 *items2 = (const uint2 *)pr.items;
      Sub s = fresh_sub(pr, gw);
      s.t0 = __builtin_amdgcn_s_memrealtime();
      // level 1: vertex items; level 2: arc items; level 3: arc items where
      // (v, kNone) stands for the whole vertex subproblem of v
      bool vertex_item = pr.level == 1;
      uint32_t iv = 0;
      uint2 ia = make_uint2(0, 0);
      if (vertex_item) {
        iv = uniform(items1[it]);
      } else {
        ia = items2[it];
        ia.x = uniform(ia.x);
        ia.y = uniform(ia.y);
        if (pr.level == 3 && ia.y == kNone) {
          vertex_item = true;
          iv = ia.x;
        }
      }
      if (vertex_item) {
        const uint32_t v = iv;
        const uint64_t b0 = pr.rp[v], s0 = pr.split[v], e0 = pr.rp[v + 1];
        const uint32_t p = (uint32_t)(e0 - s0), q = (uint32_t)(s0 - b0);
        if (p == 0) continue;
        const uint32_t W = (p + 63) / 64;
        bool bits = kIPX && q <= kMaxXRows;
        // outside rows: all of them, or (many more than |P|, as at hubs) only
        // those with a neighbour in P, in order; a hub with more than 4096
        // earlier neighbours takes the bitmap path when its live rows, less
        // repeated one-neighbour rows, fit
        uint32_t qb = q;
        bool filter = false;
        if (kIPX && !bits) {
          qb = live_count(pr.oc + s0, p, pr.oc + b0, q, s.cover);
          bits = filter = qb <= kMaxXRows;
          if (!bits) qb = q;
        }
        const uint64_t keep = !bits || filter ? 0ull
                              : q > 2 * p     ? live_rows<kInGlb>(pr.oc + s0, p, pr.oc + b0, q, qb)
                                              : all_rows(q);
        const Region rg = bits ? pool_take_wait<kFn>(pl, bits_want(p, qb, W, lv), bits_want_inner(p, qb, W, lv),
                                                bits_fs(W, (qb + 63) / 64) * min(p, lv),
                                                bits_want_inner(p, qb, W, lv))
                               : pool_take_wait<kFn>(pl, list_want(p, q, W, kIPX, lv), 0, (16 * W + 16) * min(p, lv),
                                                list_want(p, q, W, kIPX, lv));
        if (!(bits ? place_bits(s, p, qb, W, rg.ptr, rg.bytes, hbm, pr.hbm_bytes, pr.stack_lds)
                   : place(s, p, q, W, kIPX, rg.ptr, rg.bytes, hbm, pr.hbm_bytes, pr.stack_lds))) {
          pool_put<kFn>(pl, rg);
          defer(pr, it);
          continue;
        }
        s.p = p;
        s.q = bits ? qb : q;
        s.W = W;
        s.rsize = 1;
        s.root = v;
        s.rmix = splitmix64(v);
        for (uint32_t i = L; i < p; i += kWave) s.S[i] = pr.oc[s0 + i];
        if (bits) {
          finish_bits<kWL, kStat>(pr, s, pr.oc + b0, q, filter, keep, hist_lds, wa, clk);
        } else {
          for (uint32_t i = L; i < q; i += kWave) s.XL[i] = pr.oc[b0 + i];
          solve_list<kIPX, kWL, kStat, true>(pr, s, full_word(p), 0, hist_lds, wa, clk);
        }
        pool_put<kFn>(pl, rg);
      } else {
        const uint32_t u = ia.x, w = ia.y;
        const uint64_t su = pr.split[u], eu = pr.rp[u + 1], bu = pr.rp[u];
        const uint64_t sw = pr.split[w], ew = pr.rp[w + 1], bw = pr.rp[w];
        const uint32_t pb = (uint32_t)min(eu - su, ew - sw), qb = (uint32_t)min(eu - bu, sw - bw);
        Sub t = s;
        const uint32_t Wb = (pb + 63) / 64;
        const Region rg = pool_take_wait<kFn>(pl, list_want(pb, qb, Wb, kIPX, lv), 0, (16 * Wb + 16) * min(pb, lv),
                                         list_want(pb, qb, Wb, kIPX, lv));
        if (!place(t, pb, qb, Wb, kIPX, rg.ptr, rg.bytes, hbm, pr.hbm_bytes, pr.stack_lds)) {
          pool_put<kFn>(pl, rg);
          defer(pr, it);
          continue;
        }
        const uint32_t p = intersect_into<kFn>(pr.oc + su, (uint32_t)(eu - su), pr.oc + sw, (uint32_t)(ew - sw), t.S);
        const uint32_t q = intersect_into<kFn>(pr.ci + bu, (uint32_t)(eu - bu), pr.oc + bw, (uint32_t)(sw - bw), t.XL);
        const uint64_t rmix = splitmix64(u) + splitmix64(w);
        if (p == 0) {
          if (q == 0) {
            LdsHandover *ho = handover(wa.io);
            if constexpr (kFn) {
              WaveAcc w = lds_get(&ho->w);
              report(pr, hist_lds, w, 2, rmix);
              lds_put(&ho->w, w);
            } else {
              report(pr, hist_lds, wa, 2, rmix);
            }
            if (pr.sub_cliques && L == 0) atomicAdd(&pr.sub_cliques[u], 1ull);
          }
          pool_put<kFn>(pl, rg);
          continue;
        }
        // re-lay the arena for the actual sizes (and, bitmap path, the kept rows)
        const uint32_t W = (p + 63) / 64;
        const bool bits = kIPX && q <= kMaxXRows;
        uint32_t qk = q;
        const uint64_t keep = !bits ? 0ull : q > 2 * p ? live_rows<kAnywhere>(t.S, p, t.XL, q, qk) : all_rows(q);
        if (!(bits ? place_bits(s, p, qk, W, rg.ptr, rg.bytes, hbm, pr.hbm_bytes, pr.stack_lds)
                   : place(s, p, q, W, kIPX, rg.ptr, rg.bytes, hbm, pr.hbm_bytes, pr.stack_lds))) {
          pool_put<kFn>(pl, rg);
          defer(pr, it);
          continue;
        }
        // the bitmap layout ends before the staging list t.XL when both share
        // a base, and lives in a different memory otherwise
        if (s.S != t.S) wave_copy(s.S, t.S, p);
        if (!bits && s.XL != t.XL) wave_copy(s.XL, t.XL, q);
        s.p = p;
        s.q = bits ? qk : q;
        s.W = W;
        s.rsize = 2;
        s.root = u;
        s.rmix = rmix;
        if (bits) finish_bits<kWL, kStat>(pr, s, t.XL, q, false, keep, hist_lds, wa, clk);
        else solve_list<kIPX, kWL, kStat, true>(pr, s, full_word(p), 0, hist_lds, wa, clk);
        pool_put<kFn>(pl, rg);
      }
    }
  }
  clk.to(kBdSetOps);
  finish_lanes<kStat>(hist_lds, wa);
  // (the launch cannot end before this wave gets here: its tickets leave the
  // outstanding count together)
  if (kWL && tickets) tasks_done(pr, tickets);
  // phase 2: donated subtrees until no work is outstanding. An idle wave puts
  // itself on the idle queue and waits on its own mailbox line; a donor takes
  // it off the queue and writes the task into its slot, so no line is polled
  // by many waves. The receiver takes LDS from its pool once the task is in
  // (holding LDS while idle would starve the waves still at work).
  if constexpr (kWL) {
    bool registered = false;
    Region rsv{pl.base, 0, 0, 0};
    uint32_t backoff = 1, polls = 0;
    uint64_t t0 = __builtin_amdgcn_s_memrealtime();
    unsigned long long seen_out = ~0ull, seen_beat = ~0ull;
    const uint8_t *slot = pr.ring + (uint64_t)gw * pr.slot_bytes;
    while (true) {
      clk.to(kBdQueue);
      if (!registered) registered = register_idle(pr, gw, wa.xq);
      if (registered) {
        const unsigned long long got = uniform64(L == 0 ? ld_relaxed(&pr.mbox[(uint64_t)gw * kMboxStride]) : 0ull);
        if (got == kMboxDone) break;
        if (got) {
          const BkParams &pr = fresh_params<kFn>(args);
          Sub s = fresh_sub(pr, gw);
          registered = false;
          backoff = 1;
          // (empty again before this wave can be registered again; it stays
          // empty until then, with this task outstanding)
          if (L == 0) st_shared(&pr.mbox[(uint64_t)gw * kMboxStride], 0ull);
          drain();
          const uint64_t *h = (const uint64_t *)slot;
          const uint64_t h0 = uniform64(ld_shared(h)), h1 = uniform64(ld_shared(h + 1)), h2 = uniform64(ld_shared(h + 2)),
                         rmix = uniform64(ld_shared(h + 3));
          const uint32_t root = (uint32_t)h0, rsize = (uint32_t)(h0 >> 32), p = (uint32_t)h1, W = (uint32_t)(h1 >> 32),
                         nx = (uint32_t)h2, kind = (uint32_t)(h2 >> 32);
          if (kIPX && kind == kTaskBits) {
            const bool shape = p <= pr.slot_pmax && W == (p + 63) / 64 && nx <= pr.slot_xcap && nx <= kMaxXRows;
            if (shape)
              rsv = pool_take_wait<kFn>(pl, bits_want(p, nx, W, lv), bits_want_inner(p, nx, W, lv),
                                   bits_fs(W, (nx + 63) / 64) * min(p, lv), bits_want_inner(p, nx, W, lv));
            const Region rg = rsv;
            const bool okb = shape && place_bits(s, p, nx, W, rg.ptr, rg.bytes, hbm, pr.hbm_bytes, pr.stack_lds);
            uint64_t P0 = 0, X0 = 0, E0 = 0;
            if (okb) {
              const uint64_t *sp = (const uint64_t *)(slot + pr.slot_oP);
              if (L < W) {
                P0 = ld_shared(sp + L);
                X0 = ld_shared(sp + pr.slot_wmax + L);
              }
              if (L < s.WX) E0 = ld_shared(sp + 2 * pr.slot_wmax + L);
              wave_copy<false, true>(s.S, (const uint32_t *)(slot + pr.slot_oS), p);
              copy64<false, true>(s.A, (const uint64_t *)(slot + pr.slot_oA), (uint64_t)p * W);
              copy64<false, true>(s.XR, (const uint64_t *)(slot + pr.slot_oXR), (uint64_t)nx * W);
              s.p = p;
              fill_hash_terms(s);
            }
            if (okb) {
              __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
              s.p = p;
              s.q = nx;
              s.W = W;
              s.rsize = rsize;
              s.root = root;
              s.rmix = rmix;
              s.t0 = __builtin_amdgcn_s_memrealtime();
              if constexpr (kFn) lds_put(&handover(wa.io)->s, s);
              solve_bits<kWL, kStat>(pr, s, P0, X0, E0, hist_lds, wa, clk);
              finish_lanes<kStat>(hist_lds, wa);  // before the task counts as done
            } else if (L == 0) {
              atomicOr(&pr.acc[kAccError], 2ull);
            }
            tasks_done(pr, 1);
            pool_put<kFn>(pl, rsv);
            rsv = Region{pl.base, 0, 0, 0};
            t0 = __builtin_amdgcn_s_memrealtime();
            continue;
          }
          const bool shape = kind == kTaskList && p <= pr.slot_pmax && W == (p + 63) / 64 && nx <= pr.slot_xcap;
          if (shape)
            rsv = pool_take_wait<kFn>(pl, list_want(p, nx, W, kIPX, lv), 0, (16 * W + 16) * min(p, lv),
                                 list_want(p, nx, W, kIPX, lv));
          const Region rg = rsv;
          const bool ok = shape && place(s, p, nx, W, kIPX, rg.ptr, rg.bytes, hbm, pr.hbm_bytes, pr.stack_lds);
          uint64_t P0 = 0, X0 = 0;
          if (ok) {
            const uint64_t *sp = (const uint64_t *)(slot + pr.slot_oP);
            if (L < W) {
              P0 = ld_shared(sp + L);
              X0 = ld_shared(sp + pr.slot_wmax + L);
            }
            wave_copy<false, true>(s.S, (const uint32_t *)(slot + pr.slot_oS), p);
            copy64<false, true>(s.A, (const uint64_t *)(slot + pr.slot_oA), (uint64_t)p * W);
            const uint32_t *sXI = (const uint32_t *)(slot + pr.slot_oXI);
            if (kIPX) {
              wave_copy<false, true>(s.XV, sXI, nx);
              copy64<false, true>(s.XR, (const uint64_t *)(slot + pr.slot_oXR), (uint64_t)nx * W);
              for (uint32_t i = L; i < nx; i += kWave) s.XL[i] = i;
            } else {
              wave_copy<false, true>(s.XL, sXI, nx);
            }
          }
          if (ok) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            s.p = p;
            s.q = nx;
            s.W = W;
            s.xe0 = nx;
            s.rsize = rsize;
            s.root = root;
            s.rmix = rmix;
            s.t0 = __builtin_amdgcn_s_memrealtime();
            solve_list<kIPX, kWL, kStat, false>(pr, s, P0, X0, hist_lds, wa, clk);
          } else if (L == 0) {
            atomicOr(&pr.acc[kAccError], 2ull);  // donors only publish what fits
          }
          tasks_done(pr, 1);
          pool_put<kFn>(pl, rsv);
          rsv = Region{pl.base, 0, 0, 0};
          t0 = __builtin_amdgcn_s_memrealtime();
          continue;
        }
      }
      // the shared outstanding count is read every 16th poll only
      if ((++polls & 15) == 0 || !registered) {
        const unsigned long long out = uniform64(L == 0 ? ld_relaxed(pr.ctl + kCtlOutstanding) : 0);
        if (out == 0) break;
        const unsigned long long beat = uniform64(L == 0 ? ld_relaxed(pr.ctl + kCtlProgress) : 0);
        if (out != seen_out || beat != seen_beat) {
          // some wave made progress: the wait starts over
          seen_out = out;
          seen_beat = beat;
          t0 = __builtin_amdgcn_s_memrealtime();
        }
      }
      if (__builtin_amdgcn_s_memrealtime() - t0 > pr.watchdog_ticks) {
        if (L == 0) atomicOr(&pr.acc[kAccError], 1ull);
        break;
      }
      // a registered wave polls only its own line: short sleeps
      for (uint32_t z = 0; z < backoff; ++z) __builtin_amdgcn_s_sleep(32);
      backoff = min(backoff * 2, registered ? 16u : 64u);
    }
    pool_put<kFn>(pl, rsv);
  }
  clk.to(kBdOther);
  if constexpr (kFn) wa = lds_get(&handover(wa.io)->w);
  if (L == 0) {
    if (pr.wave_val) {
      pr.wave_val[gw] = kStat == kStatDonor ? wa.donations : wa.nodes;
      pr.wave_cu[gw] = hw_cu_id();
    }
    if constexpr (kStat == kStatBd) {
      if (pr.wave_bd)
        for (int i = 0; i < 7; ++i) pr.wave_bd[(uint64_t)gw * 7 + i] = clk.acc[i];
    }
  }
  wa.count += wa.ls_count;
  wa.nodes += wa.ls_nodes;
  // totals: summed over the workgroup in the pool's mask words (the pool is
  // done), one update each and workgroup (five by every wave, on one line,
  // were 0.2 ms of every launch)
  unsigned long long *tot = (unsigned long long *)pl.mask;
  static_assert(kPoolWords >= 5 && kAccCount == 0 && kAccHash == 1 && kAccNodes == 2 && kAccDonations == 3,
                "tot[0..3] in the order of acc, then the maximum size");
  __syncthreads();
  if (threadIdx.x < 5) tot[threadIdx.x] = 0;
  __syncthreads();
  if (L == 0 && wa.nodes + wa.count) {
    atomicAdd(&tot[kAccCount], (unsigned long long)wa.count);
    atomicAdd(&tot[kAccHash], (unsigned long long)wa.hash);
    atomicAdd(&tot[kAccNodes], (unsigned long long)wa.nodes);
    atomicAdd(&tot[kAccDonations], (unsigned long long)wa.donations);
    atomicMax(&tot[4], (unsigned long long)wa.max_size);
  }
  __syncthreads();
  if (threadIdx.x < 4 && tot[threadIdx.x]) atomicAdd(&pr.acc[threadIdx.x], tot[threadIdx.x]);
  if (threadIdx.x == 4 && tot[4] > ld_relaxed(&pr.acc[kAccMaxSize])) atomicMax(&pr.acc[kAccMaxSize], tot[4]);
  for (uint32_t i = threadIdx.x; i < pr.hist_lds; i += blockDim.x)
    if (const unsigned long long h = hist_lds[i]) atomicAdd(&pr.hist[min(i, pr.hist_len - 1)], h);
}

__global__ void reset_kernel(unsigned long long *acc, uint32_t n, uint32_t *ticket) {
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) acc[i] = 0;
  if (threadIdx.x == 0) *ticket = 0;
}

__global__ void ring_init(unsigned long long *seq, uint32_t cap, unsigned long long *ctl, unsigned long long outstanding,
                          unsigned long long *mbox) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < cap; i += gridDim.x * blockDim.x) {
    for (uint32_t q = 0; q < kQueues; ++q) seq[(uint64_t)q * cap + i] = i;
    mbox[(uint64_t)i * kMboxStride] = 0;
  }
  if (blockIdx.x == 0 && threadIdx.x < kCtlWords) ctl[threadIdx.x] = threadIdx.x == kCtlOutstanding ? outstanding : 0;
}

// Largest HBM arena any item needs, and how many need more than `cap`.
__global__ void need_kernel(const uint64_t *rp, const uint64_t *split, const void *items, uint64_t n_items,
                            uint32_t level, bool ipx, uint64_t cap, unsigned long long *out) {
  unsigned long long mx = 0, over = 0;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_items; i += stride) {
    uint32_t p, q;
    bool arc = false;
    if (level == 1) {
      const uint32_t v = ((const uint32_t *)items)[i];
      p = (uint32_t)(rp[v + 1] - split[v]);
      q = (uint32_t)(split[v] - rp[v]);
    } else {
      const uint2 a = ((const uint2 *)items)[i];
      if (level == 3 && a.y == kNone) {
        p = (uint32_t)(rp[a.x + 1] - split[a.x]);
        q = (uint32_t)(split[a.x] - rp[a.x]);
      } else {
        arc = true;
        p = (uint32_t)min(rp[a.x + 1] - split[a.x], rp[a.y + 1] - split[a.y]);
        q = (uint32_t)min(rp[a.x + 1] - rp[a.x], split[a.y] - rp[a.y]);
      }
    }
    const uint64_t need = item_need(p, q, arc, ipx);
    mx = max(mx, (unsigned long long)need);
    over += need > cap;
  }
  // one update per workgroup, and only of a maximum that it raises
  __shared__ unsigned long long smx, sover;
  if (threadIdx.x == 0) smx = sover = 0;
  __syncthreads();
  atomicMax(&smx, mx);
  if (over) atomicAdd(&sover, over);
  __syncthreads();
  if (threadIdx.x == 0) {
    if (smx > ld_relaxed(&out[0])) atomicMax(&out[0], smx);
    if (sover) atomicAdd(&out[1], sover);
  }
}

template <bool kIPX, bool kWL, int kStat>
int launch_one(const BkParams &pr, uint32_t groups, uint32_t wpg, size_t lds, hipStream_t s) {
  auto kern = bk_kernel<kIPX, kWL, kStat>;
  MCE_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(kern, dim3(groups), dim3(wpg * kWave), lds, s, pr);
  MCE_HIP(hipGetLastError());
  return MCE_OK;
}

template <bool kIPX, bool kWL, int kStat>
int occupancy_one(int *nb, uint32_t wpg, size_t lds) {
  MCE_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(nb, bk_kernel<kIPX, kWL, kStat>, wpg * kWave, lds));
  return MCE_OK;
}

template <bool kIPX, bool kWL>
int dispatch_stat(int stat, bool occ, int *nb, const BkParams &pr, uint32_t groups, uint32_t wpg, size_t lds,
                  hipStream_t s) {
  switch (stat) {
    case kStatLb:
      return occ ? occupancy_one<kIPX, kWL, kStatLb>(nb, wpg, lds)
                 : launch_one<kIPX, kWL, kStatLb>(pr, groups, wpg, lds, s);
    case kStatDonor:
      return occ ? occupancy_one<kIPX, kWL, kStatDonor>(nb, wpg, lds)
                 : launch_one<kIPX, kWL, kStatDonor>(pr, groups, wpg, lds, s);
    case kStatBd:
      return occ ? occupancy_one<kIPX, kWL, kStatBd>(nb, wpg, lds)
                 : launch_one<kIPX, kWL, kStatBd>(pr, groups, wpg, lds, s);
    case kStatLane:
      // the lane solver lives in the bitmap path, which only IPX takes
      if constexpr (kIPX)
        return occ ? occupancy_one<kIPX, kWL, kStatLane>(nb, wpg, lds)
                   : launch_one<kIPX, kWL, kStatLane>(pr, groups, wpg, lds, s);
      [[fallthrough]];
    default:
      return occ ? occupancy_one<kIPX, kWL, kStatNone>(nb, wpg, lds)
                 : launch_one<kIPX, kWL, kStatNone>(pr, groups, wpg, lds, s);
  }
}

// Launches (occ == false) or sizes (occ == true) the kernel variant.
int dispatch(bool ipx, bool wl, int stat, bool occ, int *nb, const BkParams &pr, uint32_t groups, uint32_t wpg,
             size_t lds, hipStream_t s) {
  if (ipx)
    return wl ? dispatch_stat<true, true>(stat, occ, nb, pr, groups, wpg, lds, s)
              : dispatch_stat<true, false>(stat, occ, nb, pr, groups, wpg, lds, s);
  return wl ? dispatch_stat<false, true>(stat, occ, nb, pr, groups, wpg, lds, s)
            : dispatch_stat<false, false>(stat, occ, nb, pr, groups, wpg, lds, s);
}

int stat_of(int task) {
  switch (task) {
    case MCE_TASK_LB_EVAL: return kStatLb;
    case MCE_TASK_DONOR_EVAL: return kStatDonor;
    case MCE_TASK_BD_EVAL: return kStatBd;
    default: return kStatNone;
  }
}

}  // namespace

void *Workspace::get(int slot, size_t n) {
  n = std::max<size_t>(n, 1);
  if (bytes[slot] >= n) return p[slot];
  if (p[slot]) {
    (void)hipFree(p[slot]);
    p[slot] = nullptr;
    bytes[slot] = 0;
  }
  if (hipMalloc(&p[slot], n) != hipSuccess) {
    p[slot] = nullptr;
    return nullptr;
  }
  bytes[slot] = n;
  return p[slot];
}

size_t Workspace::held() const {
  size_t b = 0;
  for (int k : {kWsArena, kWsRing, kWsSeq, kWsIdle, kWsMbox}) b += bytes[k];
  return b;
}

void Workspace::drop_graph() {
  if (exec) (void)hipGraphExecDestroy(exec);
  if (graph) (void)hipGraphDestroy(graph);
  exec = nullptr;
  graph = nullptr;
  key.clear();
}

void Workspace::release() {
  drop_graph();
  for (int k = 0; k < kWsSlots; ++k) {
    if (p[k]) (void)hipFree(p[k]);
    p[k] = nullptr;
    bytes[k] = 0;
  }
  if (pinned) (void)hipHostFree(pinned);
  pinned = nullptr;
}

// Waits for the enumeration launch on `s`. With progress_s > 0 it prints the
// launch's own counters to stderr every progress_s seconds while it runs:
// the kernel posts a recent ticket claim and (worker list) its heartbeat
// count (one per kBeatNodes tree nodes of a long task) into `posted`, pinned
// host memory.
static int wait_launch(hipStream_t s, uint32_t progress_s, const volatile unsigned long long *posted,
                       uint64_t n_tickets, bool wl) {
  if (progress_s && posted) {
    const auto t0 = std::chrono::steady_clock::now();
    auto next = t0 + std::chrono::seconds(progress_s);
    hipError_t e;
    while ((e = hipStreamQuery(s)) == hipErrorNotReady) {
      std::this_thread::sleep_for(std::chrono::milliseconds(20));
      if (std::chrono::steady_clock::now() < next) continue;
      next += std::chrono::seconds(progress_s);
      const double el = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
      fprintf(stderr, "[mce] enumeration %.0f s: about %llu of %llu tickets claimed", el,
              (unsigned long long)std::min<uint64_t>(posted[0], n_tickets), (unsigned long long)n_tickets);
      if (wl) fprintf(stderr, ", %llu heartbeats", (unsigned long long)posted[1]);
      fprintf(stderr, "\n");
      fflush(stderr);
    }
    if (e != hipSuccess) return hip_fail(e, "enumeration launch");
  }
  MCE_HIP(hipStreamSynchronize(s));
  return MCE_OK;
}

int bk_run(const DevGraph &g, const OrderInfo &info, const void *d_items, uint64_t n_items, const BkLaunch &cfg,
           uint64_t *d_hist, uint32_t hist_len, uint64_t *d_sub_nodes, uint64_t *d_sub_cliques,
           mce_wave_stat *wave_stats, uint32_t wave_stats_cap, uint32_t *wave_stats_len, hipStream_t s, BkOut *out,
           Scratch *sc, Workspace *ws) {
  *out = BkOut{};
  if (wave_stats_len) *wave_stats_len = 0;
  if (sc && (cfg.wl || wave_stats || cfg.capture))
    return set_error(MCE_EINVAL, "the allocation-free launch has no worker list, per-wave statistics or capture");
  if (n_items == 0) return MCE_OK;
  if (info.max_out_degree > MCE_MAX_OUT_DEGREE)
    return set_error(MCE_ELIMIT, "out-degree %u exceeds the engine limit %u", info.max_out_degree,
                     MCE_MAX_OUT_DEGREE);
  int dev = 0;
  MCE_HIP(hipGetDevice(&dev));
  int cus = 0;
  MCE_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  // the lane solver runs in its own kernel instance (IPX, no statistics)
  const uint32_t ls_max = stat_of(cfg.task) == kStatNone && cfg.ipx ? std::min<uint32_t>(cfg.lane_max, kLsP + kLsX) : 0;
  const int stat = ls_max ? kStatLane : stat_of(cfg.task);
  const uint32_t hist_lds = std::min<uint32_t>(hist_len, 128);
  const size_t hist_bytes = (8ull * hist_lds + 7) & ~7ull;
  const size_t lds_cu = 160 * 1024;
  // Waves per workgroup: by default all the waves the registers let one CU
  // hold, in as few workgroups as the launch bound allows, so that one LDS
  // pool serves the whole CU.
  const uint32_t max_wpg = max_wpg_of(cfg.wl);
  uint32_t wpg = cfg.waves_per_group;
  uint32_t groups_cu = std::max<uint32_t>(cfg.groups_per_cu, 1);
  if (!wpg) {
    int nb_regs = 0;
    BkParams probe{};
    int rc0 = dispatch(cfg.ipx, cfg.wl, stat, true, &nb_regs, probe, 0, 4, hist_bytes + kPoolHeader + 4096, s);
    if (rc0) return rc0;
    // (never more than the four waves per SIMD that buffers and pools are
    // sized for, also where an instance needs fewer registers)
    const uint32_t waves_cu = 4 * std::min((uint32_t)std::max(nb_regs, 1), waves_per_simd_of(cfg.wl));
    groups_cu = std::max<uint32_t>(groups_cu, (waves_cu + max_wpg - 1) / max_wpg);
    wpg = std::max<uint32_t>(1, waves_cu / groups_cu);
  }
  wpg = std::max<uint32_t>(1, std::min<uint32_t>(wpg, max_wpg));
  // the waves' hand-over blocks and the lane solver's LDS parts follow the pool
  const size_t ls_total = (kHandoverBytes + (ls_max ? (size_t)kLsLds : 0)) * wpg;
  const size_t fixed = hist_bytes + kPoolHeader + ls_total, share = lds_cu / groups_cu;
  size_t pool = cfg.lds_bytes ? (size_t)cfg.lds_bytes * wpg : share > fixed + kGranule ? share - fixed : kGranule;
  pool = std::min<size_t>(pool, lds_cu - fixed);
  pool = std::min<size_t>(pool, (size_t)kPoolWords * 64 * kGranule) / kGranule * kGranule;
  const size_t lds = fixed + pool;
  if (lds > lds_cu) return set_error(MCE_EINVAL, "LDS per workgroup %zu exceeds 160 KiB", lds);

  // every device buffer of this call: carved from the caller's scratch
  // region, kept in the graph's workspace slot `slot` (slot >= 0), or
  // allocated for this call and released on all paths
  std::vector<void *> bufs;
  auto dmalloc = [&](void **p, size_t bytes, int slot) -> int {
    if (sc) {
      *p = sc->take(std::max<size_t>(bytes, 1));
      if (!*p) return set_error(MCE_ELIMIT, "scratch region too small: %zu more bytes needed", bytes);
      return MCE_OK;
    }
    if (ws && slot >= 0) {
      *p = ws->get(slot, bytes);
      if (!*p) return set_error(MCE_ENOMEM, "device allocation of %zu bytes failed", bytes);
      return MCE_OK;
    }
    if (hipMalloc(p, std::max<size_t>(bytes, 1)) != hipSuccess)
      return set_error(MCE_ENOMEM, "device allocation of %zu bytes failed", bytes);
    bufs.push_back(*p);
    return MCE_OK;
  };
  struct Free {
    std::vector<void *> &b;
    ~Free() {
      for (void *p : b) hipFree(p);
    }
  } release{bufs};
  int rc;

  unsigned long long *acc = nullptr;
  uint32_t *ticket = nullptr;
  // counters, the 2 need words and the ticket in one buffer
  if ((rc = dmalloc((void **)&acc, sizeof(unsigned long long) * (kAccN + 3), kWsAcc))) return rc;
  ticket = (uint32_t *)(acc + kAccN + 2);
  unsigned long long *need = acc + kAccN;
  MCE_HIP(hipMemsetAsync(acc, 0, sizeof(unsigned long long) * (kAccN + 3), s));
  // hub row filter: 64 words per wave, for every wave a launch can hold (four
  // per SIMD), taken before the arenas size themselves to what is left
  uint64_t *cover = nullptr;
  const uint32_t max_waves = (uint32_t)cus * 16;
  if (cfg.ipx && (rc = dmalloc((void **)&cover, 8ull * kWave * max_waves, kWsCover))) return rc;
  // per-wave HBM arena cap: items that need more are deferred to a second
  // pass with arenas sized for the largest. From a scratch region, one
  // workgroup's arenas must fit what is left of it, and there is no second
  // pass.
  uint64_t cap = cfg.hbm_bytes ? cfg.hbm_bytes : 16ull << 20;
  if (sc) cap = std::min<uint64_t>(cap, (sc->left() / wpg) & ~255ull);
  // (with small maxima the need of an item that has them all stands for the
  // largest: the kernel, the copy and the wait for it are 25 us)
  unsigned long long hneed[2] = {item_need(info.max_out_degree, info.max_in_degree, cfg.level != 1, cfg.ipx), 0};
  if (cfg.level == 3)
    hneed[0] = std::max<unsigned long long>(hneed[0], item_need(info.max_out_degree, info.max_in_degree, false, cfg.ipx));
  if (sc || info.max_in_degree > kMaxXRows || hneed[0] > kSmallNeed || hneed[0] > cap) {
    need_kernel<<<(uint32_t)std::min<uint64_t>(1024, (n_items + 255) / 256), 256, 0, s>>>(g.rp, g.split, d_items, n_items, (uint32_t)cfg.level, cfg.ipx, cap, need);
    MCE_HIP(hipMemcpyAsync(hneed, need, sizeof(hneed), hipMemcpyDeviceToHost, s));
    MCE_HIP(hipStreamSynchronize(s));
  }
  if (sc && hneed[1])
    return set_error(MCE_ELIMIT, "%llu subproblems need more than the %llu scratch bytes per wave left (largest: %llu)",
                     (unsigned long long)hneed[1], (unsigned long long)cap, (unsigned long long)hneed[0]);

  int nb = 0;
  BkParams pr{};
  if ((rc = dispatch(cfg.ipx, cfg.wl, stat, true, &nb, pr, 0, wpg, lds, s))) return rc;
  nb = std::max(nb, 1);
  if (cfg.groups_per_cu) nb = std::min<int>(nb, (int)cfg.groups_per_cu);
  uint32_t groups = (uint32_t)(nb * cus);  // all waves co-resident
  uint64_t arena = std::min<uint64_t>(hneed[0], cap);
  arena = (arena + 255) & ~255ull;
  size_t freeb = 0, totalb = 0;
  if (sc) {
    freeb = 4 * sc->left();  // the arenas may take all that is left
  } else {
    MCE_HIP(hipMemGetInfo(&freeb, &totalb));
    if (ws) freeb += ws->held();  // kept buffers are reused or regrown
  }
  if (arena && (uint64_t)groups * wpg * arena > freeb / 4)
    groups = (uint32_t)std::max<uint64_t>(1, (freeb / 4) / ((uint64_t)wpg * arena));
  // Worker list: one task slot per wave. A slot holds a donor's vertex set
  // and bit matrix, the child's P/X words (and the 64-word outside-row
  // bitmap) and its outside-X ids (and rows with IPX). The outside-X capacity
  // covers the largest in-degree when the ring fits a quarter of the free
  // memory, else what that budget leaves (at least 64: a child with more
  // outside X is then not donated); when even 64 do not fit, fewer waves run.
  uint64_t slot_fixed = 0, slot_per_x = 0, slot_xcap = 0;
  uint32_t slot_pmax = 0, slot_wmax = 0;
  if (cfg.wl) {
    slot_pmax = std::max<uint32_t>(info.max_out_degree, 1);
    slot_wmax = (slot_pmax + 63) / 64;
    slot_fixed = kSlotHeader + 8ull * (2 * slot_wmax + 64) + align8(4ull * slot_pmax) + 8ull * slot_pmax * slot_wmax;
    slot_per_x = 4ull + (cfg.ipx ? 8ull * slot_wmax : 0);
    const uint64_t want_x = std::max<uint64_t>(info.max_in_degree, 64);
    const uint64_t budget = freeb / 4;
    const uint64_t min_slot = slot_fixed + 64 * slot_per_x + 512;
    if ((uint64_t)groups * wpg * min_slot > budget) {
      groups = (uint32_t)(budget / ((uint64_t)wpg * min_slot));
      if (!groups) return set_error(MCE_ENOMEM, "worker-list task slots of %llu bytes do not fit in device memory",
                                    (unsigned long long)min_slot);
    }
    const uint64_t per_slot = budget / ((uint64_t)groups * wpg);
    slot_xcap = std::min<uint64_t>(want_x, (per_slot - slot_fixed - 512) / slot_per_x);
  }
  // without the worker list, workgroups past one per item have nothing to do
  if (!cfg.wl && !wave_stats) groups = (uint32_t)std::min<uint64_t>(groups, n_items);
  const uint32_t waves = groups * wpg;

  uint8_t *hbm = nullptr;
  uint64_t *overflow = nullptr;
  unsigned long long *wave_val = nullptr, *wave_bd = nullptr;
  uint32_t *wave_cu = nullptr;
  if (arena && (rc = dmalloc((void **)&hbm, arena * waves, kWsArena))) return rc;
  uint8_t *ls = nullptr;
  if (ls_max && (rc = dmalloc((void **)&ls, (uint64_t)kLsBytes * waves, kWsLane))) return rc;
  if (cover && waves > max_waves) return set_error(MCE_EINTERNAL, "%u waves exceed the hub filter's %u", waves, max_waves);
  if (hneed[1] && (rc = dmalloc((void **)&overflow, sizeof(uint64_t) * hneed[1], kWsOverflow))) return rc;
  if (wave_stats) {
    if ((rc = dmalloc((void **)&wave_val, sizeof(unsigned long long) * waves, -1))) return rc;
    if ((rc = dmalloc((void **)&wave_cu, sizeof(uint32_t) * waves, -1))) return rc;
    if (stat == kStatBd && (rc = dmalloc((void **)&wave_bd, sizeof(unsigned long long) * 7 * waves, -1))) return rc;
  }

  pr.rp = g.rp;
  pr.ci = g.ci;
  pr.oc = g.oc;
  pr.split = g.split;
  pr.items = d_items;
  pr.n_items = n_items;
  pr.ticket = ticket;
  pr.t1 = std::min<uint64_t>(n_items, (uint64_t)waves * 8);
  pr.chunk = 8;
  pr.level = (uint32_t)cfg.level;
  pr.pool_bytes = (uint32_t)pool;
  pr.stack_lds = cfg.stack_lds_levels;
  pr.want_levels = cfg.stack_lds_levels ? cfg.stack_lds_levels : 24;
  pr.small_max = std::min<uint32_t>(cfg.small_max, kSmallMax);
  pr.small_pmax = kSmallMaxPWl;
  pr.ls_max = ls_max;
  pr.io_off = (uint32_t)(hist_bytes + kPoolHeader + pool);
  pr.ls_off = pr.io_off + kHandoverBytes * wpg;
  pr.ls = ls;
  pr.cover = cover;
  pr.watchdog_ticks = cfg.watchdog_us ? (uint64_t)cfg.watchdog_us * 100 : kWatchdogTicks;
  pr.hbm = hbm;
  pr.hbm_bytes = arena;
  pr.acc = acc;
  pr.hist = (unsigned long long *)d_hist;
  pr.hist_len = hist_len;
  pr.hist_lds = hist_lds;
  pr.sub_nodes = (unsigned long long *)d_sub_nodes;
  pr.sub_cliques = (unsigned long long *)d_sub_cliques;
  pr.overflow = overflow;
  pr.overflow_cap = hneed[1];
  pr.wave_val = wave_val;
  pr.wave_cu = wave_cu;
  pr.wave_bd = wave_bd;
  pr.wpg = wpg;
  const uint64_t n_tickets = n_items <= pr.t1 ? n_items : pr.t1 + (n_items - pr.t1 + pr.chunk - 1) / pr.chunk;
  // (a wave's claims run past the last ticket by at most one, from `waves` on)
  if (n_tickets + 2ull * waves >= 0xFFFFFF00ull) return set_error(MCE_ELIMIT, "too many work tickets");
  if (cfg.wl) {
    pr.slot_pmax = slot_pmax;
    pr.slot_wmax = slot_wmax;
    pr.slot_oP = kSlotHeader;
    pr.slot_oS = pr.slot_oP + 8 * (2 * pr.slot_wmax + 64);  // P, X, and the 64-word outside-X bitmap
    pr.slot_oA = pr.slot_oS + (uint32_t)align8(4ull * pr.slot_pmax);
    pr.slot_xcap = (uint32_t)slot_xcap;
    pr.slot_oXI = (uint32_t)slot_fixed;
    pr.slot_oXR = (uint32_t)(slot_fixed + align8(4ull * pr.slot_xcap));
    pr.slot_bytes = ((uint64_t)pr.slot_oXR + (cfg.ipx ? 8ull * pr.slot_xcap * pr.slot_wmax : 0) + 255) & ~255ull;
    pr.ring_cap = waves;
    pr.donate_min_p = std::max<uint32_t>(cfg.donate_min_p, 1);
    pr.donate_check = std::max<uint32_t>(cfg.donate_check_nodes, 1);
    pr.donate_age = (uint64_t)cfg.donate_age_us * 100;
    // looks at the idle queues at least 20 us apart, or the age if less
    pr.poll_ticks = cfg.donate_auto ? 2000 : std::min<uint64_t>(2000, pr.donate_age);
    if ((rc = dmalloc((void **)&pr.ctl, sizeof(unsigned long long) * kCtlWords, kWsCtl))) return rc;
    if ((rc = dmalloc((void **)&pr.seq, sizeof(unsigned long long) * kQueues * pr.ring_cap, kWsSeq))) return rc;
    if ((rc = dmalloc((void **)&pr.ring, pr.slot_bytes * pr.ring_cap, kWsRing))) return rc;
    if ((rc = dmalloc((void **)&pr.idle_ids, sizeof(uint32_t) * kQueues * pr.ring_cap, kWsIdle))) return rc;
    if ((rc = dmalloc((void **)&pr.mbox, sizeof(unsigned long long) * kMboxStride * pr.ring_cap, kWsMbox))) return rc;
    if (!cfg.capture) ring_init<<<64, 256, 0, s>>>(pr.seq, pr.ring_cap, pr.ctl, n_tickets, pr.mbox);
  }

  // pinned host words for the kernel's progress posts: the workspace's (kept
  // with the graph) or this call's own, freed on all paths
  struct Pinned {
    unsigned long long *h = nullptr;
    bool own = false;
    ~Pinned() {
      if (own && h) (void)hipHostFree(h);
    }
  } pin;
  volatile unsigned long long *posted = nullptr;
  if (cfg.progress_s && !sc) {
    if (ws && ws->pinned) {
      pin.h = ws->pinned;
    } else if (hipHostMalloc((void **)&pin.h, 2 * sizeof(unsigned long long), hipHostMallocMapped) == hipSuccess) {
      if (ws) ws->pinned = pin.h;
      else pin.own = true;
    } else {
      pin.h = nullptr;
    }
    void *dp = nullptr;
    if (pin.h && hipHostGetDevicePointer(&dp, pin.h, 0) == hipSuccess) {
      pin.h[0] = pin.h[1] = 0;
      posted = pin.h;
      pr.host_progress = (unsigned long long *)dp;
    }
  }
  // device-time events, except from a scratch region (event creation may
  // allocate): then host time around the synchronised launch
  struct Events {
    hipEvent_t a = nullptr, b = nullptr;
    ~Events() {
      if (a) (void)hipEventDestroy(a);
      if (b) (void)hipEventDestroy(b);
    }
  } ev;
  if (!sc) {
    MCE_HIP(hipEventCreate(&ev.a));
    MCE_HIP(hipEventCreate(&ev.b));
  }
  hipEvent_t e0 = ev.a, e1 = ev.b;
  const auto host_t0 = std::chrono::steady_clock::now();
  if (cfg.capture) {
    // one persistent launch captured into a graph: counters reset by a kernel
    // (no memset nodes), then the worker-list set-up and the enumeration
    // kernel. A graph handle keeps the instantiated graph and relaunches it
    // while every launch parameter (buffers, settings, work list) is the same.
    std::vector<uint8_t> key(sizeof(BkParams));
    memcpy(key.data(), &pr, sizeof(BkParams));  // pr is zero-initialised, padding included
    for (uint64_t v : {(uint64_t)groups, (uint64_t)wpg, (uint64_t)lds, (uint64_t)stat, (uint64_t)cfg.ipx,
                       (uint64_t)cfg.wl, (uint64_t)n_tickets})
      key.insert(key.end(), (const uint8_t *)&v, (const uint8_t *)&v + sizeof(v));
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    const bool reuse = ws && ws->exec && ws->key == key;
    if (reuse) {
      exec = ws->exec;
    } else {
      if (ws) ws->drop_graph();
      MCE_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
      reset_kernel<<<1, 64, 0, s>>>(acc, kAccN, ticket);
      if (cfg.wl) ring_init<<<64, 256, 0, s>>>(pr.seq, pr.ring_cap, pr.ctl, n_tickets, pr.mbox);
      rc = dispatch(cfg.ipx, cfg.wl, stat, false, nullptr, pr, groups, wpg, lds, s);
      const hipError_t ec = hipStreamEndCapture(s, &graph);
      if (rc) {
        if (graph) (void)hipGraphDestroy(graph);
        return rc;
      }
      MCE_HIP(ec);
      const hipError_t ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
      if (ei != hipSuccess) {
        (void)hipGraphDestroy(graph);
        return hip_fail(ei, "hipGraphInstantiate");
      }
      if (ws) {
        ws->graph = graph;
        ws->exec = exec;
        ws->key = std::move(key);
      }
    }
    MCE_HIP(hipEventRecord(e0, s));
    const hipError_t el = hipGraphLaunch(exec, s);
    const int rw = el == hipSuccess ? wait_launch(s, cfg.progress_s, posted, n_tickets, cfg.wl) : MCE_OK;
    if (!ws) {
      (void)hipGraphExecDestroy(exec);
      (void)hipGraphDestroy(graph);
    } else if (el != hipSuccess || rw) {
      ws->drop_graph();
    }
    MCE_HIP(el);
    if (rw) return rw;
  } else {
    if (e0) MCE_HIP(hipEventRecord(e0, s));
    if ((rc = dispatch(cfg.ipx, cfg.wl, stat, false, nullptr, pr, groups, wpg, lds, s))) return rc;
    if ((rc = wait_launch(s, cfg.progress_s, posted, n_tickets, cfg.wl))) return rc;
  }
  // items that did not fit: rerun them with arenas sized for the largest.
  // The deferred count is always read: an item deferred beyond what
  // need_kernel predicted would otherwise be lost without an error.
  if (e1) MCE_HIP(hipEventRecord(e1, s));
  unsigned long long h[kAccN];
  MCE_HIP(hipMemcpyAsync(h, acc, sizeof(h), hipMemcpyDeviceToHost, s));
  MCE_HIP(hipStreamSynchronize(s));
  const unsigned long long novf = h[kAccOverflow];
  if (novf > hneed[1])
    return set_error(MCE_EINTERNAL, "%llu items did not fit their arena, %llu predicted", novf, hneed[1]);
  if (novf) {
    const uint64_t big = (hneed[0] + 255) & ~255ull;
    // at most the first launch's workgroups: the lane solver's regions are
    // sized for its waves
    const uint32_t g2 = (uint32_t)std::max<uint64_t>(
        1, std::min<uint64_t>({(novf + wpg - 1) / wpg, (freeb / 2) / ((uint64_t)wpg * big), (uint64_t)groups}));
    uint8_t *hbm2 = nullptr;
    if ((rc = dmalloc((void **)&hbm2, big * g2 * wpg, -1))) return rc;
    std::vector<uint64_t> idx(novf);
    MCE_HIP(hipMemcpy(idx.data(), overflow, sizeof(uint64_t) * novf, hipMemcpyDeviceToHost));
    std::sort(idx.begin(), idx.end());
    const size_t isz = cfg.level == 1 ? sizeof(uint32_t) : sizeof(uint2);
    std::vector<uint8_t> hitems(isz * novf);
    for (uint64_t i = 0; i < novf; ++i)
      MCE_HIP(hipMemcpy(hitems.data() + i * isz, (const uint8_t *)d_items + idx[i] * isz, isz, hipMemcpyDeviceToHost));
    void *ditems2 = nullptr;
    if ((rc = dmalloc(&ditems2, isz * novf, -1))) return rc;
    MCE_HIP(hipMemcpy(ditems2, hitems.data(), isz * novf, hipMemcpyHostToDevice));
    BkParams p2 = pr;
    p2.items = ditems2;
    p2.n_items = novf;
    p2.t1 = novf;
    p2.hbm = hbm2;
    p2.hbm_bytes = big;
    p2.wave_val = nullptr;
    p2.wave_bd = nullptr;
    p2.overflow = nullptr;
    p2.overflow_cap = 0;
    MCE_HIP(hipMemsetAsync(ticket, 0, sizeof(uint32_t), s));
    if ((rc = dispatch(cfg.ipx, false, ls_max ? kStatLane : kStatNone, false, nullptr, p2, g2, wpg, lds, s)))
      return rc;
    if (e1) MCE_HIP(hipEventRecord(e1, s));
    MCE_HIP(hipMemcpyAsync(h, acc, sizeof(h), hipMemcpyDeviceToHost, s));
    MCE_HIP(hipStreamSynchronize(s));
    if (h[kAccOverflow] != novf) return set_error(MCE_EINTERNAL, "items did not fit the large arena");
  }
  float ms = 0;
  if (e0) {
    MCE_HIP(hipEventElapsedTime(&ms, e0, e1));
  } else {
    ms = std::chrono::duration<float, std::milli>(std::chrono::steady_clock::now() - host_t0).count();
  }
  if (h[kAccError] & 1ull) return set_error(MCE_EINTERNAL, "worker list watchdog expired (termination not reached)");
  if (h[kAccError] & 2ull) return set_error(MCE_EINTERNAL, "a donated subproblem did not fit its receiver");
  out->count = h[kAccCount];
  out->hash = h[kAccHash];
  out->nodes = h[kAccNodes];
  out->donations = h[kAccDonations];
  out->max_size = (uint32_t)h[kAccMaxSize];
  out->waves = waves;
  out->ms = ms;
  if (wave_stats && wave_stats_cap) {
    std::vector<unsigned long long> wv(waves), wb(stat == kStatBd ? 7ull * waves : 0);
    std::vector<uint32_t> wc(waves);
    MCE_HIP(hipMemcpy(wv.data(), wave_val, sizeof(unsigned long long) * waves, hipMemcpyDeviceToHost));
    MCE_HIP(hipMemcpy(wc.data(), wave_cu, sizeof(uint32_t) * waves, hipMemcpyDeviceToHost));
    if (stat == kStatBd)
      MCE_HIP(hipMemcpy(wb.data(), wave_bd, sizeof(unsigned long long) * 7 * waves, hipMemcpyDeviceToHost));
    const uint32_t k = std::min<uint32_t>(waves, wave_stats_cap);
    for (uint32_t i = 0; i < k; ++i) {
      wave_stats[i] = mce_wave_stat{};
      wave_stats[i].wave = i;
      wave_stats[i].cu = wc[i];
      wave_stats[i].value = wv[i];
      if (stat == kStatBd)
        for (int c = 0; c < 7; ++c) wave_stats[i].bd[c] = wb[(uint64_t)i * 7 + c];
    }
    if (wave_stats_len) *wave_stats_len = k;
  }
  return MCE_OK;
}

}  // namespace mce

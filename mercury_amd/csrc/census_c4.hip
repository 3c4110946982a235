// 4-cycles of the census graph (relabelled in DAG order: rank = id, rows
// sorted), each counted once at the pair {v, w} of opposite vertices that
// holds its highest vertex v: with n(v, w) the wedges v-u-w whose middle u
// lies below v, the pair lies on C(n, 2) cycles.
//
// The wedges of one owner are walked as ranges of sorted rows and counted
// per target in LDS.  Counters cover a window, the 65536 highest ids, so
// pairs are split by where their lower vertex w lies:
//   top   v and w in the window: owner v, target w; middles u below v, the
//         part of u's row in the window before v;
//   low   w below the window, v in it: owner w (its targets, the window's
//         vertices, fit the counters where v's would not); every neighbour
//         u of w, the part of u's row past u in the window;
//   rest  v and w below the window (small degrees): owner v, target w;
//         middles u below v, u's row before v.
// An increment returns the count before it, and those sum to C(n, 2), so
// no counter is read again for the count alone.  With the 5-vertex census a
// second walk over the same wedges takes each wedge's n - 1 cycles for the
// banner and house sums.  Range ends come from the DAG arc of the CSR entry
// (u's row position of v) and from one offset per vertex (first entry in
// the window): no searches.
//
// Owners with at most kLightWedges wedges take one wave and a hash table of
// 1024 slots; the others one workgroup and 32 to 128 KB of counters of 4, 8
// or 16 bits (32-bit counters over half the window in two rounds when the
// owner has 65536 or more middles, so a count could not overflow), or, for
// `rest`, a dense array in global memory.
//
// Measured on one MI355X, RMAT-20 (16 draws per vertex, 5.7e9 wedges): 8.3
// ms per count (top 4.8, low 3.3, rest 0.2); 24.5 ms (7.7, 16.5, 0.3) with
// 16-bit counters and one workgroup per CU for every heavy owner; 295 ms
// with one workgroup per highest vertex and global atomics on an array per
// workgroup (19e9 increments per second, each a cache miss).  The window
// covers 77% of the targets there, all of them up to 65536 vertices.  What
// bounds it: an LDS atomic per wedge, 64 wedges per 35 cycles and CU in the
// 16-bit class, behind loads that 16 waves cannot hide.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "census.hpp"
#include "choose.hpp"
#include "lanes.hpp"
#include "wave.hpp"

namespace mgpm {

namespace {

typedef unsigned long long u64;

constexpr int kDenseT = 1024;      // threads per heavy owner of `rest`
constexpr int kLanes = 16;         // lanes that walk one range
constexpr int kUnroll = 4;         // loads in flight per lane
constexpr int kWindow = kRowWindow;
constexpr int kLogSlots = 10;      // light owners' hash table
constexpr int kLightWedges = 512;
constexpr int kLightWaves = 4;
constexpr uint32_t kGrab = 4;         // most light owners per queue access

enum Kind : int { kTop = 0, kLow = 1, kRest = 2 };

// The wedges through one CSR entry of the owner: u's row from b to e.
struct Range {
  uint32_t b, e;
};

template <int KIND>
__device__ __forceinline__ Range range_of(const CensusArgs &c, uint32_t i) {
  const int32_t u = c.col[i];
  const uint32_t end = static_cast<uint32_t>(c.rowptr[u + 1]);
  const uint32_t dend = static_cast<uint32_t>(c.drp[u + 1]);
  Range r;
  if (KIND == kLow) {
    const uint32_t up = end - (dend - static_cast<uint32_t>(c.drp[u]));
    const uint32_t win = c.win[u];
    r.b = win > up ? win : up;
    r.e = end;
  } else {
    // The owner's position in u's row, from the arc u -> owner.
    r.b = KIND == kTop ? c.win[u] : static_cast<uint32_t>(c.rowptr[u]);
    r.e = end - (dend - c.arc[i]);
  }
  return r;
}

// The owner's CSR entries that are middles: below it, or all of them.
template <int KIND>
__device__ __forceinline__ void middles_of(const CensusArgs &c, int32_t o,
                                           uint32_t &i0, uint32_t &cnt) {
  const uint32_t b = static_cast<uint32_t>(c.rowptr[o]);
  const uint32_t e = static_cast<uint32_t>(c.rowptr[o + 1]);
  const uint32_t up = static_cast<uint32_t>(c.drp[o + 1] - c.drp[o]);
  i0 = b;
  cnt = KIND == kLow ? e - b : e - b - up;
}

// Walks the wedges of entries [i0, i0 + cnt) with `groups` groups of 16
// lanes (this one `grp`): the entries are dealt to the groups in turn (they
// are sorted by degree: neighbours in a hub's row have ranges alike), and
// each takes up to 16 of its entries at a time, one per lane for their
// ranges, then walks them one after the other.
// on_item(entry, j, w, ok) sees every item, idle lanes with ok = false.
template <int KIND, class F>
__device__ __forceinline__ void walk(const CensusArgs &c, uint32_t i0,
                                     uint32_t cnt, uint32_t grp,
                                     uint32_t groups, int gl,
                                     const F &on_item) {
  for (uint32_t k = grp; k < cnt; k += groups * kLanes) {
    const uint32_t mine = k + static_cast<uint32_t>(gl) * groups;
    Range r{0, 0};
    if (mine < cnt) r = range_of<KIND>(c, i0 + mine);
    for (uint32_t x = 0, i = k; x < kLanes && i < cnt; ++x, i += groups) {
      const uint32_t b = __shfl(r.b, static_cast<int>(x), kLanes);
      const uint32_t e = __shfl(r.e, static_cast<int>(x), kLanes);
      lane_walk<kLanes, kUnroll>(
          b, e, static_cast<uint32_t>(gl),
          [&](const uint32_t(&j)[kUnroll], const bool(&ok)[kUnroll]) {
            int32_t w[kUnroll];
#pragma unroll
            for (int q = 0; q < kUnroll; ++q) w[q] = c.col[j[q]];
#pragma unroll
            for (int q = 0; q < kUnroll; ++q) on_item(i0 + i, j[q], w[q], ok[q]);
          });
    }
  }
}

// The same wedges walked by a workgroup of W waves: 64 entries at a time,
// an entry per lane for its range; the ranges are cut in pieces of 64 items,
// and the waves of a team (all for at most 64 entries) take the pieces in
// turn, four at once, so that an owner with three middles keeps every wave
// busy.  Owners with hundreds of middles and more keep 64 groups busy by
// themselves and take walk, where an item costs less: RMAT-20's 16-bit owners
// 8.7 ms there and 12.7 in pieces (the two heaviest by one workgroup each;
// 4.0 ms since).
template <int KIND, int W, class F>
__device__ __forceinline__ void walk_pieces(const CensusArgs &c, uint32_t i0,
                                            uint32_t cnt, const F &on_item) {
  constexpr uint32_t kLogW = W == 16 ? 4 : 3;
  static_assert(W == 1 << kLogW, "8 or 16 waves");
  const int lane = lane64();
  const uint32_t wv = wave_first(threadIdx.x >> 6);
  const uint32_t batches = (cnt + 63) >> 6;
  const uint32_t lg =
      batches <= 1 ? 0u : min(kLogW, 32u - __builtin_clz(batches - 1));
  const uint32_t tw = W >> lg;  // waves of a team
  for (uint32_t bt = wv >> (kLogW - lg); bt < batches; bt += 1u << lg) {
    const uint32_t k = bt + batches * static_cast<uint32_t>(lane);
    Range r{0, 0};
    if (k < cnt) r = range_of<KIND>(c, i0 + k);
    const uint32_t len = r.e > r.b ? r.e - r.b : 0u;
    const uint32_t pieces = (len + 63) >> 6;
    uint32_t incl = pieces;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t x = __shfl_up(incl, o, 64);
      if (lane >= o) incl += x;
    }
    const uint32_t excl = incl - pieces;
    const uint32_t total = __builtin_amdgcn_readlane(incl, 63);
    for (uint32_t p = wv & (tw - 1u); p < total; p += tw * kUnroll) {
      uint32_t x[kUnroll], j[kUnroll];
      int32_t w[kUnroll];
      bool ok[kUnroll];
#pragma unroll
      for (int q = 0; q < kUnroll; ++q) {
        const uint32_t pq = min(p + tw * q, total - 1u);
        x[q] = static_cast<uint32_t>(__popcll(__ballot(incl <= pq)));
        const uint32_t lx = __builtin_amdgcn_readlane(len, x[q]);
        const uint32_t at =
            64u * (pq - __builtin_amdgcn_readlane(excl, x[q])) + lane;
        ok[q] = p + tw * q < total && at < lx;
        j[q] = __builtin_amdgcn_readlane(r.b, x[q]) + (at < lx ? at : lx - 1u);
        w[q] = c.col[j[q]];
      }
#pragma unroll
      for (int q = 0; q < kUnroll; ++q)
        on_item(i0 + bt + batches * x[q], j[q], w[q], ok[q]);
    }
  }
}

// Counters: add returns the count before it, get the final count.  The
// window's in LDS: B bits each, targets kWords apart share a word (adjacent
// ids, which one wave counts at once, lie in different banks).
template <int B>
struct Win {
  static constexpr int kWords = kWindow * B / 32;
  uint32_t *c;
  int32_t lo;
  __device__ __forceinline__ bool covers(int32_t) const { return true; }
  __device__ __forceinline__ uint32_t add(int32_t w) const {
    const uint32_t k = static_cast<uint32_t>(w - lo), s = k / kWords * B;
    return __builtin_amdgcn_ubfe(atomicAdd(&c[k % kWords], 1u << s), s, B);
  }
  __device__ __forceinline__ uint32_t get(int32_t w) const {
    const uint32_t k = static_cast<uint32_t>(w - lo);
    return __builtin_amdgcn_ubfe(c[k % kWords], k / kWords * B, B);
  }
};

struct Win32 {  // half the window from lo
  uint32_t *c;
  int32_t lo;
  __device__ __forceinline__ bool covers(int32_t w) const {
    return static_cast<uint32_t>(w - lo) < static_cast<uint32_t>(kWindow / 2);
  }
  __device__ __forceinline__ uint32_t add(int32_t w) const {
    return atomicAdd(&c[w - lo], 1u);
  }
  __device__ __forceinline__ uint32_t get(int32_t w) const {
    return c[w - lo];
  }
};

struct Dense {  // global: made by atomics in L2, read past the vector L1
  uint32_t *c;
  __device__ __forceinline__ bool covers(int32_t) const { return true; }
  __device__ __forceinline__ uint32_t add(int32_t w) const {
    return atomicAdd(&c[w], 1u);
  }
  __device__ __forceinline__ uint32_t get(int32_t w) const {
    return __hip_atomic_load(&c[w], __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
  }
  __device__ __forceinline__ void clear(int32_t w) const {
    __hip_atomic_store(&c[w], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
};

// Wave-private open addressing, 64-bit slots {id + 1, count}; at most
// kLightWedges of 1024 slots are taken.
struct Hash {
  u64 *s;
  __device__ __forceinline__ bool covers(int32_t) const { return true; }
  __device__ __forceinline__ uint32_t slot(int32_t w, bool insert,
                                           uint32_t *old) const {
    const u64 key = static_cast<u64>(static_cast<uint32_t>(w) + 1u) << 32;
    uint32_t h = slot_of(w, kLogSlots);
    for (;;) {
      u64 v = s[h];
      if (v == 0 && insert) {
        v = atomicCAS(&s[h], u64(0), key | 1u);
        if (v == 0) {
          *old = 0;
          return h;
        }
      }
      if ((v & ~u64(0xffffffffu)) == key) {
        *old = static_cast<uint32_t>(
            insert ? atomicAdd(&s[h], u64(1)) : v);
        return h;
      }
      h = (h + 1) & ((1u << kLogSlots) - 1u);
    }
  }
  __device__ __forceinline__ uint32_t add(int32_t w) const {
    uint32_t old;
    slot(w, true, &old);
    return old;
  }
  __device__ __forceinline__ uint32_t get(int32_t w) const {
    uint32_t n;
    slot(w, false, &n);
    return n;
  }
};

struct Sums {
  u64 acc = 0, ban = 0, tq = 0;
};

// First walk of one owner: counts, C(n, 2) as the sum of the counts before
// each increment, and with full5 the cycles' ends.
template <class W, class C>
__device__ __forceinline__ void count_walk(const CensusArgs &c, int32_t o,
                                           const W &walk, const C &ctr,
                                           Sums &s) {
  const int d4 = c.deg[o] - 4;
  walk([&](uint32_t, uint32_t, int32_t w, bool ok) {
    if (ok && ctr.covers(w)) {
      const u64 old = ctr.add(w);
      if (old) {
        s.acc += old;
        if (c.full5) s.ban += old * static_cast<u64>(d4 + c.deg[w]);
      }
    }
  });
}

// Second walk: the wedge o-u-w lies on n(o, w) - 1 cycles of its pair, and
// each puts its edges ou, uw and its middle u on them.
template <class W, class C>
__device__ __forceinline__ void cycle_walk(const CensusArgs &c, const W &walk,
                                           const C &ctr, Sums &s) {
  walk([&](uint32_t i, uint32_t j, int32_t w, bool ok) {
    if (ok && ctr.covers(w)) {
      const u64 x = ctr.get(w) - 1u;
      if (x) {
        s.ban += x * static_cast<u64>(c.deg[c.col[i]] - 2);
        s.tq += x * (static_cast<u64>(c.t_csr[i]) + c.t_csr[j]);
      }
    }
  });
}

__device__ __forceinline__ void flush(const CensusArgs &c, Sums &s) {
  s.acc = wave_sum_u64(s.acc);
  s.ban = wave_sum_u64(s.ban);
  s.tq = wave_sum_u64(s.tq);
  if (lane64() == 0) {
    if (s.acc) atomicAdd(&c.acc[kCensusC4], s.acc);
    if (s.ban) atomicAdd(&c.acc[kCensusBanner], s.ban);
    if (s.tq) atomicAdd(&c.acc[kCensusCycEdgeT], s.tq);
  }
}

// The next owners of a workgroup: its first by its number, then from the
// queue (an atomic on one address takes 11 ns, so several at a time where
// there are many).  Every thread calls it between barriers of its own.
__device__ __forceinline__ void next_owners(const C4List &l,
                                            unsigned *s_next) {
  if (threadIdx.x == 0)
    *s_next = (gridDim.x * l.grab < l.count ? atomicAdd(l.cursor, l.grab)
                                            : l.count) +
              gridDim.x * l.grab;
}

// Threads of a workgroup with B-bit counters.
constexpr int threads_of(int b) { return b == 4 ? 512 : 1024; }

// One workgroup per owner, with both ends' counters in LDS.  The counters
// are as narrow as the owner's middles allow (a count is at most their
// number): 4 bits for up to 15 of them, 8 for up to 255, 16 above, so four,
// two or one workgroups share a CU.  An owner's serial steps (its record,
// the ranges, the rows, the clearing) take microseconds whatever its size:
// with 16 bits for all, the 471000 heavy `low` owners of RMAT-20 (2800
// wedges on average) took 8.6 us each, 15.9 ms together (3.0 now).
template <int KIND, int B>
__global__ __launch_bounds__(threads_of(B)) void c4_heavy(CensusArgs c,
                                                          C4List l) {
  constexpr int T = threads_of(B);
  extern __shared__ uint4 s_dyn[];
  __shared__ unsigned s_next;
  uint32_t *ctr = reinterpret_cast<uint32_t *>(s_dyn);
  const int tid = threadIdx.x;
  // Words that hold a counter, in fours.
  const int used = (min(Win<B>::kWords, c.n - c.winlo) + 3) / 4;
  Sums s;
  auto clear = [&](int fours) {
    for (int i = tid; i < fours; i += T) s_dyn[i] = make_uint4(0, 0, 0, 0);
  };
  clear(used);
  for (uint32_t first = blockIdx.x * l.grab;; first = s_next) {
    __syncthreads();  // counters clear, s_next read
    if (first >= l.count) break;
    next_owners(l, &s_next);
    const uint32_t last = min(first + l.grab, l.count);
    for (uint32_t at = first; at < last; ++at) {
      const int32_t o = l.list[at];
      uint32_t i0, cnt;
      middles_of<KIND>(c, o, i0, cnt);
      auto each = [&](const auto &f) {
        if (B == 16)
          walk<KIND>(c, i0, cnt, tid / kLanes, T / kLanes, tid & (kLanes - 1),
                     f);
        else
          walk_pieces<KIND, T / 64>(c, i0, cnt, f);
      };
      auto run = [&](const auto &counters) {
        count_walk(c, o, each, counters, s);
        if (!c.full5) return;
        __syncthreads();
        cycle_walk(c, each, counters, s);
      };
      if (B == 16 && cnt >= 65536u) {
        for (int round = 0; round < 2; ++round) {
          run(Win32{ctr, c.winlo + round * (kWindow / 2)});
          __syncthreads();
          clear(kWindow / 8);
          if (round == 0) __syncthreads();  // clear for the second half
        }
      } else {
        run(Win<B>{ctr, c.winlo});
        __syncthreads();
        clear(used);
      }
      if (at + 1 < last) __syncthreads();  // clear for the next owner
    }
  }
  flush(c, s);
}

// One workgroup per owner, the heavy ones of `rest`, counters in global
// memory.
__global__ __launch_bounds__(kDenseT) void c4_dense(CensusArgs c, C4List l) {
  __shared__ unsigned s_next;
  const int tid = threadIdx.x;
  const int gl = tid & (kLanes - 1);
  const int grp = tid / kLanes;
  constexpr int groups = kDenseT / kLanes;
  const Dense ctr{c.wedges + size_t(blockIdx.x) * size_t(c.winlo)};
  Sums s;
  for (uint32_t at = blockIdx.x;; at = s_next) {
    __syncthreads();  // counters clear, s_next read
    if (at >= l.count) break;
    next_owners(l, &s_next);
    const int32_t o = l.list[at];
    uint32_t i0, cnt;
    middles_of<kRest>(c, o, i0, cnt);
    auto run = [&](const auto &f) {
      walk<kRest>(c, i0, cnt, grp, groups, gl, f);
    };
    count_walk(c, o, run, ctr, s);
    __syncthreads();
    if (c.full5) {
      cycle_walk(c, run, ctr, s);
      __syncthreads();
    }
    run([&](uint32_t, uint32_t, int32_t w, bool ok) {
      if (ok) ctr.clear(w);
    });
  }
  flush(c, s);
}

// One wave per owner, the light ones of a kind.
template <int KIND>
__global__ __launch_bounds__(kLightWaves * 64) void c4_light(CensusArgs c,
                                                             C4List l) {
  __shared__ u64 s_slots[kLightWaves][1 << kLogSlots];
  const int lane = lane64();
  u64 *slots = s_slots[threadIdx.x >> 6];
  const Hash ctr{slots};
  const int gl = lane & (kLanes - 1);
  const int grp = lane / kLanes;
  constexpr int groups = 64 / kLanes;
  Sums s;
  for (;;) {
    unsigned at = 0;
    if (lane == 0) at = atomicAdd(l.cursor, l.grab);
    at = wave_first(at);
    if (at >= l.count) break;
    const unsigned last = min(at + l.grab, l.count);
    for (; at < last; ++at) {
      const int32_t o = l.list[at];
      uint32_t i0, cnt;
      middles_of<KIND>(c, o, i0, cnt);
      for (int i = lane; i < (1 << kLogSlots); i += 64) slots[i] = 0;
      wave_sync();
      auto run = [&](const auto &f) {
        walk<KIND>(c, i0, cnt, grp, groups, gl, f);
      };
      count_walk(c, o, run, ctr, s);
      if (c.full5) {
        wave_sync();
        cycle_walk(c, run, ctr, s);
      }
      wave_sync();
    }
  }
  flush(c, s);
}

// First entry of every row in the window.
__global__ void c4_window(CensusArgs c, uint32_t *__restrict__ win) {
  for (int64_t v = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; v < c.n;
       v += int64_t(gridDim.x) * blockDim.x) {
    int64_t lo = c.rowptr[v], hi = c.rowptr[v + 1];
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (c.col[mid] < c.winlo) lo = mid + 1;
      else hi = mid;
    }
    win[v] = static_cast<uint32_t>(lo);
  }
}

// Class of every owner of a kind, one wave per owner, by its wedges and
// middles; -1 none (a pair of wedges has two middles).
template <int KIND>
__global__ void c4_classes(CensusArgs c, int32_t first, int32_t count,
                           int8_t *__restrict__ cls) {
  const int lane = lane64();
  const int64_t nw = (int64_t(gridDim.x) * blockDim.x) >> 6;
  for (int64_t k = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
       k < count; k += nw) {
    uint32_t i0, cnt;
    middles_of<KIND>(c, first + static_cast<int32_t>(k), i0, cnt);
    u64 w = 0;  // stops at the first 64 entries that make the owner heavy
    for (uint32_t b = 0; b < cnt && w <= kLightWedges; b += 64) {
      u64 mine = 0;
      if (b + lane < cnt) {
        const Range r = range_of<KIND>(c, i0 + b + lane);
        if (r.e > r.b) mine = r.e - r.b;
      }
      w += wave_sum_u64(mine);
    }
    if (lane == 0)
      cls[k] = static_cast<int8_t>(
          w < 2 || cnt < 2         ? -1
          : w <= kLightWedges      ? kC4Light
          : KIND == kRest          ? kC4Bits16
          : cnt <= 15              ? kC4Bits4
          : cnt <= 255             ? kC4Bits8
                                   : kC4Bits16);
  }
}

// The owners of each class from the top id down, 1024 at a time with one
// atomic per class for all (at list + start[class]), or (list null) only the
// class sizes, into fill (zeroed).
struct C4Starts {
  uint32_t at[kC4Classes];
};
constexpr int kClassT = 1024;
__global__ __launch_bounds__(kClassT) void c4_scatter(
    const int8_t *__restrict__ cls, int32_t first, int32_t count,
    unsigned *__restrict__ fill, int32_t *__restrict__ list, C4Starts start) {
  __shared__ unsigned s_wave[kClassT / 64];
  __shared__ unsigned s_base;
  const int64_t k =
      int64_t(count) - 1 - (int64_t(blockIdx.x) * kClassT + threadIdx.x);
  const int q = k >= 0 ? cls[k] : -1;
#pragma unroll
  for (int p = 0; p < kC4Classes; ++p) {
    const u64 m = __ballot(q == p);
    if (lane64() == 0) s_wave[threadIdx.x >> 6] = __popcll(m);
    __syncthreads();
    unsigned before = static_cast<unsigned>(bits_below(m)), total = 0;
    for (int w = 0; w < kClassT / 64; ++w) {
      if (w < static_cast<int>(threadIdx.x >> 6)) before += s_wave[w];
      total += s_wave[w];
    }
    if (threadIdx.x == 0) s_base = total ? atomicAdd(&fill[p], total) : 0u;
    __syncthreads();
    if (q == p && list)
      list[start.at[p] + s_base + before] = first + static_cast<int32_t>(k);
  }
}

void scatter(const int8_t *cls, int32_t first, int32_t count, unsigned *fill,
             int32_t *list, const uint32_t *sizes, hipStream_t s) {
  C4Starts start{};
  if (sizes)
    for (int q = 1; q < kC4Classes; ++q)
      start.at[q] = start.at[q - 1] + sizes[q - 1];
  hipLaunchKernelGGL(c4_scatter, dim3(count / kClassT + 1), dim3(kClassT), 0,
                     s, cls, first, count, fill, list, start);
}

template <int KIND>
void classes(const CensusArgs &c, int32_t first, int32_t count, int8_t *cls,
             hipStream_t s) {
  const int g = static_cast<int>(
      std::min<int64_t>(4096, (int64_t(count) + 3) / 4));
  hipLaunchKernelGGL((c4_classes<KIND>), dim3(g), dim3(256), 0, s, c, first,
                     count, cls);
}

template <int KIND, int B>
int launch_heavy(const CensusArgs &c, const int32_t *list, uint32_t count,
                 unsigned *cursor, int cus, hipStream_t s) {
  if (!count) return 0;
  const uint32_t most = static_cast<uint32_t>(cus) * (16 / B);
  // The heaviest owners one at a time: RMAT-20's first, 1.8e7 wedges, lasts
  // 4 ms, as long as the launch (8.7 ms when one workgroup took the first
  // two).
  const C4List l{list, count, cursor,
                 B == 16 ? 1 : std::max(1u, std::min(8u, count / (8 * most)))};
  const uint32_t g = std::min((count + l.grab - 1) / l.grab, most);
  hipLaunchKernelGGL((c4_heavy<KIND, B>), dim3(g), dim3(threads_of(B)),
                     Win<B>::kWords * sizeof(uint32_t), s, c, l);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// The classes of a kind, the heaviest first.
template <int KIND>
int launch_kind(const CensusArgs &c, const C4Plan &p, unsigned *cursor,
                int cus, int dense_groups, hipStream_t s) {
  const uint32_t *n = p.count[KIND];
  const int32_t *list[kC4Classes];
  for (int q = 0; q < kC4Classes; ++q)
    list[q] = q ? list[q - 1] + n[q - 1] : p.list[KIND];
  if constexpr (KIND == kRest) {
    if (const uint32_t k = n[kC4Bits16]) {
      const C4List l{list[kC4Bits16], k, cursor + kC4Bits16, 1};
      hipLaunchKernelGGL(c4_dense,
                         dim3(std::min<uint32_t>(k, dense_groups)),
                         dim3(kDenseT), 0, s, c, l);
    }
  } else {
    if (launch_heavy<KIND, 16>(c, list[kC4Bits16], n[kC4Bits16],
                               cursor + kC4Bits16, cus, s) ||
        launch_heavy<KIND, 8>(c, list[kC4Bits8], n[kC4Bits8],
                              cursor + kC4Bits8, cus, s) ||
        launch_heavy<KIND, 4>(c, list[kC4Bits4], n[kC4Bits4],
                              cursor + kC4Bits4, cus, s))
      return -1;
  }
  if (n[kC4Light]) {
    // One owner per access while waves are left idle.
    const uint32_t waves = static_cast<uint32_t>(cus) * 4 * kLightWaves;
    const C4List l{list[kC4Light], n[kC4Light], cursor + kC4Light,
                   std::max(1u, std::min(kGrab, n[kC4Light] / waves))};
    const uint32_t per = kLightWaves * l.grab;
    const int64_t blocks = (int64_t(l.count) + per - 1) / per;
    hipLaunchKernelGGL((c4_light<KIND>),
                       dim3(static_cast<unsigned>(
                           std::min<int64_t>(blocks, int64_t(cus) * 4))),
                       dim3(kLightWaves * 64), 0, s, c, l);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int B>
bool raise_lds() {
  const void *k[] = {reinterpret_cast<const void *>(&c4_heavy<kTop, B>),
                     reinterpret_cast<const void *>(&c4_heavy<kLow, B>)};
  for (const void *f : k)
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                            Win<B>::kWords *
                                static_cast<int>(sizeof(uint32_t))) !=
        hipSuccess)
      return false;
  return true;
}

}  // namespace

int census_c4_init() { return raise_lds<16>() && raise_lds<8>() ? 0 : -1; }

int census_c4_window(const CensusArgs &c, uint32_t *win, hipStream_t s) {
  const int g = std::max(1, std::min(4096, c.n / 256 + 1));
  hipLaunchKernelGGL(c4_window, dim3(g), dim3(256), 0, s, c, win);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int census_c4_classes(const CensusArgs &c, int8_t *cls, unsigned *fill,
                      hipStream_t s) {
  const int32_t low = c.winlo, top = c.n - c.winlo;
  if (top > 0) {
    classes<kTop>(c, low, top, cls, s);
    scatter(cls, low, top, fill, nullptr, nullptr, s);
  }
  if (low > 0) {
    classes<kLow>(c, 0, low, cls + top, s);
    scatter(cls + top, 0, low, fill + kC4Classes, nullptr, nullptr, s);
    classes<kRest>(c, 0, low, cls + top + low, s);
    scatter(cls + top + low, 0, low, fill + 2 * kC4Classes, nullptr, nullptr,
            s);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int census_c4_lists(const CensusArgs &c, const int8_t *cls, unsigned *fill,
                    const C4Plan &p, hipStream_t s) {
  const int32_t low = c.winlo, top = c.n - c.winlo;
  if (top > 0)
    scatter(cls, low, top, fill, p.list[kTop], p.count[kTop], s);
  if (low > 0) {
    scatter(cls + top, 0, low, fill + kC4Classes, p.list[kLow], p.count[kLow],
            s);
    scatter(cls + top + low, 0, low, fill + 2 * kC4Classes, p.list[kRest],
            p.count[kRest], s);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int census_c4_launch(const CensusArgs &c, const C4Plan &p, int dense_groups,
                     int cus, hipStream_t s) {
  if (launch_kind<kTop>(c, p, c.c4_cursor, cus, dense_groups, s) ||
      launch_kind<kLow>(c, p, c.c4_cursor + kC4Classes, cus, dense_groups,
                        s) ||
      launch_kind<kRest>(c, p, c.c4_cursor + 2 * kC4Classes, cus,
                         dense_groups, s))
    return -1;
  return 0;
}

}  // namespace mgpm

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
// 1024 slots; the others one workgroup of 1024 threads and 128 KB of 16-bit
// counters (32-bit counters over half the window in two rounds when the
// owner has 65536 or more middles, so a count could not overflow), or, for
// `rest`, a dense array in global memory.
//
// Measured on one MI355X, RMAT-20 (16 draws per vertex, 5.7e9 wedges):
// 24.5 ms per count (top 7.7, low 16.5, rest 0.3) against 295 ms with one
// workgroup per highest vertex and global atomics on an array per workgroup
// (19e9 increments per second, each a cache miss).  The window covers 77% of
// the targets there, all of them up to 65536 vertices.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "census.hpp"
#include "choose.hpp"
#include "wave.hpp"

namespace mgpm {

namespace {

typedef unsigned long long u64;

constexpr int kT = 1024;           // threads per heavy owner
constexpr int kLanes = 16;         // lanes that walk one range
constexpr int kUnroll = 4;         // loads in flight per lane
constexpr int kWindow = kRowWindow;
constexpr int kLogSlots = 10;      // light owners' hash table
constexpr int kLightWedges = 512;
constexpr int kLightWaves = 4;
constexpr int kGrab = 4;           // light owners per queue access

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
// lanes (this one `grp`): each group takes up to 16 entries at a time, one
// per lane for their ranges, then walks them one after the other.
// on_item(entry, j, ok) sees every item, idle lanes with ok = false.
template <int KIND, class F>
__device__ __forceinline__ void walk(const CensusArgs &c, uint32_t i0,
                                     uint32_t cnt, int grp, int groups,
                                     int gl, const F &on_item) {
  uint32_t per = (cnt + groups - 1) / groups;
  per = per > kLanes ? kLanes : (per < 1 ? 1 : per);
  for (uint32_t k = grp * per; k < cnt; k += groups * per) {
    const uint32_t take = min(per, cnt - k);
    Range mine{0, 0};
    if (static_cast<uint32_t>(gl) < take) mine = range_of<KIND>(c, i0 + k + gl);
    for (uint32_t x = 0; x < take; ++x) {
      const uint32_t b = __shfl(mine.b, static_cast<int>(x), kLanes);
      const uint32_t e = __shfl(mine.e, static_cast<int>(x), kLanes);
      for (uint32_t j = b + gl; j < e; j += kLanes * kUnroll) {
        int32_t w[kUnroll];
#pragma unroll
        for (int q = 0; q < kUnroll; ++q) {
          const uint32_t jj = j + kLanes * q;
          w[q] = c.col[jj < e ? jj : j];
        }
#pragma unroll
        for (int q = 0; q < kUnroll; ++q) {
          const uint32_t jj = j + kLanes * q;
          on_item(i0 + k + x, jj, w[q], jj < e);
        }
      }
    }
  }
}

// Counters: add returns the count before it, get the final count.
struct Win16 {
  uint32_t *c;
  int32_t lo;
  __device__ __forceinline__ bool covers(int32_t) const { return true; }
  __device__ __forceinline__ uint32_t add(int32_t w) const {
    const uint32_t k = static_cast<uint32_t>(w - lo);
    const uint32_t s = (k & 1u) * 16u;
    return (atomicAdd(&c[k >> 1], 1u << s) >> s) & 0xffffu;
  }
  __device__ __forceinline__ uint32_t get(int32_t w) const {
    const uint32_t k = static_cast<uint32_t>(w - lo);
    return (c[k >> 1] >> ((k & 1u) * 16u)) & 0xffffu;
  }
  __device__ __forceinline__ void clear(int32_t w) const {
    c[static_cast<uint32_t>(w - lo) >> 1] = 0;
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
  __device__ __forceinline__ void clear(int32_t w) const { c[w - lo] = 0; }
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
  __device__ __forceinline__ void clear(int32_t) const {}
};

struct Sums {
  u64 acc = 0, ban = 0, tq = 0;
};

// First walk of one owner: counts, C(n, 2) as the sum of the counts before
// each increment, and with full5 the cycles' ends.
template <int KIND, class C>
__device__ __forceinline__ uint32_t count_walk(const CensusArgs &c, int32_t o,
                                               uint32_t i0, uint32_t cnt,
                                               int grp, int groups, int gl,
                                               const C &ctr, Sums &s) {
  const int d4 = c.deg[o] - 4;
  uint32_t items = 0;
  walk<KIND>(c, i0, cnt, grp, groups, gl,
             [&](uint32_t, uint32_t, int32_t w, bool ok) {
               if (ok && ctr.covers(w)) {
                 ++items;
                 const u64 old = ctr.add(w);
                 if (old) {
                   s.acc += old;
                   if (c.full5) s.ban += old * static_cast<u64>(d4 + c.deg[w]);
                 }
               }
             });
  return items;
}

// Second walk: the wedge o-u-w lies on n(o, w) - 1 cycles of its pair, and
// each puts its edges ou, uw and its middle u on them.
template <int KIND, class C>
__device__ __forceinline__ void cycle_walk(const CensusArgs &c, uint32_t i0,
                                           uint32_t cnt, int grp, int groups,
                                           int gl, const C &ctr, Sums &s) {
  walk<KIND>(c, i0, cnt, grp, groups, gl,
             [&](uint32_t i, uint32_t j, int32_t w, bool ok) {
               if (ok && ctr.covers(w)) {
                 const u64 x = ctr.get(w) - 1u;
                 if (x) {
                   s.ban += x * static_cast<u64>(c.deg[c.col[i]] - 2);
                   s.tq += x * (static_cast<u64>(c.t_csr[i]) + c.t_csr[j]);
                 }
               }
             });
}

template <int KIND, class C>
__device__ __forceinline__ void clear_walk(const CensusArgs &c, uint32_t i0,
                                           uint32_t cnt, int grp, int groups,
                                           int gl, const C &ctr) {
  walk<KIND>(c, i0, cnt, grp, groups, gl,
             [&](uint32_t, uint32_t, int32_t w, bool ok) {
               if (ok && ctr.covers(w)) ctr.clear(w);
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

constexpr int kCtrWords = kWindow / 2;       // LDS counters of heavy owners
constexpr unsigned kLinearClear = kWindow / 4;  // wedges from which clearing
                                                // every counter is cheaper

// One workgroup per owner, the heavy ones of a kind.
template <int KIND>
__global__ __launch_bounds__(kT) void c4_heavy(CensusArgs c, C4List l) {
  extern __shared__ uint32_t s_ctr[];  // kCtrWords (top, low)
  __shared__ unsigned s_next, s_items;
  const int tid = threadIdx.x;
  const int gl = tid & (kLanes - 1);
  const int grp = tid / kLanes;
  constexpr int groups = kT / kLanes;
  Sums s;
  if (KIND != kRest)
    for (int i = tid; i < kCtrWords; i += kT) s_ctr[i] = 0;
  for (;;) {
    __syncthreads();  // counters clear, s_next and s_items read
    if (tid == 0) {
      s_next = atomicAdd(l.cursor, 1u);
      s_items = 0;
    }
    __syncthreads();
    const unsigned at = s_next;
    if (at >= l.count) break;
    const int32_t o = l.list[at];
    uint32_t i0, cnt;
    middles_of<KIND>(c, o, i0, cnt);
    const bool wide = KIND != kRest && cnt >= 65536u;
    for (int round = 0; round < (wide ? 2 : 1); ++round) {
      uint32_t items = 0;
      auto run = [&](const auto &ctr) {
        items = count_walk<KIND>(c, o, i0, cnt, grp, groups, gl, ctr, s);
        if (KIND == kRest || c.full5) __syncthreads();
        if (c.full5) cycle_walk<KIND>(c, i0, cnt, grp, groups, gl, ctr, s);
      };
      if constexpr (KIND == kRest) {
        const Dense ctr{c.wedges + size_t(blockIdx.x) * size_t(c.winlo)};
        run(ctr);
        __syncthreads();
        clear_walk<KIND>(c, i0, cnt, grp, groups, gl, ctr);
      } else {
        const Win16 n16{s_ctr, c.winlo};
        const Win32 n32{s_ctr, c.winlo + round * (kWindow / 2)};
        if (wide) run(n32);
        else run(n16);
        atomicAdd(&s_items, items);
        __syncthreads();
        if (wide || s_items >= kLinearClear)
          for (int i = tid; i < kCtrWords; i += kT) s_ctr[i] = 0;
        else
          clear_walk<KIND>(c, i0, cnt, grp, groups, gl, n16);
        if (wide) __syncthreads();  // counters clear for the next round
      }
    }
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
    if (lane == 0) at = atomicAdd(l.cursor, static_cast<unsigned>(kGrab));
    at = wave_first(at);
    if (at >= l.count) break;
    const unsigned last = min(at + kGrab, l.count);
    for (; at < last; ++at) {
      const int32_t o = l.list[at];
      uint32_t i0, cnt;
      middles_of<KIND>(c, o, i0, cnt);
      for (int i = lane; i < (1 << kLogSlots); i += 64) slots[i] = 0;
      wave_sync();
      count_walk<KIND>(c, o, i0, cnt, grp, groups, gl, ctr, s);
      if (c.full5) {
        wave_sync();
        cycle_walk<KIND>(c, i0, cnt, grp, groups, gl, ctr, s);
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

// Wedges of every owner of a kind, one wave per owner; -> its class: 0
// light, 1 heavy, -1 none (fewer than two wedges make no pair).
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
      cls[k] = w < 2 ? int8_t(-1) : (w <= kLightWedges ? int8_t(0) : int8_t(1));
  }
}

// The owners of each class from the top id down, or (lists null) only the
// class sizes, into fill[0..1] (zeroed).
__global__ void c4_scatter(const int8_t *__restrict__ cls, int32_t first,
                           int32_t count, unsigned *__restrict__ fill,
                           int32_t *__restrict__ light,
                           int32_t *__restrict__ heavy) {
  const int64_t stride = int64_t(gridDim.x) * blockDim.x;
  for (int64_t k0 = int64_t(blockIdx.x) * blockDim.x; k0 < count;
       k0 += stride) {
    const int64_t k = int64_t(count) - 1 - (k0 + threadIdx.x);
    const int q = k >= 0 ? cls[k] : -1;
    for (int p = 0; p < 2; ++p) {
      const u64 m = __ballot(q == p);
      if (!m) continue;
      unsigned base = 0;
      if (lane64() == 0)
        base = atomicAdd(&fill[p], static_cast<unsigned>(__popcll(m)));
      base = __shfl(base, 0, 64);
      if (q == p && light)
        (p ? heavy : light)[base + bits_below(m)] =
            first + static_cast<int32_t>(k);
    }
  }
}

void scatter(const int8_t *cls, int32_t first, int32_t count, unsigned *fill,
             int32_t *light, int32_t *heavy, hipStream_t s) {
  const int g = std::min(1024, count / 256 + 1);
  hipLaunchKernelGGL(c4_scatter, dim3(g), dim3(256), 0, s, cls, first, count,
                     fill, light, heavy);
}

template <int KIND>
void classes(const CensusArgs &c, int32_t first, int32_t count, int8_t *cls,
             hipStream_t s) {
  const int g = static_cast<int>(
      std::min<int64_t>(4096, (int64_t(count) + 3) / 4));
  hipLaunchKernelGGL((c4_classes<KIND>), dim3(g), dim3(256), 0, s, c, first,
                     count, cls);
}

template <int KIND>
int launch_kind(const CensusArgs &c, const C4Plan &p, unsigned *cursor,
                int cus, int dense_groups, hipStream_t s) {
  if (p.heavy[KIND]) {
    C4List l{p.heavy_list[KIND], p.heavy[KIND], cursor};
    const size_t lds = KIND == kRest ? 0 : kCtrWords * sizeof(uint32_t);
    const int64_t most = KIND == kRest ? dense_groups : cus;
    hipLaunchKernelGGL((c4_heavy<KIND>),
                       dim3(static_cast<unsigned>(
                           std::min<int64_t>(p.heavy[KIND], most))),
                       dim3(kT), lds, s, c, l);
  }
  if (p.light[KIND]) {
    C4List l{p.light_list[KIND], p.light[KIND], cursor + 1};
    const int64_t blocks =
        (int64_t(p.light[KIND]) + kLightWaves * kGrab - 1) /
        (kLightWaves * kGrab);
    hipLaunchKernelGGL((c4_light<KIND>),
                       dim3(static_cast<unsigned>(
                           std::min<int64_t>(blocks, int64_t(cus) * 4))),
                       dim3(kLightWaves * 64), 0, s, c, l);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace

int census_c4_init() {
  const void *big[] = {reinterpret_cast<const void *>(&c4_heavy<kTop>),
                       reinterpret_cast<const void *>(&c4_heavy<kLow>)};
  for (const void *k : big)
    if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize,
                            kCtrWords * static_cast<int>(sizeof(uint32_t))) !=
        hipSuccess)
      return -1;
  return 0;
}

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
    scatter(cls + top, 0, low, fill + 2, nullptr, nullptr, s);
    classes<kRest>(c, 0, low, cls + top + low, s);
    scatter(cls + top + low, 0, low, fill + 4, nullptr, nullptr, s);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int census_c4_lists(const CensusArgs &c, const int8_t *cls, unsigned *fill,
                    const C4Plan &p, hipStream_t s) {
  const int32_t low = c.winlo, top = c.n - c.winlo;
  if (top > 0)
    scatter(cls, low, top, fill, p.light_list[kTop], p.heavy_list[kTop], s);
  if (low > 0) {
    scatter(cls + top, 0, low, fill + 2, p.light_list[kLow],
            p.heavy_list[kLow], s);
    scatter(cls + top + low, 0, low, fill + 4, p.light_list[kRest],
            p.heavy_list[kRest], s);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int census_c4_launch(const CensusArgs &c, const C4Plan &p, int dense_groups,
                     int cus, hipStream_t s) {
  if (launch_kind<kTop>(c, p, c.c4_cursor, cus, dense_groups, s) ||
      launch_kind<kLow>(c, p, c.c4_cursor + 2, cus, dense_groups, s) ||
      launch_kind<kRest>(c, p, c.c4_cursor + 4, cus, dense_groups, s))
    return -1;
  return 0;
}

}  // namespace mgpm

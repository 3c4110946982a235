// Pair passes of the 5-vertex census: the subgraph counts behind P2, P3,
// P5 and P6 that no per-edge or per-triangle sum gives -- wheels W4 (a hub
// and a 4-cycle in its neighbourhood), K2,3 and K2,3 plus an edge between
// two of its three middle vertices.  All three are sums over vertex pairs
// {a, c} of functions of the common neighbourhood S = N(a) ∩ N(c):
//   K2,3 = sum C(|S|, 3),  K2,3+e = sum E(S) (|S| - 2),
//   W4 = 1/2 sum wedges(S) (each wheel has two rim diagonals).
// Every occurrence is charged to its lowest-ranked vertex in the DAG order
// (degree, then id; graph.cc:205-235), whose pattern neighbours all lie in
// its DAG out-neighbourhood N+ (at most ~sqrt(2m) vertices):
//   * anchor pass, per anchor a and every c above a: the mask
//     M = N+(a) ∩ N(c) over N+(a) and lo = |{z below a: z->a, z->c}|, so
//     codeg(a, c) = lo + |M| (common neighbours above a lie in N+(a));
//     K2,3 += C(codeg, 3); wheels whose lowest vertex is the rim vertex a
//     (opposite rim vertex c) += wedges of G[M]; diamonds whose lowest
//     vertex is the tip a (other tip c, hinge inside M) give
//     E(G[M]) (codeg - 2) of K2,3+e; and codeg of every pair with lo >= 1
//     goes into a table hashed per a;
//   * out-neighbourhood pass, per anchor x: wheels whose lowest vertex is
//     the hub x are 4-cycles inside G[N+(x)]; diamonds whose lowest vertex
//     is the hinge end x (tips p, q and hinge end y in N+(x)) give
//     |N+(x) ∩ N(p) ∩ N(q)| (codeg(p, q) - 2) of K2,3+e, codeg from the
//     table (x lies below p and q, so the pair is there).
// G[N+(a)] is held as adjacency bit rows, in LDS for d+ up to 512.  The
// passes run on the census graph, relabelled in DAG order (census_build):
// ids compare as ranks, and each sorted row lists the vertices below its
// own first, then N+.
#include <hip/hip_runtime.h>

#include <hipcub/device/device_scan.hpp>

#include <algorithm>
#include <type_traits>

#include "census.hpp"
#include "choose.hpp"
#include "wave.hpp"

namespace mgpm {

namespace {

constexpr int kT = 256;  // threads per workgroup
constexpr int kTW = kT / 64;

__device__ __forceinline__ uint64_t tab_slot(int32_t key, int logc) {
  return logc == 0 ? 0
                   : (static_cast<uint64_t>(static_cast<uint32_t>(key)) *
                      0x9E3779B97F4A7C15ull) >> (64 - logc);
}

__device__ __forceinline__ int log2_pow2(uint64_t cap) {
  return 63 - __clzll(static_cast<long long>(cap));
}

// Entries: (key + 1) << 32 | value; 0 = empty.  Load factor <= 1/2 when
// the count pass and the anchor pass agree; false if no slot was free.
__device__ bool tab_insert(unsigned long long *tab, uint64_t cap, int32_t key,
                           uint32_t val) {
  if (cap == 0) return false;
  const unsigned long long e =
      (static_cast<unsigned long long>(static_cast<uint32_t>(key) + 1u) << 32) |
      val;
  const int lc = log2_pow2(cap);
  uint64_t s = tab_slot(key, lc);
  for (uint64_t probes = 0; probes < cap; ++probes) {
    if (atomicCAS(&tab[s], 0ull, e) == 0ull) return true;
    s = (s + 1) & (cap - 1);
  }
  return false;
}

__device__ bool tab_find(const unsigned long long *tab, uint64_t cap,
                         int32_t key, uint32_t *val) {
  if (cap == 0) return false;
  const unsigned long long k1 = static_cast<uint32_t>(key) + 1u;
  const int lc = log2_pow2(cap);
  uint64_t s = tab_slot(key, lc);
  for (uint64_t probes = 0; probes < cap; ++probes) {
    const unsigned long long e = tab[s];
    if (e == 0) return false;
    if ((e >> 32) == k1) {
      *val = static_cast<uint32_t>(e);
      return true;
    }
    s = (s + 1) & (cap - 1);
  }
  return false;
}

__device__ __forceinline__ unsigned long long wg_sum(unsigned long long x,
                                                     unsigned long long *red) {
  x = wave_sum_u64(x);
  __syncthreads();
  if (lane64() == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  unsigned long long t = 0;
  for (int k = 0; k < kTW; ++k) t += red[k];
  return t;
}

// Sums over vertices of C(t_v, 2) and t_v C(d_v - 2, 2), and of t_v s_v as
// a sum over CSR arcs (v, x) of t_v (d_x - 1).
constexpr int kFlatT = 1024;
__global__ __launch_bounds__(kFlatT) void c5_flat(Census5Args c) {
  __shared__ unsigned long long s_sum[3];
  if (threadIdx.x < 3) s_sum[threadIdx.x] = 0;
  __syncthreads();
  unsigned long long ts = 0, t2 = 0, crk = 0;
  const int64_t stride = int64_t(gridDim.x) * blockDim.x;
  const int64_t i0 = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  for (int64_t j = i0; j < c.nnz; j += stride) {
    const unsigned long long tv = c.tv[c.src[j]] >> 1;
    ts += tv * static_cast<unsigned long long>(c.deg[c.col[j]] - 1);
  }
  for (int64_t v = i0; v < c.n; v += stride) {
    const unsigned long long tv = c.tv[v] >> 1;  // > 0: degree >= 2
    t2 += choose2(tv);
    if (tv) crk += tv * choose2(static_cast<unsigned long long>(c.deg[v]) - 2);
  }
  ts = wave_sum_u64(ts);
  t2 = wave_sum_u64(t2);
  crk = wave_sum_u64(crk);
  if (lane64() == 0) {
    atomicAdd(&s_sum[0], ts);
    atomicAdd(&s_sum[1], t2);
    atomicAdd(&s_sum[2], crk);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (s_sum[0]) atomicAdd(&c.acc[kCensusTriS], s_sum[0]);
    if (s_sum[1]) atomicAdd(&c.acc[kCensusTv2], s_sum[1]);
    if (s_sum[2]) atomicAdd(&c.acc[kCensusCricket], s_sum[2]);
  }
}

// Class of an anchor by its out-degree and the items it streams at most.
__device__ __forceinline__ int class_of(int dp, unsigned long long items) {
  if (items == 0) return -1;  // no pair with a common neighbour
  if (items <= kLightItems && dp <= 64) return kC5Light;
  int k = 0;
  while (k < kC5Windowed && dp > 64 * kC5Words[k]) ++k;
  return 1 + k;
}

// One wave per anchor: the items are the rows of its upper neighbours and
// the tails of its lower ones past it (counted to the first 64 entries that
// make it heavy).
__global__ void c5_classes(Census5Args c, int8_t *__restrict__ cls) {
  const int lane = lane64();
  const int64_t nw = (int64_t(gridDim.x) * blockDim.x) >> 6;
  for (int64_t a = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
       a < c.n; a += nw) {
    const int64_t rb = c.rowptr[a], re = c.rowptr[a + 1];
    unsigned long long items = 0;
    for (int64_t k = rb; k < re && items <= kLightItems; k += 64) {
      unsigned long long mine = 0;
      if (k + lane < re) {
        const int32_t v = c.col[k + lane];
        mine = v > a ? c.rowptr[v + 1] - c.rowptr[v] - 1
                     : c.drp[v + 1] - 1 - int64_t(c.arc[k + lane]);
      }
      items += wave_sum_u64(mine);
    }
    if (lane == 0)
      cls[a] = static_cast<int8_t>(
          class_of(static_cast<int>(c.drp[a + 1] - c.drp[a]), items));
  }
}

// The anchors class by class from the top id down (list null: only the class
// sizes, into fill), 1024 at a time with one atomic per class for all.
constexpr int kClassT = 1024;
__global__ __launch_bounds__(kClassT) void c5_scatter(
    const int8_t *__restrict__ cls, int32_t n,
    const unsigned *__restrict__ start, unsigned *__restrict__ fill,
    int32_t *__restrict__ list) {
  __shared__ unsigned s_wave[kClassT / 64];
  __shared__ unsigned s_base;
  const int64_t v =
      int64_t(n) - 1 - (int64_t(blockIdx.x) * kClassT + threadIdx.x);
  const int k = v >= 0 ? cls[v] : -1;
  for (int q = 0; q < kC5Lists; ++q) {
    const unsigned long long m = __ballot(k == q);
    if (lane64() == 0) s_wave[threadIdx.x >> 6] = __popcll(m);
    __syncthreads();
    unsigned before = static_cast<unsigned>(bits_below(m)), total = 0;
    for (int w = 0; w < kClassT / 64; ++w) {
      if (w < static_cast<int>(threadIdx.x >> 6)) before += s_wave[w];
      total += s_wave[w];
    }
    if (threadIdx.x == 0) s_base = total ? atomicAdd(&fill[q], total) : 0u;
    __syncthreads();
    if (list && k == q)
      list[start[q] + s_base + before] = static_cast<int32_t>(v);
  }
}

// The first vertex of at least two neighbours (ids are ranks by degree).
__global__ void c5_first(Census5Args c, unsigned *__restrict__ first) {
  int32_t lo = 0, hi = c.n;
  while (lo < hi) {
    const int32_t mid = lo + (hi - lo) / 2;
    if (c.deg[mid] < 2) lo = mid + 1;
    else hi = mid;
  }
  *first = static_cast<unsigned>(lo);
}

// The row of vertex v in the fine windows' offsets.
__device__ __forceinline__ int64_t woff_row(const Census5Args &c, int32_t v) {
  return max(v - c.first, -1) + 1;
}

// First entry of every row in each of the nf fine windows (kFine ids each
// from winlo), relative to the row's first entry in the window; entry nf:
// the row's entries in the window.  One thread per entry fills the windows
// that begin at it, one per row those past its last entry.
__global__ void c5_window_offsets(Census5Args c, uint16_t *__restrict__ woff) {
  const int stride = c.nf + 1;
  const int64_t step = int64_t(gridDim.x) * blockDim.x;
  const int64_t i0 = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  for (int64_t j = i0; j < c.nnz; j += step) {
    const int32_t u = c.col[j];
    if (u < c.winlo) continue;
    const int32_t v = c.src[j];
    if (v < c.first) continue;
    const int64_t w = c.win[v];
    const int f = (u - c.winlo) / kFine;
    const int from = j == w ? 0 : (c.col[j - 1] - c.winlo) / kFine + 1;
    for (int g = from; g <= f; ++g)
      woff[woff_row(c, v) * stride + g] = static_cast<uint16_t>(j - w);
  }
  for (int64_t v = c.first + i0; v < c.n; v += step) {
    const int64_t w = c.win[v], e = c.rowptr[v + 1];
    const int from = e > w ? (c.col[e - 1] - c.winlo) / kFine + 1 : 0;
    for (int g = from; g <= c.nf; ++g)
      woff[woff_row(c, static_cast<int32_t>(v)) * stride + g] =
          static_cast<uint16_t>(e - w);
  }
  if (i0 <= c.nf) woff[i0] = 0;
}

// Adjacency bit rows of G[N+(a)]: bit j of row i iff nb[j] ~ nb[i].
// `rows` (stride rs words) must be zero; built with atomics by T threads.
// Groups of 16 lanes take the neighbours in turn, each up to 16 at a time
// whose ranges are loaded one per lane, and search four items per lane in
// lockstep: with a wave per neighbour and one search at a time the chain of
// loads and searches was longer (RMAT-18's c5_outnb, all classes: 6.2 ms,
// now 5.4; c5_anchor 1.2 ms less).
constexpr int kRowLanes = 16, kRowUnroll = 4;
template <int T, class NB, class ROWS>
__device__ __forceinline__ void build_rows(const Census5Args &c, NB nb, int dp,
                                           ROWS rows, int rs) {
  constexpr int kGroups = T / kRowLanes;
  const int gl = threadIdx.x & (kRowLanes - 1);
  const int grp = static_cast<int>(threadIdx.x % T) / kRowLanes;
  for (int k = grp; k < dp; k += kGroups * kRowLanes) {
    const int mine = k + gl * kGroups;
    uint32_t mb = 0, me = 0;
    if (mine < dp) {
      const int32_t u = nb[mine];
      mb = static_cast<uint32_t>(c.drp[u]);
      me = static_cast<uint32_t>(c.drp[u + 1]);
    }
    for (int x = 0, i = k; x < kRowLanes && i < dp; ++x, i += kGroups) {
      const uint32_t b = __shfl(mb, x, kRowLanes);
      const uint32_t e = __shfl(me, x, kRowLanes);
      for (uint32_t q = b + gl; q < e; q += kRowLanes * kRowUnroll) {
        int32_t z[kRowUnroll];
        int lo[kRowUnroll];
#pragma unroll
        for (int r = 0; r < kRowUnroll; ++r) {
          const uint32_t qq = q + kRowLanes * r;
          z[r] = c.dcol[qq < e ? qq : q];
          lo[r] = 0;
        }
        // The last neighbour <= z (z lies above nb[i]).
        for (int len = dp; len > 1; len -= len >> 1) {
#pragma unroll
          for (int r = 0; r < kRowUnroll; ++r)
            if (nb[lo[r] + (len >> 1)] <= z[r]) lo[r] += len >> 1;
        }
#pragma unroll
        for (int r = 0; r < kRowUnroll; ++r) {
          const int j = lo[r];
          if (q + kRowLanes * r < e && nb[j] == z[r]) {
            atomicOr(&rows[int64_t(i) * rs + (j >> 6)], 1ull << (j & 63));
            atomicOr(&rows[int64_t(j) * rs + (i >> 6)], 1ull << (i & 63));
          }
        }
      }
    }
  }
}

// Reads a row word built by atomics: LDS words directly, global words past
// the vector L1 (the atomics ran in L2).
__device__ __forceinline__ unsigned long long row_word(
    const unsigned long long *r, bool global) {
  return global ? __hip_atomic_load(r, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT)
                : *r;
}

struct AnchorSums {
  unsigned long long k23 = 0, w4 = 0, a16 = 0, miss = 0;
};

// C(x, 3), in 32 bits where x (x - 1) (x - 2) fits (64-bit remainders and
// products cost ten times as much).
__device__ __forceinline__ unsigned long long choose3_of(unsigned x) {
  if (x < 1600) return x < 3 ? 0u : x * (x - 1) * (x - 2) / 6;
  return choose3(x);
}

// One pair (a, cc): l common neighbours below a, the mask m over N+(a), of
// which 32 H bits can be set.  The mask's bits are a loop of about 14
// instructions each in 32 bits; this half of the anchor pass took as long as
// the windows (RMAT-18, d+ <= 64: 9 of 19.8 ms, 16.4 now) with 64-bit masks
// and sums.
template <int W, int H = 2 * W>
__device__ __forceinline__ void pair_terms(
    const Census5Args &c, const unsigned long long (&m)[W],
    const unsigned long long *rows, unsigned l, int32_t cc, uint64_t toff,
    uint64_t tcap, AnchorSums &s) {
  unsigned pc = 0;
#pragma unroll
  for (int w = 0; w < W; ++w) pc += __popcll(m[w]);
  const unsigned cd = l + pc;
  s.k23 += choose3_of(cd);
  if (pc >= 2) {
    unsigned e2 = 0, sq = 0;  // sums of dm and dm^2 (at most 512 of 512)
#pragma unroll
    for (int h = 0; h < H; ++h) {
      for (unsigned b = static_cast<unsigned>(m[h >> 1] >> (32 * (h & 1))); b;
           b &= b - 1) {
        const int p = h * 32 + __builtin_ctz(b);
        unsigned dm = 0;
        if constexpr (H == 1) {
          dm = __popc(static_cast<unsigned>(rows[p]) &
                      static_cast<unsigned>(m[0]));
        } else {
#pragma unroll
          for (int w2 = 0; w2 < W; ++w2)
            dm += __popcll(rows[p * W + w2] & m[w2]);
        }
        e2 += dm;
        sq += dm * dm;
      }
    }
    s.w4 += (sq - e2) >> 1;
    s.a16 += static_cast<unsigned long long>(e2 >> 1) * (cd - 2);
  }
  if (l && !tab_insert(c.table + toff, tcap, cc, cd)) ++s.miss;
}

__device__ __forceinline__ void flush_anchor(const Census5Args &c,
                                             AnchorSums &s) {
  s.k23 = wave_sum_u64(s.k23);
  s.w4 = wave_sum_u64(s.w4);
  s.a16 = wave_sum_u64(s.a16);
  s.miss = wave_sum_u64(s.miss);
  if (lane64() == 0) {
    if (s.k23) atomicAdd(&c.acc[kCensusK23], s.k23);
    if (s.w4) atomicAdd(&c.acc[kCensusW4], s.w4);
    if (s.a16) atomicAdd(&c.acc[kCensusK23e], s.a16);
    if (s.miss) atomicAdd(&c.acc[kCensusTableMiss], s.miss);
  }
}

constexpr uint32_t kListed = 0x80000000u;  // in lo: the target is listed

// Masks and counts of anchor a over the targets in (a, top) in global
// arrays of the workgroup (zero, left zero), the targets touched listed;
// masks of rs words.  All threads call it; the list is complete after it.
template <int WAVES>
__device__ __forceinline__ void anchor_global(
    const Census5Args &c, int32_t a, int32_t top, const int32_t *nb, int dp,
    int rs, unsigned long long *mask, uint32_t *lo, int32_t *list,
    unsigned *s_nt) {
  const int lane = lane64(), wv = threadIdx.x >> 6;
  auto touch = [&](int32_t cc, uint32_t seen) {
    if (!(seen & kListed) && !(atomicOr(&lo[cc], kListed) & kListed))
      list[atomicAdd(s_nt, 1u)] = cc;
  };
  for (int i = wv; i < dp; i += WAVES) {
    const int32_t y = nb[i];
    const unsigned long long bit = 1ull << (i & 63);
    const int64_t ey = top < c.n ? int64_t(c.win[y]) : c.rowptr[y + 1];
    const int64_t ky = wave_first_greater(c.col, a, c.rowptr[y], ey);
    for (int64_t k = ky + lane; k < ey; k += 64) {
      const int32_t cc = c.col[k];
      atomicOr(&mask[size_t(cc) * rs + (i >> 6)], bit);
      touch(cc, __hip_atomic_load(&lo[cc], __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT));
    }
  }
  // Through every z below a: the tail of N+(z) past a.
  const int64_t rb = c.rowptr[a], ea = c.rowptr[a + 1] - dp;
  for (int64_t k = rb + wv; k < ea; k += WAVES) {
    const int32_t z = c.col[k];
    const int64_t dz = c.drp[z + 1];
    const int64_t e =
        top < c.n ? dz - (c.rowptr[z + 1] - int64_t(c.win[z])) : dz;
    for (int64_t q = int64_t(c.arc[k]) + 1 + lane; q < e; q += 64) {
      const int32_t cc = c.dcol[q];
      touch(cc, atomicAdd(&lo[cc], 1u));
    }
  }
  __syncthreads();
}

constexpr int kWinT = 1024;
constexpr int kWinWaves = kWinT / 64;

// Windows of targets in LDS, left zero by every scan.  Masks over N+(a) of W
// words and counts of the neighbours below a, FW fine windows at a time.
template <int W, int FW>
struct WideWin {
  static constexpr int kHalves = 2 * W;  // of a mask, with bits set
  static constexpr int kWords = W, kFines = FW, kTargets = FW * kFine;
  static constexpr size_t kBytes = size_t(kTargets) * (8 * W + 4);
  unsigned long long *mask;
  uint32_t *lo;
  __device__ explicit WideWin(unsigned long long *lds)
      : mask(lds), lo(reinterpret_cast<uint32_t *>(lds + kTargets * W)) {}
  __device__ void add(unsigned k, unsigned dl, int t) const {
    if (k >= dl) {
      const unsigned i = k - dl;
      uint32_t *half = reinterpret_cast<uint32_t *>(mask + t * W + (i >> 6));
      atomicOr(half + ((i >> 5) & 1u), 1u << (i & 31u));
    } else {
      atomicAdd(&lo[t], 1u);
    }
  }
  template <class F>
  __device__ void scan(int span, unsigned, const F &f) const {
    for (int t = threadIdx.x; t < span; t += kWinT) {
      const unsigned low = lo[t];
      unsigned long long m[W], all = low;
#pragma unroll
      for (int w = 0; w < W; ++w) {
        m[w] = mask[t * W + w];
        all |= m[w];
      }
      if (!all) continue;
      lo[t] = 0;
#pragma unroll
      for (int w = 0; w < W; ++w) mask[t * W + w] = 0;
      f(t, low, m);
    }
  }
};

// Anchors of at most B neighbours, below and above: one bit each, in words
// of 32 (for B = 16 two targets half the window apart, so that adjacent ones
// lie in different banks) or 64 bits.
template <int B>
struct SmallWin {
  static constexpr int kHalves = B == 64 ? 2 : 1;
  static constexpr int kWords = 1, kFines = 320 / B, kTargets = kFines * kFine;
  static constexpr size_t kBytes = size_t(kTargets) * (B / 8);
  static constexpr int kHalf = kTargets / 2;
  unsigned long long *lds;
  __device__ explicit SmallWin(unsigned long long *l) : lds(l) {}
  __device__ void add(unsigned k, unsigned, int t) const {
    uint32_t *w = reinterpret_cast<uint32_t *>(lds);
    if (B == 16)
      atomicOr(&w[t < kHalf ? t : t - kHalf],
               1u << (t < kHalf ? k : k + 16u));
    else
      atomicOr(&w[B == 32 ? t : 2 * t + (k >> 5)], 1u << (k & 31u));
  }
  template <class F>
  __device__ void scan(int span, unsigned dl, const F &f) const {
    const unsigned long long below =
        dl < 64 ? (1ull << dl) - 1 : ~0ull;  // the neighbours below a
    auto one = [&](int t, unsigned long long x) {
      if (!x) return;
      const unsigned long long m[1] = {dl < 64 ? x >> dl : 0ull};
      f(t, static_cast<unsigned>(__popcll(x & below)), m);
    };
    if (B == 64) {
      for (int t = threadIdx.x; t < span; t += kWinT) {
        const unsigned long long x = lds[t];
        if (!x) continue;
        lds[t] = 0;
        one(t, x);
      }
    } else {
      uint32_t *w = reinterpret_cast<uint32_t *>(lds);
      const int words = B == 16 ? min(span, kHalf) : span;
      for (int i = threadIdx.x; i < words; i += kWinT) {
        const uint32_t x = w[i];
        if (!x) continue;
        w[i] = 0;
        if (B == 16) {
          one(i, x & 0xffffu);
          one(i + kHalf, x >> 16);
        } else {
          one(i, x);
        }
      }
    }
  }
};

// Adds the items of the anchor's d entries from rb in fine windows [f0, f1)
// (first id base).  64 entries at a time, dealt to the batches in turn (they
// are sorted by degree), an entry per lane for its range;
// the ranges are cut in pieces of 64 items, and the waves of a team (all 16
// for at most 64 entries, one each from 1024) take the pieces in turn: rows
// of hubs are far longer than the others.  True if there was an item.
template <class V>
__device__ __forceinline__ bool add_window(const Census5Args &c, int32_t a,
                                           int64_t rb, unsigned d, unsigned dl,
                                           int f0, int f1, int32_t base,
                                           const V &v) {
  constexpr int kU = 4;
  const int lane = lane64();
  const unsigned wv = wave_first(threadIdx.x >> 6);
  const int64_t stride = c.nf + 1;
  const unsigned batches = (d + 63) >> 6;
  const unsigned lg =
      batches <= 1 ? 0u : min(4u, 32u - __builtin_clz(batches - 1));
  const unsigned tw = kWinWaves >> lg;  // waves of a team
  bool any = false;
  for (unsigned bt = wv >> (4u - lg); bt < batches; bt += 1u << lg) {
    const unsigned k = bt + batches * lane;
    uint32_t b = 0, len = 0;
    if (k < d) {
      const int32_t y = c.col[rb + k];
      const uint16_t *wo = c.woff + woff_row(c, y) * stride;
      b = c.win[y] + wo[f0];
      len = uint32_t(wo[f1]) - wo[f0];
    }
    const uint32_t pieces = (len + 63) >> 6;
    uint32_t incl = pieces;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t x = __shfl_up(incl, o, 64);
      if (lane >= o) incl += x;
    }
    const uint32_t excl = incl - pieces;
    const uint32_t total = __builtin_amdgcn_readlane(incl, 63);
    any |= total != 0;
    for (uint32_t p = wv & (tw - 1u); p < total; p += tw * kU) {
      int32_t u[kU];
      uint32_t x[kU];
      bool ok[kU];
#pragma unroll
      for (int q = 0; q < kU; ++q) {
        const uint32_t pq = min(p + tw * q, total - 1u);
        x[q] = static_cast<uint32_t>(__popcll(__ballot(incl <= pq)));
        const uint32_t lx = __builtin_amdgcn_readlane(len, x[q]);
        const uint32_t at =
            64u * (pq - __builtin_amdgcn_readlane(excl, x[q])) + lane;
        ok[q] = p + tw * q < total && at < lx;
        u[q] = c.col[__builtin_amdgcn_readlane(b, x[q]) +
                     (at < lx ? at : lx - 1u)];
      }
#pragma unroll
      for (int q = 0; q < kU; ++q)
        if (ok[q] && u[q] > a) v.add(bt + batches * x[q], dl, u[q] - base);
    }
  }
  return any;
}

// All windows of anchor a, from the fine window of its first target.
template <class V>
__device__ __forceinline__ void anchor_windows(
    const Census5Args &c, int32_t a, int64_t rb, unsigned d, unsigned dl,
    unsigned long long *lds, const unsigned long long *rows, uint64_t toff,
    uint64_t tcap, AnchorSums &sums) {
  const V v(lds);
  for (int f0 = a < c.winlo ? 0 : (a + 1 - c.winlo) / kFine; f0 < c.nf;
       f0 += V::kFines) {
    const int32_t base = c.winlo + f0 * kFine;
    const int f1 = min(f0 + V::kFines, c.nf);
    const int any = add_window(c, a, rb, d, dl, f0, f1, base, v);
    if (!__syncthreads_or(any)) continue;
    v.scan(min(V::kTargets, c.n - base), dl,
           [&](int t, unsigned low, const unsigned long long(&m)[V::kWords]) {
             pair_terms<V::kWords, V::kHalves>(c, m, rows, low, base + t,
                                               toff, tcap, sums);
           });
    __syncthreads();  // the window is clear
  }
}

// 64-bit words of the window of class W: masks and counts of WideWin, or
// half the window at 16 bits a target (W = 1).
__host__ __device__ constexpr int win_words(int w) {
  return w == 1   ? static_cast<int>(SmallWin<16>::kBytes / 8)
         : w == 2 ? static_cast<int>(WideWin<2, 2>::kBytes / 8)
         : w == 4 ? static_cast<int>(WideWin<4, 1>::kBytes / 8)
                  : static_cast<int>(WideWin<8, 1>::kBytes / 8);
}
static_assert(WideWin<1, 3>::kBytes <= SmallWin<16>::kBytes &&
              SmallWin<32>::kBytes <= SmallWin<16>::kBytes &&
              SmallWin<64>::kBytes <= SmallWin<16>::kBytes);

// Anchors with d+ <= 64 W.  The targets in the window (the 65536 highest
// ids) take masks and counts in LDS, as many at a time as fit, from the
// anchor up: an item is one LDS atomic, and the window is read and cleared
// in order.  Most anchors have at most 16 neighbours and see the window in
// two parts.  Targets below it take the global arrays (a cache miss per item:
// 19e9 items per second for the whole device).  RMAT-18 (5.6e9 items), the
// four classes: 234 ms with every target in global arrays, 57 ms with windows
// of 1664 to 11648 targets for all anchors and a group of 16 lanes per row,
// 33 ms with a bit per neighbour and the rows cut in pieces, 29 ms with the
// entries dealt to the batches in turn, 23 ms with 32-bit mask sums, 18.6 ms
// with windows of half the size and two workgroups per CU.  Bound by the
// serial steps of an anchor (10 to 40 us) and, for half of the time, by the
// loops over the masks' bits.
constexpr int win_groups(int w) { return w <= 4 ? 2 : 1; }  // per CU
template <int W>
__global__ __launch_bounds__(kWinT, 4 * win_groups(W)) void c5_anchor(
    Census5Args c, C5List l) {
  using Wide = WideWin<W, W == 1 ? 3 : W == 2 ? 2 : 1>;
  extern __shared__ unsigned long long s_win[];
  unsigned long long *rows = s_win + win_words(W);
  int32_t *nb = reinterpret_cast<int32_t *>(rows + 64 * W * W);
  __shared__ unsigned s_a, s_nt;
  const int tid = threadIdx.x;
  const size_t below = static_cast<size_t>(c.winlo);
  unsigned long long *mask = c.mask + size_t(blockIdx.x) * below * W;
  uint32_t *lo = c.lo + size_t(blockIdx.x) * below;
  int32_t *list = c.list + size_t(blockIdx.x) * below;
  AnchorSums sums;
  for (int i = tid; i < win_words(W); i += kWinT) s_win[i] = 0;
  for (;;) {
    __syncthreads();
    if (tid == 0) {
      s_a = atomicAdd(l.cursor, 1u);
      s_nt = 0;
    }
    __syncthreads();
    const unsigned at = s_a;
    if (at >= l.count) break;
    const int32_t a = l.list[at];
    const int64_t ba = c.drp[a], rb = c.rowptr[a];
    const int dp = static_cast<int>(c.drp[a + 1] - ba);
    const unsigned d = static_cast<unsigned>(c.rowptr[a + 1] - rb);
    const unsigned dl = d - static_cast<unsigned>(dp);
    for (int i = tid; i < dp; i += kWinT) nb[i] = c.dcol[ba + i];
    for (int i = tid; i < dp * W; i += kWinT) rows[i] = 0;
    __syncthreads();
    build_rows<kWinT>(c, nb, dp, rows, W);
    const uint64_t toff = c.tab_off[a];
    const uint64_t tcap = c.tab_off[a + 1] - toff;
    if (a + 1 < c.winlo) {
      anchor_global<kWinWaves>(c, a, c.winlo, nb, dp, W, mask, lo, list,
                               &s_nt);
      const unsigned nt = s_nt;
      for (unsigned k = tid; k < nt; k += kWinT) {
        const int32_t cc = list[k];
        // Read and clear in one atomic each (made by atomics).
        unsigned long long m[W];
#pragma unroll
        for (int w = 0; w < W; ++w)
          m[w] = atomicExch(&mask[size_t(cc) * W + w], 0ull);
        pair_terms<W>(c, m, rows, atomicExch(&lo[cc], 0u) & ~kListed, cc,
                      toff, tcap, sums);
      }
    }
    // The rows are complete past the first window's barrier.
    if (W == 1 && d <= 16)
      anchor_windows<SmallWin<16>>(c, a, rb, d, dl, s_win, rows, toff, tcap,
                                   sums);
    else if (W == 1 && d <= 32)
      anchor_windows<SmallWin<32>>(c, a, rb, d, dl, s_win, rows, toff, tcap,
                                   sums);
    else if (W == 1 && d <= 64)
      anchor_windows<SmallWin<64>>(c, a, rb, d, dl, s_win, rows, toff, tcap,
                                   sums);
    else
      anchor_windows<Wide>(c, a, rb, d, dl, s_win, rows, toff, tcap, sums);
  }
  flush_anchor(c, sums);
}

// Light anchors (at most kLightItems items, d+ <= 64): one wave each, the
// targets in a hash table of 512 slots {target + 1, count}, {mask}.
constexpr int kLogSlots = 9;
constexpr int kLightWaves = 4;

__global__ __launch_bounds__(kLightWaves * 64) void c5_anchor_light(
    Census5Args c, C5List l) {
  constexpr int kSlots = 1 << kLogSlots;
  __shared__ unsigned long long s_key[kLightWaves][kSlots];
  __shared__ unsigned long long s_mask[kLightWaves][kSlots];
  __shared__ unsigned long long s_rows[kLightWaves][64];
  __shared__ int32_t s_nb[kLightWaves][64];
  const int lane = lane64(), wv = threadIdx.x >> 6;
  unsigned long long *key = s_key[wv], *mask = s_mask[wv], *rows = s_rows[wv];
  int32_t *nb = s_nb[wv];
  AnchorSums sums;
  auto slot = [&](int32_t u) {
    const unsigned long long k =
        static_cast<unsigned long long>(static_cast<uint32_t>(u) + 1u) << 32;
    uint32_t h = slot_of(u, kLogSlots);
    for (;;) {
      unsigned long long v = key[h];
      if (v == 0) v = atomicCAS(&key[h], 0ull, k);
      if (v == 0 || (v & ~0xffffffffull) == k) return h;
      h = (h + 1) & (kSlots - 1u);
    }
  };
  for (;;) {
    unsigned at = 0;
    if (lane == 0) at = atomicAdd(l.cursor, l.grab);
    at = wave_first(at);
    if (at >= l.count) break;
    const unsigned last = min(at + l.grab, l.count);
    for (; at < last; ++at) {
      const int32_t a = l.list[at];
      const int64_t ba = c.drp[a], rb = c.rowptr[a];
      const int dp = static_cast<int>(c.drp[a + 1] - ba);
      const int64_t ea = c.rowptr[a + 1] - dp;
      for (int i = lane; i < kSlots; i += 64) {
        key[i] = 0;
        mask[i] = 0;
      }
      if (lane < dp) nb[lane] = c.dcol[ba + lane];
      rows[lane] = 0;
      wave_sync();
      build_rows<64>(c, nb, dp, rows, 1);
      // A neighbour per lane for its range, then 16 lanes per range.
      for (int64_t k0 = rb; k0 < ea + dp; k0 += 64) {
        const int64_t k = k0 + lane;
        const bool in = k < ea + dp;
        uint32_t b = 0, e = 0;
        if (in) {
          const int32_t v = c.col[k];
          if (k < ea) {  // z below a: CSR positions of the tail past a
            e = static_cast<uint32_t>(c.rowptr[v + 1]);
            b = e - static_cast<uint32_t>(c.drp[v + 1]) + c.arc[k] + 1u;
          } else {       // y above a: entries past a are filtered
            b = static_cast<uint32_t>(c.rowptr[v]);
            e = static_cast<uint32_t>(c.rowptr[v + 1]);
          }
        }
        const int cnt = static_cast<int>(min(int64_t(64), ea + dp - k0));
        for (int x0 = 0; x0 < cnt; x0 += 4) {
          const int x = x0 + (lane >> 4);  // past cnt: an empty range
          const uint32_t bx = __shfl(b, x, 64);
          const uint32_t len = __shfl(e, x, 64) - bx;
          const int64_t kx = k0 + x;
          for (uint32_t j = lane & 15; j < len; j += 16u) {
            const int32_t u = c.col[bx + j];
            if (u <= a) continue;
            const uint32_t h = slot(u);
            if (kx >= ea) atomicOr(&mask[h], 1ull << (kx - ea));
            else atomicAdd(&key[h], 1ull);
          }
        }
      }
      wave_sync();
      const uint64_t toff = c.tab_off[a];
      const uint64_t tcap = c.tab_off[a + 1] - toff;
      for (int i = lane; i < kSlots; i += 64) {
        const unsigned long long v = key[i];
        if (!v) continue;
        const unsigned long long m[1] = {mask[i]};
        pair_terms<1>(c, m, rows, static_cast<uint32_t>(v),
                      static_cast<int32_t>(v >> 32) - 1, toff, tcap, sums);
      }
      wave_sync();
    }
  }
  flush_anchor(c, sums);
}

// Anchors with larger d+: rows in the workgroup's global slab, every target
// in the global arrays, masks of gen_words words.
__global__ __launch_bounds__(kT) void c5_anchor_gen(Census5Args c, C5List l) {
  __shared__ unsigned s_a, s_nt;
  const int rs = c.gen_words;
  const size_t n = static_cast<size_t>(c.n);
  unsigned long long *mask = c.mask + size_t(blockIdx.x) * n * rs;
  uint32_t *lo = c.lo + size_t(blockIdx.x) * n;
  int32_t *list = c.list + size_t(blockIdx.x) * n;
  unsigned long long *rows = c.grows + size_t(blockIdx.x) * c.grows_len;
  AnchorSums sums;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) {
      s_a = atomicAdd(l.cursor, 1u);
      s_nt = 0;
    }
    __syncthreads();
    const unsigned at = s_a;
    if (at >= l.count) break;
    const int32_t a = l.list[at];
    const int64_t ba = c.drp[a];
    const int dp = static_cast<int>(c.drp[a + 1] - ba);
    const int ru = (dp + 63) >> 6;  // words in use
    const int32_t *nb = c.dcol + ba;
    for (int64_t i = threadIdx.x; i < int64_t(dp) * rs; i += kT) rows[i] = 0;
    __syncthreads();
    build_rows<kT>(c, nb, dp, rows, rs);
    anchor_global<kTW>(c, a, c.n, nb, dp, rs, mask, lo, list, &s_nt);
    const unsigned nt = s_nt;
    const uint64_t toff = c.tab_off[a];
    const uint64_t tcap = c.tab_off[a + 1] - toff;
    for (unsigned k = threadIdx.x; k < nt; k += kT) {
      const int32_t cc = list[k];
      unsigned long long *mc = mask + size_t(cc) * rs;
      const uint32_t low = atomicExch(&lo[cc], 0u) & ~kListed;
      unsigned pc = 0;
      for (int w = 0; w < ru; ++w)
        pc += __popcll(__hip_atomic_load(&mc[w], __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT));
      const unsigned long long cd = static_cast<unsigned long long>(low) + pc;
      sums.k23 += choose3(cd);
      if (pc >= 2) {
        unsigned long long e2 = 0, wg = 0;
        for (int w = 0; w < ru; ++w) {
          const unsigned long long mw = __hip_atomic_load(
              &mc[w], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          for (unsigned long long b = mw; b; b &= b - 1) {
            const int p = w * 64 + __builtin_ctzll(b);
            unsigned dm = 0;
            for (int w2 = 0; w2 < ru; ++w2) {
              const unsigned long long m2 = __hip_atomic_load(
                  &mc[w2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              dm += __popcll(row_word(&rows[int64_t(p) * rs + w2], true) & m2);
            }
            e2 += dm;
            wg += choose2(dm);
          }
        }
        sums.w4 += wg;
        sums.a16 += (e2 >> 1) * (cd - 2);
      }
      for (int w = 0; w < ru; ++w) atomicExch(&mc[w], 0ull);
      if (low &&
          !tab_insert(c.table + toff, tcap, cc, static_cast<uint32_t>(cd)))
        ++sums.miss;
    }
  }
  flush_anchor(c, sums);
}

// Capacity of a table part of cnt pairs: a power of two, load at most 1/2.
__device__ __forceinline__ unsigned long long tab_capacity(unsigned cnt) {
  unsigned long long cap = cnt ? 2 : 0;
  while (cap < 2ull * cnt) cap <<= 1;
  return cap;
}

// The tails past a of the rows of the z below a (entries [rb, rb + cnt) of
// its row), with groups of 16 lanes, each up to 16 entries at a time.
template <class F>
__device__ __forceinline__ void walk_tails(const Census5Args &c, int64_t rb,
                                           unsigned cnt, int grp, int groups,
                                           int gl, const F &on_item) {
  unsigned per = (cnt + groups - 1) / groups;
  per = per > 16 ? 16 : (per < 1 ? 1 : per);
  for (unsigned k = grp * per; k < cnt; k += groups * per) {
    const unsigned take = min(per, cnt - k);
    uint32_t mb = 0, me = 0;
    if (static_cast<unsigned>(gl) < take) {
      mb = c.arc[rb + k + gl] + 1u;
      me = static_cast<uint32_t>(c.drp[c.col[rb + k + gl] + 1]);
    }
    for (unsigned x = 0; x < take; ++x) {
      const uint32_t b = __shfl(mb, static_cast<int>(x), 16);
      const uint32_t len = __shfl(me, static_cast<int>(x), 16) - b;
      for (uint32_t j = gl; j < len; j += 16u) on_item(c.dcol[b + j]);
    }
  }
}

// Table sizes: per anchor a, the distinct c above a with a common neighbour
// z below a (z->a, z->c).  Targets in the window are marked in a bitmap in
// LDS, the rest in the workgroup's stamps.  A hub has most of its
// neighbours below it and short tails: a serial chain of loads per
// neighbour, so a whole workgroup walks them, 1024 at a time (RMAT-18 with
// four waves per anchor and one neighbour each at a time: 12.0 ms).
__global__ __launch_bounds__(kWinT) void c5_tab_count(Census5Args c,
                                                      C5List l) {
  __shared__ uint32_t s_seen[kRowWindow / 32];
  __shared__ unsigned s_a, s_cnt;
  uint32_t *stamp = c.stamp + size_t(blockIdx.x) * size_t(c.winlo);
  for (int i = threadIdx.x; i < kRowWindow / 32; i += kWinT) s_seen[i] = 0;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) {
      s_a = atomicAdd(l.cursor, 1u);
      s_cnt = 0;
    }
    __syncthreads();
    const unsigned at = s_a;
    if (at >= l.count) break;
    const int32_t a = l.list[at];
    const int64_t rb = c.rowptr[a];
    const int64_t dp = c.drp[a + 1] - c.drp[a];
    const uint32_t tag = static_cast<uint32_t>(a) + 1u;
    unsigned mine = 0;
    walk_tails(c, rb, static_cast<unsigned>(c.rowptr[a + 1] - rb - dp),
               threadIdx.x >> 4, kWinT / 16, threadIdx.x & 15,
               [&](int32_t u) {
                 if (u >= c.winlo) {
                   const unsigned t = static_cast<unsigned>(u - c.winlo);
                   const uint32_t bit = 1u << (t & 31u);
                   mine += !(atomicOr(&s_seen[t >> 5], bit) & bit);
                 } else {
                   mine += atomicExch(&stamp[u], tag) != tag;
                 }
               });
    if (mine) atomicAdd(&s_cnt, mine);
    __syncthreads();
    if (threadIdx.x == 0) c.tab_cap[a] = tab_capacity(s_cnt);
    if (s_cnt)
      for (int i = threadIdx.x; i < kRowWindow / 32; i += kWinT) s_seen[i] = 0;
  }
}

// The same for the light anchors, a wave each, targets hashed.
__global__ __launch_bounds__(kLightWaves * 64) void c5_tab_count_light(
    Census5Args c, C5List l) {
  constexpr int kSlots = 1 << kLogSlots;
  __shared__ uint32_t s_key[kLightWaves][kSlots];
  const int lane = lane64();
  uint32_t *key = s_key[threadIdx.x >> 6];
  for (int i = lane; i < kSlots; i += 64) key[i] = 0;
  for (;;) {
    unsigned at = 0;
    if (lane == 0) at = atomicAdd(l.cursor, l.grab);
    at = wave_first(at);
    if (at >= l.count) break;
    const unsigned last = min(at + l.grab, l.count);
    for (; at < last; ++at) {
      const int32_t a = l.list[at];
      const int64_t rb = c.rowptr[a];
      const int64_t dp = c.drp[a + 1] - c.drp[a];
      wave_sync();
      unsigned long long mine = 0;
      walk_tails(c, rb, static_cast<unsigned>(c.rowptr[a + 1] - rb - dp),
                 lane >> 4, 4, lane & 15, [&](int32_t u) {
                   const uint32_t k = static_cast<uint32_t>(u) + 1u;
                   for (uint32_t h = slot_of(u, kLogSlots);;
                        h = (h + 1) & (kSlots - 1u)) {
                     const uint32_t v = atomicCAS(&key[h], 0u, k);
                     if (v == 0) ++mine;
                     if (v == 0 || v == k) break;
                   }
                 });
      mine = wave_sum_u64(mine);
      if (lane == 0) c.tab_cap[a] = tab_capacity(static_cast<unsigned>(mine));
      wave_sync();
      if (mine)
        for (int i = lane; i < kSlots; i += 64) key[i] = 0;
    }
  }
}

// The pairs of N+(x) seen from threads [tid, T): h(p, q) common neighbours
// inside it, each pair's 4-cycles into cyc, its diamonds' codegree from the
// table.
template <bool GLOBAL>
__device__ __forceinline__ void outnb_pairs(
    const Census5Args &c, const int32_t *nb, int dp,
    const unsigned long long *rows, int rs, int tid, int T,
    unsigned long long &cyc, unsigned long long &b16,
    unsigned long long &miss) {
  const int ru = (dp + 63) >> 6;
  // 32-bit division where dp is at most 512.
  using Index = typename std::conditional<GLOBAL, uint64_t, uint32_t>::type;
  const Index np = static_cast<Index>(dp) * static_cast<Index>(dp);
  for (Index k = tid; k < np; k += T) {
    const Index row = k / static_cast<Index>(dp);
    const int i = static_cast<int>(row);
    const int j = static_cast<int>(k - row * static_cast<Index>(dp));
    if (j <= i) continue;
    unsigned h = 0;
    for (int w = 0; w < ru; ++w)
      h += __popcll(row_word(&rows[int64_t(i) * rs + w], GLOBAL) &
                    row_word(&rows[int64_t(j) * rs + w], GLOBAL));
    if (!h) continue;
    cyc += choose2(h);
    const int32_t p = nb[i], q = nb[j];  // ascending: p below q
    const uint64_t off = c.tab_off[p];
    uint32_t cd = 0;
    if (tab_find(c.table + off, c.tab_off[p + 1] - off, q, &cd))
      b16 += static_cast<unsigned long long>(h) * (cd - 2ull);
    else
      ++miss;
  }
}

// Each 4-cycle of G[N+(x)] is seen at both of its diagonals.
__device__ __forceinline__ void flush_outnb(const Census5Args &c,
                                            unsigned long long w4,
                                            unsigned long long b16,
                                            unsigned long long miss) {
  w4 = wave_sum_u64(w4);
  b16 = wave_sum_u64(b16);
  miss = wave_sum_u64(miss);
  if (lane64() == 0) {
    if (w4) atomicAdd(&c.acc[kCensusW4], w4);
    if (b16) atomicAdd(&c.acc[kCensusK23e], b16);
    if (miss) atomicAdd(&c.acc[kCensusTableMiss], miss);
  }
}

template <int W>
__global__ __launch_bounds__(kT) void c5_outnb(Census5Args c, C5List l) {
  __shared__ int32_t s_nb[W > 0 ? 64 * W : 1];
  __shared__ unsigned long long s_rows[W > 0 ? 64 * W * W : 1];
  __shared__ unsigned s_a;
  __shared__ unsigned long long s_red[kTW];
  const int rs = W > 0 ? W : c.gen_words;
  unsigned long long *grows = c.grows + size_t(blockIdx.x) * c.grows_len;
  unsigned long long w4 = 0, b16 = 0, miss = 0;
  for (;;) {
    if (threadIdx.x == 0) s_a = atomicAdd(l.cursor, 1u);
    __syncthreads();
    const unsigned at = s_a;
    if (at >= l.count) break;
    const int32_t x = l.list[at];
    const int64_t bx = c.drp[x];
    const int dp = static_cast<int>(c.drp[x + 1] - bx);
    const int32_t *nb = W > 0 ? s_nb : c.dcol + bx;
    unsigned long long *rows = W > 0 ? s_rows : grows;
    if (W > 0)
      for (int i = threadIdx.x; i < dp; i += kT) s_nb[i] = c.dcol[bx + i];
    for (int64_t i = threadIdx.x; i < int64_t(dp) * rs; i += kT) rows[i] = 0;
    __syncthreads();
    build_rows<kT>(c, nb, dp, rows, rs);
    __syncthreads();
    unsigned long long cyc = 0;
    outnb_pairs<W == 0>(c, nb, dp, rows, rs, threadIdx.x, kT, cyc, b16, miss);
    const unsigned long long tot = wg_sum(cyc, s_red);
    if (threadIdx.x == 0) w4 += tot >> 1;
    __syncthreads();  // s_a and the rows are reused
  }
  flush_outnb(c, w4, b16, miss);
}

// Light anchors, nearly all with a handful of out-neighbours: a wave each.
__global__ __launch_bounds__(kLightWaves * 64) void c5_outnb_light(
    Census5Args c, C5List l) {
  __shared__ int32_t s_nb[kLightWaves][64];
  __shared__ unsigned long long s_rows[kLightWaves][64];
  const int lane = lane64(), wv = threadIdx.x >> 6;
  int32_t *nb = s_nb[wv];
  unsigned long long *rows = s_rows[wv];
  unsigned long long w4 = 0, b16 = 0, miss = 0;
  for (;;) {
    unsigned at = 0;
    if (lane == 0) at = atomicAdd(l.cursor, l.grab);
    at = wave_first(at);
    if (at >= l.count) break;
    const unsigned last = min(at + l.grab, l.count);
    for (; at < last; ++at) {
      const int32_t x = l.list[at];
      const int64_t bx = c.drp[x];
      const int dp = static_cast<int>(c.drp[x + 1] - bx);
      if (dp < 2) continue;
      if (lane < dp) nb[lane] = c.dcol[bx + lane];
      rows[lane] = 0;
      wave_sync();
      build_rows<64>(c, nb, dp, rows, 1);
      wave_sync();
      unsigned long long cyc = 0;
      outnb_pairs<false>(c, nb, dp, rows, 1, lane, 64, cyc, b16, miss);
      w4 += wave_sum_u64(cyc) >> 1;
      wave_sync();
    }
  }
  if (lane) w4 = 0;
  flush_outnb(c, w4, b16, miss);
}

}  // namespace

int census5_flat_launch(const Census5Args &c, int cus, hipStream_t s) {
  const int64_t items = std::max<int64_t>(c.n, c.nnz);
  const int g = static_cast<int>(std::max<int64_t>(
      1, std::min<int64_t>((items + kFlatT - 1) / kFlatT, int64_t(cus) * 2)));
  hipLaunchKernelGGL(c5_flat, dim3(g), dim3(kFlatT), 0, s, c);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int census5_classes(const Census5Args &c, int8_t *cls, unsigned *fill,
                    hipStream_t s) {
  const int g = std::max(1, std::min(8192, (c.n + 3) / 4));
  hipLaunchKernelGGL(c5_classes, dim3(g), dim3(256), 0, s, c, cls);
  hipLaunchKernelGGL(c5_scatter, dim3(c.n / kClassT + 1), dim3(kClassT), 0, s,
                     cls, c.n, nullptr, fill, nullptr);
  hipLaunchKernelGGL(c5_first, dim3(1), dim3(1), 0, s, c, fill + kC5Lists);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int census5_lists(int32_t n, const int8_t *cls, const unsigned *start,
                  unsigned *fill, int32_t *list, hipStream_t s) {
  hipLaunchKernelGGL(c5_scatter, dim3(n / kClassT + 1), dim3(kClassT), 0, s,
                     cls, n, start, fill, list);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int census5_fine_windows(int32_t n, int32_t winlo) {
  return (n - winlo + kFine - 1) / kFine;
}

int census5_window_offsets(const Census5Args &c, uint16_t *woff, int cus,
                           hipStream_t s) {
  const int64_t items = std::max<int64_t>(c.n, c.nnz);
  const int g = static_cast<int>(std::max<int64_t>(
      1, std::min<int64_t>((items + 255) / 256, int64_t(cus) * 32)));
  hipLaunchKernelGGL(c5_window_offsets, dim3(g), dim3(256), 0, s, c, woff);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int census5_scan_bytes(int64_t count, size_t *bytes) {
  size_t b = 0;
  const hipError_t e = hipcub::DeviceScan::ExclusiveSum(
      nullptr, b, static_cast<const unsigned long long *>(nullptr),
      static_cast<unsigned long long *>(nullptr), count);
  *bytes = b;
  return e == hipSuccess ? 0 : -1;
}

int census5_scan(const unsigned long long *in, unsigned long long *out,
                 int64_t count, void *tmp, size_t tmp_bytes, hipStream_t s) {
  size_t b = tmp_bytes;
  return hipcub::DeviceScan::ExclusiveSum(tmp, b, in, out, count, s) ==
                 hipSuccess
             ? 0
             : -1;
}

namespace {

size_t win_lds(int w) {
  return (size_t(win_words(w)) + 64 * w * w) * 8 + 64 * w * 4;
}

template <int K>
int launch_windowed(const Census5Args &c, const C5List &l, int grid,
                    hipStream_t s) {
  constexpr int W = kC5Words[K];
  if (!l.count) return 0;
  hipLaunchKernelGGL((c5_anchor<W>), dim3(grid), dim3(kWinT), win_lds(W), s, c,
                     l);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// The lists of the anchors, queued on cursors from `cursor` on; light ones
// up to 8 per queue access, one while waves are left idle.
void lists_of(const Census5Args &c, const uint32_t *count, unsigned *cursor,
              int cus, C5List *l) {
  const int32_t *at = c.anchors;
  for (int k = 0; k < kC5Lists; ++k) {
    l[k].list = at;
    l[k].count = count[k];
    l[k].cursor = cursor + k;
    at += count[k];
  }
  l[kC5Light].grab = static_cast<uint32_t>(std::max<int64_t>(
      1, std::min<int64_t>(8, count[kC5Light] / (cus * 8 * kLightWaves))));
}

int light_grid(const C5List &l, int cus) {
  return static_cast<int>(std::min<int64_t>(
      (int64_t(l.count) + kLightWaves - 1) / kLightWaves, int64_t(cus) * 4));
}

template <int W>
int launch_outnb(const Census5Args &c, const C5List &l, int most,
                 hipStream_t s) {
  if (!l.count) return 0;
  const int g = static_cast<int>(std::min<int64_t>(l.count, most));
  hipLaunchKernelGGL((c5_outnb<W>), dim3(g), dim3(kT), 0, s, c, l);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace

int census5_init() {
  const void *kern[kC5Windowed] = {
      reinterpret_cast<const void *>(&c5_anchor<1>),
      reinterpret_cast<const void *>(&c5_anchor<2>),
      reinterpret_cast<const void *>(&c5_anchor<4>),
      reinterpret_cast<const void *>(&c5_anchor<8>)};
  for (int k = 0; k < kC5Windowed; ++k)
    if (hipFuncSetAttribute(kern[k],
                            hipFuncAttributeMaxDynamicSharedMemorySize,
                            static_cast<int>(win_lds(kC5Words[k]))) !=
        hipSuccess)
      return -1;
  return 0;
}

int census5_groups(int cls, int64_t count, int32_t n, int32_t winlo,
                   int gen_words, size_t budget, int cus) {
  if (count <= 0 || cls == kC5Light) return 0;
  const bool gen = cls == kC5Lists - 1;
  // Two to a CU pay where every workgroup gets several anchors: RMAT-18's
  // 134000 of d+ <= 64 16.4 -> 11.8 ms, RMAT-10's 390 78 -> 103 us.
  const int64_t per_cu =
      gen ? 4 : count >= int64_t(cus) * 4 ? win_groups(kC5Words[cls - 1]) : 1;
  int64_t g = std::min<int64_t>(count, cus * per_cu);
  const size_t range = static_cast<size_t>(gen ? n : winlo);
  const size_t words = static_cast<size_t>(gen ? gen_words
                                               : kC5Words[cls - 1]);
  if (range)
    g = std::min<int64_t>(
        g, static_cast<int64_t>(budget / (range * (8 * words + 8))));
  return static_cast<int>(std::max<int64_t>(g, 1));
}

int census5_table_count_launch(const Census5Args &c, const uint32_t *count,
                               int cus, hipStream_t s) {
  C5List l[kC5Lists];
  lists_of(c, count, c.cursor, cus, l);
  // The heavy anchors follow the light ones as one list.
  C5List heavy = l[1];
  for (int k = 2; k < kC5Lists; ++k) heavy.count += l[k].count;
  const int g = static_cast<int>(std::min<int64_t>(heavy.count, c.groups));
  if (g) hipLaunchKernelGGL(c5_tab_count, dim3(g), dim3(kWinT), 0, s, c, heavy);
  if (const int lg = light_grid(l[kC5Light], cus))
    hipLaunchKernelGGL(c5_tab_count_light, dim3(lg), dim3(kLightWaves * 64), 0,
                       s, c, l[kC5Light]);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int census5_pairs_launch(const Census5Args &c, const uint32_t *count,
                         const int *groups, int cus, hipStream_t s) {
  C5List l[kC5Lists];
  lists_of(c, count, c.cursor, cus, l);
  if (l[kC5Lists - 1].count)
    hipLaunchKernelGGL(c5_anchor_gen, dim3(groups[kC5Lists - 1]), dim3(kT), 0,
                       s, c, l[kC5Lists - 1]);
  if (launch_windowed<3>(c, l[4], groups[4], s) ||
      launch_windowed<2>(c, l[3], groups[3], s) ||
      launch_windowed<1>(c, l[2], groups[2], s) ||
      launch_windowed<0>(c, l[1], groups[1], s))
    return -1;
  const int lg = light_grid(l[kC5Light], cus);
  if (lg)
    hipLaunchKernelGGL(c5_anchor_light, dim3(lg), dim3(kLightWaves * 64), 0,
                       s, c, l[kC5Light]);
  lists_of(c, count, c.cursor + kC5Lists, cus, l);
  if (lg)
    hipLaunchKernelGGL(c5_outnb_light, dim3(lg), dim3(kLightWaves * 64), 0, s,
                       c, l[kC5Light]);
  const int most = cus * 8;
  if (launch_outnb<1>(c, l[1], most, s)) return -1;
  if (launch_outnb<2>(c, l[2], most, s) || launch_outnb<4>(c, l[3], most, s) ||
      launch_outnb<8>(c, l[4], most, s) ||
      launch_outnb<0>(c, l[5], groups[kC5Lists - 1], s))
    return -1;
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace mgpm

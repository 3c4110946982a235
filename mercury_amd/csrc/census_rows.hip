// Triangles per edge, 4- and 5-cliques by bit rows inside out-neighbourhoods.
//
// One workgroup takes one vertex x of the census graph (relabelled in DAG
// order, rank = id) with its out-neighbours N+(x) = {y_0 < y_1 < ...}, and
// streams two sets of sorted lists against N+(x):
//   * N+(y) for every y in N+(x): a hit z closes the triangle {x, y, z}.
//     The hits are the adjacency inside N+(x), kept as bit rows
//     U[i] (bit j: y_i ~ y_j);
//   * the tail of N+(w) past x for every w below x: a hit y closes the
//     triangle {w, x, y}.  The hits are the rows L[i] over the lower
//     neighbours of x (bit k: y_i ~ w_k), taken in chunks of columns that
//     fit the rows' storage.
// U[i] and L[i] together are N(x) ∩ N(y_i), so
//   t(x, y_i)  = |U[i]| + |L[i]|                (triangles on the edge),
//   k(x, y_i, y_j) = |U[i] & U[j]| + |L[i] & L[j]|  (4-cliques on the
//     triangle), and the 4- and 5-cliques whose lowest vertex is x are row
//     intersections of U restricted to the bits above the last vertex.
// Every list is streamed with one membership test per item -- no search --
// and a 4-clique test costs 1/64 of a word operation.
//
// Membership: a bitmap over the 65536 highest ids in LDS (8 KB) with, per
// word, the index in N+(x) of the first neighbour in it, so a hit's position
// is that index plus a popcount.  Ids below the window (a thousandth of the
// items on RMAT graphs, most of them on large graphs without skew, where
// lists are short) are searched in the sorted head of N+(x) below it.
//
// What bounds it: the lists are gathered from the DAG's columns (63 MB at
// RMAT-20, in the last-level cache), four loads per lane in flight, and the
// row intersections are LDS reads.  RMAT-20 (16 draws per vertex) streams
// 4.4e9 + 1.2e9 items and intersects 9.6e9 word pairs.  Measured on one
// MI355X against one wave per DAG arc with binary searches (arcs from one
// atomic cursor, 11 ns each): t and 4-cliques at RMAT-20 329 -> 7.3 ms;
// P7 at RMAT-18 280 -> 8.0 ms; P1 on 300007 vertices of degree 16
// (2.4 million arcs) 27.4 -> 0.26 ms (census_tiny).  Before the vertices with many lower
// neighbours went to the large workgroups and the ranges were loaded 16 at a
// time, 20.3 and 17.9 ms.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "census.hpp"
#include "choose.hpp"
#include "wave.hpp"

namespace mgpm {

namespace {

typedef unsigned long long u64;

constexpr int kWindow = 65536;           // ids of the bitmap
constexpr int kWindowWords = kWindow / 32;
constexpr int kLanesPerList = 16;        // lanes that walk one list
constexpr int kUnroll = 4;               // loads in flight per lane

// Classes by the neighbours above and below x: rows in LDS up to 704 above,
// in the workgroup's global slab beyond.  The lower neighbours cost a chain
// of loads each and the highest ids have few neighbours but thousands below
// them, so those go to the large workgroups: with classes by |N+(x)| alone
// the 64 highest ids of RMAT-20 (1e6 lower neighbours, 0.3% of the items)
// kept eight workgroups of 256 busy for 13 of the class's 15.4 ms.
// `words`: 64-bit words of row storage (U, then as many columns of L as
// fit); `grab`: most vertices per queue access.
struct RowClass {
  int max_out, max_below, threads, words, words_u, grab;
};
constexpr int kAnyBelow = 0x7fffffff;
constexpr int kTinyMax = 32;
enum : int { kSmallClass = 0, kTinyClass = 1 };
// Tiny vertices up to this number, and all in the pass over cliques, are
// taken with the small class: RMAT-10's 800 cost a launch of 12 us more than
// they save.
constexpr int64_t kTinyFew = 4096;
constexpr RowClass kRowClasses[kRowClassCount] = {
    {64, 256, 256, 320, 64, 8},
    {kTinyMax, kTinyMax, 256, 1, 1, 1},  // a wave each (census_tiny)
    {256, 1024, 512, 4096, 1024, 1},
    {704, kAnyBelow, 1024, 13312, 7744, 1},
    {0x7fffffff, kAnyBelow, 1024, 0, 0, 1},
};
constexpr int kSlabL = 8;  // words of L per row in the global slab

struct Locator {
  const uint32_t *bits;
  const uint16_t *base;
  const int32_t *nb;
  int32_t winlo;
  int low;  // neighbours below the window
  // The index of z in N+(x), or -1.
  __device__ __forceinline__ int find(int32_t z, bool ok) const {
    const uint32_t k = static_cast<uint32_t>(z - winlo);
    const bool in = k < static_cast<uint32_t>(kWindow);
    const uint32_t word = bits[in ? k >> 5 : 0u];
    int pos = -1;
    if (in) {
      if (ok && (word >> (k & 31)) & 1u)
        pos = base[k >> 5] + __popc(word & ((1u << (k & 31)) - 1u));
    } else if (ok && low > 0) {
      int lo = 0, hi = low;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (nb[mid] < z) lo = mid + 1;
        else hi = mid;
      }
      if (lo < low && nb[lo] == z) pos = lo;
    }
    return pos;
  }
};

// Items [b, e) of the DAG columns, walked by 16 lanes: on_item(q, pos, hit)
// for every item, called by all active lanes together.
template <class F>
__device__ __forceinline__ void stream_list(const int32_t *__restrict__ dcol,
                                            uint32_t b, uint32_t e, int gl,
                                            const Locator &loc,
                                            const F &on_item) {
  for (uint32_t q = b + gl; q < e; q += kLanesPerList * kUnroll) {
    int32_t z[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const uint32_t qq = q + kLanesPerList * u;
      z[u] = dcol[qq < e ? qq : q];
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const uint32_t qq = q + kLanesPerList * u;
      on_item(qq, loc.find(z[u], qq < e));
    }
  }
}

// Lists [0, cnt) dealt in turn to `groups` groups of 16 lanes (this one
// `grp`), each up to 16 of its lists at a time: their ranges are loaded one per lane, so the
// chain of loads to a range is paid once for all of them.  In turn, as the
// lists are sorted by degree: with 16 in a row per group the two classes of
// large workgroups took 8.9 ms on RMAT-20, in turn 4.9.
// on_item(list, q, pos) as in stream_list.
template <class R, class F>
__device__ __forceinline__ void walk_lists(const int32_t *__restrict__ dcol,
                                           int cnt, int grp, int groups,
                                           int gl, const Locator &loc,
                                           const R &range, const F &on_item) {
  for (int k = grp; k < cnt; k += groups * kLanesPerList) {
    const int mine = k + gl * groups;
    uint32_t mb = 0, me = 0;
    if (mine < cnt) range(mine, mb, me);
    for (int i = 0, at = k; i < kLanesPerList && at < cnt;
         ++i, at += groups) {
      const uint32_t b = __shfl(mb, i, kLanesPerList);
      const uint32_t e = __shfl(me, i, kLanesPerList);
      stream_list(dcol, b, e, gl, loc,
                  [&](uint32_t q, int pos) { on_item(at, q, pos); });
    }
  }
}

__device__ __forceinline__ void or_bit(u64 *row, int bit) {
  atomicOr(reinterpret_cast<uint32_t *>(row) + (bit >> 5), 1u << (bit & 31));
}

// Words of a row written by atomics: LDS rows read plainly, rows in global
// memory past the vector L1 (the atomics ran in L2).
template <bool LDS>
__device__ __forceinline__ u64 row_get(const u64 *r) {
  return LDS ? *r
             : __hip_atomic_load(r, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
}

// Word w of the bits above position j.
__device__ __forceinline__ u64 above_word(int j, int w) {
  const int s = j - 64 * w;  // bits 0..s are cleared
  return s < 0 ? ~0ull : (s >= 63 ? 0ull : ~0ull << (s + 1));
}

// CLIQUES = false: t of every arc and the 4-cliques.  CLIQUES = true: the
// sums over triangles and the 5-cliques (t complete).  WU: words of a row
// of U that are kept in registers (0: rows in the global slab).
template <int T, int WU, bool CLIQUES>
__global__ __launch_bounds__(T) void census_rows(CensusArgs c, RowArgs r) {
  constexpr bool LDS = WU > 0;
  extern __shared__ u64 s_dyn[];
  __shared__ uint32_t s_bits[kWindowWords];
  __shared__ uint16_t s_base[kWindowWords];
  __shared__ unsigned s_next, s_nt;
  __shared__ int s_low;
  const int tid = threadIdx.x;
  const int lane = lane64();
  const int gl = tid & (kLanesPerList - 1);
  const int grp = tid / kLanesPerList;
  constexpr int kGroups = T / kLanesPerList;
  // Row storage, then neighbour ids and counters (LDS classes); the slab of
  // the workgroup holds what is not in LDS.
  char *slab = r.slab + size_t(blockIdx.x) * r.slab_bytes;
  u64 *rows;
  int32_t *nbs;
  uint32_t *cnt;
  if (LDS) {
    rows = s_dyn;
    nbs = reinterpret_cast<int32_t *>(s_dyn + r.words);
    cnt = reinterpret_cast<uint32_t *>(nbs + r.pcap);
  } else {
    rows = reinterpret_cast<u64 *>(slab);
    cnt = reinterpret_cast<uint32_t *>(rows + r.words);
    nbs = nullptr;
    slab += size_t(r.words) * 8 + size_t(r.pcap) * 4;
    slab = reinterpret_cast<char *>(
        (reinterpret_cast<uintptr_t>(slab) + 7) & ~uintptr_t(7));
  }
  uint2 *tri = reinterpret_cast<uint2 *>(slab);
  uint32_t *kacc = reinterpret_cast<uint32_t *>(slab + size_t(r.tri_cap) * 8);
  u64 k4 = 0, k5 = 0, kk = 0, tek = 0, tdk = 0, dp2 = 0, gem = 0, bad = 0;
  for (int i = tid; i < kWindowWords; i += T) s_bits[i] = 0;
  // The first vertices by workgroup, the rest from the queue.
  const unsigned grab = static_cast<unsigned>(r.grab);
  unsigned first = blockIdx.x * grab;
  for (;; first = s_next) {
    __syncthreads();
    if (first >= r.count) break;
    if (tid == 0) s_next = (gridDim.x * grab < r.count
                                ? atomicAdd(r.cursor, grab)
                                : r.count) +
                           gridDim.x * grab;
    const unsigned last = min(first + grab, r.count);
    for (unsigned ai = first; ai < last; ++ai) {
      const int32_t x = r.list[ai];
      const int64_t bx = c.drp[x];
      const int P = static_cast<int>(c.drp[x + 1] - bx);
      const int64_t rb = c.rowptr[x];
      const int dx = c.deg[x];
      const int DL = dx - P;
      const int wu = (P + 63) >> 6;
      const int32_t *nb = LDS ? nbs : c.dcol + bx;
      for (int i = tid; i < P; i += T) {
        if (LDS) nbs[i] = c.dcol[bx + i];
        cnt[i] = 0;
      }
      for (int i = tid; i < P * wu; i += T) rows[i] = 0;
      if (tid == 0) {
        s_low = 0;
        s_nt = 0;
      }
      __syncthreads();
      for (int i = tid; i < P; i += T) {
        const int32_t k = nb[i] - c.winlo;
        if (k >= 0) {
          const int w = k >> 5;
          atomicOr(&s_bits[w], 1u << (k & 31));
          if (i == 0 || ((nb[i - 1] - c.winlo) >> 5) != w)
            s_base[w] = static_cast<uint16_t>(i);
        } else if (i + 1 == P || nb[i + 1] >= c.winlo) {
          s_low = i + 1;
        }
      }
      __syncthreads();
      const Locator loc{s_bits, s_base, nb, c.winlo, s_low};
      u64 *U = rows;
      if (P >= 2) {
        auto above = [&](int i, uint32_t &b, uint32_t &e) {
          const int32_t y = nb[i];
          b = static_cast<uint32_t>(c.drp[y]);
          e = static_cast<uint32_t>(c.drp[y + 1]);
        };
        walk_lists(
            c.dcol, P, grp, kGroups, gl, loc, above,
            [&](int i, uint32_t q, int pos) {
              if constexpr (CLIQUES) {
                const bool hit = pos >= 0;
                const u64 m = __ballot(hit);
                if (m) {
                  const int lead = __builtin_ctzll(m);
                  unsigned o = 0;
                  if (lane == lead)
                    o = atomicAdd(&s_nt, static_cast<unsigned>(__popcll(m)));
                  o = __shfl(o, lead, 64) + bits_below(m);
                  if (hit) {
                    or_bit(U + size_t(i) * wu, pos);
                    or_bit(U + size_t(pos) * wu, i);
                    tri[o] = make_uint2(static_cast<unsigned>(i) |
                                            static_cast<unsigned>(pos) << 16,
                                        q);
                  }
                }
              } else if (pos >= 0) {
                or_bit(U + size_t(i) * wu, pos);
                atomicAdd(&cnt[pos], 1u);
              }
            });
      }
      // The tails past x of the lower neighbours' lists.
      auto below = [&](int64_t k, uint32_t &b, uint32_t &e) {
        b = c.arc[rb + k] + 1u;
        e = static_cast<uint32_t>(c.drp[c.col[rb + k] + 1]);
      };
      if constexpr (!CLIQUES) {
        walk_lists(c.dcol, DL, grp, kGroups, gl, loc, below,
                   [&](int, uint32_t, int pos) {
                     if (pos >= 0) atomicAdd(&cnt[pos], 1u);
                   });
        __syncthreads();
        for (int i = tid; i < P; i += T) {
          uint32_t t = LDS ? cnt[i]
                           : __hip_atomic_load(&cnt[i], __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
          for (int w = i >> 6; w < wu; ++w)
            t += __popcll(row_get<LDS>(&U[size_t(i) * wu + w]));
          c.t[bx + i] = t;
        }
        // 4-cliques: U holds only the bits above the row, so the shared
        // bits of rows i and j (j in row i) lie above j.
        for (int p = tid; p < P * wu; p += T) {
          const int i = p / wu, w0 = p - i * wu;
          for (u64 b = row_get<LDS>(&U[p]); b; b &= b - 1) {
            const int j = 64 * w0 + __builtin_ctzll(b);
            for (int w = w0; w < wu; ++w)
              k4 += static_cast<u64>(
                  __popcll(row_get<LDS>(&U[size_t(i) * wu + w]) &
                           row_get<LDS>(&U[size_t(j) * wu + w])));
          }
        }
      } else {
        // Columns of L per chunk: what the storage holds beside U, whole
        // words, at most the words there are.
        const int WL = (DL + 63) >> 6;
        int wl = LDS ? (r.words - P * wu) / P : kSlabL;
        if (wl > WL) wl = WL;
        u64 *Lr = rows + size_t(P) * wu;
        const int chunks = WL > 0 ? (WL + wl - 1) / wl : 1;
        for (int ch = 0; ch < chunks; ++ch) {
          const int k0 = ch * wl * 64;
          const int k1 = min(DL, k0 + wl * 64);
          const int wc = (k1 - k0 + 63) >> 6;  // 0 when DL = 0
          for (int i = tid; i < P * wc; i += T) Lr[i] = 0;
          __syncthreads();
          walk_lists(c.dcol, k1 - k0, grp, kGroups, gl, loc,
                     [&](int k, uint32_t &b, uint32_t &e) {
                       below(k0 + k, b, e);
                     },
                     [&](int k, uint32_t, int pos) {
                       if (pos >= 0) or_bit(Lr + size_t(pos) * wc, k);
                     });
          __syncthreads();
          for (int i = tid; i < P; i += T) {
            uint32_t t = 0;
            if (ch == 0)
              for (int w = 0; w < wu; ++w)
                t += __popcll(row_get<LDS>(&U[size_t(i) * wu + w]));
            for (int w = 0; w < wc; ++w)
              t += __popcll(row_get<LDS>(&Lr[size_t(i) * wc + w]));
            t += cnt[i];  // this thread's own sum of the earlier chunks
            cnt[i] = t;
            if (ch == chunks - 1 && t != c.t[bx + i]) ++bad;
          }
          const unsigned nt = s_nt;
          for (unsigned p = tid; p < nt; p += T) {
            const uint2 e = tri[p];
            const int i = static_cast<int>(e.x & 0xffffu);
            const int j = static_cast<int>(e.x >> 16);
            unsigned kt = 0;
            if (ch == 0) {
              // The shared bits of rows i and j; those above j are the
              // 4-cliques with lowest vertex x, the pairs among them the
              // 5-cliques.
              if constexpr (LDS) {
                u64 S[WU];
#pragma unroll
                for (int w = 0; w < WU; ++w) {
                  S[w] = 0;
                  if (w < wu) {
                    const u64 a = U[size_t(i) * wu + w] & U[size_t(j) * wu + w];
                    kt += __popcll(a);
                    S[w] = a & above_word(j, w);
                    k4 += static_cast<u64>(__popcll(S[w]));
                  }
                }
#pragma unroll
                for (int w = 0; w < WU; ++w) {
                  for (u64 b = S[w]; b; b &= b - 1) {
                    const int v = __builtin_ctzll(b);
                    const u64 *rv = U + size_t(64 * w + v) * wu;
                    unsigned s5 = __popcll(rv[w] & (b & (b - 1)));
#pragma unroll
                    for (int w2 = w + 1; w2 < WU; ++w2)
                      if (w2 < wu) s5 += __popcll(rv[w2] & S[w2]);
                    k5 += s5;
                  }
                }
              } else {
                for (int w = 0; w < wu; ++w) {
                  const u64 a = row_get<LDS>(&U[size_t(i) * wu + w]) &
                                row_get<LDS>(&U[size_t(j) * wu + w]);
                  kt += __popcll(a);
                  const u64 s = a & above_word(j, w);
                  k4 += static_cast<u64>(__popcll(s));
                  for (u64 b = s; b; b &= b - 1) {
                    const int v = 64 * w + __builtin_ctzll(b);
                    for (int w2 = w; w2 < wu; ++w2)
                      k5 += static_cast<u64>(__popcll(
                          row_get<LDS>(&U[size_t(i) * wu + w2]) &
                          row_get<LDS>(&U[size_t(j) * wu + w2]) &
                          row_get<LDS>(&U[size_t(v) * wu + w2]) &
                          above_word(v, w2)));
                  }
                }
              }
            } else {
              kt = kacc[p];
            }
            for (int w = 0; w < wc; ++w)
              kt += __popcll(row_get<LDS>(&Lr[size_t(i) * wc + w]) &
                             row_get<LDS>(&Lr[size_t(j) * wc + w]));
            if (ch + 1 < chunks) {
              kacc[p] = kt;
              continue;
            }
            const u64 txy = c.t[bx + i], txz = c.t[bx + j], tyz = c.t[e.y];
            const u64 dy = c.deg[nb[i]], dz = c.deg[nb[j]];
            const u64 k = kt;
            kk += choose2(k);
            tek += k * (txy + txz + tyz - 6);
            tdk += k * (static_cast<u64>(dx) + dy + dz - 9);
            if (c.full5) {  // edge counts >= 1, degrees >= 2
              const u64 a = txy - 1, b = txz - 1, g = tyz - 1;
              dp2 += a * (dz - 2) + b * (dy - 2) +
                     g * static_cast<u64>(dx - 2);
              gem += a * b + a * g + b * g;
            }
          }
          __syncthreads();  // the chunk's rows are cleared next
        }
      }
      __syncthreads();
      for (int i = tid; i < P; i += T) {
        const int32_t k = nb[i] - c.winlo;
        if (k >= 0) s_bits[k >> 5] = 0;
      }
      __syncthreads();  // the neighbours and rows are overwritten
    }
  }
  k4 = wave_sum_u64(k4);
  if constexpr (CLIQUES) {
    k5 = wave_sum_u64(k5);
    kk = wave_sum_u64(kk);
    tek = wave_sum_u64(tek);
    tdk = wave_sum_u64(tdk);
    dp2 = wave_sum_u64(dp2);
    gem = wave_sum_u64(gem);
    bad = wave_sum_u64(bad);
  }
  if (lane == 0) {
    if (k4) atomicAdd(&c.acc[CLIQUES ? kCensusK4Rows : kCensusK4], k4);
    if constexpr (CLIQUES) {
      if (k5) atomicAdd(&c.acc[kCensusK5], k5);
      if (kk) atomicAdd(&c.acc[kCensusTriPairs], kk);
      if (tek) atomicAdd(&c.acc[kCensusTriEdgeK], tek);
      if (tdk) atomicAdd(&c.acc[kCensusTriDegK], tdk);
      if (dp2) atomicAdd(&c.acc[kCensusDp2], dp2);
      if (gem) atomicAdd(&c.acc[kCensusGem], gem);
      if (bad) atomicAdd(&c.acc[kCensusMismatch], bad);
    }
  }
}

// t of every arc and the 4-cliques for vertices of at most 32 neighbours on
// either side: one wave each, nothing shared, no barriers.  All ranges are
// loaded at once, one list per lane; groups of eight lanes walk the lists; an
// item is looked up in a hash table of 128 slots (the bitmap of the other
// classes would leave room for 12 waves per CU); a row of U is one word.
// The steps of a vertex are a chain of loads whoever takes them: P1 on 300007
// vertices of degree 16 793 us with a workgroup of 256 per vertex, 262 us with
// a wave; RMAT-20's 586000 vertices of up to 64 out-neighbours 2.4 ms, now
// 0.7 and, for the tiny ones, 1.4.
constexpr int kTinyWaves = 4;
constexpr int kLogTiny = 7;

__global__ __launch_bounds__(kTinyWaves * 64, 8) void census_tiny(
    CensusArgs c, const int32_t *__restrict__ list, uint32_t count) {
  constexpr uint32_t kSlots = 1u << kLogTiny;
  constexpr int kL = 8, kG = 64 / kL, kMax = kTinyMax;
  __shared__ int32_t s_key[kTinyWaves][kSlots];
  __shared__ uint8_t s_idx[kTinyWaves][kSlots];
  __shared__ uint32_t s_row[kTinyWaves][kMax], s_cnt[kTinyWaves][kMax];
  const int lane = lane64(), wv = threadIdx.x >> 6;
  int32_t *key = s_key[wv];
  uint8_t *idx = s_idx[wv];
  uint32_t *U = s_row[wv], *cnt = s_cnt[wv];
  const int gl = lane & (kL - 1), grp = lane / kL;
  for (uint32_t i = lane; i < kSlots; i += 64) key[i] = -1;
  u64 k4 = 0;
  const uint32_t waves = gridDim.x * kTinyWaves;
  for (uint32_t at = blockIdx.x * kTinyWaves + wv; at < count; at += waves) {
    const int32_t x = list[at];
    const int64_t bx = c.drp[x], rb = c.rowptr[x];
    const int P = static_cast<int>(c.drp[x + 1] - bx);
    const int d = static_cast<int>(c.rowptr[x + 1] - rb);  // at most 64
    // The last P entries of the row are N+(x).
    uint32_t mb = 0, me = 0, slot = 0;
    const int i0 = lane - (d - P);  // position in N+(x)
    const bool mine = lane < d && i0 >= 0;
    if (lane < d) {
      const int32_t y = c.col[rb + lane];
      me = static_cast<uint32_t>(c.drp[y + 1]);
      mb = mine ? static_cast<uint32_t>(c.drp[y]) : c.arc[rb + lane] + 1u;
      if (mine) {
        slot = slot_of(y, kLogTiny);
        while (atomicCAS(&key[slot], -1, y) != -1)
          slot = (slot + 1) & (kSlots - 1);
        idx[slot] = static_cast<uint8_t>(i0);
      }
    }
    if (lane < kMax) {
      U[lane] = 0;
      cnt[lane] = 0;
    }
    wave_sync();
    // The whole wave steps together (a shuffle reads active lanes only);
    // lists past the last are empty.
    for (int first = 0; first < d; first += kG) {
      const uint32_t b = __shfl(mb, first + grp, 64);
      const uint32_t e = __shfl(me, first + grp, 64);
      const int row = first + grp - (d - P);
      for (uint32_t q = b + gl; q < e; q += kL * kUnroll) {
        int32_t z[kUnroll], k[kUnroll];
        uint32_t h[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          const uint32_t qq = q + kL * u;
          z[u] = c.dcol[qq < e ? qq : q];
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          h[u] = slot_of(z[u], kLogTiny);
          k[u] = key[h[u]];
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          while (k[u] != -1 && k[u] != z[u]) {
            h[u] = (h[u] + 1) & (kSlots - 1);
            k[u] = key[h[u]];
          }
          if (k[u] == z[u] && q + kL * u < e) {
            const uint32_t pos = idx[h[u]];
            if (row >= 0) atomicOr(&U[row], 1u << pos);
            atomicAdd(&cnt[pos], 1u);
          }
        }
      }
    }
    wave_sync();
    if (mine) {
      const uint32_t u = U[i0];
      c.t[bx + i0] = cnt[i0] + __popc(u);
      uint32_t four = 0;
      for (uint32_t b = u; b; b &= b - 1) four += __popc(u & U[__ffs(b) - 1]);
      k4 += four;
      key[slot] = -1;
    }
    wave_sync();
  }
  k4 = wave_sum_u64(k4);
  if (lane == 0 && k4) atomicAdd(&c.acc[kCensusK4], k4);
}

// Vertices per class, then their ids class by class, hubs first (the
// vertex's index from the top of the id range): one atomic per class per
// wave.
__device__ __forceinline__ int row_class(const int64_t *__restrict__ drp,
                                         const int32_t *__restrict__ deg,
                                         int64_t v, int32_t n) {
  if (v < 0 || v >= n) return -1;
  const int P = static_cast<int>(drp[v + 1] - drp[v]);
  if (P < 1) return -1;
  const int below = deg[v] - P;
  auto holds = [&](int k) {
    return P <= kRowClasses[k].max_out && below <= kRowClasses[k].max_below;
  };
  if (holds(kTinyClass)) return kTinyClass;
  int k = kSmallClass;
  while (!holds(k)) ++k;
  return k;
}

// 1024 vertices at a time, one atomic per class for all of them (one per
// wave took 0.4 ms on 4 million vertices).
constexpr int kClassT = 1024;

// The count of class q in this workgroup's vertices, and the vertices of the
// class before this thread's.
struct ClassAt {
  unsigned total, before;
};
__device__ __forceinline__ ClassAt class_at(int k, int q, unsigned *s_wave) {
  const u64 m = __ballot(k == q);
  if (lane64() == 0) s_wave[threadIdx.x >> 6] = __popcll(m);
  __syncthreads();
  ClassAt r{0u, static_cast<unsigned>(bits_below(m))};
  for (int w = 0; w < kClassT / 64; ++w) {
    if (w < static_cast<int>(threadIdx.x >> 6)) r.before += s_wave[w];
    r.total += s_wave[w];
  }
  __syncthreads();
  return r;
}

__global__ __launch_bounds__(kClassT) void rows_count(
    const int64_t *__restrict__ drp, const int32_t *__restrict__ deg,
    int32_t n, unsigned *__restrict__ count) {
  __shared__ unsigned s_wave[kClassT / 64];
  const int64_t v = int64_t(blockIdx.x) * kClassT + threadIdx.x;
  const int k = row_class(drp, deg, v, n);
  for (int q = 0; q < kRowClassCount; ++q) {
    const ClassAt c = class_at(k, q, s_wave);
    if (threadIdx.x == 0 && c.total) atomicAdd(&count[q], c.total);
  }
}

__global__ __launch_bounds__(kClassT) void rows_scatter(
    const int64_t *__restrict__ drp, const int32_t *__restrict__ deg,
    int32_t n, const unsigned *__restrict__ count, unsigned *__restrict__ fill,
    int32_t *__restrict__ list) {
  __shared__ unsigned s_wave[kClassT / 64];
  __shared__ unsigned s_base;
  const int64_t v =
      int64_t(n) - 1 - (int64_t(blockIdx.x) * kClassT + threadIdx.x);
  const int k = row_class(drp, deg, v, n);
  unsigned start = 0;
  for (int q = 0; q < kRowClassCount; ++q) {
    const ClassAt c = class_at(k, q, s_wave);
    if (threadIdx.x == 0) s_base = c.total ? atomicAdd(&fill[q], c.total) : 0u;
    __syncthreads();
    if (k == q) list[start + s_base + c.before] = static_cast<int32_t>(v);
    start += count[q];
  }
}

template <int T, int WU, bool CLIQUES>
int launch_class(const CensusArgs &c, const RowArgs &r, int grid,
                 size_t lds, hipStream_t s) {
  hipLaunchKernelGGL((census_rows<T, WU, CLIQUES>), dim3(grid), dim3(T), lds,
                     s, c, r);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

size_t rows_lds(int cls, bool cliques) {
  const RowClass &k = kRowClasses[cls];
  if (k.words == 0) return 0;
  return size_t(cliques ? k.words : k.words_u) * 8 + size_t(k.max_out) * 8;
}

int rows_threads(int cls) { return kRowClasses[cls].threads; }

// Workgroups of a class that a CU holds at once (LDS and waves).
int rows_per_cu(int cls, bool cliques) {
  const size_t lds = rows_lds(cls, cliques) + kWindowWords * 6 + 64;
  const int by_lds = static_cast<int>((size_t(160) << 10) / lds);
  const int by_waves = 32 / (rows_threads(cls) / 64);
  return std::max(1, std::min(by_lds, by_waves));
}

}  // namespace

int64_t rows_members(int cls, const int64_t *count, bool cliques) {
  if (cls > kTinyClass || !(cliques || count[kTinyClass] <= kTinyFew))
    return count[cls];
  return cls == kSmallClass ? count[kSmallClass] + count[kTinyClass] : 0;
}

// 64-bit words of rows in the slab of a vertex of P out-neighbours: U and,
// in the pass over cliques, the columns of L.
int64_t slab_words(int64_t P, bool cliques) {
  return P * ((P + 63) / 64 + (cliques ? kSlabL : 0));
}

size_t rows_slab_bytes(int cls, int64_t max_out, bool cliques) {
  const RowClass &k = kRowClasses[cls];
  const int64_t P = std::min<int64_t>(max_out, k.max_out);
  // The triangles and their counts: of the pass over cliques alone (P1 on
  // 900 vertices in a clique took 977 MB with them, 23 without).
  size_t b = cliques ? size_t(P) * size_t(P - 1) / 2 * 12 : 0;
  if (k.words == 0)
    b += size_t(slab_words(P, cliques)) * 8 + size_t(P) * 4 + 16;
  return (b + 255) & ~size_t(255);
}

// Vertices per queue access: one while that leaves no workgroup more than
// eight turns (RMAT-10 at eight each: 112 workgroups on 256 CUs).
int rows_grab(int cls, int64_t count, bool cliques, int cus) {
  const int64_t wgs = int64_t(cus) * rows_per_cu(cls, cliques);
  return static_cast<int>(
      std::max<int64_t>(1, std::min<int64_t>(kRowClasses[cls].grab,
                                             count / (8 * wgs))));
}

int rows_grid(int cls, int64_t max_out, int64_t count, bool cliques,
              size_t budget, int cus) {
  if (count <= 0) return 0;
  const RowClass &k = kRowClasses[cls];
  const int64_t grab = rows_grab(cls, count, cliques, cus);
  int64_t g = std::min<int64_t>((count + grab - 1) / grab,
                                int64_t(cus) * rows_per_cu(cls, cliques));
  if (cliques || k.words == 0) {
    const size_t per =
        std::max<size_t>(rows_slab_bytes(cls, max_out, cliques), 1);
    g = std::min<int64_t>(g, static_cast<int64_t>(budget / per));
  }
  return static_cast<int>(std::max<int64_t>(g, 1));
}

int census_rows_init() {
  const void *big[] = {
      reinterpret_cast<const void *>(&census_rows<1024, 11, false>),
      reinterpret_cast<const void *>(&census_rows<1024, 11, true>)};
  for (const void *k : big)
    if (hipFuncSetAttribute(
            k, hipFuncAttributeMaxDynamicSharedMemorySize,
            static_cast<int>(rows_lds(kRowClassCount - 2, true))) !=
        hipSuccess)
      return -1;
  return 0;
}

int census_rows_launch(const CensusArgs &c, const int64_t *cls_count,
                       int64_t max_out, bool cliques, char *slab,
                       size_t budget, int cus, hipStream_t s) {
  const int32_t *list = c.order;
  int64_t start[kRowClassCount];
  int64_t at = 0;
  for (int k = 0; k < kRowClassCount; ++k) {
    start[k] = at;
    at += cls_count[k];
  }
  for (int cls = kRowClassCount - 1; cls >= 0; --cls) {  // heaviest first
    const int64_t members = rows_members(cls, cls_count, cliques);
    const int grid = rows_grid(cls, max_out, members, cliques, budget, cus);
    if (grid == 0) continue;
    if (cls == kTinyClass) {
      const int64_t g = std::min<int64_t>(
          (members + kTinyWaves - 1) / kTinyWaves, int64_t(cus) * 8);
      hipLaunchKernelGGL(census_tiny, dim3(static_cast<unsigned>(g)),
                         dim3(kTinyWaves * 64), 0, s, c, list + start[cls],
                         static_cast<uint32_t>(members));
      if (hipGetLastError() != hipSuccess) return -1;
      continue;
    }
    const RowClass &k = kRowClasses[cls];
    RowArgs r;
    r.list = list + start[cls];
    r.count = static_cast<uint32_t>(members);
    r.cursor = c.cursor + (cliques ? 8 : 0) + cls;
    r.grab = rows_grab(cls, members, cliques, cus);
    r.slab = slab;
    r.slab_bytes = rows_slab_bytes(cls, max_out, cliques);
    const int64_t P = std::min<int64_t>(max_out, k.max_out);
    r.tri_cap = cliques ? static_cast<uint32_t>(P * (P - 1) / 2) : 0;
    r.pcap = static_cast<int>(P);
    r.words = k.words == 0 ? slab_words(P, cliques)
                           : (cliques ? k.words : k.words_u);
    const size_t lds = rows_lds(cls, cliques);
    int rc = 0;
    if (cls == kSmallClass)
      rc = cliques ? launch_class<256, 1, true>(c, r, grid, lds, s)
                   : launch_class<256, 1, false>(c, r, grid, lds, s);
    else if (cls == 2)
      rc = cliques ? launch_class<512, 4, true>(c, r, grid, lds, s)
                   : launch_class<512, 4, false>(c, r, grid, lds, s);
    else if (cls == 3)
      rc = cliques ? launch_class<1024, 11, true>(c, r, grid, lds, s)
                   : launch_class<1024, 11, false>(c, r, grid, lds, s);
    else
      rc = cliques ? launch_class<1024, 0, true>(c, r, grid, lds, s)
                   : launch_class<1024, 0, false>(c, r, grid, lds, s);
    if (rc) return rc;
  }
  return 0;
}

int census_rows_classify(const int64_t *drp, const int32_t *deg, int32_t n,
                         unsigned *count, unsigned *fill, int32_t *list,
                         hipStream_t s) {
  const int g = n / kClassT + 1;
  hipLaunchKernelGGL(rows_count, dim3(g), dim3(kClassT), 0, s, drp, deg, n,
                     count);
  hipLaunchKernelGGL(rows_scatter, dim3(g), dim3(kClassT), 0, s, drp, deg, n,
                     count, fill, list);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace mgpm

// Triangle count against hub bitmaps.
//
// On the graph relabelled in DAG order (rank = id) the hubs are the 65535
// highest ids, and the DAG's lists lead into them: on RMAT-22 99.4% of the
// items that can close a triangle are hubs.  Every triangle a < b < z with a
// hub z is counted at its owner b: z lies in N+(a) past b and in N+(b), so
// for every a below b adjacent to it the part of a's row past b is tested
// against N+(b).
//   * Rows hold hub numbers n - 1 - z in 16 bits, ascending: the part past
//     b is a prefix, so the lists of every owner start on the rows' 16-byte
//     boundaries.  Whole chunks of eight are read; what a chunk holds past
//     the prefix has numbers of b or below, which N+(b) cannot hold, so no
//     item needs a guard.
//   * N+(b) is a bitmap of all hub numbers, 8 KB of LDS per wave: a test is
//     one LDS read and about five vector instructions, against 45 for a hash
//     probe of the table kernels (tc_kernels.hip).  Only the bits set are
//     cleared again.
//   * Eight lanes walk one partner (64 items a step; a list of RMAT-22 takes
//     2.3 steps), each group on its own, with three chunks per lane in flight
//     and the partners' records 64 at a time, a batch ahead.
//   * The partners of all owners lie in one array; a wave takes blocks of
//     it, whatever owners they hold, so hubs with 10^5 partners and vertices
//     with two need no task lists.  Most owners are small: the loads of the
//     next two run ahead of the one being counted.
// Triangles without a hub (both lists short) are found by binary search
// (hub_rest).
//
// Measured on one MI355X, per count: RMAT-22 (16 draws per vertex) 15.8 ms
// with hash tables on laid-out lists -> 3.6 ms (hub_count 3.0, hub_rest
// 0.69), with 0.8 GB of plan beside the census graph's 1.9 GB instead of 48
// GB of lists; RMAT-16 708 -> 67 us.  What bounds it: the rows come from the
// last-level cache (20 GB per count on RMAT-22 at 6.5 TB/s: the L2 catches a
// sixth; the plan names 15.4 GB of records and chunks), 73 vector instructions
// and eight LDS reads per step of 512 items behind that.
#include <hip/hip_runtime.h>

#include <hipcub/device/device_scan.hpp>

#include <algorithm>

#include "lanes.hpp"
#include "tc_hub.hpp"
#include "wave.hpp"

namespace mgpm {

namespace {

typedef unsigned long long u64;

constexpr int kWaves = 4;
constexpr int kWords = (kHubIds + 1) / 32;  // bitmap words
constexpr int kLanes = 8;                   // lanes per partner
constexpr int kGroups = 64 / kLanes;
constexpr uint32_t kPad = 0xffffu;
constexpr u64 kOwnerCost = 16;  // steps of a group that an owner's bitmap costs

// Hits of one 32-bit word, two hub numbers.
__device__ __forceinline__ uint32_t test2(const uint32_t *bits, uint32_t w) {
  const uint32_t lo = bits[(w & 0xffffu) >> 5], hi = bits[w >> 21];
  return __builtin_amdgcn_ubfe(lo, w, 1) +
         __builtin_amdgcn_ubfe(hi, w >> 16, 1);
}

template <class F>
__device__ __forceinline__ void each_id(const uint4 &v, const F &f) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    f(w[k] & 0xffffu);
    f(w[k] >> 16);
  }
}

// One owner's share of a block: its partners [q0, q1) and its row.
struct Share {
  uint32_t q0, q1, base, chunks;
};

// What a wave has loaded for a share before it is counted.
struct Loaded {
  HubPartner rec;  // partner q0 + lane
  uint4 own;       // this lane's chunk of the owner's row
  uint4 v;         // this lane's chunk of partner q0 + its group
};

// What a group of lanes walks: chunk c of a partner, of which `chunks` from
// `base` can hold hits (none: the group is idle).
struct Walk {
  uint32_t base, chunks, c;
};

// Adds a workgroup's sum to the launch's total.  Atomics on one address take
// 11 ns each, so the workgroups of a queue meet on its cache line first, and
// the last of each queue adds that line's sum to the total; the last of
// those moves the total to the host address and leaves every counter zero
// for the next launch.  Each atomic's value is waited for before the next
// one, which orders them without a fence (a fence writes the L2 back: 0.04
// ms for a launch).
__device__ __forceinline__ void finish(u64 acc, const HubOut &out, u64 *red) {
  acc = wave_sum_u64(acc);
  __syncthreads();  // red is the bitmaps' memory
  if (lane64() == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x != 0) return;
  acc = 0;
  for (int k = 0; k < kWaves; ++k) acc += red[k];
  if (!out.host) {
    if (acc) atomicAdd(out.result, acc);
    return;
  }
  const unsigned q = blockIdx.x % kHubQueues;
  unsigned *line = out.queue + q * kHubQueueStride;
  u64 *sum = reinterpret_cast<u64 *>(line + 2);
  u64 old = atomicAdd(sum, acc);
  asm volatile("" ::"v"(old));
  const unsigned mine = (gridDim.x - q + kHubQueues - 1) / kHubQueues;
  if (atomicAdd(line + 4, 1u) != mine - 1u) return;
  old = atomicAdd(out.result, atomicExch(sum, u64(0)));
  asm volatile("" ::"v"(old));
  line[0] = 0;
  line[4] = 0;
  unsigned *queues = out.queue + kHubQueueWords - 1;
  if (atomicAdd(queues, 1u) != kHubQueues - 1u) return;
  *queues = 0;
  const u64 total = atomicExch(out.result, u64(0));
  __hip_atomic_store(out.host, total, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ __launch_bounds__(kWaves * 64, 5) void hub_count(TcHubPlan p,
                                                         HubOut out) {
  __shared__ uint32_t s_bits[kWaves][kWords];
  const int lane = lane64();
  uint32_t *bits = s_bits[threadIdx.x >> 6];
  const uint4 *rows = static_cast<const uint4 *>(p.rows);
  const uint32_t gl = static_cast<uint32_t>(lane & (kLanes - 1));
  const uint32_t grp = static_cast<uint32_t>(lane / kLanes);
  const int words = min(kWords, static_cast<int>(p.n / 32u + 1u));
  for (int i = lane; i < words; i += 64) bits[i] = 0;
  if (lane == 0) bits[kWords - 1] = 0;  // the padding's word
  wave_sync();
  u64 acc = 0;
  // Blocks of about equal cost in turn, or, where a wave gets five or more,
  // from one of eight queues (queue q holds blocks q, q + 8, ...; an atomic
  // on one address takes 11 ns), the next one taken before this one is
  // counted.  RMAT-22 3.9 ms from queues, 4.9 in turn; RMAT-16 (2.8 blocks
  // per wave) 77 and 66 us.  Batches have no queues.
  const uint32_t wave = blockIdx.x * kWaves + (threadIdx.x >> 6);
  const uint32_t q = blockIdx.x % kHubQueues;
  unsigned *queue = out.queue && p.blocks > 4u * gridDim.x * kWaves
                        ? out.queue + q * kHubQueueStride
                        : nullptr;
  uint32_t ahead = 0;  // lane 0: the next block's place in its queue
  if (queue && lane == 0) ahead = atomicAdd(queue, 1u);
  uint32_t turn = wave;
  for (;;) {
    uint32_t g;
    if (queue) {
      g = wave_first(ahead) * kHubQueues + q;
      if (g < p.blocks && lane == 0) ahead = atomicAdd(queue, 1u);
    } else {
      g = turn;
      turn += gridDim.x * kWaves;
    }
    if (g >= p.blocks) break;
    uint32_t at = wave_first(p.bound[g]);
    const uint32_t stop = wave_first(p.bound[g + 1]);
    if (at >= stop) continue;
    // 64 owners at a time, one per lane.
    uint32_t k0 = wave_first(p.start[g]);
    HubOwner own;
    auto owners = [&]() {
      own = p.owner[min(k0 + static_cast<uint32_t>(lane), p.owners - 1u)];
    };
    owners();
    auto lane_of = [&](uint32_t x, int k) {
      return static_cast<uint32_t>(
          __builtin_amdgcn_readlane(static_cast<int>(x), k));
    };
    auto take = [&](Share &s) -> bool {
      while (at < stop && k0 < p.owners) {
        const u64 m = __ballot(own.end > at);
        if (!m) {
          k0 += 64;
          owners();
          continue;
        }
        const int k = __builtin_ctzll(m);
        s.q0 = max(at, lane_of(own.beg, k));
        s.q1 = min(lane_of(own.end, k), stop);
        s.base = lane_of(own.base, k);
        s.chunks = lane_of(own.chunks, k);
        at = max(s.q1, at);
        if (s.q0 >= stop) return false;
        return true;
      }
      return false;
    };
    auto load = [&](const Share &s, Loaded &l) {
      l.rec = p.part[min(s.q0 + static_cast<uint32_t>(lane), s.q1 - 1u)];
      l.own = rows[static_cast<uint32_t>(lane) < s.chunks ? s.base + lane : 0u];
    };
    auto pick = [&](const HubPartner &rec, uint32_t i, uint32_t cnt) {
      Walk w;
      const int from = static_cast<int>(min(i, 63u));
      w.base = __shfl(rec.base, from, 64);
      w.chunks = __shfl(rec.chunks, from, 64);
      if (i >= cnt) w.chunks = 0;
      w.c = gl;
      return w;
    };
    auto fetch = [&](const Walk &w) {
      return rows[w.c < w.chunks ? w.base + w.c : 0u];
    };
    auto load_items = [&](const Share &s, Loaded &l) {
      l.v = fetch(pick(l.rec, grp, min(s.q1 - s.q0, 64u)));
    };
    // Two shares ahead: records and owner rows; one ahead: first chunks.
    Share s0, s1, s2;
    Loaded l0, l1, l2;
    bool h0 = take(s0);
    if (!h0) continue;
    load(s0, l0);
    bool h1 = take(s1);
    if (h1) load(s1, l1);
    load_items(s0, l0);
    while (h0) {
      const bool h2 = h1 && take(s2);
      if (h1) load_items(s1, l1);
      if (h2) load(s2, l2);
      each_id(l0.own, [&](uint32_t id) {
        if (id != kPad) atomicOr(&bits[id >> 5], 1u << (id & 31u));
      });
      for (uint32_t r = lane + 64u; r < s0.chunks; r += 64u)
        each_id(rows[s0.base + r], [&](uint32_t id) {
          if (id != kPad) atomicOr(&bits[id >> 5], 1u << (id & 31u));
        });
      wave_sync();
      uint32_t hits = 0;
      HubPartner rec = l0.rec;
      uint4 v0 = l0.v;
      for (uint32_t qb = s0.q0;;) {
        // 64 partners at a time, their records one per lane; a group that
        // is done with its partner takes the next one.  Three chunks per
        // lane are in flight: every load is issued (idle lanes read the
        // padding), as a load on one branch only would make the compiler
        // wait for all of them at the join.
        const uint32_t cnt = min(s0.q1 - qb, 64u);
        const HubPartner ahead_rec =
            p.part[min(qb + 64u + static_cast<uint32_t>(lane), s0.q1 - 1u)];
        Walk w = pick(rec, grp, cnt);
        uint32_t taken = kGroups;
        // Partners without a chunk leave a group idle for a step.
        auto alive = [&]() { return taken < cnt || __any(w.chunks != 0); };
        auto step = [&]() {
          w.c += kLanes;
          const bool done = w.c - gl >= w.chunks;
          const u64 m = __ballot(done);
          if (m) {
            const uint32_t i =
                taken + static_cast<uint32_t>(
                            __popcll(m & ((u64(1) << (lane & ~(kLanes - 1))) -
                                          u64(1)))) / kLanes;
            const Walk n = pick(rec, i, cnt);
            if (done) w = n;
            taken += static_cast<uint32_t>(__popcll(m)) / kLanes;
          }
        };
        auto test = [&](const uint4 &v) {
          hits += test2(bits, v.x) + test2(bits, v.y) + test2(bits, v.z) +
                  test2(bits, v.w);
        };
        step();
        bool f0, f1 = alive();
        uint4 v1 = fetch(w);
        step();
        bool f2 = f1 && alive();
        uint4 v2 = fetch(w);
        for (;;) {
          test(v0);
          step();
          f0 = f2 && alive();
          v0 = fetch(w);
          if (!f1) break;
          test(v1);
          step();
          f1 = f0 && alive();
          v1 = fetch(w);
          if (!f2) break;
          test(v2);
          step();
          f2 = f1 && alive();
          v2 = fetch(w);
          if (!f0) break;
        }
        qb += 64u;
        if (qb >= s0.q1) break;
        rec = ahead_rec;
        v0 = fetch(pick(rec, grp, min(s0.q1 - qb, 64u)));
      }
      acc += hits;
      wave_sync();
      each_id(l0.own, [&](uint32_t id) {
        if (id != kPad) bits[id >> 5] = 0;
      });
      for (uint32_t r = lane + 64u; r < s0.chunks; r += 64u)
        each_id(rows[s0.base + r], [&](uint32_t id) {
          if (id != kPad) bits[id >> 5] = 0;
        });
      wave_sync();
      s0 = s1;
      l0 = l1;
      s1 = s2;
      l1 = l2;
      h0 = h1;
      h1 = h2;
    }
  }
  finish(acc, out, reinterpret_cast<u64 *>(s_bits));
}

// Triangles below the hubs: the pairs of heads b < z of a vertex a below the
// hubs, z searched in b's heads below them.  16 lanes per vertex, four pairs
// per lane whose searches run in lockstep (their loads overlap: a search is
// a chain of about eight loads, and the chains are what the pass takes; one
// pair per lane took 0.95 ms on RMAT-22, 4.2e7 pairs).
constexpr int kPairs = 4;

__global__ __launch_bounds__(kWaves * 64) void hub_rest(TcHubPlan p,
                                                        u64 *result) {
  __shared__ u64 s_sum[kWaves];
  constexpr uint32_t kL = 16;
  const uint32_t gl = threadIdx.x & (kL - 1);
  const uint32_t groups = gridDim.x * (kWaves * 64 / kL);
  u64 acc = 0;
  for (uint32_t at = (blockIdx.x * kWaves * 64 + threadIdx.x) / kL;
       at < p.nrest; at += groups) {
    const int32_t a = p.rest[at];
    const int32_t *N = p.dcol + p.drp[a];
    // Out-degrees are at most 65535 (below 2^31 arcs).
    const uint32_t s = p.split[a] - static_cast<uint32_t>(p.drp[a]);
    for (uint32_t q0 = gl; q0 < s * s; q0 += kL * kPairs) {
      uint32_t lo[kPairs], len[kPairs], most = 1;
      int32_t z[kPairs];
      bool ok[kPairs];
#pragma unroll
      for (int k = 0; k < kPairs; ++k) {
        const uint32_t q = q0 + kL * k;
        const uint32_t i = q / s, j = q - i * s;
        ok[k] = q < s * s && j > i;
        const int32_t b = N[ok[k] ? i : 0];
        z[k] = N[ok[k] ? j : 0];
        const uint32_t lb = static_cast<uint32_t>(p.drp[b]);
        ok[k] = ok[k] && p.split[b] > lb;
        const Window w = search_window(lb, p.split[b], ok[k]);
        lo[k] = w.lo;
        len[k] = w.len;
        most = max(most, len[k]);
      }
      // The last element <= z of each list, every window halving until it
      // is one element.
      for (; most > 1; most -= most >> 1) {
        int32_t v[kPairs];
#pragma unroll
        for (int k = 0; k < kPairs; ++k) v[k] = p.dcol[lo[k] + (len[k] >> 1)];
#pragma unroll
        for (int k = 0; k < kPairs; ++k) {
          if (v[k] <= z[k]) lo[k] += len[k] >> 1;
          len[k] -= len[k] >> 1;
        }
      }
#pragma unroll
      for (int k = 0; k < kPairs; ++k)
        acc += ok[k] && p.dcol[lo[k]] == z[k] ? 1 : 0;
    }
  }
  acc = wave_sum_u64(acc);
  if (lane64() == 0) s_sum[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < kWaves; ++k) acc += s_sum[k];
    if (acc) atomicAdd(result, acc);
  }
}

__global__ void hub_counts(const int64_t *__restrict__ drp,
                           const int32_t *__restrict__ dcol, int32_t n,
                           int32_t hublo, uint32_t *__restrict__ split,
                           uint32_t *__restrict__ chunks) {
  for (int64_t v = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; v <= n;
       v += int64_t(gridDim.x) * blockDim.x) {
    if (v == n) {
      chunks[v] = 0;
      continue;
    }
    int64_t lo = drp[v], hi = drp[v + 1];
    const int64_t e = hi;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (dcol[mid] < hublo) lo = mid + 1;
      else hi = mid;
    }
    split[v] = static_cast<uint32_t>(lo);
    // Chunk 0 of the array is padding: row 0 starts at chunk 1.
    chunks[v] = static_cast<uint32_t>((e - lo + kHubChunk - 1) / kHubChunk) +
                (v == 0 ? 1u : 0u);
  }
}

// Rows: the hubs of N+(v), last first, padded; one wave per row.
__global__ void hub_rows(const int64_t *__restrict__ drp,
                         const int32_t *__restrict__ dcol, int32_t n,
                         const uint32_t *__restrict__ split,
                         uint32_t *__restrict__ rowbase,
                         uint16_t *__restrict__ rows) {
  const int lane = lane64();
  const int64_t nw = (int64_t(gridDim.x) * blockDim.x) >> 6;
  const int64_t w0 = (int64_t(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
  if (w0 == 0 && lane < kHubChunk) rows[lane] = static_cast<uint16_t>(kPad);
  for (int64_t v = w0; v < n; v += nw) {
    // The scan put row 0 at chunk 0; its padding chunk comes first.
    const uint32_t b = rowbase[v] + (v == 0 ? 1u : 0u);
    const int64_t s = split[v], e = drp[v + 1];
    const int64_t len = e - s;
    const int64_t padded = (len + kHubChunk - 1) / kHubChunk * kHubChunk;
    for (int64_t i = lane; i < padded; i += 64)
      rows[int64_t(b) * kHubChunk + i] = static_cast<uint16_t>(
          i < len ? static_cast<uint32_t>(n - 1 - dcol[e - 1 - i]) : kPad);
  }
}

__global__ void hub_first_row(uint32_t *rowbase) { rowbase[0] = 1; }

// Owners: vertices with partners (CSR entries below them; the partners of b
// start at rowptr[b] - drp[b]) and a row.  Flags for a scan, then the list
// in id order.  Vertices without either are left out: they are most of a
// sparse graph's, and skipping them one 64 at a time made single blocks last
// as long as the rest of the launch.
__device__ __forceinline__ HubOwner owner_of(
    const int64_t *__restrict__ rowptr, const int64_t *__restrict__ drp,
    const uint32_t *__restrict__ rowbase, int64_t b) {
  HubOwner o;
  o.beg = static_cast<uint32_t>(rowptr[b] - drp[b]);
  o.end = static_cast<uint32_t>(rowptr[b + 1] - drp[b + 1]);
  o.base = rowbase[b];
  o.chunks = rowbase[b + 1] - o.base;
  return o;
}

__global__ void hub_owner_flags(const int64_t *__restrict__ rowptr,
                                const int64_t *__restrict__ drp,
                                const uint32_t *__restrict__ rowbase,
                                int32_t n, uint32_t *__restrict__ flag) {
  for (int64_t b = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; b <= n;
       b += int64_t(gridDim.x) * blockDim.x) {
    uint32_t f = 0;
    if (b < n) {
      const HubOwner o = owner_of(rowptr, drp, rowbase, b);
      f = o.end > o.beg && o.chunks > 0 ? 1u : 0u;
    }
    flag[b] = f;
  }
}

__global__ void hub_owner_list(const int64_t *__restrict__ rowptr,
                               const int64_t *__restrict__ drp,
                               const uint32_t *__restrict__ rowbase,
                               int32_t n, const uint32_t *__restrict__ pos,
                               HubOwner *__restrict__ owner) {
  for (int64_t b = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; b < n;
       b += int64_t(gridDim.x) * blockDim.x)
    if (pos[b + 1] > pos[b])
      owner[pos[b]] = owner_of(rowptr, drp, rowbase, b);
}

// What a partner record needs of its row's vertex, in one 16-byte load.
__global__ void hub_meta(const int64_t *__restrict__ drp, int32_t n,
                         const uint32_t *__restrict__ split,
                         const uint32_t *__restrict__ rowbase,
                         uint4 *__restrict__ meta) {
  for (int64_t v = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; v < n;
       v += int64_t(gridDim.x) * blockDim.x) {
    const uint32_t e = static_cast<uint32_t>(drp[v + 1]);
    meta[v] = make_uint4(e, e - split[v], rowbase[v], 0u);
  }
}

// One partner per CSR entry a below its row's vertex b: the chunks of a's
// row that hold hubs past b (the heads past b are the last ones of N+(a)).
__global__ void hub_partners(const int32_t *__restrict__ col,
                             const int32_t *__restrict__ src, int64_t nnz,
                             const int64_t *__restrict__ drp,
                             const uint32_t *__restrict__ arc,
                             const uint4 *__restrict__ meta,
                             HubPartner *__restrict__ part) {
  for (int64_t j = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; j < nnz;
       j += int64_t(gridDim.x) * blockDim.x) {
    const int32_t b = src[j], a = col[j];
    if (a > b) continue;
    const uint4 r = meta[a];  // end of N+(a), its hubs, its row
    const uint32_t past = r.x - 1u - arc[j];
    HubPartner h;
    h.base = r.z;
    h.chunks = (min(past, r.y) + kHubChunk - 1) / kHubChunk;
    part[j - drp[b]] = h;
  }
}

// Adds a workgroup's sum to one of the kHubSums places.
__device__ __forceinline__ void add_sum(u64 x, u64 *__restrict__ sums) {
  __shared__ u64 s_sum;
  if (threadIdx.x == 0) s_sum = 0;
  __syncthreads();
  x = wave_sum_u64(x);
  if (lane64() == 0) atomicAdd(&s_sum, x);
  __syncthreads();
  if (threadIdx.x == 0 && s_sum)
    atomicAdd(&sums[blockIdx.x % kHubSums * kHubSumStride], s_sum);
}

// Cost of every run of kHubRun partners, in steps of one group of lanes,
// with kOwnerCost more where an owner with a row begins (hub_owner_costs).
// Both also add up the chunks that a count reads.
__global__ void hub_costs(const HubPartner *__restrict__ part,
                          uint32_t nparts, uint32_t runs,
                          u64 *__restrict__ cost, u64 *__restrict__ sums) {
  static_assert(kHubRun == 16, "a run per 16 lanes");
  u64 chunks = 0;
  const uint32_t gl = threadIdx.x % kHubRun;
  for (uint32_t r = (blockIdx.x * blockDim.x + threadIdx.x) / kHubRun;
       r <= runs; r += gridDim.x * blockDim.x / kHubRun) {
    const uint32_t i = r * kHubRun + gl;
    int c = 0;
    if (r < runs && i < nparts) {
      const uint32_t k = part[i].chunks;
      chunks += k;
      c = static_cast<int>(max(1u, (k + kLanes - 1u) / kLanes));
    }
#pragma unroll
    for (int d = 8; d >= 1; d >>= 1) c += __shfl_xor(c, d, 16);
    if (gl == 0) cost[r] = static_cast<u64>(c);
  }
  add_sum(chunks, sums);
}

__global__ void hub_owner_costs(const HubOwner *__restrict__ owner,
                                const uint32_t *__restrict__ owners,
                                u64 *__restrict__ cost,
                                u64 *__restrict__ sums) {
  u64 chunks = 0;
  for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < *owners;
       k += gridDim.x * blockDim.x) {
    const HubOwner o = owner[k];
    chunks += o.chunks;
    atomicAdd(&cost[o.beg / kHubRun], kOwnerCost);
  }
  add_sum(chunks, sums + 1);
}

// Block g holds the runs whose cost prefix starts in [g, g + 1) / blocks of
// the total.
__global__ void hub_blocks(const u64 *__restrict__ prefix, uint32_t runs,
                           const HubOwner *__restrict__ owner,
                           const uint32_t *__restrict__ owners,
                           uint32_t nparts, uint32_t blocks,
                           uint32_t *__restrict__ bound,
                           uint32_t *__restrict__ start) {
  const u64 total = prefix[runs];
  for (uint32_t g = blockIdx.x * blockDim.x + threadIdx.x; g <= blocks;
       g += gridDim.x * blockDim.x) {
    const u64 want = total / blocks * g + total % blocks * g / blocks;
    uint32_t a = 0, b = runs;  // first run with prefix >= want
    while (a < b) {
      const uint32_t mid = a + (b - a) / 2;
      if (prefix[mid] < want) a = mid + 1;
      else b = mid;
    }
    const uint32_t at = g == blocks ? nparts : min(a * kHubRun, nparts);
    bound[g] = at;
    if (g == blocks) continue;
    uint32_t lo = 0, hi = *owners;  // first owner with end > at
    while (lo < hi) {
      const uint32_t mid = lo + (hi - lo) / 2;
      if (owner[mid].end <= at) lo = mid + 1;
      else hi = mid;
    }
    start[g] = lo;
  }
}

// Vertices with two or more heads below the hubs, one atomic per 1024.
constexpr int kRestT = 1024;
__global__ __launch_bounds__(kRestT) void hub_rest_list(
    const int64_t *__restrict__ drp, const uint32_t *__restrict__ split,
    int32_t n, int32_t *__restrict__ rest, uint32_t *__restrict__ nrest) {
  __shared__ uint32_t s_wave[kRestT / 64];
  __shared__ uint32_t s_base;
  const int64_t v = int64_t(blockIdx.x) * kRestT + threadIdx.x;
  const bool in = v < n && static_cast<int64_t>(split[v]) - drp[v] >= 2;
  const u64 m = __ballot(in);
  if (lane64() == 0) s_wave[threadIdx.x >> 6] = __popcll(m);
  __syncthreads();
  uint32_t before = bits_below(m), total = 0;
  for (int w = 0; w < kRestT / 64; ++w) {
    if (w < static_cast<int>(threadIdx.x >> 6)) before += s_wave[w];
    total += s_wave[w];
  }
  if (threadIdx.x == 0) s_base = total ? atomicAdd(nrest, total) : 0u;
  __syncthreads();
  if (in) rest[s_base + before] = static_cast<int32_t>(v);
}

int flat(int64_t items, int most) {
  return static_cast<int>(
      std::max<int64_t>(1, std::min<int64_t>((items + 255) / 256, most)));
}

}  // namespace

int tc_hub_launch(const TcHubPlan &p, const HubOut &out, int cus,
                  hipStream_t s) {
  if (p.nrest) {
    const int64_t g = std::min<int64_t>((int64_t(p.nrest) + 15) / 16,
                                        int64_t(cus) * 8);
    hipLaunchKernelGGL(hub_rest, dim3(static_cast<unsigned>(g)),
                       dim3(kWaves * 64), 0, s, p, out.result);
  }
  // Last: it reports the total.  Five workgroups per CU by LDS (32 KB each),
  // and at least one per queue.
  const int64_t g = std::max<int64_t>(
      kHubQueues, std::min<int64_t>((int64_t(p.blocks) + kWaves - 1) / kWaves,
                           int64_t(cus) * 5));
  hipLaunchKernelGGL(hub_count, dim3(static_cast<unsigned>(g)),
                     dim3(kWaves * 64), 0, s, p, out);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int tc_hub_counts(const int64_t *drp, const int32_t *dcol, int32_t n,
                  int32_t hublo, uint32_t *split, uint32_t *chunks,
                  hipStream_t s) {
  hipLaunchKernelGGL(hub_counts, dim3(flat(int64_t(n) + 1, 4096)), dim3(256),
                     0, s, drp, dcol, n, hublo, split, chunks);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

size_t tc_hub_scan_bytes(int32_t n, uint32_t runs) {
  size_t a = 0, b = 0;
  if (hipcub::DeviceScan::ExclusiveSum(
          nullptr, a, static_cast<const uint32_t *>(nullptr),
          static_cast<uint32_t *>(nullptr), int64_t(n) + 1) != hipSuccess ||
      hipcub::DeviceScan::ExclusiveSum(
          nullptr, b, static_cast<const u64 *>(nullptr),
          static_cast<u64 *>(nullptr), int64_t(runs) + 1) != hipSuccess)
    return 0;
  return std::max<size_t>({a, b, 1});
}

int tc_hub_scan(const uint32_t *chunks, uint32_t *rowbase, int32_t n,
                void *tmp, size_t bytes, hipStream_t s) {
  return hipcub::DeviceScan::ExclusiveSum(tmp, bytes, chunks, rowbase,
                                          int64_t(n) + 1, s) == hipSuccess
             ? 0
             : -1;
}

int tc_hub_blocks(const TcHubPlan &p, const uint32_t *owners, uint32_t runs,
                  unsigned long long *cost, unsigned long long *prefix,
                  void *tmp, size_t bytes, uint32_t *bound, uint32_t *start,
                  unsigned long long *sums, hipStream_t s) {
  hipLaunchKernelGGL(hub_costs, dim3(flat((int64_t(runs) + 1) * kHubRun,
                                          8192)),
                     dim3(256), 0, s, p.part, p.nparts, runs, cost, sums);
  hipLaunchKernelGGL(hub_owner_costs, dim3(flat(p.n, 4096)), dim3(256), 0, s,
                     p.owner, owners, cost, sums);
  if (hipcub::DeviceScan::ExclusiveSum(tmp, bytes, cost, prefix,
                                       int64_t(runs) + 1, s) != hipSuccess)
    return -1;
  hipLaunchKernelGGL(hub_blocks, dim3(flat(int64_t(p.blocks) + 1, 4096)),
                     dim3(256), 0, s, prefix, runs, p.owner, owners,
                     p.nparts, p.blocks, bound, start);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int tc_hub_fill(const int64_t *rowptr, const int32_t *col,
                const int32_t *src, int64_t nnz, const int64_t *drp,
                const int32_t *dcol, const uint32_t *arc, int32_t n,
                const uint32_t *split, uint32_t *rowbase, void *rows,
                uint32_t *flag, uint32_t *pos, void *meta, HubOwner *owner,
                HubPartner *part, int32_t *rest, uint32_t *nrest, void *tmp,
                size_t bytes, int cus, hipStream_t s) {
  hipLaunchKernelGGL(hub_rows, dim3(flat(int64_t(n) * 64, cus * 32)),
                     dim3(256), 0, s, drp, dcol, n, split, rowbase,
                     static_cast<uint16_t *>(rows));
  hipLaunchKernelGGL(hub_first_row, dim3(1), dim3(1), 0, s, rowbase);
  hipLaunchKernelGGL(hub_owner_flags, dim3(flat(int64_t(n) + 1, 4096)),
                     dim3(256), 0, s, rowptr, drp, rowbase, n, flag);
  if (tc_hub_scan(flag, pos, n, tmp, bytes, s)) return -1;
  hipLaunchKernelGGL(hub_owner_list, dim3(flat(n, 4096)), dim3(256), 0, s,
                     rowptr, drp, rowbase, n, pos, owner);
  hipLaunchKernelGGL(hub_meta, dim3(flat(n, 4096)), dim3(256), 0, s, drp, n,
                     split, rowbase, static_cast<uint4 *>(meta));
  hipLaunchKernelGGL(hub_partners, dim3(flat(nnz, cus * 32)), dim3(256), 0, s,
                     col, src, nnz, drp, arc,
                     static_cast<const uint4 *>(meta), part);
  hipLaunchKernelGGL(hub_rest_list, dim3(n / kRestT + 1), dim3(kRestT), 0, s,
                     drp, split, n, rest, nrest);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace mgpm

// Sums over vertices and edges of the census graph, and its 4-cycles: with
// the triangle, 4- and 5-clique counts of census_rows.hip, the terms from
// which P1, P4, P7 and P8 follow in closed form.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "census.hpp"
#include "choose.hpp"
#include "wave.hpp"

namespace mgpm {

namespace {

// Sums over vertices (C(d,3)) and over DAG arcs (t, t (d_x + d_y - 4) in
// two halves, C(t,2), C(t,3) and (d_x - t - 1)(d_y - t - 1)).
// With full5 also C(d,4), the fork, bull and diamond-pendant sums per edge,
// and twice the triangles per vertex into tv.
__global__ void census_sums(CensusArgs c) {
  unsigned long long s3 = 0, s2 = 0, sp = 0, st = 0, s4 = 0, fk = 0, dp3 = 0,
                     s1 = 0, tlo = 0, thi = 0, bdeg = 0;
  for (int64_t v = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; v < c.n;
       v += int64_t(gridDim.x) * blockDim.x) {
    const unsigned long long d = static_cast<unsigned long long>(c.deg[v]);
    s3 += choose3(d);
    if (c.full5) s4 += choose4(d);
    unsigned long long tsum = 0;
    for (int64_t a = c.drp[v]; a < c.drp[v + 1]; ++a) {
      const unsigned long long t = c.t[a];
      const int32_t y = c.dcol[a];
      const unsigned long long dy = static_cast<unsigned long long>(c.deg[y]);
      // t > 0 only when both degrees are >= 2.
      const unsigned long long td = t * (d + dy - 4);
      s1 += t;
      tlo += td & 0xffffffffull;
      thi += td >> 32;
      s2 += choose2(t);
      st += choose3(t);
      sp += (d - t - 1) * (dy - t - 1);
      if (c.full5) {
        // d, dy >= 1; t > 0 only when both are >= 2, so t (d - 2) is 0
        // whenever d - 2 would wrap.
        fk += choose2(d - 1) * (dy - 1) - t * (d - 2) +
              choose2(dy - 1) * (d - 1) - t * (dy - 2);
        dp3 += choose2(t) * (d + dy - 6);
        bdeg += t * (d - 2) * (dy - 2);
        tsum += t;
        if (t) atomicAdd(&c.tv[y], t);
      }
    }
    if (c.full5 && tsum) atomicAdd(&c.tv[v], tsum);
  }
  s3 = wave_sum_u64(s3);
  s2 = wave_sum_u64(s2);
  sp = wave_sum_u64(sp);
  st = wave_sum_u64(st);
  s4 = wave_sum_u64(s4);
  fk = wave_sum_u64(fk);
  dp3 = wave_sum_u64(dp3);
  s1 = wave_sum_u64(s1);
  tlo = wave_sum_u64(tlo);
  thi = wave_sum_u64(thi);
  bdeg = wave_sum_u64(bdeg);
  if (lane64() == 0) {
    if (s1) atomicAdd(&c.acc[kCensusTriangles], s1);
    if (tlo) atomicAdd(&c.acc[kCensusTriDegrees], tlo);
    if (thi) atomicAdd(&c.acc[kCensusTriDegreesHi], thi);
    if (bdeg) atomicAdd(&c.acc[kCensusBullDeg], bdeg);
    if (s3) atomicAdd(&c.acc[kCensusDeg3], s3);
    if (s2) atomicAdd(&c.acc[kCensusEdgePairs], s2);
    if (sp) atomicAdd(&c.acc[kCensusPathPairs], sp);
    if (st) atomicAdd(&c.acc[kCensusEdgeTriples], st);
    if (s4) atomicAdd(&c.acc[kCensusDeg4], s4);
    if (fk) atomicAdd(&c.acc[kCensusFork], fk);
    if (dp3) atomicAdd(&c.acc[kCensusDp3], dp3);
  }
}

// 4-cycles as subgraphs, each counted once at its highest-ranked vertex v
// (rank: degree, then id -- the DAG order): for every neighbour u of v
// ranked below v and every neighbour w of u ranked below v, count the
// wedge v-u-w at w; a cycle v-u-w-u' is one pair of wedges at w, so v adds
// sum_w C(wedges(w), 2).  One workgroup per v (vertices handed out by an
// atomic cursor), with its own dense counter array over all vertices
// (left zeroed) and the list of the w it touched.
constexpr int kC4Threads = 256;

__global__ __launch_bounds__(kC4Threads) void census_c4(CensusArgs c) {
  uint32_t *cnt = c.wedges + size_t(blockIdx.x) * size_t(c.n);
  int32_t *touched = c.touched + size_t(blockIdx.x) * size_t(c.n);
  __shared__ unsigned s_v, s_nt;
  __shared__ unsigned long long s_acc[kC4Threads / 64],
      s_ban[kC4Threads / 64], s_tq[kC4Threads / 64];
  const int lane = lane64(), wv = threadIdx.x >> 6;
  constexpr int nwv = kC4Threads / 64;
  unsigned long long acc = 0, ban = 0, tq = 0;
  for (;;) {
    if (threadIdx.x == 0) {
      s_v = atomicAdd(c.cursor + 1, 1u);
      s_nt = 0;
    }
    __syncthreads();
    const unsigned v = s_v;
    if (v >= static_cast<unsigned>(c.n)) break;
    // u below v: the first d(v) - d+(v) entries of v's sorted row; w below
    // v: the entries of u's row before v (the graph is relabelled in DAG
    // order, so rank is id).
    const int64_t ev = c.rowptr[v + 1] - (c.drp[v + 1] - c.drp[v]);
    for (int64_t i = c.rowptr[v] + wv; i < ev; i += nwv) {
      const int32_t u = c.col[i];
      const int64_t bu = c.rowptr[u];
      const int64_t eu = wave_first_greater(
          c.col, static_cast<int32_t>(v) - 1, bu, c.rowptr[u + 1]);
      for (int64_t j = bu + lane; j < eu; j += 64) {
        const int32_t w = c.col[j];
        if (atomicAdd(&cnt[w], 1u) == 0u) touched[atomicAdd(&s_nt, 1u)] = w;
      }
    }
    __syncthreads();
    if (c.full5) {
      // Second walk over the same wedges with the final counts: the wedge
      // v-u-w lies on cnt[w] - 1 cycles of the pair (v, w), and each puts
      // its edges vu, uw and its middle u on them (4-cycles per edge and
      // per vertex, weighted by t_e and d_u - 2).
      for (int64_t i = c.rowptr[v] + wv; i < ev; i += nwv) {
        const int32_t u = c.col[i];
        const unsigned long long tvu = c.t_csr[i];
        const unsigned long long du2 = c.deg[u] - 2;
        const int64_t bu = c.rowptr[u];
        const int64_t eu = wave_first_greater(
            c.col, static_cast<int32_t>(v) - 1, bu, c.rowptr[u + 1]);
        for (int64_t j = bu + lane; j < eu; j += 64) {
          const int32_t w = c.col[j];
          // The counts were made by atomics (in L2): read them past L1.
          const unsigned long long x =
              __hip_atomic_load(&cnt[w], __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT) - 1u;
          ban += x * du2;
          tq += x * (tvu + c.t_csr[j]);
        }
      }
      __syncthreads();  // every count read before the clear below
    }
    const unsigned nt = s_nt;
    const unsigned long long dv = c.deg[v];
    for (unsigned k = threadIdx.x; k < nt; k += kC4Threads) {
      // Read and clear in one atomic (the counts were made by atomics).
      const int32_t w = touched[k];
      const unsigned long long x = atomicExch(&cnt[w], 0u);
      const unsigned long long cyc = choose2(x);
      acc += cyc;
      if (c.full5) ban += cyc * (dv + c.deg[w] - 4);
    }
    __syncthreads();  // s_v, s_nt and the list are reused
  }
  acc = wave_sum_u64(acc);
  ban = wave_sum_u64(ban);
  tq = wave_sum_u64(tq);
  if (lane == 0) {
    s_acc[wv] = acc;
    s_ban[wv] = ban;
    s_tq[wv] = tq;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0, b = 0, q = 0;
    for (int k = 0; k < nwv; ++k) {
      t += s_acc[k];
      b += s_ban[k];
      q += s_tq[k];
    }
    if (t) atomicAdd(&c.acc[kCensusC4], t);
    if (b) atomicAdd(&c.acc[kCensusBanner], b);
    if (q) atomicAdd(&c.acc[kCensusCycEdgeT], q);
  }
}

}  // namespace

int census_c4_launch(const CensusArgs &c, hipStream_t s) {
  hipLaunchKernelGGL(census_c4, dim3(std::max(c.c4_groups, 1)),
                     dim3(kC4Threads), 0, s, c);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int census_sums_launch(const CensusArgs &c, int cus, hipStream_t s) {
  const int gv = static_cast<int>(std::max<int64_t>(
      1, std::min<int64_t>((int64_t(c.n) + 255) / 256, int64_t(cus) * 16)));
  hipLaunchKernelGGL(census_sums, dim3(gv), dim3(256), 0, s, c);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace mgpm

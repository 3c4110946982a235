// Sums over vertices and edges of the census graph: with the triangle, 4-
// and 5-clique counts of census_rows.hip and the 4-cycles of census_c4.hip,
// the terms from which P1, P4, P7 and P8 follow in closed form.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "census.hpp"
#include "choose.hpp"
#include "wave.hpp"

namespace mgpm {

namespace {

constexpr int kT = 1024;

// Sums over vertices (C(d,3)) and over edges (t, t (d_x + d_y - 4) in two
// halves, C(t,2), C(t,3) and (d_x - t - 1)(d_y - t - 1)).
// With full5 also C(d,4), the fork, bull and diamond-pendant sums per edge,
// t of every CSR entry, and twice the triangles per vertex into tv.
//
// One thread per CSR entry (an edge counts at its upper entry), so hub rows
// are spread over the device, and one atomic per workgroup and sum on two
// workgroups per CU: a vertex per thread with an atomic per wave took 0.97
// ms on RMAT-20, most of it the 164000 atomics on one cache line.
__global__ __launch_bounds__(kT) void census_sums(CensusArgs c) {
  constexpr int kSums = 11;
  __shared__ unsigned long long s_sum[kSums];
  const int lane = lane64();
  if (threadIdx.x < kSums) s_sum[threadIdx.x] = 0;
  __syncthreads();
  unsigned long long s3 = 0, s2 = 0, sp = 0, st = 0, s4 = 0, fk = 0, dp3 = 0,
                     s1 = 0, tlo = 0, thi = 0, bdeg = 0;
  const int64_t stride = int64_t(gridDim.x) * kT;
  const int64_t first = int64_t(blockIdx.x) * kT;
  for (int64_t v = first + threadIdx.x; v < c.n; v += stride) {
    const unsigned long long d = static_cast<unsigned long long>(c.deg[v]);
    s3 += choose3(d);
    if (c.full5) s4 += choose4(d);
  }
  for (int64_t j0 = first; j0 < 2 * c.m; j0 += stride) {  // whole waves
    const int64_t j = j0 + threadIdx.x;
    const bool in = j < 2 * c.m;
    const int32_t v = in ? c.src[j] : -1, y = in ? c.col[j] : -1;
    const unsigned long long t = in ? c.t[c.arc[j]] : 0u;
    if (c.full5) {
      if (in) c.t_csr[j] = static_cast<uint32_t>(t);
      // Rows are runs of lanes: the last lane of a run adds its sum.
      unsigned long long run = t;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const unsigned long long up = __shfl_up(run, d, 64);
        const int32_t vu = __shfl_up(v, d, 64);
        if (lane >= d && vu == v) run += up;
      }
      const int32_t next = __shfl_down(v, 1, 64);
      if (in && run && (lane == 63 || next != v)) atomicAdd(&c.tv[v], run);
    }
    if (y > v) {
      const unsigned long long d = static_cast<unsigned long long>(c.deg[v]);
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
      }
    }
  }
  const unsigned long long mine[kSums] = {s1, tlo, thi, bdeg, s3, s2,
                                          sp, st,  s4,  fk,   dp3};
#pragma unroll
  for (int k = 0; k < kSums; ++k) {
    const unsigned long long w = wave_sum_u64(mine[k]);
    if (lane == 0 && w) atomicAdd(&s_sum[k], w);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    constexpr int slot[kSums] = {
        kCensusTriangles, kCensusTriDegrees, kCensusTriDegreesHi,
        kCensusBullDeg,   kCensusDeg3,       kCensusEdgePairs,
        kCensusPathPairs, kCensusEdgeTriples, kCensusDeg4,
        kCensusFork,      kCensusDp3};
    for (int k = 0; k < kSums; ++k)
      if (s_sum[k]) atomicAdd(&c.acc[slot[k]], s_sum[k]);
  }
}

}  // namespace

int census_sums_launch(const CensusArgs &c, int cus, hipStream_t s) {
  const int64_t items = std::max<int64_t>(c.n, 2 * c.m);
  const int g = static_cast<int>(std::max<int64_t>(
      1, std::min<int64_t>((items + kT - 1) / kT, int64_t(cus) * 2)));
  hipLaunchKernelGGL(census_sums, dim3(g), dim3(kT), 0, s, c);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace mgpm

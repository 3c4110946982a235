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

}  // namespace

int census_sums_launch(const CensusArgs &c, int cus, hipStream_t s) {
  const int gv = static_cast<int>(std::max<int64_t>(
      1, std::min<int64_t>((int64_t(c.n) + 255) / 256, int64_t(cus) * 16)));
  hipLaunchKernelGGL(census_sums, dim3(gv), dim3(256), 0, s, c);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace mgpm

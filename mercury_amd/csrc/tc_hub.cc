// The triangle count's hub plan (tc_hub.hip): when it is taken, and its
// preparation from the census graph (the graph relabelled in DAG order),
// once per graph and kept with it.
#include <algorithm>
#include <vector>

#include "capi_common.hpp"

namespace mgpm {

namespace {

// Blocks: eight per wave of the counting kernel (20 waves per CU, by LDS),
// of at least 64 partners once every wave has one (a block costs about 5 us
// of latency to start), and never under one run.
uint32_t block_count(uint32_t nparts, uint32_t runs, int cus) {
  const uint32_t waves = static_cast<uint32_t>(cus) * 20;
  return std::min(runs, std::max(waves, std::min(8 * waves, nparts / 64)));
}

// The degrees of the 65535 highest-degree vertices add up to `num` / `den` of
// all degrees or more (each arc into a hub counts once there, arcs between
// hubs twice).
bool hubs_hold(const CsrGraph &g, int64_t num, int64_t den) {
  int32_t top = 0;
#pragma omp parallel for reduction(max : top)
  for (int32_t v = 0; v < g.n; ++v) top = std::max(top, g.degree(v));
  if (den * kHubIds * top < num * g.nnz) return false;
  std::vector<int64_t> count(static_cast<size_t>(top) + 1, 0);
  for (int32_t v = 0; v < g.n; ++v) count[g.degree(v)]++;
  int64_t left = kHubIds, sum = 0;
  for (int32_t d = top; d > 0 && left > 0; --d) {
    const int64_t k = std::min<int64_t>(left, count[d]);
    sum += k * d;
    left -= k;
  }
  return den * sum >= num * g.nnz;
}

// When the hub bitmaps count faster than the table plans (one MI355X, us per
// count, bitmaps / laid-out tables):
//   from 16384 arcs (8192 arcs 37 / 34, RMAT-12's 49000 41 / 96; smaller
//   graphs also keep the shorter preparation of the tables);
//   up to 65535 vertices, where every vertex is a hub (60001 vertices of
//   degree 33: 86 / 151);
//   beyond, where the hubs hold half of all degrees (uniform graphs: 150001
//   vertices 142 / 146, 200003 vertices 262 / 181), or a quarter and the
//   lists that the tables would stream average 32 items or more, which a
//   hash probe each makes dear (RMAT-22: 3650 / 15700).
bool hubs_pay(const mgpm_dgraph *dg) {
  const CsrGraph &g = *dg->host;
  if (g.nnz / 2 < 16384 || g.nnz >= (int64_t(1) << 32)) return false;
  if (g.n <= kHubIds) return true;
  const bool long_lists = dg->tc.probes >= 32 * dg->tc.npart;
  return hubs_hold(g, 1, long_lists ? 4 : 2);
}

}  // namespace

bool tc_hub_wanted(mgpm_dgraph *dg) {
  TcHub &h = dg->hub;
  if (h.wanted < 0) h.wanted = hubs_pay(dg) ? 1 : 0;
  return h.wanted > 0;
}

int tc_hub_prepare(mgpm_dgraph *dg, hipStream_t s) {
  TcHub &h = dg->hub;
  if (h.ready) return MGPM_OK;
  int rc = census_graph_ready(dg, s);
  if (rc) return rc;
  const CensusGraph &cg = dg->census;
  const int32_t n = dg->host->n;
  const int64_t nnz = dg->host->nnz, m = nnz / 2;
  const int32_t hublo = std::max<int32_t>(0, n - kHubIds);
  const size_t n1 = static_cast<size_t>(n) + 1;
  DevBuf split, rowbase, rows, flag, pos, owner, part, bound, start, rest,
      chunks, tmp, own, total, cost, prefix;
  const uint32_t runs = static_cast<uint32_t>((m + kHubRun - 1) / kHubRun);
  MGPM_HIP(split.alloc(n1 * 4));
  MGPM_HIP(chunks.alloc(n1 * 4));
  MGPM_HIP(rowbase.alloc(n1 * 4));
  const size_t sb = tc_hub_scan_bytes(n, runs);
  if (sb == 0) return fail(MGPM_ERR_HIP, "scan size query");
  MGPM_HIP(tmp.alloc(sb));
  const int64_t *drp = cg.drp.as<int64_t>();
  const int32_t *dcol = cg.dcol.as<int32_t>();
  if (tc_hub_counts(drp, dcol, n, hublo, split.as<uint32_t>(),
                    chunks.as<uint32_t>(), s) ||
      tc_hub_scan(chunks.as<uint32_t>(), rowbase.as<uint32_t>(), n, tmp.p, sb,
                  s))
    return fail(MGPM_ERR_HIP, "hub plan kernel launch failed");
  uint32_t nchunks = 0;
  MGPM_HIP(hipMemcpyAsync(&nchunks, rowbase.as<uint32_t>() + n, 4,
                          hipMemcpyDeviceToHost, s));
  MGPM_HIP(hipStreamSynchronize(s));
  if (nchunks < 1 || nchunks > m / kHubChunk + n + 1)
    return fail(MGPM_ERR_INTERNAL, "hub plan: bad row sizes");
  TcHubPlan p;
  p.n = static_cast<uint32_t>(n);
  p.nparts = static_cast<uint32_t>(m);
  p.blocks = block_count(p.nparts, runs, dg->cus);
  MGPM_HIP(rows.alloc(size_t(nchunks) * kHubChunk * 2));
  MGPM_HIP(flag.alloc(n1 * 4));
  MGPM_HIP(pos.alloc(n1 * 4));
  MGPM_HIP(owner.alloc(static_cast<size_t>(n) * sizeof(HubOwner)));
  MGPM_HIP(part.alloc(size_t(m) * sizeof(HubPartner)));
  MGPM_HIP(bound.alloc((size_t(p.blocks) + 1) * 4));
  MGPM_HIP(start.alloc(size_t(p.blocks) * 4));
  MGPM_HIP(cost.alloc((size_t(runs) + 1) * 8));
  MGPM_HIP(prefix.alloc((size_t(runs) + 1) * 8));
  MGPM_HIP(rest.alloc(static_cast<size_t>(n) * 4));
  MGPM_HIP(total.alloc(4));
  constexpr size_t kOwnWords = kHubQueueStride + kHubQueueWords;
  MGPM_HIP(own.alloc(kOwnWords * 4));
  if (device_zero(total.p, 1, s) || device_zero(own.p, kOwnWords, s) ||
      tc_hub_fill(cg.rowptr.as<int64_t>(), cg.col.as<int32_t>(),
                  cg.src.as<int32_t>(), nnz, drp, dcol, cg.arc.as<uint32_t>(),
                  n, split.as<uint32_t>(), rowbase.as<uint32_t>(), rows.p,
                  flag.as<uint32_t>(), pos.as<uint32_t>(),
                  owner.as<HubOwner>(), part.as<HubPartner>(),
                  rest.as<int32_t>(), total.as<uint32_t>(), tmp.p, sb,
                  dg->cus, s))
    return fail(MGPM_ERR_HIP, "hub plan kernel launch failed");
  MGPM_HIP(hipMemcpyAsync(&p.nrest, total.p, 4, hipMemcpyDeviceToHost, s));
  MGPM_HIP(hipMemcpyAsync(&p.owners, pos.as<uint32_t>() + n, 4,
                          hipMemcpyDeviceToHost, s));
  MGPM_HIP(hipStreamSynchronize(s));
  if (p.owners == 0) p.blocks = 0;  // no arc follows another: no triangle
  p.owner = owner.as<HubOwner>();
  p.part = part.as<HubPartner>();
  if (p.blocks &&
      tc_hub_blocks(p, runs, cost.as<unsigned long long>(),
                    prefix.as<unsigned long long>(), tmp.p, sb,
                    bound.as<uint32_t>(), start.as<uint32_t>(), s))
    return fail(MGPM_ERR_HIP, "hub plan kernel launch failed");
  MGPM_HIP(hipStreamSynchronize(s));  // the work arrays die here
  p.rows = rows.p;
  p.bound = bound.as<uint32_t>();
  p.start = start.as<uint32_t>();
  p.rest = rest.as<int32_t>();
  p.drp = drp;
  p.dcol = dcol;
  p.split = split.as<uint32_t>();
  h.split.swap(split);
  h.rows.swap(rows);
  h.owner.swap(owner);
  h.part.swap(part);
  h.bound.swap(bound);
  h.start.swap(start);
  h.rest.swap(rest);
  h.own.swap(own);
  h.plan = p;
  h.ready = true;
  return MGPM_OK;
}

}  // namespace mgpm

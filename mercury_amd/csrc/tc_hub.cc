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
// hubs twice); with more than 65535 degrees of 4096 and up, by a lower bound.
bool hubs_hold(const CsrGraph &g, int64_t num, int64_t den) {
  // Degrees below kFine by value, the rest (on large graphs fewer vertices
  // than there are hubs) as one bin.
  constexpr int32_t kFine = 4096;
  std::vector<int64_t> count(kFine + 1, 0);
  int64_t high = 0;  // sum of the degrees in the last bin
#pragma omp parallel
  {
    std::vector<int64_t> mine(kFine + 1, 0);
    int64_t sum = 0;
#pragma omp for nowait
    for (int32_t v = 0; v < g.n; ++v) {
      const int32_t d = g.degree(v);
      mine[std::min(d, kFine)]++;
      if (d >= kFine) sum += d;
    }
#pragma omp critical
    {
      for (int32_t d = 0; d <= kFine; ++d) count[d] += mine[d];
      high += sum;
    }
  }
  if (count[kFine] >= kHubIds)  // every hub is in the last bin
    return den * kFine * int64_t(kHubIds) >= num * g.nnz ||
           den * high * kHubIds >= num * g.nnz * count[kFine];
  int64_t left = kHubIds - count[kFine], sum = high;
  for (int32_t d = kFine - 1; d > 0 && left > 0; --d) {
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
//   hash probe each makes dear (RMAT-22: 3600 / 15800).
// These are the counts of a resident plan.  A handle's first count also builds
// it, from the census graph (ms, bitmaps / laid-out tables): RMAT-11 0.38 /
// 0.16, RMAT-12 0.43 / 0.21, RMAT-14 0.62 / 0.44, RMAT-15 0.72 / 0.76, RMAT-16
// 0.85 / 1.05, RMAT-18 1.74 / 2.35: below about 300000 arcs 0.2 ms more, which
// one to ten further counts give back.
bool hubs_pay(const mgpm_dgraph *dg) {
  const CsrGraph &g = *dg->host;
  if (g.nnz / 2 < 16384 || g.nnz >= (int64_t(1) << 32)) return false;
  if (g.n <= kHubIds) return true;
  const bool long_lists = dg->tc.probes >= 32 * dg->tc.npart;
  return hubs_hold(g, 1, long_lists ? 4 : 2);
}

// What a plan keeps: its sizes in p, its arrays added to `keep`.
struct HubKeep {
  DevView rows, owner, part, bound, start, rest, split, own;
};
constexpr size_t kOwnWords = kHubQueueStride + kHubQueueWords;

uint32_t runs_of(const mgpm_dgraph *dg) {
  return static_cast<uint32_t>((dg->host->nnz / 2 + kHubRun - 1) / kHubRun);
}

void keep_layout(const mgpm_dgraph *dg, TcHubPlan &p, HubKeep &k,
                 DevArena &keep) {
  const int64_t m = dg->host->nnz / 2;
  const size_t n1 = static_cast<size_t>(dg->host->n) + 1;
  p.n = static_cast<uint32_t>(dg->host->n);
  p.nparts = static_cast<uint32_t>(m);
  p.blocks = block_count(p.nparts, runs_of(dg), dg->cus);
  // Chunks of all rows: every row rounded up, and the padding chunk.
  const size_t nchunks = static_cast<size_t>(m) / kHubChunk + n1;
  keep.add(k.rows, nchunks * kHubChunk * 2);
  keep.add(k.owner, n1 * sizeof(HubOwner));
  keep.add(k.part, static_cast<size_t>(m) * sizeof(HubPartner));
  keep.add(k.bound, (size_t(p.blocks) + 1) * 4);
  keep.add(k.start, (size_t(p.blocks) + 1) * 4);
  keep.add(k.rest, n1 * 4);
  keep.add(k.split, n1 * 4);
  keep.add(k.own, kOwnWords * 4);
}

// Builds the plan (prep_mu held).
int prepare(mgpm_dgraph *dg, hipStream_t s) {
  TcHub &h = dg->hub;
  int rc = census_graph_ready(dg, s);
  if (rc) return rc;
  const CensusGraph &cg = dg->census;
  const int32_t n = dg->host->n;
  const int64_t nnz = dg->host->nnz;
  const int32_t hublo = std::max<int32_t>(0, n - kHubIds);
  const size_t n1 = static_cast<size_t>(n) + 1;
  const uint32_t runs = runs_of(dg);
  const int64_t *drp = cg.drp.as<int64_t>();
  const int32_t *dcol = cg.dcol.as<int32_t>();
  TcHubPlan p;
  HubKeep k;
  DevArena keep;
  keep_layout(dg, p, k, keep);
  DevBuf mem, tmp_mem;  // mem becomes h.mem when it is complete
  DevView rowbase, chunks, flag, pos, meta, cost, prefix, sums, scan;
  const size_t sb = tc_hub_scan_bytes(n, runs);
  if (sb == 0) return fail(MGPM_ERR_HIP, "scan size query");
  DevArena work;
  for (DevView *v : {&rowbase, &chunks, &flag, &pos}) work.add(*v, n1 * 4);
  work.add(meta, n1 * 16);
  work.add(cost, (size_t(runs) + 1) * 8);
  work.add(prefix, (size_t(runs) + 1) * 8);
  // The sums of chunks, and in the first place's third word the rest's size:
  // one fill, one copy back.
  constexpr size_t kSums = size_t(kHubSums) * kHubSumStride;
  work.add(sums, kSums * 8);
  work.add(scan, sb);
  MGPM_HIP(keep.alloc(mem));
  MGPM_HIP(work.alloc(tmp_mem));
  p.rows = k.rows.p;
  p.owner = k.owner.as<HubOwner>();
  p.part = k.part.as<HubPartner>();
  p.bound = k.bound.as<uint32_t>();
  p.start = k.start.as<uint32_t>();
  p.rest = k.rest.as<int32_t>();
  p.drp = drp;
  p.dcol = dcol;
  p.split = k.split.as<uint32_t>();
  const uint32_t *owners = pos.as<uint32_t>() + n;
  uint32_t *nrest =
      reinterpret_cast<uint32_t *>(sums.as<unsigned long long>() + 2);
  if (tc_hub_counts(drp, dcol, n, hublo, k.split.as<uint32_t>(),
                    chunks.as<uint32_t>(), s) ||
      tc_hub_scan(chunks.as<uint32_t>(), rowbase.as<uint32_t>(), n, scan.p,
                  sb, s) ||
      device_zero(sums.p, 2 * kSums, s) || device_zero(k.own.p, kOwnWords, s) ||
      tc_hub_fill(cg.rowptr.as<int64_t>(), cg.col.as<int32_t>(),
                  cg.src.as<int32_t>(), nnz, drp, dcol, cg.arc.as<uint32_t>(),
                  n, k.split.as<uint32_t>(), rowbase.as<uint32_t>(), k.rows.p,
                  flag.as<uint32_t>(), pos.as<uint32_t>(), meta.p,
                  k.owner.as<HubOwner>(), k.part.as<HubPartner>(),
                  k.rest.as<int32_t>(), nrest, scan.p, sb,
                  dg->cus, s) ||
      tc_hub_blocks(p, owners, runs, cost.as<unsigned long long>(),
                    prefix.as<unsigned long long>(), scan.p, sb,
                    k.bound.as<uint32_t>(), k.start.as<uint32_t>(),
                    sums.as<unsigned long long>(), s))
    return fail(MGPM_ERR_HIP, "hub plan kernel launch failed");
  MGPM_HIP(hipMemcpyAsync(&p.owners, owners, 4, hipMemcpyDeviceToHost, s));
  unsigned long long got[kSums];
  MGPM_HIP(hipMemcpyAsync(got, sums.p, sizeof(got), hipMemcpyDeviceToHost, s));
  MGPM_HIP(hipStreamSynchronize(s));  // the work arrays die here
  p.nrest = static_cast<uint32_t>(got[2]);
  if (p.owners == 0) p.blocks = 0;  // no arc follows another: no triangle
  h.mem.swap(mem);
  h.plan = p;
  h.own = k.own;
  h.part_chunks = h.row_chunks = 0;
  for (int i = 0; i < kHubSums; ++i) {
    h.part_chunks += got[i * kHubSumStride];
    h.row_chunks += got[i * kHubSumStride + 1];
  }
  h.ready = true;
  return MGPM_OK;
}

}  // namespace

bool tc_hub_wanted(mgpm_dgraph *dg) {
  TcHub &h = dg->hub;
  if (h.off || h.refused) return false;
  if (h.wanted < 0) h.wanted = hubs_pay(dg) ? 1 : 0;
  return h.wanted > 0;
}

uint64_t tc_hub_bytes(const mgpm_dgraph *dg) {
  TcHubPlan p;
  HubKeep k;
  DevArena keep;
  keep_layout(dg, p, k, keep);
  return keep.bytes();
}

int tc_hub_use(mgpm_dgraph *dg, hipStream_t s, bool *use) {
  TcHub &h = dg->hub;
  *use = false;
  if (!tc_hub_wanted(dg)) return MGPM_OK;
  if ((*use = h.ready)) return MGPM_OK;
  std::lock_guard<std::mutex> lk(dg->prep_mu);
  if ((*use = h.ready)) return MGPM_OK;
  size_t free_b = 0, total_b = 0;
  if (h.short_of) {
    MGPM_HIP(hipMemGetInfo(&free_b, &total_b));
    if (free_b <= h.short_of) return MGPM_OK;
  }
  const bool had = dg->census.ready;
  const int rc = prepare(dg, s);
  if (rc == MGPM_ERR_NOMEM) {
    // Cleared, so that no launch check sees it; without the census graph if
    // that was built for this plan alone.
    (void)hipGetLastError();
    if (!had) census_graph_drop(dg);
    MGPM_HIP(hipMemGetInfo(&free_b, &total_b));
    h.short_of = std::max<size_t>(free_b, 1);
    return MGPM_OK;
  }
  *use = rc == MGPM_OK;
  return rc;
}

void tc_hub_release(mgpm_dgraph *dg) {
  std::lock_guard<std::mutex> lk(dg->prep_mu);
  TcHub &h = dg->hub;
  h.refused = true;
  h.ready = false;
  h.mem.reset();
}

}  // namespace mgpm

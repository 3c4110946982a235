// P1..P8 in closed form from a subgraph census on the device.
//
// The reference counts every pattern per directed edge with set algebra
// (pattern_kernels.cuh:6-963, combined as sm_multigpu.cu:209-232).  Summed
// over the edges, each pattern's counters are a fixed combination of
// induced-subgraph counts:
//   P1 = claws K1,3, P2 = forks, P3 = 4 K1,4 + 3 claws, P4 = paths P4,
//   P5 = 2 bulls, P6 = 2 (diamond + pendant at a degree-3 vertex) + 2 paws,
//   P7 = 2 K1,1,3, P8 = 3 (K4 + pendant).
// Induced counts follow from subgraph counts N(H) (copies of H as a
// subgraph, not necessarily induced) by inverting the containment matrix
// of the graphs on 4 and 5 vertices.  Every N(H) needed is a sum the device
// forms from per-edge triangle counts t_e, per-triangle 4-clique counts k_T,
// 4-cycles and 5-cliques, and -- for wheels, K2,3 and K2,3 plus an edge --
// from the pair passes of census5_kernels.hip.
//
// P1 = sum_v C(d_v,3) - sum_triangles (d_x + d_y + d_z - 6)
//      + 2 sum_e C(t_e,2) - 4 K4                      (claws by centre)
// P4 = sum_e (d_x - t_e - 1)(d_y - t_e - 1)
//      - 4 (C4 - sum_e C(t_e,2) + 3 K4)                 (per task edge)
// P7 = 2 sum_e C(t_e,3) - sum_T k_T (t_ab + t_ac + t_bc - 6)
//      + 6 sum_T C(k_T,2) - 20 K5
// P8 = sum_T k_T (d_a + d_b + d_c - 9) - 3 sum_T k_T (t_ab + t_ac + t_bc - 6)
//      + 18 sum_T C(k_T,2) - 60 K5
// and, with the subgraph counts of census_combine below,
//   K1,4 = star - cricket + dp3 + bowtie - 2 book3 - k4pend - gem
//          + 2 k4wing + W4 - 3 k5e + 5 K5
//   fork = fork - 2 cricket - 2 bull - lolli - 2 banner + 5 dp3 + 4 bowtie
//          + 4 dp2 + 4 house + 6 K23 - 12 book3 - 9 k4pend - 10 gem
//          - 10 K23e + 20 k4wing + 20 W4 - 36 k5e + 60 K5
//   bull = bull - 2 dp3 - 2 dp2 - house + 6 book3 + 6 k4pend + 5 gem
//          + 4 K23e - 14 k4wing - 12 W4 + 30 k5e - 60 K5
//   dp3i = dp3 - 6 book3 - 3 k4pend - 2 gem + 10 k4wing + 4 W4
//          - 24 k5e + 60 K5
//   paw  = sum_T (d_a + d_b + d_c - 6) - 4 sum_e C(t_e,2) + 12 K4.
// The identities are checked term by term against brute-force induced
// counts in tests/test_census5_identity.py (and census_identity.py).
// Counts are uint64 modulo 2^64 throughout, like the reference's unsigned
// counters; no intermediate sum is divided except by 3, through its
// inverse modulo 2^64 (exact for a multiple of 3 whatever the wrap).
#include <algorithm>
#include <cstring>
#include <mutex>

#include "capi_common.hpp"
#include "census.hpp"

namespace mgpm {

namespace {

constexpr int kMaxCensusDevices = 64;

// Per-caller budgets of the per-workgroup arrays.
constexpr size_t kCensusC4Budget = size_t(4) << 30;
constexpr size_t kCensusRowBudget = size_t(8) << 30;  // row passes' slabs
constexpr size_t kCensus5Budget = size_t(8) << 30;  // pair-table layout

// Layout of the small buffer: census cursors, accumulators, pair-pass and
// 4-cycle cursors.
constexpr size_t kSmallBytes = 1024;
constexpr size_t kAccOff = 64;
constexpr size_t kC5CursorOff = 384;
constexpr size_t kC4CursorOff = 512;

// `passes` is a census_passes mask: the triangle pass and the sums always
// run, the 4-cycle, 5-clique and pair passes on request; the pair passes
// also add the 5-vertex terms to the others.
bool is_k5(int passes) { return (passes & kCensusPassK5) != 0; }
bool is_full5(int passes) { return (passes & kCensusPassPairs) != 0; }
bool needs_c4(int passes) { return (passes & kCensusPassC4) != 0; }

// The inverse of 3 modulo 2^64.
constexpr uint64_t kInv3 = 0xAAAAAAAAAAAAAAABull;

template <class T>
int grow(DevBuf &b, size_t count) {
  const size_t want = std::max<size_t>(count, 1) * sizeof(T);
  if (b.bytes >= want) return MGPM_OK;
  MGPM_HIP(b.alloc(want));
  return MGPM_OK;
}

int zero(void *p, size_t bytes, hipStream_t s) {
  if (!p || !bytes) return MGPM_OK;
  if (device_zero(p, (bytes + 3) / 4, s))
    return fail(MGPM_ERR_HIP, "census fill kernel launch failed");
  return MGPM_OK;
}

// Sizes of the workspace for one pattern on one graph.
struct Need {
  size_t t = 0, t_csr = 0, tv = 0, slab = 0, wedges = 0;
  size_t lo = 0, mask = 0, grows = 0, table = 0;
  int c4_groups = 0, c5_groups[kC5Lists] = {};
  int64_t grows_len = 0;
};

// Slab bytes of the row passes: the classes run one after the other on one
// slab.  Without class sizes (count null) every class counts n vertices.
size_t row_slab(const mgpm_dgraph *dg, int passes, int64_t max_out,
                const int64_t *count) {
  size_t b = 0;
  for (int cls = 0; cls < kRowClassCount; ++cls)
    for (const bool cliques : {false, true})
      if (cliques ? is_k5(passes) : cls == kRowClassCount - 1)
        b = std::max(b, rows_slab_bytes(cls, max_out, cliques) *
                            rows_grid(cls, max_out,
                                      count ? rows_members(cls, count, cliques)
                                            : dg->host->n,
                                      cliques, kCensusRowBudget, dg->cus));
  return b;
}

Need need_for(const mgpm_dgraph *dg, int passes, size_t budget) {
  const CsrGraph &G = *dg->host;
  const int64_t n = std::max<int32_t>(G.n, 1);
  const int64_t m = std::max<int64_t>(G.nnz / 2, 1);
  const int64_t nnz = std::max<int64_t>(G.nnz, 1);
  const CensusGraph &cg = dg->census;
  Need k;
  k.t = static_cast<size_t>(m);
  k.slab = row_slab(dg, passes, cg.max_out, cg.row_count);
  // Heavy 4-cycle owners below the window (before the plan is built: as if
  // there were some).
  if (needs_c4(passes) && G.n > kRowWindow &&
      (!cg.c4_ready || cg.c4_count[2][kC4Bits16])) {
    const size_t low = static_cast<size_t>(G.n - kRowWindow);
    const size_t owners = cg.c4_ready ? cg.c4_count[2][kC4Bits16] : low;
    k.c4_groups = static_cast<int>(std::max<size_t>(
        1, std::min<size_t>({size_t(dg->cus) * 2, owners,
                             kCensusC4Budget / (4 * low)})));
    k.wedges = static_cast<size_t>(k.c4_groups) * low;
  }
  if (is_full5(passes)) {
    k.t_csr = static_cast<size_t>(nnz);
    k.tv = static_cast<size_t>(n);
    const int gen_words = static_cast<int>((cg.max_out + 63) / 64);
    // Half the budget per list of anchors: the lists run one after the
    // other on arrays as large as the largest of each kind (before the plan
    // is built: as if every list held all vertices).
    const int32_t winlo = std::max<int32_t>(0, G.n - kRowWindow);
    for (int q = 0; q < kC5Lists; ++q) {
      const bool gen = q == kC5Lists - 1;
      int64_t count = cg.pairs_ready ? cg.c5_count[q] : n;
      if (gen && gen_words <= kC5Words[kC5Windowed - 1]) count = 0;
      const int g = census5_groups(q, count, G.n, winlo, gen_words,
                                   budget / 2, dg->cus);
      k.c5_groups[q] = g;
      if (!g) continue;
      const size_t range = size_t(g) * size_t(gen ? n : winlo);
      const size_t words = size_t(gen ? gen_words : kC5Words[q - 1]);
      k.lo = std::max(k.lo, range);
      k.mask = std::max(k.mask, range * words);
      if (gen) k.grows = size_t(g) * cg.max_out * gen_words;
    }
    k.grows_len = cg.max_out * gen_words;
    k.table = cg.tab_total;
  }
  return k;
}

// Builds the census graph on the device, once: the graph relabelled in DAG
// order, then its DAG.
int graph_ready(mgpm_dgraph *dg, hipStream_t s) {
  CensusGraph &cg = dg->census;
  if (cg.ready) return MGPM_OK;
  const CsrGraph &G = *dg->host;
  const int64_t nnz = G.nnz;
  const int32_t n = G.n;
  if (nnz >= (int64_t(1) << 32))
    return fail(MGPM_ERR_CAPACITY, "census: 2^32 or more arcs");
  const size_t n1 = static_cast<size_t>(n) + 1;
  const size_t na = static_cast<size_t>(nnz);
  DevArena keep, work;
  keep.add(cg.rowptr, n1 * 8);
  keep.add(cg.drp, n1 * 8);
  keep.add(cg.deg, n1 * 4);
  keep.add(cg.order, n1 * 4);
  keep.add(cg.col, na * 4);
  keep.add(cg.src, na * 4);
  keep.add(cg.arc, na * 4);
  keep.add(cg.dcol, na / 2 * 4);
  DevBuf mem, tmp_mem;  // mem becomes cg.mem when it is complete
  DevView tmp, cls;  // cls: class sizes and fill counters
  const size_t tb = census_build_bytes(n, nnz);
  if (tb == 0) return fail(MGPM_ERR_HIP, "sort size query");
  constexpr size_t kCls = 2 * kRowClassCount * sizeof(unsigned);
  work.add(tmp, tb);
  work.add(cls, kCls);
  MGPM_HIP(keep.alloc(mem));
  MGPM_HIP(work.alloc(tmp_mem));
  CensusBuild c;
  c.in_rowptr = dg->csr.rowptr.as<int64_t>();
  c.in_col = dg->csr.colidx.as<int32_t>();
  c.n = n;
  c.nnz = nnz;
  c.cus = dg->cus;
  c.rowptr = cg.rowptr.as<int64_t>();
  c.drp = cg.drp.as<int64_t>();
  c.col = cg.col.as<int32_t>();
  c.src = cg.src.as<int32_t>();
  c.deg = cg.deg.as<int32_t>();
  c.dcol = cg.dcol.as<int32_t>();
  c.arc = cg.arc.as<uint32_t>();
  c.tmp = tmp.p;
  c.tmp_bytes = tb;
  if (census_build(c, s)) return fail(MGPM_ERR_HIP, "census graph build failed");
  int rc = zero(cls.p, kCls, s);
  if (rc) return rc;
  unsigned *cnt = cls.as<unsigned>();
  if (census_rows_classify(c.drp, c.deg, n, cnt, cnt + kRowClassCount,
                           cg.order.as<int32_t>(), s))
    return fail(MGPM_ERR_HIP, "census kernel launch failed");
  unsigned sizes[kRowClassCount];
  MGPM_HIP(hipMemcpyAsync(sizes, cnt, sizeof(sizes), hipMemcpyDeviceToHost,
                          s));
  MGPM_HIP(hipStreamSynchronize(s));  // the work arrays die here
  for (int k = 0; k < kRowClassCount; ++k) cg.row_count[k] = sizes[k];
  // The triangle plan knows the largest DAG out-degree (the same DAG).
  cg.max_out = std::max<int64_t>(dg->tc.max_out, 1);
  cg.mem.swap(mem);
  cg.ready = true;
  return MGPM_OK;
}

unsigned *cursor_of(const CensusWork &w) { return w.small.as<unsigned>(); }

CensusArgs args_of(mgpm_dgraph *dg, int passes, CensusWork &w,
                   const Need &k) {
  const CensusGraph &cg = dg->census;
  CensusArgs c;
  c.drp = cg.drp.as<int64_t>();
  c.dcol = cg.dcol.as<int32_t>();
  c.deg = cg.deg.as<int32_t>();
  c.n = dg->host->n;
  c.m = dg->host->nnz / 2;
  c.t = w.t.as<uint32_t>();
  c.arc = cg.arc.as<uint32_t>();
  c.src = cg.src.as<int32_t>();
  c.order = cg.order.as<int32_t>();
  c.winlo = std::max<int32_t>(0, c.n - kRowWindow);
  c.cursor = cursor_of(w);
  c.acc = census_acc(w);
  c.rowptr = cg.rowptr.as<int64_t>();
  c.col = cg.col.as<int32_t>();
  c.win = cg.c4_win.as<uint32_t>();
  c.c4_cursor = reinterpret_cast<unsigned *>(w.small.as<char>() + kC4CursorOff);
  c.wedges = w.wedges.as<uint32_t>();
  c.full5 = is_full5(passes);
  c.t_csr = w.t_csr.as<uint32_t>();
  c.tv = w.tv.as<unsigned long long>();
  return c;
}

Census5Args args5_of(mgpm_dgraph *dg, CensusWork &w, const Need &k) {
  const CensusGraph &cg = dg->census;
  Census5Args c;
  c.rowptr = cg.rowptr.as<int64_t>();
  c.col = cg.col.as<int32_t>();
  c.src = cg.src.as<int32_t>();
  c.deg = cg.deg.as<int32_t>();
  c.n = dg->host->n;
  c.nnz = dg->host->nnz;
  c.drp = cg.drp.as<int64_t>();
  c.dcol = cg.dcol.as<int32_t>();
  c.t = w.t.as<uint32_t>();
  c.tv = w.tv.as<unsigned long long>();
  c.arc = cg.arc.as<uint32_t>();
  c.anchors = cg.c5_list.as<int32_t>();
  c.winlo = std::max<int32_t>(0, c.n - kRowWindow);
  c.nf = census5_fine_windows(c.n, c.winlo);
  c.win = cg.c4_win.as<uint32_t>();
  c.first = cg.c5_first;
  c.woff = cg.c5_woff.as<uint16_t>();
  c.lo = w.lo.as<uint32_t>();
  c.mask = w.mask.as<unsigned long long>();
  c.list = w.list.as<int32_t>();
  c.gen_words = static_cast<int>((cg.max_out + 63) / 64);
  c.grows = w.grows.as<unsigned long long>();
  c.grows_len = k.grows_len;
  c.tab_off = cg.tab_off.as<unsigned long long>();
  c.table = w.table.as<unsigned long long>();
  c.cursor =
      reinterpret_cast<unsigned *>(w.small.as<char>() + kC5CursorOff);
  c.acc = census_acc(w);
  return c;
}

// Grows `w` to hold `k` (every buffer grow-only by bytes, so each query's
// own layout -- derived from its graph by need_for at enqueue -- fits
// whatever larger queries grew it to).  Arrays the kernels leave zeroed
// are zeroed when (re)allocated; the rest is filled per call.
int work_grow(CensusWork &w, const Need &k, hipStream_t s) {
  int rc;
  auto grow_z = [&](DevBuf &b, size_t bytes) -> int {
    if (b.bytes >= std::max<size_t>(bytes, 1)) return MGPM_OK;
    MGPM_HIP(b.alloc(std::max<size_t>(bytes, 1)));
    return zero(b.p, b.bytes, s);
  };
  if ((rc = grow<uint32_t>(w.t, k.t))) return rc;
  if ((rc = grow<char>(w.small, kSmallBytes))) return rc;
  if ((rc = grow<char>(w.slab, k.slab))) return rc;
  if (k.wedges && (rc = grow_z(w.wedges, k.wedges * 4))) return rc;
  if (k.t_csr) {
    if ((rc = grow<uint32_t>(w.t_csr, k.t_csr))) return rc;
    if ((rc = grow<unsigned long long>(w.tv, k.tv))) return rc;
    if ((rc = grow<unsigned long long>(w.table, k.table))) return rc;
    if ((rc = grow<int32_t>(w.list, k.lo))) return rc;
    if ((rc = grow_z(w.lo, k.lo * 4))) return rc;
    if ((rc = grow_z(w.mask, k.mask * 8))) return rc;
    if ((rc = grow<unsigned long long>(w.grows, k.grows))) return rc;
  }
  return MGPM_OK;
}

}  // namespace

unsigned long long *census_acc(const CensusWork &w) {
  return reinterpret_cast<unsigned long long *>(w.small.as<char>() + kAccOff);
}

uint64_t census_work_bytes(const mgpm_dgraph *dg, int passes,
                           size_t budget) {
  if (!dg->census.ready) {
    // What the graph will keep (a bound), plus a bound on the workspace.
    const CsrGraph &G = *dg->host;
    const uint64_t n1 = static_cast<uint64_t>(G.n) + 1;
    uint64_t dag = 24ull * n1 + 14ull * G.nnz;  // the census graph
    if (needs_c4(passes)) dag += 16ull * n1;    // windows, three lists
    if (is_full5(passes)) {                     // table, list, offsets
      const int32_t winlo = std::max<int32_t>(0, G.n - kRowWindow);
      dag += (12ull + 2ull * (census5_fine_windows(G.n, winlo) + 1)) * n1;
    }
    const uint64_t work = is_full5(passes) ? budget + 16ull * G.nnz
                                           : 32ull * G.nnz;
    return dag + work +
           row_slab(dg, passes, std::max<int64_t>(dg->tc.max_out, 1), nullptr);
  }
  const Need k = need_for(dg, passes, budget);
  return 4ull * k.t + kSmallBytes + k.slab + 4ull * k.wedges +
         4ull * k.t_csr + 8ull * k.tv + 8ull * k.lo + 8ull * k.mask +
         8ull * k.grows + 8ull * k.table;
}

namespace {

// The 4-cycle pass's plan of the graph (once): row offsets of the window,
// and the owners of every kind and class.
C4Plan c4_plan_of(const CensusGraph &cg) {
  C4Plan p;
  int32_t *at = cg.c4_list.as<int32_t>();
  for (int k = 0; k < kC4Kinds; ++k) {
    p.list[k] = at;
    for (int q = 0; q < kC4Classes; ++q) {
      p.count[k][q] = cg.c4_count[k][q];
      at += p.count[k][q];
    }
  }
  return p;
}

int c4_layout(mgpm_dgraph *dg, hipStream_t s) {
  CensusGraph &cg = dg->census;
  if (cg.c4_ready) return MGPM_OK;
  CensusArgs c;
  c.drp = cg.drp.as<int64_t>();
  c.rowptr = cg.rowptr.as<int64_t>();
  c.col = cg.col.as<int32_t>();
  c.arc = cg.arc.as<uint32_t>();
  c.n = dg->host->n;
  c.winlo = std::max<int32_t>(0, c.n - kRowWindow);
  const size_t n = std::max<size_t>(c.n, 1);
  DevBuf win, cls, fill;
  unsigned sizes[kC4Kinds * kC4Classes];
  MGPM_HIP(win.alloc(n * sizeof(uint32_t)));
  MGPM_HIP(cls.alloc(n + static_cast<size_t>(c.winlo)));
  MGPM_HIP(fill.alloc(sizeof(sizes)));
  c.win = win.as<uint32_t>();
  int rc = zero(fill.p, sizeof(sizes), s);
  if (rc) return rc;
  if (census_c4_window(c, win.as<uint32_t>(), s) ||
      census_c4_classes(c, cls.as<int8_t>(), fill.as<unsigned>(), s))
    return fail(MGPM_ERR_HIP, "census kernel launch failed");
  MGPM_HIP(hipMemcpyAsync(sizes, fill.p, sizeof(sizes), hipMemcpyDeviceToHost,
                          s));
  MGPM_HIP(hipStreamSynchronize(s));
  size_t total = 0;
  for (const unsigned x : sizes) total += x;
  MGPM_HIP(cg.c4_list.alloc(std::max<size_t>(total, 1) * sizeof(int32_t)));
  for (int k = 0; k < kC4Kinds; ++k)
    for (int q = 0; q < kC4Classes; ++q)
      cg.c4_count[k][q] = sizes[kC4Classes * k + q];
  if ((rc = zero(fill.p, sizeof(sizes), s))) return rc;
  if (census_c4_lists(c, cls.as<int8_t>(), fill.as<unsigned>(),
                      c4_plan_of(cg), s))
    return fail(MGPM_ERR_HIP, "census kernel launch failed");
  MGPM_HIP(hipStreamSynchronize(s));  // the work arrays die here
  cg.c4_win.swap(win);
  cg.c4_ready = true;
  return MGPM_OK;
}

// The pair passes' plan of the graph (once): per anchor, a power of two of
// table slots at least twice the pairs it will hold, from one count pass
// over temporary stamps and one scan; the anchors by list; the offsets of
// the fine windows in every row.  Two reads: list sizes, table slots.
int pairs_layout(mgpm_dgraph *dg, hipStream_t s) {
  CensusGraph &cg = dg->census;
  if (cg.pairs_ready) return MGPM_OK;
  const int32_t n = dg->host->n;
  const int64_t nnz = dg->host->nnz;
  const size_t n0 = std::max<size_t>(n, 1), n1 = static_cast<size_t>(n) + 1;
  Census5Args c;
  c.rowptr = cg.rowptr.as<int64_t>();
  c.col = cg.col.as<int32_t>();
  c.src = cg.src.as<int32_t>();
  c.deg = cg.deg.as<int32_t>();
  c.n = n;
  c.nnz = nnz;
  c.drp = cg.drp.as<int64_t>();
  c.dcol = cg.dcol.as<int32_t>();
  c.arc = cg.arc.as<uint32_t>();
  c.winlo = std::max<int32_t>(0, n - kRowWindow);
  c.nf = census5_fine_windows(n, c.winlo);
  c.win = cg.c4_win.as<uint32_t>();
  const size_t below = std::max<size_t>(c.winlo, 1);
  c.groups = static_cast<int>(std::max<size_t>(
      1, std::min<size_t>(size_t(dg->cus) * 2,
                          (kCensus5Budget / 4) / (4 * below))));
  constexpr size_t kCls = (3 * kC5Lists + 1) * sizeof(unsigned);
  size_t sb = 0;
  if (census5_scan_bytes(int64_t(n1), &sb))
    return fail(MGPM_ERR_HIP, "scan size query");
  DevBuf off, list, woff, mem;
  DevArena work;
  // cnt: list sizes, the first row with offsets, starts, fills.
  DevView cap, stamp, small, scan, cls, cnt;
  work.add(cap, n1 * 8);
  work.add(stamp, size_t(c.groups) * below * 4);
  work.add(small, kSmallBytes);
  work.add(scan, std::max<size_t>(sb, 1));
  work.add(cls, n0);
  work.add(cnt, kCls);
  MGPM_HIP(off.alloc(n1 * 8));
  MGPM_HIP(work.alloc(mem));
  c.stamp = stamp.as<uint32_t>();
  c.tab_cap = cap.as<unsigned long long>();
  c.cursor = reinterpret_cast<unsigned *>(small.as<char>() + kC5CursorOff);
  unsigned *sizes_d = cnt.as<unsigned>();
  int rc;
  if ((rc = zero(small.p, kSmallBytes, s))) return rc;
  if (c.winlo && (rc = zero(stamp.p, size_t(c.groups) * below * 4, s)))
    return rc;
  if ((rc = zero(cap.p, n1 * 8, s))) return rc;
  if ((rc = zero(cnt.p, kCls, s))) return rc;
  if (census5_classes(c, cls.as<int8_t>(), sizes_d, s))
    return fail(MGPM_ERR_HIP, "census kernel launch failed");
  unsigned sizes[kC5Lists + 1], starts[kC5Lists];
  MGPM_HIP(hipMemcpyAsync(sizes, sizes_d, sizeof(sizes),
                          hipMemcpyDeviceToHost, s));
  MGPM_HIP(hipStreamSynchronize(s));
  size_t at = 0;
  for (int k = 0; k < kC5Lists; ++k) {
    starts[k] = static_cast<unsigned>(at);
    at += sizes[k];
  }
  MGPM_HIP(list.alloc(std::max<size_t>(at, 1) * sizeof(int32_t)));
  c.anchors = list.as<int32_t>();
  c.first = static_cast<int32_t>(sizes[kC5Lists]);
  // Only the anchors whose targets take LDS windows read the offsets.
  if (starts[kC5Lists - 1] > starts[kC5Light + 1]) {
    MGPM_HIP(woff.alloc((n1 - c.first) * (c.nf + 1) * sizeof(uint16_t)));
    if (census5_window_offsets(c, woff.as<uint16_t>(), dg->cus, s))
      return fail(MGPM_ERR_HIP, "census kernel launch failed");
  }
  unsigned *starts_d = sizes_d + kC5Lists + 1;
  MGPM_HIP(hipMemcpyAsync(starts_d, starts, sizeof(starts),
                          hipMemcpyHostToDevice, s));
  if (census5_lists(n, cls.as<int8_t>(), starts_d, starts_d + kC5Lists,
                    list.as<int32_t>(), s) ||
      census5_table_count_launch(c, sizes, dg->cus, s))
    return fail(MGPM_ERR_HIP, "census kernel launch failed");
  if (census5_scan(cap.as<unsigned long long>(), off.as<unsigned long long>(),
                   int64_t(n1), scan.p, sb, s))
    return fail(MGPM_ERR_HIP, "census scan failed");
  unsigned long long total = 0;
  MGPM_HIP(hipMemcpyAsync(&total, off.as<unsigned long long>() + n, 8,
                          hipMemcpyDeviceToHost, s));
  MGPM_HIP(hipStreamSynchronize(s));  // the work arrays die here
  for (int k = 0; k < kC5Lists; ++k) cg.c5_count[k] = sizes[k];
  cg.c5_first = c.first;
  cg.tab_off.swap(off);
  cg.c5_list.swap(list);
  cg.c5_woff.swap(woff);
  cg.tab_total = total;
  cg.pairs_ready = true;
  return MGPM_OK;
}

}  // namespace

int census_graph_ready(mgpm_dgraph *dg, hipStream_t s) {
  return graph_ready(dg, s);
}

void census_graph_drop(mgpm_dgraph *dg) {
  dg->census.ready = false;
  dg->census.mem.reset();
}

int census_graph_prepare(mgpm_dgraph *dg, hipStream_t s) {
  std::lock_guard<std::mutex> lk(dg->prep_mu);
  int rc = graph_ready(dg, s);
  if (rc) return rc;
  if ((rc = c4_layout(dg, s))) return rc;
  return pairs_layout(dg, s);
}

int census_passes(int pattern) {
  switch (pattern) {
    case MGPM_P1: return 0;
    case MGPM_P4: return kCensusPassC4;
    case MGPM_P7: case MGPM_P8: return kCensusPassK5;
    default:  // P2, P3, P5, P6
      return kCensusPassC4 | kCensusPassK5 | kCensusPassPairs;
  }
}

int census_prepare(mgpm_dgraph *dg, int passes, CensusWork &w,
                   hipStream_t s) {
  {
    std::lock_guard<std::mutex> lk(dg->prep_mu);
    int rc = graph_ready(dg, s);
    if (rc) return rc;
    if (needs_c4(passes) && (rc = c4_layout(dg, s))) return rc;
    if (is_full5(passes) && (rc = pairs_layout(dg, s))) return rc;
  }
  return work_grow(w, need_for(dg, passes, w.budget), s);
}

int census_enqueue(mgpm_dgraph *dg, int passes, CensusWork &w,
                   hipStream_t s) {
  const Need k = need_for(dg, passes, w.budget);
  CensusArgs c = args_of(dg, passes, w, k);
  int rc;
  if ((rc = zero(w.small.p, kSmallBytes, s))) return rc;
  const bool f5 = is_full5(passes);
  if (f5 && (rc = zero(w.tv.p, static_cast<size_t>(c.n) * 8, s))) return rc;
  const CensusGraph &cg = dg->census;
  if (census_rows_launch(c, cg.row_count, cg.max_out, false,
                         w.slab.as<char>(), kCensusRowBudget, dg->cus, s) ||
      census_sums_launch(c, dg->cus, s))
    return fail(MGPM_ERR_HIP, "census kernel launch failed");
  Census5Args c5;
  if (f5) {
    c5 = args5_of(dg, w, k);
    if (census5_flat_launch(c5, dg->cus, s))
      return fail(MGPM_ERR_HIP, "census kernel launch failed");
  }
  if (needs_c4(passes) &&
      census_c4_launch(c, c4_plan_of(cg), k.c4_groups, dg->cus, s))
    return fail(MGPM_ERR_HIP, "census kernel launch failed");
  if (is_k5(passes) &&
      census_rows_launch(c, cg.row_count, cg.max_out, true, w.slab.as<char>(),
                         kCensusRowBudget, dg->cus, s))
    return fail(MGPM_ERR_HIP, "census kernel launch failed");
  if (f5) {
    if ((rc = zero(w.table.p, cg.tab_total * 8, s))) return rc;
    if (census5_pairs_launch(c5, cg.c5_count, k.c5_groups, dg->cus, s))
      return fail(MGPM_ERR_HIP, "census kernel launch failed");
  }
  return MGPM_OK;
}

int census_combine(int pattern, const unsigned long long *acc,
                   uint64_t *count) {
  const uint64_t pairs_t = acc[kCensusEdgePairs], k4 = acc[kCensusK4];
  // Half of a sum kept in two halves of 32 bits, exact modulo 2^64.
  const unsigned __int128 tdeg2 =
      static_cast<unsigned __int128>(acc[kCensusTriDegrees]) +
      (static_cast<unsigned __int128>(acc[kCensusTriDegreesHi]) << 32);
  const uint64_t tdeg = static_cast<uint64_t>(tdeg2 >> 1);
  if (pattern == MGPM_P1) {
    *count = acc[kCensusDeg3] - tdeg + 2 * pairs_t - 4 * k4;
    return MGPM_OK;
  }
  if (pattern == MGPM_P4) {  // induced 4-cycles = C4 - sum C(t_e,2) + 3 K4
    *count = acc[kCensusPathPairs] - 4 * (acc[kCensusC4] - pairs_t + 3 * k4);
    return MGPM_OK;
  }
  // Two independent counts of the 4-cliques, every common neighbourhood of
  // the size its triangle count says, the halved sum even (parity survives
  // the wrap modulo 2^64), and every pair lookup found.
  if (acc[kCensusMismatch] != 0 || acc[kCensusK4Rows] != k4 ||
      acc[kCensusTriEdgeK] % 2 != 0 || acc[kCensusTableMiss] != 0)
    return fail(MGPM_ERR_INTERNAL, "census: self-checks disagree");
  const uint64_t tek = acc[kCensusTriEdgeK];  // 2 k4wing
  const uint64_t tdk = acc[kCensusTriDegK];   // 3 k4pend
  const uint64_t k5e = acc[kCensusTriPairs], k5 = acc[kCensusK5];
  const uint64_t book3 = acc[kCensusEdgeTriples];
  if (pattern == MGPM_P7) {
    *count = 2 * book3 - tek + 6 * k5e - 20 * k5;
    return MGPM_OK;
  }
  if (pattern == MGPM_P8) {
    *count = tdk - 3 * tek + 18 * k5e - 60 * k5;
    return MGPM_OK;
  }
  const uint64_t tri = acc[kCensusTriangles] / 3;
  const uint64_t k4pend = tdk * kInv3;
  const uint64_t gem = acc[kCensusGem] - 12 * k4;
  const uint64_t w4 = acc[kCensusW4];
  const uint64_t dp3 = acc[kCensusDp3];
  const uint64_t cricket = acc[kCensusCricket];
  const uint64_t bowtie = acc[kCensusTv2] - 2 * pairs_t;
  const uint64_t star = acc[kCensusDeg4] - cricket + dp3 + bowtie -
                        2 * book3 - k4pend - gem + tek + w4 - 3 * k5e +
                        5 * k5;
  const uint64_t dp3i = dp3 - 6 * book3 - 3 * k4pend - 2 * gem + 5 * tek +
                        4 * w4 - 24 * k5e + 60 * k5;
  if (pattern == MGPM_P3) {
    const uint64_t claw = acc[kCensusDeg3] - tdeg + 2 * pairs_t - 4 * k4;
    *count = 4 * star + 3 * claw;
    return MGPM_OK;
  }
  if (pattern == MGPM_P6) {
    const uint64_t paw = tdeg - 4 * pairs_t + 12 * k4;
    *count = 2 * dp3i + 2 * paw;
    return MGPM_OK;
  }
  const uint64_t bull = acc[kCensusBullDeg] - 2 * pairs_t;
  const uint64_t dp2 = acc[kCensusDp2] - 12 * k4;
  const uint64_t house = acc[kCensusCycEdgeT] - 4 * pairs_t;
  const uint64_t k23e = acc[kCensusK23e];
  if (pattern == MGPM_P5) {
    const uint64_t bulli = bull - 2 * dp3 - 2 * dp2 - house + 6 * book3 +
                           6 * k4pend + 5 * gem + 4 * k23e - 7 * tek -
                           12 * w4 + 30 * k5e - 60 * k5;
    *count = 2 * bulli;
    return MGPM_OK;
  }
  // P2: induced forks.  sum_T (d sum) = tdeg + 6 triangles.
  const uint64_t lolli =
      acc[kCensusTriS] - 2 * (tdeg + 6 * tri) + 6 * tri - 4 * pairs_t;
  const uint64_t banner = acc[kCensusBanner] - 2 * pairs_t;
  *count = acc[kCensusFork] - 2 * cricket - 2 * bull - lolli - 2 * banner +
           5 * dp3 + 4 * bowtie + 4 * dp2 + 4 * house + 6 * acc[kCensusK23] -
           12 * book3 - 9 * k4pend - 10 * gem - 10 * k23e + 10 * tek +
           20 * w4 - 36 * k5e + 60 * k5;
  return MGPM_OK;
}

namespace {

// The single-query path's workspace: one per device, shared by every
// graph on it (a workspace per graph would hold gigabytes per handle), so
// single-query census calls on one device run one at a time.  Never freed:
// it lives until the process ends.
struct SharedWork {
  std::mutex mu;
  CensusWork w;
};

SharedWork &shared_work(int device) {
  static SharedWork *all = new SharedWork[kMaxCensusDevices];
  return all[device];
}

}  // namespace

int census_pattern_count(mgpm_dgraph *dg, int pattern, hipStream_t s,
                         uint64_t *count, float *kernel_ms) {
  if (pattern < MGPM_P1 || pattern > MGPM_P8)
    return fail(MGPM_ERR_PATTERN, "Not support.");
  if (dg->device < 0 || dg->device >= kMaxCensusDevices)
    return fail(MGPM_ERR_NODEVICE, "census: device index out of range");
  SharedWork &sw = shared_work(dg->device);
  std::lock_guard<std::mutex> lk(sw.mu);
  CensusWork &w = sw.w;
  const int passes = census_passes(pattern);
  int rc = census_prepare(dg, passes, w, s);
  if (rc) return rc;
  MGPM_HIP(hipEventRecord(dg->ev0, s));
  if ((rc = census_enqueue(dg, passes, w, s))) return rc;
  MGPM_HIP(hipEventRecord(dg->ev1, s));
  unsigned long long acc[kCensusSlots];
  MGPM_HIP(hipMemcpyAsync(acc, census_acc(w), sizeof(acc),
                          hipMemcpyDeviceToHost, s));
  MGPM_HIP(hipStreamSynchronize(s));
  MGPM_HIP(hipEventElapsedTime(kernel_ms, dg->ev0, dg->ev1));
  return census_combine(pattern, acc, count);
}

}  // namespace mgpm

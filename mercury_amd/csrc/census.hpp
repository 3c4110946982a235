// Subgraph census (census_rows.hip, census_kernels.hip,
// census5_kernels.hip): per-edge triangle counts and the sums from which
// the pattern counts follow in closed form.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstdint>

namespace mgpm {

// Accumulator slots (uint64, zeroed by the caller).
enum CensusAcc : int {
  kCensusTriangles = 0,   // sum over edges of t_e: 3 x triangles
  kCensusTriDegrees = 1,  // sum over edges of t_e (d_x + d_y - 4), low 32
                          //   bits of each term (the high ones in
                          //   kCensusTriDegreesHi): twice the sum over
                          //   triangles of d(x) + d(y) + d(z) - 6
  kCensusK4 = 2,          // 4-cliques
  kCensusDeg3 = 3,        // sum over vertices of C(d, 3)
  kCensusEdgePairs = 4,   // sum over edges of C(t_e, 2)
  kCensusPathPairs = 5,   // sum over edges {x,y} of (d_x - t - 1)(d_y - t - 1)
  kCensusC4 = 6,          // 4-cycles (as subgraphs, not necessarily induced)
  kCensusEdgeTriples = 7, // sum over edges of C(t_e, 3)
  // census_rows_launch with cliques, k_T = 4-cliques on triangle T:
  kCensusTriPairs = 8,    // sum over triangles of C(k_T, 2)
  kCensusTriEdgeK = 9,    // sum over triangles of k_T (t_ab + t_ac + t_bc - 6)
  kCensusTriDegK = 10,    // sum over triangles of k_T (d_a + d_b + d_c - 9)
  kCensusK4Rows = 11,     // 4-cliques again (from the adjacency rows)
  kCensusK5 = 12,         // 5-cliques
  kCensusMismatch = 13,   // arcs whose common neighbourhood != t_e (0)
  // Subgraph counts of the 5-vertex census (P2, P3, P5, P6; full5 set):
  kCensusDeg4 = 14,       // sum over vertices of C(d, 4)
  kCensusFork = 15,       // sum over ordered edges (c, x) of
                          //   C(d_c - 1, 2)(d_x - 1) - t_cx (d_c - 2)
  kCensusCricket = 16,    // sum over triangles, vertices of C(d - 2, 2)
  kCensusBullDeg = 17,    // sum over edges of t_e (d_a - 2)(d_b - 2): over
                          //   triangles, vertex pairs of (d_a - 2)(d_b - 2)
  kCensusTriS = 18,       // sum over vertices of t_v s_v,
                          //   s_v = sum over neighbours x of (d_x - 1)
  kCensusDp3 = 19,        // sum over edges of C(t_e, 2)(d_a + d_b - 6)
  kCensusTv2 = 20,        // sum over vertices of C(t_v, 2)
  kCensusBanner = 21,     // sum over 4-cycles, vertices of (d_v - 2)
  kCensusCycEdgeT = 22,   // sum over edges of t_e q_e (q_e: 4-cycles on e)
  kCensusDp2 = 23,        // sum over triangles, edges of (t_e - 1)(d_opp - 2)
  kCensusGem = 24,        // sum over triangles, vertices h of
                          //   (t_hx - 1)(t_hy - 1)
  kCensusW4 = 25,         // wheels: sum over h of 4-cycles inside N(h)
  kCensusK23 = 26,        // sum over vertex pairs of C(codeg, 3)
  kCensusK23e = 27,       // sum over vertex pairs {a,c} of
                          //   E(N(a) ∩ N(c)) (codeg(a,c) - 2)
  kCensusTableMiss = 28,  // pair lookups that found no entry (0)
  kCensusTriDegreesHi = 29,  // high 32 bits of kCensusTriDegrees' terms
  kCensusSlots = 32
};

// The census runs on the graph relabelled in DAG order (census_build):
// rank is id, so "ranked below v" is "id below v", every CSR row is sorted
// with the vertices below its own first, and the DAG rows are the tails.
//
// Its construction (census_graph.hip): from the CSR (in_rowptr, in_col) the
// relabelled CSR (rowptr n + 1, col nnz, the row of every entry src nnz), the
// degrees, the DAG (drp n + 1, dcol nnz / 2) and the DAG arc of every entry
// (nnz); tmp holds census_build_bytes.  Returns 0, or -1 if a launch, scan
// or sort failed.
struct CensusBuild {
  const int64_t *in_rowptr = nullptr;
  const int32_t *in_col = nullptr;
  int32_t n = 0;
  int64_t nnz = 0;
  int cus = 256;
  int64_t *rowptr = nullptr, *drp = nullptr;
  int32_t *col = nullptr, *src = nullptr, *deg = nullptr, *dcol = nullptr;
  uint32_t *arc = nullptr;
  void *tmp = nullptr;
  size_t tmp_bytes = 0;
};
size_t census_build_bytes(int32_t n, int64_t nnz);  // 0: query failed
int census_build(const CensusBuild &c, hipStream_t s);

struct CensusArgs {
  const int64_t *drp = nullptr;  // DAG row offsets (n + 1)
  const int32_t *dcol = nullptr; // DAG column array (m)
  const int32_t *deg = nullptr;  // undirected degrees (n)
  int32_t n = 0;
  int64_t m = 0;
  uint32_t *t = nullptr;         // per DAG arc: triangles on the edge (out)
  unsigned *cursor = nullptr;    // 16 queue counters (zeroed)
  unsigned long long *acc = nullptr;  // kCensusSlots (zeroed)
  // Undirected CSR (relabelled, rows sorted), and the DAG arc of each entry.
  const int64_t *rowptr = nullptr;
  const int32_t *col = nullptr;
  const uint32_t *arc = nullptr;
  const int32_t *src = nullptr;  // row of every CSR entry
  // Vertices with out-neighbours, by class of their number (RowClass), and
  // the lowest id of the rows' bitmap window.
  const int32_t *order = nullptr;
  int32_t winlo = 0;
  // 4-cycle pass (census_c4.hip): first entry of every row in the window,
  // queue counters (12, zeroed) and, for heavy owners below the window, per
  // workgroup a dense counter array (winlo entries, zeroed; left zeroed).
  const uint32_t *win = nullptr;
  unsigned *c4_cursor = nullptr;
  uint32_t *wedges = nullptr;
  // 5-vertex census extras (P2, P3, P5, P6): the terms above marked full5
  // are accumulated only when set; t_csr gets t_e per CSR entry and tv twice
  // the triangles per vertex (zeroed) from census_sums_launch.
  bool full5 = false;
  uint32_t *t_csr = nullptr;
  unsigned long long *tv = nullptr;
};

// Classes of vertices of the row passes (census_rows.hip): up to 64
// out-neighbours, up to 32 neighbours on either side, up to 256 and 704
// out-neighbours with their bit rows in LDS, and the rest with rows in the
// workgroup's slab.
constexpr int kRowClassCount = 5;
constexpr int32_t kRowWindow = 65536;  // ids of the bitmap, the highest ones

struct RowArgs {
  const int32_t *list = nullptr;  // the class's vertices
  uint32_t count = 0;
  unsigned *cursor = nullptr;
  int grab = 1;                   // vertices per queue access
  char *slab = nullptr;           // per workgroup slab_bytes
  size_t slab_bytes = 0;
  uint32_t tri_cap = 0;           // triangles a vertex of the class can have
  int pcap = 0;                   // out-neighbours it can have
  int64_t words = 0;              // 64-bit words of row storage
};

// The pair passes of the 5-vertex census (census5_kernels.hip).  Anchors
// are the vertices, each processed as the lowest-ranked vertex (DAG order:
// degree, then id) of the occurrences it accounts for, in lists: light ones
// (few items), then by DAG out-degree d+ up to 64 * kC5Words[k] with the
// targets of the window in LDS, then the rest with everything in global
// memory.
constexpr int kC5Windowed = 4;
constexpr int kC5Words[kC5Windowed] = {1, 2, 4, 8};
constexpr int kC5Light = 0;                  // list of the light anchors
constexpr int kC5Lists = kC5Windowed + 2;
constexpr unsigned kLightItems = 256;
constexpr int kFine = 1664;                  // ids of a fine window

struct C5List {
  const int32_t *list = nullptr;
  uint32_t count = 0;
  uint32_t grab = 1;  // per queue access
  unsigned *cursor = nullptr;
};

struct Census5Args {
  const int64_t *rowptr = nullptr;   // undirected CSR
  const int32_t *col = nullptr;
  const int32_t *src = nullptr;      // row of every CSR arc (nnz)
  const int32_t *deg = nullptr;      // n
  int32_t n = 0;
  int64_t nnz = 0;
  const int64_t *drp = nullptr;      // DAG
  const int32_t *dcol = nullptr;
  const uint32_t *t = nullptr;       // per DAG arc triangles
  const unsigned long long *tv = nullptr;  // twice the triangles per vertex
  const uint32_t *arc = nullptr;     // DAG arc of every CSR entry
  const int32_t *anchors = nullptr;  // the lists of anchors, in order
  // The window: its lowest id, the first entry of every row in it, and the
  // entries of a row before each of nf fine windows (nf + 1 per row): zeros
  // for the rows below `first`, the first vertex of two neighbours (one of a
  // single neighbour leads only back to the anchor), then a row each.
  int32_t winlo = 0;
  int nf = 0;
  int32_t first = 0;
  const uint32_t *win = nullptr;
  const uint16_t *woff = nullptr;
  // Per workgroup, for the targets below the window (or, last list, all):
  // counts (u32) and masks (words x u64), zero and left zero, and a list of
  // the targets touched; stamps of the count pass.
  uint32_t *stamp = nullptr;
  uint32_t *lo = nullptr;
  unsigned long long *mask = nullptr;
  int32_t *list = nullptr;
  int groups = 0;                    // workgroups of the count pass
  int gen_words = 1;                 // words per mask of the last list
  unsigned long long *grows = nullptr;  // last class: rows per workgroup
  int64_t grows_len = 0;             // max d+ x gen_words
  // Pair table: codeg(p, q) of every pair (p below q) with a common
  // neighbour below p, hashed per p into tab_off[p] .. tab_off[p + 1]
  // (a power of two of slots, or none).
  unsigned long long *tab_cap = nullptr;  // n + 1 (out of the count pass)
  unsigned long long *tab_off = nullptr;  // n + 1 (exclusive scan of cap)
  unsigned long long *table = nullptr;    // zeroed
  unsigned *cursor = nullptr;        // 16 queue counters (zeroed)
  unsigned long long *acc = nullptr; // kCensusSlots
};

// Enqueues the per-vertex sums (kCensusTriS, kCensusTv2, kCensusCricket);
// needs tv from census_sums_launch.
int census5_flat_launch(const Census5Args &c, int cus, hipStream_t s);
// Enqueues the pair-table count pass (tab_cap, from zeroed stamps); the
// caller scans tab_cap into tab_off and sizes the table from tab_off[n].
int census5_table_count_launch(const Census5Args &c, const uint32_t *count,
                               int cus, hipStream_t s);
// The anchors' lists: classes of all vertices (n; list sizes into fill,
// kC5Lists entries, zeroed, and Census5Args::first after them), then, with fill zeroed again and the starts of
// the lists, the lists.
int census5_classes(const Census5Args &c, int8_t *cls, unsigned *fill,
                    hipStream_t s);
int census5_lists(int32_t n, const int8_t *cls, const unsigned *start,
                  unsigned *fill, int32_t *list, hipStream_t s);
// Fine windows of a graph, and their offsets (n - first + 1 rows of nf + 1).
int census5_fine_windows(int32_t n, int32_t winlo);
int census5_window_offsets(const Census5Args &c, uint16_t *woff, int cus,
                           hipStream_t s);
// Raises the dynamic-LDS limits (once per process).
int census5_init();
// Workgroups of list `cls` whose global arrays fit `budget` bytes.
int census5_groups(int cls, int64_t count, int32_t n, int32_t winlo,
                   int gen_words, size_t budget, int cus);
// Exclusive prefix sum of `count` uint64 values; tmp of census5_scan_bytes.
int census5_scan_bytes(int64_t count, size_t *bytes);
int census5_scan(const unsigned long long *in, unsigned long long *out,
                 int64_t count, void *tmp, size_t tmp_bytes, hipStream_t s);
// Enqueues the anchor and out-neighbourhood passes of every list (sizes
// count, workgroups groups; kCensusW4, kCensusK23, kCensusK23e,
// kCensusTableMiss).
int census5_pairs_launch(const Census5Args &c, const uint32_t *count,
                         const int *groups, int cus, hipStream_t s);

// Raises the dynamic-LDS limit of the row kernels (once per process).
int census_rows_init();

// Slab bytes per workgroup of class `cls`, and its workgroups (0 for an
// empty class) within `budget` bytes of slab, for graphs whose largest DAG
// out-degree is max_out.  cliques: the pass of that setting.
size_t rows_slab_bytes(int cls, int64_t max_out, bool cliques);
// Vertices of class `cls` in a pass, of the class sizes count.
int64_t rows_members(int cls, const int64_t *count, bool cliques);
int rows_grid(int cls, int64_t max_out, int64_t count, bool cliques,
              size_t budget, int cus);

// Enqueues the vertices by class into list (n entries), the class sizes
// into count (kRowClassCount, with fill zeroed before the call).
int census_rows_classify(const int64_t *drp, const int32_t *deg, int32_t n,
                         unsigned *count, unsigned *fill, int32_t *list,
                         hipStream_t s);

// Enqueues one row pass over every class.  cliques = false: t of every arc
// and kCensusK4; cliques = true (t complete): the per-triangle 4-clique
// terms and the 5-cliques (kCensusTriPairs .. kCensusMismatch, with full5
// also kCensusDp2 and kCensusGem).  Each pass has cursors of its own (zero).
// Returns 0, or -1 if a launch failed.
int census_rows_launch(const CensusArgs &c, const int64_t *cls_count,
                       int64_t max_out, bool cliques, char *slab,
                       size_t budget, int cus, hipStream_t s);

// Enqueues the sums over vertices and edges (needs t), with full5 also t_csr
// and tv.
int census_sums_launch(const CensusArgs &c, int cus, hipStream_t s);

// The 4-cycle pass's owners by kind (both ends in the window, the lower
// one below it, both below) and class (light, or by the bits of a counter);
// a kind's list holds its classes one after the other.
constexpr int kC4Kinds = 3;
enum C4Class : int { kC4Light, kC4Bits4, kC4Bits8, kC4Bits16, kC4Classes };
struct C4Plan {
  uint32_t count[kC4Kinds][kC4Classes] = {};
  int32_t *list[kC4Kinds] = {nullptr, nullptr, nullptr};
};
struct C4List {
  const int32_t *list = nullptr;
  uint32_t count = 0;
  unsigned *cursor = nullptr;
  uint32_t grab = 1;  // owners per queue access
};

// Raises the dynamic-LDS limit of the 4-cycle kernels (once per process).
int census_c4_init();
// Enqueues the window offsets of the rows (n entries), the classes of the
// owners (cls: n + winlo entries; the class sizes of each kind into fill,
// zeroed), and, with fill zeroed again, the lists of a plan that
// points at room for those sizes.
int census_c4_window(const CensusArgs &c, uint32_t *win, hipStream_t s);
int census_c4_classes(const CensusArgs &c, int8_t *cls, unsigned *fill,
                      hipStream_t s);
int census_c4_lists(const CensusArgs &c, const int8_t *cls, unsigned *fill,
                    const C4Plan &p, hipStream_t s);
// Enqueues the 4-cycle count into acc[kCensusC4], with full5 also
// kCensusBanner and kCensusCycEdgeT; dense_groups: workgroups c.wedges holds
// arrays for.  Returns 0, or -1 if a launch failed.
int census_c4_launch(const CensusArgs &c, const C4Plan &p, int dense_groups,
                     int cus, hipStream_t s);

}  // namespace mgpm

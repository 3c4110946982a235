// Triangle count against hub bitmaps (tc_hub.hip): what a graph keeps for
// it, and the launcher.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

namespace mgpm {

constexpr int32_t kHubIds = 65535;  // hubs: the highest-ranked vertices
constexpr int kHubChunk = 8;        // 16-bit ids per chunk (16 bytes)
constexpr uint32_t kHubRun = 16;    // partners per run (the blocks' unit)

// One partner of an owner: the chunks of its row that can hold a hit.
struct HubPartner {
  uint32_t base, chunks;
};

// One owner: its partners [beg, end) and its row's chunks.
struct HubOwner {
  uint32_t beg, end, base, chunks;
};

// Device view (relabelled graph: rank = id; hub z is the 16-bit number
// n - 1 - z).
struct TcHubPlan {
  const void *rows = nullptr;         // chunks of hub numbers, ascending per
                                      // row, padded with 65535; chunk 0 is
                                      // all padding
  const HubOwner *owner = nullptr;    // owners in id order
  const HubPartner *part = nullptr;   // partners by owner
  // Blocks of about equal cost: first partners (blocks + 1) and the first
  // owner each block can hold.
  const uint32_t *bound = nullptr;
  const uint32_t *start = nullptr;
  uint32_t n = 0, owners = 0, nparts = 0, blocks = 0;
  // Triangles without a hub: vertices with two or more heads below the hubs
  // (rest), and the DAG with the end of every row's heads below the hubs.
  const int32_t *rest = nullptr;
  uint32_t nrest = 0;
  const int64_t *drp = nullptr;
  const int32_t *dcol = nullptr;
  const uint32_t *split = nullptr;
};

// Queues of a launch: eight cache lines (next block, sum at word 2, finished
// workgroups at word 4) and a counter of finished queues, zero before a
// launch and left zero by it.
constexpr int kHubQueues = 8;
constexpr int kHubQueueStride = 32;  // words
constexpr int kHubQueueWords = kHubQueues * kHubQueueStride + 1;

// Where a count goes: added to *result (device), and with `host` set
// (pinned memory; needs the queue) moved there by the launch's end, *result
// left zero as it must be before it.
struct HubOut {
  unsigned long long *result = nullptr;
  unsigned *queue = nullptr;
  unsigned long long *host = nullptr;
};

// Enqueues the count.  Returns 0, or -1 if a launch failed.
int tc_hub_launch(const TcHubPlan &p, const HubOut &out, int cus,
                  hipStream_t s);

// The chunks that a plan names, added up in kHubSums places, kHubSumStride
// 64-bit words apart: of the partners, then of the owners' rows.
constexpr int kHubSums = 16;
constexpr int kHubSumStride = 16;

// Preparation: split (n) and the chunks of every row (n + 1, the last 0);
// the caller scans them into rowbase, then the rows, owners (flag and pos
// hold n + 1 entries, pos[n] their number; meta 16 bytes per vertex),
// partners and the rest list
// (its size into *nrest, zeroed), then the blocks (runs = ceil(nparts /
// kHubRun); cost and prefix hold runs + 1 entries; sums zeroed).
int tc_hub_counts(const int64_t *drp, const int32_t *dcol, int32_t n,
                  int32_t hublo, uint32_t *split, uint32_t *chunks,
                  hipStream_t s);
size_t tc_hub_scan_bytes(int32_t n, uint32_t runs);
int tc_hub_scan(const uint32_t *chunks, uint32_t *rowbase, int32_t n,
                void *tmp, size_t bytes, hipStream_t s);
int tc_hub_fill(const int64_t *rowptr, const int32_t *col,
                const int32_t *src, int64_t nnz, const int64_t *drp,
                const int32_t *dcol, const uint32_t *arc, int32_t n,
                const uint32_t *split, uint32_t *rowbase, void *rows,
                uint32_t *flag, uint32_t *pos, void *meta, HubOwner *owner,
                HubPartner *part, int32_t *rest, uint32_t *nrest, void *tmp,
                size_t bytes, int cus, hipStream_t s);
int tc_hub_blocks(const TcHubPlan &p, const uint32_t *owners, uint32_t runs,
                  unsigned long long *cost, unsigned long long *prefix,
                  void *tmp, size_t bytes, uint32_t *bound, uint32_t *start,
                  unsigned long long *sums, hipStream_t s);

}  // namespace mgpm

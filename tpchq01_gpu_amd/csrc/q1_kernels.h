// Internal interface between the C-ABI layer (q1_api.cpp) and the gfx950 kernels
// (q1_kernels.hip).  Host-only declarations; no HIP types leak into the public header.
#pragma once

#include <stdint.h>

#include "../../include/q1_hip.h"

namespace q1 {

// Value ranges of host columns.  Inside the TPC-H domain the narrow 32-bit kernels are exact;
// outside it the 64-bit kernels run.  Device tables are checked by launch_domain_check.
struct Domain {
  int64_t min_disc, max_disc, min_tax, max_tax, min_qty, max_qty, min_price, max_price;
};

bool domain_is_tpch(q1_layout layout, const Domain& d);

// The blocks of a launch over rows [row_begin, row_end) start at row_begin rounded down to
// a multiple of kRowAlign rows (rows before row_begin are masked off in the first block).
// 128 rows are a whole number of tiles of every layout and kernel, and of 128-byte lines of
// the 1-, 2- and 4-byte columns, so every wavefront load of a column starts on a line,
// wherever the range starts: a range starting at an arbitrary row otherwise made every
// load touch one line more and ran 10 % slower.
constexpr uint64_t kRowAlign = 128;
inline uint64_t align_rows_down(uint64_t row) { return row / kRowAlign * kRowAlign; }

// The tiles the host counts in (q1_launch's tuples_per_thread is a whole number of them), each
// split into the smaller tiles the kernels read.
template <int L>
constexpr int kHostTileRows = L == Q1_LAYOUT_REFERENCE ? 4 : L == Q1_LAYOUT_UNCOMPRESSED ? 8 : 16;

struct LaunchShape {
  uint32_t blocks, threads, tiles_per_thread;
};

// Spread merge.  Thousands of blocks adding into one 48-word table serialise on those
// words' atomics at the end of the grid; instead the blocks of a range merge into several
// tables, block b into table b mod their number, and the last block to finish folds the
// tables into the destination.  Tables are all zero before a launch and after it (the fold
// clears what it read), and must not be shared by launches that can overlap.
// A table takes up to 16 blocks while there are fewer than 64: the fold reads fewer tables,
// and 16 blocks' atomics on one table still pass within 0.5 us.  Kernel time with 64 / 32-4
// tables: 64 blocks 8.3 / 6.5 us, 128 blocks 8.7 / 6.7, 293 blocks 8.8 / 7.4; a table per 2,
// 4, 8 or 16 blocks: a 256-request batch 911, 908, 899, 896 us.
constexpr uint32_t kBlocksPerTable = 16;
constexpr uint32_t kSpreadTables = 64;      // the most tables a range merges into; a power of two
struct alignas(128) MergeTable {
  q1_device_aggregates sums;
  // Blocks that have merged here count in `merged`, the last of them in the range's first
  // table's tables_merged, so that no counter sees more than its share of a large grid.
  alignas(128) uint32_t merged;
  uint32_t tables_merged;
};
static_assert(sizeof(MergeTable) == 512, "sums and counters on cache lines of their own");
// How many tables the blocks of a range merge into (a power of two, at most the blocks).
inline uint32_t merge_tables(uint64_t blocks) {
  uint32_t t = 1;
  while (t < kSpreadTables && (uint64_t)t * kBlocksPerTable < blocks) t <<= 1;
  return t;
}

// The tables of a stream's scan launches.
struct MergeSet {
  MergeTable table[kSpreadTables];
  uint64_t clock_begin;       // device clock at the start of block 0
  uint64_t outside;           // number of the last domain check that found a value outside
};

// What a launch leaves in pinned host memory for a caller that waits for it.
struct HostResult {
  q1_device_aggregates sums;
  uint64_t clock_begin, clock_end;  // device clock at the start of block 0 and at the fold
  uint64_t outside;                 // domain check: whether a value lies outside the TPC-H domain
  uint64_t sequence;                // the launch's number, written after everything else
};
// How a kernel that leaves no sums tells the host that all its blocks are done: through the
// counters of a merge set, into a HostResult.
struct Completion {
  MergeSet* set;
  HostResult* host;           // as the device addresses it
  uint64_t sequence;
};

// Kernel-level request: accumulate rows [row_begin, row_end) of `cols` into `out`.
struct ScanArgs {
  q1_columns cols;          // device pointers
  uint64_t row_begin, row_end;
  int32_t cutoff_day;       // MonetDB day number (ignored for pushdown)
  q1_device_aggregates* out;
  // Set by launch_scan: without a merge set the blocks add into *out.  With one, block b
  // merges into the set's table b & table_mask, and the last block folds the tables into
  // *host (stored, with the clocks and `sequence`; host memory as the device addresses it),
  // or, when host is null, into *out (added; `sequence` then goes to *done if not null, once
  // the set is zero again).  A direct launch (launch_direct) leaves a record per block in
  // host[0 ..].
  uint32_t table_mask;
  MergeSet* set;
  HostResult* host;
  uint64_t* done;
  uint64_t sequence;
};

// Rows per lane for which the any-value kernel's LDS words are exact.
constexpr uint32_t any_value_lane_rows(q1_layout l) {
  return l == Q1_LAYOUT_COMPRESSED || l == Q1_LAYOUT_COMPRESSED_PUSHDOWN ? 128 : 256;
}

// Validate and complete a launch shape for `rows` rows (0 fields filled from defaults).
// fast: for the narrow kernels.  The any-value kernel takes no more than
// any_value_lane_rows rows per lane: a larger tuples_per_thread becomes more blocks.
q1_status make_shape(q1_placement placement, q1_layout layout, bool fast, const q1_launch* launch,
                     uint64_t row_begin, uint64_t row_end, LaunchShape* shape, const char** why);

// Smaller grids add straight into a device destination.  Device-scope atomics on one address
// from all compute units serialise, about 0.03 us per block; counting the blocks and the
// fold add a fixed 3 us.  Back-to-back q1_enqueue of 64 lanes x 64 rows blocks, direct /
// through a set: 64 blocks 12.2 / 14.8 us, 128 blocks 14.5 / 15.1, 176 blocks 16.1 / 15.1,
// 512 blocks 30.8 / 16.5, 4096 blocks 167 / 35.5.
constexpr uint32_t kSpreadMinBlocks = 144;

// The shortest fast launches of the LDS-table placement may instead leave each block's sums in a
// record of its own, a.host[block], for the host to add.  The line: 5 blocks 14.3 us per q1_run
// with a set, 12.4 with records; 10 blocks 13.7 / 12.8; 16 blocks 13.5 / 14.2.
constexpr uint32_t kDirectBlocks = 8;
bool can_launch_direct(q1_placement placement, q1_layout layout, bool fast, const LaunchShape& shape);
q1_status launch_direct(q1_layout layout, const ScanArgs& a, const LaunchShape& shape, void* stream);

// Where a scan's sums go.  host: stored into a.host (needs `set`; every grid merges through
// it).  Otherwise added into *a.out, through `set` when there is one and the grid has at
// least kSpreadMinBlocks blocks.
// fast: the rows lie inside the TPC-H domain.  Otherwise the any-value kernel runs.
q1_status launch_scan(q1_placement placement, q1_layout layout, bool fast, const ScanArgs& a,
                      const LaunchShape& shape, void* workspace, void* stream, MergeSet* set = nullptr);
// The workspace launch_scan needs: the global placement's per-block tables, which the any-value
// kernel does without.
uint64_t scan_workspace_bytes(q1_placement placement, bool fast, const LaunchShape& shape);

// Zero device memory (whole 64-bit words; a fill kernel, safe inside graph capture).
q1_status launch_zero(void* p, uint64_t bytes, void* stream);

// Device-side generator: rows [0, rows) of `layout` into the device columns.
q1_status launch_generate(q1_layout layout, uint64_t seed, uint64_t rows, const q1_columns& cols,
                          void* stream);

// Device-side domain check of a table's columns (rows > 0): host->outside, 0 before, becomes 1
// if any value lies outside the TPC-H domain.  *counted: `done` tells when; otherwise the
// kernel's end does.
q1_status launch_domain_check(q1_layout layout, const q1_columns& cols, uint64_t rows, const Completion& done,
                              void* stream, bool* counted);

// Copies up to 8 columns out of pinned host memory with one kernel.  src: as the device addresses
// it, on 8 bytes, as dst is; a column of 0 bytes is left out.  The kernel leaves its start in
// *clock_begin (host memory) if not null.
// Each of seven copies through the copy engine costs a few microseconds to start and to wait for:
// a whole q1_run_streaming call of 5,003 compressed rows takes 66 us with copies, 29 with this;
// 300,000 rows (2.8 MB) 160 / 77; 1M (9.4 MB) 275 / 198; 4M 770 / 697; 10M (94 MB) 1762 / 1682; 60M in two chunks 10100-10170 / 9930.
struct FetchArgs {
  const void* src[8];
  void* dst[8];
  uint64_t bytes[8];
  uint64_t* clock_begin;
};
q1_status launch_fetch(const FetchArgs& f, void* stream);

// Device-side pushdown producer: filter bitmap of a compressed ship_date column; the clocks and
// `sequence` in *host once it is there.
q1_status launch_build_filter(const uint16_t* ship, uint64_t rows, int32_t cutoff_day, uint32_t* filter,
                              HostResult* host, uint64_t sequence, void* stream);

// Batched scan: one launch over many requests of one layout, TPC-H domain.  The device
// buffer starts with a BatchHeader followed by `n` BatchDesc records and the n first blocks.
// Request r is cut into the blocks launch_scan would run over its rows alone (256 lanes x
// tiles_per_thread tiles each); the blocks of all requests, in request order, form one
// list of total_blocks entries.  A grid of G blocks works through the list with a
// fixed stride (block b runs entries b, b + G, b + 2G, ...).  The entries of a request merge
// through tables of its own as a scan's blocks do, and the last of them stores the sums into
// results[r], in pinned host memory.
struct BatchDesc {
  q1_columns cols;
  uint64_t row_begin, row_end;
  MergeTable* tables;         // table_mask + 1 of them, all zero
  uint32_t table_mask;
  uint32_t first_block;       // request's first entry in the block list
  uint32_t blocks;            // its entries
  int32_t cutoff_day;
};
struct BatchHeader {
  uint32_t n;                 // requests
  uint32_t with_rows;         // requests with entries
  uint32_t total_blocks;      // entries of the block list (below 2^31)
  uint32_t tiles_per_thread;  // tiles of layout_tile_rows rows per lane and entry
  uint64_t sequence;          // written to the done record at the end
  uint64_t pad[5];
};
// All zero before a batch and after it.
struct alignas(128) BatchControl {
  uint64_t clock_begin;       // device clock at the start of block 0
  uint32_t requests_done;
};
// What a batch leaves in pinned host memory after its results.
struct BatchDone {
  uint64_t clock_begin, clock_end;
  uint64_t sequence;          // written after everything else
};
constexpr uint32_t kBatchThreads = 256;
// The tables of a batch: a request with many blocks gets up to kSpreadTables of them while
// all fit (32 MiB).
constexpr uint32_t kBatchMaxTables = 65536;
uint32_t layout_tile_rows(q1_layout layout);
// The placement the batched kernel runs for a requested one (shared or in registers),
// the largest rows per lane it accepts for it, and how many of its blocks fit on a CU.
q1_placement batch_placement(q1_placement p);
uint32_t batch_max_lane_rows(q1_placement p);
uint32_t batch_blocks_per_cu(q1_layout layout, q1_placement p);
// The batched kernel over the list in dev_buffer (of n requests).
q1_status launch_batch(q1_layout layout, q1_placement placement, const BatchHeader* dev_buffer, uint32_t n,
                       BatchControl* control, q1_device_aggregates* results, BatchDone* done, uint32_t blocks,
                       void* stream);

// The scratch of q1_enqueue_noalloc (q1_noalloc.hip): a static per-device array holding the
// merge set and kNoallocWorkspaceBytes of per-block tables for the global placement.
// noalloc_setup looks up the array's address on `device` (which must be current) and
// clears its merge set, once per device; noalloc_launch_scan is launch_scan with the
// array as its scratch, refusing launches that need more (*why says which).
constexpr uint64_t kNoallocWorkspaceBytes = 8ull << 20;
constexpr const char* kNoallocRefused =
    "the launch needs more scratch than the static array holds (the global placement: at most 34952 blocks)";
q1_status noalloc_setup(int device, void* stream);
q1_status noalloc_launch_scan(int device, q1_placement placement, q1_layout layout, bool fast, const ScanArgs& a,
                              const LaunchShape& shape, void* stream, const char** why);

}  // namespace q1

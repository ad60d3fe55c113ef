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

struct LaunchShape {
  uint32_t blocks, threads, tiles_per_thread;
};

// Spread merge.  Thousands of blocks adding into one 48-word table serialise on those
// words' atomics at the end of the grid; instead block b of a launch merges into
// tables[b % kSpreadTables] of a merge set, and the last block to finish folds the tables
// into the destination.  A set is all zero before a launch and after it (the fold clears
// what it read), and must not be shared by launches that can overlap.
constexpr uint32_t kSpreadTables = 64;      // power of two
struct MergeSet {
  q1_device_aggregates tables[kSpreadTables];
  // Blocks that have merged: those of one table (the blocks b with the same b mod 64) count
  // in finished[b % 64], each on a cache line of its own, and the last of them in
  // tables_finished, so that no counter sees more than a 64th of a large grid.
  struct alignas(128) Count {
    uint32_t n;
  } finished[kSpreadTables];
  Count tables_finished;
  uint64_t clock_begin;       // device clock at the start of block 0
};

// What a launch leaves in pinned host memory for a caller that waits for it.
struct HostResult {
  q1_device_aggregates sums;
  uint64_t clock_begin, clock_end;  // device clock at the start of block 0 and at the fold
  uint64_t sequence;                // the launch's number, written after everything else
};

// Kernel-level request: accumulate rows [row_begin, row_end) of `cols` into `out`.
struct ScanArgs {
  q1_columns cols;          // device pointers
  uint64_t row_begin, row_end;
  int32_t cutoff_day;       // MonetDB day number (ignored for pushdown)
  q1_device_aggregates* out;
  // Set by launch_scan: block b merges into out[b & out_mask]; with a merge set, `out` are
  // the set's tables and the last block folds them into *dest (added), or, when dest is
  // null, into *host (stored, with the clocks and `sequence`; host memory as the device
  // addresses it).
  uint32_t out_mask;
  MergeSet* set;
  q1_device_aggregates* dest;
  HostResult* host;
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

// Where a scan's sums go.  host: stored into a.host (needs `set`; every grid merges through
// it).  Otherwise added into *a.out, through `set` when there is one and the grid has at
// least kSpreadMinBlocks blocks.
// fast: the rows lie inside the TPC-H domain.  Otherwise the any-value kernel runs.
q1_status launch_scan(q1_placement placement, q1_layout layout, bool fast, const ScanArgs& a,
                      const LaunchShape& shape, void* workspace, void* stream, MergeSet* set = nullptr);
uint64_t scan_workspace_bytes(q1_placement placement, const LaunchShape& shape);

// Zero device aggregate tables or a merge set (a fill kernel, safe inside graph capture).
q1_status launch_zero(q1_device_aggregates* table, uint32_t count, void* stream);
q1_status launch_zero(MergeSet* set, void* stream);

// Device-side generator: rows [0, rows) of `layout` into the device columns.
q1_status launch_generate(q1_layout layout, uint64_t seed, uint64_t rows, const q1_columns& cols,
                          void* stream);

// Device-side domain check of a table's columns: *outside (device-visible) is set to 1 if any
// value lies outside the TPC-H domain, and not written otherwise.
q1_status launch_domain_check(q1_layout layout, const q1_columns& cols, uint64_t rows, uint32_t* outside,
                              void* stream);

// Device-side pushdown producer: filter bitmap of a compressed ship_date column.
q1_status launch_build_filter(const uint16_t* ship, uint64_t rows, int32_t cutoff_day,
                              uint32_t* filter, void* stream);

// Batched scan: one launch over many requests of one layout, TPC-H domain.  The device
// buffer starts with a BatchHeader followed by `n` BatchDesc records.  Request r is cut
// into the blocks launch_scan would run over its rows alone (256 lanes x
// tiles_per_thread tiles each); the blocks of all requests, in request order, form one
// list of total_blocks entries.  A resident grid of G blocks works through the list with a
// fixed stride (block b runs entries b, b + G, b + 2G, ...).  Entry v of request r merges
// into spread table v mod 64 of the request (spread + 64 r) when r < spread_requests, and
// into outs[r] otherwise; after the kernel, fold_spread (one block per request with spread
// tables) adds each request's 64 tables into outs[r] and clears them.
struct BatchDesc {
  q1_columns cols;
  uint64_t row_begin, row_end;
  uint64_t block_begin;       // request's first entry in the block list
  int32_t cutoff_day;
  uint32_t pad;
};
struct BatchHeader {
  uint64_t n;                 // requests
  uint64_t total_blocks;      // entries of the block list (below 2^31)
  uint32_t tiles_per_thread;  // tiles of layout_tile_rows rows per lane and entry
  uint32_t spread_requests;   // requests 0 .. spread_requests-1 merge through spread tables
  uint64_t pad[5];
};
constexpr uint32_t kBatchThreads = 256;
// Requests of a batch that get spread tables: 64 x 384 B each, at most 24 MiB.
constexpr uint32_t kBatchSpreadRequests = 1024;
uint32_t layout_tile_rows(q1_layout layout);
// The placement the batched kernel runs for a requested one (shared or in registers),
// the largest rows per lane it accepts for it, and how many of its blocks fit on a CU.
q1_placement batch_placement(q1_placement p);
uint32_t batch_max_lane_rows(q1_placement p);
uint32_t batch_blocks_per_cu(q1_layout layout, q1_placement p);
// The batched kernel over the list in dev_buffer, then, with `spread` (spread_requests x
// kSpreadTables tables, all zero), the fold of the first spread_requests requests' tables:
// added into outs, or, with store_results (a device-visible pointer to the results in
// pinned host memory, when every request has spread tables), stored there directly.
q1_status launch_batch(q1_layout layout, q1_placement placement, BatchHeader* dev_buffer,
                       q1_device_aggregates* outs, q1_device_aggregates* spread, uint32_t spread_requests,
                       q1_device_aggregates* store_results, uint32_t blocks, uint32_t threads, void* stream);
// The host function launch_batch launches for (layout, placement), e.g. to find its node in
// a captured graph.
const void* batch_kernel_function(q1_layout layout, q1_placement placement);

// The scratch of q1_enqueue_noalloc (q1_noalloc.hip): a static per-device array holding the
// spread tables and kNoallocWorkspaceBytes of per-block tables for the global placement.
// noalloc_setup looks up the array's address on `device` (which must be current) and
// clears its spread tables, once per device; noalloc_launch_scan is launch_scan with the
// array as its scratch, refusing launches that need more (*why says which).
constexpr uint64_t kNoallocWorkspaceBytes = 8ull << 20;
q1_status noalloc_setup(int device, void* stream);
q1_status noalloc_launch_scan(int device, q1_placement placement, q1_layout layout, bool fast, const ScanArgs& a,
                              const LaunchShape& shape, void* stream, const char** why);

}  // namespace q1

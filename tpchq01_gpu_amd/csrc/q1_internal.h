// Internal host-side state shared by the C-ABI translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <mutex>
#include <string>
#include <unordered_set>
#include <vector>

#include "../../include/q1_hip.h"
#include "q1_kernels.h"

struct q1_table {
  q1_ctx* ctx = nullptr;
  q1_layout layout = Q1_LAYOUT_COMPRESSED;
  uint64_t rows = 0;
  q1_columns dev{};
  void* owned[8] = {};           // allocations this table frees
  bool fast = false;             // inside the TPC-H value domain
  uint64_t device_bytes = 0;
  int32_t filter_cutoff = 0;     // pushdown tables: the cutoff their bitmap encodes
  uint64_t filter_bytes = 0;     // ... and what is allocated for it
  // Whether work on other streams than the context's may read the table (its pointers were
  // handed out, or a server got a request on it).
  mutable std::atomic<bool> shared{false};
};

// q1_run_streaming's chunk rows and stream count when neither the caller nor the tuning
// table gives them.
constexpr uint64_t kStreamChunkRows = 1ull << 24;
constexpr int kStreamCount = 4;

namespace q1 {
struct BatchBuffers;
struct StreamState;     // q1_stream.cpp: the host-resident streaming pipeline
// Merge sets for launches on callers' streams: each launch in flight has one of its own, so
// nothing orders the streams (or a destroyed stream and one made at its address).  A launch's
// last block writes the launch's number to its set's word in `done`, and a set is free again
// once the number is there.
constexpr size_t kPoolSets = 256;
struct SetPool {
  MergeSet* sets = nullptr;       // kPoolSets
  uint64_t* done = nullptr;       // pinned words
  uint64_t* done_dev = nullptr;   // ... as the device addresses them
  uint64_t last[kPoolSets] = {};  // number of the last launch given the set
  uint64_t sequence = 0;
  size_t cursor = 0;
  bool stalled = false;           // the last wait for a set was in vain
};
// The filter bitmap of a freed table, kept for the next q1_build_filter (a query per cutoff
// builds, reads and frees one: hipMalloc and hipFree were 40 of the 160 us of such a query over
// 60M rows).  At most kSpareFilterBytes (a bitmap of 512M rows), given back when an allocation
// of the library on the device fails (device_malloc) and with the context.
constexpr uint64_t kSpareFilterBytes = 64ull << 20;
struct SpareFilter {
  void* p = nullptr;
  uint64_t bytes = 0;
};
// A launch shape tuned on ranges of `rows` rows ("launch_at" lines of the tuning file).
struct SizedLaunch {
  uint64_t rows;
  uint32_t threads_per_block, tuples_per_thread;
};
}

struct q1_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  // Work may be on the stream that no call has waited for: q1_enqueue's since the last wait, or
  // the caller's own once it has got the stream (q1_stream).
  bool queued = false;
  std::atomic<bool> stream_out{false};
  hipEvent_t ev_begin = nullptr, ev_end = nullptr, ev_h2d_begin = nullptr, ev_h2d_end = nullptr;
  q1::HostResult* h_result = nullptr;      // pinned, kDirectBlocks: what q1_run's kernel leaves (and
                                           // a copy's start clock behind them)
  uint32_t results = 0;                    // records that the last launch leaves
  q1::HostResult* d_result = nullptr;      // ... as the device addresses it
  uint64_t sequence = 0;                   // number of the last launch that wrote h_result
  int32_t clock_khz = 0;                   // rate of the device clock in h_result
  q1_device_aggregates* d_aggr = nullptr;  // the table q1_run_streaming's chunks add into
  q1_device_aggregates* h_aggr = nullptr;  // pinned host copy
  void* workspace = nullptr;
  uint64_t workspace_bytes = 0;
  q1_timing last{};
  std::string error;
  int32_t compute_units = 0;
  q1_launch tuning[4][5]{};                // [layout][placement]
  // Shapes tuned at several row counts, ascending; a launch takes the one tuned nearest its
  // own row count (by ratio) and falls back to tuning[][] when there is none.
  std::vector<q1::SizedLaunch> tuning_at[4][5];
  // The batched kernel's tuned shape per [layout][placement]: num_blocks holds blocks per
  // compute unit, tuples_per_thread rows per lane; zero = not tuned.
  q1_launch batch_tuning[4][5]{};
  // The host-resident streaming pipeline's tuned chunk rows and stream count per layout
  // (0 = not tuned: kStreamChunkRows, kStreamCount).
  uint64_t stream_chunk_rows[4] = {};
  int stream_count[4] = {};
  q1_placement best[4] = {Q1_PLACE_IN_REGISTERS, Q1_PLACE_IN_REGISTERS, Q1_PLACE_IN_REGISTERS,
                          Q1_PLACE_IN_REGISTERS};
  q1::BatchBuffers* batch = nullptr;       // q1_run_batch's buffers
  q1::StreamState* streaming = nullptr;    // cached staging buffers and streams of q1_run_streaming
  q1::MergeSet* set = nullptr;             // merge set of the context stream
  q1::SetPool pool;                        // merge sets of launches on callers' streams
  q1::SpareFilter spare;                   // a freed table's filter bitmap, for the next one
  std::mutex spare_lock;                   // guards it: server threads allocate without `lock`
  std::unordered_set<q1_table*> tables;    // live tables (released device memory at shutdown)
  std::mutex lock;                         // serialises calls that share the context stream
};

namespace q1 {
q1_status fail(q1_ctx* ctx, q1_status s, const std::string& why);
q1_status hip_fail(q1_ctx* ctx, hipError_t e, const char* what);
q1_placement resolve_placement(q1_ctx* ctx, q1_layout layout, q1_placement p);
// Fills a launch from the caller's, with the tuned values where it leaves them 0.  fast: for
// the narrow kernels; launches that run the any-value kernel take that kernel's own shape
// instead, since it runs every placement alike.  table: the columns are a table's.
void resolve_launch(q1_ctx* ctx, q1_layout layout, q1_placement p, bool fast, uint64_t rows, const q1_launch* in,
                    q1_launch* out, bool table = true);
inline bool in_domain_flag(const q1_launch* l) { return l && (l->flags & Q1_LAUNCH_ASSUME_TPCH_DOMAIN); }
uint64_t algorithmic_bytes(q1_layout layout, uint64_t rows);
// hipMalloc that gives the spare bitmap back when there is no more memory; needs no lock held.
hipError_t device_malloc(q1_ctx* ctx, void** p, uint64_t bytes);
q1_status ensure_workspace(q1_ctx* ctx, uint64_t bytes);
// launch_scan for q1_enqueue: with the context's merge set on the context stream, one of the
// pool's on a caller's, none on a stream that is being captured.
q1_status scan_on(q1_ctx* ctx, q1_placement placement, q1_layout layout, bool fast, const ScanArgs& a,
                  const LaunchShape& shape, void* stream);
// launch_scan on the context stream with the sums going to ctx->h_result, and the wait for
// them: fills *out and returns the kernel's device time in *kernel_ms.  A launch with no
// blocks leaves zeros.
q1_status scan_to_host(q1_ctx* ctx, q1_placement placement, q1_layout layout, bool fast, ScanArgs a,
                       const LaunchShape& shape);
q1_status wait_result(q1_ctx* ctx, q1_result* out, double* kernel_ms, uint64_t* begin = nullptr);
// Waits until a launch on the context stream has written `sequence` to *word (pinned).
q1_status wait_sequence(q1_ctx* ctx, const uint64_t* word, uint64_t sequence);
double clock_ms(const q1_ctx* ctx, uint64_t begin, uint64_t end);

// The buffers of batched launches on one stream, kept between launches and grown when a
// larger batch comes: the descriptors (pinned and on the device), the results (pinned,
// written by the kernel) and the requests' merge tables.
struct BatchBuffers {
  uint32_t capacity = 0;                    // requests
  uint32_t tables = 0;
  BatchHeader* h_buf = nullptr;             // header, descriptors, first blocks
  BatchHeader* d_buf = nullptr;
  q1_device_aggregates* h_out = nullptr;    // results, then a BatchDone
  q1_device_aggregates* h_out_dev = nullptr;  // ... as the device addresses them
  BatchControl* control = nullptr;          // on the device, the tables behind it
  uint64_t sequence = 0;                    // of the last launch
  const BatchDone* done() const { return reinterpret_cast<const BatchDone*>(h_out + capacity); }
};
void batch_free(BatchBuffers* b);
// Launches n requests of one layout inside the domain on `stream` (whose earlier launches with
// these buffers have finished): results in b->h_out[0 .. n-1] once b->done() holds
// b->sequence, or the stream has got there.  lane_rows and grid of 0 take the tuned rows per
// lane, less for a batch too small to fill the chip, and a block per entry up to the tuned
// grid.  *lane_rows_planned, *grid_planned: the tuned shape or the caller's.  *why: what
// failed (of ctx only the spare bitmap is changed: the server's threads launch without its lock).
q1_status batch_launch(q1_ctx* ctx, BatchBuffers* b, const q1_request* reqs, uint32_t n, q1_placement placement,
                       uint32_t lane_rows, uint32_t grid, hipStream_t stream, uint32_t* lane_rows_planned,
                       uint32_t* grid_planned, const char** why);
void stream_state_release(q1_ctx* ctx);
}  // namespace q1

// q1_run_batch: many filter-aggregate requests (uneven row counts, their own cutoffs) in
// one launch of the batched kernel: the descriptors are copied to the device, the kernel runs
// every request's blocks, and the last block of each request stores its result straight into
// the pinned host results, with a done record after all of them that the caller waits for.
// Two commands on the stream and no per-batch set-up: a batch of any size runs at once in
// the same buffers.
#include <algorithm>
#include <chrono>
#include <cstring>
#include <vector>

#include "q1_internal.h"

namespace q1 {

void batch_free(BatchBuffers* b) {
  if (b->h_buf) (void)hipHostFree(b->h_buf);
  if (b->h_out) (void)hipHostFree(b->h_out);
  if (b->d_buf) (void)hipFree(b->d_buf);
  if (b->control) (void)hipFree(b->control);
  *b = BatchBuffers{};
}

static uint64_t buf_bytes(uint32_t n) {
  return sizeof(BatchHeader) + (uint64_t)n * (sizeof(BatchDesc) + sizeof(uint32_t));
}

// Rows per lane: the autotuner's batch value for the layout and placement, else the
// scan's tuned value, within the batched kernel's limit.
static uint32_t batch_lane_rows(q1_ctx* ctx, q1_layout layout, q1_placement p) {
  const uint32_t most = batch_max_lane_rows(p);
  const uint32_t batch_tuned = ctx->batch_tuning[layout][p].tuples_per_thread;
  if (batch_tuned >= 16 && batch_tuned <= most) return batch_tuned / 16 * 16;
  const uint32_t tuned = ctx->tuning[layout][p].tuples_per_thread;
  return tuned >= 16 && tuned <= most ? tuned / 16 * 16 : std::min<uint32_t>(256, most);
}

static uint32_t compute_units(const q1_ctx* ctx) { return (uint32_t)(ctx->compute_units > 0 ? ctx->compute_units : 256); }

// Grid: the autotuner's blocks per compute unit for the layout and placement, else as many
// blocks as are resident at once.
static uint32_t batch_default_blocks(q1_ctx* ctx, q1_layout layout, q1_placement p) {
  const uint32_t per_cu = ctx->batch_tuning[layout][p].num_blocks;
  return compute_units(ctx) * (per_cu ? per_cu : batch_blocks_per_cu(layout, p));
}

static uint64_t request_blocks(const q1_request& r, uint32_t lane_rows) {
  if (r.row_count == 0) return 0;
  const uint64_t trows = layout_tile_rows(r.table->layout);
  const uint64_t tiles = (r.row_begin + r.row_count + trows - 1) / trows - align_rows_down(r.row_begin) / trows;
  const uint64_t per_block = (uint64_t)kBatchThreads * (lane_rows / trows);
  return (tiles + per_block - 1) / per_block;
}

// Makes room for n requests and `tables` merge tables.  The stream's earlier launches with
// the buffers have finished.
static q1_status reserve(q1_ctx* ctx, BatchBuffers* b, uint32_t n, uint32_t tables, hipStream_t stream,
                         const char** why) {
  auto give_up = [&](q1_status s, const char* text) {
    *why = text;
    return s;
  };
  if (b->capacity < n) {
    uint32_t cap = 16;
    while (cap < n) cap <<= 1;
    if (b->h_buf) (void)hipHostFree(b->h_buf);
    if (b->h_out) (void)hipHostFree(b->h_out);
    if (b->d_buf) (void)hipFree(b->d_buf);
    b->h_buf = b->d_buf = nullptr;
    b->h_out = b->h_out_dev = nullptr;
    b->capacity = 0;
    const uint64_t out_bytes = (uint64_t)cap * sizeof(q1_device_aggregates) + sizeof(BatchDone);
    if (hipHostMalloc(&b->h_buf, buf_bytes(cap), hipHostMallocDefault) != hipSuccess ||
        hipHostMalloc(&b->h_out, out_bytes, hipHostMallocMapped) != hipSuccess ||
        hipHostGetDevicePointer((void**)&b->h_out_dev, b->h_out, 0) != hipSuccess ||
        device_malloc(ctx, (void**)&b->d_buf, buf_bytes(cap)) != hipSuccess)
      return give_up(Q1_ENOMEM, "batch buffers could not be allocated");
    std::memset((void*)b->h_out, 0, out_bytes);
    b->capacity = cap;
  }
  if (!b->control || b->tables < tables) {
    uint32_t t = 64;
    while (t < tables) t <<= 1;
    if (b->control) (void)hipFree(b->control);
    b->control = nullptr;
    b->tables = 0;
    const uint64_t bytes = sizeof(BatchControl) + (uint64_t)t * sizeof(MergeTable);
    if (device_malloc(ctx, (void**)&b->control, bytes) != hipSuccess)
      return give_up(Q1_ENOMEM, "batch tables could not be allocated");
    if (launch_zero(b->control, bytes, stream) != Q1_OK) {
      (void)hipFree(b->control);
      b->control = nullptr;
      return give_up(Q1_EDEVICE, "clearing the batch tables failed");
    }
    b->tables = t;
  }
  return Q1_OK;
}

q1_status batch_launch(q1_ctx* ctx, BatchBuffers* b, const q1_request* reqs, uint32_t n, q1_placement placement,
                       uint32_t lane_rows, uint32_t grid, hipStream_t stream, uint32_t* lane_rows_planned,
                       uint32_t* grid_planned, const char** why) {
  auto give_up = [&](q1_status s, const char* text) {
    *why = text;
    return s;
  };
  const q1_layout layout = reqs[0].table->layout;
  placement = batch_placement(placement);
  *lane_rows_planned = lane_rows ? lane_rows : batch_lane_rows(ctx, layout, placement);
  *grid_planned = grid ? grid : batch_default_blocks(ctx, layout, placement);
  if (!lane_rows) {
    // The tuned rows per lane, halved while the batch has fewer than 4 blocks per compute
    // unit, so that a small batch spreads over the chip too.
    lane_rows = *lane_rows_planned;
    uint64_t rows = 0;
    for (uint32_t i = 0; i < n; i++) rows += reqs[i].row_count;
    while (lane_rows > 16 && rows < 4ull * compute_units(ctx) * kBatchThreads * lane_rows)
      lane_rows = std::max<uint32_t>(16, (lane_rows / 2) & ~15u);
  }
  // A request's tables: as a scan of its blocks would have, fewer for all while the batch
  // would need more than kBatchMaxTables.
  uint64_t entries = 0, tables = 0;
  uint32_t most = kSpreadTables;
  for (;; most >>= 1) {
    entries = tables = 0;
    for (uint32_t i = 0; i < n; i++) {
      const uint64_t blocks = request_blocks(reqs[i], lane_rows);
      entries += blocks;
      tables += std::min(merge_tables(blocks), most);
    }
    if (tables <= kBatchMaxTables || most == 1) break;
  }
  if (entries >= (1ull << 31)) return give_up(Q1_EINVAL, "batch too large (2^31 blocks of rows)");
  const q1_status s = reserve(ctx, b, n, (uint32_t)tables, stream, why);
  if (s != Q1_OK) return s;
  BatchDesc* d = reinterpret_cast<BatchDesc*>(b->h_buf + 1);
  uint32_t* first = reinterpret_cast<uint32_t*>(d + n);
  MergeTable* next = reinterpret_cast<MergeTable*>(b->control + 1);
  uint32_t block = 0, with_rows = 0;
  for (uint32_t i = 0; i < n; i++) {
    const q1_request& r = reqs[i];
    const q1_table* t = r.table;
    const uint32_t blocks = (uint32_t)request_blocks(r, lane_rows);
    const uint32_t own = std::min(merge_tables(blocks), most);
    d[i].cols = t->dev;
    d[i].row_begin = r.row_begin;
    d[i].row_end = r.row_begin + r.row_count;
    d[i].tables = next;
    d[i].table_mask = own - 1;
    d[i].first_block = first[i] = block;
    d[i].blocks = blocks;
    d[i].cutoff_day = t->layout == Q1_LAYOUT_COMPRESSED_PUSHDOWN ? t->filter_cutoff : r.cutoff_day;
    next += own;
    block += blocks;
    if (blocks)
      with_rows++;
    else
      std::memset((void*)&b->h_out[i], 0, sizeof(q1_device_aggregates));
  }
  b->sequence++;
  BatchHeader* h = b->h_buf;
  *h = BatchHeader{};
  h->n = n;
  h->with_rows = with_rows;
  h->total_blocks = block;
  h->tiles_per_thread = lane_rows / layout_tile_rows(layout);
  h->sequence = b->sequence;
  if (!with_rows) {
    BatchDone* done = const_cast<BatchDone*>(b->done());
    *done = BatchDone{0, 0, b->sequence};
    return Q1_OK;
  }
  if (!grid) grid = std::min(block, *grid_planned);
  if (hipMemcpyAsync(b->d_buf, b->h_buf, buf_bytes(n), hipMemcpyHostToDevice, stream) != hipSuccess)
    return give_up(Q1_EDEVICE, "copying the batch descriptors failed");
  BatchDone* done = reinterpret_cast<BatchDone*>(b->h_out_dev + b->capacity);
  if (launch_batch(layout, placement, b->d_buf, n, b->control, b->h_out_dev, done, grid, stream) != Q1_OK) {
    (void)hipStreamSynchronize(stream);  // the copy still reads the pinned descriptors
    return give_up(Q1_EDEVICE, "batch kernel launch failed");
  }
  return Q1_OK;
}

}  // namespace q1

using namespace q1;

extern "C" q1_status q1_run_batch(q1_ctx* ctx, const q1_request* reqs, uint32_t n, const q1_launch* launch,
                                  q1_result* outs) {
  if (!ctx || (!reqs && n) || (!outs && n)) return fail(ctx, Q1_EINVAL, "bad argument");
  if (n == 0) return Q1_OK;
  if (n > (1u << 16)) return fail(ctx, Q1_EINVAL, "at most 65536 requests per batch");
  for (uint32_t i = 0; i < n; i++) {
    const q1_table* t = reqs[i].table;
    if (!t) return fail(ctx, Q1_EINVAL, "request without a table");
    if (reqs[i].row_begin > t->rows || reqs[i].row_count > t->rows - reqs[i].row_begin)
      return fail(ctx, Q1_EINVAL, "request row range outside its table");
  }
  try {
    // One launch needs one layout and the TPC-H domain; any other mix runs
    // request by request (same results, no batching).
    const q1_layout layout = reqs[0].table->layout;
    bool batchable = true;
    for (uint32_t i = 0; i < n; i++)
      batchable = batchable && reqs[i].table->layout == layout && reqs[i].table->fast;
    if (!batchable) {
      for (uint32_t i = 0; i < n; i++) {
        const q1_status s = q1_run(ctx, reqs[i].table, reqs[i].row_begin, reqs[i].row_count, reqs[i].cutoff_day,
                                   Q1_PLACE_AUTO, nullptr, &outs[i]);
        if (s != Q1_OK) return s;
      }
      return Q1_OK;
    }
    std::lock_guard<std::mutex> g(ctx->lock);
    const q1_placement p = batch_placement(ctx->best[layout]);
    // The batched kernel runs 256-thread blocks; the grid and rows per lane are tunable.
    if (launch && launch->threads_per_block && launch->threads_per_block != kBatchThreads)
      return fail(ctx, Q1_EINVAL, "the batched kernel runs 256 threads per block");
    const uint32_t lane_rows = launch ? launch->tuples_per_thread : 0, grid = launch ? launch->num_blocks : 0;
    if (lane_rows % 16 != 0 || lane_rows > batch_max_lane_rows(p))
      return fail(ctx, Q1_EINVAL,
                  "batched tuples_per_thread must be a multiple of 16, at most 256 (shared placement) or 16384");
    // The grid's work-items (blocks x 256) must stay below 2^32.
    if (grid >= (1u << 24)) return fail(ctx, Q1_EINVAL, "batched num_blocks must be below 2^24");
    if (!ctx->batch) ctx->batch = new BatchBuffers();
    BatchBuffers* b = ctx->batch;
    const auto w0 = std::chrono::steady_clock::now();
    uint32_t plan_rows = 0, plan_grid = 0;
    const char* why = "";
    q1_status s = batch_launch(ctx, b, reqs, n, p, lane_rows, grid, ctx->stream, &plan_rows, &plan_grid, &why);
    if (s != Q1_OK) return fail(ctx, s, why);
    // a batch without rows has launched nothing to wait for
    if (__atomic_load_n(&b->done()->sequence, __ATOMIC_ACQUIRE) != b->sequence)
      s = wait_sequence(ctx, &b->done()->sequence, b->sequence);
    if (s != Q1_OK) {
      // The tables may hold partial sums: the next call makes new ones.
      batch_free(b);
      return s;
    }
    uint64_t rows = 0;
    for (uint32_t i = 0; i < n; i++) {
      q1_aggregates_to_result(&b->h_out[i], &outs[i]);
      rows += reqs[i].row_count;
    }
    ctx->last = q1_timing{};
    ctx->last.kernel_ms = clock_ms(ctx, b->done()->clock_begin, b->done()->clock_end);
    ctx->last.wall_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - w0).count();
    ctx->last.rows = rows;
    ctx->last.bytes_read = algorithmic_bytes(layout, rows);
    ctx->last.num_blocks = plan_grid;
    ctx->last.threads_per_block = kBatchThreads;
    ctx->last.tuples_per_thread = plan_rows;
    ctx->last.placement = (uint32_t)p;
    return Q1_OK;
  } catch (const std::exception& e) {
    return fail(ctx, Q1_ENOMEM, e.what());
  }
}

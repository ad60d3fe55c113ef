// The CPU/GPU split (src/main.cu:513-550 with the CoProc of src/cpu.h:23-38) and the
// host-resident streaming pipeline (src/main.cu:567-724): chunks of host columns are
// copied into per-stream device staging buffers and aggregated by the scan kernel on the
// same stream, so copies of one chunk overlap kernels of others; all launches add into
// one device table.  A call of one chunk runs on the context stream alone.
#include <algorithm>
#include <chrono>
#include <cstring>
#include <thread>
#include <vector>

#include "q1_internal.h"

namespace q1 {

struct StreamState {
  q1_layout layout = Q1_LAYOUT_COMPRESSED;
  uint64_t chunk_rows = 0;
  int streams = 0;
  std::vector<hipStream_t> s;
  std::vector<hipEvent_t> done;
  std::vector<q1_columns> staging;
  std::vector<void*> allocs;
  std::vector<void*> workspace;
  std::vector<MergeSet*> set;   // each stream's launches merge through its own
  uint64_t workspace_bytes = 0;
};

static void stream_state_free(StreamState* st) {
  if (!st) return;
  for (hipStream_t s : st->s) (void)hipStreamSynchronize(s);
  for (void* p : st->allocs) (void)hipFree(p);
  for (void* p : st->workspace)
    if (p) (void)hipFree(p);
  for (MergeSet* p : st->set) (void)hipFree(p);
  for (hipEvent_t e : st->done) (void)hipEventDestroy(e);
  for (hipStream_t s : st->s) (void)hipStreamDestroy(s);
  delete st;
}

void stream_state_release(q1_ctx* ctx) {
  stream_state_free(ctx->streaming);
  ctx->streaming = nullptr;
}

// Whether a kernel can read the bytes at p: pinned memory, at the address the host uses, and all of
// them in the one range that holds the first (a buffer may be pinned in pieces, with pageable
// memory between them).
static bool kernel_reads(const void* p, uint64_t bytes) {
  if ((uintptr_t)p % 8) return false;
  hipPointerAttribute_t a{};
  hipDeviceptr_t base = nullptr;
  size_t size = 0;
  if (hipPointerGetAttributes(&a, p) != hipSuccess || a.type != hipMemoryTypeHost || a.devicePointer != p ||
      hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  const uint64_t offset = (uint64_t)((const char*)p - (const char*)base);
  return (const char*)p >= (const char*)base && offset <= size && bytes <= size - offset;
}

static void column_bytes_local(q1_layout layout, uint64_t n, uint64_t b[8]) {
  q1_layout_column_bytes(layout, n, b);
}

// The context's cached pipeline for (layout, chunk_rows, streams), rebuilt when those
// change.  A pipeline is stored only once all of its streams, events and staging buffers
// exist, so a failed build leaves nothing half-made behind.
static q1_status prepare(q1_ctx* ctx, q1_layout layout, uint64_t chunk_rows, int streams, StreamState** out) {
  StreamState* cur = ctx->streaming;
  if (cur && cur->layout == layout && cur->chunk_rows == chunk_rows && cur->streams == streams) {
    *out = cur;
    return Q1_OK;
  }
  stream_state_free(cur);
  ctx->streaming = nullptr;
  StreamState* st = new StreamState();
  auto give_up = [&](q1_status code, const char* why) {
    stream_state_free(st);
    return fail(ctx, code, why);
  };
  uint64_t b[8];
  column_bytes_local(layout, chunk_rows, b);
  for (int i = 0; i < streams; i++) {
    hipStream_t s;
    hipEvent_t e;
    if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess) return give_up(Q1_EDEVICE, "stream creation failed");
    st->s.push_back(s);
    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return give_up(Q1_EDEVICE, "event creation failed");
    st->done.push_back(e);
    MergeSet* set = nullptr;
    if (device_malloc(ctx, (void**)&set, sizeof(MergeSet)) != hipSuccess)
      return give_up(Q1_ENOMEM, "staging allocation failed");
    st->set.push_back(set);
    if (launch_zero(set, sizeof(MergeSet), s) != Q1_OK) return give_up(Q1_EDEVICE, "zero kernel failed");
    q1_columns c{};
    const void** slots[8] = {&c.ship_date, &c.quantity, &c.extended_price, &c.discount,
                             &c.tax, &c.return_flag, &c.line_status, &c.filter};
    for (int k = 0; k < 8; k++) {
      if (!b[k]) continue;
      void* p = nullptr;
      if (device_malloc(ctx, &p, b[k]) != hipSuccess) return give_up(Q1_ENOMEM, "staging allocation failed");
      st->allocs.push_back(p);
      *slots[k] = p;
    }
    st->staging.push_back(c);
    st->workspace.push_back(nullptr);
  }
  st->layout = layout;
  st->chunk_rows = chunk_rows;
  st->streams = streams;
  ctx->streaming = st;
  *out = st;
  return Q1_OK;
}

}  // namespace q1

using namespace q1;

extern "C" {

q1_status q1_run_streaming(q1_ctx* ctx, q1_layout layout, const q1_columns* host, uint64_t rows, int32_t cutoff_day,
                           q1_placement placement, const q1_launch* launch, uint64_t chunk_rows, int num_streams,
                           q1_result* out) {
  if (!ctx || !host || !out || layout < Q1_LAYOUT_REFERENCE || layout > Q1_LAYOUT_COMPRESSED_PUSHDOWN)
    return fail(ctx, Q1_EINVAL, "bad argument");
  // 0 = the autotuning table's value for the layout ("streaming" lines), else 16M rows / 4 streams
  if (chunk_rows == 0) chunk_rows = ctx->stream_chunk_rows[layout] ? ctx->stream_chunk_rows[layout] : kStreamChunkRows;
  if (num_streams == 0) num_streams = ctx->stream_count[layout] ? ctx->stream_count[layout] : kStreamCount;
  if (chunk_rows % 32 || num_streams < 1 || num_streams > 16)
    return fail(ctx, Q1_EINVAL, "chunk_rows must be a positive multiple of 32 and streams in [1, 16]");
  try {
    std::lock_guard<std::mutex> g(ctx->lock);
    const q1_placement p = resolve_placement(ctx, layout, placement);
    q1_launch l;
    const bool fast = in_domain_flag(launch);
    resolve_launch(ctx, layout, p, fast, chunk_rows, launch, &l, false);
    // A call of fewer rows than a chunk takes the shape for its rows.
    const uint64_t most = std::min(rows, chunk_rows);
    StreamState* st = nullptr;
    q1_status s = prepare(ctx, layout, chunk_rows, num_streams, &st);
    if (s != Q1_OK) return s;
    LaunchShape full_shape;
    const char* why = "";
    s = make_shape(p, layout, fast, &l, 0, chunk_rows, &full_shape, &why);
    if (s != Q1_OK) return fail(ctx, s, why);
    if (most < chunk_rows) {
      if (!l.num_blocks) resolve_launch(ctx, layout, p, fast, most, launch, &l, false);
      s = make_shape(p, layout, fast, &l, 0, most, &full_shape, &why);
      if (s != Q1_OK) return fail(ctx, s, why);
    }
    const uint64_t ws_bytes = scan_workspace_bytes(p, fast, full_shape);
    if (rows > chunk_rows && ws_bytes > st->workspace_bytes) {
      st->workspace_bytes = 0;  // until every stream has its own
      for (auto& w : st->workspace) {
        if (w) (void)hipFree(w);
        w = nullptr;
        void* grown = nullptr;
        if (device_malloc(ctx, &grown, ws_bytes) != hipSuccess)
          return fail(ctx, Q1_ENOMEM, "workspace allocation failed");
        w = grown;
      }
      st->workspace_bytes = ws_bytes;
    }
    uint64_t elem[8];
    column_bytes_local(layout, 1, elem);  // per-row bytes of the unpacked columns
    const bool packed = layout == Q1_LAYOUT_COMPRESSED || layout == Q1_LAYOUT_COMPRESSED_PUSHDOWN;
    const auto w0 = std::chrono::steady_clock::now();
    // Once copies are queued, an error return first drains every stream, so no copy is
    // still reading the caller's host columns when the call returns.
    auto drain_fail = [&](q1_status code, const char* why) {
      for (hipStream_t ss : st->s) (void)hipStreamSynchronize(ss);
      (void)hipStreamSynchronize(ctx->stream);
      return fail(ctx, code, why);
    };
    const void* hsrc[8] = {host->ship_date, host->quantity, host->extended_price, host->discount,
                           host->tax, host->return_flag, host->line_status, host->filter};
    // Column k's share of the n rows from `off`.
    struct Piece {
      const char* src;
      void* dst;
      uint64_t len;
    };
    auto piece = [&](const q1_columns& dst, int k, uint64_t off, uint64_t n) {
      const void* ddst[8] = {dst.ship_date, dst.quantity, dst.extended_price, dst.discount,
                             dst.tax, dst.return_flag, dst.line_status, dst.filter};
      Piece c{(const char*)hsrc[k], (void*)ddst[k], 0};
      if (!c.dst || !c.src) return c;
      if (packed && k == 5) {          // return flags: 16 rows per word
        c.src += off / 16 * 4;
        c.len = (n + 15) / 16 * 4;
      } else if (packed && k >= 6) {   // line status / filter: 32 rows per word
        c.src += off / 32 * 4;
        c.len = (n + 31) / 32 * 4;
      } else {
        c.src += off * elem[k];
        c.len = n * elem[k];
      }
      return c;
    };
    uint64_t bytes = 0;
    double ms = 0;
    if (rows <= chunk_rows) {
      // One chunk: copies, scan and result one after another on the context stream, as q1_run.
      // The join of six streams, the table's clearing and its copy back took 80 us of such a
      // call (5,003 rows 146 -> 66 us).
      const q1_columns& dst = st->staging[0];
      FetchArgs f{};
      f.clock_begin = &ctx->d_result[kDirectBlocks].clock_begin;
      Piece c[8];
      for (int k = 0; k < 8; k++) {
        c[k] = piece(dst, k, 0, rows);
        if (!c[k].dst || !rows) continue;
        if (!c[k].src) return fail(ctx, Q1_EINVAL, "a column required by the layout is NULL");
        bytes += c[k].len;
        f.src[k] = c[k].src;
        f.dst[k] = c[k].dst;
        f.bytes[k] = c[k].len;
      }
      bool fetch = true;
      for (int k = 0; k < 8 && fetch; k++) fetch = !f.bytes[k] || kernel_reads(f.src[k], f.bytes[k]);
      if (!fetch) std::memset(f.bytes, 0, sizeof(f.bytes));
      if (rows && launch_fetch(f, ctx->stream) != Q1_OK) return drain_fail(Q1_EDEVICE, "chunk copy failed");
      for (int k = 0; k < 8 && !fetch; k++)
        if (c[k].len && hipMemcpyAsync(c[k].dst, c[k].src, c[k].len, hipMemcpyHostToDevice, ctx->stream) != hipSuccess)
          return drain_fail(Q1_EDEVICE, "chunk copy failed");
      s = ensure_workspace(ctx, ws_bytes);
      if (s != Q1_OK) return drain_fail(s, "workspace allocation failed");
      ScanArgs a{};
      a.cols = dst;
      a.row_end = rows;
      a.cutoff_day = cutoff_day;
      s = scan_to_host(ctx, p, layout, fast, a, full_shape);
      if (s != Q1_OK) return drain_fail(s, "scan kernel launch failed");
      double scan_ms = 0;
      uint64_t begin = 0;
      s = wait_result(ctx, out, &scan_ms, &begin);
      if (s != Q1_OK) return s;
      if (rows) ms = scan_ms + clock_ms(ctx, ctx->h_result[kDirectBlocks].clock_begin, begin);
    } else {
      const int used = (int)std::min<uint64_t>((uint64_t)num_streams, (rows + chunk_rows - 1) / chunk_rows);
      s = launch_zero(ctx->d_aggr, sizeof(q1_device_aggregates), ctx->stream);
      if (s != Q1_OK) return fail(ctx, s, "zero kernel failed");
      if (hipEventRecord(ctx->ev_begin, ctx->stream) != hipSuccess) return fail(ctx, Q1_EDEVICE, "event record failed");
      for (int i = 0; i < used; i++)
        if (hipStreamWaitEvent(st->s[(size_t)i], ctx->ev_begin, 0) != hipSuccess)
          return drain_fail(Q1_EDEVICE, "stream wait failed");
      int idx = 0;
      for (uint64_t off = 0; off < rows; off += chunk_rows, idx = (idx + 1) % num_streams) {
        const uint64_t n = rows - off < chunk_rows ? rows - off : chunk_rows;
        const q1_columns& dst = st->staging[(size_t)idx];
        hipStream_t ss = st->s[(size_t)idx];
        FetchArgs f{};
        Piece c[8];
        bool fetch = true;
        for (int k = 0; k < 8; k++) {
          c[k] = piece(dst, k, off, n);
          if (!c[k].dst) continue;
          if (!c[k].src) return drain_fail(Q1_EINVAL, "a column required by the layout is NULL");
          fetch = fetch && kernel_reads(c[k].src, c[k].len);
          f.src[k] = c[k].src;
          f.dst[k] = c[k].dst;
          f.bytes[k] = c[k].len;
          bytes += c[k].len;
        }
        if (fetch && launch_fetch(f, ss) != Q1_OK) return drain_fail(Q1_EDEVICE, "chunk copy failed");
        for (int k = 0; k < 8 && !fetch; k++)
          if (c[k].len && hipMemcpyAsync(c[k].dst, c[k].src, c[k].len, hipMemcpyHostToDevice, ss) != hipSuccess)
            return drain_fail(Q1_EDEVICE, "chunk copy failed");
        LaunchShape shape;
        s = make_shape(p, layout, fast, &l, 0, n, &shape, &why);
        if (s != Q1_OK) return drain_fail(s, why);
        ScanArgs a{};
        a.cols = dst;
        a.row_begin = 0;
        a.row_end = n;
        a.cutoff_day = cutoff_day;
        a.out = ctx->d_aggr;
        s = launch_scan(p, layout, fast, a, shape, st->workspace[(size_t)idx], ss, st->set[(size_t)idx]);
        if (s != Q1_OK) return drain_fail(s, "scan kernel launch failed");
      }
      for (int i = 0; i < used; i++) {
        if (hipEventRecord(st->done[(size_t)i], st->s[(size_t)i]) != hipSuccess ||
            hipStreamWaitEvent(ctx->stream, st->done[(size_t)i], 0) != hipSuccess)
          return drain_fail(Q1_EDEVICE, "stream join failed");
      }
      if (hipEventRecord(ctx->ev_end, ctx->stream) != hipSuccess ||
          hipMemcpyAsync(ctx->h_aggr, ctx->d_aggr, sizeof(q1_device_aggregates), hipMemcpyDeviceToHost, ctx->stream) !=
              hipSuccess ||
          hipStreamSynchronize(ctx->stream) != hipSuccess)
        return drain_fail(Q1_EDEVICE, "final copy failed");
      q1_aggregates_to_result(ctx->h_aggr, out);
      float device_ms = 0;
      (void)hipEventElapsedTime(&device_ms, ctx->ev_begin, ctx->ev_end);
      ms = device_ms;
    }
    ctx->last = q1_timing{};
    ctx->last.kernel_ms = ms;
    ctx->last.h2d_ms = ms;
    ctx->last.wall_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - w0).count();
    ctx->last.rows = rows;
    ctx->last.bytes_read = bytes;
    ctx->last.threads_per_block = l.threads_per_block;
    ctx->last.tuples_per_thread = l.tuples_per_thread;
    ctx->last.placement = fast ? (uint32_t)p : (uint32_t)Q1_PLACE_IN_REGISTERS_PER_THREAD;
    return Q1_OK;
  } catch (const std::exception& e) {
    return fail(ctx, Q1_ENOMEM, e.what());
  }
}

q1_status q1_run_split(q1_ctx* ctx, const q1_table* t, const q1_columns* host, uint64_t rows, int32_t cutoff_day,
                       q1_placement placement, const q1_launch* launch, double cpu_fraction, uint64_t align_rows,
                       int cpu_threads, q1_result* out, double* cpu_ms, double* gpu_ms) {
  if (!ctx || !t || !host || !out || cpu_fraction < 0.0 || cpu_fraction > 1.0 || rows > t->rows)
    return fail(ctx, Q1_EINVAL, "bad argument");
  try {
    // split = rows - rows*fraction, rounded down to the alignment (src/main.cu:518-529);
    // packed columns additionally need a 32-row boundary.
    uint64_t split = rows - (uint64_t)((double)rows * cpu_fraction);
    uint64_t align = align_rows ? align_rows : 1;
    if (t->layout == Q1_LAYOUT_COMPRESSED || t->layout == Q1_LAYOUT_COMPRESSED_PUSHDOWN)
      align = (align + 31) / 32 * 32;
    split -= split % align;
    std::lock_guard<std::mutex> g(ctx->lock);
    const q1_placement p = resolve_placement(ctx, t->layout, placement);
    q1_launch l;
    resolve_launch(ctx, t->layout, p, t->fast, split, launch, &l);
    LaunchShape shape;
    const char* why = "";
    q1_status s = make_shape(p, t->layout, t->fast, &l, 0, split, &shape, &why);
    if (s != Q1_OK) return fail(ctx, s, why);
    s = ensure_workspace(ctx, scan_workspace_bytes(p, t->fast, shape));
    if (s != Q1_OK) return s;
    ScanArgs a{};
    a.cols = t->dev;
    a.row_begin = 0;
    a.row_end = split;
    a.cutoff_day = t->layout == Q1_LAYOUT_COMPRESSED_PUSHDOWN ? t->filter_cutoff : cutoff_day;
    const auto w0 = std::chrono::steady_clock::now();
    s = scan_to_host(ctx, p, t->layout, t->fast, a, shape);
    if (s != Q1_OK) return s;
    // The host share runs while the device works.
    q1_result cpu{};
    const auto c0 = std::chrono::steady_clock::now();
    s = q1_cpu_run(t->layout, host, split, rows - split, a.cutoff_day, cpu_threads, &cpu);
    const double cms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - c0).count();
    q1_result gpu;
    double ms = 0;
    const q1_status device = wait_result(ctx, &gpu, &ms);
    if (device != Q1_OK) return device;
    if (s != Q1_OK) return fail(ctx, s, "host part of the split failed");
    q1_result_merge(&gpu, &cpu, out);
    ctx->last = q1_timing{};
    ctx->last.kernel_ms = ms;
    ctx->last.wall_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - w0).count();
    ctx->last.rows = rows;
    ctx->last.bytes_read = algorithmic_bytes(t->layout, split);
    ctx->last.num_blocks = shape.blocks;
    ctx->last.threads_per_block = shape.threads;
    ctx->last.tuples_per_thread = l.tuples_per_thread;
    ctx->last.placement = (uint32_t)p;
    if (cpu_ms) *cpu_ms = cms;
    if (gpu_ms) *gpu_ms = ms;
    return Q1_OK;
  } catch (const std::exception& e) {
    return fail(ctx, Q1_ENOMEM, e.what());
  }
}

}  // extern "C"

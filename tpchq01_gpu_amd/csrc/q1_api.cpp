// C-ABI implementation: contexts, device-resident tables, the query entry points,
// timing, autotuning table, the CPU/GPU split and the host-resident streaming pipeline.
// Every entry point catches C++ exceptions and returns a status (nothing crosses the ABI).
#include <dlfcn.h>

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <sstream>
#include <thread>
#include <vector>

#include "q1_common.h"
#include "q1_internal.h"

namespace q1 {

q1_status fail(q1_ctx* ctx, q1_status s, const std::string& why) {
  if (ctx) ctx->error = why;
  return s;
}

q1_status hip_fail(q1_ctx* ctx, hipError_t e, const char* what) {
  if (ctx) ctx->error = std::string(what) + ": " + hipGetErrorString(e);
  return Q1_EDEVICE;
}

#define Q1_HIP(ctx, call)                                   \
  do {                                                      \
    const hipError_t e_ = (call);                           \
    if (e_ != hipSuccess) return q1::hip_fail(ctx, e_, #call); \
  } while (0)

static bool valid_layout(int l) { return l >= Q1_LAYOUT_REFERENCE && l <= Q1_LAYOUT_COMPRESSED_PUSHDOWN; }
static bool valid_placement(int p) { return p >= Q1_PLACE_IN_REGISTERS && p <= Q1_PLACE_AUTO; }

uint64_t algorithmic_bytes(q1_layout layout, uint64_t rows) {
  // bits per row: 304 reference, 160 uncompressed, 75 compressed, 60 pushdown
  static const uint64_t bits[4] = {304, 160, 75, 60};
  return rows * bits[layout] / 8;
}

q1_placement resolve_placement(q1_ctx* ctx, q1_layout layout, q1_placement p) {
  return p == Q1_PLACE_AUTO ? ctx->best[layout] : p;
}

// The any-value kernel's shape.  Lanes per block: 256 for the compressed layouts, 128 for the
// others, whose LDS tables of 61 and 86 KB per 256 lanes leave a compute unit two blocks or
// one (60M reference rows 371 us with 256 lanes, 354 with 128; 2M compressed rows 10.0 and
// 11.2 us).  Rows per lane: what makes the grid one round of the chip, since the last of two
// or three rounds leaves compute units idle (8.4M reference rows 56 us with 128 rows per lane,
// one round, and 63 with 64; 12M uncompressed rows 47 with 96 and 55 with 64; 20M compressed
// rows 38 with 80 and 41 with 64): 16 while all lanes' tables fit the LDS (`fit` lanes per
// compute unit), else the fewest for which `lanes` do, an even share of its four SIMDs, at
// most 128.  Above that, many rounds of short blocks, whose last round is short: 60M rows with
// 32 / 64 / 128 per lane: compressed 101 / 98 / 102, uncompressed 193 / 197 / 207, reference
// 345 / 349 / 353.
struct AnyShape {
  uint32_t threads, fit, lanes, many;
};
constexpr uint32_t kAnyTuples = 128;
static AnyShape any_value_shape(q1_layout l) {
  return l == Q1_LAYOUT_REFERENCE      ? AnyShape{128, 384, 256, 32}
         : l == Q1_LAYOUT_UNCOMPRESSED ? AnyShape{128, 640, 512, 32}
                                       : AnyShape{256, 1024, 1024, 64};
}

// The tuned shape for a range of `rows` rows: of the shapes tuned at several row counts,
// the one whose row count is nearest by ratio (the larger on a tie); the single tuned
// shape when the table has none.
static q1_launch tuned_for_rows(const q1_ctx* ctx, q1_layout layout, q1_placement p, uint64_t rows) {
  q1_launch t = ctx->tuning[layout][p];
  const std::vector<SizedLaunch>& at = ctx->tuning_at[layout][p];
  if (at.empty()) return t;
  const double r = (double)std::max<uint64_t>(rows, 1);
  double best = 0;
  for (size_t i = 0; i < at.size(); i++) {
    const double n = (double)at[i].rows, d = r > n ? r / n : n / r;
    if (i == 0 || d <= best) {
      best = d;
      t.threads_per_block = at[i].threads_per_block;
      t.tuples_per_thread = at[i].tuples_per_thread;
    }
  }
  return t;
}

void resolve_launch(q1_ctx* ctx, q1_layout layout, q1_placement p, bool fast, uint64_t rows, const q1_launch* in,
                    q1_launch* out, bool table) {
  const AnyShape any = any_value_shape(layout);
  q1_launch t{any.threads, kAnyTuples, 0, 0};
  if (fast)
    t = tuned_for_rows(ctx, layout, p, rows);
  else if (in && in->num_blocks)
    // a caller's grid is held against the tuned shape for a table, 256 x 1024 for raw pointers
    t = table ? tuned_for_rows(ctx, layout, p, rows) : q1_launch{256, 1024, 0, 0};
  out->threads_per_block = in && in->threads_per_block ? in->threads_per_block : t.threads_per_block;
  out->tuples_per_thread = in && in->tuples_per_thread ? in->tuples_per_thread : t.tuples_per_thread;
  out->num_blocks = in ? in->num_blocks : 0;
  out->flags = in ? in->flags : 0;
  // A caller-chosen value is kept as given.
  if ((in && in->tuples_per_thread) || out->num_blocks) return;
  const uint64_t units = ctx->compute_units > 0 ? ctx->compute_units : 256;
  if (!fast) {
    const uint64_t a_round = 16 * units * any.lanes;
    if (rows <= 16 * units * any.fit)
      out->tuples_per_thread = 16;
    else if (rows <= a_round * (kAnyTuples / 16))
      out->tuples_per_thread = 16 * (uint32_t)((rows + a_round - 1) / a_round);
    else
      out->tuples_per_thread = any.many;
    return;
  }
  // A range smaller than the row counts the shape was tuned at halves its tuples_per_thread
  // until the grid has at least 4 blocks or 384 lanes per compute unit, so small requests still
  // spread over the whole chip.  6M compressed rows in 256 x 32, 732 lanes per compute unit: 24.4
  // us; halved to 1,465: 27.8 (4 blocks of 256 lanes used to be asked for).
  const uint64_t tpb = out->threads_per_block ? out->threads_per_block : 256;
  const uint64_t lanes = std::min<uint64_t>(4 * tpb, 384) * units;
  while (out->tuples_per_thread > 16 && rows < lanes * out->tuples_per_thread)
    out->tuples_per_thread = (out->tuples_per_thread / 2 + 15) & ~15u;
}

// The spare bitmap if it holds at least `bytes` bytes; it is then the caller's.
static SpareFilter take_spare(q1_ctx* ctx, uint64_t bytes) {
  std::lock_guard<std::mutex> g(ctx->spare_lock);
  SpareFilter spare;
  if (ctx->spare.bytes >= bytes) std::swap(spare, ctx->spare);
  return spare;
}

hipError_t device_malloc(q1_ctx* ctx, void** p, uint64_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipSuccess) return e;
  const SpareFilter spare = take_spare(ctx, 0);
  if (!spare.p) return e;
  (void)hipGetLastError();
  (void)hipFree(spare.p);
  return hipMalloc(p, bytes);
}

q1_status ensure_workspace(q1_ctx* ctx, uint64_t bytes) {
  if (bytes <= ctx->workspace_bytes) return Q1_OK;
  if (ctx->workspace) {
    Q1_HIP(ctx, hipStreamSynchronize(ctx->stream));
    Q1_HIP(ctx, hipFree(ctx->workspace));
    ctx->workspace = nullptr;
    ctx->workspace_bytes = 0;
  }
  Q1_HIP(ctx, device_malloc(ctx, &ctx->workspace, bytes));
  ctx->workspace_bytes = bytes;
  return Q1_OK;
}

// The longest wait for a set, with the context's lock held: beyond it a launch merges directly.  The
// oldest of 256 launches in flight usually ends within its own few microseconds.
constexpr int kPoolWaitMs = 2;

// A free set of the pool for a large launch on a caller's stream, its index in *index; nullptr
// (merge directly) when the sets stay in flight.
static MergeSet* pool_set(q1_ctx* ctx, size_t* index) {
  SetPool& pool = ctx->pool;
  // Launches on one stream end in order, so the set after the last one given is the first to
  // come free unless streams of very different pace share the pool.
  auto free_set = [&](size_t i) { return __atomic_load_n(&pool.done[i], __ATOMIC_ACQUIRE) == pool.last[i]; };
  auto take = [&](size_t i) {
    pool.cursor = (i + 1) % kPoolSets;
    pool.stalled = false;
    *index = i;
    return pool.sets + i;
  };
  for (size_t looked = 0; looked < 8; looked++)
    if (free_set((pool.cursor + looked) % kPoolSets)) return take((pool.cursor + looked) % kPoolSets);
  // All in flight: the caller is 256 launches ahead of the device.  Waiting for the oldest
  // keeps it there; a direct merge would cost this launch up to 0.03 us per block.  A stream
  // that does not move (it may be waiting for the caller) is waited for once only.
  if (!pool.stalled) {
    const size_t i = pool.cursor;
    const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(kPoolWaitMs);
    while (!free_set(i) && std::chrono::steady_clock::now() < until) __builtin_ia32_pause();
    if (free_set(i)) return take(i);
    pool.stalled = true;
  }
  pool.cursor = (pool.cursor + 8) % kPoolSets;
  return nullptr;
}

// Whether a launch on the stream goes into a graph, whose replays, on any stream and beside any
// other launch, would use its merge set again: it merges directly.
static bool captured(void* stream) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing((hipStream_t)stream, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone;
}

q1_status scan_on(q1_ctx* ctx, q1_placement placement, q1_layout layout, bool fast, const ScanArgs& args,
                  const LaunchShape& shape, void* stream) {
  ScanArgs a = args;
  size_t i = 0;
  MergeSet *set = nullptr, *pooled = nullptr;
  if (shape.blocks >= kSpreadMinBlocks && !captured(stream)) {
    if (stream == (void*)ctx->stream)  // its launches run one after another
      set = ctx->set;
    else
      set = pooled = pool_set(ctx, &i);
  }
  if (pooled) {
    a.done = ctx->pool.done_dev + i;
    a.sequence = ++ctx->pool.sequence;
  }
  const q1_status s = launch_scan(placement, layout, fast, a, shape, ctx->workspace, stream, set);
  if (s == Q1_OK && pooled) ctx->pool.last[i] = a.sequence;
  return s;
}

q1_status scan_to_host(q1_ctx* ctx, q1_placement placement, q1_layout layout, bool fast, ScanArgs a,
                       const LaunchShape& shape) {
  a.host = ctx->d_result;
  a.sequence = ++ctx->sequence;
  const bool direct = can_launch_direct(placement, layout, fast, shape);
  ctx->results = direct ? shape.blocks : shape.blocks ? 1 : 0;
  if (shape.blocks == 0) return Q1_OK;
  const q1_status s = direct ? launch_direct(layout, a, shape, (void*)ctx->stream)
                             : launch_scan(placement, layout, fast, a, shape, ctx->workspace, (void*)ctx->stream, ctx->set);
  return s == Q1_OK ? Q1_OK : fail(ctx, s, "scan kernel launch failed");
}

// The kernel's last store is the launch's number in pinned host memory, for which the host
// watches: an empty kernel launched and awaited so takes 6.2 us, 10.9 with the stream's wait,
// and a call of 820 us 5 us less.  Under HIP's default schedule the stream's wait keeps the
// processor as busy (1.00 of a core over such calls), so nothing is lost by watching for as long as
// a scan of 1.4G compressed rows takes; then the stream's wait, which also tells when the launch
// has failed.  A process that asked for blocking waits gets the stream's after 20 us: asking the
// runtime costs 0.5 us, of calls that mostly have their result before (5,003 rows 12.7 -> 11.7 us).
static bool blocking_waits(const q1_ctx* ctx) {
  int current = ctx->device;
  unsigned flags = 0;
  (void)hipGetDevice(&current);
  if (current != ctx->device) (void)hipSetDevice(ctx->device);
  const bool got = hipGetDeviceFlags(&flags) == hipSuccess;
  if (current != ctx->device) (void)hipSetDevice(current);
  return got && (flags & hipDeviceScheduleMask) == hipDeviceScheduleBlockingSync;
}
constexpr int kWatchMicroseconds = 2000, kShortWatchMicroseconds = 20;
q1_status wait_sequence(q1_ctx* ctx, const uint64_t* word, uint64_t sequence) {
  auto arrived = [&] { return __atomic_load_n(word, __ATOMIC_ACQUIRE) == sequence; };
  auto watch = [&](int us) {
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(us);
    while (!arrived() && std::chrono::steady_clock::now() < until)
      for (int i = 0; i < 16 && !arrived(); i++) __builtin_ia32_pause();
    return arrived();
  };
  if (!watch(kShortWatchMicroseconds) && !blocking_waits(ctx)) watch(kWatchMicroseconds);
  if (!arrived()) {
    Q1_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (!arrived()) {
      // The launch's blocks were not counted to the end: the set may hold partial sums.
      (void)launch_zero(ctx->set, sizeof(MergeSet), ctx->stream);
      return fail(ctx, Q1_EDEVICE, "the scan kernel ended without a result");
    }
  }
  ctx->queued = false;  // what was before the launch on the stream has ended too
  return Q1_OK;
}

double clock_ms(const q1_ctx* ctx, uint64_t begin, uint64_t end) {
  return ctx->clock_khz > 0 ? (double)(end - begin) / ctx->clock_khz : 0.0;
}

// sum += other, the 128-bit fields as (lo, hi) pairs.
static void add_aggregates(q1_device_aggregates* sum, const q1_device_aggregates& other) {
  for (int g = 0; g < Q1_NUM_GROUPS; g++) {
    sum->sum_qty[g] += other.sum_qty[g];
    sum->sum_base_price[g] += other.sum_base_price[g];
    sum->sum_disc[g] += other.sum_disc[g];
    sum->count[g] += other.count[g];
    sum->sum_disc_price_lo[g] += other.sum_disc_price_lo[g];
    sum->sum_disc_price_hi[g] += other.sum_disc_price_hi[g] + (sum->sum_disc_price_lo[g] < other.sum_disc_price_lo[g]);
    sum->sum_charge_lo[g] += other.sum_charge_lo[g];
    sum->sum_charge_hi[g] += other.sum_charge_hi[g] + (sum->sum_charge_lo[g] < other.sum_charge_lo[g]);
  }
}

q1_status wait_result(q1_ctx* ctx, q1_result* out, double* kernel_ms, uint64_t* begin_clock) {
  const HostResult* r = ctx->h_result;
  for (uint32_t i = 0; i < ctx->results; i++) {
    const q1_status s = wait_sequence(ctx, &r[i].sequence, ctx->sequence);
    if (s != Q1_OK) return s;
  }
  q1_device_aggregates sum{};
  uint64_t begin = 0, end = 0;
  if (ctx->results) {
    sum = r[0].sums;
    begin = r[0].clock_begin;
    end = r[0].clock_end;
  }
  for (uint32_t i = 1; i < ctx->results; i++) {
    add_aggregates(&sum, r[i].sums);
    begin = std::min(begin, r[i].clock_begin);
    end = std::max(end, r[i].clock_end);
  }
  q1_aggregates_to_result(&sum, out);
  *kernel_ms = clock_ms(ctx, begin, end);
  if (begin_clock) *begin_clock = begin;
  return Q1_OK;
}

// Column sizes in bytes, in q1_columns order.
static void column_bytes(q1_layout layout, uint64_t n, uint64_t b[8]) {
  std::memset(b, 0, 8 * sizeof(uint64_t));
  const uint64_t rf_words = (n + 15) / 16, ls_words = (n + 31) / 32;
  switch (layout) {
    case Q1_LAYOUT_REFERENCE:
      b[0] = 4 * n; b[1] = 8 * n; b[2] = 8 * n; b[3] = 8 * n; b[4] = 8 * n; b[5] = n; b[6] = n;
      break;
    case Q1_LAYOUT_UNCOMPRESSED:
      b[0] = 4 * n; b[1] = 4 * n; b[2] = 8 * n; b[3] = n; b[4] = n; b[5] = n; b[6] = n;
      break;
    case Q1_LAYOUT_COMPRESSED:
      b[0] = 2 * n; b[1] = n; b[2] = 4 * n; b[3] = n; b[4] = n; b[5] = 4 * rf_words; b[6] = 4 * ls_words;
      break;
    case Q1_LAYOUT_COMPRESSED_PUSHDOWN:
      b[1] = n; b[2] = 4 * n; b[3] = n; b[4] = n; b[5] = 4 * rf_words; b[6] = 4 * ls_words; b[7] = 4 * ls_words;
      break;
  }
}

static const void*& col(q1_columns& c, int i) {
  const void** p[8] = {&c.ship_date, &c.quantity, &c.extended_price, &c.discount,
                       &c.tax, &c.return_flag, &c.line_status, &c.filter};
  return *p[i];
}
static const void* colc(const q1_columns& c, int i) { return col(const_cast<q1_columns&>(c), i); }

// Sets t->fast: whether the table's values lie inside the TPC-H domain.  The columns of a
// pushdown table are those of a compressed one.
static q1_status measure_domain(q1_ctx* ctx, q1_table* t) {
  const q1_layout l = t->layout == Q1_LAYOUT_COMPRESSED_PUSHDOWN ? Q1_LAYOUT_COMPRESSED : t->layout;
  if (t->rows == 0) {
    t->fast = true;
    return Q1_OK;
  }
  const Completion done{ctx->set, ctx->d_result, ++ctx->sequence};
  bool counted = false;
  ctx->h_result->outside = 0;
  q1_status s = launch_domain_check(l, t->dev, t->rows, done, ctx->stream, &counted);
  if (s != Q1_OK) return fail(ctx, s, "domain check kernel launch failed");
  if (!counted) {
    Q1_HIP(ctx, hipStreamSynchronize(ctx->stream));
  } else {
    s = wait_sequence(ctx, &ctx->h_result->sequence, done.sequence);
    if (s != Q1_OK) return s;
  }
  t->fast = ctx->h_result->outside == 0;
  return Q1_OK;
}

static void load_tuning_file(q1_ctx* ctx) {
  std::string path;
  if (const char* env = std::getenv("Q1_TUNING_FILE")) {
    path = env;
  } else {
    Dl_info info;
    if (dladdr((void*)&load_tuning_file, &info) && info.dli_fname) {
      std::string so = info.dli_fname;
      const size_t slash = so.rfind('/');
      const std::string dir = slash == std::string::npos ? "." : so.substr(0, slash);
      path = dir + "/../tuning/gfx950.txt";
    }
  }
  std::ifstream in(path);
  std::string line;
  while (std::getline(in, line)) {
    std::istringstream ls(line);
    std::string kind;
    ls >> kind;
    int l = -1, p = -1;
    if (kind == "launch") {
      uint32_t tpb = 0, tpt = 0;
      ls >> l >> p >> tpb >> tpt;
      // same limits as make_shape: a bad line is ignored rather than failing every launch
      const bool shape_ok = (tpb == 64 || tpb == 128 || tpb == 256) && tpt && tpt % 16 == 0 && tpt <= 16384;
      if (valid_layout(l) && p >= 0 && p <= Q1_PLACE_GLOBAL && shape_ok) {
        ctx->tuning[l][p].threads_per_block = tpb;
        ctx->tuning[l][p].tuples_per_thread = tpt;
      }
    } else if (kind == "launch_at") {
      // launch_at <rows> <layout> <placement> <threads_per_block> <tuples_per_thread>
      uint64_t rows = 0;
      uint32_t tpb = 0, tpt = 0;
      ls >> rows >> l >> p >> tpb >> tpt;
      const bool shape_ok = (tpb == 64 || tpb == 128 || tpb == 256) && tpt && tpt % 16 == 0 && tpt <= 16384;
      if (rows && valid_layout(l) && p >= 0 && p <= Q1_PLACE_GLOBAL && shape_ok) {
        std::vector<SizedLaunch>& at = ctx->tuning_at[l][p];
        auto it = std::lower_bound(at.begin(), at.end(), rows,
                                   [](const SizedLaunch& a, uint64_t r) { return a.rows < r; });
        if (it != at.end() && it->rows == rows)
          *it = SizedLaunch{rows, tpb, tpt};
        else
          at.insert(it, SizedLaunch{rows, tpb, tpt});
      }
    } else if (kind == "streaming") {
      // streaming <layout> <chunk rows> <streams>
      uint64_t chunk = 0;
      int streams = 0;
      ls >> l >> chunk >> streams;
      if (valid_layout(l) && chunk && chunk % 32 == 0 && streams >= 1 && streams <= 16) {
        ctx->stream_chunk_rows[l] = chunk;
        ctx->stream_count[l] = streams;
      }
    } else if (kind == "best") {
      ls >> l >> p;
      if (valid_layout(l) && p >= 0 && p <= Q1_PLACE_GLOBAL) ctx->best[l] = (q1_placement)p;
    } else if (kind == "batch") {
      // batch <layout> <placement> <blocks per compute unit> <rows per lane>
      uint32_t per_cu = 0, lane_rows = 0;
      ls >> l >> p >> per_cu >> lane_rows;
      const bool shape_ok = per_cu >= 1 && per_cu <= 64 && lane_rows && lane_rows % 16 == 0 && lane_rows <= 16384;
      if (valid_layout(l) && p >= 0 && p <= Q1_PLACE_GLOBAL && shape_ok) {
        ctx->batch_tuning[l][p].num_blocks = per_cu;
        ctx->batch_tuning[l][p].tuples_per_thread = lane_rows;
      }
    }
  }
}

// A bitmap of at least `bytes` bytes.
static bool filter_malloc(q1_ctx* ctx, uint64_t bytes, q1_table* t) {
  const SpareFilter spare = take_spare(ctx, bytes);
  if (spare.p) {
    t->owned[7] = spare.p;
    t->filter_bytes = spare.bytes;
    return true;
  }
  void* p = nullptr;
  if (device_malloc(ctx, &p, bytes) != hipSuccess) return false;
  t->owned[7] = p;
  t->filter_bytes = bytes;
  return true;
}

// Frees a table with its context's lock held (every entry point that creates tables
// holds it when a creation fails).  Whatever may still read the table ends first: hipFree waits
// for the device, and where nothing may be freed, the waits here are those that are needed.
static void release_table(q1_table* t) {
  if (q1_ctx* ctx = t->ctx) {
    if (ctx->queued || ctx->stream_out) {
      (void)hipStreamSynchronize(ctx->stream);
      ctx->queued = false;
    }
    if (t->filter_bytes && t->filter_bytes <= kSpareFilterBytes) {
      if (t->shared) (void)hipDeviceSynchronize();
      std::lock_guard<std::mutex> g(ctx->spare_lock);
      if (t->filter_bytes > ctx->spare.bytes) {
        const SpareFilter kept{t->owned[7], t->filter_bytes};
        t->owned[7] = ctx->spare.p;
        ctx->spare = kept;
      }
    }
    for (void* p : t->owned)
      if (p) (void)hipFree(p);
    ctx->tables.erase(t);
  }
  delete t;
}

}  // namespace q1

using namespace q1;

#define GUARD_BEGIN try {
#define GUARD_END(ctx)                                         \
  }                                                            \
  catch (const std::bad_alloc&) {                              \
    return q1::fail(ctx, Q1_ENOMEM, "host allocation failed"); \
  }                                                            \
  catch (const std::exception& ex) {                           \
    return q1::fail(ctx, Q1_EINVAL, ex.what());                \
  }

extern "C" {

const char* q1_strerror(q1_status s) {
  switch (s) {
    case Q1_OK: return "ok";
    case Q1_EINVAL: return "invalid argument";
    case Q1_ENOMEM: return "out of memory";
    case Q1_EDEVICE: return "device error";
    case Q1_EOVERFLOW: return "overflow";
    case Q1_EBUSY: return "busy";
    case Q1_ETIMEOUT: return "timed out";
    case Q1_ECANCELED: return "canceled";
  }
  return "unknown status";
}

int q1_abi_version(void) { return Q1_ABI_VERSION; }

const char* q1_last_error(q1_ctx* ctx) { return ctx ? ctx->error.c_str() : ""; }

q1_status q1_init(int device, q1_ctx** out) {
  if (!out) return Q1_EINVAL;
  *out = nullptr;
  GUARD_BEGIN
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess || count == 0) return Q1_EDEVICE;
  if (device < 0 || device >= count) return Q1_EINVAL;
  if (hipSetDevice(device) != hipSuccess) return Q1_EDEVICE;
  q1_ctx* ctx = new q1_ctx();
  ctx->device = device;
  for (int l = 0; l < 4; l++)
    for (int p = 0; p < 5; p++) ctx->tuning[l][p] = q1_launch{256, 1024, 0, 0};
  hipDeviceProp_t prop;
  bool ok = hipGetDeviceProperties(&prop, device) == hipSuccess;
  ctx->compute_units = ok ? prop.multiProcessorCount : 0;
  ok = ok && hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) == hipSuccess;
  ok = ok && hipEventCreate(&ctx->ev_begin) == hipSuccess && hipEventCreate(&ctx->ev_end) == hipSuccess;
  ok = ok && hipEventCreate(&ctx->ev_h2d_begin) == hipSuccess && hipEventCreate(&ctx->ev_h2d_end) == hipSuccess;
  ok = ok && hipMalloc(&ctx->d_aggr, sizeof(q1_device_aggregates)) == hipSuccess;
  ok = ok && hipHostMalloc(&ctx->h_aggr, sizeof(q1_device_aggregates), hipHostMallocDefault) == hipSuccess;
  ok = ok && hipHostMalloc(&ctx->h_result, (kDirectBlocks + 1) * sizeof(HostResult), hipHostMallocMapped) == hipSuccess &&
       hipHostGetDevicePointer((void**)&ctx->d_result, ctx->h_result, 0) == hipSuccess;
  if (ok) std::memset(ctx->h_result, 0, (kDirectBlocks + 1) * sizeof(HostResult));
  ok = ok && hipDeviceGetAttribute(&ctx->clock_khz, hipDeviceAttributeWallClockRate, device) == hipSuccess;
  ok = ok && hipMalloc(&ctx->set, sizeof(MergeSet)) == hipSuccess;
  ok = ok && hipMemset(ctx->set, 0, sizeof(MergeSet)) == hipSuccess;
  SetPool& pool = ctx->pool;
  ok = ok && hipMalloc(&pool.sets, kPoolSets * sizeof(MergeSet)) == hipSuccess &&
       hipMemset(pool.sets, 0, kPoolSets * sizeof(MergeSet)) == hipSuccess &&
       hipHostMalloc(&pool.done, kPoolSets * sizeof(uint64_t), hipHostMallocMapped) == hipSuccess &&
       hipHostGetDevicePointer((void**)&pool.done_dev, pool.done, 0) == hipSuccess;
  if (ok) std::memset(pool.done, 0, kPoolSets * sizeof(uint64_t));
  // the scratch of q1_enqueue_noalloc on this device (once per device and process)
  ok = ok && noalloc_setup(device, ctx->stream) == Q1_OK;
  ok = ok && hipDeviceSynchronize() == hipSuccess;
  if (!ok) {
    q1_shutdown(ctx);
    return Q1_EDEVICE;
  }
  load_tuning_file(ctx);
  *out = ctx;
  return Q1_OK;
  GUARD_END(nullptr)
}

void q1_shutdown(q1_ctx* ctx) {
  if (!ctx) return;
  if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
  // Tables still alive lose their device memory; their handles stay valid for
  // q1_table_free only.
  for (q1_table* t : ctx->tables) {
    for (void*& p : t->owned) {
      if (p) (void)hipFree(p);
      p = nullptr;
    }
    t->ctx = nullptr;
    t->dev = q1_columns{};
    t->rows = 0;
  }
  ctx->tables.clear();
  if (ctx->spare.p) (void)hipFree(ctx->spare.p);
  if (ctx->batch) {
    batch_free(ctx->batch);
    delete ctx->batch;
  }
  stream_state_release(ctx);
  if (ctx->workspace) (void)hipFree(ctx->workspace);
  if (ctx->set) (void)hipFree(ctx->set);
  if (ctx->pool.sets) (void)hipDeviceSynchronize();  // callers' streams may still use the pool
  if (ctx->pool.sets) (void)hipFree(ctx->pool.sets);
  if (ctx->pool.done) (void)hipHostFree(ctx->pool.done);
  if (ctx->h_aggr) (void)hipHostFree(ctx->h_aggr);
  if (ctx->h_result) (void)hipHostFree(ctx->h_result);
  if (ctx->d_aggr) (void)hipFree(ctx->d_aggr);
  for (hipEvent_t e : {ctx->ev_begin, ctx->ev_end, ctx->ev_h2d_begin, ctx->ev_h2d_end})
    if (e) (void)hipEventDestroy(e);
  if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
  delete ctx;
}

q1_status q1_device_info_get(q1_ctx* ctx, q1_device_info* out) {
  if (!ctx || !out) return Q1_EINVAL;
  hipDeviceProp_t p;
  Q1_HIP(ctx, hipGetDeviceProperties(&p, ctx->device));
  std::memset(out, 0, sizeof(*out));
  std::snprintf(out->name, sizeof(out->name), "%.63s", p.name);
  std::snprintf(out->arch, sizeof(out->arch), "%.31s", p.gcnArchName);
  out->compute_units = p.multiProcessorCount;
  out->clock_khz = p.clockRate;
  out->memory_clock_khz = p.memoryClockRate;
  out->memory_bus_width = p.memoryBusWidth;
  out->total_memory = p.totalGlobalMem;
  out->lds_per_block = p.sharedMemPerBlock;
  out->wavefront_size = p.warpSize;
  out->max_threads_per_block = p.maxThreadsPerBlock;
  return Q1_OK;
}

q1_status q1_synchronize(q1_ctx* ctx) {
  if (!ctx) return Q1_EINVAL;
  Q1_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return Q1_OK;
}

void* q1_stream(q1_ctx* ctx) {
  if (!ctx) return nullptr;
  ctx->stream_out = true;
  return (void*)ctx->stream;
}

q1_status q1_layout_column_bytes(q1_layout layout, uint64_t rows, uint64_t bytes_out[8]) {
  if (!valid_layout(layout) || !bytes_out) return Q1_EINVAL;
  column_bytes(layout, rows, bytes_out);
  return Q1_OK;
}

// ---------------------------------------------------------------------------------------
// Tables
// ---------------------------------------------------------------------------------------
static q1_status alloc_table(q1_ctx* ctx, q1_layout layout, uint64_t rows, q1_table** out) {
  uint64_t b[8];
  column_bytes(layout, rows, b);
  q1_table* t = new q1_table();
  t->ctx = ctx;
  t->layout = layout;
  t->rows = rows;
  ctx->tables.insert(t);
  for (int i = 0; i < 8; i++) {
    if (!b[i]) continue;
    void* p = nullptr;
    const hipError_t e = device_malloc(ctx, &p, b[i]);
    if (e != hipSuccess) {
      release_table(t);
      return fail(ctx, Q1_ENOMEM, "device allocation of a table column failed");
    }
    t->owned[i] = p;
    col(t->dev, i) = p;
    t->device_bytes += b[i];
  }
  *out = t;
  return Q1_OK;
}

q1_status q1_table_upload(q1_ctx* ctx, q1_layout layout, const q1_columns* host, uint64_t rows,
                          q1_table** out) {
  if (!ctx || !host || !out || !valid_layout(layout)) return fail(ctx, Q1_EINVAL, "bad argument");
  *out = nullptr;
  GUARD_BEGIN
  std::lock_guard<std::mutex> g(ctx->lock);
  Q1_HIP(ctx, hipSetDevice(ctx->device));
  uint64_t b[8];
  column_bytes(layout, rows, b);
  for (int i = 0; i < 8; i++)
    if (b[i] && !colc(*host, i)) return fail(ctx, Q1_EINVAL, "a column required by the layout is NULL");
  q1_table* t = nullptr;
  q1_status s = alloc_table(ctx, layout, rows, &t);
  if (s != Q1_OK) return s;
  const auto w0 = std::chrono::steady_clock::now();
  bool ok = hipEventRecord(ctx->ev_h2d_begin, ctx->stream) == hipSuccess;
  for (int i = 0; i < 8 && ok; i++)
    if (b[i])
      ok = hipMemcpyAsync((void*)colc(t->dev, i), colc(*host, i), b[i], hipMemcpyHostToDevice, ctx->stream) ==
           hipSuccess;
  ok = ok && hipEventRecord(ctx->ev_h2d_end, ctx->stream) == hipSuccess;
  ok = hipStreamSynchronize(ctx->stream) == hipSuccess && ok;
  if (!ok) {
    release_table(t);
    return fail(ctx, Q1_EDEVICE, "upload of the table columns failed");
  }
  float ms = 0;
  (void)hipEventElapsedTime(&ms, ctx->ev_h2d_begin, ctx->ev_h2d_end);
  ctx->last = q1_timing{};
  ctx->last.h2d_ms = ms;
  ctx->last.wall_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - w0).count();
  ctx->last.bytes_read = t->device_bytes;
  s = measure_domain(ctx, t);
  if (s != Q1_OK) {
    release_table(t);
    return s;
  }
  *out = t;
  return Q1_OK;
  GUARD_END(ctx)
}

q1_status q1_table_wrap(q1_ctx* ctx, q1_layout layout, const q1_columns* device, uint64_t rows,
                        q1_table** out) {
  if (!ctx || !device || !out || !valid_layout(layout)) return fail(ctx, Q1_EINVAL, "bad argument");
  *out = nullptr;
  GUARD_BEGIN
  std::lock_guard<std::mutex> g(ctx->lock);
  uint64_t b[8];
  column_bytes(layout, rows, b);
  for (int i = 0; i < 8; i++) {
    if (!b[i]) continue;
    const void* p = colc(*device, i);
    if (!p) return fail(ctx, Q1_EINVAL, "a column required by the layout is NULL");
    if ((uintptr_t)p % 16) return fail(ctx, Q1_EINVAL, "device columns must be 16-byte aligned");
  }
  q1_table* t = new q1_table();
  t->ctx = ctx;
  t->layout = layout;
  t->rows = rows;
  t->dev = *device;
  for (int i = 0; i < 8; i++)
    if (!b[i]) col(t->dev, i) = nullptr;
  const q1_status s = measure_domain(ctx, t);
  if (s != Q1_OK) {
    delete t;
    return s;
  }
  ctx->tables.insert(t);
  *out = t;
  return Q1_OK;
  GUARD_END(ctx)
}

q1_status q1_table_refresh_domain(q1_ctx* ctx, q1_table* t) {
  if (!ctx || !t || t->ctx != ctx) return fail(ctx, Q1_EINVAL, "bad argument");
  GUARD_BEGIN
  std::lock_guard<std::mutex> g(ctx->lock);
  return measure_domain(ctx, t);
  GUARD_END(ctx)
}

q1_status q1_table_generate(q1_ctx* ctx, q1_layout layout, uint64_t seed, uint64_t rows, q1_table** out) {
  if (!ctx || !out || !valid_layout(layout) || layout == Q1_LAYOUT_COMPRESSED_PUSHDOWN)
    return fail(ctx, Q1_EINVAL, "bad argument (pushdown tables come from q1_build_filter)");
  *out = nullptr;
  GUARD_BEGIN
  std::lock_guard<std::mutex> g(ctx->lock);
  Q1_HIP(ctx, hipSetDevice(ctx->device));
  q1_table* t = nullptr;
  q1_status s = alloc_table(ctx, layout, rows, &t);
  if (s != Q1_OK) return s;
  s = launch_generate(layout, seed, rows, t->dev, ctx->stream);
  if (s == Q1_OK) s = measure_domain(ctx, t);
  if (s != Q1_OK) {
    release_table(t);
    return fail(ctx, s, "generator failed");
  }
  *out = t;
  return Q1_OK;
  GUARD_END(ctx)
}

q1_status q1_table_info(const q1_table* t, q1_layout* layout, uint64_t* rows, q1_columns* device) {
  if (!t) return Q1_EINVAL;
  if (layout) *layout = t->layout;
  if (rows) *rows = t->rows;
  if (device) {
    t->shared = true;
    *device = t->dev;
  }
  return Q1_OK;
}

q1_status q1_table_download(q1_ctx* ctx, const q1_table* t, const q1_columns* host_out) {
  if (!ctx || !t || !host_out) return fail(ctx, Q1_EINVAL, "bad argument");
  GUARD_BEGIN
  std::lock_guard<std::mutex> g(ctx->lock);
  uint64_t b[8];
  column_bytes(t->layout, t->rows, b);
  for (int i = 0; i < 8; i++) {
    if (!b[i] || !colc(*host_out, i)) continue;
    Q1_HIP(ctx, hipMemcpyAsync((void*)colc(*host_out, i), colc(t->dev, i), b[i], hipMemcpyDeviceToHost, ctx->stream));
  }
  Q1_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return Q1_OK;
  GUARD_END(ctx)
}

uint64_t q1_table_device_bytes(const q1_table* t) { return t ? t->device_bytes : 0; }

// A table freed after its context was shut down has already lost its device memory
// (q1_shutdown releases it); only the handle is deleted then.
void q1_table_free(q1_table* t) {
  if (!t) return;
  if (q1_ctx* ctx = t->ctx) {
    std::lock_guard<std::mutex> g(ctx->lock);
    release_table(t);
  } else {
    delete t;
  }
}

q1_status q1_build_filter(q1_ctx* ctx, const q1_table* compressed, int32_t cutoff_day, q1_table** out) {
  if (!ctx || !compressed || !out || compressed->layout != Q1_LAYOUT_COMPRESSED)
    return fail(ctx, Q1_EINVAL, "q1_build_filter needs a COMPRESSED table");
  *out = nullptr;
  GUARD_BEGIN
  std::lock_guard<std::mutex> g(ctx->lock);
  Q1_HIP(ctx, hipSetDevice(ctx->device));
  q1_table* t = new q1_table();
  t->ctx = ctx;
  t->layout = Q1_LAYOUT_COMPRESSED_PUSHDOWN;
  t->rows = compressed->rows;
  t->dev = compressed->dev;
  t->dev.ship_date = nullptr;
  t->fast = compressed->fast;
  t->filter_cutoff = cutoff_day;
  ctx->tables.insert(t);
  const uint64_t words = (t->rows + 31) / 32;
  if (words) {
    if (!filter_malloc(ctx, words * 4, t)) {
      release_table(t);
      return fail(ctx, Q1_ENOMEM, "filter allocation failed");
    }
    void* const f = t->owned[7];
    t->dev.filter = f;
    t->device_bytes = words * 4;
    q1_status s = launch_build_filter((const uint16_t*)compressed->dev.ship_date, t->rows, cutoff_day, (uint32_t*)f,
                                      ctx->d_result, ++ctx->sequence, ctx->stream);
    if (s == Q1_OK) s = wait_sequence(ctx, &ctx->h_result->sequence, ctx->sequence);
    if (s != Q1_OK) {
      release_table(t);
      return fail(ctx, s, "building the filter bitmap failed");
    }
    ctx->last = q1_timing{};
    ctx->last.kernel_ms = clock_ms(ctx, ctx->h_result->clock_begin, ctx->h_result->clock_end);
    ctx->last.rows = t->rows;
    ctx->last.bytes_read = 2 * t->rows + 4 * words;
  }
  *out = t;
  return Q1_OK;
  GUARD_END(ctx)
}

// ---------------------------------------------------------------------------------------
// Results
// ---------------------------------------------------------------------------------------
void q1_aggregates_to_result(const q1_device_aggregates* a, q1_result* out) {
  if (!a || !out) return;
  for (int g = 0; g < Q1_NUM_GROUPS; g++) {
    q1_group& r = out->g[g];
    r.sum_qty = (int64_t)a->sum_qty[g];
    r.sum_base_price = (int64_t)a->sum_base_price[g];
    r.sum_disc_price_lo = a->sum_disc_price_lo[g];
    r.sum_disc_price_hi = (int64_t)a->sum_disc_price_hi[g];
    r.sum_charge_lo = a->sum_charge_lo[g];
    r.sum_charge_hi = (int64_t)a->sum_charge_hi[g];
    r.sum_disc = (int64_t)a->sum_disc[g];
    r.count = (int64_t)a->count[g];
  }
}

void q1_result_merge(const q1_result* a, const q1_result* b, q1_result* out) {
  if (!a || !b || !out) return;
  q1_result r;
  for (int g = 0; g < Q1_NUM_GROUPS; g++) {
    const q1_group &x = a->g[g], &y = b->g[g];
    q1_group& z = r.g[g];
    z.sum_qty = (int64_t)((uint64_t)x.sum_qty + (uint64_t)y.sum_qty);
    z.sum_base_price = (int64_t)((uint64_t)x.sum_base_price + (uint64_t)y.sum_base_price);
    z.sum_disc = (int64_t)((uint64_t)x.sum_disc + (uint64_t)y.sum_disc);
    z.count = (int64_t)((uint64_t)x.count + (uint64_t)y.count);
    z.sum_disc_price_lo = x.sum_disc_price_lo + y.sum_disc_price_lo;
    z.sum_disc_price_hi = (int64_t)((uint64_t)x.sum_disc_price_hi + (uint64_t)y.sum_disc_price_hi +
                                    (z.sum_disc_price_lo < x.sum_disc_price_lo));
    z.sum_charge_lo = x.sum_charge_lo + y.sum_charge_lo;
    z.sum_charge_hi = (int64_t)((uint64_t)x.sum_charge_hi + (uint64_t)y.sum_charge_hi +
                                (z.sum_charge_lo < x.sum_charge_lo));
  }
  *out = r;
}

// ---------------------------------------------------------------------------------------
// The query
// ---------------------------------------------------------------------------------------
static q1_status run_locked(q1_ctx* ctx, const q1_table* t, uint64_t row_begin, uint64_t row_count,
                            int32_t cutoff_day, q1_placement placement, const q1_launch* launch,
                            q1_result* out) {
  if (row_begin > t->rows || row_count > t->rows - row_begin)
    return fail(ctx, Q1_EINVAL, "row range outside the table");
  const q1_placement p = resolve_placement(ctx, t->layout, placement);
  q1_launch l;
  resolve_launch(ctx, t->layout, p, t->fast, row_count, launch, &l);
  LaunchShape shape;
  const char* why = "";
  q1_status s = make_shape(p, t->layout, t->fast, &l, row_begin, row_begin + row_count, &shape, &why);
  if (s != Q1_OK) return fail(ctx, s, why);
  s = ensure_workspace(ctx, scan_workspace_bytes(p, t->fast, shape));
  if (s != Q1_OK) return s;
  ScanArgs a{};
  a.cols = t->dev;
  a.row_begin = row_begin;
  a.row_end = row_begin + row_count;
  a.cutoff_day = t->layout == Q1_LAYOUT_COMPRESSED_PUSHDOWN ? t->filter_cutoff : cutoff_day;
  const auto w0 = std::chrono::steady_clock::now();
  double ms = 0;
  s = scan_to_host(ctx, p, t->layout, t->fast, a, shape);
  if (s == Q1_OK) s = wait_result(ctx, out, &ms);
  if (s != Q1_OK) return s;
  ctx->last = q1_timing{};
  ctx->last.kernel_ms = ms;
  ctx->last.wall_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - w0).count();
  ctx->last.rows = row_count;
  ctx->last.bytes_read = algorithmic_bytes(t->layout, row_count);
  ctx->last.num_blocks = shape.blocks;
  ctx->last.threads_per_block = shape.threads;
  ctx->last.tuples_per_thread = shape.tiles_per_thread * layout_tile_rows(t->layout);
  ctx->last.placement = t->fast ? (uint32_t)p : (uint32_t)Q1_PLACE_IN_REGISTERS_PER_THREAD;
  return Q1_OK;
}

q1_status q1_run(q1_ctx* ctx, const q1_table* t, uint64_t row_begin, uint64_t row_count, int32_t cutoff_day,
                 q1_placement placement, const q1_launch* launch, q1_result* out) {
  if (!ctx || !t || !out || !valid_placement(placement)) return fail(ctx, Q1_EINVAL, "bad argument");
  GUARD_BEGIN
  std::lock_guard<std::mutex> g(ctx->lock);
  return run_locked(ctx, t, row_begin, row_count, cutoff_day, placement, launch, out);
  GUARD_END(ctx)
}

q1_status q1_last_timing(q1_ctx* ctx, q1_timing* out) {
  if (!ctx || !out) return Q1_EINVAL;
  *out = ctx->last;
  return Q1_OK;
}

q1_status q1_enqueue_noalloc(q1_ctx* ctx, q1_placement placement, q1_layout layout, const q1_launch* launch,
                             q1_device_aggregates* aggregates, const q1_columns* device, uint64_t row_begin,
                             uint64_t num_tuples, int32_t cutoff_day, void* hip_stream) {
  if (!ctx || !aggregates || !device || !valid_layout(layout) || !valid_placement(placement))
    return fail(ctx, Q1_EINVAL, "bad argument");
  GUARD_BEGIN
  std::lock_guard<std::mutex> g(ctx->lock);
  uint64_t b[8];
  column_bytes(layout, row_begin + num_tuples, b);
  for (int i = 0; i < 8; i++) {
    if (!b[i]) continue;
    const void* p = colc(*device, i);
    if (!p) return fail(ctx, Q1_EINVAL, "a column required by the layout is NULL");
    if ((uintptr_t)p % 16) return fail(ctx, Q1_EINVAL, "device columns must be 16-byte aligned");
  }
  const q1_placement p = resolve_placement(ctx, layout, placement);
  q1_launch l;
  const bool fast = in_domain_flag(launch);
  resolve_launch(ctx, layout, p, fast, num_tuples, launch, &l, false);
  LaunchShape shape;
  const char* why = "";
  q1_status s = make_shape(p, layout, fast, &l, row_begin, row_begin + num_tuples, &shape, &why);
  if (s != Q1_OK) return fail(ctx, s, why);
  if (!fast && p == Q1_PLACE_GLOBAL) {
    // The any-value kernel runs this launch without per-block tables, with as many blocks as its
    // rows per lane make; the limit on the caller's own grid holds all the same.
    const q1_launch own{launch && launch->threads_per_block ? launch->threads_per_block : 256,
                        launch && launch->tuples_per_thread ? launch->tuples_per_thread : 1024, l.num_blocks, 0};
    LaunchShape asked;
    s = make_shape(p, layout, true, &own, row_begin, row_begin + num_tuples, &asked, &why);
    if (s != Q1_OK) return fail(ctx, s, why);
    if (scan_workspace_bytes(p, true, asked) > kNoallocWorkspaceBytes) return fail(ctx, Q1_EINVAL, kNoallocRefused);
  }
  ScanArgs a{};
  a.cols = *device;
  a.row_begin = row_begin;
  a.row_end = row_begin + num_tuples;
  a.cutoff_day = cutoff_day;
  a.out = aggregates;
  if (!hip_stream) ctx->queued = true;
  // the device's static scratch array instead of the context's merge set and workspace
  s = noalloc_launch_scan(ctx->device, p, layout, fast, a, shape,
                          hip_stream ? hip_stream : (void*)ctx->stream, &why);
  return s == Q1_OK ? Q1_OK : fail(ctx, s, why);
  GUARD_END(ctx)
}

q1_status q1_enqueue(q1_ctx* ctx, q1_placement placement, q1_layout layout, const q1_launch* launch,
                     q1_device_aggregates* aggregates, const q1_columns* device, uint64_t row_begin,
                     uint64_t num_tuples, int32_t cutoff_day, void* hip_stream) {
  if (!ctx || !aggregates || !device || !valid_layout(layout) || !valid_placement(placement))
    return fail(ctx, Q1_EINVAL, "bad argument");
  GUARD_BEGIN
  std::lock_guard<std::mutex> g(ctx->lock);
  uint64_t b[8];
  column_bytes(layout, row_begin + num_tuples, b);
  for (int i = 0; i < 8; i++) {
    if (!b[i]) continue;
    const void* p = colc(*device, i);
    if (!p) return fail(ctx, Q1_EINVAL, "a column required by the layout is NULL");
    if ((uintptr_t)p % 16) return fail(ctx, Q1_EINVAL, "device columns must be 16-byte aligned");
  }
  const q1_placement p = resolve_placement(ctx, layout, placement);
  q1_launch l;
  const bool fast = in_domain_flag(launch);
  resolve_launch(ctx, layout, p, fast, num_tuples, launch, &l, false);
  LaunchShape shape;
  const char* why = "";
  q1_status s = make_shape(p, layout, fast, &l, row_begin, row_begin + num_tuples, &shape, &why);
  if (s != Q1_OK) return fail(ctx, s, why);
  void* stream = hip_stream ? hip_stream : (void*)ctx->stream;
  // The global placement's workspace is per launch: size it and keep launches that
  // share it ordered on the context stream.
  if (p == Q1_PLACE_GLOBAL && stream != (void*)ctx->stream)
    return fail(ctx, Q1_EINVAL, "the global placement enqueues on the context stream only");
  s = ensure_workspace(ctx, scan_workspace_bytes(p, fast, shape));
  if (s != Q1_OK) return s;
  ScanArgs a{};
  a.cols = *device;
  a.row_begin = row_begin;
  a.row_end = row_begin + num_tuples;
  a.cutoff_day = cutoff_day;
  a.out = aggregates;
  if (stream == (void*)ctx->stream) ctx->queued = true;
  s = scan_on(ctx, p, layout, fast, a, shape, stream);
  return s == Q1_OK ? Q1_OK : fail(ctx, s, "scan kernel launch failed");
  GUARD_END(ctx)
}

// ---------------------------------------------------------------------------------------
// Host memory and the autotuning table
// ---------------------------------------------------------------------------------------
void* q1_host_alloc(q1_ctx* ctx, size_t bytes) {
  void* p = nullptr;
  if (hipHostMalloc(&p, bytes ? bytes : 1, hipHostMallocDefault) != hipSuccess) {
    if (ctx) ctx->error = "hipHostMalloc failed";
    return nullptr;
  }
  return p;
}

void q1_host_free(q1_ctx*, void* p) {
  if (p) (void)hipHostFree(p);
}

q1_status q1_tuning_set(q1_ctx* ctx, q1_layout layout, q1_placement placement, const q1_launch* best) {
  if (!ctx || !best || !valid_layout(layout) || placement < 0 || placement > Q1_PLACE_GLOBAL)
    return fail(ctx, Q1_EINVAL, "bad argument");
  LaunchShape shape;
  const char* why = "";
  const q1_status s = make_shape(placement, layout, true, best, 0, 1, &shape, &why);
  if (s != Q1_OK) return fail(ctx, s, why);
  ctx->tuning[layout][placement] = *best;
  ctx->tuning[layout][placement].num_blocks = 0;
  ctx->tuning_at[layout][placement].clear();
  return Q1_OK;
}

q1_status q1_tuning_get(q1_ctx* ctx, q1_layout layout, q1_placement placement, q1_launch* out) {
  if (!ctx || !out || !valid_layout(layout) || !valid_placement(placement)) return Q1_EINVAL;
  *out = ctx->tuning[layout][resolve_placement(ctx, layout, placement)];
  return Q1_OK;
}

q1_status q1_tuning_resolve(q1_ctx* ctx, q1_layout layout, q1_placement placement, uint64_t rows,
                            q1_launch* out) {
  if (!ctx || !out || !valid_layout(layout) || !valid_placement(placement)) return Q1_EINVAL;
  resolve_launch(ctx, layout, resolve_placement(ctx, layout, placement), true, rows, nullptr, out);
  return Q1_OK;
}

q1_status q1_tuning_get_streaming(q1_ctx* ctx, q1_layout layout, uint64_t* chunk_rows, int* num_streams) {
  if (!ctx || !chunk_rows || !num_streams || !valid_layout(layout)) return Q1_EINVAL;
  *chunk_rows = ctx->stream_chunk_rows[layout] ? ctx->stream_chunk_rows[layout] : kStreamChunkRows;
  *num_streams = ctx->stream_count[layout] ? ctx->stream_count[layout] : kStreamCount;
  return Q1_OK;
}

q1_status q1_tuning_set_best_placement(q1_ctx* ctx, q1_layout layout, q1_placement placement) {
  if (!ctx || !valid_layout(layout) || placement < 0 || placement > Q1_PLACE_GLOBAL) return Q1_EINVAL;
  ctx->best[layout] = placement;
  return Q1_OK;
}

int32_t q1_day_number(int32_t year, int32_t month, int32_t day) { return q1::day_number(year, month, day); }

}  // extern "C"

// Cases of the library's host code over the stand-in runtime (hip_standin.h), each run in a
// process of its own: host_cases NAME.  A failed expectation prints its line and exits with 1.
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#include <sys/mman.h>

#include "../../tpchq01_gpu_amd/csrc/q1_internal.h"
#include "hip_standin.h"

using namespace q1;
using standin::state;

#define EXPECT(x)                                                     \
  do {                                                                \
    if (!(x)) {                                                       \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);             \
      std::exit(1);                                                   \
    }                                                                 \
  } while (0)

namespace {

q1_ctx* context() {
  q1_ctx* ctx = nullptr;
  EXPECT(q1_init(0, &ctx) == Q1_OK);
  state().launches.clear();
  state().copies.clear();
  return ctx;
}

// The columns of `rows` rows of a layout at one address each.
struct HostColumns {
  q1_columns c{};
  uint64_t bytes[8] = {};
  const void** slot(int i) {
    const void** s[8] = {&c.ship_date, &c.quantity, &c.extended_price, &c.discount,
                         &c.tax, &c.return_flag, &c.line_status, &c.filter};
    return s[i];
  }
  HostColumns(q1_layout layout, uint64_t rows) {
    q1_layout_column_bytes(layout, rows, bytes);
    for (int i = 0; i < 8; i++)
      if (bytes[i]) {
        *slot(i) = mmap(nullptr, bytes[i], PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
        EXPECT(*slot(i) != MAP_FAILED);
      }
  }
};

const ScanArgs& scan_args(const standin::Launch& l) { return *(const ScanArgs*)l.scan_args.data(); }

// The bytes that copy kernels read from host memory.
uint64_t fetched() {
  uint64_t n = 0;
  for (const standin::Launch& l : state().launches)
    if (l.is("fetch_columns"))
      for (uint64_t b : ((const FetchArgs*)l.fetch_args.data())->bytes) n += b;
  return n;
}
uint64_t copied_in() {
  uint64_t n = 0;
  for (const standin::Copy& c : state().copies) n += c.to_device ? c.bytes : 0;
  return n;
}

// ---------------------------------------------------------------------------------------------
// Host columns pinned in pieces, with pageable memory between them: no kernel may read them.
void streaming_columns_pinned_in_pieces() {
  const uint64_t rows = 1u << 20;
  for (uint64_t chunk : {rows, rows / 4}) {
    for (int holed = 0; holed < 7; holed++) {
      q1_ctx* ctx = context();
      HostColumns h(Q1_LAYOUT_COMPRESSED, rows);
      for (int i = 0; i < 7; i++) {
        const char* p = (const char*)*h.slot(i);
        if (i != holed) {
          standin::pin(p, h.bytes[i]);
          continue;
        }
        // every chunk's first and last 4 KiB pinned, the middle of it not
        const uint64_t piece = h.bytes[i] / (rows / chunk);
        for (uint64_t at = 0; at < h.bytes[i]; at += piece) {
          standin::pin(p + at, 4096);
          standin::pin(p + at + piece - 4096, 4096);
        }
      }
      q1_result r;
      EXPECT(q1_run_streaming(ctx, Q1_LAYOUT_COMPRESSED, &h.c, rows, 729999, Q1_PLACE_AUTO, nullptr, chunk, 2, &r) == Q1_OK);
      uint64_t all = 0;
      for (uint64_t b : h.bytes) all += b;
      EXPECT(fetched() == 0);
      EXPECT(copied_in() == all);
      q1_shutdown(ctx);
    }
  }
}

// Pinned columns, also where they begin inside their range, are read by the copy kernel.
void streaming_pinned_columns() {
  const uint64_t rows = 1u << 20;
  q1_ctx* ctx = context();
  HostColumns h(Q1_LAYOUT_COMPRESSED, rows);
  uint64_t all = 0;
  for (int i = 0; i < 7; i++) {
    char* range = (char*)std::calloc(1, h.bytes[i] + 16);
    standin::pin(range, h.bytes[i] + 16);
    *h.slot(i) = range + (i % 2 ? 16 : 0);
    all += h.bytes[i];
  }
  q1_result r;
  EXPECT(q1_run_streaming(ctx, Q1_LAYOUT_COMPRESSED, &h.c, rows, 729999, Q1_PLACE_AUTO, nullptr, rows / 4, 2, &r) == Q1_OK);
  EXPECT(fetched() == all && copied_in() == 0);
  q1_shutdown(ctx);
}

// Device columns that nothing reads.
q1_columns device_columns(q1_layout layout, uint64_t rows) { return HostColumns(layout, rows).c; }

const standin::Launch& last_scan() {
  for (size_t i = state().launches.size(); i-- > 0;)
    if (!state().launches[i].scan_args.empty()) return state().launches[i];
  std::printf("no scan was launched\n");
  std::exit(1);
}

// A launch that a graph records uses no merge set, on the context's stream as on a caller's: its
// replays may overlap whatever else uses the set.
void enqueue_under_capture() {
  q1_ctx* ctx = context();
  const uint64_t rows = 1u << 20;
  const q1_columns cols = device_columns(Q1_LAYOUT_COMPRESSED, rows);
  static q1_device_aggregates sums;
  hipStream_t own = nullptr;
  EXPECT(hipStreamCreateWithFlags(&own, 0) == hipSuccess);
  for (uint32_t flags : {0u, Q1_LAUNCH_ASSUME_TPCH_DOMAIN})
    for (void* stream : {q1_stream(ctx), (void*)own})
      for (bool capture : {false, true, false}) {
        const q1_launch l{64, 16, 0, flags};  // 1024 blocks
        state().capturing = capture ? stream : nullptr;
        EXPECT(q1_enqueue(ctx, Q1_PLACE_IN_REGISTERS, Q1_LAYOUT_COMPRESSED, &l, &sums, &cols, 0, rows, 729999, stream) ==
               Q1_OK);
        state().capturing = nullptr;
        const standin::Launch& scan = last_scan();
        EXPECT(scan.captured == capture && scan.grid == 1024 && scan.stream == stream);
        EXPECT((scan_args(scan).set == nullptr) == capture);
        EXPECT(!capture || scan_args(scan).done == nullptr);
      }
  q1_shutdown(ctx);
}

// A launch that ends without its result leaves no partial sums or block counts behind for the
// launches after it.
void merge_set_after_a_lost_result() {
  q1_ctx* ctx = context();
  HostColumns h(Q1_LAYOUT_COMPRESSED, 1u << 20);
  q1_table* t = nullptr;
  EXPECT(q1_table_wrap(ctx, Q1_LAYOUT_COMPRESSED, &h.c, 1u << 20, &t) == Q1_OK);
  std::memset((void*)ctx->set, 0x55, sizeof(MergeSet));
  state().silent = true;
  q1_result r;
  EXPECT(q1_run(ctx, t, 0, 1u << 20, 729999, Q1_PLACE_AUTO, nullptr, &r) == Q1_EDEVICE);
  state().silent = false;
  for (uint32_t i = 0; i < kSpreadTables; i++) {
    EXPECT(ctx->set->table[i].merged == 0 && ctx->set->table[i].tables_merged == 0);
    EXPECT(ctx->set->table[i].sums.count[0] == 0);
  }
  EXPECT(ctx->set->clock_begin == 0);
  EXPECT(q1_run(ctx, t, 0, 1u << 20, 729999, Q1_PLACE_AUTO, nullptr, &r) == Q1_OK);
  q1_table_free(t);
  q1_shutdown(ctx);
}

// Calls of q1_enqueue_noalloc that overlapped spoil their own results only: whatever they left in
// the merge set they share is cleared, in the later call's own stream, before its scan.
void noalloc_after_an_overlap() {
  q1_ctx* ctx = context();
  const uint64_t rows = 1u << 20;
  const q1_columns cols = device_columns(Q1_LAYOUT_COMPRESSED, rows);
  static q1_device_aggregates sums;
  hipStream_t own = nullptr;
  EXPECT(hipStreamCreateWithFlags(&own, 0) == hipSuccess);
  for (uint32_t flags : {0u, Q1_LAUNCH_ASSUME_TPCH_DOMAIN})
    for (void* stream : {q1_stream(ctx), (void*)own})
      for (bool capture : {false, true}) {
        const q1_launch l{64, 16, 0, flags};  // 1024 blocks
        auto enqueue = [&] {
          return q1_enqueue_noalloc(ctx, Q1_PLACE_IN_REGISTERS, Q1_LAYOUT_COMPRESSED, &l, &sums, &cols, 0, rows, 729999,
                                    stream);
        };
        EXPECT(enqueue() == Q1_OK);
        MergeSet* set = scan_args(last_scan()).set;
        EXPECT(set != nullptr);
        std::memset((void*)set, 0x55, sizeof(MergeSet));
        state().launches.clear();
        state().capturing = capture ? stream : nullptr;
        EXPECT(enqueue() == Q1_OK);
        state().capturing = nullptr;
        EXPECT(scan_args(last_scan()).set == set);
        EXPECT(state().launches.size() == 2 && state().launches[0].is("zero_words"));
        for (const standin::Launch& k : state().launches) EXPECT(k.stream == stream && k.captured == capture);
        EXPECT(state().launches[0].grid * state().launches[0].block * 8ull >= sizeof(MergeSet));
        const MergeSet clear{};
        EXPECT(capture || std::memcmp(set, &clear, sizeof(MergeSet)) == 0);
      }
  q1_shutdown(ctx);
}

// The global placement's workspaces of the streaming pipeline grow until memory runs out: the next
// call, which needs no more than the first had, launches no kernel without one.
void streaming_workspace_after_a_failed_growth() {
  q1_ctx* ctx = context();
  const uint64_t rows = 1u << 22, chunk = 1u << 20;
  HostColumns h(Q1_LAYOUT_COMPRESSED, rows);
  auto stream = [&](uint32_t threads, uint32_t tuples) {
    const q1_launch l{threads, tuples, 0, Q1_LAUNCH_ASSUME_TPCH_DOMAIN};
    q1_result r;
    state().launches.clear();
    const q1_status s =
        q1_run_streaming(ctx, Q1_LAYOUT_COMPRESSED, &h.c, rows, 729999, Q1_PLACE_GLOBAL, &l, chunk, 2, &r);
    for (const standin::Launch& k : state().launches) EXPECT(!k.is("scan_fast") || k.workspace != nullptr);
    return s;
  };
  EXPECT(stream(256, 1024) == Q1_OK);
  const uint64_t larger = 1024 * 240;  // the tables of a chunk's 1024 blocks
  state().budget = state().device_bytes + larger;
  EXPECT(stream(64, 16) == Q1_ENOMEM);
  state().budget = UINT64_MAX;
  EXPECT(stream(256, 1024) == Q1_OK);
  EXPECT(stream(64, 16) == Q1_OK);
  q1_shutdown(ctx);
}

// The bitmap of a freed pushdown table, kept for the next one, is given back to whatever allocation
// of the library finds no memory left.
void spare_bitmap_given_back() {
  const uint64_t rows = 1u << 26;  // a bitmap of 8 MiB
  static HostColumns h(Q1_LAYOUT_COMPRESSED, rows);
  auto with_spare = [&](q1_ctx* ctx, const q1_table* t) {
    q1_table* f = nullptr;
    EXPECT(q1_build_filter(ctx, t, 729999, &f) == Q1_OK);
    q1_table_free(f);
    EXPECT(ctx->spare.bytes == rows / 8);
    state().budget = state().device_bytes;
  };
  auto given_back = [&](const q1_ctx* ctx) {
    state().budget = UINT64_MAX;
    return ctx->spare.p == nullptr;
  };
  q1_ctx* ctx = context();
  q1_table* t = nullptr;
  EXPECT(q1_table_wrap(ctx, Q1_LAYOUT_COMPRESSED, &h.c, rows, &t) == Q1_OK);
  q1_result r[2];
  // a table's columns
  with_spare(ctx, t);
  q1_table* made = nullptr;
  EXPECT(q1_table_generate(ctx, Q1_LAYOUT_COMPRESSED, 1, 10000, &made) == Q1_OK && given_back(ctx));
  q1_table_free(made);
  // the staging buffers of the streaming pipeline, and its workspaces
  const q1_launch few{256, 16, 0, Q1_LAUNCH_ASSUME_TPCH_DOMAIN};
  for (q1_placement p : {Q1_PLACE_IN_REGISTERS, Q1_PLACE_GLOBAL}) {
    with_spare(ctx, t);
    EXPECT(q1_run_streaming(ctx, Q1_LAYOUT_COMPRESSED, &h.c, 4096, 729999, p, &few, 1024, 2, r) == Q1_OK && given_back(ctx));
  }
  // the buffers of a batch
  with_spare(ctx, t);
  const q1_request reqs[2] = {{t, 0, 1000, 729999, 0}, {t, 5, 1000, 729999, 0}};
  EXPECT(q1_run_batch(ctx, reqs, 2, nullptr, r) == Q1_OK && given_back(ctx));
  // a server's merge sets
  with_spare(ctx, t);
  q1_server* sv = nullptr;
  EXPECT(q1_server_create(ctx, nullptr, &sv) == Q1_OK && given_back(ctx));
  q1_server_destroy(sv);
  q1_table_free(t);
  q1_shutdown(ctx);
}

// Launches of the any-value kernel need no per-block tables, whatever the placement and however
// many blocks the kernel's own limit of rows per lane makes of the launch: q1_enqueue_noalloc takes
// them, except for grids of more than 34952 blocks that the caller asks for itself.
void any_value_launches_need_no_workspace() {
  q1_ctx* ctx = context();
  static q1_device_aggregates sums;
  const uint64_t rows = 600'000'000;
  for (q1_layout layout : {Q1_LAYOUT_REFERENCE, Q1_LAYOUT_UNCOMPRESSED, Q1_LAYOUT_COMPRESSED, Q1_LAYOUT_COMPRESSED_PUSHDOWN}) {
    const q1_columns cols = device_columns(layout, rows);
    auto noalloc = [&](uint32_t threads, uint32_t tuples, uint32_t blocks, uint32_t flags = 0) {
      const q1_launch l{threads, tuples, blocks, flags};
      return q1_enqueue_noalloc(ctx, Q1_PLACE_GLOBAL, layout, &l, &sums, &cols, 0, rows, 729999, q1_stream(ctx));
    };
    EXPECT(q1_enqueue_noalloc(ctx, Q1_PLACE_GLOBAL, layout, nullptr, &sums, &cols, 0, rows, 729999, nullptr) == Q1_OK);
    EXPECT(noalloc(0, 0, 0) == Q1_OK);
    EXPECT(noalloc(256, 1024, 0) == Q1_OK);   // 2289 blocks asked for
    EXPECT(noalloc(64, 16384, 0) == Q1_OK);
    EXPECT(noalloc(64, 512, 0) == Q1_OK);     // 18311
    EXPECT(noalloc(0, 0, 3000) == Q1_OK);
    EXPECT(noalloc(64, 1024, 34952) == Q1_OK);
    EXPECT(noalloc(64, 1024, 34953) == Q1_EINVAL);
    EXPECT(noalloc(64, 256, 0) == Q1_EINVAL);  // 36622
    EXPECT(noalloc(64, 16, 0) == Q1_EINVAL);
    EXPECT(noalloc(64, 256, 0, Q1_LAUNCH_ASSUME_TPCH_DOMAIN) == Q1_EINVAL);
    // nor does the launch that may allocate
    const uint64_t before = state().device_bytes;
    EXPECT(q1_enqueue(ctx, Q1_PLACE_GLOBAL, layout, nullptr, &sums, &cols, 0, rows, 729999, nullptr) == Q1_OK);
    EXPECT(state().device_bytes == before);
  }
  q1_shutdown(ctx);
}

// q1_table_free returns once the work that may read the table has ended, as freeing its memory did:
// queued on the context's stream, which callers can also get and use themselves, or for a filter
// bitmap whose address was handed out, on any stream.
void table_free_waits() {
  const uint64_t rows = 1u << 20;
  HostColumns h(Q1_LAYOUT_COMPRESSED, rows);
  static q1_device_aggregates sums;
  q1_result r;
  auto wrapped = [&](q1_ctx* ctx) {
    q1_table* t = nullptr;
    EXPECT(q1_table_wrap(ctx, Q1_LAYOUT_COMPRESSED, &h.c, rows, &t) == Q1_OK);
    return t;
  };
  auto waits_for_stream = [&](q1_table* t) {
    state().stream_waits = 0;
    q1_table_free(t);
    return state().stream_waits > 0;
  };
  q1_ctx* ctx = context();
  auto enqueue = [&](bool noalloc) {
    EXPECT((noalloc ? q1_enqueue_noalloc : q1_enqueue)(ctx, Q1_PLACE_IN_REGISTERS, Q1_LAYOUT_COMPRESSED, nullptr, &sums,
                                                       &h.c, 0, rows, 729999, nullptr) == Q1_OK);
  };
  for (bool noalloc : {false, true}) {
    q1_table* t = wrapped(ctx);
    enqueue(noalloc);
    EXPECT(waits_for_stream(t));
    // calls without rows launch nothing that could be waited for
    t = wrapped(ctx);
    enqueue(noalloc);
    EXPECT(q1_run(ctx, t, 0, 0, 729999, Q1_PLACE_AUTO, nullptr, &r) == Q1_OK);
    const q1_request none{t, 5, 0, 729999, 0};
    EXPECT(q1_run_batch(ctx, &none, 1, nullptr, &r) == Q1_OK);
    EXPECT(waits_for_stream(t));
    // nothing is queued behind a query's result
    t = wrapped(ctx);
    enqueue(noalloc);
    EXPECT(q1_run(ctx, t, 0, rows, 729999, Q1_PLACE_AUTO, nullptr, &r) == Q1_OK);
    EXPECT(!waits_for_stream(t));
  }
  // a bitmap on other streams
  q1_table *t = wrapped(ctx), *f = nullptr;
  EXPECT(q1_build_filter(ctx, t, 729999, &f) == Q1_OK);
  q1_columns dev;
  EXPECT(q1_table_info(f, nullptr, nullptr, &dev) == Q1_OK);
  state().device_waits = state().frees = 0;
  q1_table_free(f);
  EXPECT(state().device_waits + state().frees > 0);
  // the caller's own work on the context's stream
  EXPECT(q1_stream(ctx) != nullptr);
  EXPECT(waits_for_stream(t));
  q1_shutdown(ctx);
}

// A process that asked for blocking waits (hipDeviceScheduleBlockingSync) gets the runtime's wait,
// which sleeps, for a result that takes a while; by default the host watches for it.
void waits_follow_the_device_flags() {
  q1_ctx* ctx = context();
  const uint64_t rows = 1u << 20;
  HostColumns h(Q1_LAYOUT_COMPRESSED, rows);
  q1_table* t = nullptr;
  EXPECT(q1_table_wrap(ctx, Q1_LAYOUT_COMPRESSED, &h.c, rows, &t) == Q1_OK);
  state().late_stream = (void*)ctx->stream;
  state().late_us = 300;
  for (unsigned flags : {(unsigned)hipDeviceScheduleAuto, (unsigned)hipDeviceScheduleSpin,
                         (unsigned)(hipDeviceScheduleBlockingSync | hipDeviceMapHost)}) {
    state().device_flags = flags;
    const bool blocking = flags & hipDeviceScheduleBlockingSync;
    q1_result r;
    state().stream_waits = 0;
    EXPECT(q1_run(ctx, t, 0, rows, 729999, Q1_PLACE_AUTO, nullptr, &r) == Q1_OK);
    EXPECT((state().stream_waits > 0) == blocking);
    const q1_request reqs[2] = {{t, 0, rows, 729999, 0}, {t, 32, 1000, 729999, 0}};
    q1_result rs[2];
    state().stream_waits = 0;
    EXPECT(q1_run_batch(ctx, reqs, 2, nullptr, rs) == Q1_OK);
    EXPECT((state().stream_waits > 0) == blocking);
  }
  state().late_us = 0;
  q1_table_free(t);
  q1_shutdown(ctx);
}

const std::map<std::string, void (*)()> kCases = {
    {"waits_follow_the_device_flags", waits_follow_the_device_flags},
    {"table_free_waits", table_free_waits},
    {"any_value_launches_need_no_workspace", any_value_launches_need_no_workspace},
    {"spare_bitmap_given_back", spare_bitmap_given_back},
    {"streaming_workspace_after_a_failed_growth", streaming_workspace_after_a_failed_growth},
    {"noalloc_after_an_overlap", noalloc_after_an_overlap},
    {"merge_set_after_a_lost_result", merge_set_after_a_lost_result},
    {"enqueue_under_capture", enqueue_under_capture},
    {"streaming_columns_pinned_in_pieces", streaming_columns_pinned_in_pieces},
    {"streaming_pinned_columns", streaming_pinned_columns},
};

}  // namespace

int main(int argc, char** argv) {
  if (argc < 2) {
    for (const auto& c : kCases) std::printf("%s\n", c.first.c_str());
    return 0;
  }
  const auto it = kCases.find(argv[1]);
  if (it == kCases.end()) return 2;
  it->second();
  return 0;
}

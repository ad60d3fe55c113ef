// gfx950 utility kernels (zero fill, generator, domain check, pushdown producer), kernel dispatch
// and the host-side launch helpers of the TPC-H Q1 path.  The scan kernels themselves are in
// q1_scan.h, instantiated per layout.
#include <algorithm>
#include <type_traits>

#include "q1_scan.h"

namespace q1 {
namespace {

// ------------------------------------------------------------------------------------
// Utility kernels: zero fill, generator, domain check, pushdown producer.
// ------------------------------------------------------------------------------------
__global__ void zero_words(uint64_t* p, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// One thread per 32-row group writes the rows' values and the packed words of the group.
template <int L>
__global__ void generate_rows(uint64_t seed, uint64_t rows, q1_columns c) {
  const uint64_t grp = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t r0 = grp * 32;
  if (r0 >= rows) return;
  const uint64_t r1 = r0 + 32 < rows ? r0 + 32 : rows;
  uint32_t rfw[2] = {0, 0}, lsw = 0;
  for (uint64_t r = r0; r < r1; r++) {
    const GenRow g = gen_row(seed, r);
    const uint32_t j = (uint32_t)(r - r0);
    if (L == Q1_LAYOUT_REFERENCE) {
      ((int32_t*)c.ship_date)[r] = g.ship_date;
      ((int64_t*)c.quantity)[r] = (int64_t)g.quantity * 100;
      ((int64_t*)c.extended_price)[r] = g.extended_price;
      ((int64_t*)c.discount)[r] = g.discount;
      ((int64_t*)c.tax)[r] = g.tax;
      ((char*)c.return_flag)[r] = g.return_flag;
      ((char*)c.line_status)[r] = g.line_status;
    } else if (L == Q1_LAYOUT_UNCOMPRESSED) {
      ((int32_t*)c.ship_date)[r] = g.ship_date;
      ((int32_t*)c.quantity)[r] = g.quantity * 100;
      ((int64_t*)c.extended_price)[r] = g.extended_price;
      ((int8_t*)c.discount)[r] = (int8_t)g.discount;
      ((int8_t*)c.tax)[r] = (int8_t)g.tax;
      ((char*)c.return_flag)[r] = g.return_flag;
      ((char*)c.line_status)[r] = g.line_status;
    } else {
      ((uint16_t*)c.ship_date)[r] = (uint16_t)(g.ship_date - kShipDateFrameOfReference);
      ((uint8_t*)c.quantity)[r] = (uint8_t)g.quantity;
      ((uint32_t*)c.extended_price)[r] = (uint32_t)g.extended_price;
      ((uint8_t*)c.discount)[r] = (uint8_t)g.discount;
      ((uint8_t*)c.tax)[r] = (uint8_t)g.tax;
      rfw[j >> 4] |= encode_return_flag((uint32_t)g.return_flag) << (2 * (j & 15));
      lsw |= encode_line_status((uint32_t)g.line_status) << j;
    }
  }
  if (L == Q1_LAYOUT_COMPRESSED || L == Q1_LAYOUT_COMPRESSED_PUSHDOWN) {
    uint32_t* rf = (uint32_t*)c.return_flag;
    rf[2 * grp] = rfw[0];
    if (r0 + 16 < rows) rf[2 * grp + 1] = rfw[1];
    ((uint32_t*)c.line_status)[grp] = lsw;
  }
}

// The end of a kernel that leaves no sums, called by wavefront 0 of a block: the count of
// finished blocks, whose last one tells the host.
__device__ __forceinline__ void end_counted(const Completion& c) {
  MergeSet* const set = c.set;
  const uint32_t grid = gridDim.x, b = blockIdx.x, mask = kSpreadTables - 1;
  const uint32_t used = grid < kSpreadTables ? grid : kSpreadTables;
  if (!count_block(set->table, b & mask, blocks_sharing(grid, b, mask), used)) return;
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if ((threadIdx.x & 63) == 0) store_host(&c.host->sequence, c.sequence);
}

// The value-domain check: host->outside becomes whether any discount, tax, quantity or price
// lies outside the TPC-H domain (domain_is_tpch's limits).
// HBM bounds it: 7 (compressed), 14 or 32 bytes per row are read once and nothing is written
// for a table inside the domain.  Each column is read as 16-byte vectors with no regard to
// rows: a limit of the form 2^k - 1 is a test of bits, so a lane ORs what it reads of such a
// column and tests the OR; quantities in hundredths (at most 6300) keep a maximum.  A block
// takes kDomainRows rows: its 14 to 16 loads per lane, each a contiguous stretch of the
// block's share of a column, are all issued before any is used.  The loads are ordinary ones,
// which pass through the memory-side cache and so write back what the columns' producer
// left there: after them the first query of 600M freshly written rows takes 880 us, after
// non-temporal ones 990 (checks 0.67 and 0.61 ms).
// With its launch and wait, 60M compressed rows take 72 us.  Grid-strided columns one after
// another, four vectors in flight per lane, took 83 us; the per-row minimum and maximum of
// every column, merged with eight 64-bit atomics per wavefront into one line, 1.55 ms.
template <int L>
constexpr int kDomainRows = L == Q1_LAYOUT_REFERENCE ? 2048 : L == Q1_LAYOUT_UNCOMPRESSED ? 4096 : 8192;

// A lane's vectors of one block's share of a column of T values, at most LIMIT each.
template <typename T, uint32_t LIMIT, int ROWS>
struct DomainColumn {
  static constexpr bool kBits = (LIMIT & (LIMIT + 1)) == 0;
  static constexpr int kPer = 16 / sizeof(T);              // values per vector
  static constexpr int kVectors = ROWS / kPer / 256;       // vectors per lane
  static_assert(kVectors >= 1 && (kBits || sizeof(T) >= 4), "whole vectors; byte columns have limits 2^k - 1");
  uint4 v[kVectors];

  // WHOLE: the block's rows all lie in the column; otherwise vectors past its last whole
  // one are taken as zero.
  template <bool WHOLE>
  __device__ __forceinline__ void load(const void* col, uint64_t block, uint64_t rows) {
    const uint64_t first = block * (ROWS / kPer) + threadIdx.x;
#pragma unroll
    for (int k = 0; k < kVectors; k++) {
      const uint64_t i = first + k * 256;
      v[k] = WHOLE || i < rows / kPer ? reinterpret_cast<const uint4*>(col)[i] : make_uint4(0, 0, 0, 0);
    }
  }
  __device__ __forceinline__ bool outside() const {
    uint4 a = v[0];
#pragma unroll
    for (int k = 1; k < kVectors; k++) {
      if (kBits) {
        a.x |= v[k].x; a.y |= v[k].y; a.z |= v[k].z; a.w |= v[k].w;
      } else {
        a.x = max(a.x, v[k].x); a.y = max(a.y, v[k].y); a.z = max(a.z, v[k].z); a.w = max(a.w, v[k].w);
      }
    }
    if constexpr (kBits) {
      constexpr uint32_t low = sizeof(T) == 1 ? (~LIMIT & 0xFFu) * 0x01010101u : ~LIMIT;
      constexpr uint32_t high = sizeof(T) == 8 ? 0xFFFFFFFFu : low;
      return ((a.x | a.z) & low) != 0 || ((a.y | a.w) & high) != 0;
    } else {
      return max(a.x, a.z) > LIMIT || max(a.y, a.w) > (sizeof(T) == 8 ? 0u : LIMIT);
    }
  }
  // One of the up to 15 values behind the column's last whole vector.
  __device__ __forceinline__ static bool tail_outside(const void* col, uint64_t rows) {
    const uint64_t r = rows / kPer * kPer + threadIdx.x;
    if (r >= rows) return false;
    const int64_t x = (int64_t)reinterpret_cast<const T*>(col)[r];
    return x < 0 || x > (int64_t)LIMIT;
  }
};

template <typename Narrow, typename Qty, uint32_t QTY_LIMIT, typename Price, int ROWS>
__device__ __forceinline__ bool block_outside(const q1_columns& c, uint64_t rows) {
  DomainColumn<Narrow, 15, ROWS> d, x;
  DomainColumn<Qty, QTY_LIMIT, ROWS> q;
  DomainColumn<Price, (1u << 24) - 1, ROWS> p;
  const uint64_t b = blockIdx.x;
  bool tail = false;
  if ((b + 1) * ROWS <= rows) {
    d.template load<true>(c.discount, b, rows);
    x.template load<true>(c.tax, b, rows);
    q.template load<true>(c.quantity, b, rows);
    p.template load<true>(c.extended_price, b, rows);
  } else {
    d.template load<false>(c.discount, b, rows);
    x.template load<false>(c.tax, b, rows);
    q.template load<false>(c.quantity, b, rows);
    p.template load<false>(c.extended_price, b, rows);
    tail = d.tail_outside(c.discount, rows) | x.tail_outside(c.tax, rows) | q.tail_outside(c.quantity, rows) |
           p.tail_outside(c.extended_price, rows);
  }
  return tail | d.outside() | x.outside() | q.outside() | p.outside();
}

// Larger grids do not count their blocks: a block lives for one round of loads, which the
// count lengthens.  Check and wait, counted / not: 1M compressed rows (123 blocks) 10.1 / 12.3
// us, 60M (7,325 blocks) 77 / 77, 600M 694 / 672.
constexpr uint64_t kDomainCountedBlocks = 4096;
// COUNTED: the last of its blocks tells the host; otherwise the caller waits for the kernel's
// end, host->outside being 0 before.
template <int L, bool COUNTED>
__global__ void __launch_bounds__(256) domain_check(q1_columns c, uint64_t rows, Completion done) {
  bool bad;
  if constexpr (L == Q1_LAYOUT_REFERENCE)
    bad = block_outside<int64_t, int64_t, 6300, int64_t, kDomainRows<L>>(c, rows);
  else if constexpr (L == Q1_LAYOUT_UNCOMPRESSED)
    bad = block_outside<int8_t, int32_t, 6300, int64_t, kDomainRows<L>>(c, rows);
  else
    bad = block_outside<uint8_t, uint8_t, 63, uint32_t, kDomainRows<L>>(c, rows);
  // The first block to find a value outside tells the host: a table with many would have
  // every wavefront write to it over PCIe (1.1 ms at 60M rows).
  auto report = [&] {
    uint64_t* const seen = &done.set->outside;
    if (__hip_atomic_load(seen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != done.sequence &&
        atomicExch((unsigned long long*)seen, (unsigned long long)done.sequence) != done.sequence)
      store_host(&done.host->outside, 1);
  };
  if (COUNTED) {
    const bool outside = __syncthreads_or(bad);
    if (threadIdx.x < 64) {
      if (outside && threadIdx.x == 0) report();
      end_counted(done);
    }
  } else if (ballot(bad) && (threadIdx.x & 63) == 0) {
    report();
  }
}

// The pushdown producer (src/main.cu:362-389 semantics, runtime cutoff).  A lane turns the
// 8 ship dates of rows [8g, 8g + 8) -- one 16-byte load -- into 8 filter bits, and four
// neighbouring lanes' bytes make one 32-bit word of the bitmap, which the first of them
// writes.  Each lane takes kFilterGroups such groups a block-width apart (a wavefront
// reads 1 KiB of the column contiguously per group) and issues all their loads before it
// uses any: a block covers 8,192 rows, a quarter of the blocks of one lane per group, and
// each lane keeps 64 bytes in flight.  At 600M rows 4 groups per lane took 0.200-0.209 ms,
// 1, 8, 16 and 32 groups 0.232, 0.211, 0.218 and 0.228 ms.  The column must be 16-byte
// aligned (as every table column is).
// The host watches for report_end's word: with its launch and wait 60M rows take 29 us, with two
// events and the stream's wait 34; 100,000 rows 11 and 18.
constexpr int kFilterGroups = 4;
__global__ void __launch_bounds__(256) build_filter(const uint16_t* ship, uint64_t rows, int32_t cut,
                                                    uint32_t* filter, uint64_t* clock_begin) {
  if (blockIdx.x == 0 && threadIdx.x == 0) store_host(clock_begin, wall_clock64());
  const uint64_t full = rows / 8;  // groups of 8 rows inside the column
  const uint64_t g0 = (uint64_t)blockIdx.x * 256 * kFilterGroups + threadIdx.x;
  uint4 v[kFilterGroups];
#pragma unroll
  for (int k = 0; k < kFilterGroups; k++) {
    const uint64_t g = g0 + (uint64_t)k * 256;
    v[k] = g < full ? nt_load(reinterpret_cast<const uint4*>(ship) + g) : make_uint4(0, 0, 0, 0);
  }
#pragma unroll
  for (int k = 0; k < kFilterGroups; k++) {
    const uint64_t g = g0 + (uint64_t)k * 256, r0 = g * 8;
    uint32_t bits = 0;
    if (g < full) {
      const uint32_t w[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
#pragma unroll
      for (int q = 0; q < 4; q++)
        bits |= (uint32_t)((int32_t)(w[q] & 0xFFFFu) <= cut) << (2 * q) |
                (uint32_t)((int32_t)(w[q] >> 16) <= cut) << (2 * q + 1);
    } else if (r0 < rows) {
      for (uint32_t j = 0; r0 + j < rows; j++) bits |= (uint32_t)((int32_t)ship[r0 + j] <= cut) << j;
    }
    // every lane takes part in the exchange, inside the range or not
    uint32_t word = bits << (8 * (threadIdx.x & 3));
    word |= __shfl_xor(word, 1, 64);
    word |= __shfl_xor(word, 2, 64);
    if ((threadIdx.x & 3) == 0 && r0 < rows) filter[g / 4] = word;
  }
  if (blockIdx.x == 0) __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the clock is there before report_end's
}

// Columns out of pinned host memory.  PCIe bounds it (57 GB/s), or its latency.  A block takes
// pieces of 16 KiB of one column, every lane's loads all issued before any is stored: 128 blocks
// keep 2 MiB in flight, which PCIe fills (200M rows 32.8-33.0 ms, as with 512; 64 blocks 33.2-33.4),
// and leave the compute units to the scans of other streams.  System-scope loads go past the caches, where lines of host memory
// that the caller has written since may be, and do not wait for them: 45 GB/s with ordinary ones.
__device__ __forceinline__ uint64_t load_host(const uint64_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
constexpr uint32_t kFetchPiece = 256 * 8 * 8, kFetchBlocks = 128;
inline uint64_t fetch_pieces(const FetchArgs& f) {
  uint64_t n = 0;
  for (uint64_t bytes : f.bytes) n += (bytes + kFetchPiece - 1) / kFetchPiece;
  return n;
}
__global__ void __launch_bounds__(256) fetch_columns(FetchArgs f, uint64_t pieces) {
  if (blockIdx.x == 0 && threadIdx.x == 0 && f.clock_begin) {
    store_host(f.clock_begin, wall_clock64());
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  for (uint64_t next = blockIdx.x; next < pieces; next += gridDim.x) {
    uint64_t piece = next;
    int k = 0;
    for (;; k++) {
      const uint64_t n = (f.bytes[k] + kFetchPiece - 1) / kFetchPiece;
      if (piece < n) break;
      piece -= n;
    }
    const uint64_t bytes = f.bytes[k], words = bytes / 8, w0 = piece * (kFetchPiece / 8) + threadIdx.x;
    const uint64_t* src = reinterpret_cast<const uint64_t*>(f.src[k]);
    uint64_t* dst = reinterpret_cast<uint64_t*>(f.dst[k]);
    uint64_t v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = w0 + i * 256 < words ? load_host(src + w0 + i * 256) : 0;
#pragma unroll
    for (int i = 0; i < 8; i++)
      if (w0 + i * 256 < words) dst[w0 + i * 256] = v[i];
    // the column's last bytes behind its last whole word, with its last piece
    const uint64_t tail = words * 8 + threadIdx.x;
    if ((piece + 1) * kFetchPiece >= bytes && tail < bytes)
      reinterpret_cast<uint8_t*>(f.dst[k])[tail] = __hip_atomic_load(
          reinterpret_cast<const uint8_t*>(f.src[k]) + tail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// ------------------------------------------------------------------------------------
// Dispatch
// ------------------------------------------------------------------------------------
FastFn fast_kernel(q1_layout l, int p, uint32_t threads) {
  switch (l) {
    case Q1_LAYOUT_REFERENCE: return fast_kernel_reference(p, threads);
    case Q1_LAYOUT_UNCOMPRESSED: return fast_kernel_uncompressed(p, threads);
    case Q1_LAYOUT_COMPRESSED: return fast_kernel_compressed(p, threads);
    default: return fast_kernel_pushdown(p, threads);
  }
}

GenFn direct_kernel(q1_layout l, uint32_t threads) {
  switch (l) {
    case Q1_LAYOUT_REFERENCE: return direct_kernel_reference(threads);
    case Q1_LAYOUT_UNCOMPRESSED: return direct_kernel_uncompressed(threads);
    case Q1_LAYOUT_COMPRESSED: return direct_kernel_compressed(threads);
    default: return direct_kernel_pushdown(threads);
  }
}

GenFn any_kernel(q1_layout l, uint32_t threads) {
  switch (l) {
    case Q1_LAYOUT_REFERENCE: return any_kernel_reference(threads);
    case Q1_LAYOUT_UNCOMPRESSED: return any_kernel_uncompressed(threads);
    case Q1_LAYOUT_COMPRESSED: return any_kernel_compressed(threads);
    default: return any_kernel_pushdown(threads);
  }
}

uint32_t any_kernel_lds(q1_layout l, uint32_t threads) {
  switch (l) {
    case Q1_LAYOUT_REFERENCE: return any_kernel_lds_reference(threads);
    case Q1_LAYOUT_UNCOMPRESSED: return any_kernel_lds_uncompressed(threads);
    case Q1_LAYOUT_COMPRESSED: return any_kernel_lds_compressed(threads);
    default: return any_kernel_lds_pushdown(threads);
  }
}

uint32_t tile_rows(q1_layout l) {
  return l == Q1_LAYOUT_REFERENCE      ? kHostTileRows<Q1_LAYOUT_REFERENCE>
         : l == Q1_LAYOUT_UNCOMPRESSED ? kHostTileRows<Q1_LAYOUT_UNCOMPRESSED>
                                       : kHostTileRows<Q1_LAYOUT_COMPRESSED>;
}

q1_status hip_status(hipError_t e) { return e == hipSuccess ? Q1_OK : Q1_EDEVICE; }

}  // namespace

// ------------------------------------------------------------------------------------
// Host-side launch helpers
// ------------------------------------------------------------------------------------
bool domain_is_tpch(q1_layout layout, const Domain& d) {
  const int64_t max_qty =
      (layout == Q1_LAYOUT_COMPRESSED || layout == Q1_LAYOUT_COMPRESSED_PUSHDOWN) ? 63 : 6300;
  return d.min_disc >= 0 && d.max_disc <= 15 && d.min_tax >= 0 && d.max_tax <= 15 && d.min_qty >= 0 &&
         d.max_qty <= max_qty && d.min_price >= 0 && d.max_price < (1ll << 24);
}

q1_status make_shape(q1_placement placement, q1_layout layout, bool fast, const q1_launch* launch,
                     uint64_t row_begin, uint64_t row_end, LaunchShape* shape, const char** why) {
  const uint32_t trows = tile_rows(layout);
  uint32_t threads = launch && launch->threads_per_block ? launch->threads_per_block : 256;
  uint32_t tpt = launch && launch->tuples_per_thread ? launch->tuples_per_thread : 1024;
  if (threads != 64 && threads != 128 && threads != 256) {
    *why = "threads_per_block must be 64, 128 or 256";
    return Q1_EINVAL;
  }
  if (tpt % 16 != 0 || tpt == 0 || tpt > 16384) {
    *why = "tuples_per_thread must be a multiple of 16 in [16, 16384]";
    return Q1_EINVAL;
  }
  if ((int)placement < 0 || placement > Q1_PLACE_GLOBAL) {
    *why = "unknown placement";
    return Q1_EINVAL;
  }
  uint32_t tiles_per_thread = tpt / trows;
  const uint64_t first = align_rows_down(row_begin) / trows, end = (row_end + trows - 1) / trows;
  const uint64_t tiles = end > first ? end - first : 0;
  uint64_t per_block = (uint64_t)threads * tiles_per_thread;
  uint64_t blocks = (tiles + per_block - 1) / per_block;
  if (launch && launch->num_blocks) {
    // A caller-chosen grid must still cover the range with the chosen tuples per thread.
    if ((uint64_t)launch->num_blocks < blocks) {
      *why = "num_blocks too small to cover the rows with tuples_per_thread";
      return Q1_EINVAL;
    }
    blocks = launch->num_blocks;
  }
  if (!fast && tpt > any_value_lane_rows(layout)) {
    tiles_per_thread = any_value_lane_rows(layout) / trows;
    per_block = (uint64_t)threads * tiles_per_thread;
    const uint64_t needed = (tiles + per_block - 1) / per_block;
    blocks = needed > blocks ? needed : blocks;
  }
  // HIP's grid size counts work-items in 32 bits.
  if (blocks * threads > 0xFFFFFFFFull) {
    *why = "grid too large (blocks x threads_per_block must stay below 2^32)";
    return Q1_EINVAL;
  }
  shape->blocks = (uint32_t)blocks;
  shape->threads = threads;
  shape->tiles_per_thread = tiles_per_thread;
  return Q1_OK;
}

uint64_t scan_workspace_bytes(q1_placement placement, bool fast, const LaunchShape& shape) {
  return fast && placement == Q1_PLACE_GLOBAL ? (uint64_t)shape.blocks * AccGlobal::W * kNumGroups * 8 : 0;
}

// The kernel variant of a fast launch, and its LDS.  The packed slot holds quantities in whole
// units: the compressed layouts only.
static int fast_variant(q1_placement placement, q1_layout layout, const LaunchShape& shape) {
  const bool units = layout == Q1_LAYOUT_COMPRESSED || layout == Q1_LAYOUT_COMPRESSED_PUSHDOWN;
  if (placement != Q1_PLACE_PER_THREAD_SHARED_MEM || (uint64_t)shape.tiles_per_thread * tile_rows(layout) > 256)
    return (int)placement;
  return units ? kPlaceSharedPacked : kPlaceSharedNarrow;
}

static uint32_t fast_lds(int variant, const LaunchShape& shape) {
  const bool shared = variant == kPlaceSharedNarrow || variant == (int)Q1_PLACE_PER_THREAD_SHARED_MEM;
  const uint32_t table = variant == kPlaceSharedPacked ? packed_table_bytes(shape.threads)
                         : shared                     ? shared_table_bytes(shape.threads)
                                                      : stage_bytes(shape.threads);
  return table + shape.threads / 64 * kNumGroups * NF * 8;
}

bool can_launch_direct(q1_placement placement, q1_layout layout, bool fast, const LaunchShape& shape) {
  return fast && shape.blocks >= 1 && shape.blocks <= kDirectBlocks &&
         fast_variant(placement, layout, shape) != (int)placement;
}

q1_status launch_direct(q1_layout layout, const ScanArgs& a, const LaunchShape& shape, void* stream) {
  const int variant = fast_variant(Q1_PLACE_PER_THREAD_SHARED_MEM, layout, shape);
  uint32_t tiles = shape.tiles_per_thread;
  void* params[] = {(void*)&a, (void*)&tiles};
  return hip_status(hipLaunchKernel((const void*)direct_kernel(layout, shape.threads), dim3(shape.blocks),
                                    dim3(shape.threads), params, fast_lds(variant, shape), (hipStream_t)stream));
}

q1_status launch_scan(q1_placement placement, q1_layout layout, bool fast, const ScanArgs& args,
                      const LaunchShape& shape, void* workspace, void* stream, MergeSet* set) {
  if (args.host && !set) return Q1_EINVAL;
  if (shape.blocks == 0) return Q1_OK;
  const hipStream_t s = (hipStream_t)stream;
  ScanArgs a = args;
  a.set = set && (a.host || shape.blocks >= kSpreadMinBlocks) ? set : nullptr;
  a.table_mask = merge_tables(shape.blocks) - 1;
  if (fast) {
    const int variant = fast_variant(placement, layout, shape);
    uint32_t tiles = shape.tiles_per_thread;
    void* params[] = {(void*)&a, (void*)&tiles, (void*)&workspace};
    return hip_status(hipLaunchKernel((const void*)fast_kernel(layout, variant, shape.threads), dim3(shape.blocks),
                                      dim3(shape.threads), params, fast_lds(variant, shape), s));
  }
  uint32_t tiles = shape.tiles_per_thread;
  void* params[] = {(void*)&a, (void*)&tiles};
  return hip_status(hipLaunchKernel((const void*)any_kernel(layout, shape.threads), dim3(shape.blocks),
                                    dim3(shape.threads), params, any_kernel_lds(layout, shape.threads), s));
}

q1_status launch_fetch(const FetchArgs& f, void* stream) {
  const uint64_t pieces = fetch_pieces(f);
  const uint32_t blocks = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(pieces, kFetchBlocks));
  hipLaunchKernelGGL(fetch_columns, dim3(blocks), dim3(256), 0, (hipStream_t)stream, f, pieces);
  return hip_status(hipGetLastError());
}

q1_status launch_zero(void* p, uint64_t bytes, void* stream) {
  const uint64_t n = bytes / 8;
  if (n == 0) return Q1_OK;
  hipLaunchKernelGGL(zero_words, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     (uint64_t*)p, n);
  return hip_status(hipGetLastError());
}

q1_status launch_generate(q1_layout layout, uint64_t seed, uint64_t rows, const q1_columns& cols,
                          void* stream) {
  if (rows == 0) return Q1_OK;
  const uint64_t groups = (rows + 31) / 32;
  const dim3 grid((uint32_t)((groups + 255) / 256)), block(256);
  const hipStream_t s = (hipStream_t)stream;
  switch (layout) {
    case Q1_LAYOUT_REFERENCE: hipLaunchKernelGGL(generate_rows<Q1_LAYOUT_REFERENCE>, grid, block, 0, s, seed, rows, cols); break;
    case Q1_LAYOUT_UNCOMPRESSED: hipLaunchKernelGGL(generate_rows<Q1_LAYOUT_UNCOMPRESSED>, grid, block, 0, s, seed, rows, cols); break;
    default: hipLaunchKernelGGL(generate_rows<Q1_LAYOUT_COMPRESSED>, grid, block, 0, s, seed, rows, cols); break;
  }
  return hip_status(hipGetLastError());
}

q1_status launch_domain_check(q1_layout layout, const q1_columns& cols, uint64_t rows, const Completion& done,
                              void* stream, bool* counted) {
  if (rows == 0) return Q1_EINVAL;
  const uint64_t per = layout == Q1_LAYOUT_REFERENCE      ? kDomainRows<Q1_LAYOUT_REFERENCE>
                       : layout == Q1_LAYOUT_UNCOMPRESSED ? kDomainRows<Q1_LAYOUT_UNCOMPRESSED>
                                                          : kDomainRows<Q1_LAYOUT_COMPRESSED>;
  const uint64_t blocks = (rows + per - 1) / per;
  if (blocks * 256 > 0xFFFFFFFFull) return Q1_EINVAL;  // HIP counts work-items in 32 bits
  const dim3 grid((uint32_t)blocks), block(256);
  const hipStream_t s = (hipStream_t)stream;
  *counted = blocks <= kDomainCountedBlocks;
  auto run = [&](auto layout_const) {
    constexpr int L = decltype(layout_const)::value;
    if (*counted)
      hipLaunchKernelGGL((domain_check<L, true>), grid, block, 0, s, cols, rows, done);
    else
      hipLaunchKernelGGL((domain_check<L, false>), grid, block, 0, s, cols, rows, done);
  };
  switch (layout) {
    case Q1_LAYOUT_REFERENCE: run(std::integral_constant<int, Q1_LAYOUT_REFERENCE>()); break;
    case Q1_LAYOUT_UNCOMPRESSED: run(std::integral_constant<int, Q1_LAYOUT_UNCOMPRESSED>()); break;
    default: run(std::integral_constant<int, Q1_LAYOUT_COMPRESSED>()); break;
  }
  return hip_status(hipGetLastError());
}

// The end of the kernel before it on the stream, for a host that watches.  A kernel of its own:
// were build_filter's blocks counted, the query could start before its writes have left the
// caches (248 us of a query that takes 234).  A domain check writes nothing and counts its
// blocks (1M rows 9.6 us; with this kernel 10.7).
__global__ void __launch_bounds__(64) report_end(HostResult* host, uint64_t sequence) {
  if (threadIdx.x != 0) return;
  store_host(&host->clock_end, wall_clock64());
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  store_host(&host->sequence, sequence);
}

q1_status launch_build_filter(const uint16_t* ship, uint64_t rows, int32_t cutoff_day, uint32_t* filter,
                              HostResult* host, uint64_t sequence, void* stream) {
  if (rows == 0) return Q1_OK;
  const int64_t c = (int64_t)cutoff_day - kShipDateFrameOfReference;
  const int32_t cut = c < -1 ? -1 : (c > 65535 ? 65535 : (int32_t)c);
  const uint64_t groups = (rows + 7) / 8;   // 8 rows per lane and group
  const uint64_t per_block = 256ull * kFilterGroups;
  hipLaunchKernelGGL(build_filter, dim3((uint32_t)((groups + per_block - 1) / per_block)), dim3(256), 0,
                     (hipStream_t)stream, ship, rows, cut, filter, &host->clock_begin);
  hipLaunchKernelGGL(report_end, dim3(1), dim3(64), 0, (hipStream_t)stream, host, sequence);
  return hip_status(hipGetLastError());
}

uint32_t layout_tile_rows(q1_layout layout) { return tile_rows(layout); }

static void* batch_kernel(q1_layout layout, q1_placement p) {
  switch (layout) {
    case Q1_LAYOUT_REFERENCE: return batch_kernel_reference(p);
    case Q1_LAYOUT_UNCOMPRESSED: return batch_kernel_uncompressed(p);
    case Q1_LAYOUT_COMPRESSED: return batch_kernel_compressed(p);
    default: return batch_kernel_pushdown(p);
  }
}

static uint32_t batch_lds(q1_layout layout, q1_placement p) {
  const bool units = layout == Q1_LAYOUT_COMPRESSED || layout == Q1_LAYOUT_COMPRESSED_PUSHDOWN;
  uint32_t lds = p != Q1_PLACE_PER_THREAD_SHARED_MEM ? stage_bytes(kBatchBlock)
                 : units                            ? packed_table_bytes(kBatchBlock)
                                                    : shared_table_bytes(kBatchBlock);
  return lds + kBatchBlock / 64 * kNumGroups * NF * 8;
}

q1_placement batch_placement(q1_placement p) {
  return p == Q1_PLACE_PER_THREAD_SHARED_MEM ? p : Q1_PLACE_IN_REGISTERS;
}

uint32_t batch_max_lane_rows(q1_placement p) { return batch_placement(p) == Q1_PLACE_PER_THREAD_SHARED_MEM ? 256 : 16384; }

uint32_t batch_blocks_per_cu(q1_layout layout, q1_placement p) {
  p = batch_placement(p);
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)batch_kernel(layout, p), kBatchBlock,
                                                   batch_lds(layout, p)) != hipSuccess ||
      per_cu < 1)
    per_cu = 1;
  return (uint32_t)per_cu;
}

q1_status launch_batch(q1_layout layout, q1_placement placement, const BatchHeader* buf, uint32_t n,
                       BatchControl* control, q1_device_aggregates* results, BatchDone* done, uint32_t blocks,
                       void* stream) {
  placement = batch_placement(placement);
  if (blocks == 0) return Q1_EINVAL;
  const BatchDesc* descs = reinterpret_cast<const BatchDesc*>(buf + 1);
  const uint32_t* first = reinterpret_cast<const uint32_t*>(descs + n);
  void* args[] = {(void*)&buf, (void*)&descs, (void*)&first, (void*)&control, (void*)&results, (void*)&done};
  return hip_status(hipLaunchKernel(batch_kernel(layout, placement), dim3(blocks), dim3(kBatchBlock), args,
                                    batch_lds(layout, placement), (hipStream_t)stream));
}

}  // namespace q1

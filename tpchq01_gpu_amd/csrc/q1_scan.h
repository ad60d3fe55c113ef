// gfx950 scan kernels of the TPC-H Q1 scan -> filter -> group-aggregate path: device code
// shared by the translation units that instantiate it, one per column layout
// (q1_scan_<layout>.hip), so the layouts compile in parallel.
//
// Work decomposition (all layouts, all placements):
//   * rows are cut into lane tiles of consecutive rows (4 for the compressed layouts, 2 for
//     the uncompressed and reference ones), four in flight per lane, so that every load
//     instruction of a wavefront reads whole cache lines of its column and the loads can be
//     non-temporal;
//   * a block owns tiles_per_thread * blockDim consecutive tiles; in iteration k thread i
//     takes tile base + k*blockDim + i, so each load instruction of a wavefront covers one
//     contiguous stretch of a column;
//   * only the first and the last tile of a range can be partial: groups of tiles at the
//     range's ends take a guarded path, every other one straight-line loads and rows;
//   * each placement keeps its partial aggregation table in its own memory space
//     (registers, scratch, LDS or global memory); at the end of the block the per-lane
//     partials are reduced across the wavefront, across the
//     block through LDS in 128-bit arithmetic, and merged into the destination table with
//     one set of 64-bit atomics per block (128-bit sums as carry-propagating word pairs).
//
// Arithmetic (cpu/kernel_naive.hpp:14-25): disc_1 = 100 - disc, disc_price = disc_1*price,
// charge = disc_price*(100 + tax), all exact.  Inside the TPC-H value domain (discount and
// tax <= 15, quantity <= 63 units, price < 2^24; measured per table) the "fast" kernels use
// 24-bit multiplies and narrow per-tile accumulators:
//   small    = 1 | disc << 5 | qty << 13       (count, discount, quantity in one dword)
//   dprod    = disc * price                     (then sum_disc_price = 100*sum_price - sum_dprod)
//   charge   = (100-disc)*(100+tax) * price     (v_mul_u32_u24 + v_mul_hi_u32_u24)
// Outside the domain the any-value kernel computes in wrapping int64 with 128-bit
// signed sums, which is the reference CPU kernels' arithmetic for any input.
#pragma once

#include <hip/hip_runtime.h>

#include "q1_common.h"
#include "q1_kernels.h"

namespace q1 {
using FastFn = void (*)(ScanArgs, uint32_t, uint64_t*);
using GenFn = void (*)(ScanArgs, uint32_t);

namespace {

constexpr int kBatchBlock = (int)kBatchThreads;  // the batched kernel's block size

// ------------------------------------------------------------------------------------
// Small helpers
// ------------------------------------------------------------------------------------
// The thread's index in its block (threadIdx.x), hidden from the optimizer by an empty asm.
// Every use reads the index afresh, so values derived from it (lane offsets into the
// columns and the LDS table) are recomputed where they are used instead of being hoisted
// out of the row and entry loops and kept live across them.  That costs a few integer
// operations per tile and saves 8 to 40 vector registers per kernel.  Where that adds a
// wavefront per SIMD it pays only for the batched kernel with in-register sums (179 to 161
// registers, 2 to 3 wavefronts): the 256-request batch takes 1.28 ms instead of 1.67.  The
// scans (compressed LDS table 122 to 106, uncompressed 132 to 112, 3 to 4 wavefronts) and
// the LDS-table batched kernel (148 to 109) measured the same as before, within 0.5 %.
__device__ __forceinline__ uint32_t thread_index() {
  uint32_t t = __builtin_amdgcn_workitem_id_x();
  __asm__ volatile("" : "+v"(t));
  return t;
}
__device__ __forceinline__ uint32_t comp(const uint4& v, int i) {
  return i == 0 ? v.x : (i == 1 ? v.y : (i == 2 ? v.z : v.w));
}
__device__ __forceinline__ void comp_set(uint4& v, int i, uint32_t bits) {
  if (i == 0) v.x = bits; else if (i == 1) v.y = bits; else if (i == 2) v.z = bits; else v.w = bits;
}
__device__ __forceinline__ uint32_t comp(const uint2& v, int i) { return i == 0 ? v.x : v.y; }
__device__ __forceinline__ void comp_set(uint2& v, int i, uint32_t bits) {
  if (i == 0) v.x = bits; else v.y = bits;
}
__device__ __forceinline__ uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }

// Rows of the tile that lie inside [lo, hi): bit j set for row tile*TILE + j.
template <int TILE>
__device__ __forceinline__ uint32_t valid_mask(uint64_t tile, uint64_t lo, uint64_t hi) {
  const uint64_t r0 = tile * TILE;
  uint32_t m = 0;
#pragma unroll
  for (int j = 0; j < TILE; j++) m |= (uint32_t)(r0 + j >= lo && r0 + j < hi) << j;
  return m;
}

// The rows a streaming tile at an end of the range reads: its rows outside [lo, hi) stand for
// the nearest one inside (they never count, whatever they hold), so that all its loads are
// issued together, with no branch per row.  At least one row of the tile is inside.
struct EdgeRows {
  uint64_t lo, hi;
  __device__ __forceinline__ uint64_t row(uint64_t r) const { return r < lo ? lo : r >= hi ? hi - 1 : r; }
};

// One row of the fast path: values already narrowed.  gid is the raw 3-bit slot code
// (6 and 7 only arise from the unused return-flag code 3 and never count).
struct FastRow {
  bool pass;     // inside the row range and ship_date <= cutoff
  uint32_t gid;
  uint32_t qty, disc, tax, price;
  __device__ __forceinline__ bool counts() const { return pass && gid < kNumGroups; }
};

// One row of the any-value path, for layouts whose values are wider than 32 bits.
struct WideRow {
  bool pass;
  uint32_t gid;
  int64_t qty, price, disc, tax;
  __device__ __forceinline__ bool counts() const { return pass && gid < kNumGroups; }
};

// ------------------------------------------------------------------------------------
// Tile loaders, one per layout.  load() reads a whole tile with vector loads; load_edge()
// reads a partial tile row by row into the same vector form, its rows outside the range replaced by
// the nearest one inside (EdgeRows).
// Accessors extract row j (j is a compile-time constant after unrolling).
// ------------------------------------------------------------------------------------

// Non-temporal (streaming) vector loads.  A column is read once, so its lines need not
// stay in the caches; on gfx950 this raises the rate at which HBM feeds a streaming kernel
// (measured: 6.2 -> 7.1 TB/s for these columns) when every load instruction of a
// wavefront covers whole cache lines, as the 4-row tiles below do.
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint4 nt_load(const uint4* p) {
  const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint2 nt_load(const uint2* p) {
  const u32x2_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x2_t*>(p));
  return make_uint2(v.x, v.y);
}
__device__ __forceinline__ uint32_t nt_load(const uint32_t* p) { return __builtin_nontemporal_load(p); }
__device__ __forceinline__ uint32_t nt_load(const uint16_t* p) { return __builtin_nontemporal_load(p); }

// Q1_LAYOUT_COMPRESSED / Q1_LAYOUT_COMPRESSED_PUSHDOWN: 4 rows per tile, so that each load
// instruction of a wavefront reads one contiguous, line-aligned stretch of its column:
// 64 lanes x 8 bytes of ship dates, x 4 bytes of quantity / discount / tax, x 16 bytes of
// prices.  The 4 rows' return flags are one byte of the packed column (2 bits per row)
// and their line statuses / filter bits one nibble (1 bit per row).
template <bool PUSHDOWN>
struct CompressedStreamTile {
  static constexpr int TILE = 4;
  static constexpr int GROUP = 4;  // tiles loaded together per lane
  uint2 sd;         // 4 x uint16 ship dates (unused for pushdown)
  uint32_t q, d, x; // 4 x uint8 quantity, discount, tax
  uint4 p;          // 4 x uint32 extended price
  uint32_t rf;      // 4 x 2-bit return flag codes
  uint32_t ls;      // 4 x 1-bit line status codes
  uint32_t flt;     // 4 x filter bits (pushdown)

  __device__ __forceinline__ static uint32_t nibble(const void* col, uint64_t t) {
    return (reinterpret_cast<const uint8_t*>(col)[t >> 1] >> (4 * (t & 1))) & 0xFu;
  }
  __device__ __forceinline__ void load(const q1_columns& c, uint64_t t) {
    if (!PUSHDOWN)
      sd = nt_load(reinterpret_cast<const uint2*>(c.ship_date) + t);
    else
      flt = nibble(c.filter, t);
    q = nt_load(reinterpret_cast<const uint32_t*>(c.quantity) + t);
    d = nt_load(reinterpret_cast<const uint32_t*>(c.discount) + t);
    x = nt_load(reinterpret_cast<const uint32_t*>(c.tax) + t);
    p = nt_load(reinterpret_cast<const uint4*>(c.extended_price) + t);
    rf = reinterpret_cast<const uint8_t*>(c.return_flag)[t];
    ls = nibble(c.line_status, t);
  }
  __device__ __forceinline__ void load_edge(const q1_columns& c, uint64_t t, const EdgeRows& e) {
    // The packed byte / nibble of a tile holds rows of the tile only, so reading it for a
    // tile that has at least one row in the range stays inside the column.
    rf = reinterpret_cast<const uint8_t*>(c.return_flag)[t];
    ls = nibble(c.line_status, t);
    if (PUSHDOWN) flt = nibble(c.filter, t);
    uint32_t sv[TILE], qv[TILE], dv[TILE], xv[TILE];
#pragma unroll
    for (int j = 0; j < TILE; j++) {
      const uint64_t r = e.row(t * TILE + j);
      sv[j] = PUSHDOWN ? 0 : reinterpret_cast<const uint16_t*>(c.ship_date)[r];
      qv[j] = reinterpret_cast<const uint8_t*>(c.quantity)[r];
      dv[j] = reinterpret_cast<const uint8_t*>(c.discount)[r];
      xv[j] = reinterpret_cast<const uint8_t*>(c.tax)[r];
      comp_set(p, j, reinterpret_cast<const uint32_t*>(c.extended_price)[r]);
    }
    sd = make_uint2(sv[0] | sv[1] << 16, sv[2] | sv[3] << 16);
    q = qv[0] | qv[1] << 8 | qv[2] << 16 | qv[3] << 24;
    d = dv[0] | dv[1] << 8 | dv[2] << 16 | dv[3] << 24;
    x = xv[0] | xv[1] << 8 | xv[2] << 16 | xv[3] << 24;
  }
  // `cut` is the cutoff relative to the frame of reference (may be < 0 or > 65535).
  __device__ __forceinline__ bool pass(int j, int32_t cut) const {
    if (PUSHDOWN) return (flt >> j) & 1;
    const uint32_t s = ((j < 2 ? sd.x : sd.y) >> (16 * (j & 1))) & 0xFFFFu;
    return (int32_t)s <= cut;
  }
  __device__ __forceinline__ uint32_t gid(int j) const {
    return __builtin_amdgcn_ubfe(rf, 2 * j, 2) << 1 | __builtin_amdgcn_ubfe(ls, j, 1);
  }
  __device__ __forceinline__ static uint32_t byte(uint32_t v, int j) { return (v >> (8 * j)) & 0xFFu; }
  // Rows carrying the unused return-flag code 3 (slot 6 or 7): bit 2j set for row j.
  __device__ __forceinline__ uint32_t bad_codes() const { return rf & (rf >> 1) & 0x55u; }
  // Turns those rows into rows that fail the filter (ship date 0xFFFF, above every
  // cutoff below 65535; pushdown: filter bit cleared) with code 0, so every row's slot is
  // below 6.
  __device__ void drop_bad_codes() {
    const uint32_t inv = bad_codes();
    rf &= ~(inv * 3u);
    if (PUSHDOWN) {
      flt &= ~((inv & 1u) | (inv >> 1 & 2u) | (inv >> 2 & 4u) | (inv >> 3 & 8u));
    } else {
      sd.x |= (inv & 1u ? 0xFFFFu : 0u) | (inv & 4u ? 0xFFFF0000u : 0u);
      sd.y |= (inv & 0x10u ? 0xFFFFu : 0u) | (inv & 0x40u ? 0xFFFF0000u : 0u);
    }
  }
  // U tiles a block-stride apart (stride even): their packed line-status / filter nibbles
  // sit stride / 2 bytes apart from one base and at the same half of their byte.
  template <int U>
  __device__ __forceinline__ static void load_group(CompressedStreamTile (&g)[U], const q1_columns& c, uint64_t t0,
                                                    uint64_t stride) {
    const uint8_t* lsb = reinterpret_cast<const uint8_t*>(c.line_status) + (t0 >> 1);
    const uint32_t sh = 4u * (uint32_t)(t0 & 1);
#pragma unroll
    for (int m = 0; m < U; m++) {
      const uint64_t t = t0 + (uint64_t)m * stride;
      if (!PUSHDOWN)
        g[m].sd = nt_load(reinterpret_cast<const uint2*>(c.ship_date) + t);
      else
        g[m].flt = (reinterpret_cast<const uint8_t*>(c.filter)[(t0 >> 1) + (uint64_t)m * (stride >> 1)] >> sh) & 0xFu;
      g[m].q = nt_load(reinterpret_cast<const uint32_t*>(c.quantity) + t);
      g[m].d = nt_load(reinterpret_cast<const uint32_t*>(c.discount) + t);
      g[m].x = nt_load(reinterpret_cast<const uint32_t*>(c.tax) + t);
      g[m].p = nt_load(reinterpret_cast<const uint4*>(c.extended_price) + t);
      g[m].rf = reinterpret_cast<const uint8_t*>(c.return_flag)[t];
      g[m].ls = (lsb[(uint64_t)m * (stride >> 1)] >> sh) & 0xFu;
    }
  }
  template <bool EDGE>
  __device__ __forceinline__ FastRow fast(int j, int32_t cut, uint32_t valid) const {
    FastRow r;
    r.pass = EDGE ? ((valid >> j & 1) && pass(j, cut)) : pass(j, cut);
    r.gid = gid(j);
    r.qty = byte(q, j);
    r.disc = byte(d, j);
    r.tax = byte(x, j);
    r.price = comp(p, j);
    return r;
  }
};

// Q1_LAYOUT_UNCOMPRESSED: int32 ship, int32 qty, int64 price, int8 disc/tax, char rf/ls; 2 rows
// per tile, so that each load instruction of a wavefront reads one contiguous stretch of
// its column with at most 16 bytes per lane: 64 lanes x 8 bytes of ship dates and
// quantities, x 16 bytes of prices, x 2 bytes of discounts, taxes, return flags and line
// statuses.  All loads are non-temporal (each byte is read once).
struct UncompressedStreamTile {
  static constexpr int TILE = 2;
  static constexpr int GROUP = 4;  // tiles loaded together per lane
  uint2 s, q;              // 2 x int32 ship date, quantity (hundredths)
  uint4 p;                 // 2 x int64 price as (lo, hi) pairs
  uint32_t d, x, rf, ls;   // 2 x int8 / char in the low half-word

  __device__ __forceinline__ void load(const q1_columns& c, uint64_t t) {
    s = nt_load(reinterpret_cast<const uint2*>(c.ship_date) + t);
    q = nt_load(reinterpret_cast<const uint2*>(c.quantity) + t);
    p = nt_load(reinterpret_cast<const uint4*>(c.extended_price) + t);
    d = nt_load(reinterpret_cast<const uint16_t*>(c.discount) + t);
    x = nt_load(reinterpret_cast<const uint16_t*>(c.tax) + t);
    rf = nt_load(reinterpret_cast<const uint16_t*>(c.return_flag) + t);
    ls = nt_load(reinterpret_cast<const uint16_t*>(c.line_status) + t);
  }
  __device__ __forceinline__ void load_edge(const q1_columns& c, uint64_t t, const EdgeRows& e) {
    uint32_t dv[TILE], xv[TILE], rv[TILE], lv[TILE];
#pragma unroll
    for (int j = 0; j < TILE; j++) {
      const uint64_t r = e.row(t * TILE + j);
      comp_set(s, j, (uint32_t)reinterpret_cast<const int32_t*>(c.ship_date)[r]);
      comp_set(q, j, (uint32_t)reinterpret_cast<const int32_t*>(c.quantity)[r]);
      const uint64_t pv = (uint64_t)reinterpret_cast<const int64_t*>(c.extended_price)[r];
      comp_set(p, 2 * j, (uint32_t)pv);
      comp_set(p, 2 * j + 1, (uint32_t)(pv >> 32));
      dv[j] = reinterpret_cast<const uint8_t*>(c.discount)[r];
      xv[j] = reinterpret_cast<const uint8_t*>(c.tax)[r];
      rv[j] = reinterpret_cast<const uint8_t*>(c.return_flag)[r];
      lv[j] = reinterpret_cast<const uint8_t*>(c.line_status)[r];
    }
    d = dv[0] | dv[1] << 8;
    x = xv[0] | xv[1] << 8;
    rf = rv[0] | rv[1] << 8;
    ls = lv[0] | lv[1] << 8;
  }
  __device__ __forceinline__ static uint32_t byte(uint32_t v, int j) { return (v >> (8 * j)) & 0xFFu; }
  __device__ __forceinline__ uint32_t gid(int j) const {
    return encode_return_flag(byte(rf, j)) << 1 | encode_line_status(byte(ls, j));
  }
  __device__ __forceinline__ bool pass(int j, int32_t cut) const { return (int32_t)comp(s, j) <= cut; }
  // Character flags encode to slots 0..5 only.
  __device__ __forceinline__ static constexpr uint32_t bad_codes() { return 0; }
  __device__ __forceinline__ void drop_bad_codes() {}
  template <int U>
  __device__ __forceinline__ static void load_group(UncompressedStreamTile (&g)[U], const q1_columns& c, uint64_t t0,
                                                    uint64_t stride) {
#pragma unroll
    for (int m = 0; m < U; m++) g[m].load(c, t0 + (uint64_t)m * stride);
  }
  template <bool EDGE>
  __device__ __forceinline__ FastRow fast(int j, int32_t cut, uint32_t valid) const {
    FastRow r;
    r.pass = EDGE ? ((valid >> j & 1) && pass(j, cut)) : pass(j, cut);
    r.gid = gid(j);
    r.qty = comp(q, j);
    r.disc = byte(d, j);
    r.tax = byte(x, j);
    r.price = comp(p, 2 * j);
    return r;
  }
  template <bool EDGE>
  __device__ __forceinline__ WideRow wide(int j, int32_t cut, uint32_t valid) const {
    WideRow r;
    r.pass = EDGE ? ((valid >> j & 1) && pass(j, cut)) : pass(j, cut);
    r.gid = gid(j);
    r.qty = (int32_t)comp(q, j);
    r.disc = (int8_t)byte(d, j);
    r.tax = (int8_t)byte(x, j);
    r.price = (int64_t)((uint64_t)comp(p, 2 * j + 1) << 32 | comp(p, 2 * j));
    return r;
  }
};

// Q1_LAYOUT_REFERENCE: int32 ship, int64 qty/price/disc/tax, char rf/ls; 2 rows per
// tile, each load instruction of a wavefront one contiguous stretch of its column with at
// most 16 bytes per lane (64 lanes x 8 bytes of ship dates, x 16 bytes of each int64
// column, x 2 bytes of return flags and line statuses), all loads non-temporal.
struct ReferenceStreamTile {
  static constexpr int TILE = 2;
  static constexpr int GROUP = 4;  // tiles loaded together per lane
  uint2 s;                 // 2 x int32 ship date
  uint4 q, p, d, x;        // 2 x int64 as (lo, hi) pairs
  uint32_t rf, ls;         // 2 x char in the low half-word

  __device__ __forceinline__ void load(const q1_columns& c, uint64_t t) {
    s = nt_load(reinterpret_cast<const uint2*>(c.ship_date) + t);
    q = nt_load(reinterpret_cast<const uint4*>(c.quantity) + t);
    p = nt_load(reinterpret_cast<const uint4*>(c.extended_price) + t);
    d = nt_load(reinterpret_cast<const uint4*>(c.discount) + t);
    x = nt_load(reinterpret_cast<const uint4*>(c.tax) + t);
    rf = nt_load(reinterpret_cast<const uint16_t*>(c.return_flag) + t);
    ls = nt_load(reinterpret_cast<const uint16_t*>(c.line_status) + t);
  }
  __device__ __forceinline__ static void put64(uint4& v, int j, uint64_t val) {
    comp_set(v, 2 * j, (uint32_t)val);
    comp_set(v, 2 * j + 1, (uint32_t)(val >> 32));
  }
  __device__ __forceinline__ void load_edge(const q1_columns& c, uint64_t t, const EdgeRows& e) {
    uint32_t rv[TILE], lv[TILE];
#pragma unroll
    for (int j = 0; j < TILE; j++) {
      const uint64_t r = e.row(t * TILE + j);
      comp_set(s, j, (uint32_t)reinterpret_cast<const int32_t*>(c.ship_date)[r]);
      put64(q, j, (uint64_t)reinterpret_cast<const int64_t*>(c.quantity)[r]);
      put64(p, j, (uint64_t)reinterpret_cast<const int64_t*>(c.extended_price)[r]);
      put64(d, j, (uint64_t)reinterpret_cast<const int64_t*>(c.discount)[r]);
      put64(x, j, (uint64_t)reinterpret_cast<const int64_t*>(c.tax)[r]);
      rv[j] = reinterpret_cast<const uint8_t*>(c.return_flag)[r];
      lv[j] = reinterpret_cast<const uint8_t*>(c.line_status)[r];
    }
    rf = rv[0] | rv[1] << 8;
    ls = lv[0] | lv[1] << 8;
  }
  __device__ __forceinline__ static uint32_t lo32(const uint4& v, int j) { return comp(v, 2 * j); }
  __device__ __forceinline__ static int64_t get64(const uint4& v, int j) {
    return (int64_t)((uint64_t)comp(v, 2 * j + 1) << 32 | comp(v, 2 * j));
  }
  __device__ __forceinline__ uint32_t gid(int j) const {
    return encode_return_flag((rf >> (8 * j)) & 0xFFu) << 1 | encode_line_status((ls >> (8 * j)) & 0xFFu);
  }
  __device__ __forceinline__ bool pass(int j, int32_t cut) const { return (int32_t)comp(s, j) <= cut; }
  // Character flags encode to slots 0..5 only.
  __device__ __forceinline__ static constexpr uint32_t bad_codes() { return 0; }
  __device__ __forceinline__ void drop_bad_codes() {}
  template <int U>
  __device__ __forceinline__ static void load_group(ReferenceStreamTile (&g)[U], const q1_columns& c, uint64_t t0,
                                                    uint64_t stride) {
#pragma unroll
    for (int m = 0; m < U; m++) g[m].load(c, t0 + (uint64_t)m * stride);
  }
  template <bool EDGE>
  __device__ __forceinline__ FastRow fast(int j, int32_t cut, uint32_t valid) const {
    FastRow r;
    r.pass = EDGE ? ((valid >> j & 1) && pass(j, cut)) : pass(j, cut);
    r.gid = gid(j);
    r.qty = lo32(q, j);
    r.disc = lo32(d, j);
    r.tax = lo32(x, j);
    r.price = lo32(p, j);
    return r;
  }
  template <bool EDGE>
  __device__ __forceinline__ WideRow wide(int j, int32_t cut, uint32_t valid) const {
    WideRow r;
    r.pass = EDGE ? ((valid >> j & 1) && pass(j, cut)) : pass(j, cut);
    r.gid = gid(j);
    r.qty = get64(q, j);
    r.disc = get64(d, j);
    r.tax = get64(x, j);
    r.price = get64(p, j);
    return r;
  }
};

// Every placement reads these tiles.  The register placements read tiles of 16, 8 and 4 rows
// with ordinary loads before, half a stretch per load instruction: 600M compressed rows per
// thread / in registers / global 982 / 990 / 1007 us (now 873 / 929 / 930), 60M uncompressed
// 210 / 208 / 210 (188 / 189 / 190), 60M reference 382 / 378 / 386 (345 / 344 / 346).
template <int L> struct TileOf;
template <> struct TileOf<Q1_LAYOUT_REFERENCE> { using T = ReferenceStreamTile; };
template <> struct TileOf<Q1_LAYOUT_UNCOMPRESSED> { using T = UncompressedStreamTile; };
template <> struct TileOf<Q1_LAYOUT_COMPRESSED> { using T = CompressedStreamTile<false>; };
template <> struct TileOf<Q1_LAYOUT_COMPRESSED_PUSHDOWN> { using T = CompressedStreamTile<true>; };

// A group of U lane tiles t0 + m * stride (m < U, at most `count` of them, below
// `end_tile`), all loaded before any of their rows is used, so that a wavefront keeps 16 rows'
// (4-row tiles) or 8 rows' (2-row tiles) worth of loads per lane in flight.
template <class Tile, int U>
struct TileGroup {
  Tile tile[U];
  uint32_t valid[U];  // rows of the tile inside [row_begin, row_end)
  bool use[U], edge[U];
  // Straight-line loads of all U tiles, for a group the caller knows to be whole and inside
  // the range for every lane.
  __device__ __forceinline__ void load_plain(const q1_columns& c, uint64_t t0, uint64_t stride) {
    Tile::template load_group<U>(tile, c, t0, stride);
  }
  // The whole tiles are loaded first, then the partial ones (at most one at each end of the
  // range).  A partial tile read row by row, each under its own branch, and inside the tile
  // loop, made every range with a ragged end wait four more times for memory (kernel of 5,003
  // rows 8.5 us, now 6.9, of whole blocks 6.7) and kept 26 (compressed) to 78 (reference)
  // more vector registers.
  __device__ __forceinline__ void load(const q1_columns& c, uint64_t t0, uint64_t stride, uint32_t count,
                                       uint64_t end_tile, uint64_t row_begin, uint64_t row_end) {
    constexpr int TILE = Tile::TILE;
#pragma unroll
    for (int m = 0; m < U; m++) {
      const uint64_t t = t0 + (uint64_t)m * stride;
      edge[m] = t * TILE < row_begin || (t + 1) * TILE > row_end;
      valid[m] = edge[m] ? valid_mask<TILE>(t, row_begin, row_end) : (1u << TILE) - 1;
      use[m] = (uint32_t)m < count && t < end_tile && valid[m];
      if (use[m] && !edge[m]) tile[m].load(c, t);
    }
#pragma unroll
    for (int m = 0; m < U; m++) {
      const uint64_t t = t0 + (uint64_t)m * stride;
      if (use[m] && edge[m]) tile[m].load_edge(c, t, EdgeRows{row_begin, row_end});
    }
  }
};

// Cutoff in the units of the layout's ship_date column.
template <int L>
__device__ __forceinline__ int32_t column_cutoff(int32_t cutoff_day) {
  if (L == Q1_LAYOUT_COMPRESSED || L == Q1_LAYOUT_COMPRESSED_PUSHDOWN) {
    const int64_t c = (int64_t)cutoff_day - kShipDateFrameOfReference;
    return c < -1 ? -1 : (c > 65535 ? 65535 : (int32_t)c);
  }
  return cutoff_day;
}

// ------------------------------------------------------------------------------------
// Per-lane partial table handed to the block merge: six base sums per group.
//   F_QTY quantity (layout units), F_PRICE price, F_DISC discount, F_CNT count,
//   F_DPROD sum of disc*price, F_CHARGE charge.  All exact in uint64 per lane.
// ------------------------------------------------------------------------------------
enum { F_QTY, F_PRICE, F_DISC, F_CNT, F_DPROD, F_CHARGE, NF };

// A lane's sums as the register tables hand them over: per group the packed (count |
// discount | quantity) word (pack_small64), price, discount product and charge.
typedef uint64_t LaneWords[kNumGroups][4];
// The LDS rows that their sum over a wavefront goes through (sum_lane_words).
constexpr uint32_t stage_bytes(uint32_t threads) { return 2u * kNumGroups * 8u * threads; }

__device__ __forceinline__ uint32_t pack_small(const FastRow& r) {
  return 1u | r.disc << 5 | r.qty << 13;
}
__device__ __forceinline__ uint32_t disc_prod(const FastRow& r) { return __umul24(r.disc, r.price); }
__device__ __forceinline__ uint64_t fast_charge(const FastRow& r) {
  const uint32_t f = __umul24(100u - r.disc, 100u + r.tax);  // <= 100*115, fits 24 bits
  const uint64_t prod = (uint64_t)(f & 0xFFFFFFu) * (r.price & 0xFFFFFFu);
  return prod;
}

// DPP move of a 64-bit value (two 32-bit lane permutes); CTRL is a gfx9 DPP control.
template <int CTRL>
__device__ __forceinline__ uint64_t dpp_u64(uint64_t v) {
  const uint2 w = __builtin_bit_cast(uint2, v);
  const uint2 r = make_uint2((uint32_t)__builtin_amdgcn_mov_dpp((int)w.x, CTRL, 0xF, 0xF, false),
                             (uint32_t)__builtin_amdgcn_mov_dpp((int)w.y, CTRL, 0xF, 0xF, false));
  return __builtin_bit_cast(uint64_t, r);
}

// Q1_PLACE_IN_REGISTERS: narrow per-tile accumulators in registers; a group's block of
// adds is skipped by the whole wavefront when no lane holds a row of that group.  Price
// and price x discount share one 64-bit word (price in the low half, below 16 * 2^24 =
// 2^28 over a tile; the product in the high half, below 16 * 15 * 2^24 < 2^32), so a row
// costs three adds per group: that word, the packed count|discount|quantity and the charge.
struct AccRegisters {
  static constexpr bool kWideRows = false, kCompactEnds = true;
  uint32_t ns[kNumGroups];
  uint64_t npd[kNumGroups];
  uint64_t ch[kNumGroups], pr[kNumGroups], dp[kNumGroups];
  uint32_t cnt[kNumGroups], dsc[kNumGroups], qty[kNumGroups];

  __device__ __forceinline__ void init(char*) {
#pragma unroll
    for (int g = 0; g < kNumGroups; g++) {
      ns[g] = 0;
      npd[g] = 0;
      ch[g] = pr[g] = dp[g] = 0;
      cnt[g] = dsc[g] = qty[g] = 0;
    }
  }
  __device__ __forceinline__ void add(const FastRow& r) {
    const uint32_t s = pack_small(r);
    const uint64_t pd = (uint64_t)disc_prod(r) << 32 | r.price;
    const uint64_t c = fast_charge(r);
    const uint64_t pass_mask = ballot(r.pass);
#pragma unroll
    for (int g = 0; g < kNumGroups; g++) {
      const bool mine = r.pass && r.gid == (uint32_t)g;
      if (ballot(r.gid == (uint32_t)g) & pass_mask) {
        // The empty asm keeps this a separate, wavefront-uniform branch (it cannot be
        // folded into the lane mask), so a group no lane holds costs no adds at all.
        __asm__ volatile("");
        if (mine) {
          ns[g] += s;
          npd[g] += pd;
          ch[g] += c;
        }
      }
    }
  }
  // Called after at most 16 rows: moves the narrow sums into the wide ones.
  __device__ __forceinline__ void flush(bool = false) {
#pragma unroll
    for (int g = 0; g < kNumGroups; g++) {
      if (ballot(ns[g] != 0)) {
        cnt[g] += ns[g] & 31u;
        dsc[g] += (ns[g] >> 5) & 255u;
        qty[g] += ns[g] >> 13;
        pr[g] += (uint32_t)npd[g];
        dp[g] += npd[g] >> 32;
        ns[g] = 0;
        npd[g] = 0;
      }
    }
  }
  __device__ __forceinline__ void words(LaneWords& w) const {
#pragma unroll
    for (int g = 0; g < kNumGroups; g++) {
      w[g][0] = (uint64_t)cnt[g] | (uint64_t)dsc[g] << 17 | (uint64_t)qty[g] << 37;
      w[g][1] = pr[g];
      w[g][2] = dp[g];
      w[g][3] = ch[g];
    }
  }
  static constexpr uint32_t lds_bytes(uint32_t threads) { return stage_bytes(threads); }
};

// Packed (count | discount | quantity) in 64 bits for the per-lane 64-bit tables:
// count bits [0,17), discount [17,37), quantity [37,64).  Exact while a lane's table
// sees at most 16384 rows (tuples_per_thread is capped there).
__device__ __forceinline__ uint64_t pack_small64(const FastRow& r) {
  return 1ull | (uint64_t)r.disc << 17 | (uint64_t)r.qty << 37;
}
__device__ __forceinline__ void unpack_small64(uint64_t s, uint64_t* out) {
  out[F_CNT] = s & ((1ull << 17) - 1);
  out[F_DISC] = (s >> 17) & ((1ull << 20) - 1);
  out[F_QTY] = s >> 37;
}
// The narrow per-tile word (pack_small: count [0,5), discount [5,13), quantity [13,32),
// at most 16 rows) re-packed in the pack_small64 layout.
__device__ __forceinline__ uint64_t small_to_small64(uint32_t s) {
  return (uint64_t)(s & 31u) | (uint64_t)((s >> 5) & 255u) << 17 | (uint64_t)(s >> 13) << 37;
}

// Q1_PLACE_IN_REGISTERS_PER_THREAD: the per-thread table of the reference
// (src/kernels/ht_in_registers_per_thread.cuh:54-64): full-width 64-bit sums per group in
// the lane's registers, updated by every row.  The reference selects the row's group with
// a compare-select over all six groups and every field; here each group is one
// wavefront-uniform branch taken only when some lane of the wavefront holds a passing row
// of it (real data fills four of the six groups), and its four 64-bit adds run under the
// lanes' mask: count, discount and quantity share one word (pack_small64).
struct AccPerThread {
  static constexpr bool kWideRows = false, kCompactEnds = true;
  uint64_t sm[kNumGroups], pr[kNumGroups], dp[kNumGroups], ch[kNumGroups];
  __device__ __forceinline__ void init(char*) {
#pragma unroll
    for (int g = 0; g < kNumGroups; g++) sm[g] = pr[g] = dp[g] = ch[g] = 0;
  }
  __device__ __forceinline__ void add(const FastRow& r) {
    const uint64_t s = pack_small64(r);
    const uint64_t dprod = disc_prod(r);
    const uint64_t c = fast_charge(r);
    const uint64_t pass_mask = ballot(r.pass);
#pragma unroll
    for (int g = 0; g < kNumGroups; g++) {
      if (ballot(r.gid == (uint32_t)g) & pass_mask) {
        // a real, wavefront-uniform branch (not folded into the lane mask), as in AccRegisters
        __asm__ volatile("");
        if (r.pass && r.gid == (uint32_t)g) {
          sm[g] += s;
          pr[g] += r.price;
          dp[g] += dprod;
          ch[g] += c;
        }
      }
    }
  }
  __device__ __forceinline__ void flush(bool = false) {}
  __device__ __forceinline__ void words(LaneWords& w) const {
#pragma unroll
    for (int g = 0; g < kNumGroups; g++) {
      w[g][0] = sm[g];
      w[g][1] = pr[g];
      w[g][2] = dp[g];
      w[g][3] = ch[g];
    }
  }
  static constexpr uint32_t lds_bytes(uint32_t threads) { return stage_bytes(threads); }
};

// Q1_PLACE_LOCAL_MEM: the per-thread table of the reference
// (src/kernels/ht_in_local_mem.cuh:54-59) lives in the lane's private (scratch) memory:
// [group][count|discount|quantity, price, discount product, charge], 64-bit words.  Rows
// are first summed over kLocalFlushRows rows of the lane in registers, with the
// wavefront-uniform group skip of AccRegisters; those sums then go into the private table:
// the first time as plain stores (the table is never zero-filled), later as one
// read-modify-write of the whole table, and once more after the lane's last row unless
// the last periodic update just happened.  A row costs registers only.  The private tables
// of the resident wavefronts (192 B per lane) outgrow the L2, so their updates reach HBM;
// the update interval sets their cost at 600M compressed rows: every 16 rows 3.2 ms,
// 64 rows 1.46 ms, 256 rows 1.35 ms, 1024 rows 1.19 ms.
constexpr uint32_t kLocalFlushRows = 1024;
struct AccLocal {
  static constexpr bool kWideRows = false, kCompactEnds = true;
  // Per group: narrow sums of at most 16 rows as in AccRegisters (pack_small word; price
  // and discount product in one 64-bit word), folded every 16 rows into 64-bit
  // register sums of at most kLocalFlushRows rows (count, discount and quantity in the
  // pack_small64 layout, exact up to 16384 rows; price; discount product), with the charge
  // summed in 64 bits directly.
  static constexpr uint32_t kTableWords = kNumGroups * 4;
  static constexpr uint32_t kFlushCalls = kLocalFlushRows / 16;
  uint32_t ns[kNumGroups];
  uint64_t npd[kNumGroups];
  uint64_t sm[kNumGroups], pr[kNumGroups], dp[kNumGroups], ch[kNumGroups];
  uint32_t calls;
  // The table (kTableWords words of the caller's private array) is used only through this
  // pointer, which an empty asm hides from the optimizer: the array cannot become
  // registers, so it stays in private memory, and its loads and stores are ordinary ones
  // the compiler may overlap (volatile accesses would each wait for the previous one).
  uint64_t* t;
  __device__ __forceinline__ void init(char* private_table) {
    calls = 0;
    t = reinterpret_cast<uint64_t*>(private_table);
    __asm__ volatile("" : "+v"(t));
#pragma unroll
    for (int g = 0; g < kNumGroups; g++) {
      ns[g] = 0;
      npd[g] = 0;
      sm[g] = pr[g] = dp[g] = ch[g] = 0;
    }
  }
  __device__ __forceinline__ void add(const FastRow& r) {
    const uint32_t s = pack_small(r);
    const uint64_t pd = (uint64_t)disc_prod(r) << 32 | r.price;
    const uint64_t c = fast_charge(r);
    const uint64_t pass_mask = ballot(r.pass);
#pragma unroll
    for (int g = 0; g < kNumGroups; g++) {
      if (ballot(r.gid == (uint32_t)g) & pass_mask) {
        __asm__ volatile("");
        if (r.pass && r.gid == (uint32_t)g) {
          ns[g] += s;
          npd[g] += pd;
          ch[g] += c;
        }
      }
    }
  }
  // Called every 16 rows of a lane (at the same points in every lane; a lane's rows are a
  // whole number of 16-row periods, so the last such call comes right before the final
  // one) and after its last row (last = true).  Every call folds the narrow sums into the
  // register sums; every kLocalFlushRows rows, and at the end unless that just happened,
  // the register sums go into the private table.
  __device__ __forceinline__ void flush(bool last = false) {
    static_assert(kLocalFlushRows <= 16384, "pack_small64 is exact up to 16384 rows");
    if (last) {
      if (calls > 0 && calls % kFlushCalls == 0) return;  // nothing summed since the last update
    } else {
#pragma unroll
      for (int g = 0; g < kNumGroups; g++) {
        if (ballot(ns[g] != 0)) {
          sm[g] += small_to_small64(ns[g]);
          pr[g] += (uint32_t)npd[g];
          dp[g] += npd[g] >> 32;
          ns[g] = 0;
          npd[g] = 0;
        }
      }
      if (++calls % kFlushCalls != 0) return;
    }
    // The table is updated in two halves of three groups: each half's words are loaded
    // before any is added to and stored, with no branch between the loads (groups without
    // rows add zero), so the lane waits for its private memory twice per update while
    // holding only half the table in registers.
    const bool first = calls <= kFlushCalls;
    constexpr int kHalf = kNumGroups / 2;
#pragma unroll
    for (int h = 0; h < kNumGroups; h += kHalf) {
      uint64_t w[kHalf * 4];
#pragma unroll
      for (int i = 0; i < kHalf * 4; i++) w[i] = first ? 0 : t[h * 4 + i];
#pragma unroll
      for (int g = 0; g < kHalf; g++) {
        w[g * 4 + 0] += sm[h + g];
        w[g * 4 + 1] += pr[h + g];
        w[g * 4 + 2] += dp[h + g];
        w[g * 4 + 3] += ch[h + g];
        sm[h + g] = pr[h + g] = dp[h + g] = ch[h + g] = 0;
      }
#pragma unroll
      for (int i = 0; i < kHalf * 4; i++) t[h * 4 + i] = w[i];
    }
  }
  // The private table (after the last flush).
  __device__ __forceinline__ void words(LaneWords& w) const {
#pragma unroll
    for (int g = 0; g < kNumGroups; g++)
#pragma unroll
      for (int j = 0; j < 4; j++) w[g][j] = t[g * 4 + j];
  }
  static constexpr uint32_t lds_bytes(uint32_t threads) { return stage_bytes(threads); }
};

// The LDS tables of the shared placement: [group][word][thread] words of 64 bits, W words per
// group.  A wavefront clears, updates and sums only its own 64 threads' words of every row,
// and LDS operations of a wavefront take effect in order, so none of it needs a barrier.
// Clearing: one 16-byte store covers a wavefront's words of two rows.
template <int B, int W>
__device__ __forceinline__ void clear_wave_table(uint64_t* tab) {
  const uint32_t wave = thread_index() >> 6, lane = thread_index() & 63;
  uint64_t* p = tab + (lane >> 5) * B + wave * 64 + (lane & 31) * 2;
#pragma unroll
  for (int row = 0; row < W * kNumGroups; row += 2) *reinterpret_cast<uint4*>(p + row * B) = make_uint4(0, 0, 0, 0);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Sums a wavefront's part of the table over its threads into red[wave][group][words].  Lane 8g + k
// takes group g and threads k, k + 8, ... (rotated by g, so that the groups' reads fall on
// different banks), then the eight lanes of a group are added with DPP.  All groups go at
// once: about 200 vector instructions per wavefront, where a butterfly over all lanes for
// each word of each group took 1,560 -- half the vector work of a block of 128 rows per
// lane, and 2 us of every short launch.  Kernel time of 5,003 compressed rows 10.5 -> 8.5 us,
// of 1M rows 12.3 -> 10.4, of 6M rows 20.9 -> 18.6; the 256-request batch 1,019 -> 977 us
// per call; 600M rows 847 -> 843 us.
__device__ __forceinline__ void add_eight(uint32_t& v) {
  v += (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
  v += (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
  v += (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, false);  // row_half_mirror
}
__device__ __forceinline__ void add_eight(uint64_t& v) {
  v += dpp_u64<0xB1>(v);
  v += dpp_u64<0x4E>(v);
  v += dpp_u64<0x141>(v);
}
template <int B, int W, class GroupSums>
__device__ __forceinline__ void sum_wave_table(const uint64_t* tab, uint64_t* red) {
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const uint32_t wave = thread_index() >> 6, lane = thread_index() & 63, g = lane >> 3, k = lane & 7;
  GroupSums sums;
  if (g < kNumGroups) {
    const uint64_t* p = tab + g * (W * B) + wave * 64 + k;
#pragma unroll
    for (uint32_t i = 0; i < 8; i++) {
      uint64_t w[W];
#pragma unroll
      for (int j = 0; j < W; j++) w[j] = p[j * B + 8 * ((i + g) & 7)];
      sums.add(w);
    }
  }
  sums.reduce([](auto& v) { add_eight(v); });
  if (g < kNumGroups && k == 0) sums.store(red + (wave * kNumGroups + g) * GroupSums::kWords);
}

// Q1_PLACE_PER_THREAD_SHARED_MEM: each lane owns a table in LDS laid out
// [group][field][thread] (consecutive lanes -> consecutive 8-byte words, so a wavefront's
// update of any mix of groups is bank-conflict free); rows are added with return-less
// LDS atomics, which need no VALU add and no read-back.  With the block size known at
// compile time a row's address is one shift-add and the four fields are immediate offsets.
constexpr uint32_t shared_table_bytes(uint32_t threads) { return 4u * kNumGroups * 8u * threads; }

// NARROW: at most 256 rows per lane, so a lane's price sum stays below 256 * 2^24 = 2^32
// and the price field takes a 32-bit LDS atomic on the low word of its 64-bit slot (no
// register pair to build per row); the slot's high word stays zero.
template <int B, bool NARROW = false>
struct AccShared {
  static constexpr bool kWideRows = false, kCompactEnds = false;
  uint64_t* tab;  // dynamic LDS: 6 * 4 * B words
  __device__ __forceinline__ void init(char* lds) {
    tab = reinterpret_cast<uint64_t*>(lds);
    clear_wave_table<B, 4>(tab);
  }
  __device__ __forceinline__ void add(const FastRow& r) {
    // Nearly every row passes: lay the atomics out inline, with no branch around them.
    if (__builtin_expect(r.counts(), 1)) {
      uint64_t* base = tab + r.gid * (4 * B) + thread_index();
      __hip_atomic_fetch_add(base, pack_small64(r), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (NARROW)
        __hip_atomic_fetch_add(reinterpret_cast<uint32_t*>(base + B), r.price, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
      else
        __hip_atomic_fetch_add(base + B, (uint64_t)r.price, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __hip_atomic_fetch_add(base + 2 * B, (uint64_t)disc_prod(r), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __hip_atomic_fetch_add(base + 3 * B, fast_charge(r), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
  __device__ __forceinline__ void flush(bool = false) {}
  // The wavefront's sums of one group's words (sum_wave_table).  A wavefront's sum of the
  // packed word fits its fields for NARROW tables (count <= 64 * 256, discount < 2^18,
  // quantity <= 64 * 256 * 6300 < 2^27); the others take the fields apart first.
  struct GroupSums {
    static constexpr int kWords = NF;
    uint64_t small = 0, price = 0, dprod = 0, charge = 0;
    uint32_t cnt = 0, disc = 0;
    uint64_t qty = 0;
    __device__ __forceinline__ void add(const uint64_t (&w)[4]) {
      if (NARROW) {
        small += w[0];
      } else {
        cnt += (uint32_t)w[0] & ((1u << 17) - 1);
        disc += (uint32_t)(w[0] >> 17) & ((1u << 20) - 1);
        qty += w[0] >> 37;
      }
      price += w[1];
      dprod += w[2];
      charge += w[3];
    }
    template <class F>
    __device__ __forceinline__ void reduce(F f) {
      if (NARROW) {
        f(small);
      } else {
        f(cnt);
        f(disc);
        f(qty);
      }
      f(price);
      f(dprod);
      f(charge);
    }
    __device__ __forceinline__ void store(uint64_t* r) const {
      if (NARROW) {
        unpack_small64(small, r);
      } else {
        r[F_CNT] = cnt;
        r[F_DISC] = disc;
        r[F_QTY] = qty;
      }
      r[F_PRICE] = price;
      r[F_DPROD] = dprod;
      r[F_CHARGE] = charge;
    }
  };
  __device__ __forceinline__ void wave_totals(uint64_t* red) const { sum_wave_table<B, 4, GroupSums>(tab, red); }
  static constexpr uint32_t lds_bytes(uint32_t) { return shared_table_bytes(B); }
};

// Variant of the LDS table for compressed-layout launches of at most 256 rows per lane
// (quantities in whole units, at most 63): three slots per group instead of four.
//   slot 0: price sum (< 256 * 2^24 = 2^32) in bits [0,32), discount sum (<= 256 * 15
//           < 2^12) in [32,44), quantity sum (<= 256 * 63 < 2^14) in [44,58);
//   slot 1: discount-price product sum (< 256 * 15 * 2^24 < 2^36) in [0,36), count
//           (<= 256) in [48,57);
//   slot 2: charge.
// Three return-less 64-bit LDS atomics per passing row instead of four, and a table of
// 6 * 3 * 8 bytes per lane, so four 256-thread blocks fit a compute unit's LDS.
constexpr uint32_t packed_table_bytes(uint32_t threads) { return 3u * kNumGroups * 8u * threads; }

template <int B>
struct AccSharedPacked {
  static constexpr bool kWideRows = false, kCompactEnds = false;
  uint64_t* tab;  // dynamic LDS: 6 * 3 * B words
  __device__ __forceinline__ void init(char* lds) {
    tab = reinterpret_cast<uint64_t*>(lds);
    clear_wave_table<B, 3>(tab);
  }
  __device__ __forceinline__ void add(const FastRow& r) {
    // Nearly every row passes: lay the atomics out inline, with no branch around them.
    if (__builtin_expect(r.counts(), 1)) {
      uint64_t* base = tab + r.gid * (3 * B) + thread_index();
      const uint64_t w0 = (uint64_t)r.price | (uint64_t)(r.disc | r.qty << 12) << 32;
      const uint64_t w1 = (uint64_t)disc_prod(r) | 1ull << 48;
      __hip_atomic_fetch_add(base, w0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __hip_atomic_fetch_add(base + B, w1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __hip_atomic_fetch_add(base + 2 * B, fast_charge(r), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
  __device__ __forceinline__ void flush(bool = false) {}
  // The wavefront's sums of one group's words (sum_wave_table): slot 0 is taken apart, slot
  // 1's fields hold a wavefront's sums (product < 2^42, count <= 64 * 256).
  struct GroupSums {
    static constexpr int kWords = NF;
    uint64_t price = 0, dprod_cnt = 0, charge = 0;
    uint32_t disc = 0, qty = 0;
    __device__ __forceinline__ void add(const uint64_t (&w)[3]) {
      price += (uint32_t)w[0];
      disc += (uint32_t)(w[0] >> 32) & 0xFFFu;
      qty += (uint32_t)(w[0] >> 44);
      dprod_cnt += w[1];
      charge += w[2];
    }
    template <class F>
    __device__ __forceinline__ void reduce(F f) {
      f(price);
      f(disc);
      f(qty);
      f(dprod_cnt);
      f(charge);
    }
    __device__ __forceinline__ void store(uint64_t* r) const {
      r[F_PRICE] = price;
      r[F_DISC] = disc;
      r[F_QTY] = qty;
      r[F_DPROD] = dprod_cnt & ((1ull << 48) - 1);
      r[F_CNT] = dprod_cnt >> 48;
      r[F_CHARGE] = charge;
    }
  };
  __device__ __forceinline__ void wave_totals(uint64_t* red) const { sum_wave_table<B, 3, GroupSums>(tab, red); }
  static constexpr uint32_t lds_bytes(uint32_t) { return packed_table_bytes(B); }
};

// The register tables' sums over a wavefront, through LDS like the LDS tables' own: two of a
// lane's four words per group at a time are staged in rows of 64 lanes (6 KB per wavefront,
// so that registers, not LDS, go on limiting the wavefronts of a compute unit), and eight
// lanes per group add them.  A butterfly over all lanes for each word of each
// group took 3 us more of every launch: 1M compressed rows per thread 15.2 us, now 12.0; 6M
// uncompressed rows 31.9, now 28.8.
__device__ __forceinline__ void sum_lane_words(const LaneWords& w, uint64_t* stage, uint64_t* red) {
  const uint32_t wave = thread_index() >> 6, lane = thread_index() & 63, g = lane >> 3, k = lane & 7;
  uint64_t* mine = stage + wave * (2 * kNumGroups * 64);
  typename AccShared<64>::GroupSums sums;
  uint64_t v[8][4];
#pragma unroll
  for (int half = 0; half < 4; half += 2) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < kNumGroups; i++) {
      mine[(2 * i) * 64 + lane] = w[i][half];
      mine[(2 * i + 1) * 64 + lane] = w[i][half + 1];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const uint32_t row = g < kNumGroups ? g : 0;
#pragma unroll
    for (uint32_t i = 0; i < 8; i++) {
      const uint32_t at = 2 * row * 64 + k + 8 * ((i + g) & 7);
      v[i][half] = mine[at];
      v[i][half + 1] = mine[at + 64];
    }
  }
#pragma unroll
  for (int i = 0; i < 8; i++) sums.add(v[i]);
  sums.reduce([](auto& x) { add_eight(x); });
  if (g < kNumGroups && k == 0) sums.store(red + (wave * kNumGroups + g) * NF);
}

// Q1_PLACE_GLOBAL: the block's aggregation table lives in global memory (the kernel's
// workspace, one table per block), as the reference's table does
// (src/kernels/ht_in_global_mem.hpp:12-52).  The reference adds every row into it with
// five device atomics; here rows are summed in the lanes' registers (AccRegisters), each
// wavefront reduces its lanes' sums with DPP and adds them into the block's table with
// one atomic per (group, field) from one lane, and the block then merges its table into
// the destination once: thread g reads group g's words and issues its destination atomics.
// The table sees up to blockDim * 16384 <= 2^22 rows: count and discount share one word
// (count bits [0,24), discount [24,64)), the other sums have a word each; every block sum
// fits 64 bits (price < 2^46, discount product < 2^50, charge < 2^60).
__device__ __forceinline__ void atomic_add128(uint64_t* lo_p, uint64_t* hi_p, uint64_t lo, uint64_t hi);
struct AccGlobal {
  static constexpr bool kWideRows = false, kCompactEnds = true;
  static constexpr int W = 5;  // words per group: count|disc, qty, price, dprod, charge
  AccRegisters regs;
  uint64_t* tab;               // [W][6] words of this block
  __device__ __forceinline__ void init_global(uint64_t* ws) {
    tab = ws + (uint64_t)blockIdx.x * (W * kNumGroups);
    if (thread_index() < W * kNumGroups)
      __hip_atomic_store(tab + thread_index(), 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
  }
  __device__ __forceinline__ void init(char* lds) { regs.init(lds); }
  __device__ __forceinline__ void add(const FastRow& r) { regs.add(r); }
  __device__ __forceinline__ void flush(bool = false) { regs.flush(); }
  // The block's whole merge (called by every thread of the block; `stage` is its LDS).
  __device__ __forceinline__ void merge(uint64_t* stage, uint64_t* red, q1_device_aggregates* out,
                                        uint64_t qty_scale) const {
    LaneWords o;
    regs.words(o);
    sum_lane_words(o, stage, red);
    const uint32_t wave = thread_index() >> 6, lane = thread_index() & 63;
    // lane 5g + w adds word w of group g into the block's table (a wavefront's count is below
    // 2^21 and its discount sum below 2^24)
    if (lane < W * kNumGroups) {
      const uint32_t g = lane / W, w = lane % W;
      const uint64_t* r = red + (wave * kNumGroups + g) * NF;
      const uint64_t v = w == 0   ? r[F_CNT] | r[F_DISC] << 24
                         : w == 1 ? r[F_QTY]
                         : w == 2 ? r[F_PRICE]
                         : w == 3 ? r[F_DPROD]
                                  : r[F_CHARGE];
      if (v) atomicAdd((unsigned long long*)(tab + w * kNumGroups + g), (unsigned long long)v);
    }
    // Only this block reads its table back, and every wave of the block shares one L2 (where
    // the atomics are performed): the barrier's workgroup-scope release and acquire order
    // them before the read-back.  A device-scope fence here would make each block wait for
    // an L2 write-back towards the other XCDs.
    __syncthreads();
    if (thread_index() < kNumGroups) {
      const int g = thread_index();
      auto ld = [&](int w) {
        return __hip_atomic_load(tab + w * kNumGroups + g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      };
      const uint64_t cd = ld(0), q = ld(1), p = ld(2), d = ld(3), c = ld(4);
      if (cd) {
        atomicAdd((unsigned long long*)&out->sum_qty[g], (unsigned long long)(q * qty_scale));
        atomicAdd((unsigned long long*)&out->sum_base_price[g], (unsigned long long)p);
        atomicAdd((unsigned long long*)&out->sum_disc[g], (unsigned long long)(cd >> 24));
        atomicAdd((unsigned long long*)&out->count[g], (unsigned long long)(cd & ((1ull << 24) - 1)));
        // sum_disc_price = 100 * sum_price - sum(disc * price) >= 0 (every disc <= 15)
        atomic_add128(&out->sum_disc_price_lo[g], &out->sum_disc_price_hi[g], 100 * p - d, 0);
        atomic_add128(&out->sum_charge_lo[g], &out->sum_charge_hi[g], c, 0);
      }
    }
  }
  static constexpr uint32_t lds_bytes(uint32_t threads) { return stage_bytes(threads); }
};

template <int P, int B> struct AccOf;
template <int B> struct AccOf<Q1_PLACE_IN_REGISTERS, B> { using A = AccRegisters; };
template <int B> struct AccOf<Q1_PLACE_IN_REGISTERS_PER_THREAD, B> { using A = AccPerThread; };
template <int B> struct AccOf<Q1_PLACE_LOCAL_MEM, B> { using A = AccLocal; };
template <int B> struct AccOf<Q1_PLACE_PER_THREAD_SHARED_MEM, B> { using A = AccShared<B>; };
template <int B> struct AccOf<Q1_PLACE_GLOBAL, B> { using A = AccGlobal; };
// Internal kernel variant of the shared placement for launches of at most 256 rows per lane.
constexpr int kPlaceSharedNarrow = 8;
template <int B> struct AccOf<kPlaceSharedNarrow, B> { using A = AccShared<B, true>; };
// ... and, for the compressed layouts, the packed table with three slots per group.
constexpr int kPlaceSharedPacked = 9;
template <int B> struct AccOf<kPlaceSharedPacked, B> { using A = AccSharedPacked<B>; };

// ------------------------------------------------------------------------------------
// Block merge and the single global merge per block.
// ------------------------------------------------------------------------------------
// 128-bit signed add of (lo, hi) into a device (lo, hi) word pair with two atomics.
__device__ __forceinline__ void atomic_add128(uint64_t* lo_p, uint64_t* hi_p, uint64_t lo, uint64_t hi) {
  uint64_t carry = 0;
  if (lo) {
    const uint64_t old = atomicAdd((unsigned long long*)lo_p, (unsigned long long)lo);
    carry = (old + lo) < old;
  }
  if (hi + carry) atomicAdd((unsigned long long*)hi_p, (unsigned long long)(hi + carry));
}

// A store to pinned host memory.  System-scope stores go past every cache of the device, so
// the wait for them (vmcnt 0) is all that orders them before a later one; a system-scope
// fence would also write back the XCD's L2.
__device__ __forceinline__ void store_host(uint64_t* p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A word, or a (lo, hi) pair, of a block's sums: added into a device table, or (DIRECT) stored
// into the block's own record in host memory.
template <bool DIRECT>
__device__ __forceinline__ void put_word(uint64_t* p, uint64_t v) {
  if (DIRECT)
    store_host(p, v);
  else
    atomicAdd((unsigned long long*)p, (unsigned long long)v);
}
template <bool DIRECT>
__device__ __forceinline__ void put_pair(uint64_t* lo_p, uint64_t* hi_p, uint64_t lo, uint64_t hi) {
  if (DIRECT) {
    store_host(lo_p, lo);
    store_host(hi_p, hi);
  } else {
    atomic_add128(lo_p, hi_p, lo, hi);
  }
}

// The block's merge into `out`: the wavefronts' sums red[wave][group][NF] are added in 128
// bits.  qty_scale turns layout units into x100.
template <bool DIRECT = false>
__device__ __forceinline__ void block_merge(const uint64_t* red, q1_device_aggregates* out, uint64_t qty_scale) {
  const uint32_t nwaves = blockDim.x >> 6;
  __syncthreads();
  // Thread g*NF + f sums field f of group g over the waves (128-bit) and issues that
  // field's atomics, so a block's destination atomics go out together.
  if (thread_index() < kNumGroups * NF) {
    const int g = thread_index() / NF, f = thread_index() % NF;
    uint64_t lo = 0, hi = 0, cnt = 0, plo = 0, phi = 0;
    for (uint32_t w = 0; w < nwaves; w++) {
      const uint64_t* r = red + (w * kNumGroups + g) * NF;
      const uint64_t v = r[f];
      lo += v;
      hi += lo < v;
      cnt |= r[F_CNT];
      const uint64_t pv = r[F_PRICE];
      plo += pv;
      phi += plo < pv;
    }
    if (DIRECT || cnt) {
      switch (f) {
        case F_QTY: put_word<DIRECT>(&out->sum_qty[g], lo * qty_scale); break;
        case F_PRICE: put_word<DIRECT>(&out->sum_base_price[g], lo); break;
        case F_DISC: put_word<DIRECT>(&out->sum_disc[g], lo); break;
        case F_CNT: put_word<DIRECT>(&out->count[g], lo); break;
        case F_DPROD: {
          // sum_disc_price = 100 * sum_price - sum(disc * price), in 128 bits
          const unsigned __int128 p100 = ((unsigned __int128)phi << 64 | plo) * 100u;
          const unsigned __int128 dp = p100 - ((unsigned __int128)hi << 64 | lo);
          put_pair<DIRECT>(&out->sum_disc_price_lo[g], &out->sum_disc_price_hi[g], (uint64_t)dp, (uint64_t)(dp >> 64));
          break;
        }
        default: put_pair<DIRECT>(&out->sum_charge_lo[g], &out->sum_charge_hi[g], lo, hi); break;
      }
    }
  }
}

// The end of a block that merged into table t of the tables its range's blocks share, called
// by wavefront 0 of the block, which issued the merge atomics; `sharing` blocks merge into
// table t, and `used` tables have blocks.  Returns whether this is the last block of the
// range (count_block): lane w then holds word w of the sums (w < 48), lane 48 what was in *extra
// (if not null), and all of it is zero again.
// Ordering: the tables and the counters are only ever touched by device-scope
// atomics, which are performed at memory, past the XCDs' L2 caches.  A block counts itself
// only after its own atomics have been performed (the wait below), so the block that draws
// the last count finds every table complete; it takes the words with exchanges, which read
// memory and clear it in one.  No fence is needed, and none is affordable: a release
// writes back the XCD's L2, under the loads of all its blocks (one per block makes 600M rows
// take 1.41 ms instead of 0.85).
// What it replaces is a zero-fill launch before the scan, a fold launch and a copy to the
// host after it, each 2-5 us of a short call: q1_run of 5,003 rows 32.3 -> 18.9 us, of 1M
// rows 39.0 -> 23.9.  A block's own part is two waits for an atomic; the other blocks of
// its compute unit cover them (600M rows, 18,311 blocks: 862 -> 847 us per call).  The start
// clock is read with the tables and the counts clear themselves: 10 blocks 14.4 -> 13.8 us, 1M
// rows 15.8 -> 15.3, a launch of 2M rows on a caller's stream 22.7 -> 22.2.
__device__ __forceinline__ bool count_block(MergeTable* tables, uint32_t t, uint32_t sharing, uint32_t used) {
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  uint32_t last = 0;
  if ((thread_index() & 63) == 0) {
    // atomicInc goes from its second argument back to 0: the last one clears the count.
    last = sharing == 1 || atomicInc(&tables[t].merged, sharing - 1) == sharing - 1;
    if (last && used > 1) last = atomicInc(&tables[0].tables_merged, used - 1) == used - 1;
  }
  last = (uint32_t)__builtin_amdgcn_readfirstlane((int)last);
  __asm__ volatile("" ::: "memory");
  return last;
}
__device__ __forceinline__ bool finish_tables(MergeTable* tables, uint32_t t, uint32_t sharing, uint32_t used,
                                              uint64_t& sum, uint64_t* extra = nullptr) {
  if (!count_block(tables, t, sharing, used)) return false;
  const uint32_t lane = thread_index() & 63;
  // Lane w sums word w of the tables in use.  A 128-bit field is two words: the lane of the
  // low one counts its carries, which then go to the lane of the high one, 6 lanes on.
  constexpr uint32_t kWords = sizeof(q1_device_aggregates) / 8;
  static_assert(kWords == 48 && kNumGroups == 6, "8 fields of 6 groups, the 128-bit ones at words 12..35");
  uint64_t s = 0, carry = 0, other = 0;
  if (extra && lane == kWords) other = atomicExch((unsigned long long*)extra, 0ull);
  if (lane < kWords) {
    for (uint32_t k = 0; k < used; k += 16) {
      uint64_t v[16];
#pragma unroll
      for (uint32_t i = 0; i < 16; i++)
        v[i] = k + i < used ? __hip_atomic_exchange(reinterpret_cast<uint64_t*>(&tables[k + i].sums) + lane, 0ull,
                                                    __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                            : 0;
#pragma unroll
      for (uint32_t i = 0; i < 16; i++) {
        s += v[i];
        carry += s < v[i];
      }
    }
  }
  const uint64_t carried = __shfl(carry, (int)lane - kNumGroups, 64);  // lanes below 6 ignore it
  if ((lane >= 18 && lane < 24) || (lane >= 30 && lane < 36)) s += carried;
  sum = lane == kWords ? other : s;
  return true;
}

// Blocks of a range of `blocks` blocks that share the table of block b.
__device__ __forceinline__ uint32_t blocks_sharing(uint32_t blocks, uint32_t b, uint32_t table_mask) {
  return (blocks - (b & table_mask) + table_mask) / (table_mask + 1);
}

// Around a scan kernel's body: the launch's start clock, where block b merges, and the end of
// the merge.
__device__ __forceinline__ void begin_scan(const ScanArgs& a) {
  if (a.host && blockIdx.x == 0 && thread_index() == 0)
    __hip_atomic_store(&a.set->clock_begin, (uint64_t)wall_clock64(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ q1_device_aggregates* merge_target(const ScanArgs& a) {
  return a.set ? &a.set->table[blockIdx.x & a.table_mask].sums : a.out;
}
__device__ __forceinline__ void finish_scan(const ScanArgs& a) {
  if (!a.set || thread_index() >= 64) return;
  MergeSet* const set = a.set;
  const uint32_t lane = thread_index() & 63;
  const uint32_t grid = gridDim.x, b = blockIdx.x, used = grid <= a.table_mask ? grid : a.table_mask + 1;
  uint64_t sum;
  if (!finish_tables(set->table, b & a.table_mask, blocks_sharing(grid, b, a.table_mask), used, sum,
                     a.host ? &set->clock_begin : nullptr))
    return;
  if (!a.host) {
    if (a.done) {
      __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the set is zero
      if (lane == 0) store_host(a.done, a.sequence);
    }
    uint64_t* d = reinterpret_cast<uint64_t*>(a.out);
    const uint64_t hi = __shfl(sum, (int)lane + kNumGroups, 64);  // of a low lane: its high word
    const bool low = (lane >= 12 && lane < 18) || (lane >= 24 && lane < 30);
    const bool high = (lane >= 18 && lane < 24) || (lane >= 30 && lane < 36);
    if (low) {
      atomic_add128(d + lane, d + lane + kNumGroups, sum, hi);
    } else if (lane < 48 && !high && sum) {
      atomicAdd((unsigned long long*)(d + lane), (unsigned long long)sum);
    }
    return;
  }
  // Everything but the sequence number, then the number.
  static_assert(offsetof(HostResult, clock_begin) == sizeof(q1_device_aggregates), "word 48");
  if (lane < 49) store_host(reinterpret_cast<uint64_t*>(&a.host->sums) + lane, sum);
  if (lane == 0) store_host(&a.host->clock_end, wall_clock64());
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (lane == 0) store_host(&a.host->sequence, a.sequence);
}

// ------------------------------------------------------------------------------------
// Row bodies of one tile group.
// ------------------------------------------------------------------------------------
// Row j of a tile into an accumulator, in the row form the accumulator takes.  SLOT: the
// caller knows that the row's slot is below 6.
template <bool EDGE, bool SLOT, class Tile, class Acc>
__device__ __forceinline__ void add_row(const Tile& tile, int j, Acc& acc, int32_t cut, uint32_t valid) {
  if constexpr (Acc::kWideRows) {
    const WideRow r = tile.template wide<EDGE>(j, cut, valid);
    if (SLOT) __builtin_assume(r.gid < kNumGroups);
    acc.add(r);
  } else {
    const FastRow r = tile.template fast<EDGE>(j, cut, valid);
    if (SLOT) __builtin_assume(r.gid < kNumGroups);
    acc.add(r);
  }
}

// A whole group inside the range.  Rows with the unused return-flag code are first made
// to fail the filter (a wavefront-uniform branch that real data never takes), so every
// row's slot is below 6 and the slot test drops out of the row body.
template <class Tile, int U, class Acc>
__device__ __forceinline__ void add_whole_group(TileGroup<Tile, U>& grp, Acc& acc, int32_t cut) {
  constexpr int TILE = Tile::TILE;
  uint32_t bad = 0;
#pragma unroll
  for (int m = 0; m < U; m++) bad |= grp.tile[m].bad_codes();
  if (ballot(bad != 0)) {
#pragma unroll
    for (int m = 0; m < U; m++) grp.tile[m].drop_bad_codes();
  }
#pragma unroll
  for (int m = 0; m < U; m++)
#pragma unroll
    for (int j = 0; j < TILE; j++) add_row<false, true>(grp.tile[m], j, acc, cut, 0);
}

// Any group: tiles may be unused, or partial at the range's ends.
template <class Tile, int U, class Acc>
__device__ __forceinline__ void add_any_group(const TileGroup<Tile, U>& grp, Acc& acc, int32_t cut) {
  constexpr int TILE = Tile::TILE;
#pragma unroll
  for (int m = 0; m < U; m++) {
    if (!grp.use[m]) continue;
#pragma unroll
    for (int j = 0; j < TILE; j++) add_row<true, false>(grp.tile[m], j, acc, cut, grp.valid[m]);
  }
}

// A group at an end of the range for the register tables: tile by tile, so that the kernel
// holds one guarded copy of a tile's rows beside the whole groups' (with a guarded copy of
// every row of a group the compressed kernels take 142-180 registers and spill, 106-136 so).
template <class Tile, int U, class Acc>
__device__ __forceinline__ void add_end_tiles(const ScanArgs& a, uint64_t t0, uint64_t stride, uint32_t count,
                                              uint64_t end_tile, Acc& acc, int32_t cut) {
#pragma unroll 1
  for (uint32_t m = 0; m < U; m++) {
    TileGroup<Tile, 1> one;
    one.load(a.cols, t0 + m * stride, stride, m < count ? 1 : 0, end_tile, a.row_begin, a.row_end);
    add_any_group(one, acc, cut);
  }
}

// The tiles base + k * B + lane (k < tiles_per_thread) of a block's lanes into a table.
// Groups k in [k_lo, k_end) are whole and inside the range for every lane of the
// block: the tiles of group k are base + (k + m) * B + lane, and they all lie in
// [whole_begin, whole_end), the tiles with no row outside [row_begin, row_end).  They
// run a branch-free body; the few others (the range's first and last groups) a
// guarded one.  A dropped row's ship date 0xFFFF must fail the filter: compressed
// cutoffs of 65535 and above (beyond the year 2170) take the guarded body throughout.
template <int L, class Tile, int B, class Acc>
__device__ __forceinline__ void add_tiles(const ScanArgs& a, uint64_t base, uint32_t tiles_per_thread, Acc& acc,
                                          int32_t cut) {
  constexpr int TILE = Tile::TILE;
  constexpr int U = Tile::GROUP;
  constexpr int FLUSH = U * TILE >= 16 ? 1 : 16 / (U * TILE);  // groups per 16 rows
  const uint64_t end_tile = (a.row_end + TILE - 1) / TILE;
  const uint64_t whole_begin = (a.row_begin + TILE - 1) / TILE, whole_end = a.row_end / TILE;
  uint32_t k_lo = 0, k_end = 0;
  if ((L != Q1_LAYOUT_COMPRESSED || cut < 65535) && whole_end > base) {
    const uint64_t lo = base >= whole_begin ? 0 : (whole_begin - base + B - 1) / B;
    const uint64_t klo = (lo + U - 1) / U * U;
    uint64_t kmax = (whole_end - base) / B;  // groups with k + U <= kmax are inside
    if (kmax > tiles_per_thread) kmax = tiles_per_thread;
    if (kmax >= klo + U) {
      k_lo = (uint32_t)klo;
      k_end = (uint32_t)(klo + (kmax - klo) / U * U);
    }
  }
  auto add_end_group = [&](uint32_t k) {
    const uint64_t t0 = base + (uint64_t)k * B + thread_index();
    if constexpr (Acc::kCompactEnds) {
      add_end_tiles<Tile, U>(a, t0, B, tiles_per_thread - k, end_tile, acc, cut);
    } else {
      TileGroup<Tile, U> grp;
      grp.load(a.cols, t0, B, tiles_per_thread - k, end_tile, a.row_begin, a.row_end);
      add_any_group(grp, acc, cut);
    }
  };
  uint32_t k = 0;
  for (; k < k_lo; k += U) {
    add_end_group(k);
    if ((k / U + 1) % FLUSH == 0) acc.flush();
  }
  for (; k < k_end; k += U) {
    TileGroup<Tile, U> grp;
    grp.load_plain(a.cols, base + (uint64_t)k * B + thread_index(), B);
    add_whole_group(grp, acc, cut);
    if ((k / U + 1) % FLUSH == 0) acc.flush();
  }
  for (; k < tiles_per_thread; k += U) {
    add_end_group(k);
    if ((k / U + 1) % FLUSH == 0) acc.flush();
  }
}

// ------------------------------------------------------------------------------------
// The fast scan kernel: layout L, placement P.
// ------------------------------------------------------------------------------------
// One block's share of a range: block `block` of the grid that launch_scan would run over
// a's rows, merged into *out.  `lds` is the block's dynamic LDS.
template <int L, int P, int B, bool DIRECT = false>
__device__ __forceinline__ void scan_block(const ScanArgs& a, uint64_t block, uint32_t host_tiles_per_thread,
                                           uint64_t* ws, uint64_t* lds, q1_device_aggregates* out) {
  using Tile = typename TileOf<L>::T;
  using Acc = typename AccOf<P, B>::A;
  constexpr int TILE = Tile::TILE;
  constexpr int SUB = kHostTileRows<L> / TILE;  // kernel tiles per tile the host counts

  const int32_t cut = column_cutoff<L>(a.cutoff_day);
  // Block b covers kernel tiles [first_tile + b*B*tpt, +B*tpt): SUB times the host's
  // tiles per lane, so the grid covers every row of the range.  The first tile is that of
  // row_begin rounded down to kRowAlign rows, as the host counts them.
  static_assert(kRowAlign % TILE == 0, "kRowAlign is a whole number of tiles");
  const uint32_t tiles_per_thread = host_tiles_per_thread * SUB;
  const uint64_t first_tile = a.row_begin / kRowAlign * kRowAlign / TILE;
  const uint64_t base = first_tile + block * B * tiles_per_thread;

  Acc acc;
  // the local placement's table in the lane's private memory (unused by the others)
  uint64_t private_table[P == Q1_PLACE_LOCAL_MEM ? AccLocal::kTableWords : 1];
  if constexpr (P == Q1_PLACE_GLOBAL) acc.init_global(ws);
  if constexpr (P == Q1_PLACE_LOCAL_MEM)
    acc.init(reinterpret_cast<char*>(private_table));
  else
    acc.init(reinterpret_cast<char*>(lds));

  add_tiles<L, Tile, B>(a, base, tiles_per_thread, acc, cut);
  acc.flush(true);

  const uint64_t qty_scale =
      (L == Q1_LAYOUT_COMPRESSED || L == Q1_LAYOUT_COMPRESSED_PUSHDOWN) ? kQuantityScaleCompressed : 1;
  // The reduction scratch follows the placement's own LDS table or staging rows.
  uint64_t* red = lds + Acc::lds_bytes(B) / 8;
  if constexpr (P == Q1_PLACE_GLOBAL) {
    acc.merge(lds, red, out, qty_scale);  // through the block's table in global memory
  } else {
    if constexpr (P == Q1_PLACE_PER_THREAD_SHARED_MEM || P == kPlaceSharedNarrow || P == kPlaceSharedPacked) {
      acc.wave_totals(red);
    } else {
      LaneWords w;
      acc.words(w);
      sum_lane_words(w, lds, red);
    }
    block_merge<DIRECT>(red, out, qty_scale);
  }
}

template <int L, int P, int B>
__global__ void __launch_bounds__(B)
scan_fast(ScanArgs a, uint32_t host_tiles_per_thread, uint64_t* ws) {
  extern __shared__ uint64_t lds[];
  begin_scan(a);
  scan_block<L, P, B>(a, blockIdx.x, host_tiles_per_thread, ws, lds, merge_target(a));
  finish_scan(a);
}

// The shortest queries: a grid of at most kDirectBlocks blocks, each of which leaves its sums,
// clocks and `sequence` in a host record of its own, for the host to add.  What it saves is the
// chain at a short kernel's end of an atomic, the block count, the exchange and the store, each
// waiting a microsecond for the last: 5,003 rows (2 blocks) 13.2 -> 11.5 us per call, kernel 5.5
// -> 3.7; 5 blocks 14.3 -> 12.4; 10 blocks 13.7 -> 12.8.  At 16 blocks the host's reading of the
// records costs more (13.5 -> 14.2 us).  A kernel of its own, without an argument for it: the
// choice at run time in every kernel's tail, and one more word of ScanArgs, each made all
// longer launches 0.3 us slower.
template <int L, int P, int B>
__global__ void __launch_bounds__(B)
scan_direct(ScanArgs a, uint32_t host_tiles_per_thread) {
  extern __shared__ uint64_t lds[];
  HostResult* const mine = a.host + blockIdx.x;
  if (thread_index() == 0) store_host(&mine->clock_begin, wall_clock64());
  scan_block<L, P, B, true>(a, blockIdx.x, host_tiles_per_thread, nullptr, lds, &mine->sums);
  if (thread_index() < 64) {  // wavefront 0 stored the sums
    if (thread_index() == 0) store_host(&mine->clock_end, wall_clock64());
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (thread_index() == 0) store_host(&mine->sequence, a.sequence);
  }
}

// ------------------------------------------------------------------------------------
// The any-value scan kernel (tables outside the TPC-H domain, and launches without
// Q1_LAUNCH_ASSUME_TPCH_DOMAIN): exact for every input with the reference's arithmetic,
// wrapping int64 per-row products and 128-bit signed sums, whatever the values.  It is the
// shared placement's kernel with LDS tables whose words hold any value of the layout's
// types, so a row takes the same branch-free path inside and outside the domain: streaming
// tiles, 3 (compressed), 5 (uncompressed) or 7 (reference) return-less 64-bit LDS atomics.
// The fields of a word are exact for any_value_lane_rows rows per lane, which make_shape
// keeps to.
// Bound by HBM, as the narrow kernel: 600M compressed rows 0.82-0.84 ms (narrow 0.83), 60M
// uncompressed 190 us, 60M reference 341 us (6.7 TB/s).  Testing each tile for the domain and
// sending the others to 128-bit sums in registers or private memory took 281 us for 60M
// compressed rows with two thirds of them outside (now 93), and 27 us for a 1M-row launch,
// whose blocks each reduced both kinds of sums (now 12).
// ------------------------------------------------------------------------------------
// A wavefront's sums of one group in red[wave][group][NA]: 64-bit (wrapping, as the
// reference's int64 sums), the products as 128-bit word pairs.
enum { A_QTY, A_PRICE, A_DISC, A_CNT, A_DP_LO, A_DP_HI, A_CH_LO, A_CH_HI, NA };

__device__ __forceinline__ void store_i128(uint64_t* lo_hi, __int128 v) {
  lo_hi[0] = (uint64_t)v;
  lo_hi[1] = (uint64_t)((unsigned __int128)v >> 64);
}
// The two halves of the sum of up to 2^23 int64 values, split into unsigned low and signed
// high 32-bit words.
__device__ __forceinline__ __int128 join_i128(uint64_t lo_sum, int64_t hi_sum) {
  return (__int128)hi_sum * ((__int128)1 << 32) + (__int128)lo_sum;
}
// a word's signed sum in bits [0,40) and the rest of it, sum >> 40 (below 2^24)
__device__ __forceinline__ int64_t low40(uint64_t w) { return (int64_t)(w << 24) >> 24; }
__device__ __forceinline__ uint32_t high24(uint64_t w) { return (uint32_t)((w - (uint64_t)low40(w)) >> 40); }

// Compressed layouts: quantity, discount and tax are bytes and the price has 32 bits, so every
// product fits 64 bits and a lane's sums over 128 rows fit three words:
//   word 0: price (< 2^39) in bits [0,39), discount (< 2^15) in [39,54), count in [54,62)
//   word 1: discount x price (< 2^47) in [0,47), quantity (< 2^15) in [47,62)
//   word 2: (f + 55025) x price, f = (100 - discount)(100 + tax) in [-55025, 35500] (< 2^56)
// Two multiplications a row beyond the narrow table's, both with a 64-bit result.
template <int B>
struct AnyCompressed {
  static constexpr bool kWideRows = false, kCompactEnds = false;
  static constexpr int W = 3;
  static_assert(any_value_lane_rows(Q1_LAYOUT_COMPRESSED) <= 128, "the fields' widths");
  static constexpr uint32_t kFactorBias = 55025;
  uint64_t* tab;
  __device__ __forceinline__ void flush(bool = false) {}
  __device__ __forceinline__ void init(uint64_t* lds) {
    tab = lds;
    clear_wave_table<B, W>(tab);
  }
  __device__ __forceinline__ void add(const FastRow& r) {
    if (__builtin_expect(r.counts(), 1)) {
      uint64_t* base = tab + r.gid * (W * B) + thread_index();
      const uint32_t f = (uint32_t)(__mul24(100 - (int)r.disc, 100 + (int)r.tax) + (int)kFactorBias);
      const uint64_t w0 = (uint64_t)r.price | (uint64_t)(r.disc << 7 | 1u << 22) << 32;
      const uint64_t w1 = (uint64_t)r.disc * r.price + ((uint64_t)(r.qty << 15) << 32);
      __hip_atomic_fetch_add(base, w0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __hip_atomic_fetch_add(base + B, w1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __hip_atomic_fetch_add(base + 2 * B, (uint64_t)f * r.price, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
  struct GroupSums {
    static constexpr int kWords = NA;
    uint64_t price = 0, dprod = 0, charge = 0;
    uint32_t disc = 0, cnt = 0, qty = 0;
    __device__ __forceinline__ void add(const uint64_t (&w)[W]) {
      price += w[0] & ((1ull << 39) - 1);
      disc += (uint32_t)(w[0] >> 39) & 0x7FFFu;
      cnt += (uint32_t)(w[0] >> 54);
      dprod += w[1] & ((1ull << 47) - 1);
      qty += (uint32_t)(w[1] >> 47);
      charge += w[2];
    }
    template <class F>
    __device__ __forceinline__ void reduce(F f) {
      f(price);
      f(disc);
      f(cnt);
      f(dprod);
      f(qty);
      f(charge);
    }
    // over a wavefront: price < 2^45, discount x price < 2^53, word 2 < 2^62
    __device__ __forceinline__ void store(uint64_t* r) const {
      r[A_QTY] = qty;
      r[A_PRICE] = price;
      r[A_DISC] = disc;
      r[A_CNT] = cnt;
      store_i128(r + A_DP_LO, (__int128)((int64_t)(100 * price) - (int64_t)dprod));
      store_i128(r + A_CH_LO, (__int128)((int64_t)charge - (int64_t)(kFactorBias * price)));
    }
  };
  __device__ __forceinline__ void wave_totals(uint64_t* red) const { sum_wave_table<B, W, GroupSums>(tab, red); }
  static constexpr uint32_t lds_bytes(uint32_t threads) { return W * kNumGroups * 8u * threads; }
};

// A wrapping 64-bit product whose second factor is a signed 32-bit value.
__device__ __forceinline__ uint64_t mul_64_s32(uint64_t a, int32_t f) {
  const uint32_t lo = (uint32_t)a, hi = (uint32_t)(a >> 32);
  const uint64_t p = (uint64_t)lo * (uint32_t)f;
  const uint32_t top = (uint32_t)(p >> 32) + hi * (uint32_t)f - (f < 0 ? lo : 0u);
  return (uint64_t)top << 32 | (uint32_t)p;
}

// Uncompressed layout: int64 price, int32 quantity, int8 discount and tax; the products are
// split into unsigned low and signed high halves.  A lane's sums over 256 rows fit five words:
//   word 0: low halves of disc_price (< 2^40) in bits [0,48), count in [48,57)
//   word 1: high halves of disc_price (signed) in [0,40), discount + 128 in [40,56)
//   word 2: low halves of charge in [0,40), low half-word of quantity in [40,64)
//   word 3: high halves of charge (signed) in [0,40), high half-word of quantity + 2^15 in [40,64)
//   word 4: price (wrapping)
template <int B>
struct AnyUncompressed {
  static constexpr bool kWideRows = true, kCompactEnds = false;
  static constexpr int W = 5;
  static_assert(any_value_lane_rows(Q1_LAYOUT_UNCOMPRESSED) <= 256, "the fields' widths");
  uint64_t* tab;
  __device__ __forceinline__ void flush(bool = false) {}
  __device__ __forceinline__ void init(uint64_t* lds) {
    tab = lds;
    clear_wave_table<B, W>(tab);
  }
  __device__ __forceinline__ void add(const WideRow& r) {
    if (__builtin_expect(r.counts(), 1)) {
      uint64_t* base = tab + r.gid * (W * B) + thread_index();
      const int32_t disc = (int32_t)r.disc, qty = (int32_t)r.qty, d1 = 100 - disc;
      const uint64_t dp = mul_64_s32((uint64_t)r.price, d1);
      const uint64_t ch = mul_64_s32((uint64_t)r.price, __mul24(d1, 100 + (int32_t)r.tax));
      const uint64_t w[W] = {(uint64_t)(uint32_t)dp | 1ull << 48,
                             (uint64_t)((int64_t)dp >> 32) + ((uint64_t)(uint32_t)(disc + 128) << 40),
                             (uint64_t)(uint32_t)ch | (uint64_t)((uint32_t)qty & 0xFFFFu) << 40,
                             (uint64_t)((int64_t)ch >> 32) + ((uint64_t)(uint32_t)((qty >> 16) + 32768) << 40),
                             (uint64_t)r.price};
#pragma unroll
      for (int i = 0; i < W; i++)
        __hip_atomic_fetch_add(base + i * B, w[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
  struct GroupSums {
    static constexpr int kWords = NA;
    uint64_t dp_lo_cnt = 0, dp_hi = 0, ch_lo = 0, ch_hi = 0, price = 0;
    uint32_t disc = 0, qty_lo = 0, qty_hi = 0;
    __device__ __forceinline__ void add(const uint64_t (&w)[W]) {
      dp_lo_cnt += w[0];  // a wavefront's sums fit the fields
      dp_hi += (uint64_t)low40(w[1]);
      disc += high24(w[1]);
      ch_lo += w[2] & ((1ull << 40) - 1);
      qty_lo += (uint32_t)(w[2] >> 40);
      ch_hi += (uint64_t)low40(w[3]);
      qty_hi += high24(w[3]);
      price += w[4];
    }
    template <class F>
    __device__ __forceinline__ void reduce(F f) {
      f(dp_lo_cnt);
      f(dp_hi);
      f(disc);
      f(ch_lo);
      f(qty_lo);
      f(ch_hi);
      f(qty_hi);
      f(price);
    }
    __device__ __forceinline__ void store(uint64_t* r) const {
      const int64_t cnt = (int64_t)(dp_lo_cnt >> 48);
      r[A_QTY] = (uint64_t)((int64_t)qty_lo + ((int64_t)qty_hi - 32768 * cnt) * 65536);
      r[A_PRICE] = price;
      r[A_DISC] = (uint64_t)((int64_t)disc - 128 * cnt);
      r[A_CNT] = (uint64_t)cnt;
      store_i128(r + A_DP_LO, join_i128(dp_lo_cnt & ((1ull << 48) - 1), (int64_t)dp_hi));
      store_i128(r + A_CH_LO, join_i128(ch_lo, (int64_t)ch_hi));
    }
  };
  __device__ __forceinline__ void wave_totals(uint64_t* red) const { sum_wave_table<B, W, GroupSums>(tab, red); }
  static constexpr uint32_t lds_bytes(uint32_t threads) { return W * kNumGroups * 8u * threads; }
};

// Reference layout: every value int64.  Seven words: low halves of disc_price with the count
// in bits [48,57), its high halves, low and high halves of charge, and the wrapping sums of
// price, quantity and discount.
template <int B>
struct AnyReference {
  static constexpr bool kWideRows = true, kCompactEnds = false;
  static constexpr int W = 7;
  static_assert(any_value_lane_rows(Q1_LAYOUT_REFERENCE) <= 256, "the fields' widths");
  uint64_t* tab;
  __device__ __forceinline__ void flush(bool = false) {}
  __device__ __forceinline__ void init(uint64_t* lds) {
    tab = lds;
    clear_wave_table<B, W>(tab);
  }
  __device__ __forceinline__ void add(const WideRow& r) {
    if (__builtin_expect(r.counts(), 1)) {
      uint64_t* base = tab + r.gid * (W * B) + thread_index();
      const uint64_t dp = (100ull - (uint64_t)r.disc) * (uint64_t)r.price;
      const uint64_t ch = dp * (100ull + (uint64_t)r.tax);
      const uint64_t w[W] = {(uint64_t)(uint32_t)dp | 1ull << 48, (uint64_t)((int64_t)dp >> 32),
                             (uint64_t)(uint32_t)ch,              (uint64_t)((int64_t)ch >> 32),
                             (uint64_t)r.price,                   (uint64_t)r.qty,
                             (uint64_t)r.disc};
#pragma unroll
      for (int i = 0; i < W; i++)
        __hip_atomic_fetch_add(base + i * B, w[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  }
  struct GroupSums {
    static constexpr int kWords = NA;
    uint64_t w[W] = {};
    __device__ __forceinline__ void add(const uint64_t (&v)[W]) {
#pragma unroll
      for (int i = 0; i < W; i++) w[i] += v[i];
    }
    template <class F>
    __device__ __forceinline__ void reduce(F f) {
#pragma unroll
      for (int i = 0; i < W; i++) f(w[i]);
    }
    __device__ __forceinline__ void store(uint64_t* r) const {
      r[A_QTY] = w[5];
      r[A_PRICE] = w[4];
      r[A_DISC] = w[6];
      r[A_CNT] = w[0] >> 48;
      store_i128(r + A_DP_LO, join_i128(w[0] & ((1ull << 48) - 1), (int64_t)w[1]));
      store_i128(r + A_CH_LO, join_i128(w[2], (int64_t)w[3]));
    }
  };
  __device__ __forceinline__ void wave_totals(uint64_t* red) const { sum_wave_table<B, W, GroupSums>(tab, red); }
  static constexpr uint32_t lds_bytes(uint32_t threads) { return W * kNumGroups * 8u * threads; }
};

template <int L, int B> struct AnyOf { using A = AnyCompressed<B>; };
template <int B> struct AnyOf<Q1_LAYOUT_UNCOMPRESSED, B> { using A = AnyUncompressed<B>; };
template <int B> struct AnyOf<Q1_LAYOUT_REFERENCE, B> { using A = AnyReference<B>; };

// The block's merge: thread 8g + i of wavefront 0 adds word (or word pair) i of group g over
// the wavefronts and issues its atomics.
template <int B>
__device__ __forceinline__ void any_merge(const uint64_t* red, q1_device_aggregates* out, uint64_t qty_scale) {
  __syncthreads();
  const uint32_t g = thread_index() >> 3, f = thread_index() & 7;
  if (g >= kNumGroups || f == A_DP_HI || f == A_CH_HI) return;
  const bool pair = f == A_DP_LO || f == A_CH_LO;
  uint64_t lo = 0, hi = 0;
#pragma unroll
  for (int w = 0; w < B / 64; w++) {
    const uint64_t* r = red + (w * kNumGroups + g) * NA + f;
    lo += r[0];
    if (pair) hi += r[1] + (lo < r[0]);
  }
  if (f == A_QTY) lo *= qty_scale;
  if (pair) {
    atomic_add128(f == A_DP_LO ? &out->sum_disc_price_lo[g] : &out->sum_charge_lo[g],
                  f == A_DP_LO ? &out->sum_disc_price_hi[g] : &out->sum_charge_hi[g], lo, hi);
  } else if (lo) {
    uint64_t* d = f == A_QTY     ? out->sum_qty
                  : f == A_PRICE ? out->sum_base_price
                  : f == A_DISC  ? out->sum_disc
                                 : out->count;
    atomicAdd((unsigned long long*)(d + g), (unsigned long long)lo);
  }
}

template <int L, int B>
__global__ void __launch_bounds__(B)
scan_any(ScanArgs a, uint32_t host_tiles_per_thread) {
  using Tile = typename TileOf<L>::T;
  using Acc = typename AnyOf<L, B>::A;
  constexpr int TILE = Tile::TILE;
  constexpr int SUB = kHostTileRows<L> / TILE;  // kernel tiles per tile the host counts
  constexpr uint64_t kQtyScale =
      (L == Q1_LAYOUT_COMPRESSED || L == Q1_LAYOUT_COMPRESSED_PUSHDOWN) ? kQuantityScaleCompressed : 1;
  extern __shared__ uint64_t lds[];
  begin_scan(a);
  const uint32_t tiles_per_thread = host_tiles_per_thread * SUB;
  const uint64_t first_tile = a.row_begin / kRowAlign * kRowAlign / TILE;  // as the host counts them
  Acc acc;
  acc.init(lds);
  add_tiles<L, Tile, B>(a, first_tile + (uint64_t)blockIdx.x * B * tiles_per_thread, tiles_per_thread, acc,
                        column_cutoff<L>(a.cutoff_day));
  uint64_t* red = lds + Acc::lds_bytes(B) / 8;
  acc.wave_totals(red);
  any_merge<B>(red, merge_target(a), kQtyScale);
  finish_scan(a);
}

// ------------------------------------------------------------------------------------
// The batched persistent kernel.
// ------------------------------------------------------------------------------------
// Column pointers read from a descriptor.  Pointers that arrive as kernel arguments are
// known to be global; generic ones loaded from memory make flat loads: 64-bit vector
// addresses, and flat loads count against the LDS wait counter too, so every wait for an
// LDS atomic would also wait for them.  Reading the pointers as global-qualified values
// keeps the tile loads global (a scalar base plus a vector offset).
typedef const __attribute__((address_space(1))) void* GlobalPtr;
struct GlobalColumns {
  GlobalPtr ship_date, quantity, extended_price, discount, tax, return_flag, line_status, filter;
};
static_assert(sizeof(GlobalColumns) == sizeof(q1_columns), "same layout as q1_columns");

__device__ __forceinline__ q1_columns load_global_columns(const q1_columns* src) {
  const GlobalColumns g = *reinterpret_cast<const GlobalColumns*>(src);
  q1_columns c;
  c.ship_date = (const void*)g.ship_date;
  c.quantity = (const void*)g.quantity;
  c.extended_price = (const void*)g.extended_price;
  c.discount = (const void*)g.discount;
  c.tax = (const void*)g.tax;
  c.return_flag = (const void*)g.return_flag;
  c.line_status = (const void*)g.line_status;
  c.filter = (const void*)g.filter;
  return c;
}

// The last request whose first block is <= v, from request r on (whose first block is <= v).
// First blocks never decrease along the list, so the requests that pass form a prefix of
// those that the lanes look at.
// find_request: of the whole list (first[0] = 0): the lanes look at 64 requests evenly spread
// over what is left of it; n <= 64 takes one look, n <= 4096 two.
// next_request: forward from a block's last request, 64 neighbours at a look.
__device__ __forceinline__ uint32_t find_request(const uint32_t* first, uint32_t n, uint32_t v) {
  const uint32_t lane = thread_index() & 63;
  uint32_t r = 0, left = n;
  while (left > 1) {
    const uint32_t step = (left + 63) / 64, i = lane * step;
    const uint32_t pass = (uint32_t)__popcll(ballot(i < left && first[r + i] <= v));
    r += (pass - 1) * step;
    left = left - (pass - 1) * step < step ? left - (pass - 1) * step : step;
  }
  return r;
}
__device__ __forceinline__ uint32_t next_request(const uint32_t* first, uint32_t n, uint32_t r, uint32_t v) {
  const uint32_t lane = thread_index() & 63;
  for (;;) {
    const uint32_t i = r + 1 + lane;
    const uint32_t pass = (uint32_t)__popcll(ballot(i < n && first[i] <= v));
    r += pass;
    if (pass < 64) return r;
  }
}

// The batched kernel: the requests' scan blocks (request r's block k is the block k that
// launch_scan would run over r's rows alone, with hdr->tiles_per_thread) form one list of
// hdr->total_blocks blocks.  Block b runs entries b, b + gridDim.x, b + 2 gridDim.x, ...  The
// blocks in flight therefore read neighbouring stretches of HBM whatever the request sizes,
// with no shared counter (a claim counter that every block updates once per entry cost
// 6-11 % of the read rate of this structure).  Each entry runs the scan kernel's block body
// and merges into one of its request's tables; the last entry of a request stores its result
// into host memory, and the last request's then the done record.  Every block exits once its
// next entry lies past the list.
// The header and descriptors come as read-only pointers, so they load through the scalar
// cache into scalar registers.
// On the layouts with a tuned batch shape (the compressed one) the default grid is one block per
// entry, up to 64 per compute unit: the hardware's dispatch then balances the list.  256 requests
// of 754M rows in all: 1.03 ms (6.87 TB/s, 64 blocks per compute unit x 192 rows per lane), 1.08 ms
// striding with 8 blocks per compute unit.  Batches of the other layouts stride with as many blocks
// as are resident.
// The descriptors and results used to travel through a graph of a copy, the kernel and a
// fold, rebuilt for every power of two of requests: 16 requests of 10,000 rows 50 -> 21 us.
template <int L, int P>
__global__ void __launch_bounds__(kBatchBlock)
batch_scan(const BatchHeader* __restrict__ hdr, const BatchDesc* __restrict__ descs,
           const uint32_t* __restrict__ first, BatchControl* control, q1_device_aggregates* results, BatchDone* done) {
  extern __shared__ uint64_t lds[];
  const uint32_t n = hdr->n, tpt = hdr->tiles_per_thread, total = hdr->total_blocks;
  if (blockIdx.x == 0 && thread_index() == 0)
    __hip_atomic_store(&control->clock_begin, (uint64_t)wall_clock64(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  uint32_t v = blockIdx.x;
  if (v >= total) return;
  uint32_t r = (uint32_t)__builtin_amdgcn_readfirstlane((int)find_request(first, n, v));
  for (;;) {
    const BatchDesc d = descs[r];
    const uint32_t e = v - d.first_block, t = e & d.table_mask;
    ScanArgs a;
    a.cols = load_global_columns(&descs[r].cols);
    a.row_begin = d.row_begin;
    a.row_end = d.row_end;
    a.cutoff_day = d.cutoff_day;
    scan_block<L, P, kBatchBlock>(a, e, tpt, nullptr, lds, &d.tables[t].sums);
    if (thread_index() < 64) {
      const uint32_t lane = thread_index() & 63;
      uint64_t sum;
      if (finish_tables(d.tables, t, blocks_sharing(d.blocks, e, d.table_mask), d.table_mask + 1, sum)) {
        if (lane < 48) store_host(reinterpret_cast<uint64_t*>(results + r) + lane, sum);
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        uint32_t last = 0;
        if (lane == 0) last = atomicAdd(&control->requests_done, 1u) == hdr->with_rows - 1;
        if (last) {
          atomicExch(&control->requests_done, 0u);
          store_host(&done->clock_begin, atomicExch((unsigned long long*)&control->clock_begin, 0ull));
          store_host(&done->clock_end, wall_clock64());
          __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
          store_host(&done->sequence, hdr->sequence);
        }
      }
    }
    v += gridDim.x;
    if (v >= total) return;
    if (v - d.first_block >= d.blocks) r = (uint32_t)__builtin_amdgcn_readfirstlane((int)next_request(first, n, r, v));
    // Orders this entry's reads of the merge scratch before the next entry's writes.
    __syncthreads();
  }
}

// ------------------------------------------------------------------------------------
// Dispatch templates: the kernel of a (layout, placement, block size).
// ------------------------------------------------------------------------------------
template <int L, int B>
constexpr FastFn fast_fn_b(int p) {
  return p == Q1_PLACE_IN_REGISTERS ? scan_fast<L, Q1_PLACE_IN_REGISTERS, B>
       : p == Q1_PLACE_IN_REGISTERS_PER_THREAD ? scan_fast<L, Q1_PLACE_IN_REGISTERS_PER_THREAD, B>
       : p == Q1_PLACE_LOCAL_MEM ? scan_fast<L, Q1_PLACE_LOCAL_MEM, B>
       : p == Q1_PLACE_PER_THREAD_SHARED_MEM ? scan_fast<L, Q1_PLACE_PER_THREAD_SHARED_MEM, B>
       : p == kPlaceSharedNarrow ? scan_fast<L, kPlaceSharedNarrow, B>
       : p == kPlaceSharedPacked ? scan_fast<L, kPlaceSharedPacked, B>
       : scan_fast<L, Q1_PLACE_GLOBAL, B>;
}

template <int L>
FastFn fast_fn(int p, uint32_t threads) {
  return threads == 64 ? fast_fn_b<L, 64>(p) : threads == 128 ? fast_fn_b<L, 128>(p) : fast_fn_b<L, 256>(p);
}

// The direct kernel of the LDS table for at most 256 rows per lane.
template <int L>
GenFn direct_fn(uint32_t threads) {
  constexpr bool units = L == Q1_LAYOUT_COMPRESSED || L == Q1_LAYOUT_COMPRESSED_PUSHDOWN;
  constexpr int P = units ? kPlaceSharedPacked : kPlaceSharedNarrow;
  return threads == 64 ? scan_direct<L, P, 64> : threads == 128 ? scan_direct<L, P, 128> : scan_direct<L, P, 256>;
}

template <int L>
GenFn any_fn(uint32_t threads) {
  return threads == 64 ? scan_any<L, 64> : threads == 128 ? scan_any<L, 128> : scan_any<L, 256>;
}
template <int L>
uint32_t any_lds(uint32_t threads) {
  return AnyOf<L, 64>::A::lds_bytes(threads) + threads / 64 * kNumGroups * NA * 8;
}

// The batched kernel's variants: the shared placement runs the narrow per-lane table (the
// packed one for the compressed layouts), as launch_scan does for at most 256 rows per lane.
template <int L>
void* batch_fn(q1_placement p) {
  constexpr bool units = L == Q1_LAYOUT_COMPRESSED || L == Q1_LAYOUT_COMPRESSED_PUSHDOWN;
  if (p != Q1_PLACE_PER_THREAD_SHARED_MEM) return (void*)batch_scan<L, Q1_PLACE_IN_REGISTERS>;
  return units ? (void*)batch_scan<L, kPlaceSharedPacked> : (void*)batch_scan<L, kPlaceSharedNarrow>;
}

}  // namespace

// Kernel entry points of one layout, defined by that layout's translation unit.
#define Q1_DECLARE_LAYOUT_KERNELS(NAME)                  \
  FastFn fast_kernel_##NAME(int placement, uint32_t threads); \
  GenFn direct_kernel_##NAME(uint32_t threads);          \
  GenFn any_kernel_##NAME(uint32_t threads);             \
  uint32_t any_kernel_lds_##NAME(uint32_t threads);      \
  void* batch_kernel_##NAME(q1_placement placement);
Q1_DECLARE_LAYOUT_KERNELS(reference)
Q1_DECLARE_LAYOUT_KERNELS(uncompressed)
Q1_DECLARE_LAYOUT_KERNELS(compressed)
Q1_DECLARE_LAYOUT_KERNELS(pushdown)

#define Q1_DEFINE_LAYOUT_KERNELS(L, NAME)                                                          \
  FastFn fast_kernel_##NAME(int placement, uint32_t threads) { return fast_fn<L>(placement, threads); } \
  GenFn direct_kernel_##NAME(uint32_t threads) { return direct_fn<L>(threads); }                   \
  GenFn any_kernel_##NAME(uint32_t threads) { return any_fn<L>(threads); }                         \
  uint32_t any_kernel_lds_##NAME(uint32_t threads) { return any_lds<L>(threads); }                 \
  void* batch_kernel_##NAME(q1_placement placement) { return batch_fn<L>(placement); }

}  // namespace q1

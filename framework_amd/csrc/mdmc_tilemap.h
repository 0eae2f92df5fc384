// Workgroup -> tile map of the plane-tile classify (k_classify_pt), the chunk
// tickets of the persistent emit (k_emit), the scan's forms and reads, and the emit's
// address arithmetic.
//
// Workgroups are dispatched round-robin over the 8 XCDs (block b runs on XCD
// b % 8).  A column is one x-tile of one row block; columns form groups of B.
// In every plane block XCD x takes groups x, x+8, x+16, ... and walks them in
// memory order, plane block after plane block; the groups left over when
// their count is not a multiple of 8 are dealt out over the XCDs eight plane
// blocks at a time.  The launch has 8 * B * ceil(NKB * groups / 8) blocks.
//
// Plain C++ (no HIP types) so that a host test can check it.
#ifndef MDMC_TILEMAP_H
#define MDMC_TILEMAP_H

#include <cstdint>

#if defined(__HIPCC__)
#define MDMC_HD __host__ __device__
#else
#define MDMC_HD
#endif

namespace mdmc {

// Tile of block b (XCD b % 8, b / 8-th of that XCD's walk); blocks past the
// XCD's share get plane block NKB, a tile outside the grid.
struct PtTile {
  uint32_t xt, rb, kb;
};
MDMC_HD inline PtTile pt_tile_of(uint32_t b, uint32_t XT, uint32_t NRB, uint32_t NKB, uint32_t B) {
  const uint32_t x = b & 7u, s = b >> 3;
  const uint32_t cols = XT * NRB;
  const uint32_t ng = (cols + B - 1u) / B;  // column groups
  const uint32_t q = ng >> 3, r = ng & 7u;  // groups per XCD per plane block; left over
  const uint32_t gs = s / B, w = s - gs * B;  // group tile of the walk, column in the group
  const uint32_t per = 8u * q + r;          // group tiles per XCD per 8 plane blocks
  const uint32_t S = gs / per, o = gs - S * per;
  PtTile t{0u, 0u, NKB};
  if ((uint64_t)S * 8u >= NKB) return t;
  const uint32_t nk = NKB - 8u * S < 8u ? NKB - 8u * S : 8u;
  uint32_t kb, g;
  if (o < nk * q) {  // the XCD's own groups, plane block by plane block
    kb = 8u * S + o / q;
    g = (o % q) * 8u + x;
  } else {  // left-over group tiles e = x, x + 8, ... of these plane blocks
    const uint32_t e = x + 8u * (o - nk * q);
    if (e >= nk * r) return t;
    kb = 8u * S + e / r;
    g = 8u * q + e % r;
  }
  const uint32_t col = g * B + w;
  if (col >= cols) return t;
  t.xt = col % XT;
  t.rb = col / XT;
  t.kb = kb;
  return t;
}

// Chunk tickets of the persistent emit (k_emit).  The workgroups b with
// b % 8 == x (XCD x) take the contiguous chunk range [x n / 8, (x + 1) n / 8)
// in tickets of one chunk per wave: ticket t is chunks [lo + W t, lo + W t +
// W) for W waves per workgroup.  Workgroup b's first ticket is its slot b / 8
// (no atomic), its later ones are slots + c for the values c of counter x,
// taken only when the first tickets do not already cover the range
// (dynamic).  A workgroup stops at the first ticket that starts at or past
// hi.  G, the number of workgroups, is a multiple of 8.
struct EmitTickets {
  uint32_t lo, hi, slots;
  bool dynamic;
};
MDMC_HD inline EmitTickets emit_tickets(uint32_t n, uint32_t x, uint32_t G, uint32_t W) {
  EmitTickets e;
  e.lo = (uint32_t)((uint64_t)n * x / 8u);
  e.hi = (uint32_t)((uint64_t)n * (x + 1u) / 8u);
  e.slots = G >> 3;
  e.dynamic = e.lo + (uint64_t)e.slots * W < e.hi;
  return e;
}
// first chunk of ticket t
MDMC_HD inline uint64_t emit_ticket_chunk(const EmitTickets &e, uint64_t t, uint32_t W) { return e.lo + t * W; }

// Which scan serves a call of nsegs segments (the kernels' comments have the
// measurements behind the lines): whole cell planes of plane_segs segments and
// plane_parts sums, where a workgroup holds a plane and all sums are few
// (plane_segs = 0: no planes, as in a batch); sums per scan tile; look-back.
enum class ScanForm { lookback, planes, tiles };
constexpr uint32_t kScanTileSegs = 2048;
constexpr uint32_t kPlaneScanParts = 1u << 15;
constexpr uint32_t kTileScanMin = 96, kTileScanMax = 4096;
inline ScanForm scan_form(uint64_t nsegs, uint64_t plane_segs, uint64_t plane_parts) {
  if (plane_segs != 0 && plane_segs <= kScanTileSegs && plane_parts * (nsegs / plane_segs) <= kPlaneScanParts)
    return ScanForm::planes;
  const uint64_t tiles = (nsegs + kScanTileSegs - 1u) / kScanTileSegs;
  return tiles >= kTileScanMin && tiles <= kTileScanMax ? ScanForm::tiles : ScanForm::lookback;
}

// Whether the scan's workgroups fill the coordinate tables on the side: not
// where the rows are so long that its threads get more than 64 of the ncoord
// entries each.  A launch of its own costs an extraction 3 to 4 us, 64 entries
// about as much (20,000 x 9 x 9 points, 39 a thread: 14 us, with the launch
// 17; 100,000 x 5 x 5, 195 a thread: 25 and 17; 1,000,000 x 2 x 2,
// 3,906 a thread: 322 and 17).
inline bool scan_fills_coords(uint64_t ncoord, uint64_t scan_threads) { return ncoord <= 64u * scan_threads; }

// A scan thread's pairs of segment totals: it reads entries scan_pair(base, i,
// end) and the one after, where its segments base + 2 i and the next are below
// end, the end of its workgroup's segments.  Past that it reads the last one
// and `end` itself, the next workgroup's first or a padding entry: there is at
// least one, and behind the padding lies what other workgroups write.
MDMC_HD inline uint32_t scan_pair(uint32_t base, uint32_t i, uint32_t end) {
  const uint32_t at = base + 2u * i;
  return at < end ? at : end - 1u;
}

// Exact division of 32-bit numbers by a divisor known on the host: a multiply
// and two shifts (round-up multiplier 2^32 (2^l - d) / d + 1, l = ceil(log2 d);
// Granlund and Montgomery, "Division by invariant integers using
// multiplication").
struct FastDiv {
  uint32_t mul, sh1, sh2;
};
inline FastDiv fast_div(uint32_t d) {
  uint32_t l = 0;
  while (l < 32u && (1ull << l) < d) ++l;
  return FastDiv{(uint32_t)(((1ull << 32) * ((1ull << l) - d)) / d + 1u), l < 1u ? l : 1u, l > 1u ? l - 1u : 0u};
}
MDMC_HD inline uint32_t div_by(uint32_t n, FastDiv d) {
  const uint32_t t = (uint32_t)(((uint64_t)d.mul * n) >> 32);
  return (t + ((n - t) >> d.sh1)) >> d.sh2;
}

// Segments from a wave's first one on whose records, group maps and field rows
// lie within 2 GB of that segment's (32-bit lane offsets from its bases): a
// record is 4 bytes, and a segment lies at most 2 * (distance / XT + 1) point
// rows further on.
inline uint32_t emit_span(uint32_t X, uint32_t XT, uint32_t cap) {
  const uint64_t rec = (1ull << 31) / (4ull * cap) - 1u, rows = (1ull << 31) / (4ull * X);
  const uint64_t fld = rows > 6u ? (uint64_t)XT * ((rows - 4u) / 2u) : 0u;
  return (uint32_t)(rec < fld ? rec : fld);
}

}  // namespace mdmc

#endif

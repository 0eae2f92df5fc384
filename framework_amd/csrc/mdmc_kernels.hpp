// Dual Marching Cubes kernels for gfx950 (MI355X).
//
// Pipeline for one volume (stream-ordered launches, no host sync):
//
//   k_classify_pt  dense pass over the field in plane tiles (7 cell rows x
//               one x-tile x 1-4 cell planes per 256-thread workgroup): point
//               rows staged in LDS as sign bits, uniform 256-cell chunks
//               skipped with one ballot, active cells found by bit operations
//               and listed in LDS; listed cells get their 2B/3B table variant,
//               vertex and quad counts, a DPP-scan rank and a 32-bit record in
//               their segment's slot range (segment = one cell row of one
//               x-tile in one plane), plus a per-16-cell group map (active
//               mask, first rank).  Workgroups map to tiles XCD by XCD (mdmc_tilemap.h).
//               k_classify is the z-marching form for any row length.
//   k_scan_planes, k_scan_tiles, k_scan   scan over the segment totals:
//               vertex/quad bases per segment, the non-empty segment list and
//               where each 64-cell chunk starts.  From sums per plane that the
//               classify left, from sums per 2048 segments, or (the smallest
//               batches, the largest volumes, the z-marching classify's small
//               grids) single-pass with decoupled look-back.
//   k_emit      one wave per chunk of 64 active cells: edge crossing points
//               in the owner's orientation, dual vertices (FP32, reference
//               operation order) and quads; ring cells are found through the
//               group map in O(1).
//   k_smooth, k_reaverage   optional smoothing iterations over the mesh.
//
// Batched forms (k_classify_batch, k_batch_counts, k_emit_batch) run the
// same per-tile and per-cell code over many volumes; k_slab_info reports an
// out-of-core slab in one record; k_field_* generate the synthetic benchmark
// fields.
//
// Reference semantics: DMC_CUDA/DMC_CUDA/src/dmc.cu:1018-2208 (dmc::run_dmc).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "mdmc_tilemap.h"
#include "mdmc_wave.h"

#pragma clang fp contract(off)

namespace mdmc {

constexpr int kWave = 64;
constexpr uint32_t kStatusVertexOverflow = 1, kStatusQuadOverflow = 2, kStatusLookup = 4,
                   kStatusScanTimeout = 8, kStatusInternal = 16, kStatusIndexRange = 32;

// Case tables in constant memory (uploaded by mdmc_setup):
//   c_label[v][cfg]   12 nibbles, edge e -> iso-vertex label or 0xF
//   c_cfg_info[cfg]   bits 0-2 NV variant 0, 3-5 NV variant 1, 6 = 2B/3B,
//                     7-9 check direction (POS_X=0 .. NEG_Z=5)
__constant__ uint64_t c_label[2][256];
__constant__ uint16_t c_cfg_info[256];
// c_cfg_count[cfg]: bits 0-3 NV variant 0 + bipolar owned edges, 4-7 the same
// for variant 1, 8-10 bipolar owned edges 6/9/10, 11 = 2B/3B, 12-14 check dir.
__constant__ uint16_t c_cfg_count[256];

struct Totals {
  uint32_t num_active, num_vertices, num_quads, num_nonempty;
  uint32_t num_chunks, pad0, pad1, pad2;
};

struct FieldDesc {
  const float *f;
  uint32_t X, Y, Z;     // points
  uint32_t cx, cy, cz;  // cells
  float iso;
};

// Record of an active cell (32 bits):
//   bits  0-9   x offset inside its x-tile
//   bits 10-17  configuration
//   bit  18     uses the variant-1 table (2B/3B correction)
//   bits 19-31  first vertex, relative to the segment
// Its first quad, relative to the segment, is kept apart (16 bits): only the
// cell's own emit reads it, while a record is read by up to seven cells.
__device__ __forceinline__ uint32_t make_record(uint32_t xl, uint32_t cfg, uint32_t lut2, uint32_t lvb) {
  return xl | (cfg << 10) | (lut2 << 18) | (lvb << 19);
}
__device__ __forceinline__ uint32_t rec_x(uint32_t r) { return r & 0x3FFu; }
__device__ __forceinline__ uint32_t rec_cfg(uint32_t r) { return (r >> 10) & 0xFFu; }
__device__ __forceinline__ uint32_t rec_lut2(uint32_t r) { return (r >> 18) & 1u; }
__device__ __forceinline__ uint32_t rec_lvb(uint32_t r) { return r >> 19; }

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

// Index of the calling wave in its workgroup, as a wave-uniform (scalar)
// value so that per-wave bookkeeping compiles to scalar instructions.
__device__ __forceinline__ uint32_t wave_id() {
  return __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
}

// The wave passes this point together, with its LDS accesses before it done
// before those after it, for all lanes (mdmc_wave.h).
struct WaveOrder {
  __device__ __forceinline__ void operator()() const {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
  }
};

// Workgroups are dispatched round-robin over the 8 XCDs (block b -> XCD b%8).
// Remap so that each XCD works on a contiguous range of tiles: neighbouring
// tiles (which share halo rows) then hit the same L2.
__device__ __forceinline__ uint32_t xcd_remap(uint32_t b, uint32_t n) {
  uint32_t q = n >> 3, r = n & 7, x = b & 7;
  return x * q + min(x, r) + (b >> 3);
}

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
  const int lane = (int)lane_id();
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    uint32_t t = __shfl_up(v, d, kWave);
    if (lane >= d) v += t;
  }
  return v;
}

// DPP controls (GFX9 encoding).
constexpr int kDppRowShr = 0x110;  // + n: lane i reads lane i-n of its 16-lane row
constexpr int kDppWaveShl1 = 0x130;  // lane i reads lane i+1 across the wave
constexpr int kDppRowBcast15 = 0x142;
constexpr int kDppRowBcast31 = 0x143;

// Value of lane+1 (0 in lane 63).
__device__ __forceinline__ uint32_t lane_next(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, kDppWaveShl1, 0xF, 0xF, true);
}

// Inclusive prefix sum over the 64 lanes with DPP (no LDS traffic).
__device__ __forceinline__ uint32_t wave_incl_scan_dpp(uint32_t x) {
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kDppRowShr + 1, 0xF, 0xF, true);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kDppRowShr + 2, 0xF, 0xF, true);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kDppRowShr + 4, 0xF, 0xF, true);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kDppRowShr + 8, 0xF, 0xF, true);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kDppRowBcast15, 0xA, 0xF, false);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kDppRowBcast31, 0xC, 0xF, false);
  return x;
}

// The same over each 16 or 32 lanes.
template <int LW>
__device__ __forceinline__ uint32_t row_incl_scan_dpp(uint32_t x) {
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kDppRowShr + 1, 0xF, 0xF, true);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kDppRowShr + 2, 0xF, 0xF, true);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kDppRowShr + 4, 0xF, 0xF, true);
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kDppRowShr + 8, 0xF, 0xF, true);
  if constexpr (LW >= 32) x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, kDppRowBcast15, 0xA, 0xF, false);
  return x;
}

__device__ __forceinline__ uint32_t mbcnt64(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// Configuration of cell (x, y, z) read straight from the field (used for the
// rare 2B/3B neighbour checks whose neighbour lies outside the tile window).
__device__ __forceinline__ uint32_t cell_cfg_global(const FieldDesc &g, uint32_t x, uint32_t y,
                                                    uint32_t z) {
  const size_t sy = g.X, sz = (size_t)g.X * g.Y;
  const float *p = g.f + (size_t)z * sz + (size_t)y * sy + x;
  const float iso = g.iso;
  uint32_t c = 0;
  c |= (uint32_t)(p[0] < iso);
  c |= (uint32_t)(p[1] < iso) << 1;
  c |= (uint32_t)(p[sy + 1] < iso) << 2;
  c |= (uint32_t)(p[sy] < iso) << 3;
  c |= (uint32_t)(p[sz] < iso) << 4;
  c |= (uint32_t)(p[sz + 1] < iso) << 5;
  c |= (uint32_t)(p[sz + sy + 1] < iso) << 6;
  c |= (uint32_t)(p[sz + sy] < iso) << 7;
  return c;
}

// 2B/3B correction (dmc.cu:1345-1371): a cell whose configuration is 2B/3B
// uses the variant-1 table when its in-grid neighbour across the listed face
// is also 2B/3B.
__device__ __forceinline__ uint32_t use_variant1(const FieldDesc &g, const uint16_t *info_tab,
                                                 uint32_t info, uint32_t x, uint32_t y,
                                                 uint32_t z) {
  if (!(info & 64u)) return 0;
  uint32_t dir = (info >> 7) & 7u;
  int nx = (int)x, ny = (int)y, nz = (int)z;
  switch (dir) {
    case 0: nx += 1; break;
    case 1: nx -= 1; break;
    case 2: ny += 1; break;
    case 3: ny -= 1; break;
    case 4: nz += 1; break;
    default: nz -= 1; break;
  }
  if (nx < 0 || ny < 0 || nz < 0 || nx >= (int)g.cx || ny >= (int)g.cy || nz >= (int)g.cz) return 0;
  uint32_t ncfg = cell_cfg_global(g, (uint32_t)nx, (uint32_t)ny, (uint32_t)nz);
  return (info_tab[ncfg] >> 6) & 1u;
}

// The scan's ticket word opens a region of the scratch of kTicketBytes: word 0
// is the scan's tile ticket, and word kEmitCtr * (x + 1) the emit's chunk
// ticket counter of XCD x (k_emit), each on a 256-byte line of its own (the
// atomics on one line serialise).  The classify zeroes all nine.
constexpr uint32_t kEmitCtr = 64;
constexpr uint32_t kTicketBytes = 9 * kEmitCtr * 4;

__device__ __forceinline__ void zero_tickets(uint32_t *t, uint32_t tid) {
  if (tid < 9u) t[tid * kEmitCtr] = 0u;
}

struct ClassifyArgs {
  FieldDesc g;
  uint32_t XT, NRB, NKC, Kc;
  uint2 *seg_counts;      // per segment: {nact | nquad << 16, nvert}
  uint32_t *slots;        // per segment: 64*W record slots
  uint16_t *slot_q;       // per record slot: the cell's first quad
  uint32_t *gmap;         // per segment and 16-cell group: active mask | rank of the group's
                          // first active cell << 16; written for non-empty groups
  unsigned long long *scan_state;  // zeroed here for k_scan
  uint32_t scan_state_words;
  uint2 *part;            // per plane, row block and x-tile: the sums of its segments' totals
                          // {active | quads << 16, vertices | non-empty << 16} (null: not wanted)
  uint2 *seg_pad;         // segment totals past the last segment, up to a whole scan tile
  uint32_t seg_pad_n;     // (zeroed here, read by the scan)
  uint32_t *scan_ticket;  // the ticket region, zeroed here
  Totals *totals;
  uint32_t *counts_out;   // user mdmc_counts (4 words), zeroed here
};

// One wave per tile; see the file header.
template <int W, int R>
__global__ __launch_bounds__(64) void k_classify(ClassifyArgs a) {
  static_assert(R >= 1 && R <= 15, "rows per tile must fit the 16-bit plane fields");
  static_assert(W >= 1 && W <= 16, "x-tile is at most 1024 cells");
  __shared__ uint16_t s_info[256];
  const uint32_t lane = lane_id();
  for (uint32_t i = lane; i < 256; i += kWave) s_info[i] = c_cfg_info[i];
  if (blockIdx.x == 0) {
    for (uint32_t i = lane; i < a.scan_state_words; i += kWave) a.scan_state[i] = 0ull;
    for (uint32_t i = lane; i < a.seg_pad_n; i += kWave) a.seg_pad[i] = make_uint2(0u, 0u);
    if (lane < 8) reinterpret_cast<uint32_t *>(a.totals)[lane] = 0u;
    zero_tickets(a.scan_ticket, lane);
    if (a.counts_out != nullptr && lane < 4) a.counts_out[lane] = 0u;
  }
  __syncthreads();

  const FieldDesc g = a.g;
  const float iso = g.iso;
  constexpr uint32_t CAP = 64u * W;
  const uint32_t tile = xcd_remap(blockIdx.x, gridDim.x);
  const uint32_t xt = tile % a.XT;
  const uint32_t rest = tile / a.XT;
  const uint32_t rb = rest % a.NRB;
  const uint32_t kc = rest / a.NRB;
  const uint32_t x0 = xt * CAP;
  const uint32_t j0 = rb * R;
  const uint32_t k0 = kc * a.Kc;
  const uint32_t k1 = min(k0 + a.Kc, g.cz);
  if (k0 >= g.cz) return;
  const size_t plane = (size_t)g.X * g.Y;
  const bool has_extra = x0 + CAP < g.X;  // first point of the next x-tile
  const float qnan = __int_as_float(0x7FC00000);

  float vals[R + 1][W];
  float vext[R + 1];

  auto load_plane = [&](uint32_t z) {
#pragma unroll
    for (int r = 0; r <= R; ++r) {
      const uint32_t y = j0 + r;
      const bool row_ok = (z < g.Z) && (y < g.Y);
      const float *rowp = g.f + (size_t)z * plane + (size_t)y * g.X;
#pragma unroll
      for (int c = 0; c < W; ++c) {
        const uint32_t x = x0 + 64u * c + lane;
        vals[r][c] = (row_ok && x < g.X) ? rowp[x] : qnan;
      }
      vext[r] = (row_ok && has_extra) ? rowp[x0 + CAP] : qnan;
    }
  };
  auto plane_bits = [&](int c) {
    uint32_t b = 0;
#pragma unroll
    for (int r = 0; r <= R; ++r) b |= (uint32_t)(vals[r][c] < iso) << r;
    return b;
  };
  auto ext_bits = [&]() {
    uint32_t b = 0;
#pragma unroll
    for (int r = 0; r <= R; ++r) b |= (uint32_t)(vext[r] < iso) << r;
    return b;
  };

  uint32_t B[W];
  uint32_t E;
  load_plane(k0);
#pragma unroll
  for (int c = 0; c < W; ++c) B[c] = plane_bits(c) << 16;
  E = ext_bits() << 16;
  load_plane(k0 + 1);

  constexpr uint32_t rowmask = (1u << (R + 1)) - 1u;
  constexpr uint32_t fullmask = rowmask | (rowmask << 16);

  for (uint32_t k = k0; k < k1; ++k) {
#pragma unroll
    for (int c = 0; c < W; ++c) B[c] = (B[c] >> 16) | (plane_bits(c) << 16);
    E = (E >> 16) | (ext_bits() << 16);
    if (k + 1 < k1) load_plane(k + 2);  // prefetch the plane the next step needs

    // Neighbour columns (lane+1; lane 63 takes the next chunk's lane 0) and
    // the chunks that are not uniformly in or out over all rows.
    uint32_t N[W];
    uint32_t live = 0;
#pragma unroll
    for (int c = 0; c < W; ++c) {
      const uint32_t own = B[c];
      uint32_t nb = __shfl_down(own, 1, kWave);
      const uint32_t nxt = (c + 1 < W) ? (uint32_t)__shfl(B[(c + 1 < W) ? c + 1 : c], 0, kWave) : E;
      if (lane == kWave - 1) nb = nxt;
      N[c] = nb;
      const uint32_t uo = own & fullmask, un = nb & fullmask;
      const bool all_out = (uo | un) == 0u;
      const bool all_in = (uo & un) == fullmask;
      if (__ballot(!all_out) != 0ull && __ballot(!all_in) != 0ull) live |= 1u << c;
    }

#pragma unroll 1
    for (int r = 0; r < R; ++r) {
      const uint32_t y = j0 + r;
      if (y >= g.cy) break;
      uint32_t cnt_a = 0, cnt_v = 0, cnt_q = 0;
      const uint32_t seg = xt + a.XT * (y + g.cy * k);
#pragma unroll
      for (int c = 0; c < W; ++c) {
        if (!((live >> c) & 1u)) continue;
        const uint32_t own = B[c], nb = N[c];
        const uint32_t x = x0 + 64u * c + lane;
        const uint32_t t = ((own >> r) & 0x30003u) | (((nb >> r) & 0x30003u) << 2);
        const uint32_t key = (t & 0xFu) | ((t >> 12) & 0xF0u);
        const uint32_t cfg = (key & 0x11u) | ((key >> 1) & 0x66u) | ((key << 2) & 0x88u);
        const bool active = (x < g.cx) && (cfg != 0u) && (cfg != 0xFFu);
        const uint64_t bal = __ballot(active);
        if (bal == 0ull) continue;
        if (lane < 4u) {
          const uint32_t m16 = (uint32_t)(bal >> (16u * lane)) & 0xFFFFu;
          const uint32_t before = (uint32_t)__popcll(bal & ((1ull << (16u * lane)) - 1ull));
          if (m16) a.gmap[(size_t)seg * (4u * W) + 4u * c + lane] = m16 | ((cnt_a + before) << 16);
        }
        uint32_t nv = 0, nq = 0, lut2 = 0;
        if (active) {
          const uint32_t info = s_info[cfg];
          lut2 = use_variant1(g, s_info, info, x, y, k);
          const uint32_t b6 = ((cfg >> 2) ^ (cfg >> 6)) & 1u;
          const uint32_t b9 = ((cfg >> 5) ^ (cfg >> 6)) & 1u;
          const uint32_t b10 = ((cfg >> 7) ^ (cfg >> 6)) & 1u;
          nv = (lut2 ? ((info >> 3) & 7u) : (info & 7u)) + b6 + b9 + b10;
          const bool xin = x + 1 < g.cx, yin = y + 1 < g.cy, zin = k + 1 < g.cz;
          nq = (b6 & (uint32_t)(xin && yin)) + (b9 & (uint32_t)(xin && zin)) +
               (b10 & (uint32_t)(yin && zin));
        }
        const uint32_t packed = nv | (nq << 16);
        const uint32_t incl = wave_incl_scan(packed);
        const uint32_t excl = incl - packed;
        const uint32_t tot = __shfl(incl, kWave - 1, kWave);
        if (active) {
          const uint32_t rank = cnt_a + mbcnt64(bal);
          const uint32_t lvb = cnt_v + (excl & 0xFFFFu);
          const uint32_t lqb = cnt_q + (excl >> 16);
          a.slots[(size_t)seg * CAP + rank] = make_record(x - x0, cfg, lut2, lvb);
          a.slot_q[(size_t)seg * CAP + rank] = (uint16_t)lqb;
        }
        cnt_a += (uint32_t)__popcll(bal);
        cnt_v += tot & 0xFFFFu;
        cnt_q += tot >> 16;
      }
      if (lane == 0) a.seg_counts[seg] = make_uint2(cnt_a | (cnt_q << 16), cnt_v);
    }
  }
}

// Plane-tile classify: the main kernel, for rows of any length.  A 256-thread
// workgroup owns one tile = R cell rows x one x-tile
// (256*W4 cells) x KP cell planes.  Workgroups are dispatched round-robin over
// the 8 XCDs (block b runs on XCD b % 8), each with its own L2.  A column is
// one x-tile of one row block; columns form groups of B (the band option).
// In every plane block, XCD x takes groups x, x+8, x+16, ... and walks them
// in memory order, plane block after plane block, so the point plane shared
// by two plane blocks is read twice by the same XCD a few tiles apart and
// comes from its L2, and all XCDs stream through the same few planes at a
// time (a small working set for the address translation caches).  The groups
// left over when their count is not a multiple of 8 are dealt out over the
// XCDs eight plane blocks at a time, so every XCD gets the same number of
// tiles (within one group) and none of them finishes late.
//
// Phase 1: wave w converts point rows r = w, w+4, ... (R+1 of them, so every
// wave has the same share) of all KP+1 point planes.  A lane owns 4
// consecutive points of a 256-point chunk (one 16-byte load from a uniform
// row address plus a fixed lane offset); it packs their sign bits and the
// first bit of lane l+1 into a 5-bit value v5, pairs the values of planes
// p and p+1 into 16 bits and stores that pair into the LDS word of cell row
// r (low half) and of cell row r-1 (high half) of cell plane p:
//   byte 0: point row j,   plane k     byte 1: point row j,   plane k+1
//   byte 2: point row j+1, plane k     byte 3: point row j+1, plane k+1
// (the LDS has one padding row above and below, so every store is
// unconditional and every address is the wave's base plus a constant).
// Phase 2: each wave takes cell rows w, w+4, ...; one LDS read gives all 20
// corner bits of a lane's 4 cells.  The active ones go to a list, and the list
// is classified a cell per lane (PtList): for a cell, t = (w >> q) &
// 0x03030303 holds the corner pairs (p0,p1), (p4,p5), (p3,p2), (p7,p6) in its
// bytes and (t * 0x41041) >> 18 gathers them into an 8-bit key, which indexes
// a table of configuration and counts.
constexpr int kPtThreads = 256;

// key bits p0 p1 p4 p5 p3 p2 p7 p6 -> configuration bits p0..p7
__host__ __device__ constexpr uint32_t key_to_cfg(uint32_t key) {
  return (key & 0x03u) | ((key >> 3) & 0x04u) | ((key >> 1) & 0x08u) | ((key << 2) & 0x30u) |
         ((key & 0x40u) << 1) | ((key & 0x80u) >> 1);
}

struct PtArgs {
  ClassifyArgs c;
  uint32_t B;    // columns per group
  uint32_t NKB;  // plane blocks
  uint32_t NRB;  // row blocks
  // The last x-tiles, where they are narrow, are in the blocks from tail_block
  // on (a multiple of 8) as columns of their own.  Among the others' columns
  // they fell to the same XCDs throughout: with two x-tiles four XCDs got all
  // the full ones (603x487x399: 129 us, 107 apart).
  uint32_t tail_block;
  uint32_t NKBT;  // their plane blocks
  uint32_t tall;  // of pt_tall planes
};

// Cell rows per plane tile (R + 1 point rows, 2 per wave) and cell planes per
// tile (KP + 1 point planes), chosen so that all loads of a wave fit in
// registers: (R+1)/4 * (KP+1) * W4 float4 per lane.
constexpr uint32_t pt_rows(uint32_t) { return 7u; }
constexpr uint32_t pt_planes(uint32_t W4) { return W4 >= 4 ? 1u : (W4 == 2 ? 2u : 4u); }

// Parts of a row's last x-tile, by its points (see PtWide): full chunks << 8 |
// lanes of the narrow part.  kPtTailFull: the x-tile's full mapping (also
// where the narrow part's 32-bit lane offsets do not reach).  kPtTailTiny:
// rows of less than 4 points, which a 16-byte load would leave.
constexpr uint32_t kPtTailFull = 0u, kPtTailTiny = 1u, kPtTail16 = 16u, kPtTail32 = 32u, kPtTail64 = 64u,
                   kPtTail256_16 = 256u + 16u, kPtTail256_32 = 256u + 32u;
__host__ __device__ constexpr uint32_t pt_tail(uint32_t X, uint32_t XT, uint32_t cap) {
  const uint32_t np = X - (XT - 1u) * cap;  // points of the last x-tile
  if (X < 4u) return kPtTailTiny;
  if (X > (1u << 24) || cap > 512u) return kPtTailFull;
  if (np <= 64u) return kPtTail16;
  if (np <= 128u) return kPtTail32;
  if (cap == 256u) return kPtTailFull;
  return np <= 256u ? kPtTail64 : np <= 320u ? kPtTail256_16 : np <= 384u ? kPtTail256_32 : kPtTailFull;
}

// Cell planes of a narrow last x-tile's workgroup where it takes more than KP of
// them (a tall tile): as many as fill the LDS words and registers of a full
// tile.  A narrow tile of KP planes holds a quarter of a full one's points or
// less, but its loads, barriers and list rounds follow each other just as
// slowly, and it keeps its place on the CU for half as long (256 volumes of 32
// to 256 points a side: classify 701 us, with tall tiles 584).
__host__ __device__ constexpr uint32_t pt_tall(uint32_t tail, uint32_t W4, uint32_t R, uint32_t KP) {
  if (R != 7u || (tail != kPtTail16 && tail != kPtTail32 && tail != kPtTail64)) return KP;
  // (tail: its lanes, and LDS words, per row and plane; a full tile has 64 W4)
  const uint32_t words = KP * W4 * 64u / tail, most = words < 8u ? words : 8u;
  return most >= KP ? most / KP * KP : KP;
}
// Narrow tiles are tall where rows have full x-tiles as well (in a batch, whose
// tiles are in memory order, every pt_tall / KP-th plane block's narrow tile
// works and the others leave: kTallSome), and where a row is one narrow tile
// if enough tiles remain to fill the chip twice (kTallAll).  Where the line lies
// matters little: rows of 64 points, classify with and without tall tiles, 16.3
// and 17.3 us at 5,300 tiles, 20.7 and 21.6 at 8,400, 30.2 and 37.8 at 18,500;
// rows of 128 points 27.5 and 27.0 at 7,000, 30.5 and 29.2 at 8,400, 51.3 and
// 53.8 at 18,500; 24 volumes of 32 to 128 points (4,000) 31.0 both.
constexpr uint32_t kTallNever = 0u, kTallSome = 1u, kTallAll = 2u;
constexpr uint64_t kTallTiles = 8192;  // of KP planes
__host__ __device__ constexpr uint32_t pt_tall_when(uint32_t tail, uint32_t W4, uint32_t R, uint32_t KP, uint64_t XT,
                                                    uint64_t tiles) {
  return pt_tall(tail, W4, R, KP) == KP ? kTallNever : XT > 1u ? kTallSome : tiles >= kTallTiles ? kTallAll : kTallNever;
}

template <int W4, int R, int KP>
struct PtShape {
  static_assert(W4 >= 1 && W4 <= 4, "x-tile is at most 1024 cells");
  static_assert((R + 1) % 4 == 0 && R <= 31, "point rows are split evenly over 4 waves");
  static_assert(KP >= 1 && KP <= 4, "one to four cell planes per tile");
  static constexpr uint32_t kRowWords = W4 * kWave;           // LDS words per cell row
  static constexpr uint32_t kPlaneWords = kRowWords * (R + 2);  // incl. two padding rows
  static constexpr uint32_t kLdsWords = KP * kPlaneWords;
};

// LDS of a tile besides its corner words.
constexpr uint32_t kPtRowsMax = 64;    // cell rows of a tile
constexpr uint32_t kPtListLen = 512;   // entries of a wave's list of active cells (a ring)
struct PtShared {
  uint32_t tab[256];                        // by key: c_cfg_count of its configuration | cfg << 16
  uint2 cnt[kPtRowsMax];                    // row counts {active | quads << 16, vertices}
  uint2 cnt2[kPtRowsMax];                   // the same of a second part
  uint2 row[kPtRowsMax];                    // {segment, first list entry | y + 1, z + 1 in the grid << 16, 17}
  uint16_t list[kPtThreads / kWave][kPtListLen];  // active cells: row << 10 | x in the x-tile
};
// This thread's entry of the table (a global load).
__device__ __forceinline__ uint32_t pt_table_entry() {
  const uint32_t cfg = key_to_cfg(threadIdx.x);
  return (uint32_t)c_cfg_count[cfg] | (cfg << 16);
}

// Zeroes the state the scan expects to start from (first workgroup only).
__device__ __forceinline__ void zero_scan_state(const ClassifyArgs &a, uint32_t tid, uint32_t nthreads) {
  for (uint32_t i = tid; i < a.scan_state_words; i += nthreads) a.scan_state[i] = 0ull;
  for (uint32_t i = tid; i < a.seg_pad_n; i += nthreads) a.seg_pad[i] = make_uint2(0u, 0u);
  if (tid < 8) reinterpret_cast<uint32_t *>(a.totals)[tid] = 0u;
  zero_tickets(a.scan_ticket, tid);
}

// 4 consecutive points of a row (16 bytes at the alignment of a float).
typedef float Float4Row __attribute__((ext_vector_type(4), aligned(4)));

// Bit q: cell xb + q lies in the grid.
__device__ __forceinline__ uint32_t cells_in_grid(uint32_t xb, uint32_t cx) {
  return xb >= cx ? 0u : (cx - xb >= 4u ? 0xFu : (1u << (cx - xb)) - 1u);
}

// Cells of a lane that are active, as 4 bits, from its 20 corner bits w: cell
// q is when bits q and q + 1 of the four rows are not all alike.
__device__ __forceinline__ uint32_t active_cells(uint32_t w) {
  const uint32_t o2 = w | (w >> 16), a2 = w & (w >> 16);
  const uint32_t o = o2 | (o2 >> 8), n = a2 & (a2 >> 8);
  return (o | (o >> 1)) & ~(n & (n >> 1)) & 0xFu;
}
// Whether any of them can be (all 20 corner bits equal: none is).
__device__ __forceinline__ bool may_be_active(uint32_t w) { return w != 0u && w != 0x1F1F1F1Fu; }

// The second phase of a tile.  Each wave walks its cell rows (append): it finds
// the active cells of a chunk of 256 from their corner bits, writes the group
// maps, and appends the cells to a list of its own in LDS; whenever the list
// holds 64 (and at the end) it classifies 64 of them, a cell per lane (drain):
// table lookup, 2B/3B check, vertex and quad numbers by one wave scan over the
// list, records.  A row's cells follow each other in the list, so a record's
// numbers are the scan minus its value at the row's start.
//
// Classifying from the list instead of 4 cells per lane in place is what the
// list is for: most chunks that hold a surface hold a few active cells, and
// the lanes' 4 cells in sequence made a chain of some thousand cycles for each
// such chunk, up to 8 chunks one after the other in a wave (classify of 256^3
// blobs 33 -> 23 us, 384^3 60 -> 49 us, 603x487x399 142 -> 129 us; the 1024^3
// gyroid, where every lane has work, 1.50 -> 1.44 ms: 7.0 GB moved).
template <uint32_t CAP, uint32_t kRowWords, uint32_t kPlaneWords, int R, bool CARRY>
struct PtList {
  const ClassifyArgs &a;
  const uint32_t *s_w;
  PtShared &sh;
  uint32_t xt, xoff, k, j0;  // x-tile, first cell of the part in it, first plane and row of the tile
  uint32_t have = 0, done = 0;     // entries appended, classified
  uint32_t run = 0, row_run = 0;   // vertices | quads << 16 before the next entry, before its row
  uint16_t *list;

  __device__ __forceinline__ PtList(const ClassifyArgs &a_, const uint32_t *w, PtShared &s, uint32_t xt_,
                                    uint32_t xoff_, uint32_t k_, uint32_t j0_)
      : a(a_), s_w(w), sh(s), xt(xt_), xoff(xoff_), k(k_), j0(j0_), list(s.list[wave_id()]) {}

  static constexpr uint32_t kDivR = (1024u + R - 1u) / R;  // m / R for m < kPtRowsMax
  __device__ static constexpr bool div_ok() {
    for (uint32_t m = 0; m < kPtRowsMax; ++m)
      if (m * kDivR / 1024u != m / R) return false;
    return true;
  }
  static_assert(R >= 1 && R <= 31, "rows of a tile");

  // counts of row m before this part
  __device__ __forceinline__ uint2 before(uint32_t m) const { return CARRY ? sh.cnt[m] : make_uint2(0u, 0u); }

  // A lane's 4 cells in row m from xl in the x-tile: `act` their active bits,
  // `incl` the inclusive sum of the active cells over the row's lanes so far,
  // `pos` the list index of the lane's first.
  __device__ __forceinline__ void append(uint32_t m, uint32_t xl, uint32_t act, uint32_t pos) {
    const uint32_t e = m << 10 | xl;
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
      if ((act >> q) & 1u) {
        list[pos & (kPtListLen - 1u)] = (uint16_t)(e + q);
        ++pos;
      }
    }
  }

  // Group maps of the groups that lanes 4 i .. 4 i + 3 hold, from lane 4 i + 3
  // (grp: its group); incl: active cells of the row up to and with this lane.
  __device__ __forceinline__ void group_maps(uint32_t seg, uint32_t grp, uint32_t act, uint32_t incl) {
    const uint32_t lane = lane_id();
    uint32_t m = act << (4u * (lane & 3u));
    m |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, kDppRowShr + 1, 0xF, 0xF, true);
    m |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, kDppRowShr + 2, 0xF, 0xF, true);
    // (lanes other than 4 i + 3 hold bits of the group before)
    if ((lane & 3u) == 3u && m != 0u) a.gmap[(size_t)seg * (CAP / 16u) + grp] = m | ((incl - (uint32_t)__popc(m)) << 16);
  }

  // Variant-1 test of a 2B/3B cell (its neighbour across the listed face is
  // 2B/3B too).  Inside the part the neighbour's corner bits are in LDS (the
  // word one cell or lane over, or of the next row or plane); only a neighbour
  // outside is read from the field.
  template <int KP>
  __device__ __forceinline__ uint32_t variant1(uint32_t ent, uint32_t widx, uint32_t xl, uint32_t cp, uint32_t r) {
    const FieldDesc &g = a.g;
    const uint32_t face = (ent >> 12) & 7u, q = xl & 3u, l = (xl - xoff) >> 2;
    int nx = (int)(xt * CAP + xl), ny = (int)(j0 + r), nz = (int)(k + cp);
    bool in_part;
    uint32_t nidx = widx, nq = q;
    switch (face) {
      case 0:
        nx += 1;
        in_part = q < 3u || l + 1u < kRowWords;
        nidx = widx + (q == 3u ? 1u : 0u);
        nq = (q + 1u) & 3u;
        break;
      case 1:
        nx -= 1;
        in_part = q > 0u || l > 0u;
        nidx = widx - (q == 0u ? 1u : 0u);
        nq = (q + 3u) & 3u;
        break;
      case 2: ny += 1; in_part = r + 1u < (uint32_t)R; nidx = widx + kRowWords; break;
      case 3: ny -= 1; in_part = r > 0u; nidx = widx - kRowWords; break;
      case 4: nz += 1; in_part = cp + 1u < (uint32_t)KP; nidx = widx + kPlaneWords; break;
      default: nz -= 1; in_part = cp > 0u; nidx = widx - kPlaneWords; break;
    }
    if (nx < 0 || ny < 0 || nz < 0 || nx >= (int)g.cx || ny >= (int)g.cy || nz >= (int)g.cz) return 0u;
    uint32_t nent;
    if (in_part) {
      const uint32_t tq = (s_w[nidx] >> nq) & 0x03030303u;
      nent = sh.tab[((tq * 0x41041u) >> 18) & 0xFFu];
    } else {
      nent = c_cfg_count[cell_cfg_global(g, (uint32_t)nx, (uint32_t)ny, (uint32_t)nz)];
    }
    return (nent >> 11) & 1u;
  }

  // Classifies the next n (at most 64) entries.
  template <int KP>
  __device__ __forceinline__ void drain(uint32_t n) {
    static_assert(div_ok(), "row index division");
    const FieldDesc &g = a.g;
    const uint32_t lane = lane_id();
    const bool valid = lane < n;
    const uint32_t e = ring_take<kPtListLen>(list, done, lane, n, WaveOrder());  // (and sh.row, sh.cnt behind it)
    const uint32_t m = e >> 10, xl = e & 0x3FFu;
    const uint2 row = sh.row[m];
    const uint2 bef = before(m);
    const uint32_t cp = m * kDivR >> 10, r = m - cp * R, q = xl & 3u;
    const uint32_t widx = cp * kPlaneWords + (r + 1u) * kRowWords + ((xl - xoff) >> 2);
    const uint32_t tq = (valid ? s_w[widx] >> q : 0u) & 0x03030303u;
    const uint32_t ent = sh.tab[((tq * 0x41041u) >> 18) & 0xFFu];
    uint32_t l2 = 0u;
    const bool amb = valid && ((ent >> 11) & 1u);
    if (__ballot(amb) != 0ull) {  // rare
      if (amb) l2 = variant1<KP>(ent, widx, xl, cp, r);
    }
    const uint32_t yin = (row.y >> 16) & 1u, zin = row.y >> 17;
    const uint32_t xin = xt * CAP + xl + 1u < g.cx ? 1u : 0u;
    const uint32_t qmask = (xin & yin) | ((xin & zin) << 1) | ((yin & zin) << 2);
    const uint32_t nv = (l2 ? ent >> 4 : ent) & 0xFu, nq = (uint32_t)__popc((ent >> 8) & qmask);
    const uint32_t pk = valid ? nv | (nq << 16) : 0u;
    const uint32_t incl = run + wave_incl_scan_dpp(pk), excl = incl - pk;
    // the entry's place in its row, and the scan's value at the row's start
    const uint32_t rank = done + lane - (row.y & 0xFFFFu);
    const uint32_t at_start = (uint32_t)__shfl((int)excl, (int)((lane - rank) & 63u), kWave);
    const uint32_t st = rank <= lane ? at_start : row_run;
    const uint32_t loc = excl - st;
    if (valid) {
      const size_t at = (size_t)row.x * CAP + (bef.x & 0xFFFFu) + rank;
      a.slots[at] = make_record(xl, (ent >> 16) & 0xFFu, l2, bef.y + (loc & 0xFFFFu));
      a.slot_q[at] = (uint16_t)((bef.x >> 16) + (loc >> 16));
    }
    // the row's counts so far (its last entry writes the final ones)
    const uint32_t next = lane_next(m);
    if (valid && (lane + 1u == n || next != m)) {
      const uint32_t tot = incl - st;
      (CARRY ? sh.cnt2 : sh.cnt)[m] = make_uint2((rank + 1u) | (tot >> 16 << 16), tot & 0xFFFFu);
    }
    run = (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
    row_run = (uint32_t)__builtin_amdgcn_readlane((int)st, (int)(n - 1u));
    done += n;
  }
};

// The tile's row counts leave in one store (a store per row costs more).
template <int R, int KP, bool TWO>
__device__ __forceinline__ void store_row_counts(const ClassifyArgs &a, uint32_t xt, uint32_t j0, uint32_t k,
                                                 const PtShared &sh) {
  __syncthreads();
  if (threadIdx.x < (uint32_t)(KP * R)) {
    const uint32_t m = threadIdx.x, cp = m / R, r = m - cp * R;
    const uint32_t y = j0 + r, z = k + cp;
    const uint2 c = sh.cnt[m], c2 = TWO ? sh.cnt2[m] : make_uint2(0u, 0u);
    if (y < a.g.cy && z < a.g.cz) a.seg_counts[xt + a.XT * (y + a.g.cy * z)] = make_uint2(c.x + c2.x, c.y + c2.y);
  }
  // their sums per plane, for the scan (by another wave; rows past the grid
  // have no counts)
  const uint32_t cp = threadIdx.x - (uint32_t)kWave;
  if (a.part != nullptr && cp < (uint32_t)KP && k + cp < a.g.cz) {
    uint2 sum = make_uint2(0u, 0u);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint2 c = sh.cnt[cp * R + r], c2 = TWO ? sh.cnt2[cp * R + r] : make_uint2(0u, 0u);
      sum.x += c.x + c2.x;
      sum.y += c.y + c2.y + (((c.x + c2.x) & 0xFFFFu) != 0u ? 1u << 16 : 0u);
    }
    a.part[((size_t)(k + cp) * a.NRB + j0 / R) * a.XT + xt] = sum;
  }
}

// A tile's columns are C full chunks of 256 points (a lane holds 4 points of a
// row, a wave takes one row at a time) and then, when LW is not 0, up to 4*LW
// points of which a wave takes 64 / LW rows at a time, LW lanes each.  The
// narrow part is for narrow grids and for the end of a row: there the full
// mapping leaves most lanes past the row's end and costs as much.  x0 is the
// part's first point.
//
// All loads of a part are issued first, from in-bounds addresses: rows and
// planes past the grid are clamped to its last row / plane and lanes past the
// row end to its last 4 points; the cells that would use such values lie
// outside the grid and are never classified.
template <int C, int R, int KP>
struct PtWide {
  static constexpr int kRowsPerWave = (R + 1) / 4;
  static constexpr uint32_t kRowWords = C * kWave;
  static constexpr uint32_t kPlaneWords = kRowWords * (R + 2);
  Float4Row v[kRowsPerWave][KP + 1][C];
  float ve[kRowsPerWave][KP + 1];
  uint32_t xsh[C];  // points a lane's load starts before its first point

  __device__ __forceinline__ void load(const FieldDesc &g, uint32_t x0, uint32_t k, uint32_t j0) {
    const uint32_t lane = lane_id(), wave = wave_id();
    const size_t plane = (size_t)g.X * g.Y;
    // the lane that holds the row's end loads the row's last 4 points and
    // shifts its sign bits (lanes past the end hold bits no cell uses)
    uint32_t xob[C];  // byte offset of the lane's points in a row
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const uint32_t xs = x0 + 256u * c + 4u * lane, xl = min(xs, g.X - 4u);
      xob[c] = xl * 4u;
      xsh[c] = min(xs - xl, 4u);
    }
    const uint32_t xe = x0 + 256u * C < g.X ? x0 + 256u * C : 0u;
#pragma unroll
    for (int i = 0; i < kRowsPerWave; ++i) {
      const size_t yoff = (size_t)min(j0 + wave + 4u * i, g.Y - 1u) * g.X;
#pragma unroll
      for (int p = 0; p <= KP; ++p) {
        const float *rowp = g.f + (size_t)min(k + p, g.Z - 1u) * plane + yoff;
#pragma unroll
        for (int c = 0; c < C; ++c)
          v[i][p][c] = *reinterpret_cast<const Float4Row *>(reinterpret_cast<const char *>(rowp) + xob[c]);
        ve[i][p] = rowp[xe];
      }
    }
  }

  __device__ __forceinline__ void store(float iso, uint32_t *s_w) const {
    const uint32_t lane = lane_id(), wave = wave_id();
    uint16_t *s_h = reinterpret_cast<uint16_t *>(s_w);
    const uint32_t base = wave * kRowWords + lane;
#pragma unroll
    for (int i = 0; i < kRowsPerWave; ++i) {
      uint32_t v5[KP + 1][C];
#pragma unroll
      for (int p = 0; p <= KP; ++p) {
        uint32_t nib[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
          nib[c] = (uint32_t)(v[i][p][c].x < iso) | ((uint32_t)(v[i][p][c].y < iso) << 1) |
                   ((uint32_t)(v[i][p][c].z < iso) << 2) | ((uint32_t)(v[i][p][c].w < iso) << 3);
          nib[c] >>= xsh[c];
        }
        const uint32_t ext = (uint32_t)(ve[i][p] < iso);
#pragma unroll
        for (int c = 0; c < C; ++c) {
          // first point of lane+1, or of the next chunk / the point past the part for lane 63
          uint32_t nb = lane_next(nib[c]);
          const uint32_t nxt =
              (c + 1 < C) ? (uint32_t)__builtin_amdgcn_readfirstlane(nib[(c + 1 < C) ? c + 1 : c]) : ext;
          if (lane == kWave - 1) nb = nxt;
          v5[p][c] = nib[c] | ((nb & 1u) << 4);
        }
      }
#pragma unroll
      for (int cp = 0; cp < KP; ++cp) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
          const uint16_t h = (uint16_t)(v5[cp][c] | (v5[cp + 1][c] << 8));
          // cell row r = wave + 4i sits at padded row r + 1; cell row r - 1 at r
          s_h[2u * (base + cp * kPlaneWords + (4u * i + 1u) * kRowWords + c * kWave)] = h;
          s_h[2u * (base + cp * kPlaneWords + (4u * i) * kRowWords + c * kWave) + 1u] = h;
        }
      }
    }
  }

  // each wave classifies cell rows wave, wave+4, ... of the KP*R rows of the
  // tile; the rows' counts go to sh.cnt
  template <uint32_t CAP>
  __device__ static __forceinline__ void classify(const ClassifyArgs &a, uint32_t xt, uint32_t k, uint32_t j0,
                                                  const uint32_t *s_w, PtShared &sh) {
    const FieldDesc &g = a.g;
    const uint32_t lane = lane_id(), wave = wave_id();
    constexpr int RW = (KP * R + 3) / 4;  // rows of a wave
    static_assert(RW * C <= 32, "chunks of a wave in one mask");
    auto word = [&](uint32_t m, int c) {
      const uint32_t cp = m / R, r = m - cp * R;
      return cp * kPlaneWords + (r + 1u) * kRowWords + c * kWave + lane;
    };
    // the chunks that can hold active cells (the words are read together; rows
    // past the tile read its last row's)
    uint32_t w[RW][C], live = 0;
#pragma unroll
    for (int i = 0; i < RW; ++i) {
#pragma unroll
      for (int c = 0; c < C; ++c) w[i][c] = s_w[word(min(wave + 4u * i, (uint32_t)(KP * R - 1)), c)];
    }
#pragma unroll
    for (int i = 0; i < RW; ++i) {
#pragma unroll
      for (int c = 0; c < C; ++c) live |= __ballot(may_be_active(w[i][c])) != 0ull ? 1u << (i * C + c) : 0u;
    }
    if (live == 0u) return;
    const uint32_t x0 = xt * CAP;
    PtList<CAP, kRowWords, kPlaneWords, R, false> L(a, s_w, sh, xt, 0u, k, j0);
    for (int i = 0; i < RW; ++i) {
      if (!((live >> (i * C)) & ((1u << C) - 1u))) continue;
      const uint32_t m = wave + 4u * i, cp = m / R, y = j0 + m - cp * R, z = k + cp;
      if (m >= (uint32_t)(KP * R) || y >= g.cy || z >= g.cz) continue;
      const uint32_t seg = xt + a.XT * (y + g.cy * z), start = L.have;
      if (lane == 0)
        sh.row[m] = make_uint2(seg, start | (y + 1u < g.cy ? 1u << 16 : 0u) | (z + 1u < g.cz ? 1u << 17 : 0u));
#pragma unroll
      for (int c = 0; c < C; ++c) {
        if (!((live >> (i * C + c)) & 1u)) continue;
        const uint32_t act = active_cells(s_w[word(m, c)]) & cells_in_grid(x0 + 256u * c + 4u * lane, g.cx);
        if (__ballot(act != 0u) == 0ull) continue;
        const uint32_t cnt = (uint32_t)__popc(act), incl = wave_incl_scan_dpp(cnt);
        L.group_maps(seg, 16u * c + (lane >> 2), act, L.have - start + incl);
        L.append(m, 256u * c + 4u * lane, act, L.have + incl - cnt);
        L.have += (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
        while (L.have - L.done >= (uint32_t)kWave) L.template drain<KP>(kWave);
      }
    }
    if (L.have != L.done) L.template drain<KP>(L.have - L.done);
  }
};

// TINY: rows of 2 or 3 points, read one point at a time.
template <int LW, int R, int KP, bool TINY>
struct PtNarrow {
  static_assert(LW == 16 || LW == 32 || LW == 64, "whole DPP rows");
  static constexpr int SR = kWave / LW;                // rows side by side in a wave
  static constexpr int NS = (R + 1) / SR;              // sets of SR point rows in the tile
  static constexpr int SPLIT = NS >= 4 ? 1 : 4 / NS;   // waves that share a row set, each with its cell planes
  static constexpr int PP = (KP + SPLIT - 1) / SPLIT;  // cell planes of a wave
  static constexpr int NI = NS >= 4 ? NS / 4 : 1;      // row sets of a wave
  static constexpr uint32_t kPlaneWords = LW * (R + 2);
  static_assert((R + 1) % SR == 0 && 4 % SPLIT == 0 && (NS % 4 == 0 || NS < 4), "row sets cover the point rows");
  Float4Row v[NI][PP + 1];
  uint32_t xsh;

  __device__ static __forceinline__ uint32_t set0() { return wave_id() % (4u / SPLIT); }
  __device__ static __forceinline__ uint32_t plane0() { return wave_id() / (4u / SPLIT) * PP; }

  __device__ __forceinline__ void load(const FieldDesc &g, uint32_t x0, uint32_t k, uint32_t j0) {
    const uint32_t lane = lane_id(), l = lane % LW, sub = lane / LW;
    const size_t plane = (size_t)g.X * g.Y;
    const uint32_t xs = x0 + 4u * l, xl = TINY ? 0u : min(xs, g.X - 4u);
    xsh = TINY ? 0u : min(xs - xl, 4u);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const uint32_t row = min(j0 + (set0() + 4u * i) * SR + sub, g.Y - 1u) - j0;
      const uint32_t off = (row * g.X + xl) * 4u;
#pragma unroll
      for (int p = 0; p <= PP; ++p) {
        const float *base = g.f + (size_t)min(k + plane0() + p, g.Z - 1u) * plane + (size_t)j0 * g.X;
        if constexpr (TINY) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[i][p][e] = base[row * g.X + min((uint32_t)e, g.X - 1u)];
        } else {
          v[i][p] = *reinterpret_cast<const Float4Row *>(reinterpret_cast<const char *>(base) + off);
        }
      }
    }
  }

  __device__ __forceinline__ void store(float iso, uint32_t *s_w) const {
    const uint32_t lane = lane_id(), l = lane % LW, sub = lane / LW;
    uint16_t *s_h = reinterpret_cast<uint16_t *>(s_w);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      uint32_t v5[PP + 1];
#pragma unroll
      for (int p = 0; p <= PP; ++p) {
        const uint32_t nib = ((uint32_t)(v[i][p].x < iso) | ((uint32_t)(v[i][p].y < iso) << 1) |
                              ((uint32_t)(v[i][p].z < iso) << 2) | ((uint32_t)(v[i][p].w < iso) << 3)) >> xsh;
        v5[p] = nib | ((lane_next(nib) & 1u) << 4);  // (a row's last lane: a bit no cell uses)
      }
      const uint32_t r = (set0() + 4u * i) * SR + sub;  // cell row r sits at padded row r + 1, r - 1 at r
#pragma unroll
      for (int p = 0; p < PP; ++p) {
        const uint32_t cp = plane0() + p;
        if (cp >= (uint32_t)KP) continue;
        const uint16_t h = (uint16_t)(v5[p] | (v5[p + 1] << 8));
        s_h[2u * (cp * kPlaneWords + (r + 1u) * LW + l)] = h;
        s_h[2u * (cp * kPlaneWords + r * LW + l) + 1u] = h;
      }
    }
  }

  // the part's columns start xoff points into the x-tile; with CARRY the rows'
  // counts before it are in sh.cnt, and its own go to sh.cnt2
  template <uint32_t CAP, bool CARRY>
  __device__ static __forceinline__ void classify(const ClassifyArgs &a, uint32_t xt, uint32_t xoff, uint32_t k,
                                                  uint32_t j0, const uint32_t *s_w, PtShared &sh) {
    const FieldDesc &g = a.g;
    const uint32_t lane = lane_id(), wave = wave_id(), l = lane % LW, sub = lane / LW;
    const uint32_t in_x = cells_in_grid(xt * CAP + xoff + 4u * l, g.cx);
    PtList<CAP, (uint32_t)LW, kPlaneWords, R, CARRY> L(a, s_w, sh, xt, xoff, k, j0);
    for (uint32_t m0 = wave * SR; m0 < (uint32_t)(KP * R); m0 += 4u * SR) {
      const uint32_t m = m0 + sub, cp = m / R, r = m - cp * R;
      const uint32_t y = j0 + r, z = k + cp;
      const bool ok = m < (uint32_t)(KP * R) && y < g.cy && z < g.cz;
      const uint32_t act = ok ? active_cells(s_w[cp * kPlaneWords + (r + 1u) * LW + l]) & in_x : 0u;
      if (__ballot(act != 0u) == 0ull) continue;
      const uint32_t cnt = (uint32_t)__popc(act), seg = xt + a.XT * (y + g.cy * z);
      // active cells of the row up to this lane, and of the rows in the lanes before
      const uint32_t incl = LW == kWave ? wave_incl_scan_dpp(cnt) : row_incl_scan_dpp<LW>(cnt);
      uint32_t first = 0u, total = 0u;
#pragma unroll
      for (int i = 0; i < SR; ++i) {
        const uint32_t t = (uint32_t)__builtin_amdgcn_readlane((int)incl, i * LW + LW - 1);
        if (sub == (uint32_t)i) first = total;
        total += t;
      }
      const uint32_t start = L.have + first;
      if (l == 0u && ok)
        sh.row[m] = make_uint2(seg, start | (y + 1u < g.cy ? 1u << 16 : 0u) | (z + 1u < g.cz ? 1u << 17 : 0u));
      L.group_maps(seg, (xoff >> 4) + (l >> 2), act, (ok ? L.before(m).x & 0xFFFFu : 0u) + incl);
      L.append(m, xoff + 4u * l, act, start + incl - cnt);
      L.have += total;
      while (L.have - L.done >= (uint32_t)kWave) L.template drain<KP>(kWave);
    }
    if (L.have != L.done) L.template drain<KP>(L.have - L.done);
  }
};

// One plane tile with the parts TAIL names (pt_tail).
template <uint32_t TAIL, uint32_t CAP, int R, int KP, uint32_t WORDS>
__device__ __forceinline__ void classify_pt_parts(const ClassifyArgs &a, uint32_t xt, uint32_t k, uint32_t j0,
                                                  uint32_t (&s_w)[WORDS], PtShared &sh, uint32_t tab_entry, bool store_tab) {
  static_assert(KP * R <= (int)kPtRowsMax, "row counts are staged in kPtRowsMax LDS entries");
  constexpr bool TINY = TAIL == kPtTailTiny;
  constexpr int C = TAIL == kPtTailFull ? (int)(CAP / 256u) : TINY ? 0 : (int)(TAIL >> 8);
  constexpr int LW = TAIL == kPtTailFull ? 0 : TINY ? 16 : (int)(TAIL & 0xFFu);
  constexpr bool TWO = C != 0 && LW != 0;
  using W = PtWide<C ? C : 1, R, KP>;
  using N = PtNarrow<LW ? LW : 16, R, KP, TINY>;
  static_assert((C != 0 ? KP * W::kPlaneWords : 0u) + (LW != 0 ? KP * N::kPlaneWords : 0u) <= WORDS, "the parts' LDS words");
  const bool tile_ok = (k < a.g.cz) && (j0 < a.g.cy);  // padding tiles do nothing
  const uint32_t x0 = xt * CAP;
  uint32_t *const s_n = s_w + (C ? KP * W::kPlaneWords : 0u);  // the narrow part's words
  if (tile_ok) {
    W w;
    N n;
    if constexpr (LW != 0) n.load(a.g, x0 + 256u * C, k, j0);
    if constexpr (C != 0) w.load(a.g, x0, k, j0);
    if constexpr (LW != 0) n.store(a.g.iso, s_n);
    if constexpr (C != 0) w.store(a.g.iso, s_w);
  }
  // the table entry was loaded before the field rows; storing it here keeps
  // its wait behind theirs
  if (store_tab) sh.tab[threadIdx.x] = tab_entry;
  if (threadIdx.x < kPtRowsMax) {
    sh.cnt[threadIdx.x] = make_uint2(0u, 0u);
    if (TWO) sh.cnt2[threadIdx.x] = make_uint2(0u, 0u);
  }
  __syncthreads();
  if (!tile_ok) return;  // uniform over the workgroup
  if constexpr (C != 0) W::template classify<CAP>(a, xt, k, j0, s_w, sh);
  if constexpr (LW != 0) {
    if constexpr (C != 0) __syncthreads();  // the full chunks' counts
    N::template classify<CAP, C != 0>(a, xt, 256u * C, k, j0, s_n, sh);
  }
  store_row_counts<R, KP, TWO>(a, xt, j0, k, sh);
}

// Single volume: block b -> tile through the XCD mapping (pt_tile_of).
// TAIL: the parts of the last x-tile.
template <int W4, int R, int KP, uint32_t TAIL>
__global__ __launch_bounds__(kPtThreads) __attribute__((amdgpu_waves_per_eu(W4 >= 4 || R > 7 ? 4 : 8, W4 >= 4 ? 4 : 8))) void k_classify_pt(PtArgs pa) {
  __shared__ uint32_t s_w[PtShape<W4, R, KP>::kLdsWords];
  __shared__ PtShared sh;
  const ClassifyArgs &a = pa.c;
  const uint32_t tab = pt_table_entry();
  if (blockIdx.x == 0) {
    zero_scan_state(a, threadIdx.x, kPtThreads);
    if (a.counts_out != nullptr && threadIdx.x < 4) a.counts_out[threadIdx.x] = 0u;
  }
  constexpr uint32_t KPT = pt_tall(TAIL, W4, R, KP);
  constexpr uint32_t CAP = 256u * W4;
  if (TAIL != kPtTailFull && blockIdx.x >= pa.tail_block) {
    const PtTile t = pt_tile_of(blockIdx.x - pa.tail_block, 1u, pa.NRB, pa.NKBT, pa.B);
    if (KPT != KP && pa.tall)
      classify_pt_parts<TAIL, CAP, R, (int)KPT>(a, a.XT - 1u, t.kb * KPT, t.rb * R, s_w, sh, tab, true);
    else
      classify_pt_parts<TAIL, CAP, R, KP>(a, a.XT - 1u, t.kb * KP, t.rb * R, s_w, sh, tab, true);
  } else if (TAIL != kPtTailTiny) {
    const PtTile t = pt_tile_of(blockIdx.x, TAIL != kPtTailFull ? a.XT - 1u : a.XT, pa.NRB, pa.NKB, pa.B);
    classify_pt_parts<kPtTailFull, CAP, R, KP>(a, t.xt, t.kb * KP, t.rb * R, s_w, sh, tab, true);
  }
}

// ---------------------------------------------------------------------------
// Batches: many volumes in one launch sequence.  The segments of all volumes
// are concatenated (volume v owns segments [seg_off, seg_off + nsegs_v)), so
// the scan runs once over the whole batch and a volume's local vertex / quad
// numbers are the global ones minus the prefix at its first segment.

constexpr uint32_t kMaxBatch = 1024;  // volumes per batch call
constexpr uint32_t kPublishHead = 16;  // words before the counts of k_publish

// Per-volume part of the emit arguments.
struct EmitVol {
  FieldDesc g;
  FastDiv div_xt, div_cy;              // division by XT and by cy
  uint32_t span;                       // emit_span: segments that share 32-bit offsets
  const float *xt_c, *yt_c, *zt_c;     // coordinate of every point index per axis
  uint32_t XT, seg_off;                // x-tiles; first segment of the volume
  uint32_t vbase, qbase;               // global vertex / quad number of its first
  float *verts;
  uint64_t vcap;
  int32_t *quads;
  uint64_t qcap;
  uint32_t *status;
  // emit only cell planes [kmin, kmax); quad entries are vertex numbers plus
  // vshift (a slab of a larger grid, numbered globally)
  uint32_t kmin = 0, kmax = 0xFFFFFFFFu, vshift = 0;
};

struct BatchVol {
  ClassifyArgs c;         // per-volume field and tiling; record pointers start at seg_off
  EmitVol e;              // for the emit, except vbase and qbase (BatchEmitArgs.base)
  uint32_t NRB, NKP;      // row blocks and plane blocks of the volume
  uint32_t tall;          // kTall*
  uint32_t tail;          // parts of the last x-tile (pt_tail)
  uint32_t tile_off;      // first flattened classify tile
  uint32_t seg_off, nsegs;
  float mnx, mny, mnz, rgx, rgy, rgz;
  uint32_t *counts;       // the volume's mdmc_counts
  float *coords;          // X + Y + Z point coordinates (filled before the emit)
};

struct BatchArgs {
  BatchVol *vols;
  const uint32_t *tile_off;  // first tile of each volume, then the total
  uint32_t nvol, total_tiles;
  ClassifyArgs zero;      // scan state of the batch (zeroed by block 0)
};

// Last volume v with off[v] <= t (off ascending, off[0] <= t; volumes without
// tiles share an entry with the next).  The 64 lanes test every stride-th
// entry, then the entries of the stride found: two loads and two ballots, no
// table in LDS (a workgroup that first copied the offsets from the volume
// descriptors touched a cache line per volume).
__device__ __forceinline__ uint32_t volume_of(const uint32_t *off, uint32_t nvol, uint32_t t) {
  static_assert(kMaxBatch <= kWave * kWave, "two rounds of 64");
  const uint32_t lane = lane_id(), stride = (nvol + kWave - 1u) / kWave;
  const uint32_t i = lane * stride;
  const uint32_t m = (uint32_t)__popcll(__ballot(i < nvol && off[min(i, nvol - 1u)] <= t)) - 1u;
  const uint32_t j = m * stride + lane;
  return m * stride + (uint32_t)__popcll(__ballot(lane < stride && j < nvol && off[min(j, nvol - 1u)] <= t)) - 1u;
}

// Classify over the flattened tiles of all volumes (tiles of a volume in
// memory order): with a grid of at least the tile count a workgroup per tile,
// with a smaller grid each workgroup walks several (persistent).  6 waves per
// SIMD at 256-cell x-tiles and 5 at 512: every kind of tile is in this kernel,
// and at 8 and 6 waves it spilled 14 vector registers (256 volumes of 32 to 256
// points: 582 us at 8 waves, 567 at 7, 512 at 6, 530 at 5; 24 volumes of 300 to
// 511 points a row: 252 us at 6, 203 at 5, 219 at 4).
template <int W4, int R, int KP>
__global__ __launch_bounds__(kPtThreads) __attribute__((amdgpu_waves_per_eu(W4 == 1 ? 6 : (W4 == 2 ? 5 : 4), W4 == 1 ? 6 : (W4 == 2 ? 5 : 4)))) void k_classify_batch(BatchArgs b) {
  __shared__ uint32_t s_w[PtShape<W4, R, KP>::kLdsWords];
  __shared__ PtShared sh;
  sh.tab[threadIdx.x] = pt_table_entry();
  if (blockIdx.x == 0) {
    zero_scan_state(b.zero, threadIdx.x, kPtThreads);
    if (threadIdx.x < 4) b.zero.counts_out[threadIdx.x] = 0u;  // the batch's scan counts
  }
  __syncthreads();
  // XCD x (workgroups b with b % 8 == x) takes a contiguous eighth of the
  // flattened tiles, so tiles that share halo rows and planes meet in its L2
  const uint32_t G = gridDim.x;
  uint32_t t = blockIdx.x, t_end = b.total_tiles, t_step = G;
  if (G >= 8u) {
    const uint32_t x = blockIdx.x & 7u;
    t = (uint32_t)((uint64_t)b.total_tiles * x / 8u) + (blockIdx.x >> 3);
    t_end = (uint32_t)((uint64_t)b.total_tiles * (x + 1u) / 8u);
    t_step = (G >> 3) + (x < (G & 7u) ? 1u : 0u);
  }
  for (; t < t_end; t += t_step) {
    const uint32_t v = volume_of(b.tile_off, b.nvol, t);
    // the volume's descriptor through the constant address space (nothing in
    // this launch writes it), so that its fields are scalar loads and not
    // vector registers
    const __attribute__((address_space(4))) BatchVol *bv = (const __attribute__((address_space(4))) BatchVol *)b.vols + v;
    ClassifyArgs a{};
    a.g.f = bv->c.g.f;
    a.g.X = bv->c.g.X;
    a.g.Y = bv->c.g.Y;
    a.g.Z = bv->c.g.Z;
    a.g.cx = bv->c.g.cx;
    a.g.cy = bv->c.g.cy;
    a.g.cz = bv->c.g.cz;
    a.g.iso = bv->c.g.iso;
    a.XT = bv->c.XT;
    a.seg_counts = bv->c.seg_counts;
    a.slots = bv->c.slots;
    a.slot_q = bv->c.slot_q;
    a.gmap = bv->c.gmap;
    const uint32_t nrb = bv->NRB;
    const uint32_t local = t - bv->tile_off;
    const uint32_t xt = local % a.XT, u = local / a.XT;
    const uint32_t kb = u / nrb, k = kb * KP, j0 = (u - kb * nrb) * R;
    const uint32_t tail = xt + 1u == a.XT ? bv->tail : kPtTailFull, tall = tail == kPtTailFull ? kTallNever : bv->tall;
    constexpr uint32_t CAP = 256u * W4;
    const uint32_t kpt = pt_tall(tail, W4, R, KP);
    if (tall == kTallSome && kb % (kpt / KP) != 0u) continue;  // (uniform) another's planes
    __syncthreads();  // the previous tile's LDS words are no longer read
    const uint32_t kt = tall == kTallSome ? k : kb * kpt;
    if (W4 <= 2 && tail == kPtTail16 && tall != kTallNever)
      classify_pt_parts<kPtTail16, CAP, R, (int)pt_tall(kPtTail16, W4, R, KP)>(a, xt, kt, j0, s_w, sh, 0u, false);
    else if (W4 <= 2 && tail == kPtTail32 && tall != kTallNever)
      classify_pt_parts<kPtTail32, CAP, R, (int)pt_tall(kPtTail32, W4, R, KP)>(a, xt, kt, j0, s_w, sh, 0u, false);
    else if (W4 == 2 && tail == kPtTail64 && tall != kTallNever)
      classify_pt_parts<kPtTail64, CAP, R, (int)pt_tall(kPtTail64, W4, R, KP)>(a, xt, kt, j0, s_w, sh, 0u, false);
    else if (W4 <= 2 && tail == kPtTail16)
      classify_pt_parts<kPtTail16, CAP, R, KP>(a, xt, k, j0, s_w, sh, 0u, false);
    else if (W4 <= 2 && tail == kPtTail32)
      classify_pt_parts<kPtTail32, CAP, R, KP>(a, xt, k, j0, s_w, sh, 0u, false);
    else if (W4 == 2 && tail == kPtTail64)
      classify_pt_parts<kPtTail64, CAP, R, KP>(a, xt, k, j0, s_w, sh, 0u, false);
    else if (tail == kPtTailTiny)
      classify_pt_parts<kPtTailTiny, CAP, R, KP>(a, xt, k, j0, s_w, sh, 0u, false);
    else
      classify_pt_parts<kPtTailFull, CAP, R, KP>(a, xt, k, j0, s_w, sh, 0u, false);
  }
}

// utils::ijk_to_xyz (include/utils.hpp:118-122): i / n * range + min, three
// correctly rounded float operations.
__device__ __forceinline__ float coordf(uint32_t i, uint32_t n, float range, float mn) {
  return (float)i / (float)n * range + mn;
}

// Coordinates of the point indices of a volume, per axis (X, then Y, then Z
// entries): the same three float operations per entry as the reference.
struct CoordArgs {
  float *out;
  uint32_t X, Y, Z, cx, cy, cz;
  float mnx, mny, mnz, rgx, rgy, rgz;
  uint32_t z_off;  // global index of the first z point (a slab of a larger grid; cz is then the grid's)
};

__device__ __forceinline__ void coords_fill(const CoordArgs &c, uint32_t i0, uint32_t stride) {
  const uint32_t n = c.X + c.Y + c.Z;
  for (uint32_t i = i0; i < n; i += stride) {
    float v;
    if (i < c.X) v = coordf(i, c.cx, c.rgx, c.mnx);
    else if (i < c.X + c.Y) v = coordf(i - c.X, c.cy, c.rgy, c.mny);
    else v = coordf(i - c.X - c.Y + c.z_off, c.cz, c.rgz, c.mnz);
    c.out[i] = v;
  }
}

__global__ __launch_bounds__(256) void k_coords(CoordArgs c) {
  coords_fill(c, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

// ---------------------------------------------------------------------------
// Decoupled look-back scan over segment totals.  A tile is 2048 segments, 8
// per thread read as four 16-byte loads (the totals array is padded to a
// whole number of tiles with zeros).  Four channels are scanned: active
// cells, vertices, quads and non-empty segments.  Outputs: the first vertex
// and quad of every segment; the list of non-empty segments with the index
// of their first active cell (ne[i] = {segment, first active}, ne[NE] =
// {nsegs, A}); for every chunk of 64 active cells the list position of the
// segment holding its first cell; the grand totals.

constexpr int kScanThreads = 256;
constexpr int kScanIpt = 8;  // segments per thread (16: 1 us slower per 512^3 extraction)
constexpr int kScanTile = kScanThreads * kScanIpt;
static_assert((uint32_t)kScanTile == kScanTileSegs, "scan_form's tiles");
constexpr uint32_t kSpinLimit = 1u << 24;

struct ScanArgs {
  const uint2 *seg_counts;  // padded to ntiles * kScanTile entries
  uint32_t nsegs, ntiles;
  uint64_t max_chunks;      // capacity of chunk_ne
  uint2 *seg_vq;            // per segment: first vertex, first quad (same padding)
  uint2 *ne;                // non-empty segments: {segment, first active cell}; nsegs + 1
  uint32_t *chunk_ne;       // per 64 active cells: index into ne of its first cell's segment
  unsigned long long *state;  // 4 words per tile: (status << 32) | value
  uint32_t *ticket;
  Totals *totals;
  uint32_t *counts_out;  // optional user mdmc_counts
  CoordArgs co;          // coordinate tables, filled by the scan's workgroups
  uint32_t fill_coords;  // when the box is known at count time
};

__device__ __forceinline__ unsigned long long ld_state(const unsigned long long *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_state(unsigned long long *p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ __launch_bounds__(kScanThreads) void k_scan(ScanArgs a) {
  __shared__ uint32_t s_tile;
  __shared__ uint4 s_wave[kScanThreads / kWave];
  __shared__ uint4 s_prefix;
  const uint32_t tid = threadIdx.x, lane = lane_id(), wave = wave_id();
  if (tid == 0) s_tile = atomicAdd(a.ticket, 1u);
  __syncthreads();
  const uint32_t t = s_tile;
  const uint32_t base = t * kScanTile + tid * kScanIpt;

  uint4 c[kScanIpt / 2];
  const uint4 *src = reinterpret_cast<const uint4 *>(a.seg_counts + base);
#pragma unroll
  for (int i = 0; i < kScanIpt / 2; ++i) c[i] = src[i];
  // per segment: .x = nact | nquad << 16, .y = nvert; two segments per uint4
  uint4 sum = make_uint4(0, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < kScanIpt / 2; ++i) {
    sum.x += (c[i].x & 0xFFFFu) + (c[i].z & 0xFFFFu);
    sum.y += c[i].y + c[i].w;
    sum.z += (c[i].x >> 16) + (c[i].z >> 16);
    sum.w += ((c[i].x & 0xFFFFu) ? 1u : 0u) + ((c[i].z & 0xFFFFu) ? 1u : 0u);
  }
  uint4 inc;
  inc.x = wave_incl_scan_dpp(sum.x);
  inc.y = wave_incl_scan_dpp(sum.y);
  inc.z = wave_incl_scan_dpp(sum.z);
  inc.w = wave_incl_scan_dpp(sum.w);
  if (lane == kWave - 1) s_wave[wave] = inc;
  __syncthreads();
  uint4 woff = make_uint4(0, 0, 0, 0), agg = make_uint4(0, 0, 0, 0);
#pragma unroll
  for (int w = 0; w < kScanThreads / kWave; ++w) {
    const uint4 v = s_wave[w];
    if ((uint32_t)w < wave) { woff.x += v.x; woff.y += v.y; woff.z += v.z; woff.w += v.w; }
    agg.x += v.x; agg.y += v.y; agg.z += v.z; agg.w += v.w;
  }

  if (wave == 0) {
    unsigned long long *my = a.state + 4ull * t;
    uint4 excl = make_uint4(0, 0, 0, 0);
    const unsigned long long AGG = 1ull << 32, INC = 2ull << 32;
    if (t == 0) {
      if (lane == 0) {
        st_state(my + 0, INC | agg.x); st_state(my + 1, INC | agg.y);
        st_state(my + 2, INC | agg.z); st_state(my + 3, INC | agg.w);
      }
    } else {
      if (lane == 0) {
        st_state(my + 0, AGG | agg.x); st_state(my + 1, AGG | agg.y);
        st_state(my + 2, AGG | agg.z); st_state(my + 3, AGG | agg.w);
      }
      // Each channel word is self-describing (status, value) and a tile flips
      // its four words from aggregate to inclusive one at a time, so every
      // channel is resolved on its own: sum aggregates back to the nearest
      // tile whose word in *that* channel is inclusive.
      int64_t look = (int64_t)t - 1;
      bool timed_out = false;
      uint32_t done = 0;  // bit c: channel c resolved
      while (done != 0xFu) {
        const int64_t idx = look - (int64_t)lane;
        unsigned long long w[4] = {INC, INC, INC, INC};  // before tile 0: inclusive zeros
        if (idx >= 0) {
          const unsigned long long *p = a.state + 4ull * (uint64_t)idx;
          // the four channel words are read together; only words not yet
          // published are read again
#pragma unroll
          for (int ch = 0; ch < 4; ++ch)
            if (!((done >> ch) & 1u)) w[ch] = ld_state(p + ch);
          uint32_t spins = 0;
#pragma unroll
          for (int ch = 0; ch < 4; ++ch) {
            if ((done >> ch) & 1u) continue;
            while ((w[ch] >> 32) == 0 && ++spins < kSpinLimit) w[ch] = ld_state(p + ch);
          }
          if (spins >= kSpinLimit) timed_out = true;
        }
        uint32_t add[4];
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) {
          add[ch] = 0;
          if ((done >> ch) & 1u) continue;
          const uint64_t incmask = __ballot((w[ch] >> 32) == 2);
          const int stop = incmask ? (__ffsll((long long)incmask) - 1) : kWave;
          const uint32_t val = ((int)lane <= stop && idx >= 0) ? (uint32_t)w[ch] : 0u;
          add[ch] = __shfl(wave_incl_scan(val), kWave - 1, kWave);
          if (incmask) done |= 1u << ch;
        }
        excl.x += add[0]; excl.y += add[1]; excl.z += add[2]; excl.w += add[3];
        look -= kWave;
      }
      if (__ballot(timed_out) && lane == 0 && a.counts_out)
        atomicOr(a.counts_out + 3, kStatusScanTimeout);
      if (lane == 0) {
        st_state(my + 0, INC | (uint32_t)(excl.x + agg.x));
        st_state(my + 1, INC | (uint32_t)(excl.y + agg.y));
        st_state(my + 2, INC | (uint32_t)(excl.z + agg.z));
        st_state(my + 3, INC | (uint32_t)(excl.w + agg.w));
        // the tile where a 32-bit total first passes 2^32 - 1 sees its
        // inclusive sum wrap (vertex and quad numbers are 32-bit, as the
        // reference's)
        const bool wraps = excl.x + agg.x < excl.x || excl.y + agg.y < excl.y || excl.z + agg.z < excl.z;
        if (wraps && a.counts_out) atomicOr(a.counts_out + 3, kStatusIndexRange);
      }
    }
    if (lane == 0) s_prefix = excl;
  }
  __syncthreads();
  const uint4 tp = s_prefix;
  // exclusive prefix of this thread's first segment
  uint32_t pa = tp.x + woff.x + inc.x - sum.x;
  uint32_t pv = tp.y + woff.y + inc.y - sum.y;
  uint32_t pq = tp.z + woff.z + inc.z - sum.z;
  uint32_t pe = tp.w + woff.w + inc.w - sum.w;
  bool bad = false;
  uint4 *dst = reinterpret_cast<uint4 *>(a.seg_vq + base);
#pragma unroll
  for (int i = 0; i < kScanIpt / 2; ++i) {
    uint4 o;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t cx_ = h ? c[i].z : c[i].x, cy_ = h ? c[i].w : c[i].y;
      const uint32_t n = cx_ & 0xFFFFu;
      if (h) { o.z = pv; o.w = pq; } else { o.x = pv; o.y = pq; }
      if (n) {
        const uint32_t sg = base + 2 * i + h;
        if (pe < a.nsegs) a.ne[pe] = make_uint2(sg, pa); else bad = true;
        for (uint32_t gch = (pa + 63u) >> 6; (gch << 6) < pa + n; ++gch) {
          if (gch < a.max_chunks) a.chunk_ne[gch] = pe; else bad = true;
        }
        ++pe;
      }
      pa += n;
      pv += cy_;
      pq += cx_ >> 16;
    }
    dst[i] = o;
  }
  if (t == a.ntiles - 1 && tid == kScanThreads - 1) {
    // pa/pv/pq/pe now hold the grand totals
    Totals tot;
    tot.num_active = pa;
    tot.num_vertices = pv;
    tot.num_quads = pq;
    tot.num_nonempty = pe;
    tot.num_chunks = (pa + 63u) >> 6;
    tot.pad0 = tot.pad1 = tot.pad2 = 0;
    *a.totals = tot;
    if (pe <= a.nsegs) a.ne[pe] = make_uint2(a.nsegs, pa); else bad = true;
    if (a.counts_out) {
      a.counts_out[0] = pa;
      a.counts_out[1] = pv;
      a.counts_out[2] = pq;
    }
  }
  if (bad && a.counts_out) atomicOr(a.counts_out + 3, kStatusInternal);
  if (a.fill_coords) coords_fill(a.co, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

// The scan of a small or medium single volume, without look-back: a workgroup
// takes whole cell planes of at most a scan tile's segments and finds what
// precedes them by summing the sums the classify left per plane, row block and
// x-tile (1/7 of the totals, contiguous in scan order), so that no workgroup
// waits for another: a look-back's hops between the XCDs' caches cost more
// than reading them.  HIP events around the scan: 64^3 10.0 -> 6.7 us, 128^3
// 10.2 -> 7.4, 256^3 9.9 -> 9.1, 384^3 12.0 -> 10.5.  The reading grows with
// the square of the sums: at 512^3 (37,000 sums) it costs what the look-back
// does, so kPlaneScanParts ends there.

struct PlaneScanArgs {
  ScanArgs s;           // (state and ticket unused)
  const uint2 *part;
  uint32_t plane_segs;  // segments per cell plane
  uint32_t plane_parts; // sums per cell plane
  uint32_t planes;      // cell planes per workgroup
};

// A thread's kScanIpt segment totals from `base`, zeros from `end` on.
__device__ __forceinline__ void scan_load(const uint2 *seg_counts, uint32_t base, uint32_t end, uint2 (&c)[kScanIpt]) {
  typedef uint32_t Word4 __attribute__((ext_vector_type(4), aligned(8)));
#pragma unroll
  for (int i = 0; i < kScanIpt / 2; ++i) {
    const Word4 w = *reinterpret_cast<const Word4 *>(seg_counts + scan_pair(base, i, end));
    c[2 * i] = base + 2 * i < end ? make_uint2(w.x, w.y) : make_uint2(0u, 0u);
    c[2 * i + 1] = base + 2 * i + 1 < end ? make_uint2(w.z, w.w) : make_uint2(0u, 0u);
  }
}
// {active cells, vertices, quads, non-empty segments}
__device__ __forceinline__ uint4 scan_sum(const uint2 (&c)[kScanIpt]) {
  uint4 sum = make_uint4(0, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < kScanIpt; ++i) {
    sum.x += c[i].x & 0xFFFFu;
    sum.y += c[i].y;
    sum.z += c[i].x >> 16;
    sum.w += (c[i].x & 0xFFFFu) ? 1u : 0u;
  }
  return sum;
}
__device__ __forceinline__ uint4 scan_incl(uint4 v) {
  return make_uint4(wave_incl_scan_dpp(v.x), wave_incl_scan_dpp(v.y), wave_incl_scan_dpp(v.z), wave_incl_scan_dpp(v.w));
}

// A workgroup's segments [first, end): their bases and the lists, given the
// thread's share `bef` of the sums of everything before them.
__device__ __forceinline__ void scan_write(const ScanArgs &a, uint32_t first, uint32_t end, const uint2 (&c)[kScanIpt],
                                           uint4 bef) {
  constexpr int kWaves = kScanThreads / kWave;
  __shared__ uint4 s_before[kWaves], s_wave[kWaves];
  __shared__ uint2 s_high[kWaves];  // upper words of s_before's vertices and quads
  const uint32_t tid = threadIdx.x, lane = lane_id(), wave = wave_id(), base = first + tid * kScanIpt;
  const uint4 sum = scan_sum(c), inc = scan_incl(sum);
  // (vertices and quads may pass 2^32, which is reported: summed in halves)
  const uint32_t act = wave_incl_scan_dpp(bef.x), ne = wave_incl_scan_dpp(bef.w);
  const uint64_t bv = ((uint64_t)wave_incl_scan_dpp(bef.y >> 16) << 16) + wave_incl_scan_dpp(bef.y & 0xFFFFu);
  const uint64_t bq = ((uint64_t)wave_incl_scan_dpp(bef.z >> 16) << 16) + wave_incl_scan_dpp(bef.z & 0xFFFFu);
  if (lane == kWave - 1) {
    s_wave[wave] = inc;
    s_before[wave] = make_uint4(act, (uint32_t)bv, (uint32_t)bq, ne);
    s_high[wave] = make_uint2((uint32_t)(bv >> 32), (uint32_t)(bq >> 32));
  }
  __syncthreads();
  uint32_t pa = inc.x - sum.x, pv = inc.y - sum.y, pq = inc.z - sum.z, pe = inc.w - sum.w;
  uint64_t tot_v = 0, tot_q = 0;  // a total past 2^32 - 1 is reported
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    const uint4 v = s_wave[w], b = s_before[w];
    pa += b.x;
    pv += b.y;
    pq += b.z;
    pe += b.w;
    const uint2 h = s_high[w];
    tot_v += ((uint64_t)h.x << 32) + b.y + v.y;
    tot_q += ((uint64_t)h.y << 32) + b.z + v.z;
    if ((uint32_t)w < wave) {
      pa += v.x;
      pv += v.y;
      pq += v.z;
      pe += v.w;
    }
  }
  if (tid == 0 && ((tot_v | tot_q) >> 32) != 0u && a.counts_out) atomicOr(a.counts_out + 3, kStatusIndexRange);
  bool bad = false;
#pragma unroll
  for (int i = 0; i < kScanIpt; ++i) {
    const uint32_t sg = base + i, n = c[i].x & 0xFFFFu;
    if (sg < end) a.seg_vq[sg] = make_uint2(pv, pq);
    if (n) {
      if (pe < a.nsegs) a.ne[pe] = make_uint2(sg, pa); else bad = true;
      for (uint32_t gch = (pa + 63u) >> 6; (gch << 6) < pa + n; ++gch) {
        if (gch < a.max_chunks) a.chunk_ne[gch] = pe; else bad = true;
      }
      ++pe;
    }
    pa += n;
    pv += c[i].y;
    pq += c[i].x >> 16;
  }
  if (end == a.nsegs && tid == kScanThreads - 1) {
    // pa/pv/pq/pe now hold the grand totals
    Totals tot;
    tot.num_active = pa;
    tot.num_vertices = pv;
    tot.num_quads = pq;
    tot.num_nonempty = pe;
    tot.num_chunks = (pa + 63u) >> 6;
    tot.pad0 = tot.pad1 = tot.pad2 = 0;
    *a.totals = tot;
    a.seg_vq[a.nsegs] = make_uint2(pv, pq);
    if (pe <= a.nsegs) a.ne[pe] = make_uint2(a.nsegs, pa); else bad = true;
    if (a.counts_out) {
      a.counts_out[0] = pa;
      a.counts_out[1] = pv;
      a.counts_out[2] = pq;
    }
  }
  if (bad && a.counts_out) atomicOr(a.counts_out + 3, kStatusInternal);
}

__global__ __launch_bounds__(kScanThreads) void k_scan_planes(PlaneScanArgs p) {
  const ScanArgs &a = p.s;
  const uint32_t tid = threadIdx.x;
  const uint32_t first = blockIdx.x * p.planes * p.plane_segs;
  const uint32_t end = min(first + p.planes * p.plane_segs, a.nsegs);
  uint2 c[kScanIpt];
  scan_load(a.seg_counts, first + tid * kScanIpt, end, c);
  // sums of everything before the workgroup's planes
  const uint32_t nbefore = blockIdx.x * p.planes * p.plane_parts;
  uint4 bef = make_uint4(0, 0, 0, 0);
  const uint4 *parts2 = reinterpret_cast<const uint4 *>(p.part);
#pragma unroll 8
  for (uint32_t i = tid; i < nbefore / 2u; i += kScanThreads) {
    const uint4 q = parts2[i];
    bef.x += (q.x & 0xFFFFu) + (q.z & 0xFFFFu);
    bef.y += (q.y & 0xFFFFu) + (q.w & 0xFFFFu);
    bef.z += (q.x >> 16) + (q.z >> 16);
    bef.w += (q.y >> 16) + (q.w >> 16);
  }
  if ((nbefore & 1u) && tid == 0) {
    const uint2 q = p.part[nbefore - 1u];
    bef.x += q.x & 0xFFFFu;
    bef.y += q.y & 0xFFFFu;
    bef.z += q.x >> 16;
    bef.w += q.y >> 16;
  }
  scan_write(a, first, end, c, bef);
  if (a.fill_coords) coords_fill(a.co, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

// The scan of larger volumes and of batches, in two launches and again without
// look-back: k_scan_sums leaves the sums of every scan tile, and a workgroup of
// k_scan_tiles adds up those before its own.  HIP events around both launches:
// 512^3 (128 tiles) 13.3 -> 11.6 us, 603x487x399 (190) 13.3 -> 12.0, 1024^3
// gyroid (1024) 62.8 -> 44.9, 256 volumes of 32 to 256 points (1,460) 66.7 ->
// 40.2; with 24 volumes of 32 to 128 points (57 tiles) the look-back is ahead,
// 9.9 to 11.3.  The reading grows with the square of the tiles and the
// look-back with their number; rows of 64 points, both launches against the
// look-back: 15.6 and 26 us at 512 tiles, 37 and 66 at 2,048, 69 and 108 at
// 4,092, 130 and 189 at 8,188.  So the two are still ahead where kTileScanMax
// ends; volumes of that many cell rows need 17 GB of scratch.
__global__ __launch_bounds__(kScanThreads) void k_scan_sums(ScanArgs a, uint4 *sums) {
  __shared__ uint4 s_wave[kScanThreads / kWave];
  const uint32_t first = blockIdx.x * kScanTile, end = min(first + kScanTile, a.nsegs);
  uint2 c[kScanIpt];
  scan_load(a.seg_counts, first + threadIdx.x * kScanIpt, end, c);
  const uint4 inc = scan_incl(scan_sum(c));
  if (lane_id() == kWave - 1) s_wave[wave_id()] = inc;
  __syncthreads();
  if (threadIdx.x != 0) return;
  uint4 t = make_uint4(0, 0, 0, 0);
#pragma unroll
  for (int w = 0; w < kScanThreads / kWave; ++w) {
    const uint4 v = s_wave[w];
    t = make_uint4(t.x + v.x, t.y + v.y, t.z + v.z, t.w + v.w);
  }
  sums[blockIdx.x] = t;
}

__global__ __launch_bounds__(kScanThreads) void k_scan_tiles(ScanArgs a, const uint4 *sums) {
  const uint32_t first = blockIdx.x * kScanTile, end = min(first + kScanTile, a.nsegs);
  uint2 c[kScanIpt];
  scan_load(a.seg_counts, first + threadIdx.x * kScanIpt, end, c);
  uint4 bef = make_uint4(0, 0, 0, 0);
#pragma unroll 4
  for (uint32_t i = threadIdx.x; i < blockIdx.x; i += kScanThreads) {
    const uint4 v = sums[i];
    bef = make_uint4(bef.x + v.x, bef.y + v.y, bef.z + v.z, bef.w + v.w);
  }
  scan_write(a, first, end, c, bef);
  if (a.fill_coords) coords_fill(a.co, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

// ---------------------------------------------------------------------------
// Emit: vertices and quads.  Each wave takes chunks of 64 consecutive active
// cells (in cell order), one lane per cell, and finds each cell's segment in
// the non-empty segment list (the chunk's first list entry comes from the
// scan; a window of 64 entries is searched with shuffles).  Per cell: edge
// crossing points, dual vertices (FP32, reference operation order) and
// quads.  A ring
// neighbour of an owned edge is active by construction; its record is found
// in O(1): the +x neighbour is the next record of the same segment (or the
// first of the next x-tile's segment), and in a neighbour row the rank of
// cell x is the group's first rank plus the population count of the group's
// active mask below x.

constexpr int kEmitThreads = 256;
// Words of LDS of an emit wave: 12 sums a lane, then its vertices (up to 4 of
// 3 words a cell) or quads (up to 3 of 4 words) on their way out.
constexpr uint32_t kEmitStage = 12 * kWave;

struct EmitArgs {
  EmitVol v;  // the volume (single-volume launches)
  uint32_t cap, nsegs;
  uint64_t max_chunks;  // capacity of chunk_ne
  const uint2 *seg_counts;
  const uint2 *seg_vq;
  const uint32_t *slots;
  const uint16_t *slot_q;
  const uint32_t *gmap;
  const uint2 *ne;
  const uint32_t *chunk_ne;
  const Totals *totals;
  uint32_t *emit_ctr;  // k_emit's chunk tickets: the ticket region (zero at launch)
};

// Arrays seen through the constant address space: loads at wave-uniform
// indices become scalar loads.  Only for arrays no kernel running at the
// same time writes.
__device__ __forceinline__ const __attribute__((address_space(4))) float *as_const(const float *p) {
  return (const __attribute__((address_space(4))) float *)p;
}
// Entry i of an array of uint2 through the constant address space.
__device__ __forceinline__ uint2 const_u2(const uint2 *p, uint32_t i) {
  const __attribute__((address_space(4))) uint32_t *w = (const __attribute__((address_space(4))) uint32_t *)p;
  return make_uint2(w[2 * i], w[2 * i + 1]);
}
// Entry i of an array of words.
__device__ __forceinline__ uint32_t const_u1(const uint32_t *p, uint32_t i) {
  return ((const __attribute__((address_space(4))) uint32_t *)p)[i];
}
// First word of entry i of an array of uint2.
__device__ __forceinline__ uint32_t const_u2x(const uint2 *p, uint32_t i) {
  return ((const __attribute__((address_space(4))) uint32_t *)p)[2 * i];
}

// Kernel arguments and volume descriptors seen through the constant address
// space; fresh() makes the compiler read the fields used after it again (into
// scalar registers) instead of keeping them from before.
typedef const __attribute__((address_space(4))) EmitArgs *EmitArgsK;
typedef const __attribute__((address_space(4))) EmitVol *EmitVolK;
__device__ __forceinline__ const EmitArgs &fresh(EmitArgsK p) {
  asm volatile("" : "+s"(p));
  return *(const EmitArgs *)p;
}
__device__ __forceinline__ const EmitVol &fresh(EmitVolK p) {
  asm volatile("" : "+s"(p));
  return *(const EmitVol *)p;
}

// Address `off` bytes after a wave-uniform base.
template <class T>
__device__ __forceinline__ const T *at_off(const void *base, uint32_t off) {
  return reinterpret_cast<const T *>(static_cast<const char *>(base) + off);
}
template <class T>
__device__ __forceinline__ T *at_off(void *base, uint32_t off) {
  return reinterpret_cast<T *>(static_cast<char *>(base) + off);
}

// Two consecutive words or floats, and a vertex, at the alignment of one word.
typedef uint32_t Word2 __attribute__((ext_vector_type(2), aligned(4)));
typedef float Float2 __attribute__((ext_vector_type(2), aligned(4)));
struct Float3 {  // (a 3-vector type would be stored as 4 words)
  float x, y, z;
};
typedef int Int4 __attribute__((ext_vector_type(4)));
// (a volume's vertices begin at any multiple of 12 bytes)
typedef int Int4Row __attribute__((ext_vector_type(4), aligned(4)));

// The active cells of the calling lanes (segment s, rank within it) of volume
// vol: their vertices and the quads of their owned edges.  s0: the segment of
// the first of these lanes (uniform); all lanes' segments lie in [s0, s0 +
// vol.span], so everything a lane addresses is a uniform base, taken for s0,
// plus a 32-bit lane offset.  base: the volume's first vertex and quad.  (64-bit address arithmetic per lane and load, and
// the division of a segment number into tile, row and plane on every lane,
// were a quarter of the kernel's issue slots.)  s_lab: 512 entries (emit_label).
__device__ __forceinline__ void emit_cells(EmitArgsK pa, EmitVolK pv, uint2 base, uint32_t s0, uint32_t s,
                                           uint32_t rank, const uint64_t *s_lab, float *s_wave) {
  const EmitArgs &a = fresh(pa);
  const EmitVol &vol = fresh(pv);
  const FieldDesc &g = vol.g;
  const float iso = g.iso;
  const uint32_t cap = a.cap;
  const size_t sy = g.X, sz = (size_t)g.X * g.Y;
  const uint32_t d = s - s0;
  // this cell's record and the next active one's of its segment
  const uint32_t *const rec0 = a.slots + (size_t)s0 * cap;
  const uint32_t roff = d * cap + rank;
  const Word2 own = *at_off<Word2>(rec0, roff * 4u);
  const uint32_t lqb = *at_off<uint16_t>(a.slot_q + (size_t)s0 * cap, roff * 2u);
  // What depends only on the segment (its bases and count, the row's y and z
  // coordinates) comes through scalar loads for the lanes in s0 and through
  // vector loads for the rest (these arrays are read-only in the emit).  s0u:
  // s0 in a scalar register that the compiler cannot equate with s, so that on
  // the lanes where s == s0 it does not turn the scalar loads back into
  // per-lane vector loads at s.
  uint32_t s0u = s0;
  asm volatile("" : "+s"(s0u));
  const uint32_t sl0 = s0u - vol.seg_off;
  const uint32_t row0 = div_by(sl0, vol.div_xt), xt0 = sl0 - row0 * vol.XT;
  const uint32_t k0 = div_by(row0, vol.div_cy), j0 = row0 - k0 * g.cy;
  uint2 vq = const_u2(a.seg_vq, s0u);
  uint32_t nact = const_u2x(a.seg_counts, s0u) & 0xFFFFu;
  float Y0 = as_const(vol.yt_c)[j0], Y1 = as_const(vol.yt_c)[j0 + 1];
  float Z0 = as_const(vol.zt_c)[k0], Z1 = as_const(vol.zt_c)[k0 + 1];
  uint32_t xt = xt0, j = j0, k = k0, prow = 0;  // prow: point rows after (j0, k0)
  if (d != 0u) {
    const uint32_t sl = s - vol.seg_off, row = div_by(sl, vol.div_xt);
    xt = sl - row * vol.XT;
    k = div_by(row, vol.div_cy);
    j = row - k * g.cy;
    prow = (k - k0) * g.Y + j - j0;
    vq = *at_off<uint2>(a.seg_vq + s0, d * 8u);
    nact = at_off<uint2>(a.seg_counts + s0, d * 8u)->x & 0xFFFFu;
    const Float2 yy = *at_off<Float2>(vol.yt_c, j * 4u), zz = *at_off<Float2>(vol.zt_c, k * 4u);
    Y0 = yy.x;
    Y1 = yy.y;
    Z0 = zz.x;
    Z1 = zz.y;
  }
  const uint32_t rec = own.x;
  const uint32_t xl = rec_x(rec), cfg = rec_cfg(rec);
  const uint32_t x = xt * cap + xl;
  // a rank past the segment's count means inconsistent count-pass data
  if (x >= g.cx || xl >= cap || rank >= nact) { atomicOr(vol.status, kStatusInternal); return; }
  if (k < vol.kmin || k >= vol.kmax) return;

  // the cell's four point pairs along x
  const float *const p = g.f + (size_t)k0 * sz + (size_t)j0 * sy + (size_t)xt0 * cap;
  const uint32_t poff = (prow * g.X + x - xt0 * cap) * 4u;
  const Float2 v01 = *at_off<Float2>(p, poff), v32 = *at_off<Float2>(p + sy, poff);
  const Float2 v45 = *at_off<Float2>(p + sz, poff), v76 = *at_off<Float2>(p + sz + sy, poff);
  const Float2 xx = *at_off<Float2>(vol.xt_c, x * 4u);
  const float v[8] = {v01.x, v01.y, v32.y, v32.x, v45.x, v45.y, v76.y, v76.x};
  const float X0 = xx.x, X1 = xx.y;

  // first vertex and quad (numbers of the volume), and as offsets from those of
  // the first lane: a chunk's cells are consecutive, so the offsets are small
  const uint32_t vb = vq.x + rec_lvb(rec) - base.x, qb = vq.y + lqb - base.y;
  const uint32_t vb0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)vb);
  const uint32_t qb0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)qb);
  uint32_t dvq = (vb - vb0) | ((qb - qb0) << 16);
  if (vb - vb0 >= 1024u || qb - qb0 >= 1024u) { atomicOr(vol.status, kStatusInternal); return; }
  // what the quads need of the position, kept as lane masks over the vertices
  const bool xin = x + 1 < g.cx, yin = j + 1 < g.cy, zin = k + 1 < g.cz, n0in = rank + 1u < nact;
  asm volatile("" : "+v"(dvq));  // (one register, not its two halves)

  // Edge e runs from corner EF[e] to corner ET[e]: the orientation its
  // owning cell uses (owner edge 6: p2->p6, 9: p5->p6, 10: p6->p7), so the
  // point is bitwise the one the owner writes (dmc.cu:1468-1514).
  constexpr uint8_t EF[12] = {1, 1, 2, 0, 0, 1, 2, 3, 5, 5, 6, 4};
  constexpr uint8_t ET[12] = {0, 2, 3, 3, 4, 5, 6, 7, 4, 6, 7, 7};
  // Owner of each edge lies at a non-positive offset; an edge is skipped
  // when its owner would be outside the grid (dmc.cu:1539-1545): edges that
  // need a cell at -x (0x898), -y (0x131), -z (0x00F)
  const uint64_t labels = s_lab[(rec >> 10) & 0x1FFu];
  const uint32_t lab_hi = (uint32_t)(labels >> 32);
  const uint32_t niso = (lab_hi >> 16) & 0xFu;
  uint32_t use = lab_hi >> 20;  // crossed edges whose owner is in the grid
  if (x == 0u) use &= ~0x898u;
  if (j == 0u) use &= ~0x131u;
  if (k == 0u) use &= ~0x00Fu;
  // Group sums live in the wave's part of LDS, component c of group q of a lane
  // at s_acc[(3q + c) * T].  They start at -0.0, so the first addition yields
  // the point itself bitwise, as the reference's "assign the first, add the
  // rest" does.
  constexpr uint32_t T = kWave;
  float *const s_acc = s_wave + lane_id();
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if ((uint32_t)q < niso) {
      s_acc[(3 * q + 0) * T] = -0.0f;
      s_acc[(3 * q + 1) * T] = -0.0f;
      s_acc[(3 * q + 2) * T] = -0.0f;
    }
  }
  uint32_t cnt = 0;  // 8 bits per group
  float ex[3] = {0, 0, 0}, ey[3] = {0, 0, 0}, ez[3] = {0, 0, 0};
#pragma unroll
  for (int e = 0; e < 12; ++e) {
    // (edges 6, 9, 10 are the cell's own: used whenever crossed)
    if (!((use >> e) & 1u)) continue;
    const uint32_t lab = (e < 8 ? (uint32_t)labels >> (4 * e) : lab_hi >> (4 * e - 32)) & 0xFu;
    const int f = EF[e], to = ET[e];
    const float vf = v[f], vt = v[to];
    const float tt = (iso - vf) / (vt - vf);
    const float omt = 1.0f - tt;
    const float fx = (f == 1 || f == 2 || f == 5 || f == 6) ? X1 : X0;
    const float fy = (f == 2 || f == 3 || f == 6 || f == 7) ? Y1 : Y0;
    const float fz = (f >= 4) ? Z1 : Z0;
    const float tx = (to == 1 || to == 2 || to == 5 || to == 6) ? X1 : X0;
    const float ty = (to == 2 || to == 3 || to == 6 || to == 7) ? Y1 : Y0;
    const float tz = (to >= 4) ? Z1 : Z0;
    const float px = fx * omt + tx * tt;
    const float py = fy * omt + ty * tt;
    const float pz = fz * omt + tz * tt;
    if (e == 6) { ex[0] = px; ey[0] = py; ez[0] = pz; }
    if (e == 9) { ex[1] = px; ey[1] = py; ez[1] = pz; }
    if (e == 10) { ex[2] = px; ey[2] = py; ez[2] = pz; }
    float *acc = s_acc + 3 * lab * T;
    acc[0] = acc[0] + px;
    acc[T] = acc[T] + py;
    acc[2 * T] = acc[2 * T] + pz;
    cnt += 1u << (8 * lab);
  }
  const uint32_t b6 = (use >> 6) & 1u, b9 = (use >> 9) & 1u, b10 = (use >> 10) & 1u;
  const uint32_t nv = niso + b6 + b9 + b10, dv = dvq & 0xFFFFu;
  const uint64_t lanes = __ballot(true);
  const uint32_t idx = mbcnt64(lanes), nlanes = (uint32_t)__popcll(lanes);
  float *const out = vol.verts + 3ull * vb0;
  const float qnan = __int_as_float(0x7FC00000);
  const bool vfit = (uint64_t)vb0 + dv + nv <= vol.vcap;
  if (__ballot(niso != 1u || dv + nv > kEmitStage / 3u) == 0ull) {
    // One iso vertex in every cell (nearly all chunks): the vertices are put
    // in order in the wave's part of LDS and leave as whole lines, 16 bytes a
    // lane whatever the alignment.  A store per lane and vertex touches a
    // dozen lines each time, four times over.  The stores are nontemporal:
    // nothing here reads the mesh again, and at twice the field's bytes it
    // pushed the field's rows and the records out of the XCD's L2 before the
    // next plane's chunks asked for them (512^3 gyroid: 9.5 -> 6.5 million line
    // reads from memory; emit 634 -> 600 us, 1024^3 5.00 -> 4.72 ms of which
    // the wider stores alone give 0.2, 300x281x260 100 -> 92 us).
    const uint32_t n = cnt & 0xFFu;
    const float dn = (float)n;
    const Float3 r{n ? s_acc[0] / dn : qnan, n ? s_acc[T] / dn : qnan, n ? s_acc[2 * T] / dn : qnan};
    auto put = [&]() {
      if (!vfit) return;
      Float3 *st = reinterpret_cast<Float3 *>(s_wave + 3u * dv);
      *st++ = r;
      if (b6) *st++ = Float3{ex[0], ey[0], ez[0]};
      if (b9) *st++ = Float3{ex[1], ey[1], ez[1]};
      if (b10) *st = Float3{ex[2], ey[2], ez[2]};
    };
    auto copy = [&]() {
      const uint64_t fits = __ballot(vfit);
      const uint32_t total = fits ? (uint32_t)__builtin_amdgcn_readlane((int)(dv + nv), 63 - __builtin_clzll(fits)) : 0u;
      const uint32_t words = 3u * total, tail = words & ~3u;
      for (uint32_t i = 4u * idx; i < tail; i += 4u * nlanes)
        __builtin_nontemporal_store(*reinterpret_cast<const Int4 *>(s_wave + i), at_off<Int4Row>(out, i * 4u));
      for (uint32_t i = tail + idx; i < words; i += nlanes) __builtin_nontemporal_store(s_wave[i], at_off<float>(out, i * 4u));
    };
    wave_exchange(put, copy, WaveOrder());
  } else if (vfit) {
    uint32_t o = dv * 12u;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if ((uint32_t)q < niso) {
        const uint32_t n = (cnt >> (8 * q)) & 0xFFu;
        const float dn = (float)n;
        Float3 r;
        r.x = n ? s_acc[(3 * q + 0) * T] / dn : qnan;
        r.y = n ? s_acc[(3 * q + 1) * T] / dn : qnan;
        r.z = n ? s_acc[(3 * q + 2) * T] / dn : qnan;
        *at_off<Float3>(out, o + 12u * q) = r;
      }
    }
    o += niso * 12u;
    if (b6) { *at_off<Float3>(out, o) = Float3{ex[0], ey[0], ez[0]}; o += 12u; }
    if (b9) { *at_off<Float3>(out, o) = Float3{ex[1], ey[1], ez[1]}; o += 12u; }
    if (b10) *at_off<Float3>(out, o) = Float3{ex[2], ey[2], ez[2]};
  }
  if (!vfit) atomicOr(vol.status, kStatusVertexOverflow);

  // Quads (dmc.cu:1983-2047): rings in ccw order, reversed (0,3,2,1) when
  // the owned edge's first corner is not above iso.  The arguments are read
  // again (scalar loads that hit the cache) instead of staying in registers
  // over the vertices.
  const EmitArgs &aq = fresh(pa);
  const EmitVol &vq_ = fresh(pv);
  const bool e6 = b6 && xin && yin, e9 = b9 && xin && zin, e10 = b10 && yin && zin;
  if (__ballot(e6 || e9 || e10) == 0ull) return;
  const uint32_t nq = (uint32_t)e6 + (uint32_t)e9 + (uint32_t)e10, dq = dvq >> 16;
  // Ring cells n = 0 (+1,0,0), 1 (0,+1,0), 2 (0,0,+1), 3 (+1,+1,0),
  // 4 (+1,0,+1), 5 (0,+1,+1).  A ring cell contains the crossing edge, so it
  // is active.  Cells 1, 2 and 5 are found through their segments' group
  // maps.  Cells 0, 3 and 4 follow from this cell, 1 and 2: a ring cell and
  // its -x neighbour in the ring are both active, so the +x one is the next
  // active cell of its row, read with it (the first of the next x-tile's
  // segment when x is the tile's last cell).  Each record's x field confirms
  // the cell found.  A lookup the quads do not need reads at offset 0 of a
  // segment in range, so that every load is in bounds.
  const bool need1 = e6 || e10, need2 = e9 || e10, need5 = e10;
  const uint32_t capq = aq.cap, G = capq >> 4, dy = vq_.XT, dz = vq_.XT * vq_.g.cy, last = aq.nsegs - 1u;
  const uint32_t b1 = min(s0u + dy, last), b2 = min(s0u + dz, last), b5 = min(s0u + dy + dz, last);
  const uint32_t goff = (d * G + (xl >> 4)) * 4u;
  const uint32_t g1 = *at_off<uint32_t>(aq.gmap + (size_t)b1 * G, need1 ? goff : 0u);
  const uint32_t g2 = *at_off<uint32_t>(aq.gmap + (size_t)b2 * G, need2 ? goff : 0u);
  const uint32_t g5 = *at_off<uint32_t>(aq.gmap + (size_t)b5 * G, need5 ? goff : 0u);
  uint32_t vq1 = const_u2x(aq.seg_vq, b1), vq2 = const_u2x(aq.seg_vq, b2), vq5 = const_u2x(aq.seg_vq, b5);
  if (d != 0u) {
    vq1 = at_off<uint2>(aq.seg_vq + b1, need1 ? d * 8u : 0u)->x;
    vq2 = at_off<uint2>(aq.seg_vq + b2, need2 ? d * 8u : 0u)->x;
    vq5 = at_off<uint2>(aq.seg_vq + b5, need5 ? d * 8u : 0u)->x;
  }
  const uint32_t bit = xl & 15u, below = (1u << bit) - 1u;
  auto rank_of = [&](uint32_t gm) {  // (clamped: a group map may be stale where the lane needs no lookup)
    return min((gm >> 16) + (uint32_t)__popc(gm & below), capq - 1u);
  };
  auto in_map = [&](uint32_t gm) { return ((gm >> bit) & 1u) != 0u; };
  const uint32_t r1 = rank_of(g1), r2 = rank_of(g2), r5 = rank_of(g5);
  const Word2 c13 = *at_off<Word2>(aq.slots + (size_t)b1 * capq, need1 ? (d * capq + r1) * 4u : 0u);
  const Word2 c24 = *at_off<Word2>(aq.slots + (size_t)b2 * capq, need2 ? (d * capq + r2) * 4u : 0u);
  const uint32_t c5 = *at_off<uint32_t>(aq.slots + (size_t)b5 * capq, need5 ? (d * capq + r5) * 4u : 0u);
  uint32_t c0 = own.y, c3 = c13.y, c4 = c24.y, vq0 = vq.x, vq3 = vq1, vq4 = vq2, xn = xl + 1u;
  // the next active cell of a row is in the segment only if its count says so
  bool n0 = n0in, n3 = r1 + 1u < capq, n4 = r2 + 1u < capq;
  if (xn == capq) {  // +x lies in the next x-tile's segments of this row, row y + 1 and plane z + 1
    xn = 0u;
    n0 = n3 = n4 = true;
    uint32_t sn = s0 + d + 1u;
    asm volatile("" : "+v"(sn));  // (keeps the addresses below out of the lanes' common path)
    if (e6 || e9) {
      c0 = aq.slots[(size_t)sn * capq];
      vq0 = aq.seg_vq[sn].x;
    }
    if (e6) {
      c3 = aq.slots[(size_t)(sn + dy) * capq];
      vq3 = aq.seg_vq[sn + dy].x;
    }
    if (e9) {
      c4 = aq.slots[(size_t)(sn + dz) * capq];
      vq4 = aq.seg_vq[sn + dz].x;
    }
  }
  const bool ok0 = n0 && rec_x(c0) == xn, ok3 = n3 && rec_x(c3) == xn, ok4 = n4 && rec_x(c4) == xn;
  const bool ok1 = in_map(g1) && rec_x(c13.x) == xl, ok2 = in_map(g2) && rec_x(c24.x) == xl;
  const bool ok5 = in_map(g5) && rec_x(c5) == xl;
  bool ok = true;
  // vertex of a ring cell (record m, its segment's first vertex vqn) for its local edge e
  const uint32_t *const s_lab32 = reinterpret_cast<const uint32_t *>(s_lab);
  const uint32_t shift = vq_.vshift - base.x;
  auto vtx = [&](uint32_t m, uint32_t vqn, int e, bool found) -> int32_t {
    const uint32_t lab = (s_lab32[2u * ((m >> 10) & 0x1FFu) + (e >> 3)] >> (4 * (e & 7))) & 0xFu;
    if (!found || lab == 0xFu) ok = false;
    return (int32_t)(vqn + rec_lvb(m) + lab + shift);
  };
  // in order in the wave's part of LDS (like the vertices, 3 quads a cell fit)
  const bool qfit = (uint64_t)qb0 + dq + nq <= vq_.qcap && dq + nq <= kEmitStage / 4u;
  Int4 *st = reinterpret_cast<Int4 *>(s_wave) + (qfit ? dq : 0u);
  const int32_t self = (int32_t)(vb0 + (dvq & 0xFFFFu) + vq_.vshift);
  auto put = [&]() {
    if (e6) {
      const int32_t m0 = self + (int32_t)(((uint32_t)labels >> 24) & 0xFu);
      const int32_t m1 = vtx(c0, vq0, 7, ok0), m2 = vtx(c3, vq3, 4, ok3), m3 = vtx(c13.x, vq1, 5, ok1);
      if (qfit) *st++ = v[2] <= vq_.g.iso ? Int4{m0, m1, m2, m3} : Int4{m0, m3, m2, m1};
    }
    if (e9) {
      const int32_t m0 = self + (int32_t)((lab_hi >> 4) & 0xFu);
      const int32_t m1 = vtx(c24.x, vq2, 1, ok2), m2 = vtx(c4, vq4, 3, ok4), m3 = vtx(c0, vq0, 11, ok0);
      if (qfit) *st++ = v[5] <= vq_.g.iso ? Int4{m0, m1, m2, m3} : Int4{m0, m3, m2, m1};
    }
    if (e10) {
      const int32_t m0 = self + (int32_t)((lab_hi >> 8) & 0xFu);
      const int32_t m1 = vtx(c13.x, vq1, 8, ok1), m2 = vtx(c5, vq5, 0, ok5), m3 = vtx(c24.x, vq2, 2, ok2);
      if (qfit) *st++ = v[7] <= vq_.g.iso ? Int4{m0, m1, m2, m3} : Int4{m0, m3, m2, m1};
    }
  };
  auto copy = [&]() {
    const uint64_t fits = __ballot(qfit);
    const uint32_t total = fits ? (uint32_t)__builtin_amdgcn_readlane((int)(dq + nq), 63 - __builtin_clzll(fits)) : 0u;
    int32_t *const qout = vq_.quads + 4ull * qb0;
    for (uint32_t i = idx; i < total; i += nlanes)
      __builtin_nontemporal_store(reinterpret_cast<const Int4 *>(s_wave)[i], at_off<Int4>(qout, i * 16u));
  };
  wave_exchange(put, copy, WaveOrder());
  if (!qfit && nq) atomicOr(vq_.status, kStatusQuadOverflow);
  if (!ok) atomicOr(vq_.status, kStatusLookup);
}

// The lanes with a cell (todo), in runs whose segments lie within vol.span of
// their first lane's (nearly always one run).
__device__ __forceinline__ void emit_lanes(EmitArgsK pa, EmitVolK pv, uint2 base, bool todo, uint32_t s, uint32_t rank,
                                           const uint64_t *s_lab, float *s_wave) {
  for (uint64_t left = __ballot(todo); left != 0ull; left = __ballot(todo)) {
    const uint32_t s0 = (uint32_t)__builtin_amdgcn_readlane((int)s, __ffsll((long long)left) - 1);
    const bool mine = todo && s - s0 <= fresh(pv).span;
    if (mine) emit_cells(pa, pv, base, s0, s, rank, s_lab, s_wave);
    todo = todo && !mine;
  }
}

// Entry i of the emit's table in LDS, by configuration and variant: the label
// nibbles of edges 0..11, the number of iso vertices (bits 48-51) and the
// crossed edges (bits 52-63).
__device__ __forceinline__ uint64_t emit_label(uint32_t i) {
  const uint64_t l = (&c_label[0][0])[i];
  const uint32_t info = c_cfg_info[i & 255u], n = i >= 256u ? (info >> 3) & 7u : info & 7u;
  uint64_t cross = 0;
#pragma unroll
  for (int e = 0; e < 12; ++e) cross |= (uint64_t)(((l >> (4 * e)) & 0xFu) != 0xFu) << e;
  return (l & 0xFFFFFFFFFFFFull) | ((uint64_t)n << 48) | (cross << 52);
}

// Segment and rank of active cell ch*64 + lane: the chunk's first entry of
// the non-empty list comes from the scan, and a window of 64 entries is
// searched with shuffles (all lanes take part).  False for lanes past the
// last cell and for inconsistent inputs (reported in the status word).
__device__ __forceinline__ bool locate_cell(const EmitArgs &a, const Totals &tot, uint32_t num_ne,
                                            uint32_t ch, uint32_t lane, uint32_t &s, uint32_t &rank) {
  const uint32_t act = ch * 64u + lane;
  const uint32_t u0 = const_u1(a.chunk_ne, (uint32_t)__builtin_amdgcn_readfirstlane((int)ch));  // (ch is uniform)
  const uint2 wl = (u0 < num_ne && u0 + lane <= num_ne) ? a.ne[u0 + lane] : make_uint2(0u, 0xFFFFFFFFu);
  uint32_t m = 0;
#pragma unroll
  for (uint32_t step = 32; step >= 1; step >>= 1) {
    const uint32_t cand = m + step;
    const uint32_t wc = (uint32_t)__shfl((int)wl.y, (int)(cand & 63u), kWave);
    if (cand < 64u && wc <= act) m = cand;
  }
  const uint32_t ap = (uint32_t)__shfl((int)wl.y, (int)m, kWave);
  s = (uint32_t)__shfl((int)wl.x, (int)m, kWave);
  if (act >= tot.num_active) return false;
  rank = act - ap;
  // (the rank is checked against the segment's count by the caller, whose
  // loads that check rides along with)
  if (u0 >= num_ne || u0 + m >= num_ne || s >= a.nsegs || act < ap || rank >= a.cap) {
    atomicOr(a.v.status, kStatusInternal);
    return false;
  }
  return true;
}

// Chunks of a wave.  Workgroups are dispatched round-robin over the 8 XCDs
// (workgroup b runs on XCD b % 8); with at least 8 workgroups, XCD x takes
// the contiguous chunk range [x n / 8, (x + 1) n / 8) and its workgroups
// stride through it, so that neighbouring chunks, which share field rows and
// the records of neighbour segments, meet in one L2.
struct ChunkIter {
  uint32_t next, end, step;
};

__device__ __forceinline__ ChunkIter chunk_iter(uint32_t n, uint32_t wave) {
  constexpr uint32_t wpb = kEmitThreads / kWave;
  const uint32_t G = gridDim.x;
  if (G < 8u) return ChunkIter{blockIdx.x * wpb + wave, n, G * wpb};
  const uint32_t x = blockIdx.x & 7u, slot = blockIdx.x >> 3;
  const uint32_t gx = (G >> 3) + (x < (G & 7u) ? 1u : 0u);
  const uint32_t lo = (uint32_t)((uint64_t)n * x / 8u), hi = (uint32_t)((uint64_t)n * (x + 1u) / 8u);
  return ChunkIter{lo + slot * wpb + wave, hi, gx * wpb};
}

// Emit grid: at most this many workgroups per CU (MDMC_OPT_EMIT_BLOCKS_PER_CU
// overrides it).  The grid is sized for the chunk capacity because the count
// is still on the device when the emit is launched; on a surface-dense 1024^3
// field 128 per CU beat 8 by 8% (more, shorter-lived workgroups keep each
// XCD's chunks in dispatch order), and past 256 the workgroups that find no
// chunk cost a sparse extraction several microseconds.
constexpr int kEmitBlocksPerCu = 128;

// Whether any wave of this workgroup has a chunk (its wave 0 has the lowest
// one).  The grid is sized for the chunk capacity, so when the mesh is
// sparse most workgroups leave at once, before loading their tables.
__device__ __forceinline__ bool workgroup_has_chunks(uint32_t n) {
  const ChunkIter it = chunk_iter(n, 0);
  return it.next < it.end;
}

// Single-volume emit grid: a persistent grid of this many workgroups per CU
// (MDMC_OPT_EMIT_BLOCKS_PER_CU overrides it), the most that are resident at
// once at 8 waves per SIMD.
constexpr int kEmitPersistPerCu = 8;

// 8 waves per SIMD: the emit is latency-bound, the register cap costs a few
// scalar spills only.  Chunks come by ticket (emit_tickets, mdmc_tilemap.h):
// workgroups are dispatched round-robin over the 8 XCDs (workgroup b runs on
// XCD b % 8), so the chunks in flight on an XCD stay one contiguous window
// that moves through its range in order, and neighbouring chunks, which share
// field rows and the records of neighbour segments, meet in its L2 while both
// are in flight; the next ticket is asked for before the current one's
// chunks run and read after them, so its latency hides under the work.  The
// placement only shapes locality: any mapping of workgroups to XCDs takes
// every chunk exactly once.  The grid is a multiple of 8 workgroups, and the
// ticket counters are zero at launch (the classify zeroes them; the host
// zeroes them again before an emit that follows another).
__global__ __launch_bounds__(kEmitThreads) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_emit(EmitArgs a) {
  constexpr uint32_t wpb = kEmitThreads / kWave;
  __shared__ uint64_t s_lab[2 * 256];
  __shared__ __align__(16) float s_acc[kEmitStage * wpb];
  __shared__ uint32_t s_ticket[2];
  const Totals tot = *a.totals;
  // Counts are clamped to buffer capacities so that no access can leave the
  // scratch buffers even if the count pass produced inconsistent data.
  const uint32_t num_chunks = (uint32_t)min((uint64_t)tot.num_chunks, a.max_chunks);
  const EmitTickets et = emit_tickets(num_chunks, blockIdx.x & 7u, gridDim.x, wpb);
  uint64_t first = emit_ticket_chunk(et, blockIdx.x >> 3, wpb);
  if (first >= et.hi) return;  // (uniform: before the barrier)
  for (uint32_t i = threadIdx.x; i < 512; i += kEmitThreads) s_lab[i] = emit_label(i);
  uint32_t *ctr = a.emit_ctr + kEmitCtr * ((blockIdx.x & 7u) + 1u);
  __syncthreads();
  const uint32_t lane = lane_id(), wave = wave_id();
  const uint32_t num_ne = min(tot.num_nonempty, a.nsegs);
  const EmitArgsK pa = (EmitArgsK)__builtin_amdgcn_kernarg_segment_ptr();  // a
  const uint2 base = make_uint2(a.v.vbase, a.v.qbase);
  for (uint32_t it = 0;; ++it) {
    // the next ticket is asked for before this one's chunks run and published
    // after them; two slots, because thread 0 writes the next iteration's
    // only after every thread has passed this iteration's barrier
    uint32_t next = 0;
    if (et.dynamic && threadIdx.x == 0) next = atomicAdd(ctr, 1u);
    const uint64_t ch = first + wave;
    if (ch < et.hi) {
      uint32_t s = 0, rank = 0;
      const bool found = locate_cell(a, tot, num_ne, (uint32_t)ch, lane, s, rank);
      emit_lanes(pa, &pa->v, base, found, s, rank, s_lab, s_acc + kEmitStage * wave);
    }
    if (!et.dynamic) break;
    if (threadIdx.x == 0) s_ticket[it & 1u] = next;
    __syncthreads();
    first = emit_ticket_chunk(et, (uint64_t)et.slots + s_ticket[it & 1u], wpb);
    if (first >= et.hi) break;
  }
}

// Zeroes the emit's ticket counters (one workgroup of 64 threads).
__global__ void k_zero_tickets(uint32_t *t) { zero_tickets(t, threadIdx.x); }


// ---------------------------------------------------------------------------
// Smoothing (num_smooth > 0): smooth_edge_vertices (dmc.cu:1868-1981) then
// calc_iso_vertices_kern again (dmc.cu:1517-1593, 2157-2169), per iteration.
// Both run over the emitted mesh, one lane per active cell in the emit's
// chunks.  k_smooth moves owned edge points (reading iso vertices only);
// k_reaverage recomputes iso vertices from the stored edge points (reading
// edge points only), so neither reads what it writes.
//
// Each pass rewrites every other vertex of the mesh, so it moves all of its
// lines twice: on 3.4 M cells (256x240x272 gyroid) k_smooth moves 244 MB (52 us
// at a large copy's rate) and takes 84 us with VALU issue on at most 84% of its
// cycles (92 us with two differences, products and a root per corner instead of
// per edge and integer divisions for the position); k_reaverage moves 186 MB
// (40 us) and takes 68 us, a chain of lookups with VALU issue on at most 85%
// (83 us with a gather for each of the 12 edges, a third of the address units'
// work for nothing).
//
// The split of a convex ring is at the corner of the largest angle, taken as
// the smallest cosine (a.b) / (sqrt(a.a) sqrt(b.b)) with IEEE sqrt and
// division, first smallest wins (the reference takes acosf of rsqrtf-
// normalised vectors, dmc.cu:1818-1860); everything else is the reference's
// float operation sequence.

// Position of an active cell from its segment.
struct CellPos {
  uint32_t xl, cfg, lut2, x, j, k, vb, qb;
  uint32_t seg_vb;  // the segment's first vertex
  uint32_t nact;    // the segment's active cells
  float y1, z1;     // coordinates of point row j + 1 and plane k + 1
};

// As in the emit, what depends only on the segment (its bases and count, the
// row's coordinates) comes through scalar loads for the lanes in the wave's
// first segment and through vector loads for the others.
__device__ __forceinline__ CellPos cell_pos(const EmitArgs &a, const EmitVol &vol, uint32_t s, uint32_t rank,
                                            uint32_t &rec) {
  CellPos c;
  rec = a.slots[(size_t)s * a.cap + rank];
  c.xl = rec_x(rec);
  c.cfg = rec_cfg(rec);
  c.lut2 = rec_lut2(rec);
  const uint32_t sl = s - vol.seg_off;
  const uint32_t row = div_by(sl, vol.div_xt), xt = sl - row * vol.XT;
  c.k = div_by(row, vol.div_cy);
  c.j = row - c.k * vol.g.cy;
  c.x = xt * a.cap + c.xl;
  const uint32_t s0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)s);
  uint32_t s0u = s0;
  asm volatile("" : "+s"(s0u));
  const uint32_t row0 = div_by(s0u - vol.seg_off, vol.div_xt), k0 = div_by(row0, vol.div_cy);
  uint2 vq = const_u2(a.seg_vq, s0u);
  uint32_t nact = const_u2x(a.seg_counts, s0u) & 0xFFFFu;
  float y1 = as_const(vol.yt_c)[row0 - k0 * vol.g.cy + 1u], z1 = as_const(vol.zt_c)[k0 + 1u];
  if (s != s0) {
    vq = a.seg_vq[s];
    nact = a.seg_counts[s].x & 0xFFFFu;
    y1 = vol.yt_c[c.j + 1u];
    z1 = vol.zt_c[c.k + 1u];
  }
  c.seg_vb = vq.x;
  c.nact = nact;
  c.y1 = y1;
  c.z1 = z1;
  c.vb = vq.x + rec_lvb(rec) - vol.vbase;
  c.qb = vq.y + a.slot_q[(size_t)s * a.cap + rank] - vol.qbase;
  return c;
}

__device__ __forceinline__ uint32_t iso_count(uint32_t cfg, uint32_t lut2) {
  const uint32_t info = c_cfg_info[cfg];
  return lut2 ? ((info >> 3) & 7u) : (info & 7u);
}

// bipolar owned edges 6, 9, 10 of a configuration, as bits 0, 1, 2
__device__ __forceinline__ uint32_t owned_bipolar(uint32_t cfg) {
  return (((cfg >> 2) ^ (cfg >> 6)) & 1u) | ((((cfg >> 5) ^ (cfg >> 6)) & 1u) << 1) |
         ((((cfg >> 7) ^ (cfg >> 6)) & 1u) << 2);
}

struct P2 {
  float x, y;
};

// is_inside_triangle (dmc.cu:1894-1912)
__device__ __forceinline__ bool inside_tri(P2 p0, P2 p1, P2 p2, P2 t, float &al, float &be, float &ga) {
  const float v0x = p1.x - p0.x, v0y = p1.y - p0.y, v1x = p2.x - p0.x, v1y = p2.y - p0.y;
  const float v2x = t.x - p0.x, v2y = t.y - p0.y;
  const float d00 = v0x * v0x + v0y * v0y, d10 = v1x * v0x + v1y * v0y, d11 = v1x * v1x + v1y * v1y;
  const float d20 = v2x * v0x + v2y * v0y, d21 = v2x * v1x + v2y * v1y;
  const float inv = 1.0f / (d00 * d11 - d10 * d10);
  be = (d11 * d20 - d10 * d21) * inv;
  ga = (d00 * d21 - d10 * d20) * inv;
  al = 1.0f - be - ga;
  // The reference compares with the doubles -1e-4 and 1 + 1e-4.  Both lie just
  // below the float nearest to them, so these comparisons decide alike.
  static_assert((double)-1e-4f > -1e-4 && (double)1.0001f > 1.0 + 1e-4, "float thresholds");
  return be >= -1e-4f && ga >= -1e-4f && be + ga < 1.0001f;
}

// v[t] for t in 0..3 by selects (no indexed register array)
__device__ __forceinline__ float sel4(uint32_t t, const float (&v)[4]) {
  const float lo = (t & 1u) ? v[1] : v[0], hi = (t & 1u) ? v[3] : v[2];
  return (t & 2u) ? hi : lo;
}

// One smoothing pass over the owned edge points of a chunk's cells (found:
// this lane has a cell).  The chunk's quads are spread over its lanes, one
// quad per lane per round: the lanes' quad counts are prefix-summed and lane
// L of round r takes quad r*64 + L from the lane that owns it (a shuffle
// search over the prefix).  Taking each cell's up-to-three quads on its own
// lane would run three divergent rounds in nearly every surface-dense chunk,
// where most cells own one quad.  Every lane takes part in the shuffles.
__device__ __forceinline__ void smooth_chunk(const EmitArgs &a, const EmitVol &vol, bool found, uint32_t s,
                                             uint32_t rank) {
  const FieldDesc &g = vol.g;
  uint32_t has = 0, bip = 0, qb = 0, ev0 = 0;
  float x1 = 0.0f, y1 = 0.0f, z1 = 0.0f;
  if (found) {
    uint32_t rec;
    const CellPos c = cell_pos(a, vol, s, rank, rec);
    if (c.x >= g.cx || rank >= c.nact) {
      atomicOr(vol.status, kStatusInternal);
    } else {
      bip = owned_bipolar(c.cfg);
      const bool xin = c.x + 1 < g.cx, yin = c.j + 1 < g.cy, zin = c.k + 1 < g.cz;
      has = ((bip & 1u) && xin && yin ? 1u : 0u) | ((bip & 2u) && xin && zin ? 2u : 0u) |
            ((bip & 4u) && yin && zin ? 4u : 0u);
      if (has) x1 = vol.xt_c[c.x + 1];
      y1 = c.y1;
      z1 = c.z1;
      qb = c.qb;
      ev0 = c.vb + iso_count(c.cfg, c.lut2);
    }
  }
  const uint32_t lane = lane_id();
  const uint32_t cnt = (uint32_t)__popc(has);
  const uint32_t incl = wave_incl_scan(cnt), off = incl - cnt;
  const uint32_t K = (uint32_t)__shfl((int)incl, kWave - 1, kWave);
  for (uint32_t base = 0; base < K; base += kWave) {
    const uint32_t jq = base + lane;
    // owner: the highest lane whose prefix is <= jq (for jq < K it owns jq)
    uint32_t m = 0;
#pragma unroll
    for (uint32_t step = 32; step >= 1; step >>= 1) {
      const uint32_t cand = m + step;
      const uint32_t oc = (uint32_t)__shfl((int)off, (int)(cand & 63u), kWave);
      if (cand < 64u && oc <= jq) m = cand;
    }
    const uint32_t o_off = (uint32_t)__shfl((int)off, (int)m, kWave);
    const uint32_t o_has = (uint32_t)__shfl((int)has, (int)m, kWave);
    const uint32_t o_bip = (uint32_t)__shfl((int)bip, (int)m, kWave);
    const uint32_t o_qb = (uint32_t)__shfl((int)qb, (int)m, kWave);
    const uint32_t o_ev0 = (uint32_t)__shfl((int)ev0, (int)m, kWave);
    const float o_x1 = __shfl(x1, (int)m, kWave), o_y1 = __shfl(y1, (int)m, kWave), o_z1 = __shfl(z1, (int)m, kWave);
    if (jq >= K) continue;
    // the owner's k-th quad is on its k-th set bit l of `has`
    const uint32_t kq = jq - o_off;
    uint32_t h = o_has;
    if (kq >= 1u) h &= h - 1u;
    if (kq >= 2u) h &= h - 1u;
    const uint32_t l = (uint32_t)__builtin_ctz(h);
    const uint32_t q = o_qb + kq;
    const uint32_t e_vtx = o_ev0 + (uint32_t)__popc(o_bip & ((1u << l) - 1u));
    if ((uint64_t)q >= vol.qcap || (uint64_t)e_vtx >= vol.vcap) { atomicOr(vol.status, kStatusInternal); continue; }
    const int4 rq = reinterpret_cast<const int4 *>(vol.quads)[q];
    const int32_t iv[4] = {rq.x, rq.y, rq.z, rq.w};
    // the ring's four iso vertices, read once (k_smooth writes edge points
    // only, so they do not change while it runs); the edge's plane: x-y for
    // e6 (l = 0), x-z for e9, y-z for e10
    float vx[4], vy[4], vz[4];
    P2 P[4];
    bool bad = false;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      bad |= iv[p] < 0 || (uint64_t)iv[p] >= vol.vcap;
      const float *vp = vol.verts + 3ull * (uint32_t)(bad ? 0 : iv[p]);
      vx[p] = vp[0];
      vy[p] = vp[1];
      vz[p] = vp[2];
      P[p].x = l == 2u ? vy[p] : vx[p];
      P[p].y = l == 0u ? vy[p] : vz[p];
    }
    if (bad) { atomicOr(vol.status, kStatusInternal); continue; }
    // Edge vectors E_p = P_p+1 - P_p.  With a = P_p-1 - P_p = -E_p-1 and b = E_p
    // the reference's cross product (calc_cross_z_sign, dmc.cu:1741-1747) and
    // dot product at corner p come out of E_p-1 and E_p up to signs, which
    // change no rounding, and each length serves two corners: 8 differences
    // and 4 square roots instead of 32 and 8.
    P2 E[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) E[p] = P2{P[(p + 1) & 3].x - P[p].x, P[(p + 1) & 3].y - P[p].y};
    // calc_quadrilateral_signs (dmc.cu:1749-1780)
    uint32_t npos = 0, ipos = 0, ineg = 0;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const P2 e = E[p], f = E[(p + 3) & 3];
      if (f.x * e.y - e.x * f.y >= 0.0f) { ++npos; ipos = p; }
      else ineg = p;
    }
    if (npos == 2) continue;  // self-crossing ring (dmc.cu:1783-1786)
    uint32_t s0;
    if (npos == 0 || npos == 4) {
      // (the smallest cosine is the largest of f.e / (|f| |e|))
      float len[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) len[p] = sqrtf(E[p].x * E[p].x + E[p].y * E[p].y);
      float best = (E[3].x * E[0].x + E[3].y * E[0].y) / (len[3] * len[0]);
      s0 = 0;
#pragma unroll
      for (int p = 1; p < 4; ++p) {
        const float c = (E[p - 1].x * E[p].x + E[p - 1].y * E[p].y) / (len[p - 1] * len[p]);
        if (c > best) { best = c; s0 = p; }
      }
    } else {
      s0 = npos < 2 ? ipos : ineg;  // the concave corner
    }
    const uint32_t s1 = (s0 + 2) & 3;
    const P2 o = l == 0u ? P2{o_x1, o_y1} : (l == 1u ? P2{o_x1, o_z1} : P2{o_y1, o_z1});
    float al, be, ga;
    uint32_t ta, tb, tc;
    if (inside_tri(P[s0], P[(s0 + 1) & 3], P[s1], o, al, be, ga)) {
      ta = s0; tb = (s0 + 1) & 3; tc = s1;
    } else if (inside_tri(P[s1], P[(s1 + 1) & 3], P[s0], o, al, be, ga)) {
      ta = s1; tb = (s1 + 1) & 3; tc = s0;
    } else {
      continue;
    }
    float *out = vol.verts + 3ull * e_vtx;
    const float r0 = al * sel4(ta, vx) + be * sel4(tb, vx) + ga * sel4(tc, vx);
    const float r1 = al * sel4(ta, vy) + be * sel4(tb, vy) + ga * sel4(tc, vy);
    const float r2 = al * sel4(ta, vz) + be * sel4(tb, vz) + ga * sel4(tc, vz);
    out[0] = r0;
    out[1] = r1;
    out[2] = r2;
  }
}

// Iso vertices from the stored edge points: for each edge of the cell in
// order 0..11 with a vertex and an in-grid owner, the owner's stored point
// (owner cells n = 0 (-1,0,0), 1 (0,-1,0), 2 (0,0,-1), 3 (-1,-1,0),
// 4 (-1,0,-1), 5 (0,-1,-1), found like the quad ring cells), summed per
// group from -0.0 and divided by the count; groups with no point keep their
// value.
__device__ __forceinline__ void reaverage_cell(const EmitArgs &a, const EmitVol &vol, uint32_t s, uint32_t rank,
                                               const uint64_t *s_lab, uint32_t *s_idx) {
  uint32_t rec;
  const CellPos c = cell_pos(a, vol, s, rank, rec);
  const FieldDesc &g = vol.g;
  const uint32_t cap = a.cap;
  if (c.x >= g.cx || c.xl >= cap || rank >= c.nact) {
    atomicOr(vol.status, kStatusInternal);
    return;
  }
  const uint32_t *const s_lab32 = reinterpret_cast<const uint32_t *>(s_lab);
  const uint64_t labels = s_lab[c.lut2 * 256 + c.cfg];
  const uint32_t lab_hi = (uint32_t)(labels >> 32), niso = (lab_hi >> 16) & 0xFu;
  // crossed edges whose owner is in the grid, as in the emit
  uint32_t use = lab_hi >> 20;
  if (c.x == 0u) use &= ~0x898u;
  if (c.j == 0u) use &= ~0x131u;
  if (c.k == 0u) use &= ~0x00Fu;
  // owner n's edges: 0: 7, 11; 1: 5, 8; 2: 1, 2; 3: 4; 4: 3; 5: 0
  constexpr uint32_t OWNED[6] = {0x880u, 0x120u, 0x006u, 0x010u, 0x008u, 0x001u};
  uint32_t need = 0;
#pragma unroll
  for (int n = 0; n < 6; ++n) need |= (use & OWNED[n]) ? 1u << n : 0u;
  // Owners 1 (0,-1,0), 2 (0,0,-1) and 5 (0,-1,-1) are found through their
  // segments' group maps.  An owner needed here contains a crossing edge, so
  // it is active, and so are the other cells around that edge: owners 0
  // (-1,0,0), 3 (-1,-1,0) and 4 (-1,0,-1) are the active cells just before
  // this cell, owner 1 and owner 2 in their rows (when x is the first cell
  // of its x-tile they lie in the previous x-tile's segments and are found
  // through its group maps instead).  Each record's x field confirms the
  // cell found.  A lookup the cell does not need reads this cell's segment,
  // so that every load is in bounds.
  const bool wrap = c.xl == 0;  // -x lies in the previous x-tile's segment
  const uint32_t xlm = wrap ? cap - 1u : c.xl - 1u;
  const uint32_t dy = vol.XT, dz = vol.XT * g.cy;
  const uint32_t need1 = need & 0x0Au, need2 = need & 0x14u, need5 = need & 0x20u, needw = need & 0x19u;
  const uint32_t ns[6] = {wrap ? s - 1u : s, need1 ? s - dy : s, need2 ? s - dz : s,
                          wrap ? s - 1u - dy : s - dy, wrap ? s - 1u - dz : s - dz, need5 ? s - dy - dz : s};
  const uint32_t G = cap >> 4;
  const uint32_t g1 = a.gmap[(size_t)ns[1] * G + (c.xl >> 4)], g2 = a.gmap[(size_t)ns[2] * G + (c.xl >> 4)];
  const uint32_t g5 = a.gmap[(size_t)ns[5] * G + (c.xl >> 4)];
  uint32_t vq0[6];
  vq0[1] = a.seg_vq[ns[1]].x;
  vq0[2] = a.seg_vq[ns[2]].x;
  vq0[5] = a.seg_vq[ns[5]].x;
  const uint32_t bit = c.xl & 15u, below = (1u << bit) - 1u;
  const uint32_t r1 = (g1 >> 16) + (uint32_t)__popc(g1 & below), r2 = (g2 >> 16) + (uint32_t)__popc(g2 & below);
  const uint32_t r5 = (g5 >> 16) + (uint32_t)__popc(g5 & below);
  uint32_t nr[6] = {rank - 1u, r1, r2, r1 - 1u, r2 - 1u, r5};
  bool inmask[6] = {rank > 0u, ((g1 >> bit) & 1u) != 0, ((g2 >> bit) & 1u) != 0, r1 > 0u, r2 > 0u,
                    ((g5 >> bit) & 1u) != 0};
  vq0[0] = c.seg_vb;
  vq0[3] = vq0[1];
  vq0[4] = vq0[2];
  if (wrap && needw) {  // owners 0, 3, 4: the last cells of the previous x-tile's segments
    const uint32_t gw = (cap - 1u) >> 4;
#pragma unroll
    for (int n = 0; n < 6; ++n) {
      if (n != 0 && n != 3 && n != 4) continue;
      const uint32_t sn = ((need >> n) & 1u) ? ns[n] : s;  // in bounds when not needed
      const uint32_t gx = a.gmap[(size_t)sn * G + gw];
      nr[n] = (gx >> 16) + (uint32_t)__popc(gx & 0x7FFFu);
      inmask[n] = ((gx >> 15) & 1u) != 0;
      vq0[n] = a.seg_vq[sn].x;
    }
  }
  const uint32_t nx[6] = {xlm, c.xl, c.xl, xlm, xlm, c.xl};
  // Each edge's point (its owner's first edge point and the owner's crossed
  // edges before it) in column e of the lane's part of LDS.
  constexpr uint32_t T = kEmitThreads;
  constexpr int kOwnerEdges[7][3] = {{7, 11, -1}, {5, -1, 8}, {-1, 1, 2}, {4, -1, -1}, {-1, 3, -1}, {-1, -1, 0}, {6, 9, 10}};
  bool ok = true;
  auto put = [&](int n, uint32_t first, uint32_t bip) {
    const uint32_t i1 = first + (bip & 1u), i2 = i1 + ((bip >> 1) & 1u);
    const uint32_t at[3] = {first, i1, i2};
#pragma unroll
    for (int l = 0; l < 3; ++l) {
      const int e = kOwnerEdges[n][l];
      if (e < 0) continue;
      s_idx[e * T] = at[l];
      // (a point its owner does not have, or past the capacity, is left out)
      if (((use >> e) & 1u) && (!((bip >> l) & 1u) || (uint64_t)at[l] >= vol.vcap)) {
        ok = false;
        use &= ~(1u << e);
      }
    }
  };
  uint32_t m[6];  // (all six in flight before the first is used)
  bool ok_r[6];
#pragma unroll
  for (int n = 0; n < 6; ++n) {
    const bool used = (need >> n) & 1u;
    ok_r[n] = used && inmask[n] && nr[n] < cap;
    m[n] = a.slots[(size_t)(ok_r[n] ? ns[n] : s) * cap + (ok_r[n] ? nr[n] : rank)];
    if (used && !ok_r[n]) ok = false;
  }
#pragma unroll
  for (int n = 0; n < 6; ++n) {
    if (ok_r[n] && rec_x(m[n]) != nx[n]) ok = false;
    const uint32_t miso = (s_lab32[2u * ((m[n] >> 10) & 0x1FFu) + 1u] >> 16) & 0xFu;
    put(n, vq0[n] + rec_lvb(m[n]) - vol.vbase + miso, owned_bipolar(rec_cfg(m[n])));
  }
  put(6, c.vb + niso, owned_bipolar(c.cfg));
  if ((uint64_t)c.vb + niso > vol.vcap) { atomicOr(vol.status, kStatusVertexOverflow); return; }
  // The points are gathered three of a lane's own edges at a time, in edge
  // order: a cell crosses 4 of the 12 on average and the most of 64 lanes is
  // 5 to 6, so two rounds (a gather costs its 64 lanes' addresses whether or
  // not they contribute; a load the lane does not need reads vertex 0).
  Float3 *const out = reinterpret_cast<Float3 *>(vol.verts + 3ull * c.vb);
  auto walk = [&](auto add) {
    for (uint32_t left = use; left != 0u;) {
      const uint32_t l1 = left & (left - 1u), l2 = l1 & (l1 - 1u);
      const uint32_t e0 = (uint32_t)__builtin_ctz(left), e1 = l1 ? (uint32_t)__builtin_ctz(l1) : 12u;
      const uint32_t e2 = l2 ? (uint32_t)__builtin_ctz(l2) : 12u;
      const uint32_t i0 = s_idx[e0 * T], i1 = s_idx[e1 * T], i2 = s_idx[e2 * T];
      const Float3 *const pts = reinterpret_cast<const Float3 *>(vol.verts);
      const Float3 p0 = pts[i0], p1 = pts[i1], p2 = pts[i2];
      add(e0, p0);
      if (l1) add(e1, p1);
      if (l2) add(e2, p2);
      left = l2 & (l2 - 1u);
    }
  };
  s_idx[12 * T] = 0u;
  if (__ballot(niso != 1u) == 0ull) {
    const uint32_t n = (uint32_t)__popc(use);
    float sx = -0.0f, sy = -0.0f, sz = -0.0f;
    walk([&](uint32_t, const Float3 &p) {
      sx = sx + p.x;
      sy = sy + p.y;
      sz = sz + p.z;
    });
    const float d = (float)n;
    if (n) *out = Float3{sx / d, sy / d, sz / d};
  } else {
    float sx[4] = {-0.0f, -0.0f, -0.0f, -0.0f}, sy[4] = {-0.0f, -0.0f, -0.0f, -0.0f}, sz[4] = {-0.0f, -0.0f, -0.0f, -0.0f};
    uint32_t cnt = 0;  // 8 bits per group
    walk([&](uint32_t e, const Float3 &p) {
      const uint32_t lab = (uint32_t)(labels >> (4u * e)) & 0xFu;
      cnt += 1u << (8u * lab);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        sx[q] = lab == (uint32_t)q ? sx[q] + p.x : sx[q];
        sy[q] = lab == (uint32_t)q ? sy[q] + p.y : sy[q];
        sz[q] = lab == (uint32_t)q ? sz[q] + p.z : sz[q];
      }
    });
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if ((uint32_t)q < niso) {
        const uint32_t n = (cnt >> (8 * q)) & 0xFFu;
        const float d = (float)n;
        if (n) out[q] = Float3{sx[q] / d, sy[q] / d, sz[q] / d};
      }
    }
  }
  if (!ok) atomicOr(vol.status, kStatusLookup);
}

__global__ __launch_bounds__(kEmitThreads) void k_smooth(EmitArgs a) {
  const uint32_t lane = lane_id(), wave = wave_id();
  const Totals tot = *a.totals;
  const uint32_t num_chunks = (uint32_t)min((uint64_t)tot.num_chunks, a.max_chunks);
  const uint32_t num_ne = min(tot.num_nonempty, a.nsegs);
  const ChunkIter it = chunk_iter(num_chunks, wave);
  for (uint32_t ch = it.next; ch < it.end; ch += it.step) {
    uint32_t s = 0, rank = 0;
    const bool found = locate_cell(a, tot, num_ne, ch, lane, s, rank);
    smooth_chunk(a, a.v, found, s, rank);
  }
}

__global__ __launch_bounds__(kEmitThreads) void k_reaverage(EmitArgs a) {
  __shared__ uint64_t s_lab[2 * 256];
  __shared__ uint32_t s_idx[13 * kEmitThreads];
  const Totals tot = *a.totals;
  const uint32_t num_chunks = (uint32_t)min((uint64_t)tot.num_chunks, a.max_chunks);
  if (!workgroup_has_chunks(num_chunks)) return;  // (uniform: before the barrier)
  for (uint32_t i = threadIdx.x; i < 512; i += kEmitThreads) s_lab[i] = emit_label(i);
  __syncthreads();
  const uint32_t lane = lane_id(), wave = wave_id();
  const uint32_t num_ne = min(tot.num_nonempty, a.nsegs);
  const ChunkIter it = chunk_iter(num_chunks, wave);
  for (uint32_t ch = it.next; ch < it.end; ch += it.step) {
    uint32_t s, rank;
    if (!locate_cell(a, tot, num_ne, ch, lane, s, rank)) continue;
    reaverage_cell(a, a.v, s, rank, s_lab, s_idx + threadIdx.x);
  }
}

// ---------------------------------------------------------------------------
// Batch count and emit.

struct BatchCountArgs {
  const BatchVol *vols;
  uint32_t nvol, nsegs;
  const uint2 *seg_vq;
  const uint2 *ne;              // non-empty segments {segment, first active}, sentinel last
  const Totals *totals;
  uint2 *base;                  // per volume: global vertex / quad number of its first
  const uint32_t *batch_counts;  // the batch scan's counts (status bits in [3])
};

// Active cells before segment s: the first active of the first non-empty
// segment at or after s (the list ends with {nsegs, total}).
__device__ __forceinline__ uint32_t actives_before(const uint2 *ne, uint32_t num_ne, uint32_t s) {
  uint32_t lo = 0, hi = num_ne;  // ne[num_ne] is the sentinel
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (ne[mid].x < s) lo = mid + 1; else hi = mid;
  }
  return ne[lo].y;
}

// One slab of an out-of-core extraction, after its count: the count words,
// the vertex / quad bases of segments s_lo and s_hi (the slab's own cell
// planes) and its active cells, in one small record for one host copy:
// out[0..3] counts, out[4..7] base(s_lo).xy base(s_hi).xy, out[8] actives.
__global__ void k_slab_info(const uint2 *seg_vq, const uint2 *ne, const Totals *totals, uint32_t nsegs,
                            const uint32_t *counts, uint32_t s_lo, uint32_t s_hi, uint32_t *out) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  const uint32_t num_ne = min(totals->num_nonempty, nsegs);
  for (int i = 0; i < 4; ++i) out[i] = counts[i];
  const uint2 lo = seg_vq[s_lo], hi = seg_vq[s_hi];
  out[4] = lo.x;
  out[5] = lo.y;
  out[6] = hi.x;
  out[7] = hi.y;
  out[8] = actives_before(ne, num_ne, s_hi) - actives_before(ne, num_ne, s_lo);
}

// The same by a whole wave: 64 entries a round, so 4 rounds of loads for 16 M
// segments instead of 24 one after the other.
__device__ __forceinline__ uint32_t actives_before_wave(const uint2 *ne, uint32_t num_ne, uint32_t s) {
  uint32_t lo = 0, n = num_ne;  // the first entry at or after s is in [lo, lo + n]
  while (n != 0u) {
    const uint32_t step = (n + kWave - 1u) / kWave, i = lane_id() * step;
    const uint32_t less = (uint32_t)__popcll(__ballot(i < n && ne[lo + min(i, n - 1u)].x < s));
    if (less == 0u) break;
    const uint32_t at = (less - 1u) * step + 1u;  // entries up to the last one found less are
    n = min(step - 1u, n - at);
    lo += at;
  }
  return ne[lo].y;
}

// One wave per volume: its totals and the bases of its numbering.
__global__ __launch_bounds__(256) void k_batch_counts(BatchCountArgs b) {
  const uint32_t v = blockIdx.x * (256u / kWave) + wave_id();
  if (v >= b.nvol) return;
  const BatchVol &bv = b.vols[v];
  const uint32_t num_ne = min(b.totals->num_nonempty, b.nsegs);
  const uint2 v0 = b.seg_vq[bv.seg_off], v1 = b.seg_vq[bv.seg_off + bv.nsegs];
  uint32_t active = 0u;
  if (bv.counts && bv.nsegs)
    active = actives_before_wave(b.ne, num_ne, bv.seg_off + bv.nsegs) - actives_before_wave(b.ne, num_ne, bv.seg_off);
  if (lane_id() != 0u) return;
  b.base[v] = v0;
  if (bv.counts) {
    bv.counts[0] = active;
    bv.counts[1] = v1.x - v0.x;
    bv.counts[2] = v1.y - v0.y;
    bv.counts[3] = b.batch_counts[3];
  }
}

// Counts to pinned host memory, then the call's number in its first word: the
// host, which watches that word, has them 2-3 us after the kernels before this
// one end.  The stream's own completion and a copy out of device memory cost
// it 15-20 us (one workgroup).
__global__ __launch_bounds__(256) void k_publish(const uint32_t *src, uint32_t words, uint32_t *host, uint32_t seq) {
  for (uint32_t i = threadIdx.x; i < words; i += 256u)
    __hip_atomic_store(host + kPublishHead + i, src[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(host, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// After a batch emit: status bits the emit could only attribute to the batch
// (a chunk whose cell could not be located) go to every volume's counts, the
// words callers read.
__global__ __launch_bounds__(256) void k_batch_status(const BatchVol *vols, uint32_t nvol,
                                                      const uint32_t *batch_status) {
  const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nvol) return;
  const uint32_t st = *batch_status;
  uint32_t *const cnt = vols[v].counts;
  if (st && cnt) atomicOr(cnt + 3, st);
}

// One workgroup per volume: its coordinate tables.
__global__ __launch_bounds__(256) void k_coords_batch(const BatchVol *vols, uint32_t nvol) {
  for (uint32_t v = blockIdx.x; v < nvol; v += gridDim.x) {
    const BatchVol &bv = vols[v];
    if (bv.nsegs == 0) continue;
    CoordArgs c{bv.coords, bv.c.g.X, bv.c.g.Y, bv.c.g.Z, bv.c.g.cx, bv.c.g.cy, bv.c.g.cz,
                bv.mnx, bv.mny, bv.mnz, bv.rgx, bv.rgy, bv.rgz};
    coords_fill(c, threadIdx.x, blockDim.x);
  }
}

struct BatchEmitArgs {
  EmitArgs a;  // arrays of the whole batch; a.v.status is the batch status word
  const BatchVol *vols;
  const uint32_t *seg_off;  // first segment of each volume
  const uint2 *base;
  uint32_t nvol;
};

// Emit over the active cells of all volumes; a lane finds its volume by
// binary search over the volumes' first segments.
__global__ __launch_bounds__(kEmitThreads) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_emit_batch(BatchEmitArgs b) {
  __shared__ uint64_t s_lab[2 * 256];
  __shared__ __align__(16) float s_acc[kEmitStage * (kEmitThreads / kWave)];
  // first segment of each volume (the search below reads entries 1 .. nvol-1;
  // kMaxBatch entries keep the workgroup's LDS at 20 KB, 8 workgroups per CU)
  __shared__ uint32_t s_soff[kMaxBatch];
  const EmitArgs &a = b.a;
  static_assert(offsetof(BatchEmitArgs, a) == 0, "the kernel's arguments start with a");
  const EmitArgsK pa = (EmitArgsK)__builtin_amdgcn_kernarg_segment_ptr();  // b.a
  const Totals tot = *a.totals;
  const uint32_t num_chunks = (uint32_t)min((uint64_t)tot.num_chunks, a.max_chunks);
  if (!workgroup_has_chunks(num_chunks)) return;  // (uniform: before the barrier)
  for (uint32_t i = threadIdx.x; i < 512; i += kEmitThreads) s_lab[i] = emit_label(i);
  for (uint32_t i = threadIdx.x; i < b.nvol; i += kEmitThreads) s_soff[i] = b.seg_off[i];
  __syncthreads();
  const uint32_t lane = lane_id(), wave = wave_id();
  const uint32_t num_ne = min(tot.num_nonempty, a.nsegs);
  const ChunkIter it = chunk_iter(num_chunks, wave);
  for (uint32_t ch = it.next; ch < it.end; ch += it.step) {
    uint32_t s = 0, rank = 0;
    bool todo = locate_cell(a, tot, num_ne, ch, lane, s, rank);
    // the last volume whose first segment is <= s (empty volumes share it)
    uint32_t lo = 0, hi = b.nvol;
    while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) >> 1;
      if (s_soff[mid] <= s) lo = mid; else hi = mid;
    }
    // the lanes of one volume at a time (64 consecutive active cells rarely
    // span two volumes), so that the volume's descriptor is wave-uniform and
    // comes in through scalar loads instead of occupying vector registers
    for (uint64_t left = __ballot(todo); left != 0ull; left = __ballot(todo)) {
      const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)lo, __ffsll((long long)left) - 1);
      const __attribute__((address_space(4))) BatchVol *bv = (const __attribute__((address_space(4))) BatchVol *)b.vols + v;
      emit_lanes(pa, &bv->e, const_u2(b.base, v), todo && lo == v, s, rank, s_lab, s_acc + kEmitStage * wave);
      todo = todo && lo != v;
    }
  }
}

// ---------------------------------------------------------------------------
// Per-cell records in ascending cell order (parity and debugging): one
// workgroup per non-empty segment (grid-stride over the list).

struct CellsArgs {
  uint32_t XT, cap, cx, nsegs;
  const uint2 *seg_counts;
  const uint32_t *slots;
  const uint2 *seg_vq;
  const uint2 *ne;
  const Totals *totals;
  uint32_t *cell_index;
  uint8_t *cfg;
  uint8_t *flags;
  uint32_t *vbegin;
  uint64_t capacity;
};

__global__ __launch_bounds__(256) void k_cells(CellsArgs a) {
  const uint32_t num_ne = min(a.totals->num_nonempty, a.nsegs);
  for (uint32_t i = blockIdx.x; i < num_ne; i += gridDim.x) {
    const uint2 e = a.ne[i];
    const uint32_t sg = e.x;
    if (sg >= a.nsegs) continue;
    const uint32_t n = min(a.seg_counts[sg].x & 0xFFFFu, a.cap);
    const uint32_t vb = a.seg_vq[sg].x;
    const uint32_t xt = sg % a.XT, row = sg / a.XT;
    for (uint32_t r = threadIdx.x; r < n; r += blockDim.x) {
      const uint64_t pos = (uint64_t)e.y + r;
      if (pos >= a.capacity) break;
      const uint32_t rec = a.slots[(size_t)sg * a.cap + r];
      a.cell_index[pos] = xt * a.cap + rec_x(rec) + a.cx * row;
      a.cfg[pos] = (uint8_t)rec_cfg(rec);
      a.flags[pos] = (uint8_t)rec_lut2(rec);
      a.vbegin[pos] = vb + rec_lvb(rec);
    }
  }
}

// ---------------------------------------------------------------------------
// Synthetic fields (definitions in mdmc_fields.h).

// Blob tables, ldb = blob_ldb(nblobs) entries per blob dimension, entries
// past nblobs zero: ex is [ldb][X] (read per lane), ey and ez are transposed,
// [Y][ldb] and [Z][ldb], so that the factors of one row are contiguous and
// come in through a few wide scalar loads; amp has ldb entries.
struct BlobArgs {
  float *out;
  uint32_t X, Y, Z, nblobs, ldb;
  const double *ex, *ey, *ez, *amp;
  uint32_t per;  // planes per task
};

// Generators work in wave tasks of 64 consecutive columns x; a lane owns one
// column, and a task takes one row y in `per` consecutive planes z.  The loop
// over the task's planes is uniform over the wave, so per-plane values are
// scalar loads, the stores of a plane are one contiguous 256-byte run, and
// what depends on x and y only is computed once per task.  Consecutive tasks
// take consecutive column blocks, then rows, then plane blocks.  `per` is at
// most kGenPer, fewer for a field too small to give the chip enough waves (a
// task's planes run one after another).
constexpr uint32_t kGenPer = 16;
constexpr uint32_t kGenThreads = 256;
constexpr uint32_t kGenWaves = kGenThreads / kWave;
constexpr uint32_t kBlobRegs = 32;  // blobs kept in registers (more: per-point path)

// blob table row stride for a blob count
__host__ __device__ inline uint32_t blob_ldb(uint32_t nblobs) {
  return nblobs <= kBlobRegs ? kBlobRegs : nblobs;
}

__host__ __device__ inline uint64_t gen_tasks(uint32_t X, uint32_t Y, uint32_t Z, uint32_t per) {
  return (uint64_t)((X + 63u) / 64u) * Y * ((Z + per - 1u) / per);
}

// Wave-uniform reads through the constant address space compile to scalar
// loads (the tables are not written while a generator runs).
typedef const __attribute__((address_space(4))) double *uniform_dptr;
__device__ __forceinline__ uniform_dptr as_uniform(const double *p) { return (uniform_dptr)p; }

// A task: the lane's column x, its row y, and its planes z0 .. z0 + nz - 1
// (nz = 0 past the last task).
struct PlaneTask {
  uint32_t x, y, z0, nz;
};

__device__ __forceinline__ PlaneTask plane_task(uint32_t X, uint32_t Y, uint32_t Z, uint32_t per, uint64_t task) {
  const uint32_t ncc = (X + 63u) / 64u;
  PlaneTask t;
  t.x = (uint32_t)(task % ncc) * 64u + (threadIdx.x & 63u);
  const uint64_t rest = task / ncc;
  t.y = (uint32_t)(rest % Y);
  const uint64_t zb = rest / Y;
  t.z0 = (uint32_t)min<uint64_t>(zb * per, Z);
  t.nz = min(per, Z - t.z0);
  return t;
}

// Blob sums: a lane keeps (amp[b] * ex[b][x]) * ey[y][b] for every blob in
// registers and, plane by plane, adds it times ez[z][b] blob by blob with one
// FMA each (fma((amp*ex) * ey, ez, sum)), the same operations in the same
// order as the CPU generator.  Four planes go per pass (four independent FMA
// chains); blobs go in groups of 8 (one group of a plane's factors is one
// wide scalar load).  The zero entries that pad the last group add +0.0 to a
// sum that starts at +0.0 and so can never be -0.0, which leaves it
// unchanged.  Needs ldb == kBlobRegs.
__device__ __forceinline__ void blob_task(const BlobArgs &a, uint64_t task) {
  constexpr uint32_t P = 4;
  const PlaneTask t = plane_task(a.X, a.Y, a.Z, a.per, task);
  if (t.x >= a.X || t.nz == 0) return;
  const uniform_dptr amp = as_uniform(a.amp);
  const uniform_dptr ey = as_uniform(a.ey + (size_t)t.y * kBlobRegs);
  double txy[kBlobRegs];
#pragma unroll
  for (uint32_t g = 0; g < kBlobRegs / 8; ++g) {
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) txy[8 * g + i] = 0.0;
    if (8 * g < a.nblobs) {
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i)
        txy[8 * g + i] = (amp[8 * g + i] * a.ex[(size_t)(8 * g + i) * a.X + t.x]) * ey[8 * g + i];
    }
  }
  const uint64_t plane = (uint64_t)a.X * a.Y;
  float *out = a.out + (uint64_t)t.z0 * plane + (uint64_t)t.y * a.X + t.x;
  for (uint32_t kz = 0; kz < t.nz; kz += P) {
    // planes past the task's last repeat it (summed, not stored)
    uniform_dptr ez[P];
#pragma unroll
    for (uint32_t j = 0; j < P; ++j) ez[j] = as_uniform(a.ez + (size_t)(t.z0 + min(kz + j, t.nz - 1u)) * kBlobRegs);
    double acc[P];
#pragma unroll
    for (uint32_t j = 0; j < P; ++j) acc[j] = 0.0;
#pragma unroll
    for (uint32_t g = 0; g < kBlobRegs / 8; ++g) {
      if (8 * g < a.nblobs) {
        double f[P][8];
#pragma unroll
        for (uint32_t j = 0; j < P; ++j)
#pragma unroll
          for (uint32_t i = 0; i < 8; ++i) f[j][i] = ez[j][8 * g + i];
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i)
#pragma unroll
          for (uint32_t j = 0; j < P; ++j) acc[j] = __builtin_fma(txy[8 * g + i], f[j][i], acc[j]);
      }
    }
#pragma unroll
    for (uint32_t j = 0; j < P; ++j)
      if (kz + j < t.nz) out[(size_t)(kz + j) * plane] = (float)acc[j];
  }
}

// Per-point path (any number of blobs).
__device__ __forceinline__ void blob_points(const BlobArgs &a, size_t i0, size_t stride) {
  const size_t n = (size_t)a.X * a.Y * a.Z;
  for (size_t id = i0; id < n; id += stride) {
    const uint32_t x = (uint32_t)(id % a.X);
    const size_t r = id / a.X;
    const uint32_t y = (uint32_t)(r % a.Y), z = (uint32_t)(r / a.Y);
    double acc = 0.0;
    for (uint32_t b = 0; b < a.nblobs; ++b)
      acc = __builtin_fma((a.amp[b] * a.ex[(size_t)b * a.X + x]) * a.ey[(size_t)y * a.ldb + b],
                          a.ez[(size_t)z * a.ldb + b], acc);
    a.out[id] = (float)acc;
  }
}

struct GyroidArgs {
  float *out;
  uint32_t X, Y, Z;
  const double *sx, *cx, *sy, *cy, *sz, *cz;
  uint64_t seed;
  double amp;
  uint32_t per;  // planes per task
};

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// Gyroid plus hash noise of point id = x + X * (y + Y * z):
// sx*cy + sy*cz + sz*cx from the 1-D tables, in that order, then the noise of
// mix64(seed + (id + 1) * golden).  Along the task's planes id grows by X*Y,
// so the hash input grows by X*Y*golden (mod 2^64).
__device__ __forceinline__ void gyroid_task(const GyroidArgs &a, uint64_t task) {
  constexpr uint64_t kGolden = 0x9E3779B97F4A7C15ull;
  const PlaneTask t = plane_task(a.X, a.Y, a.Z, a.per, task);
  if (t.x >= a.X || t.nz == 0) return;
  const double sxx = a.sx[t.x], cxx = a.cx[t.x];
  const uniform_dptr sz = as_uniform(a.sz), cz = as_uniform(a.cz);
  const double syy = as_uniform(a.sy)[t.y];
  const double t1 = sxx * as_uniform(a.cy)[t.y];
  const uint64_t plane = (uint64_t)a.X * a.Y;
  const uint64_t id0 = (uint64_t)t.z0 * plane + (uint64_t)t.y * a.X + t.x;
  const uint64_t step = plane * kGolden;
  uint64_t hin = a.seed + (id0 + 1) * kGolden;
  float *out = a.out + id0;
  for (uint32_t kz = 0; kz < t.nz; ++kz, hin += step) {
    const uint32_t z = t.z0 + kz;
    const double gval = t1 + syy * cz[z] + sz[z] * cxx;
    const uint64_t h = mix64(hin);
    const double u = (double)(h >> 11) * (1.0 / 9007199254740992.0);
    out[kz * plane] = (float)(gval + a.amp * (2.0 * u - 1.0));
  }
}

// The generator kernel: the fields of one or many volumes in one launch.
// Workgroup b belongs to the volume whose range [block_off, block_off +
// nblocks) holds it, so its waves share the volume and its kind.
struct GenVol {
  float *out;
  uint32_t X, Y, Z, kind;  // kind 1: blobs, 2: gyroid
  uint32_t nblobs, block_off, nblocks, per;  // per: planes per task
  const double *t[6];      // blobs: ex, ey, ez, amp; gyroid: sx, cx, sy, cy, sz, cz
  uint64_t seed;
  double amp;              // gyroid noise amplitude
};

__global__ __launch_bounds__(kGenThreads) void k_field_batch(const GenVol *vols, uint32_t nvol) {
  uint32_t lo = 0, hi = nvol;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (vols[mid].block_off <= blockIdx.x) lo = mid; else hi = mid;
  }
  const GenVol &v = vols[__builtin_amdgcn_readfirstlane(lo)];
  const uint32_t local = blockIdx.x - v.block_off;
  const uint64_t task = (uint64_t)local * kGenWaves + wave_id();
  if (v.kind == 1) {
    const BlobArgs ba{v.out, v.X, v.Y, v.Z, v.nblobs, blob_ldb(v.nblobs), v.t[0], v.t[1], v.t[2], v.t[3], v.per};
    if (v.nblobs <= kBlobRegs) {
      if (task < gen_tasks(v.X, v.Y, v.Z, v.per)) blob_task(ba, task);
    } else {
      blob_points(ba, (size_t)local * blockDim.x + threadIdx.x, (size_t)v.nblocks * blockDim.x);
    }
    return;
  }
  if (task < gen_tasks(v.X, v.Y, v.Z, v.per)) {
    const GyroidArgs ga{v.out, v.X, v.Y, v.Z, v.t[0], v.t[1], v.t[2], v.t[3], v.t[4], v.t[5], v.seed, v.amp, v.per};
    gyroid_task(ga, task);
  }
}

}  // namespace mdmc

// nlg_attn_grid.h -- how the fp16 decode attention's chunk pass lays its work
// over a grid: the host's choice and the workgroup's reading of it, in one
// place (plain C++, so both are checked against each other on the CPU).
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define NLG_GRID_HD __host__ __device__ __forceinline__
#else
#define NLG_GRID_HD inline
#endif

#define ATTN_WAVES 8

// Workgroups of G of a kv head's grp query heads over units (row, kv head,
// first chunk), `gx` first chunks per (row, kv head).  nunits not 0: a 1-D
// grid, a unit's grp / G workgroups on one XCD; 0: x the first chunk, y the head
// group, z the row; or, with clast (asked for by `last`), x the head group, y the
// row, z the chunk: workgroups start in x, y, z order, so the chunks past the
// position come after all others.
struct AttnGrid {
  uint32_t x, y, z, nunits, clast;
};
inline AttnGrid attn_grid(uint32_t rows, uint32_t kvheads, uint32_t grp, uint32_t G, uint32_t gx, bool last) {
  // a grid's x dimension holds fewer than 2^32 threads; past it the grid is 3-D
  const uint64_t nu = (uint64_t)rows * kvheads * gx, per = grp / G;
  if ((G == 1 || G < grp) && (nu + 7) * per * (ATTN_WAVES * 64) < (1ull << 32))
    return AttnGrid{(uint32_t)((nu + 7) / 8 * 8 * per), 1, 1, (uint32_t)nu, 0};
  // (a z dimension holds 65,535)
  if (last && gx <= 65535) return AttnGrid{kvheads * (uint32_t)per, rows, gx, 0, 1};
  return AttnGrid{gx, kvheads * (uint32_t)per, rows, 0, 0};
}

// Whether a form of the pass reads nunits: the others are only launched with 0
// (eight heads in fours neither loop over chunks nor rotate rows).
constexpr bool attn_reads_units(int G, bool loop, bool rot) { return G == 1 || (G == 4 && !loop && !rot); }

// The workgroup's first chunk, first query head and row; false: nothing to do.
// Workgroups are dealt to the 8 XCDs round-robin by id, and each XCD has its own
// L2: on the 1-D grid the n = grp / G workgroups of a unit u get ids u%8 + 8(q +
// n*(u/8)), all on XCD u%8, so the unit's K/V rows come from HBM once and from
// that L2 for the other heads.
template <int G>
NLG_GRID_HD bool attn_unit(uint32_t bx, uint32_t by, uint32_t bz, uint32_t nunits, uint32_t clast, uint32_t cstep,
                           uint32_t kvheads, uint32_t grp, uint32_t &c, uint32_t &h0, uint32_t &qr) {
  if (!nunits) {
    c = clast ? bz : bx;
    h0 = (clast ? bx : by) * G;
    qr = clast ? by : bz;
    return true;
  }
  const uint32_t n = grp / G, rest = bx >> 3, q = rest % n, u = (bx & 7u) + 8u * (rest / n);
  if (u >= nunits) return false;
  c = u % cstep;
  const uint32_t r2 = u / cstep;
  h0 = (r2 % kvheads) * grp + q * G;
  qr = r2 / kvheads;
  return true;
}

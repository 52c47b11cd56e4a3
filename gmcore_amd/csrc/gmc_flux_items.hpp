// gmc_flux_items.hpp -- the work items of the tracer flux kernels
// (gmc_adv.hip).  Index arithmetic only: tests/test_index_maps.py runs it on
// the CPU.
#pragma once

#include "gmc_hflx.hpp"

namespace gmc {

// Work of the two flux kernels, in blocks of NF = 8 wavefronts.  Items
// [0, npole) are the pole rows (2 per tracer, padded to a multiple of the
// XCD count so that the interior items keep their XCD placement).  An
// interior item covers the cell rows r0 .. r0 + 6 (r0 = 1 + 7 rb) over one
// column segment, for a group of up to kGroup tracers: wavefront w forms the
// y-fluxes of V row r0 - 1 + w (into LDS, each shared by the cells either
// side) and, for w < 7, the x-fluxes and the update of cell row r0 + w.  Lane
// l sits on column 63 s - 1 + l; lanes 1..63 own the cells 63 s .. 63 s + 62,
// the x-flux on a cell's west face coming from the lane below.  Interior items
// are numbered (row block, segment, group), the group fastest, and dealt to
// the XCDs in contiguous runs, so the wind rows and the neighbouring tracer
// rows an item reads are already in its XCD's L2.
//
// The kernels are bound by instruction issue.  The wind's share of a face (its
// weights, direction, stencil address, the reciprocal of its Courant number)
// is half of a face's instructions and the same for every tracer, so a group
// forms it once: 232 vector instructions per tracer and cell instead of 430,
// 40 -> 28 us a kernel at 720 x 361 x 8 tracers.  Groups of 4 at four
// wavefronts per SIMD: groups of 2 and 8 and six wavefronts took 2 to 10 %
// longer, eight (spilling) 45 %.
constexpr int NF = 512;
constexpr int kSeg = kWave - 1;
constexpr int kRowsPerItem = NF / kWave - 1;
constexpr int kGroup = 4;
struct FluxItem {
  int pole;    // 1: pole row item
  int r, t;    // pole: cell row; interior: first cell row r0; (first) tracer
  int c0;      // first cell of the segment
  int nt;      // tracers of the group
};
// How a launch numbers its items: ng groups of `group` tracers, nseg segments,
// nrb row blocks, the first and last `edge` of them first (below); the two
// divisions of an item's number by div_mod (integer divisions were 0.4 us of a
// 4.5 us kernel).
struct FluxMap {
  int ntr, group, ng, per, nrb, edge, npole;
  uint32_t div_ng, div_per;
  FluxMap(const AdvGrid &g, int ntr_, int group_) : ntr(ntr_), group(group_) {
    ng = (ntr + group - 1) / group;
    per = (g.nlon + kSeg - 1) / kSeg * ng;
    nrb = (g.nlat - 2 + kRowsPerItem - 1) / kRowsPerItem;
    // one tracer an item: all items run at once, in the order that shares L2s
    edge = group == 1 ? 0 : nrb / 2 < 2 ? nrb / 2 : 2;
    npole = (2 * ntr + kNumXcd - 1) / kNumXcd * kNumXcd;
    div_ng = div_mul(ng);
    div_per = div_mul(per);
  }
  int blocks() const { return npole + nrb * per; }
};
// the item of workgroup b
__host__ __device__ __forceinline__ FluxItem flux_item(const AdvGrid &g, const FluxMap &m, int b) {
  FluxItem it{0, -1, 0, 0, 1};
  if (b < m.npole) {
    if (b < 2 * m.ntr) { it.pole = 1; it.r = b % 2 ? g.nlat - 1 : 0; it.t = b / 2; }
    return it;
  }
  // the `edge` row blocks at either pole, whose x-fluxes cross up to hw whole
  // cells, go first, one workgroup after the other on all XCDs
  const int e = b - m.npole, first = 2 * m.edge * m.per;
  const int L = e < first ? e : xcd_item(e - first, m.nrb * m.per - first);
  int rb, rest, seg, grp;
  div_mod(L, m.per, m.div_per, rb, rest);
  div_mod(rest, m.ng, m.div_ng, seg, grp);
  rb = e >= first ? rb + m.edge : rb & 1 ? m.nrb - 1 - rb / 2 : rb / 2;
  it.t = grp * m.group;
  it.nt = min(m.group, m.ntr - it.t);
  it.r = 1 + kRowsPerItem * rb;
  it.c0 = seg * kSeg;
  return it;
}

}  // namespace gmc

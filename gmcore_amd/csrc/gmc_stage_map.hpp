// gmc_stage_map.hpp -- which rows of a grid the stage's tiles take whole, and
// the rows and columns of every tile (gmc_fused.hip).  Host code and index
// arithmetic only: tests/test_index_maps.py runs it on the CPU.
#pragma once

#include <algorithm>
#include <utility>
#include <vector>

#include "gmc_internal.hpp"

namespace gmc {

// tendency tile: one wavefront per tile row, lane q <-> column C0 - 2 + q
constexpr int LC = kWave;               // 64 tile columns
constexpr int HXL = 2;                  // column halo: the west of pv_lat's four columns
constexpr int TX = LC - 2 * HXL;        // 60 output columns (q = 2 .. 61)
constexpr int kLaneTaps = 9;            // widest filter the lanes of a tile take

// What a tile owns: output columns c0 .. c0+nc-1 on the lanes from hl on, rows
// r0 .. r1-1 (at most TY; the tile's local row k is global row r0 - 2 + k).
struct TileGeo {
  int c0, nc, hl, r0, r1;
};

constexpr int kMaxSegs = 8;
// Bands of the short rows whose tiles have the same width: from band b0 and
// tile t0 on, nx tiles of w columns a band, first output lane hl; div = div_mul(nx).
struct TileSeg {
  int b0, t0, nx, w, hl;
  uint32_t div;
};
// What the launches of a stage share about its rows: [ra, rb) the rows of
// short filters; the polar tendencies' nx_p tiles a band, tiles_s of them
// south and tiles_p in all; bands_s polar bands south and bands_p in all.
struct StageMap {
  int ra, rb, nseg, ntiles;
  TileSeg seg[kMaxSegs];
  int nx_p, tiles_s, tiles_p, bands_s, bands_p;
  uint32_t div_p;
};
template <int TY> __host__ __device__ __forceinline__ TileGeo short_tile(const StageMap &S, int nlon, int t) {
  TileSeg s = S.seg[0];
#pragma unroll
  for (int k = 1; k < kMaxSegs; k++)
    if (k < S.nseg && t >= S.seg[k].t0) s = S.seg[k];
  int b, x;
  div_mod(t - s.t0, s.nx, s.div, b, x);
  const int r0 = S.ra + (s.b0 + b) * TY, c0 = x * s.w;
  return TileGeo{c0, min(s.w, nlon - c0), s.hl, r0, min(r0 + TY, S.rb)};
}

// Tile e of the polar tendencies: bands from the south pole to row ra, then
// from row rb to the north pole.
template <int TY> __host__ __device__ __forceinline__ TileGeo polar_tile(const StageMap &S, const Grid &g, int e) {
  const bool north = e >= S.tiles_s;
  if (north) e -= S.tiles_s;
  int b, x;
  div_mod(e, S.nx_p, S.div_p, b, x);
  const int r0 = (north ? S.rb : 0) + b * TY, c0 = x * TX;
  return TileGeo{c0, min(TX, g.nlon - c0), HXL, r0, min(r0 + TY, north ? g.nlat : S.ra)};
}

// The rows [ra, rb) that tiles take through the whole stage: rows of short
// filters (and the gz row rb that the last v row reads), at least three from
// either pole, whose sums and mirrored rows the tiles then never read.
inline void short_rows(int nlat, const std::vector<int32_t> &nb, const std::vector<int32_t> &ns,
                       const std::vector<int32_t> &nbv, int &ra, int &rb) {
  const int nhalf = nlat - 1;
  auto cell = [&](int r) { return nb[r] <= kLaneTaps && ns[r] <= kLaneTaps; };
  const int mid = nlat / 2;
  ra = rb = mid;
  while (ra > 3 && cell(ra - 1) && nbv[ra - 1] <= kLaneTaps) ra--;
  while (rb < nhalf - 3 && cell(rb) && nbv[rb] <= kLaneTaps && cell(rb + 1)) rb++;
}

// The rows of a grid that tiles of height ty take through the whole stage, and
// those tiles: bands of like width in segments (the last segment takes what
// does not fit the table at its widest filters); the tiles of the other rows'
// tendencies.  Grids of at least 64 columns and 24 rows (below that the polar
// zones are most of the grid) whose short rows are at least half of all have
// such rows; false, and every row among the others, elsewhere.
inline bool stage_map(int nlon, int nlat, const std::vector<int32_t> &nb, const std::vector<int32_t> &ns,
                      const std::vector<int32_t> &nbv, int ty, StageMap &m, bool whole = true) {
  m = StageMap{};
  auto half_width = [](int n) { return n > 1 ? (n - 1) / 2 : 0; };
  m.ra = m.rb = nlat;
  if (whole && nlon >= kWave && nlat >= 24) short_rows(nlat, nb, ns, nbv, m.ra, m.rb);
  const bool has = 2 * (m.rb - m.ra) >= nlat;
  if (!has) m.ra = m.rb = nlat;
  m.nx_p = (nlon + TX - 1) / TX;
  m.div_p = div_mul(m.nx_p);
  m.tiles_s = m.nx_p * ((m.ra + ty - 1) / ty);
  m.tiles_p = m.tiles_s + m.nx_p * ((nlat - m.rb + ty - 1) / ty);
  if (!has) return false;
  const int nbands = (m.rb - m.ra + ty - 1) / ty;
  std::vector<std::pair<int, int>> h(nbands);   // half widths of the filters of gz, and of u and v
  for (int b = 0; b < nbands; b++) {
    const int r0 = m.ra + ty * b, r1 = std::min(r0 + ty, m.rb);
    for (int r = r0; r <= r1; r++) h[b].first = std::max({h[b].first, half_width(nb[r]), half_width(ns[r])});
    for (int r = r0; r < r1; r++) h[b].second = std::max({h[b].second, half_width(nb[r]), half_width(nbv[r])});
  }
  for (int b = 0; b < nbands;) {
    int e = b + 1;
    std::pair<int, int> hh = h[b];
    while (e < nbands && (h[e] == h[b] || m.nseg == kMaxSegs - 1)) {
      hh = {std::max(hh.first, h[e].first), std::max(hh.second, h[e].second)};
      e++;
    }
    TileSeg &s = m.seg[m.nseg++];
    s.b0 = b;
    s.t0 = m.ntiles;
    s.hl = std::max(2, 1 + hh.first) + hh.second;
    s.w = std::min(61, 62 - hh.first) - hh.second - s.hl + 1;
    s.nx = (nlon + s.w - 1) / s.w;
    s.w = (nlon + s.nx - 1) / s.nx;
    s.div = div_mul(s.nx);
    m.ntiles += s.nx * (e - b);
    b = e;
  }
  return true;
}

// Where the tiles of the short rows are shared out over three launches, the
// first takes those of the bands next to the polar rows, whose gz_f the polar v
// rows of the last launch read: beside_polar tiles at least.  Of n tiles it
// takes, south_tiles are the first of the numbering and the rest the last.
inline int beside_polar(const StageMap &m) { return std::min(m.ntiles, m.seg[0].nx + m.seg[m.nseg - 1].nx); }
inline int south_tiles(const StageMap &m, int n) {
  const int first = m.seg[0].nx, last = m.seg[m.nseg - 1].nx;
  return n < first + last ? n : std::min(std::max(n / 2, first), n - last);
}

}  // namespace gmc

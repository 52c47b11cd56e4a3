// The tiles of a stage (gmcore_amd/csrc/gmc_stage_map.hpp): over grids, filter
// tables and tile heights, the tiles of the polar rows and those that do a
// whole stage own every point of the grid exactly once, from inside it, and
// the lanes of a whole-stage tile reach what its filters and stencil read.
// Prints "grids N bad M"; exits 1 on a fault.
#include <cstdio>
#include <cstdlib>

#include "../../gmcore_amd/csrc/gmc_stage_map.hpp"

using namespace gmc;

static int bad = 0;
static void fault(const char *what, int nlon, int nlat, int ty, int t) {
  if (bad++ < 8) std::printf("%s: %d x %d, tiles of %d rows, tile %d\n", what, nlon, nlat, ty, t);
}

template <int TY> static void check(int nlon, int nlat, const std::vector<int32_t> &nb, const std::vector<int32_t> &ns,
                                    const std::vector<int32_t> &nbv) {
  StageMap m;
  stage_map(nlon, nlat, nb, ns, nbv, TY, m);
  const Grid g{nlon, nlat, nlat - 1, (nlon + 31) / 32 * 32, nlon / 2};
  std::vector<char> owned((size_t)nlon * nlat, 0);
  for (int t = 0; t < m.tiles_p + m.ntiles; t++) {
    const bool polar = t < m.tiles_p;
    const TileGeo G = polar ? polar_tile<TY>(m, g, t) : short_tile<TY>(m, nlon, t - m.tiles_p);
    if (G.c0 < 0 || G.nc < 1 || G.c0 + G.nc > nlon || G.r0 < 0 || G.r1 <= G.r0 || G.r1 > nlat || G.r1 - G.r0 > TY) {
      fault("tile outside the grid", nlon, nlat, TY, t);
      continue;
    }
    for (int r = G.r0; r < G.r1; r++)
      for (int c = G.c0; c < G.c0 + G.nc; c++) owned[(size_t)r * nlon + c]++;
    if (polar) continue;
    // lanes 2 .. 61 hold tendencies and 1 .. 63 gz (as tend_tile); gz_f is a
    // filter of gz, u a difference of gz_f, u_f and v_f filters of u and v
    int hg = 0, hu = 0;
    for (int r = G.r0; r <= G.r1; r++) {
      hg = std::max({hg, (nb[r] - 1) / 2, (ns[r] - 1) / 2});
      if (r < G.r1) hu = std::max({hu, (nb[r] - 1) / 2, (nbv[r] - 1) / 2});
      if (nb[r] > kLaneTaps || ns[r] > kLaneTaps || (r < G.r1 && nbv[r] > kLaneTaps))
        fault("a wide filter in a whole-stage tile", nlon, nlat, TY, t);
    }
    const int west = G.hl - hu, east = G.hl + G.nc - 1 + hu;   // the lanes whose u and v are read
    if (west < 2 || west - hg < 1 || east > 61 || east + 1 + hg > 63)
      fault("a whole-stage tile reads beyond its lanes", nlon, nlat, TY, t);
    if (G.r0 < 3 || G.r1 > nlat - 4) fault("a whole-stage tile next to a pole", nlon, nlat, TY, t);
  }
  // the first launch's share, however many tiles it takes: the first `south` and
  // the last of the numbering, with the bands beside the polar rows among them
  for (int n = m.nseg ? beside_polar(m) : 0; n && n <= m.ntiles; n++) {
    const int south = south_tiles(m, n), north = n - south;
    if (south < 0 || north < 0 || (n < m.ntiles && (south < m.seg[0].nx || north < m.seg[m.nseg - 1].nx)))
      fault("a band beside the polar rows not in the first launch", nlon, nlat, TY, n);
  }
  for (char o : owned)
    if (o != 1) {
      fault("a point not owned exactly once", nlon, nlat, TY, -1);
      break;
    }
}

int main() {
  for (int d = 1; d <= 4096; d++) {   // div_mod against the divisions
    const uint32_t mul = div_mul(d);
    for (int64_t x = 0; x < (int64_t)1 << 31; x = x < 3 * d ? x + 1 : x + x / 7 / d * d + d)
      for (int o = -1; o <= 1; o++) {
        const int64_t y = x + o < 0 ? 0 : x + o > 0x7fffffff ? 0x7fffffff : x + o;
        int q, r;
        div_mod((int)y, d, mul, q, r);
        if (q != y / d || r != y % d) fault("div_mod", (int)y, d, 0, 0);
      }
  }
  unsigned seed = 1;
  auto rnd = [&](int n) { return (int)((seed = seed * 1664525u + 1013904223u) >> 8) % n; };
  int grids = 0;
  const int nlons[] = {8, 16, 30, 58, 60, 62, 64, 66, 118, 120, 122, 154, 180, 360, 502, 720, 1440, 2400};
  const int nlats[] = {5, 11, 12, 22, 23, 24, 25, 30, 31, 40, 61, 91, 181, 361};
  for (int nlon : nlons)
    for (int nlat : nlats)
      for (int table = 0; table < 4; table++) {
        std::vector<int32_t> nb(nlat), ns(nlat), nbv(nlat);
        const int zone = 3 + rnd(nlat / 3 + 1), most = std::min(nlon - 1, 4 * kLaneTaps + 1) | 1;
        for (int r = 0; r < nlat; r++) {
          const bool polar = r < zone || r >= nlat - zone;
          auto taps = [&] { return polar ? std::min(most, 1 + 2 * rnd(most)) : 1 + 2 * rnd(table == 3 ? 6 : table + 2); };
          nb[r] = taps();
          ns[r] = taps();
          nbv[r] = taps();
          if (table == 2 && !polar && r > nlat / 2) nb[r] = ns[r] = nbv[r] = 1;   // no filters in the north
        }
        check<5>(nlon, nlat, nb, ns, nbv);
        check<7>(nlon, nlat, nb, ns, nbv);
        check<11>(nlon, nlat, nb, ns, nbv);
        grids++;
      }
  std::printf("grids %d bad %d\n", grids, bad);
  return bad != 0;
}

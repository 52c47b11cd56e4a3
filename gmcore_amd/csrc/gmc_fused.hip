// gmc_fused.hip -- fused stage kernels used by gmc_step / gmc_time_integrate.
//
// One step_forward_backward stage (time_schemes_mod.F90:102-118) of the SW
// path is three steps:
//   tendencies  an LDS-tiled stencil: the pole sums (in the tiles next to the
//               poles), m, mass fluxes, pv, ke, tangential winds, upwind pv on
//               edges, then the forward tendencies du, dv and the updated,
//               unfiltered gz (operators_prepare_2 forward + calc_grad_mf +
//               calc_coriolis + calc_grad_ke + the gz part of update_state);
//   gz filters  the big and small zonal filters of the new gz;
//   u and v     the backward pass (pgf from gz_f), the u/v update with the
//               pole-row smoothing, and the big filters to u_f, v_f.
// k_tend, k_gzf and k_uvf are those three over the whole grid.  k_stage, which
// gmc_step runs, takes the rows of short filters through all three in one
// tile, and the polar rows in bands of whole circles or in three launches.
// The filter items are (row, column chunk) pieces from a host-built list, so
// that polar rows with hundreds of taps are spread over many workgroups.
// Every expression is the same point formula as the operator-level kernels
// (gmc_point.hpp), so all paths give the same bits.
#include <hip/hip_ext.h>

#include <algorithm>
#include <vector>

#include "gmc_internal.hpp"
#include "gmc_point.hpp"
#include "gmc_stage_map.hpp"
#include "../../include/gmcore_ens.h"

namespace gmc {

namespace {

constexpr int LX = LC + 1;              // m and v_f rows in LDS: lane 63 also holds the column east of it
// launch-shape parameters (the defaults are the measured best on MI355X;
// the macros let a sweep build other shapes)
#ifndef GMC_TY_MAIN
#define GMC_TY_MAIN 11
#endif
#ifndef GMC_FILTER_THREADS
#define GMC_FILTER_THREADS 256
#endif
#ifndef GMC_CHUNK_WORK
#define GMC_CHUNK_WORK 32768
#endif
#ifndef GMC_NARROW_CHUNK
#define GMC_NARROW_CHUNK (2 * GMC_FILTER_THREADS)
#endif
constexpr int TY_MAIN = GMC_TY_MAIN;    // output rows of the single-member k_tend tile
constexpr int NF = GMC_FILTER_THREADS;  // threads per workgroup of the filter kernels
constexpr int NXCD = 8;                 // XCDs of an MI355X
// A k_tend tile with TY output rows: LR = TY + 5 tile rows (r = R0-2 ..
// R0+TY+2), one wavefront each.
template <int TY_> struct Tile {
  static constexpr int TY = TY_;
  static constexpr int LR = TY + 5;
  static constexpr int NT = LR * kWave;
  static constexpr int SH_TILES = LR * (2 * LX + 5 * LC);   // LDS field tiles
  static constexpr int SH_ALL = SH_TILES + 8;
  static constexpr int kMaxPoleLon = SH_TILES / 3;          // the pole sums keep 3 row terms in the tile area
};

struct StagePtrs {
  const double *gz_star, *gzs, *u_f, *v_f, *gz_old;
  double *gz_new, *du, *dv;
};

// the `order` argument of pv_edge: upwind_order_pv, or the limiter for tvd
inline int pv_order(const gmc_config &cfg) {
  return cfg.pv_scheme == GMC_PV_TVD ? cfg.tvd_limiter : cfg.upwind_order_pv;
}

// pv at vertex (r, i) from global memory: rows reached through the
// cross-pole mirror next to the poles
template <class MT, class PT>
__device__ double pv_global(const Grid &g, const MT &M, double grav, double rgrav, int stokes, const double *pole,
                            const PT &P, int r, int i) {
  const int64_t p = g.pitch;
  const int ip = wrap(i + 1, g.nlon);
  auto m = [&](int rr, int ii) { return div_rn(P.gz_star[rr * p + ii] - P.gzs[rr * p + ii], grav, rgrav); };
  double vor;
  if (stokes && r == 0) vor = pole[4];
  else if (stokes && r == g.nhalf - 1) vor = pole[5];
  else vor = vor_of(P.u_f[r * p + i], P.u_f[(r + 1) * p + i], P.v_f[r * p + ip], P.v_f[r * p + i], M, r);
  return pv_of(vor, M, r, m_vtx_of(m(r, i), m(r, ip), m(r + 1, i), m(r + 1, ip), M, r));
}

// Pole reductions of the star state for one pole (zonal_sum call sites in
// calc_ke :320-349, calc_vor :640-674, calc_grad_mf :974-1003): the row
// terms go to LDS scratch, one wavefront adds them in the fixed order of
// wave_zonal_sum.  pole[north] = ke, pole[2+north] = dmfdlat at the pole
// cell, pole[4+north] = vor of the vertex row next to the pole.
template <int NT, class MT, class PT>
__device__ void pole_sums(const Grid &g, const MT &M, double grav, double rgrav, const PT &P, int north,
                          double *scratch, double *pole) {
  const int tid = threadIdx.x, n = g.nlon;
  const int64_t p = g.pitch;
  const int vr = north ? g.nhalf - 1 : 0, cr = north ? g.nlat - 1 : 0, ur = north ? g.nlat - 2 : 1;
  const double le = M(GMC_LE_LAT, vr), ac = M(GMC_AREA_CELL, cr);
  const double w1 = M(GMC_HALF_TANGENT_WGT1, vr), w2 = M(GMC_HALF_TANGENT_WGT2, vr);
  double *t0 = scratch, *t1 = scratch + n, *t2 = scratch + 2 * n;
  auto m = [&](int r, int i) { return div_rn(P.gz_star[r * p + i] - P.gzs[r * p + i], grav, rgrav); };
  for (int i = tid; i < n; i += NT) {
    const int im = wrap(i - 1, n), ip = wrap(i + 1, n);
    const double v = P.v_f[vr * p + i];
    const double m_lat = (m(vr, i) + m(vr + 1, i)) * 0.5;
    const double mu = m(ur, i);
    const double mfx_w = (m(ur, im) + mu) * 0.5 * P.u_f[ur * p + im];
    const double mfx_e = (mu + m(ur, ip)) * 0.5 * P.u_f[ur * p + i];
    // mfx_lat of the V row: the pole U row contributes zero flux
    const double t = north ? tangent_sum(w1, w2, mfx_w, mfx_e, 0.0, 0.0) : tangent_sum(w1, w2, 0.0, 0.0, mfx_w, mfx_e);
    const double ul = t / m_lat;
    const double mfy = m_lat * v;
    t0[i] = v * v;
    t1[i] = north ? -mfy : mfy;
    t2[i] = north ? ul * le : -ul * le;
  }
  __syncthreads();
  // one wavefront per sum (workgroups here have at least three)
  const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
  if (w < 3) {
    const double s = wave_zonal_sum_batched(n, tid % kWave, scratch + w * n);
    if (tid % kWave == 0) {
      const double nl = (double)n;
      pole[2 * w + north] = w == 0 ? s / nl : (w == 1 ? s * le / nl / ac : s / nl / ac);
    }
  }
  __syncthreads();
}

// Row records of the metric table in the constant address space: a record
// index uniform over the wavefront makes every access a scalar load, so the
// metric terms sit in scalar registers and take neither LDS nor vector ones.
typedef const __attribute__((address_space(4))) double *RecPtr;

// The records of rows r - 1, r, r + 1 for the point formulas: M(f, r') and
// M.div(x, f, r'), which divides through the record's reciprocal.  Rows
// beyond the table read its zero records.  (Forcing a phase's terms to be
// loaded ahead of its barrier spilled scalar registers and was slower.)
struct MeshRow {
  RecPtr m1, c0, p1;
  int r;
  __device__ __forceinline__ MeshRow(RecPtr base, int nlat, int r_) : r(r_) {
    auto rec = [&](int rr) { return base + (min(max(rr, -1), nlat) + 1) * kRowRec; };
    m1 = rec(r - 1);
    c0 = rec(r);
    p1 = rec(r + 1);
  }
  __device__ __forceinline__ RecPtr at(int rr) const { return rr == r ? c0 : rr > r ? p1 : m1; }
  __device__ __forceinline__ double operator()(int f, int rr) const { return at(rr)[f]; }
  __device__ __forceinline__ double div(double x, int f, int rr) const {
    return div_rn(x, at(rr)[f], at(rr)[GMC_MESH_NFIELDS + recip_slot(f)]);
  }
};

// Pointers typed in the global address space, and element i of a row whose
// base is uniform over the wavefront through a 32-bit byte offset: the access
// takes the scalar base and one vector register (a row is far below 4 GiB).
template <class T> using gptr = __attribute__((address_space(1))) T *;
template <class T> __device__ __forceinline__ gptr<T> glb(T *p) { return (gptr<T>)p; }
template <class PT> __device__ __forceinline__ double row_ld(PT row, unsigned i) {
  return *(gptr<const double>)((gptr<const char>)row + i * 8u);
}
template <class PT> __device__ __forceinline__ void row_st(PT row, unsigned i, double v) {
  *(gptr<double>)((gptr<char>)row + i * 8u) = v;
}

// The value of the lane west (east) of this one, by a wavefront shift of the
// vector registers: every lane must be active; lane 0 (63) gets 0.
template <int CTRL> __device__ __forceinline__ double lane_shift(double x) {
  union { double d; int i[2]; } u{x};
  u.i[0] = __builtin_amdgcn_update_dpp(0, u.i[0], CTRL, 0xf, 0xf, true);
  u.i[1] = __builtin_amdgcn_update_dpp(0, u.i[1], CTRL, 0xf, 0xf, true);
  return u.d;
}
__device__ __forceinline__ double lane_west(double x) { return lane_shift<0x138>(x); }   // wave_shr:1
__device__ __forceinline__ double lane_east(double x) { return lane_shift<0x130>(x); }   // wave_shl:1

// The global loads of one tile row per lane: gz, gzs, u_f, v_f of its tile
// point, and on lane 63 gz, gzs and v_f of the column east of the tile.
struct TileIn {
  double gz, gzs, uf, vf, gz_x, gzs_x, vf_x;
};

template <class S, class PT>
__device__ __forceinline__ TileIn tile_fetch(const Grid &g, const PT &P, const TileGeo &G) {
  const int64_t p = g.pitch;
  const int k = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int q = threadIdx.x % kWave, r = G.r0 - 2 + k;
  const int ic = G.c0 + q - G.hl;
  // a lane beyond a narrow grid's east side only has to stay in its row
  const int i = min(wrap(ic, g.nlon), g.nlon - 1);
  TileIn in{};
  if (r >= 0 && r < g.nlat) {
    in.gz = row_ld(P.gz_star + r * p, i);
    in.gzs = row_ld(P.gzs + r * p, i);
    in.uf = row_ld(P.u_f + r * p, i);
    if (r < g.nhalf) in.vf = row_ld(P.v_f + r * p, i);
    if (q == LC - 1) {
      const int ix = min(wrap(ic + 1, g.nlon), g.nlon - 1);
      in.gz_x = row_ld(P.gz_star + r * p, ix);
      in.gzs_x = row_ld(P.gzs + r * p, ix);
      if (r < g.nhalf) in.vf_x = row_ld(P.v_f + r * p, ix);
    }
  }
  return in;
}

// Pole sums of the star state into the tile's pole slots, in the tiles that
// read them (a uniform branch per workgroup); uses the tile's LDS as scratch.
template <class S, class MT, class PT>
__device__ __forceinline__ void tile_poles(const Grid &g, const MT &Mg, double grav, double rgrav, const PT &P, int R0,
                                           double *sh) {
  double *pole = sh + S::SH_TILES;
  if (R0 <= 2) pole_sums<S::NT>(g, Mg, grav, rgrav, P, 0, sh, pole);
  if (R0 + S::TY + 3 >= g.nlat - 1) pole_sums<S::NT>(g, Mg, grav, rgrav, P, 1, sh, pole);
}

// the six upwind derivatives of an edge point, column i of the row at `row` of
// the fields, into a tape
__device__ __forceinline__ void tape_upwind(double *const *dst, int64_t row, unsigned i, const UpwD &d) {
  row_st(dst[0] + row, i, d.dt);
  row_st(dst[1] + row, i, d.dn);
#pragma unroll
  for (int j = 0; j < 4; j++) row_st(dst[2 + j] + row, i, d.df[j]);
}

// A short zonal filter (half width H) of a value held one column a lane, taps
// in ascending order as filter_point.
template <int H> __device__ __forceinline__ double lane_taps(double x, RecPtr w) {
  double t[2 * H + 1];
  t[H] = x;
#pragma unroll
  for (int j = 1; j <= H; j++) {
    t[H - j] = lane_west(t[H - j + 1]);
    t[H + j] = lane_east(t[H + j - 1]);
  }
  double acc = 0.0;
#pragma unroll
  for (int j = 0; j < 2 * H + 1; j++) acc = acc + w[j] * t[j];
  return acc;
}
template <class WT> __device__ __forceinline__ double lane_filter(double x, int n, WT wgt) {
  const RecPtr w = (RecPtr)wgt;
  if (n == 5) return lane_taps<2>(x, w);
  if (n == 3) return lane_taps<1>(x, w);
  if (n == 7) return lane_taps<3>(x, w);
  if (n == 9) return lane_taps<4>(x, w);
  return x;
}

// What the rest of a stage reads and writes in a tile that does all of it.
template <class FT, class CP, class WP> struct TileRest {
  FT big, small;
  CP u_old, v_old;
  WP u, v, u_f, v_f, gz_f, gz;
};

// One tile of the forward tendencies and the unfiltered gz update of the
// points G owns, LDS scratch sh[S::SH_ALL].  The tile's pole slots hold its
// pole sums (tile_poles) and io its loads (tile_fetch) on entry.  With TAPE
// the tile also writes the star state's intermediates of its output points to
// *tape.  With FULL the tile, on rows of short filters (at most kLaneTaps)
// away from the poles, does the rest of the stage as well: the filters of gz
// by lane shifts, the gz_f of the row north through LDS, u and v and their
// filters.  A lane's filtered u takes 1 + h + h' columns either side (h, h'
// the half widths of the filters of gz and of u), 54 of 64 lanes at h = 2;
// what that recomputes is less than the gz, du, dv and gz_f that three
// kernels pass through memory.
//
// A wavefront owns one tile row in every phase and all its 64 lanes run every
// formula, so the columns on either side come from wavefront shifts and only
// the rows on either side from LDS (16 reads a point); the lanes whose stencil
// leaves the tile form values that no output point reads.  Reading both kinds
// of neighbour and the metric rows from LDS (90 reads a point) kept the LDS
// pipe, which a CU's four SIMDs share, busy for half of the launch.
struct NoRest {};
template <class S, bool TAPE, bool FULL, class MT, class PT, class RT>
__device__ __forceinline__ void tend_tile(const Grid &g, const MT &Mg, RecPtr mrows, double grav, double rgrav,
                                          double dt, int stokes, int pv_scheme, int order, double wgt, int coriolis,
                                          const PT &P, const TileGeo &G, double *sh, const TileIn &io,
                                          const TapeOut *tape, const RT &rest) {
  double(*sm)[LX] = (double(*)[LX])sh;
  double(*svf)[LX] = (double(*)[LX])(sh + S::LR * LX);
  double *shc = sh + 2 * S::LR * LX;
  double(*suf)[LC] = (double(*)[LC])shc;
  double(*smfx)[LC] = (double(*)[LC])(shc + 1 * S::LR * LC);
  double(*smfy)[LC] = (double(*)[LC])(shc + 2 * S::LR * LC);
  double(*spv)[LC] = (double(*)[LC])(shc + 3 * S::LR * LC);
  double(*ske)[LC] = (double(*)[LC])(shc + 4 * S::LR * LC);
  double(*spl)[LC] = suf;  // pv_lon and pv_lat replace u_f and v_f, which
  double(*spt)[LX] = svf;  // no row reads from LDS after phase B
  const double *pole = sh + S::SH_TILES;

  const int64_t p = g.pitch;
  const int nlat = g.nlat, nhalf = g.nhalf;
  const int k = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);   // tile row of this wavefront
  const int q = threadIdx.x % kWave;                                   // tile column of this lane
  const int r = G.r0 - 2 + k;                                          // global row
  const int ic = G.c0 + q - G.hl;                                      // output column
  const int kn = min(k + 1, S::LR - 1), ks = max(k - 1, 0), kss = max(k - 2, 0);
  const bool out_pt = k >= 2 && r < G.r1 && q >= G.hl && q < G.hl + G.nc;
  const bool u_row = r >= 1 && r <= nlat - 2, v_row = r >= 0 && r < nhalf;
  const MeshRow M(mrows, nlat, r);

  // A: m, u_f, v_f of the row
  const double uf = io.uf, vf = io.vf;
  const double m0 = div_rn(io.gz - io.gzs, grav, rgrav);   // m_of; 0 beyond the poles
  sm[k][q] = m0;
  svf[k][q] = vf;
  suf[k][q] = uf;
  if (q == LC - 1) {
    sm[k][LC] = div_rn(io.gz_x - io.gzs_x, grav, rgrav);
    svf[k][LC] = io.vf_x;
  }
  if (TAPE && out_pt && tape->u_f) {
    row_st(tape->u_f + r * p, ic, uf);
    if (v_row) row_st(tape->v_f + r * p, ic, vf);
  }
  __syncthreads();

  // B: mass fluxes (rows 1 .. TY+2), pv (rows 0 .. TY+3), ke (rows 2 .. TY+2),
  // the row's three chains in one block; then what the rows at and beyond the
  // poles hold instead
  const double m1 = sm[k][q + 1], m2 = sm[kn][q], m3 = sm[kn][q + 1];
  const double u1 = suf[kn][q], v1 = svf[k][q + 1], vs = svf[ks][q], uw = lane_west(uf);
  double mfx = (m0 + m1) * 0.5 * uf;
  double mfy = (m0 + m2) * 0.5 * vf;
  const double mv = m_vtx_of(m0, m1, m2, m3, M, r);
  double pv = pv_of(vor_of(uf, u1, v1, vf, M, r), M, r, mv);
  double ke = ke_of(uw, uf, vs, vf, M, r);
  if (r < 2 || r > nlat - 3) {
    if (!u_row) {
      mfx = 0.0;
      ke = r == 0 ? pole[0] : r == nlat - 1 ? pole[1] : 0.0;
    }
    if (!v_row) {
      mfy = 0.0;
      pv = 0.0;
      if (r >= -2 && r <= nhalf + 1) {
        int rr = r, ii = min(wrap(ic, g.nlon), g.nlon - 1);
        mirror_half(rr, ii, g);
        pv = pv_global(g, Mg, grav, rgrav, stokes, pole, P, rr, ii);
      }
    } else if (stokes && (r == 0 || r == nhalf - 1)) {
      pv = pv_of(r == 0 ? pole[4] : pole[5], M, r, mv);
    }
  }
  smfx[k][q] = mfx;
  smfy[k][q] = mfy;
  spv[k][q] = pv;
  ske[k][q] = ke;
  if (TAPE && out_pt && v_row) {
    row_st(tape->m_vtx + r * p, ic, mv);
    row_st(tape->pv + r * p, ic, pv);
    row_st(tape->mfy + r * p, ic, mfy);
    row_st(tape->m_lat + r * p, ic, (m0 + m2) * 0.5);
  }
  __syncthreads();

  // D: tangential winds and pv on the edges (U rows 2 .. TY+2, V rows 1 ..
  // TY+1); phase E's gz_old is on its way meanwhile
  double gz_old = 0.0;
  const int il = min(wrap(ic, g.nlon), g.nlon - 1);
  if (FULL ? k >= 2 && r <= G.r1 : out_pt) gz_old = row_ld(P.gz_old + r * p, FULL ? il : ic);
  const double mfy_s = smfy[ks][q], mfx_n = smfx[kn][q];
  double pl = 0.0, pt = 0.0;
  if (k >= 1 && k < S::TY + 3) {
    auto lon_tangent = [&] {
      return tangent_sum(M(GMC_FULL_TANGENT_WGT1, r), M(GMC_FULL_TANGENT_WGT2, r), mfy_s, lane_east(mfy_s), mfy,
                         lane_east(mfy));
    };
    auto lat_tangent = [&] {
      return tangent_sum(M(GMC_HALF_TANGENT_WGT1, r), M(GMC_HALF_TANGENT_WGT2, r), lane_west(mfx), mfx,
                         lane_west(mfx_n), mfx_n);
    };
    if (TAPE) {   // an edge at a time: both with their tapes are more than the registers
      {
        const double pss = spv[kss][q], ps = spv[ks][q], pn = spv[kn][q];
        const double t = lon_tangent(), ml = (m0 + m1) * 0.5, vl = div_mid(t, ml);
        pl = pv_edge(pv_scheme, order, wgt, vl, uf, 0, dt, M(GMC_LE_LON, r), pss, ps, pv, pn);
        if (!u_row) pl = 0.0;
        if (out_pt && u_row) {
          row_st(tape->m_lon + r * p, ic, ml);
          row_st(tape->mfx + r * p, ic, mfx);
          if (tape->mfy_lon) row_st(tape->mfy_lon + r * p, ic, t);
          row_st(tape->v_lon + r * p, ic, vl);
          row_st(tape->pv_lon + r * p, ic, pl);
          if (tape->dlon[0])
            tape_upwind(tape->dlon, r * p, ic, upwind_deriv(pv_scheme, order, wgt, vl, uf, 0, pss, ps, pv, pn));
        }
      }
      const double pw = lane_west(pv), pww = lane_west(pw), pe = lane_east(pv);
      const double t = lat_tangent(), ul = div_mid(t, (m0 + m2) * 0.5);
      pt = pv_edge(pv_scheme, order, wgt, ul, vf, 1, dt, M(GMC_LE_LAT, r), pww, pw, pv, pe);
      if (!v_row) pt = 0.0;
      if (out_pt && v_row) {
        if (tape->mfx_lat) row_st(tape->mfx_lat + r * p, ic, t);
        row_st(tape->u_lat + r * p, ic, ul);
        row_st(tape->pv_lat + r * p, ic, pt);
        if (tape->dlat[0])
          tape_upwind(tape->dlat, r * p, ic, upwind_deriv(pv_scheme, order, wgt, ul, vf, 1, pww, pw, pv, pe));
      }
    } else {
      const double pss = spv[kss][q], ps = spv[ks][q], pn = spv[kn][q];
      const double pw = lane_west(pv), pww = lane_west(pw), pe = lane_east(pv);
      const double vl = div_mid(lon_tangent(), (m0 + m1) * 0.5);
      const double ul = div_mid(lat_tangent(), (m0 + m2) * 0.5);
      if (pv_scheme == GMC_PV_UPWIND && order == 3) {   // both edges in one block
        pl = pv_upwind_edge(3, wgt, vl, uf, 0, pss, ps, pv, pn);
        pt = pv_upwind_edge(3, wgt, ul, vf, 1, pww, pw, pv, pe);
      } else {
        pl = pv_edge(pv_scheme, order, wgt, vl, uf, 0, dt, M(GMC_LE_LON, r), pss, ps, pv, pn);
        pt = pv_edge(pv_scheme, order, wgt, ul, vf, 1, dt, M(GMC_LE_LAT, r), pww, pw, pv, pe);
      }
      if (!u_row) pl = 0.0;
      if (!v_row) pt = 0.0;
    }
  }
  spl[k][q] = pl;
  spt[k][q] = pt;
  __syncthreads();

  // E: du, dv (forward pass) and gz_new = gz_old + dt dgz on the output rows
  // (FULL: gz also on the row north of them)
  if (!FULL && (k < 2 || k >= S::TY + 2)) return;
  double u_old = 0.0, v_old = 0.0;
  if constexpr (FULL)
    if (k >= 2 && r < G.r1) {
      u_old = row_ld(rest.u_old + r * p, il);
      v_old = row_ld(rest.v_old + r * p, il);
    }
  const double pt_s = spt[ks][q], pt_se = lane_east(pt_s), pt_e = lane_east(pt);
  const double pl_n = spl[kn][q], pl_nw = lane_west(pl_n), pl_w = lane_west(pl);
  const double mfy_e = lane_east(mfy), mfy_se = lane_east(mfy_s), mfx_w = lane_west(mfx), mfx_nw = lane_west(mfx_n);
  const double ke_0 = ske[k][q], ke_e = lane_east(ke_0), ke_n = ske[kn][q];
  const double qhv = coriolis == 1
      ? qhv_of(M, r, pl, mfy_s, pt_s, mfy_se, pt_se, mfy, pt, mfy_e, pt_e)
      : tangent_sum(M(GMC_FULL_TANGENT_WGT1, r), M(GMC_FULL_TANGENT_WGT2, r), mfy_s, mfy_se, mfy, mfy_e) * pl;
  const double qhu = coriolis == 1
      ? qhu_of(M, r, pt, mfx_w, pl_w, mfx, pl, mfx_nw, pl_nw, mfx_n, pl_n)
      : tangent_sum(M(GMC_HALF_TANGENT_WGT1, r), M(GMC_HALF_TANGENT_WGT2, r), mfx_w, mfx, mfx_nw, mfx_n) * pt;
  const double dku = M.div(ke_e - ke_0, GMC_DE_LON, r);
  const double dkv = M.div(ke_n - ke_0, GMC_DE_LAT, r);
  double dgz = -(dmfdlon_of(mfx, mfx_w, M, r) + dmfdlat_of(mfy, mfy_s, M, r)) * grav;
  if (!FULL && !u_row) {   // the pole rows: gz from the pole sums
    const double dmfdlon = 0.0, dmfdlat = r == 0 ? pole[2] : pole[3];
    dgz = -(dmfdlon + dmfdlat) * grav;
  }
  const double gz_new = gz_old + dt * dgz;
  if constexpr (!FULL) {
    if (out_pt) {
      if (u_row) row_st(P.du + r * p, ic, qhv - dku);
      if (v_row) row_st(P.dv + r * p, ic, -qhu - dkv);
      row_st(P.gz_new + r * p, ic, gz_new);
    }
  } else {
    // F: the filters of gz; the row's gz_f to the row south of it, over pv
    double gz_f = 0.0;
    if (k >= 2 && r <= G.r1) {
      const auto nb = *((const __attribute__((address_space(4))) int32_t *)rest.big.ngrid_lon + r);
      gz_f = lane_filter(gz_new, nb, rest.big.wgt_lon + (int64_t)r * rest.big.max_taps);
      spv[k][q] = gz_f;
    }
    __syncthreads();
    if (k < 2 || r >= G.r1) return;
    const auto ns = *((const __attribute__((address_space(4))) int32_t *)rest.small.ngrid_lon + r);
    const auto nu = *((const __attribute__((address_space(4))) int32_t *)rest.big.ngrid_lon + r);
    const auto nv = *((const __attribute__((address_space(4))) int32_t *)rest.big.ngrid_lat + r);
    const double gz_s = lane_filter(gz_new, ns, rest.small.wgt_lon + (int64_t)r * rest.small.max_taps);
    // G: u, v and their filters
    const double u = u_old + dt * ((qhv - dku) - pgf_lon_of(lane_east(gz_f), gz_f, M, r));
    const double v = v_old + dt * ((-qhu - dkv) - pgf_lat_of(spv[kn][q], gz_f, M, r));
    const double u_f = lane_filter(u, nu, rest.big.wgt_lon + (int64_t)r * rest.big.max_taps);
    const double v_f = lane_filter(v, nv, rest.big.wgt_lat + (int64_t)r * rest.big.max_taps);
    if (out_pt) {
      row_st(rest.gz_f + r * p, ic, gz_f);
      row_st(rest.gz + r * p, ic, gz_s);
      row_st(rest.u + r * p, ic, u);
      row_st(rest.v + r * p, ic, v);
      row_st(rest.u_f + r * p, ic, u_f);
      row_st(rest.v_f + r * p, ic, v_f);
    }
  }
}

// tile (tx, ty) of a cover of the grid by 60 x TY tiles
template <class S> __device__ __forceinline__ TileGeo tile_geo(const Grid &g, int tx, int ty) {
  const int c0 = tx * TX, r0 = ty * S::TY;
  return TileGeo{c0, min(TX, g.nlon - c0), HXL, r0, min(r0 + S::TY, g.nlat)};
}

// Forward tendencies and the unfiltered gz update on a 60 x TY_MAIN tile.
// Wavefront k owns tile row k (global row R0 - 2 + k) in every phase and lane
// q the column C0 - 2 + q, so metric terms are wave-uniform.  Blocks are
// dealt to the XCDs round-robin; each XCD gets a contiguous run of tiles
// (row-major), so vertically adjacent tiles share that XCD's L2.  The XCD
// holding the north pole walks its run backwards so that the polar tiles,
// which also form the pole sums, start first.
constexpr int kTendThreads = Tile<TY_MAIN>::NT;
template <bool TAPE>
__global__ void __launch_bounds__(kTendThreads, 8) k_tend(Grid g, Mesh Mg, const double *__restrict__ mrows,
                                                          double grav, double rgrav, double dt, int stokes,
                                                          int pv_scheme, int order, double wgt, int coriolis,
                                                          StagePtrs P, TapeOut tape) {
  using S = Tile<TY_MAIN>;
  __shared__ double sh[S::SH_ALL];
  // tile of this block
  const int nx = (g.nlon + TX - 1) / TX, ny = (g.nlat + S::TY - 1) / S::TY, T = nx * ny;
  const int b = blockIdx.x, x = b % NXCD;
  const int t = x == NXCD - 1 ? T - 1 - b / NXCD : xcd_item(b, T);
  const TileGeo G = tile_geo<S>(g, t % nx, t / nx);
  const TileIn io = tile_fetch<S>(g, P, G);
  tile_poles<S>(g, Mg, grav, rgrav, P, G.r0, sh);
  tend_tile<S, TAPE, false>(g, Mg, (RecPtr)mrows, grav, rgrav, dt, stokes, pv_scheme, order, wgt, coriolis, P, G, sh,
                            io, &tape, NoRest{});
}

// ---------------------------------------------------------------------------
// zonal filters over (row, column chunk) work items
struct Item {
  int32_t row, c0, c1, kind;  // kind: 0 gz (cell row), 1 u (U row), 2 v (V row)
  int32_t member;             // ensemble member (0 for a single context)
  int32_t n, n2;              // taps of the row's filters (copies of the filter tables): the big filter
                              // of the item's row kind, and small_filter1 for gz items
  int32_t pad;
};

// column i - h + t of a row, t in [0, nlon + 2h), h <= nlon
__device__ __forceinline__ int wrap2(int c, int n) { return c < 0 ? c + n : (c >= n ? c - n : c); }

// big filter gz_new -> gz_f and small filter gz_new -> gz
// (time_schemes_mod.F90:184-191, filter_mod.F90:25-50).  Weights and the
// row window are staged in LDS: xs = [weights big | weights small | window].
template <class FT, class CP, class WP>
__device__ __forceinline__ void gzf_item(const Grid &g, const FT &big, const FT &small, const Item &it, CP gz_new,
                                         WP gz_f, WP gz, double *xs, int tid) {
  const int r = it.row;
  const int64_t o = r * g.pitch;
  const int nb = it.n, ns = it.n2;
  const int hb = nb > 1 ? (nb - 1) / 2 : 0, hs = ns > 1 ? (ns - 1) / 2 : 0, hw = hb > hs ? hb : hs;
  double *wb = xs, *ws = wb + max(nb, 0), *x0 = ws + max(ns, 0);
  const int len = it.c1 - it.c0 + 2 * hw;
  for (int k = tid; k < nb; k += NF) wb[k] = big.wgt_lon[(int64_t)r * big.max_taps + k];
  for (int k = tid; k < ns; k += NF) ws[k] = small.wgt_lon[(int64_t)r * small.max_taps + k];
  for (int t = tid; t < len; t += 4 * NF) {
    double v[4];
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (t + u * NF < len) v[u] = gz_new[o + wrap2(it.c0 - hw + t + u * NF, g.nlon)];
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (t + u * NF < len) x0[t + u * NF] = v[u];
  }
  __syncthreads();
  for (int c = it.c0 + tid; c < it.c1; c += NF) {
    const double *x = x0 + (c - it.c0);      // x[hw] is column c
    gz_f[o + c] = nb > 1 ? filter_point(wb, nb, x + hw - hb) : x[hw];
    gz[o + c] = ns > 1 ? filter_point(ws, ns, x + hw - hs) : x[hw];
  }
}

__global__ void __launch_bounds__(NF) k_gzf(Grid g, FilterDev big, FilterDev small, const Item *__restrict__ items,
                                            const double *__restrict__ gz_new, double *gz_f, double *gz) {
  extern __shared__ double xs[];
  gzf_item(g, big, small, items[xcd_item(blockIdx.x, gridDim.x)], gz_new, gz_f, gz, xs, threadIdx.x);
}

struct UVPtrs {
  const double *u_old, *v_old, *du, *dv, *gz_f;
  double *u, *v, *u_f, *v_f;
};

// backward pass + u/v update + big filters
// (gmcore_mod.F90:552-571, time_schemes_mod.F90:198-239).  xs = [weights |
// window of the updated row].
template <class MT, class FT, class PT>
__device__ __forceinline__ void uvf_item(const Grid &g, const MT &M, double dt, const FT &big,
                                         const Item &it, const PT &P, double *xs, int tid) {
  const int r = it.row;
  const int64_t p = g.pitch, o = r * p;
  const int nl = g.nlon;
  const bool pole_u = it.kind == 1 && (r == 0 || r == g.nlat - 1);   // not updated, copied to u_f
  const int n = pole_u ? 0 : it.n;
  double *w = xs, *x0 = xs + max(n, 0);
  const int h = n > 1 ? (n - 1) / 2 : 0;
  const int len = it.c1 - it.c0 + 2 * h;
  const auto wg = (it.kind == 1 ? big.wgt_lon : big.wgt_lat) + (int64_t)r * big.max_taps;
  for (int k = tid; k < n; k += NF) w[k] = wg[k];
  if (pole_u) {
    for (int c = it.c0 + tid; c < it.c1; c += NF) P.u_f[o + c] = P.u[o + c];
  } else if (it.kind == 1) {
    const double de = M(GMC_DE_LON, r), rde = 1.0 / de;
    for (int t = tid; t < len; t += 4 * NF) {
      double uo[4], du[4], ge[4], gw[4];
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (t + u * NF < len) {
          const int i = wrap2(it.c0 - h + t + u * NF, nl);
          uo[u] = P.u_old[o + i];
          du[u] = P.du[o + i];
          ge[u] = P.gz_f[o + wrap(i + 1, nl)];
          gw[u] = P.gz_f[o + i];
        }
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (t + u * NF < len) x0[t + u * NF] = uo[u] + dt * (du[u] - div_rn(ge[u] - gw[u], de, rde));
    }
  } else {
    const int pole = r == 0 ? 1 : (r == g.nhalf - 1 ? -1 : 0);   // neighbour row of the smoothing
    const double de0 = M(GMC_DE_LAT, r), de1 = pole ? M(GMC_DE_LAT, r + pole) : 1.0;
    const double rde0 = 1.0 / de0, rde1 = 1.0 / de1;
    for (int t = tid; t < len; t += 2 * NF) {
      double a[2][8];
#pragma unroll
      for (int u = 0; u < 2; u++)
        if (t + u * NF < len) {
          const int64_t q = o + wrap2(it.c0 - h + t + u * NF, nl);
          a[u][0] = P.v_old[q]; a[u][1] = P.dv[q]; a[u][2] = P.gz_f[q + p]; a[u][3] = P.gz_f[q];
          if (pole) {
            const int64_t q1 = q + pole * p;
            a[u][4] = P.v_old[q1]; a[u][5] = P.dv[q1]; a[u][6] = P.gz_f[q1 + p]; a[u][7] = P.gz_f[q1];
          }
        }
#pragma unroll
      for (int u = 0; u < 2; u++)
        if (t + u * NF < len) {
          double v = a[u][0] + dt * (a[u][1] - div_rn(a[u][2] - a[u][3], de0, rde0));
          if (pole) v = pole_smooth(v, a[u][4] + dt * (a[u][5] - div_rn(a[u][6] - a[u][7], de1, rde1)));
          x0[t + u * NF] = v;
        }
    }
  }
  __syncthreads();
  if (pole_u) return;
  const auto out = it.kind == 1 ? P.u : P.v;
  const auto out_f = it.kind == 1 ? P.u_f : P.v_f;
  for (int c = it.c0 + tid; c < it.c1; c += NF) {
    const double *x = x0 + (c - it.c0);
    out[o + c] = x[h];
    out_f[o + c] = n > 1 ? filter_point(w, n, x) : x[h];
  }
}

__global__ void __launch_bounds__(NF) k_uvf(Grid g, Mesh M, double dt, FilterDev big, const Item *__restrict__ items,
                                            UVPtrs P) {
  extern __shared__ double xs[];
  uvf_item(g, M, dt, big, items[xcd_item(blockIdx.x, gridDim.x)], P, xs, threadIdx.x);
}


// ---------------------------------------------------------------------------
// A whole stage of a band of rows in one workgroup, for rows whose filters
// are too wide for a tile's lanes, on grids whose latitude circles fit a band
// into LDS.
//
// The workgroup owns up to TY v rows over whole circles, so every stencil and
// filter of the stage stays inside it: it forms the tendencies of its rows and
// of the rows around them, filters gz on its rows and the next one north,
// updates u and v and filters them, with a barrier where the three kernels
// have a launch.  The expressions and their order are theirs, so both forms
// give the same bits.
//
// Band b: v rows r0 .. r0+nv-1, the cell and U rows of the same numbers, and
// in the last band the pole row north of them.  Local row k is global row
// r0 - 2 + k.  The two v rows next to a pole share a band (the smoothing of
// the pole row reads both).
constexpr int NB_T = 1024;              // threads of a band's workgroup
constexpr int NB_W = NB_T / kWave;
constexpr int kBandTY = 2;              // v rows of a band
constexpr int kBandRows = kBandTY + 5;  // local rows: two south, three north of the v rows
constexpr int kBandLoads = 4;           // (row, 64-column) tasks per wavefront: loads of the local rows,
constexpr int kBandOut = 2;             // and its output rows
struct Band {
  int r0, nv;
  int part, parts;   // of several workgroups that form the same band, the columns part / parts
};
// LDS rows of nlon doubles: m, u_f, v_f; mfx and mfy (local rows 1 .. TY+2),
// pv (0 .. TY+3), ke (2 .. TY+2)
constexpr int kBandLdsRows = 3 * kBandRows + 2 * (kBandTY + 2) + (kBandTY + 4) + (kBandTY + 1);

// The (row, segment) tasks of a wavefront, every nw-th from its own: a scalar
// division per task would cost as much as the task's loads.
struct Tasks {
  int row, seg, segs, drow, dseg;
  __device__ __forceinline__ Tasks(int w, int segs_, int nw) : segs(segs_) {
    row = w / segs;
    seg = w - row * segs;
    drow = nw / segs;
    dseg = nw - drow * segs;
  }
  __device__ __forceinline__ void next() {
    row += drow;
    seg += dseg;
    if (seg >= segs) {
      seg -= segs;
      row++;
    }
  }
};

// Two neighbouring outputs of a zonal filter of n taps (filter_point's sums):
// x points at the even column's window.  Each tap needs one more value of the
// window, read in 16-byte pairs: half of filter_point's LDS reads per output,
// which bound a wide filter's workgroup.
__device__ __forceinline__ void filter_pair(const double *w, int n, const double *x, double &o0, double &o1) {
  typedef double d2 __attribute__((ext_vector_type(2)));
  double a0 = 0.0, a1 = 0.0, cur;
  int k = 0;
  if ((__builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)x) & 8) == 0) {   // x[0] on a pair's boundary
    const d2 p = *(const d2 *)x;
    a0 = a0 + w[0] * p.x;
    a1 = a1 + w[0] * p.y;
    cur = p.y;
    k = 1;
  } else {
    cur = x[0];
  }
  for (; k + 8 <= n; k += 8) {
    d2 p[4];
    double wk[8];
#pragma unroll
    for (int u = 0; u < 4; u++) p[u] = *(const d2 *)(x + k + 1 + 2 * u);
#pragma unroll
    for (int u = 0; u < 8; u++) wk[u] = w[k + u];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      a0 = a0 + wk[2 * u] * cur;
      a1 = a1 + wk[2 * u] * p[u].x;
      a0 = a0 + wk[2 * u + 1] * p[u].x;
      a1 = a1 + wk[2 * u + 1] * p[u].y;
      cur = p[u].y;
    }
  }
  for (; k < n; k++) {
    const double nx = x[k + 1];
    a0 = a0 + w[k] * cur;
    a1 = a1 + w[k] * nx;
    cur = nx;
  }
  o0 = a0;
  o1 = a1;
}

struct BandOut {
  double *gz_f, *gz;
};

template <bool TAPE>
__device__ __forceinline__ void band_stage(const Grid &g, RecPtr mrows, double grav, double rgrav, double dt,
                                           int stokes, int pv_scheme, int order, double wgt, int coriolis,
                                           const FilterDev &big, const FilterDev &small, const Band bd,
                                           const StagePtrs &P, const UVPtrs &U, const BandOut &G, const TapeOut &tape,
                                           double *xs) {
  const int n = g.nlon, nlat = g.nlat, nhalf = g.nhalf, segs = (n + kWave - 1) / kWave;
  const int64_t p = g.pitch;
  constexpr int TY = kBandTY, LR = kBandRows;
  double *sm = xs, *suf = sm + LR * n, *svf = suf + LR * n;
  double *smfx = svf + LR * n - n, *smfy = smfx + (TY + 2) * n;   // row k at + k n, from k = 1
  double *spv = smfy + (TY + 2) * n + n;
  double *ske = spv + (TY + 4) * n - 2 * n;                       // from k = 2
  double *pole = spv + (TY + 4) * n + (TY + 1) * n, *wt = pole + 8;
  double *spl = suf, *spt = svf;   // pv on the edges replaces u_f and v_f element by element
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid / kWave), q = tid % kWave;
  const int r0 = bd.r0, nv = bd.nv;
  const bool south = r0 == 0, north = r0 + nv == nhalf;
  const int nu = nv + (north ? 1 : 0);         // cell rows the band writes
  const int rows = nv + 5;                     // local rows in use

  // ---- the band's loads, all on their way before the first use -----------
  double a_gz[kBandLoads], a_gzs[kBandLoads], a_uf[kBandLoads], a_vf[kBandLoads];
  Tasks T(w, segs, NB_W);
#pragma unroll
  for (int j = 0; j < kBandLoads; j++, T.next()) {
    const int k = T.row, r = r0 - 2 + k, i = T.seg * kWave + q;
    a_gz[j] = a_gzs[j] = a_uf[j] = a_vf[j] = 0.0;
    if (k < rows && r >= 0 && r < nlat && i < n) {
      a_gz[j] = row_ld(P.gz_star + r * p, i);
      a_gzs[j] = row_ld(P.gzs + r * p, i);
      a_uf[j] = row_ld(P.u_f + r * p, i);
      if (r < nhalf) a_vf[j] = row_ld(P.v_f + r * p, i);
    }
  }
  double gz_old[kBandOut], u_old[kBandOut], v_old[kBandOut];
  T = Tasks(w, segs, NB_W);
#pragma unroll
  for (int j = 0; j < kBandOut; j++, T.next()) {
    const int k = 2 + T.row, r = r0 - 2 + k, i = T.seg * kWave + q;
    gz_old[j] = u_old[j] = v_old[j] = 0.0;
    if (k <= nv + 2 && r < nlat && i < n) {
      gz_old[j] = row_ld(P.gz_old + r * p, i);
      if (k < nv + 2) {
        u_old[j] = row_ld(U.u_old + r * p, i);
        v_old[j] = row_ld(U.v_old + r * p, i);
      }
    }
  }
  double u_pole = 0.0;   // n <= NB_T
  if ((south || north) && tid < n) u_pole = row_ld(U.u + (south ? 0 : nlat - 1) * p, tid);
  // filter weights: table rows (zero beyond a row's taps, at most nlon <= NB_T
  // of them) loaded whole, so that no load waits for the tap counts
  double wr[3 * TY + 2];
#pragma unroll
  for (int j = 0; j <= TY; j++) {
    const int r = min(r0 + j, nlat - 1), rv = min(r0 + j, nhalf - 1);
    if (tid < big.max_taps) {
      wr[j] = row_ld(big.wgt_lon + (int64_t)r * big.max_taps, tid);
      if (j < TY) wr[2 * TY + 2 + j] = row_ld(big.wgt_lat + (int64_t)rv * big.max_taps, tid);
    }
    if (tid < small.max_taps) wr[TY + 1 + j] = row_ld(small.wgt_lon + (int64_t)r * small.max_taps, tid);
  }
  // taps of row r0 + j and where its weights sit: big and small filter of the
  // cell (and U) rows, big filter of the v rows
  typedef const __attribute__((address_space(4))) int32_t *TapPtr;
  int nb[TY + 1], ns[TY + 1], nt[TY], ob[TY + 1], os[TY + 1], ot[TY], o = 0;
#pragma unroll
  for (int j = 0; j <= TY; j++) {
    const int r = min(r0 + j, nlat - 1), rv = min(r0 + j, nhalf - 1);
    nb[j] = ((TapPtr)big.ngrid_lon)[r];
    ns[j] = ((TapPtr)small.ngrid_lon)[r];
    ob[j] = o;
    os[j] = ob[j] + max(nb[j], 0);
    o = os[j] + max(ns[j], 0);
    if (j < TY) {
      nt[j] = ((TapPtr)big.ngrid_lat)[rv];
      ot[j] = o;
      o += max(nt[j], 0);
    }
  }
  T = Tasks(w, segs, NB_W);
#pragma unroll
  for (int j = 0; j < kBandLoads; j++, T.next()) {
    const int k = T.row, r = r0 - 2 + k, i = T.seg * kWave + q;
    if (k < rows && i < n) {
      const int e = k * n + i;
      sm[e] = div_rn(a_gz[j] - a_gzs[j], grav, rgrav);   // m_of
      suf[e] = a_uf[j];
      svf[e] = a_vf[j];
      if (TAPE && tape.u_f && k >= 2 && k < 2 + nu) {
        row_st(tape.u_f + r * p, i, a_uf[j]);
        if (r < nhalf) row_st(tape.v_f + r * p, i, a_vf[j]);
      }
    }
  }
#pragma unroll
  for (int j = 0; j <= TY; j++) {
    if (tid < nb[j]) wt[ob[j] + tid] = wr[j];
    if (tid < ns[j]) wt[os[j] + tid] = wr[TY + 1 + j];
    if (j < TY && tid < nt[j]) wt[ot[j] + tid] = wr[2 * TY + 2 + j];
  }
  // the entry of a per-row array for a row index known at run time
  auto pick = [](const int *v, int n_, int j) {
    int x = v[0];
    for (int e = 1; e < n_; e++) x = j == e ? v[e] : x;
    return x;
  };
  __syncthreads();

  // ---- pole sums (pole_sums' terms from LDS), one each for the last three
  // wavefronts while the others form B; the rows that read them follow
  // (the bands that read the vertex row next to a pole: its own, and with two
  // rows a band the one beside it)
  const bool sum_s = r0 <= 2, sum_n = r0 + nv >= nhalf - 2;
  if (sum_s || sum_n) {
    if (const int ws = w - (NB_W - 3); ws >= 0) {
      const int vr = sum_s ? 0 : nhalf - 1, cr = sum_s ? 0 : nlat - 1;
      const int kv = vr - r0 + 2, ku = sum_s ? kv + 1 : kv;
      const MeshRow V(mrows, nlat, vr), Cc(mrows, nlat, cr);
      const double le = V(GMC_LE_LAT, vr), ac = Cc(GMC_AREA_CELL, cr);
      const double w1 = V(GMC_HALF_TANGENT_WGT1, vr), w2 = V(GMC_HALF_TANGENT_WGT2, vr);
      auto term = [&](int i) {
        const double v = svf[kv * n + i];
        if (ws == 0) return v * v;
        const double m_lat = (sm[kv * n + i] + sm[(kv + 1) * n + i]) * 0.5;
        if (ws == 1) {
          const double mfy = m_lat * v;
          return sum_n ? -mfy : mfy;
        }
        const int im = wrap(i - 1, n), ip = wrap(i + 1, n);
        const double *mu = sm + ku * n, *uu = suf + ku * n;
        const double mfx_w = (mu[im] + mu[i]) * 0.5 * uu[im], mfx_e = (mu[i] + mu[ip]) * 0.5 * uu[i];
        const double t = sum_n ? tangent_sum(w1, w2, mfx_w, mfx_e, 0.0, 0.0) : tangent_sum(w1, w2, 0.0, 0.0, mfx_w, mfx_e);
        const double ul = t / m_lat;
        return sum_n ? ul * le : -ul * le;
      };
      // wave_zonal_sum's order, three terms of a lane formed at a time
      double sum = 0.0;
      for (int i = q; i < n; i += 3 * kWave) {
        double t[3];
#pragma unroll
        for (int u = 0; u < 3; u++) t[u] = i + u * kWave < n ? term(i + u * kWave) : 0.0;
#pragma unroll
        for (int u = 0; u < 3; u++)
          if (i + u * kWave < n) sum = sum + t[u];
      }
      for (int x = 1; x < kWave; x <<= 1) sum = sum + __shfl_xor(sum, x, kWave);
      const double nl = (double)n;
      if (q == 0) pole[ws] = ws == 0 ? sum / nl : (ws == 1 ? sum * le / nl / ac : sum / nl / ac);
    }
  }

  // ---- B: mass fluxes, pv, ke (as tend_tile) -----------------------------
  const bool sums = sum_s || sum_n;
  const int r_sum = sum_s ? 0 : nhalf - 1, c_sum = sum_s ? 0 : nlat - 1;   // vertex and cell row of the sums
  const int nw_b = sums ? NB_W - 3 : NB_W;
  for (T = Tasks(w < nw_b ? w : kBandRows * segs, segs, nw_b); T.row < nv + 4; T.next()) {
    const int k = T.row, r = r0 - 2 + k, i = T.seg * kWave + q;
    if (r < 0 || r >= nlat || i >= n) continue;
    const MeshRow M(mrows, nlat, r);
    const int ie = wrap(i + 1, n), iw = wrap(i - 1, n), ks = max(k - 1, 0);
    const double *m_ = sm + k * n, *u_ = suf + k * n, *v_ = svf + k * n;
    const double m0 = m_[i], m1 = m_[ie], m2 = m_[n + i], m3 = m_[n + ie];
    const double uf = u_[i], u1 = u_[n + i], uw = u_[iw], vf = v_[i], v1 = v_[ie], vs = svf[ks * n + i];
    const bool u_row = r >= 1 && r <= nlat - 2, v_row = r < nhalf;
    const double mv = m_vtx_of(m0, m1, m2, m3, M, r);
    // the vertex row of a pole sum keeps m_vtx until the sum is there
    const double pv = stokes && sums && r == r_sum ? mv : pv_of(vor_of(uf, u1, v1, vf, M, r), M, r, mv);
    const double mfx = (m0 + m1) * 0.5 * uf, mfy = (m0 + m2) * 0.5 * vf;
    if (v_row) spv[k * n + i] = pv;
    if (k >= 1 && k <= nv + 2) {
      smfx[k * n + i] = u_row ? mfx : 0.0;
      smfy[k * n + i] = v_row ? mfy : 0.0;
      if (k >= 2 && u_row) ske[k * n + i] = ke_of(uw, uf, vs, vf, M, r);
    }
    if (TAPE && v_row && k >= 2 && k < 2 + nv) {
      row_st(tape.m_vtx + r * p, i, mv);
      if (!(stokes && r == r_sum)) row_st(tape.pv + r * p, i, pv);
      row_st(tape.mfy + r * p, i, mfy);
      row_st(tape.m_lat + r * p, i, (m0 + m2) * 0.5);
    }
  }
  __syncthreads();

  if (sums) {
    const int kv = r_sum - r0 + 2, kc = c_sum - r0 + 2;
    const MeshRow V(mrows, nlat, r_sum);
    for (int i = tid; i < n; i += NB_T) {
      if (stokes) {
        const double pv = pv_of(pole[2], V, r_sum, spv[kv * n + i]);
        spv[kv * n + i] = pv;
        if (TAPE && kv >= 2 && kv < 2 + nv) row_st(tape.pv + r_sum * p, i, pv);
      }
      if (kc >= 2 && kc <= nv + 2) ske[kc * n + i] = pole[0];
    }
    __syncthreads();
  }

  // ---- D: tangential winds and pv on the edges ---------------------------
  // (U rows 2 .. nv+2 and V rows 1 .. nv+1, a task each)
  for (T = Tasks(w, segs, NB_W); T.row < 2 * (nv + 1); T.next()) {
    const bool lon = T.row <= nv;
    const int k = lon ? 2 + T.row : T.row - nv, r = r0 - 2 + k, i = T.seg * kWave + q;
    if (r < 0 || r >= nlat || i >= n) continue;
    const MeshRow M(mrows, nlat, r);
    const int ie = wrap(i + 1, n), iw = wrap(i - 1, n), iww = wrap(i - 2, n), ih = wrap(i + g.half, n);
    const bool u_row = r >= 1 && r <= nlat - 2, v_row = r < nhalf;
    const double *m_ = sm + k * n;
    const double m0 = m_[i];
    const double *fx = smfx + k * n, *fy = smfy + k * n;
    if (lon) {
      if (!u_row) {
        spl[k * n + i] = 0.0;
        continue;
      }
      const double uf = suf[k * n + i];
      double pl;
      const double tl = tangent_sum(M(GMC_FULL_TANGENT_WGT1, r), M(GMC_FULL_TANGENT_WGT2, r), fy[i - n], fy[ie - n], fy[i], fy[ie]);
      const double ml = (m0 + m_[ie]) * 0.5, vl = div_mid(tl, ml);
      // rows beyond a pole are rows on its other side, half a circle away
      const double *v0 = spv + k * n;
      const double a1 = r == 1 ? v0[ih - n] : v0[i - 2 * n], a2 = v0[i - n], a3 = v0[i];
      const double a4 = r == nhalf - 1 ? v0[ih] : v0[i + n];
      if (pv_scheme == GMC_PV_UPWIND && order == 3) pl = pv_upwind_edge(3, wgt, vl, uf, 0, a1, a2, a3, a4);
      else pl = pv_edge(pv_scheme, order, wgt, vl, uf, 0, dt, M(GMC_LE_LON, r), a1, a2, a3, a4);
      if (TAPE && k < 2 + nu) {
        row_st(tape.m_lon + r * p, i, ml);
        row_st(tape.mfx + r * p, i, fx[i]);
        if (tape.mfy_lon) row_st(tape.mfy_lon + r * p, i, tl);
        row_st(tape.v_lon + r * p, i, vl);
        row_st(tape.pv_lon + r * p, i, pl);
        if (tape.dlon[0]) tape_upwind(tape.dlon, r * p, i, upwind_deriv(pv_scheme, order, wgt, vl, uf, 0, a1, a2, a3, a4));
      }
      spl[k * n + i] = pl;
    }
    if (!lon) {
      if (!v_row) continue;
      const double vf = svf[k * n + i];
      double pt;
      const double tu = tangent_sum(M(GMC_HALF_TANGENT_WGT1, r), M(GMC_HALF_TANGENT_WGT2, r), fx[iw], fx[i], fx[n + iw], fx[n + i]);
      const double ul = div_mid(tu, (m0 + m_[n + i]) * 0.5);
      const double *v0 = spv + k * n;
      const double a1 = v0[iww], a2 = v0[iw], a3 = v0[i], a4 = v0[ie];
      if (pv_scheme == GMC_PV_UPWIND && order == 3) pt = pv_upwind_edge(3, wgt, ul, vf, 1, a1, a2, a3, a4);
      else pt = pv_edge(pv_scheme, order, wgt, ul, vf, 1, dt, M(GMC_LE_LAT, r), a1, a2, a3, a4);
      if (TAPE && k >= 2) {
        if (tape.mfx_lat) row_st(tape.mfx_lat + r * p, i, tu);
        row_st(tape.u_lat + r * p, i, ul);
        row_st(tape.pv_lat + r * p, i, pt);
        if (tape.dlat[0]) tape_upwind(tape.dlat, r * p, i, upwind_deriv(pv_scheme, order, wgt, ul, vf, 1, a1, a2, a3, a4));
      }
      spt[k * n + i] = pt;
    }
  }
  __syncthreads();

  // ---- E: tendencies, the unfiltered gz into rows wrapped around the circle
  // (column c of row j at x[j][c + n / 2], c in [-n/2, n + n/2)) over m
  const int hw = n / 2;
  auto put = [&](double *row, int i, double v) {
    row[i + hw] = v;
    row[i + hw + (i < n - hw ? n : -n)] = v;
  };
  double du[kBandOut], dv[kBandOut];
  T = Tasks(w, segs, NB_W);
#pragma unroll
  for (int j = 0; j < kBandOut; j++, T.next()) {
    const int k = 2 + T.row, r = r0 - 2 + k, i = T.seg * kWave + q;
    du[j] = dv[j] = 0.0;
    if (k > nv + 2 || r >= nlat || i >= n) continue;
    const MeshRow M(mrows, nlat, r);
    const int ie = wrap(i + 1, n), iw = wrap(i - 1, n);
    const double *fx = smfx + k * n, *fy = smfy + k * n, *pl = spl + k * n, *pt = spt + k * n, *ke = ske + k * n;
    const bool u_row = r >= 1 && r <= nlat - 2;
    double dgz;
    if (u_row) {
      dgz = -(dmfdlon_of(fx[i], fx[iw], M, r) + dmfdlat_of(fy[i], fy[i - n], M, r)) * grav;
    } else {
      const double dmfdlon = 0.0, dmfdlat = pole[1];
      dgz = -(dmfdlon + dmfdlat) * grav;
    }
    const double gz_new = gz_old[j] + dt * dgz;
    put(sm + (k - 2) * 2 * n, i, gz_new);
    if (k < nv + 2) {
      if (u_row) {
        const double qhv = coriolis == 1
            ? qhv_of(M, r, pl[i], fy[i - n], pt[i - n], fy[ie - n], pt[ie - n], fy[i], pt[i], fy[ie], pt[ie])
            : tangent_sum(M(GMC_FULL_TANGENT_WGT1, r), M(GMC_FULL_TANGENT_WGT2, r), fy[i - n], fy[ie - n], fy[i], fy[ie]) * pl[i];
        du[j] = qhv - M.div(ke[ie] - ke[i], GMC_DE_LON, r);
      }
      const double qhu = coriolis == 1
          ? qhu_of(M, r, pt[i], fx[iw], pl[iw], fx[i], pl[i], fx[n + iw], pl[n + iw], fx[n + i], pl[n + i])
          : tangent_sum(M(GMC_HALF_TANGENT_WGT1, r), M(GMC_HALF_TANGENT_WGT2, r), fx[iw], fx[i], fx[n + iw], fx[n + i]) * pt[i];
      dv[j] = -qhu - M.div(ke[n + i] - ke[i], GMC_DE_LAT, r);
    }
  }
  __syncthreads();

  // ---- F: the filters of gz, two columns a lane; gz_f also into LDS over ke
  // (a band in parts stores only its part's columns)
  const int segs2 = (n + 2 * kWave - 1) / (2 * kWave);
  const int p0 = n / 2 * bd.part / bd.parts * 2, p1 = n / 2 * (bd.part + 1) / bd.parts * 2;
  for (T = Tasks(w, segs2, NB_W); T.row < 2 * (nv + 1); T.next()) {
    const int j = T.row >> 1, r = r0 + j, i = 2 * (T.seg * kWave + q);
    if (r >= nlat || i >= n) continue;
    const double *x = sm + j * 2 * n + i + hw;
    const bool sml = T.row & 1, mine = i >= p0 && i < p1;
    if (sml && (T.seg * 2 * kWave >= p1 || (T.seg + 1) * 2 * kWave <= p0)) continue;
    const int nf = sml ? pick(ns, TY + 1, j) : pick(nb, TY + 1, j), of = sml ? pick(os, TY + 1, j) : pick(ob, TY + 1, j);
    double f0 = x[0], f1 = x[1];
    if (nf > 1) filter_pair(wt + of, nf, x - (nf - 1) / 2, f0, f1);
    if (!sml) {
      ske[(j + 2) * n + i] = f0;
      ske[(j + 2) * n + i + 1] = f1;
    }
    if (j < nu && mine) {
      double *out = (sml ? G.gz : G.gz_f) + r * p;
      row_st(out, i, f0);
      row_st(out, i + 1, f1);
    }
  }
  __syncthreads();

  // ---- G: u and v of the band into wrapped rows over m and u_f (u rows,
  // then v rows), then the smoothing of the v row next to a pole -----------
  T = Tasks(w, segs, NB_W);
#pragma unroll
  for (int j = 0; j < kBandOut; j++, T.next()) {
    const int jr = T.row, r = r0 + jr, i = T.seg * kWave + q;
    if (jr >= nv || i >= n) continue;
    const MeshRow M(mrows, nlat, r);
    const double *f = ske + (jr + 2) * n;
    if (r >= 1) put(sm + jr * 2 * n, i, u_old[j] + dt * (du[j] - pgf_lon_of(f[wrap(i + 1, n)], f[i], M, r)));
    put(sm + (TY + jr) * 2 * n, i, v_old[j] + dt * (dv[j] - pgf_lat_of(f[n + i], f[i], M, r)));
  }
  __syncthreads();
  if (south || north) {
    double *v0 = sm + (TY + (south ? 0 : nv - 1)) * 2 * n, *v1 = v0 + (south ? 2 * n : -2 * n);
    for (int i = tid; i < n; i += NB_T) put(v0, i, pole_smooth(v0[i + hw], v1[i + hw]));
    __syncthreads();
  }

  // ---- H: the big filters of u and v, two columns a lane -----------------
  const int segs_p = (p1 - p0 + 2 * kWave - 1) / (2 * kWave);
  for (T = Tasks(w, segs_p, NB_W); T.row < 2 * nv; T.next()) {
    const int j = T.row >> 1, r = r0 + j, i = p0 + 2 * (T.seg * kWave + q);
    const bool lat = !(T.row & 1);
    if (i >= p1 || (!lat && r == 0)) continue;
    const double *x = sm + ((lat ? TY : 0) + j) * 2 * n + i + hw;
    const int nf = lat ? pick(nt, TY, j) : pick(nb, TY + 1, j), of = lat ? pick(ot, TY, j) : pick(ob, TY + 1, j);
    double f0 = x[0], f1 = x[1];
    double *out = (lat ? U.v : U.u) + r * p, *out_f = (lat ? U.v_f : U.u_f) + r * p;
    row_st(out, i, f0);
    row_st(out, i + 1, f1);
    if (nf > 1) filter_pair(wt + of, nf, x - (nf - 1) / 2, f0, f1);
    row_st(out_f, i, f0);
    row_st(out_f, i + 1, f1);
  }
  if ((south || north) && tid < n && bd.part == 0)   // pole U rows: not updated, copied to u_f
    row_st(U.u_f + (south ? 0 : nlat - 1) * p, tid, u_pole);
}

// ---------------------------------------------------------------------------
// The stage as gmc_step runs it.
//
// Away from the poles the zonal filters have 3 to 9 taps, and one tile takes a
// point through the whole stage (tend_tile with FULL).  Only the polar rows,
// about an eighth of them, need the tendencies, the gz filters and the u / v
// part one after the other:
//   one launch    (kStageOne) where their circles fit into LDS: bands of the
//                 polar rows beside the tiles;
//   three launches (kStageTend, kStageGz, kStageUv) on wider grids of many
//                 tiles (kSpreadTiles): tiles of the polar tendencies, then
//                 four filter items a workgroup, with the tiles of the other
//                 rows spread over the three so that none of them leaves
//                 compute units idle;
//   k_tend, k_gzf and k_uvf over all rows on the others.
// A polar v row next to the tiles reads their gz_f row, so the tiles beside
// the polar rows go into the first launch.
//
// Measured per step with three models in flight on three streams (and alone),
// three kernels a stage against this: 180 x 91 wrfrk3 17.9 (50) -> 13.5 (39)
// us, 360 x 181 24.1 (62) -> 19.4 (55), 502 x 253 with damping 35 (90) -> 31
// (85); the wider grids at kSpreadTiles.  A full tile takes 5 us from its
// start to its last store; the band at a pole, 17 us at 360 columns, bounds
// the small grids, the chains of the tiles (two workgroups a compute unit, the
// VALU 34 % busy) and of the widest filter rows the large ones.
//
// A workgroup finds its work from its number and the kernel arguments alone: a
// table would put one more trip to memory (about 1 us) before its first load.
enum { kStageTend = 0, kStageGz = 1, kStageUv = 2, kStageOne = 3 };
struct StageArgs {
  Grid g;
  Mesh M;
  const double *mrows;
  double grav, rgrav, dt, wgt;
  int stokes, pv_scheme, order, coriolis;
  StagePtrs P;
  UVPtrs U;
  BandOut G;
  FilterDev big, small;
  StageMap S;
  int polar;               // workgroups of this launch with polar work
  int tile0, tiles;        // its tiles of the short rows, from tile0 on (counted around)
  const Item *items;       // filter items, kItemsPerWg a workgroup
  int item_lds;            // doubles of LDS per item
  TapeOut tape;
};
using StageTile = Tile<11>;
constexpr int kItemsPerWg = StageTile::NT / NF;

// The work of polar workgroup e: kPoleParts workgroups for the band at each
// pole, whose filters are twice as wide as the next one's, each filtering and
// storing its share of the columns; then the other bands, numbered from the
// poles, south first: kBandTY v rows each, the last of a zone what is left.
constexpr int kPoleParts = 4;
__device__ __forceinline__ Band polar_band(const StageMap &S, int nhalf, int e) {
  const bool pole = e < 2 * kPoleParts;
  const bool north = pole ? e >= kPoleParts : e - 2 * kPoleParts >= S.bands_s - 1;
  const int part = pole ? e % kPoleParts : 0, parts = pole ? kPoleParts : 1;
  const int j = pole ? 0 : e - 2 * kPoleParts + 1 - (north ? S.bands_s - 1 : 0);   // from the zone's pole
  if (!north) return Band{kBandTY * j, min(kBandTY, S.ra - kBandTY * j), part, parts};
  const int r1 = nhalf - kBandTY * j, r0 = max(r1 - kBandTY, S.rb);
  return Band{r0, r1 - r0, part, parts};
}

template <int PHASE, bool TAPE>
__global__ void __launch_bounds__(StageTile::NT, PHASE == kStageOne ? 4 : 8) k_stage(StageArgs A) {
  extern __shared__ __attribute__((aligned(16))) double xs[];
  using S = StageTile;
  const int b = blockIdx.x;
  if (b >= A.polar) {
    int t = A.tile0 + xcd_item(b - A.polar, A.tiles);
    t = t >= A.S.ntiles ? t - A.S.ntiles : t;
    const TileGeo geo = short_tile<S::TY>(A.S, A.g.nlon, t);
    const TileRest<FilterDev, const double *, double *> rest{A.big,  A.small, A.U.u_old, A.U.v_old, A.U.u,
                                                             A.U.v,  A.U.u_f, A.U.v_f,   A.G.gz_f,  A.G.gz};
    const TileIn io = tile_fetch<S>(A.g, A.P, geo);
    tend_tile<S, TAPE, true>(A.g, A.M, (RecPtr)A.mrows, A.grav, A.rgrav, A.dt, A.stokes, A.pv_scheme, A.order, A.wgt,
                             A.coriolis, A.P, geo, xs, io, &A.tape, rest);
  } else if constexpr (PHASE == kStageTend) {
    const TileGeo geo = polar_tile<S::TY>(A.S, A.g, b);
    const TileIn io = tile_fetch<S>(A.g, A.P, geo);
    tile_poles<S>(A.g, A.M, A.grav, A.rgrav, A.P, geo.r0, xs);
    tend_tile<S, TAPE, false>(A.g, A.M, (RecPtr)A.mrows, A.grav, A.rgrav, A.dt, A.stokes, A.pv_scheme, A.order, A.wgt,
                              A.coriolis, A.P, geo, xs, io, &A.tape, NoRest{});
  } else if constexpr (PHASE == kStageOne) {
    band_stage<TAPE>(A.g, (RecPtr)A.mrows, A.grav, A.rgrav, A.dt, A.stokes, A.pv_scheme, A.order, A.wgt, A.coriolis,
                     A.big, A.small, polar_band(A.S, A.g.nhalf, b), A.P, A.U, A.G, A.tape, xs);
  } else {
    // an item per group of NF threads (the list is padded with empty items)
    const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x / NF), tid = threadIdx.x % NF;
    const Item &it = A.items[b * kItemsPerWg + grp];
    double *x = xs + grp * A.item_lds;
    if constexpr (PHASE == kStageGz)
      gzf_item(A.g, A.big, A.small, it, A.P.gz_new, A.G.gz_f, A.G.gz, x, tid);
    else
      uvf_item(A.g, A.M, A.dt, A.big, it, A.U, x, tid);
  }
}

// ---------------------------------------------------------------------------
// Batched ensembles: the launches of a stage over many contexts at once.  A
// member's descriptor for one stage holds its geometry, tables, options, stage
// dt and field pointers; a list gives each tile its member (one trip to memory
// where a search over the members' first tiles took four), and an item holds
// its member's index.
//
// The tendency launch takes the polar rows' tiles; the filter launches, bound
// by the latency of their widest rows, also take as many of the tiles that do
// a whole stage as make two workgroups a compute unit, and the tendency launch
// the rest.  At 16 members (8 of 180 x 91, 6 of 360 x 181, 2 of 720 x 361) a
// stage's three launches took 38.5 + 23.5 + 12.7 us with every row in all
// three, 49.4 + 7.7 + 11.3 us with all tiles in the first and 38.0 + 13.5 +
// 12.6 us so.
struct EnsMember {
  Grid g;
  Mesh M;
  const double *mrows;
  FilterDev big, small1;
  double grav, rgrav, dt, wgt;   // rgrav = 1 / grav correctly rounded
  int stokes, pv_scheme, order, coriolis;
  StagePtrs sp;
  UVPtrs up;
  double *gz_f_out;    // gz_f of the new state (big filter output)
  double *gz_out;      // gz of the new state (small filter output)
};
// Tile `tile` of member `member`: map.tiles_p of the polar rows, then
// map.ntiles that do a whole stage.
struct EnsTile {
  int member, tile;
};

// Field pointers read from a descriptor in memory are generic (FLAT) to the
// compiler, and FLAT accesses also count against the LDS wait counter.  The
// ensemble kernels therefore hand the shared tile and item code pointers
// typed in the global address space, so that it emits global loads and
// stores as it does for pointers passed as kernel arguments.
struct MeshG {
  gptr<const double> m;
  int nlat;
  __device__ __forceinline__ double operator()(int f, int r) const { return m[f * nlat + r]; }
  __device__ __forceinline__ double div(double x, int f, int r) const { return x / (*this)(f, r); }
};
__device__ __forceinline__ MeshG glb(const Mesh &M) { return MeshG{glb(M.m), M.nlat}; }
struct FilterDevG {
  int max_taps;
  gptr<const int32_t> ngrid_lon, ngrid_lat;
  gptr<const double> wgt_lon, wgt_lat;
};
struct StagePtrsG {
  gptr<const double> gz_star, gzs, u_f, v_f, gz_old;
  gptr<double> gz_new, du, dv;
};
struct UVPtrsG {
  gptr<const double> u_old, v_old, du, dv, gz_f;
  gptr<double> u, v, u_f, v_f;
};
__device__ __forceinline__ FilterDevG glb(const FilterDev &f) {
  return FilterDevG{f.max_taps, glb(f.ngrid_lon), glb(f.ngrid_lat), glb(f.wgt_lon), glb(f.wgt_lat)};
}
__device__ __forceinline__ StagePtrsG glb(const StagePtrs &p) {
  return StagePtrsG{glb(p.gz_star), glb(p.gzs), glb(p.u_f), glb(p.v_f), glb(p.gz_old), glb(p.gz_new), glb(p.du), glb(p.dv)};
}
__device__ __forceinline__ UVPtrsG glb(const UVPtrs &p) {
  return UVPtrsG{glb(p.u_old), glb(p.v_old), glb(p.du), glb(p.dv), glb(p.gz_f), glb(p.u), glb(p.v), glb(p.u_f), glb(p.v_f)};
}

// A tile of an ensemble's member.
template <class S, bool POLAR>
__device__ __forceinline__ void ens_tile(const EnsMember *__restrict__ mem, const StageMap *__restrict__ maps,
                                         EnsTile e, double *sh) {
  const EnsMember d = mem[e.member];   // private copies: no aliasing with the stores of the tile
  const StageMap m = maps[e.member];
  const StagePtrsG sp = glb(d.sp);
  if (POLAR && e.tile < m.tiles_p) {
    const TileGeo G = polar_tile<S::TY>(m, d.g, e.tile);
    const TileIn io = tile_fetch<S>(d.g, sp, G);
    tile_poles<S>(d.g, glb(d.M), d.grav, d.rgrav, sp, G.r0, sh);
    tend_tile<S, false, false>(d.g, glb(d.M), (RecPtr)d.mrows, d.grav, d.rgrav, d.dt, d.stokes, d.pv_scheme, d.order,
                               d.wgt, d.coriolis, sp, G, sh, io, nullptr, NoRest{});
  } else {
    const TileGeo G = short_tile<S::TY>(m, d.g.nlon, e.tile - m.tiles_p);
    const UVPtrsG up = glb(d.up);
    const TileRest<FilterDevG, gptr<const double>, gptr<double>> rest{
        glb(d.big), glb(d.small1), up.u_old, up.v_old, up.u, up.v, up.u_f, up.v_f, glb(d.gz_f_out), glb(d.gz_out)};
    const TileIn io = tile_fetch<S>(d.g, sp, G);
    tend_tile<S, false, true>(d.g, glb(d.M), (RecPtr)d.mrows, d.grav, d.rgrav, d.dt, d.stokes, d.pv_scheme, d.order,
                              d.wgt, d.coriolis, sp, G, sh, io, nullptr, rest);
  }
}

// The listed tiles are cut into NXCD contiguous runs, one per XCD (workgroup b
// runs on XCD b % NXCD), so vertically adjacent tiles share that XCD's L2.
// The workgroups of one XCD stride over its run: gridDim.x may be smaller than
// the tile count (a persistent launch sized by the tuner).
template <class S>
__global__ void __launch_bounds__(S::NT, 8) k_tend_ens(const EnsMember *__restrict__ mem,
                                                       const StageMap *__restrict__ maps,
                                                       const EnsTile *__restrict__ tiles, int total) {
  __shared__ double sh[S::SH_ALL];
  const int G = gridDim.x, x = blockIdx.x % NXCD;
  const int q = total / NXCD, rem = total % NXCD;
  const int start = x * q + min(x, rem), cnt = q + (x < rem);   // this XCD's run
  const int per = (G - x + NXCD - 1) / NXCD;                    // workgroups on this XCD
  for (int s = blockIdx.x / NXCD; s < cnt; s += per) {
    ens_tile<S, true>(mem, maps, tiles[start + s], sh);
    __syncthreads();
  }
}

// Workgroups [0, groups): an item per group of NF threads (the list is padded
// with empty items); then the listed tiles, where a workgroup has their size.
template <bool GZ>
__global__ void __launch_bounds__(StageTile::NT, 8) k_filter_ens(const EnsMember *__restrict__ mem,
                                                                 const StageMap *__restrict__ maps,
                                                                 const EnsTile *__restrict__ tiles, int ntiles,
                                                                 const Item *__restrict__ items, int groups,
                                                                 int per_wg, int item_lds) {
  extern __shared__ __attribute__((aligned(16))) double xs[];
  const int b = blockIdx.x;
  if (b >= groups) {
    ens_tile<StageTile, false>(mem, maps, tiles[xcd_item(b - groups, ntiles)], xs);
    return;
  }
  const int grp = __builtin_amdgcn_readfirstlane(threadIdx.x / NF), tid = threadIdx.x % NF;
  const Item &it = items[b * per_wg + grp];
  const EnsMember *d = mem + it.member;
  double *x = xs + grp * item_lds;
  if constexpr (GZ)
    gzf_item(d->g, glb(d->big), glb(d->small1), it, glb(d->sp.gz_new), glb(d->gz_f_out), glb(d->gz_out), x, tid);
  else
    uvf_item(d->g, glb(d->M), d->dt, glb(d->big), it, glb(d->up), x, tid);
}

}  // namespace

// ---------------------------------------------------------------------------
// Work lists: a row whose filter has n taps is cut into chunks of about
// kChunkWork / n columns (a multiple of 64, at least 64) so that each
// workgroup does similar work: the taps of a chunk's outputs are LDS reads,
// and a polar row of several hundred taps over 512 columns kept one CU busy
// for the whole launch.  Rows of short filters go into chunks of at most
// kNarrowChunk columns, so that a workgroup's window is one round of loads.
static constexpr int kChunkWork = GMC_CHUNK_WORK;
static constexpr int kNarrowChunk = GMC_NARROW_CHUNK;

// One row of a filter work list: `work` taps per output sets the chunk
// width; n (and n2) are the taps of the row's filters, the window of a chunk
// is its columns and (n - 1) / 2 of the wider filter's taps on either side
// (lds: the most of weights and window).
// Returns the number of chunks the row was cut into.
static int add_row(std::vector<Item> &v, int row, int kind, int work, int nlon, size_t &lds, int n, int n2 = 0,
                   int chunk_work = kChunkWork) {
  int w = work <= 16 ? std::min(nlon, kNarrowChunk)
                     : std::min(nlon, std::max(64, (chunk_work / work + 63) / 64 * 64));
  const int parts = (nlon + w - 1) / w;
  const int taps = std::max(n, 0) + std::max(n2, 0), widest = std::max(n, n2), h = widest > 1 ? (widest - 1) / 2 : 0;
  for (int k = 0; k < parts; k++) {
    const int c0 = (int)((int64_t)nlon * k / parts), c1 = (int)((int64_t)nlon * (k + 1) / parts);
    v.push_back(Item{row, c0, c1, kind, 0, n, n2, 0});
    lds = std::max(lds, sizeof(double) * (size_t)(taps + c1 - c0 + 2 * h));
  }
  return parts;
}

struct FusedPlan {
  Item *d_items = nullptr;
  int n_gz = 0, n_uv = 0;
  size_t lds_gz = 0, lds_uv = 0;
  int rows_split = 0, max_parts = 1, widest = 0;   // reported by gmc_filter_plan
  // the stage as gmc_step runs it (launches of k_stage; none: the three kernels)
  int n_stage = 0;
  StageMap map{};
  struct Launch {
    int polar, tile0, tiles, item_lds;
    Item *d_items;
    size_t lds;
  } stage[3] = {};
  std::vector<void *> mem;   // their device allocations
};

static FusedPlan *plan_of(gmc_ctx *c) { return (FusedPlan *)c->fused_plan; }

static void plan_free(gmc_ctx *c) {
  FusedPlan *P = plan_of(c);
  if (!P) return;
  if (P->d_items) hip_note(hipFree(P->d_items), "plan free");
  for (void *m : P->mem) hip_note(hipFree(m), "plan free");
  delete P;
  c->fused_plan = nullptr;
}

// Order a work list for a launch of one workgroup per item whose workgroup b
// takes item xcd_item(b): each XCD works through one contiguous run of the
// list.  The wide items (more than twice the median work: the polar rows'
// long filters) are dealt round-robin to the XCDs and put first in each run,
// so they start first everywhere; the rest follow in their list order, so
// each XCD sweeps a band of neighbouring rows that share its L2.
template <class W>
static std::vector<Item> xcd_deal(const std::vector<Item> &v, W work) {
  const int T = (int)v.size();
  std::vector<int64_t> wk(T);
  for (int k = 0; k < T; k++) wk[k] = work(v[k]);
  std::vector<int64_t> sorted = wk;
  std::nth_element(sorted.begin(), sorted.begin() + T / 2, sorted.end());
  const int64_t med = T ? sorted[T / 2] : 0;
  std::vector<int> wide, narrow;
  for (int k = 0; k < T; k++) (wk[k] > 2 * med ? wide : narrow).push_back(k);
  std::stable_sort(wide.begin(), wide.end(), [&](int a, int b) { return wk[a] > wk[b]; });
  std::vector<std::vector<int>> run(NXCD);
  std::vector<int> size(NXCD);
  for (int x = 0; x < NXCD; x++) size[x] = T / NXCD + (x < T % NXCD ? 1 : 0);   // run lengths of xcd_item
  int x = 0;
  for (int k : wide) {   // round-robin over the XCDs that still have room
    while ((int)run[x].size() >= size[x]) x = (x + 1) % NXCD;
    run[x].push_back(k);
    x = (x + 1) % NXCD;
  }
  size_t next = 0;
  std::vector<Item> out;
  out.reserve(T);
  for (int y = 0; y < NXCD; y++) {
    while ((int)run[y].size() < size[y]) run[y].push_back(narrow[next++]);
    for (int k : run[y]) out.push_back(v[k]);
  }
  return out;
}

template <class T> static int to_device(gmc_ctx *c, FusedPlan *P, const std::vector<T> &v, T *&d, const char *what) {
  void *m = nullptr;
  int rc = check_hip(c, hipMalloc(&m, sizeof(T) * std::max<size_t>(v.size(), 1)), what);
  if (rc) return rc;
  P->mem.push_back(m);
  d = (T *)m;
  return check_hip(c, hipMemcpy(m, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice), what);
}

// The tap-outputs of a filter item of the launches that also take tiles (four
// items share a workgroup's LDS), and the workgroups those launches are filled
// up to with tiles: two on each compute unit.
static constexpr int kStageWork = 8192, kStageSlots = 2 * 256;

// Tiles of the whole grid from which a stage of wide circles goes in the three
// launches that share its tiles out, two and a half a compute unit.  A filter
// launch is as long as its widest rows' chains, 4 to 5 us longer beside tiles;
// below, k_tend's tiles run at once or nearly so and spreading them saves less
// than that.  us a step of one model (of three in flight), three launches and
// three kernels: 560 x 281 (260 tiles) 82 (35) and 70 (29), 720 x 361 (396) 94
// (41.5) and 76 (37.4), 900 x 451 (615) 104 (53) and 92 (53), 960 x 481 (704)
// 106 (57) and 101 (59), 1024 x 513 (846) 109 (62) and 104 (69), 1440 x 721
// (1584) 164 (134) and 147 to 154 (147), 2160 x 1081 (3564) 336 (289) and 348
// (322).
static constexpr int kSpreadTiles = 5 * 256 / 2;

// Tiles of 60 x 11 over all rows of all members from which an ensemble's tiles
// take the short rows whole: more than run at once.  Below, a launch is one
// workgroup's chain, which a whole tile or four filter items in a workgroup only
// make longer.  us a step, every row in three kernels with a filter item a
// workgroup, and whole tiles: 2 members of 180 x 91 (54 tiles) 54.7 and 69, 2 of
// 180 x 91 and one of 360 x 181 (156) 63.6 and 74.6, 4 of 360 x 181 (408) 87 and
// 95, 16 of 180 x 91 (432) 90.3 and 92.2; 2 of 180 x 91, one of 360 x 181 and
// one of 720 x 361 (552) 115 and 108, 3 and 6 of the first two (693) 114.6 and
// 117, 2 of 720 x 361 (792) 131 and 122, 8, 6 and 2 of the three (1620) 202 and
// 200.
static constexpr int kWholeTiles = kStageSlots;

// Heavy and light items share a workgroup of `per`: item i of the order by work
// goes to workgroup i mod the number of workgroups.
static void deal_items(std::vector<Item> &v, int per = kItemsPerWg) {
  auto taps = [](const Item &it) { return (int64_t)(it.c1 - it.c0) * std::max(it.n + it.n2, 1); };
  std::stable_sort(v.begin(), v.end(), [&](const Item &a, const Item &b) { return taps(a) > taps(b); });
  while (v.size() % per) v.push_back(Item{1, 0, 0, 1, 0, 0, 0, 0});   // no columns
  const int n = (int)v.size() / per;
  std::vector<Item> dealt(v.size());
  for (int i = 0; i < (int)v.size(); i++) dealt[i % n * per + i / n] = v[i];
  v = dealt;
}

// The launches of the stage.
static int build_stage(gmc_ctx *c, FusedPlan *P, const std::vector<int32_t> &nb, const std::vector<int32_t> &ns,
                       const std::vector<int32_t> &nbv) {
  using S = StageTile;
  const Grid &g = c->grid;
  const int nlon = g.nlon, nlat = g.nlat, nhalf = g.nhalf;
  StageMap &m = P->map;
  if (!stage_map(nlon, nlat, nb, ns, nbv, S::TY, m)) return GMC_OK;
  constexpr size_t kLds = 160 * 1024, kTileLds = sizeof(double) * S::SH_ALL;
  auto big_lds = [&](std::initializer_list<const void *> fs) {
    int rc = GMC_OK;
    for (const void *f : fs)
      if (!rc) rc = check_hip(c, hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds), "lds");
    return rc;
  };
  int rc;
  // one launch: bands of the polar rows, if their circles and weights fit
  const int segs = (nlon + kWave - 1) / kWave;
  int weights = 0;
  for (int r = 0; r < nhalf; r++) {
    if (r >= m.ra && r < m.rb) continue;
    int w = 0;
    for (int j = 0; j <= kBandTY && r + j < nlat; j++) {
      w += std::max(nb[r + j], 0) + std::max(ns[r + j], 0);
      if (j < kBandTY && r + j < nhalf) w += std::max(nbv[r + j], 0);
    }
    weights = std::max(weights, w);
  }
  const size_t lds = sizeof(double) * ((size_t)kBandLdsRows * nlon + 8 + weights);
  if (kBandRows * segs <= kBandLoads * NB_W && (kBandTY + 1) * segs <= kBandOut * NB_W && lds <= kLds) {
    m.bands_s = (m.ra + kBandTY - 1) / kBandTY;
    m.bands_p = m.bands_s + (nhalf - m.rb + kBandTY - 1) / kBandTY;
    P->stage[0] = {m.bands_p + 2 * (kPoleParts - 1), 0, m.ntiles, 0, nullptr, std::max(lds, kTileLds)};
    rc = big_lds({(const void *)k_stage<kStageOne, false>, (const void *)k_stage<kStageOne, true>});
    if (!rc) P->n_stage = 1;
    return rc;
  }
  // three launches
  if (((nlon + TX - 1) / TX) * ((nlat + S::TY - 1) / S::TY) < kSpreadTiles) return GMC_OK;
  std::vector<Item> items[3];
  size_t lgz = 0, luv = 0;
  for (int r = 0; r < nlat; r++) {
    if (r >= m.ra && r < m.rb) continue;
    add_row(items[1], r, 0, nb[r] + std::max(1, nb[r] / 2), nlon, lgz, nb[r], ns[r], kStageWork);
    add_row(items[2], r, 1, nb[r], nlon, luv, nb[r], 0, kStageWork);
    if (r < nhalf) add_row(items[2], r, 2, nbv[r], nlon, luv, nbv[r], 0, kStageWork);
  }
  for (int k = 1; k < 3; k++) deal_items(items[k]);
  const size_t item[3] = {0, lgz, luv};
  if (kItemsPerWg * std::max(item[1], item[2]) > kLds) return GMC_OK;
  // the short rows' tiles: what fills the second and third launch up to two
  // workgroups a compute unit, from the middle of the numbering
  int left = m.ntiles - beside_polar(m);
  for (int k = 1; k < 3; k++) {
    const int polar = (int)items[k].size() / kItemsPerWg, take = std::min(left, std::max(0, kStageSlots - polar));
    P->stage[k] = {polar, 0, take, (int)(item[k] / sizeof(double)), nullptr, std::max(kTileLds, kItemsPerWg * item[k])};
    left -= take;
  }
  const int n0 = beside_polar(m) + left, south = south_tiles(m, n0);
  P->stage[0] = {m.tiles_p, m.ntiles - (n0 - south), n0, 0, nullptr, kTileLds};
  P->stage[1].tile0 = south;
  P->stage[2].tile0 = south + P->stage[1].tiles;
  rc = big_lds({(const void *)k_stage<kStageTend, false>, (const void *)k_stage<kStageTend, true>,
                (const void *)k_stage<kStageGz, false>, (const void *)k_stage<kStageGz, true>,
                (const void *)k_stage<kStageUv, false>, (const void *)k_stage<kStageUv, true>});
  for (int k = 1; k < 3 && !rc; k++) rc = to_device(c, P, items[k], P->stage[k].d_items, "stage items alloc");
  if (!rc) P->n_stage = 3;
  return rc;
}

static int build_plan(gmc_ctx *c) {
  const Grid &g = c->grid;
  std::vector<int32_t> nb_lon(g.nlat), nb_lat(g.nhalf), ns_lon(g.nlat);
  int rc = check_hip(c, hipMemcpy(nb_lon.data(), c->big.ngrid_lon, sizeof(int32_t) * g.nlat, hipMemcpyDeviceToHost),
                     "plan");
  if (!rc) rc = check_hip(c, hipMemcpy(nb_lat.data(), c->big.ngrid_lat, sizeof(int32_t) * g.nhalf,
                                       hipMemcpyDeviceToHost), "plan");
  if (!rc) rc = check_hip(c, hipMemcpy(ns_lon.data(), c->small1.ngrid_lon, sizeof(int32_t) * g.nlat,
                                       hipMemcpyDeviceToHost), "plan");
  if (rc) return rc;
  for (int r = 0; r < g.nlat; r++)
    if (ns_lon[r] > g.nlon) return set_error(c, GMC_EINVAL, "filter wider than a latitude circle");
  for (int r = 0; r < g.nlat; r++)
    if (nb_lon[r] > g.nlon) return set_error(c, GMC_EINVAL, "filter wider than a latitude circle");
  for (int r = 0; r < g.nhalf; r++)
    if (nb_lat[r] > g.nlon) return set_error(c, GMC_EINVAL, "filter wider than a latitude circle");
  if (g.nlon > Tile<TY_MAIN>::kMaxPoleLon) return set_error(c, GMC_EINVAL, "nlon too large for the fused stage kernels");
  std::vector<Item> items;
  FusedPlan *P = new FusedPlan();

  {
    std::vector<Item> gz, uv;
    auto count = [&](int parts, int n) {
      P->rows_split += parts > 1;
      P->max_parts = std::max(P->max_parts, parts);
      P->widest = std::max(P->widest, n);
    };
    // gz items: the window is that of the wider of the two filters
    for (int r = 0; r < g.nlat; r++)
      count(add_row(gz, r, 0, nb_lon[r] + std::max(1, nb_lon[r] / 2), g.nlon, P->lds_gz, nb_lon[r], ns_lon[r]),
            nb_lon[r]);
    // u row r next to v rows r - 1 and r: the three read gz_f row r
    for (int r = 0; r < g.nlat; r++) {
      count(add_row(uv, r, 1, nb_lon[r], g.nlon, P->lds_uv, nb_lon[r]), nb_lon[r]);
      if (r < g.nhalf) count(add_row(uv, r, 2, nb_lat[r], g.nlon, P->lds_uv, nb_lat[r]), nb_lat[r]);
    }
    auto work = [&](const Item &it) {
      const int n = it.kind == 2 ? nb_lat[it.row] : nb_lon[it.row];
      return (int64_t)(it.c1 - it.c0) * std::max(n, 1);
    };
    const std::vector<Item> gz_d = xcd_deal(gz, work), uv_d = xcd_deal(uv, work);
    items.insert(items.end(), gz_d.begin(), gz_d.end());
    P->n_gz = (int)items.size();
    items.insert(items.end(), uv_d.begin(), uv_d.end());
    P->n_uv = (int)items.size() - P->n_gz;
  }
  rc = check_hip(c, hipMalloc((void **)&P->d_items, sizeof(Item) * items.size()), "plan alloc");
  if (!rc) rc = check_hip(c, hipMemcpy(P->d_items, items.data(), sizeof(Item) * items.size(), hipMemcpyHostToDevice),
                          "plan copy");
  if (!rc) rc = build_stage(c, P, nb_lon, ns_lon, nb_lat);
  c->fused_plan = P;
  if (rc) plan_free(c);
  return rc;
}

void fused_release(gmc_ctx *c) {
  for (auto &sg : c->graphs) hip_note(hipGraphExecDestroy(sg.exec), "step graph destroy");
  c->graphs.clear();
  plan_free(c);
}

const char *const kKernelNames[kKernelClasses] = {"k_tend", "k_gzf", "k_uvf"};

// A stage launch.  Under gmc_kernel_times the next two profiling events take
// the kernel's own start and end stamps (hipExtLaunchKernelGGL fills them from
// the dispatch itself, so no event packet sits between them and the kernel);
// every argument is converted to the kernel's parameter type first, since the
// extended launch passes the arguments' bytes as given.
template <class... P, class... A>
static void stage_launch(gmc_ctx *c, void (*k)(P...), dim3 grid, dim3 block, uint32_t lds, A &&...a) {
  static_assert(sizeof...(P) == sizeof...(A), "one argument per kernel parameter");
  if (c->prof_ev && c->prof_n + 2 <= c->prof_cap) {
    hipExtLaunchKernelGGL(k, grid, block, lds, c->stream, c->prof_ev[c->prof_n], c->prof_ev[c->prof_n + 1], 0,
                          static_cast<P>(a)...);
    c->prof_n += 2;
  } else {
    hipLaunchKernelGGL(k, grid, block, lds, c->stream, static_cast<P>(a)...);
  }
}

// one step_forward_backward stage: old -> new with the star state `star`;
// with tape, the star state's intermediates go to its state fields
static void fused_stage(gmc_ctx *c, int o, int s, int n, double dt, bool tape = false,
                        const TapeOut *dst = nullptr) {
  const Grid &g = c->grid;
  const Mesh M{c->d_mesh, g.nlat};
  FusedPlan *PL = plan_of(c);
  double **O = c->state[o], **S = c->state[s], **N = c->state[n];
  double *du = c->tend[o][T_DU], *dv = c->tend[o][T_DV];
  double *gz_new = c->tend[o][T_DGZ];   // the unfiltered gz of the new state
  StagePtrs sp{S[S_GZ], c->gzs, S[S_U_F], S[S_V_F], O[S_GZ], gz_new, du, dv};
  const int tiles = ((g.nlon + TX - 1) / TX) * ((g.nlat + TY_MAIN - 1) / TY_MAIN);
  TapeOut T{S[S_M_LON], S[S_M_LAT], S[S_M_VTX], S[S_MFX_LON], S[S_MFY_LAT], S[S_MFX_LAT], S[S_MFY_LON],
            S[S_U_LAT], S[S_V_LON], S[S_PV], S[S_PV_LON], S[S_PV_LAT], nullptr, nullptr};
  if (dst) T = *dst;
  UVPtrs up{O[S_U_LON], O[S_V_LAT], du, dv, N[S_GZ_F], N[S_U_LON], N[S_V_LAT], N[S_U_F], N[S_V_F]};
  if (PL->n_stage && !c->prof_ev) {   // gmc_kernel_times times the three kernels on every grid
    StageArgs A{g, M, c->d_mrows, c->cfg.g, 1.0 / c->cfg.g, dt, c->cfg.upwind_wgt_pv, c->cfg.pv_pole_stokes,
                c->cfg.pv_scheme, pv_order(c->cfg), c->cfg.coriolis_scheme, sp, up, BandOut{N[S_GZ_F], N[S_GZ]},
                c->big, c->small1, PL->map, 0, 0, 0, nullptr, 0, T};
    for (int k = 0; k < PL->n_stage; k++) {
      const FusedPlan::Launch &L = PL->stage[k];
      A.polar = L.polar;
      A.tile0 = L.tile0;
      A.tiles = L.tiles;
      A.items = L.d_items;
      A.item_lds = L.item_lds;
      auto fn = PL->n_stage == 1 ? (tape ? k_stage<kStageOne, true> : k_stage<kStageOne, false>)
                : k == 0         ? (tape ? k_stage<kStageTend, true> : k_stage<kStageTend, false>)
                : k == 1         ? (tape ? k_stage<kStageGz, true> : k_stage<kStageGz, false>)
                                 : (tape ? k_stage<kStageUv, true> : k_stage<kStageUv, false>);
      hipLaunchKernelGGL(fn, dim3(L.polar + L.tiles), dim3(StageTile::NT), L.lds, c->stream, A);
    }
    return;
  }
  stage_launch(c, tape ? k_tend<true> : k_tend<false>, dim3(tiles), dim3(Tile<TY_MAIN>::NT), 0, g, M,
               c->d_mrows, c->cfg.g, 1.0 / c->cfg.g, dt, c->cfg.pv_pole_stokes, c->cfg.pv_scheme,
               pv_order(c->cfg), c->cfg.upwind_wgt_pv, c->cfg.coriolis_scheme, sp, T);
  stage_launch(c, k_gzf, dim3(PL->n_gz), dim3(NF), PL->lds_gz, g, c->big, c->small1, PL->d_items, gz_new,
               N[S_GZ_F], N[S_GZ]);
  stage_launch(c, k_uvf, dim3(PL->n_uv), dim3(NF), PL->lds_uv, g, M, dt, c->big, PL->d_items + PL->n_gz, up);
}

int fused_prepare(gmc_ctx *c) { return c->fused_plan ? GMC_OK : build_plan(c); }

int fused_plan_info(gmc_ctx *c, int32_t out[4]) {
  const int rc = fused_prepare(c);
  if (rc) return rc;
  const FusedPlan *P = plan_of(c);
  out[0] = P->n_gz + P->n_uv;
  out[1] = P->rows_split;
  out[2] = P->max_parts;
  out[3] = P->widest;
  return GMC_OK;
}

int fused_stage_tape(gmc_ctx *c, int o, int s, int n, double dt, const TapeOut *dst) {
  int rc = fused_prepare(c);
  if (rc) return rc;
  fused_stage(c, o, s, n, dt, true, dst);
  return check_hip(c, hipGetLastError(), "fused stage");
}

int fused_integrate(gmc_ctx *c, int o, int n, double dt) {
  int rc = fused_prepare(c);
  if (rc) return rc;
  const bool keep = c->keep_derived != 0;
  switch (c->cfg.time_scheme) {
  case GMC_TIME_EULER:
    fused_stage(c, o, o, n, dt, keep);
    break;
  case GMC_TIME_WRFRK3:
    fused_stage(c, o, o, n, dt / 3.0, keep);
    fused_stage(c, o, n, 3, dt / 2.0, keep);
    fused_stage(c, o, 3, n, dt, keep);
    break;
  default:
    fused_stage(c, o, o, n, dt / 2.0, keep);
    fused_stage(c, o, n, 3, dt / 2.0, keep);
    fused_stage(c, o, 3, n, dt, keep);
  }
  rc = check_hip(c, hipGetLastError(), "fused stage");
  if (!rc && c->cfg.use_div_damp) rc = ops_div_damp(c, n);
  return rc;
}

void derived_after_step(gmc_ctx *c, int o, int n) {
  const int v = c->keep_derived ? 1 : 0;
  c->derived_kept[o] = v;
  if (c->cfg.time_scheme != GMC_TIME_EULER) {
    c->derived_kept[n] = v;
    c->derived_kept[3] = v;
  }
}

void derived_forget(gmc_ctx *c) {
  for (int &k : c->derived_kept) k = 0;
}

// gmc_step: replay a captured graph of `steps` fused steps from old level o
// (the levels swap after every step).  Kernels inside one graph follow each
// other with no gap, while consecutive graph launches leave one (about 9 us at
// 1440 x 721), so long runs replay graphs of several steps.
int fused_step_graph(gmc_ctx *c, int o, int n, double dt, int steps) {
  int rc = fused_prepare(c);
  if (rc) return rc;
  hipGraphExec_t exec = nullptr;
  for (auto &sg : c->graphs)
    if (sg.o == o && sg.n == n && sg.dt == dt && sg.keep == c->keep_derived && sg.steps == steps) exec = sg.exec;
  if (!exec) {
    hipGraph_t graph = nullptr;
    rc = check_hip(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal), "begin capture");
    if (rc) return rc;
    int rc2 = GMC_OK, a = o, b = n;
    for (int s = 0; s < steps && !rc2; s++) {
      rc2 = fused_integrate(c, a, b, dt);
      std::swap(a, b);
    }
    rc = check_hip(c, hipStreamEndCapture(c->stream, &graph), "end capture");
    if (rc2) return rc2;
    if (rc) return rc;
    rc = check_hip(c, hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0), "graph instantiate");
    (void)hipGraphDestroy(graph);
    if (rc) return rc;
    c->graphs.push_back({o, n, dt, c->keep_derived, steps, exec});
  }
  return check_hip(c, hipGraphLaunch(exec, c->stream), "graph launch");
}

}  // namespace gmc

// ===========================================================================
// Batched ensembles (include/gmcore_ens.h)
namespace gmc {
namespace {

// launch shapes the tuner chooses from: rows of the k_tend tile and the
// workgroups of the persistent tendency launch (0: one per tile, else
// mult x 256)
struct EnsShape {
  int ty, mult;
  const char *name;
};
constexpr EnsShape kEnsShapes[] = {
    {11, 0, "tile 60x11, one workgroup per tile"}, {7, 0, "tile 60x7, one workgroup per tile"},
    {5, 0, "tile 60x5, one workgroup per tile"},   {11, 4, "tile 60x11, 1024 persistent workgroups"},
    {7, 4, "tile 60x7, 1024 persistent workgroups"}, {5, 4, "tile 60x5, 1024 persistent workgroups"},
    {11, 8, "tile 60x11, 2048 persistent workgroups"}, {7, 8, "tile 60x7, 2048 persistent workgroups"},
    {5, 8, "tile 60x5, 2048 persistent workgroups"}};
constexpr int kNumEnsShapes = sizeof(kEnsShapes) / sizeof(kEnsShapes[0]);

int stage_count(int scheme) { return scheme == GMC_TIME_EULER ? 1 : 3; }

// (old, star, new) level of each stage and its dt, as fused_integrate
void stage_levels(int scheme, int o, int n, double dt, int st, int &so, int &ss, int &sn, double &sdt) {
  so = o;
  if (scheme == GMC_TIME_EULER) { ss = o; sn = n; sdt = dt; return; }
  if (st == 0) { ss = o; sn = n; sdt = scheme == GMC_TIME_WRFRK3 ? dt / 3.0 : dt / 2.0; }
  else if (st == 1) { ss = n; sn = 3; sdt = dt / 2.0; }
  else { ss = 3; sn = n; sdt = dt; }
}

}  // namespace
}  // namespace gmc

struct gmc_ens {
  std::vector<gmc_ctx *> m;
  int scheme = 0, nstage = 3;
  int shape = 0;
  gmc::EnsMember *d_mem = nullptr;  // [2 parities][nstage][members]; then, in the same allocation,
  gmc::StageMap *d_maps = nullptr;  // [members],
  gmc::EnsTile *d_tiles = nullptr;  // the tiles of the three launches
  gmc::Item *d_items = nullptr;
  bool whole = false;               // tiles take the rows of short filters through the whole stage
  int per_wg = 1;                   // filter items of a workgroup
  int n_gz = 0, n_uv = 0;           // workgroups of filter items
  size_t lds_gz = 0, lds_uv = 0;    // LDS of an item
  int tiles[3] = {0, 0, 0};
  std::vector<std::vector<int32_t>> nb_lon, nb_lat, ns_lon;   // taps of the members' rows
  std::vector<double> dt;           // dt the tables were built for
  int built_shape = -1;
  // graphs of one step and of kEnsBlock steps, by the parity they start from
  hipGraphExec_t graph[2] = {nullptr, nullptr}, graph_block[2] = {nullptr, nullptr};
  hipStream_t stream = nullptr;
  std::string err;
};

namespace gmc {
namespace {

int eerr(gmc_ens *e, int code, const std::string &msg) {
  if (e) e->err = msg;
  return code;
}
int ehip(gmc_ens *e, hipError_t x, const char *what) {
  if (x == hipSuccess) return GMC_OK;
  return eerr(e, x == hipErrorOutOfMemory ? GMC_ENOMEM : GMC_EDEVICE, std::string(what) + ": " + hipGetErrorString(x));
}

void drop_graphs(gmc_ens *e) {
  for (hipGraphExec_t *g : {&e->graph[0], &e->graph[1], &e->graph_block[0], &e->graph_block[1]})
    if (*g) { hip_note(hipGraphExecDestroy(*g), "ensemble graph destroy"); *g = nullptr; }
}

// the members' rows for tiles of height ty; returns the number of their tiles
int ens_maps(gmc_ens *e, int ty, std::vector<StageMap> &maps) {
  int tiles = 0;
  maps.resize(e->m.size());
  for (size_t k = 0; k < e->m.size(); k++) {
    const Grid &g = e->m[k]->grid;
    stage_map(g.nlon, g.nlat, e->nb_lon[k], e->ns_lon[k], e->nb_lat[k], ty, maps[k], e->whole);
    tiles += maps[k].tiles_p + maps[k].ntiles;
  }
  return tiles;
}

// descriptor tables for the current shape and dts
int build_tables(gmc_ens *e) {
  const int nm = (int)e->m.size(), ty = kEnsShapes[e->shape].ty;
  std::vector<EnsMember> tab((size_t)2 * e->nstage * nm);
  std::vector<StageMap> maps;
  ens_maps(e, ty, maps);
  // The tiles of each launch, member by member.  The filter launches take tiles
  // of their own workgroups' height only, and none of the two bands beside the
  // polar rows, whose gz_f the last launch's polar rows read.
  std::vector<EnsTile> tiles[3];
  const int room[2] = {std::max(0, kStageSlots - e->n_gz), std::max(0, kStageSlots - e->n_uv)};
  for (int k = 0; k < nm; k++) {
    const StageMap &m = maps[k];
    const int first = m.nseg ? m.seg[0].nx : 0, last = m.nseg ? m.ntiles - m.seg[m.nseg - 1].nx : 0;
    for (int t = 0; t < m.tiles_p + m.ntiles; t++) {
      const int s = t - m.tiles_p;
      int l = 0;
      if (ty == StageTile::TY && s >= first && s < last)
        l = (int)tiles[1].size() < room[0] ? 1 : (int)tiles[2].size() < room[1] ? 2 : 0;
      tiles[l].push_back(EnsTile{k, t});
    }
  }
  std::vector<EnsTile> list;
  for (int l = 0; l < 3; l++) {
    e->tiles[l] = (int)tiles[l].size();
    list.insert(list.end(), tiles[l].begin(), tiles[l].end());
  }
  for (int par = 0; par < 2; par++)
    for (int st = 0; st < e->nstage; st++)
      for (int k = 0; k < nm; k++) {
        gmc_ctx *c = e->m[k];
        const int o = par == 0 ? 1 : 2, n = par == 0 ? 2 : 1;
        int so, ss, sn;
        double sdt;
        stage_levels(e->scheme, o, n, e->dt[k], st, so, ss, sn, sdt);
        double **O = c->state[so], **S = c->state[ss], **N = c->state[sn];
        double *du = c->tend[so][T_DU], *dv = c->tend[so][T_DV], *gz_new = c->tend[so][T_DGZ];
        EnsMember &d = tab[((size_t)par * e->nstage + st) * nm + k];
        d.g = c->grid;
        d.M = Mesh{c->d_mesh, c->grid.nlat};
        d.mrows = c->d_mrows;
        d.big = c->big;
        d.small1 = c->small1;
        d.grav = c->cfg.g;
        d.rgrav = 1.0 / c->cfg.g;
        d.dt = sdt;
        d.wgt = c->cfg.upwind_wgt_pv;
        d.stokes = c->cfg.pv_pole_stokes;
        d.pv_scheme = c->cfg.pv_scheme;
        d.order = pv_order(c->cfg);
        d.coriolis = c->cfg.coriolis_scheme;
        d.sp = StagePtrs{S[S_GZ], c->gzs, S[S_U_F], S[S_V_F], O[S_GZ], gz_new, du, dv};
        d.up = UVPtrs{O[S_U_LON], O[S_V_LAT], du, dv, N[S_GZ_F], N[S_U_LON], N[S_V_LAT], N[S_U_F], N[S_V_F]};
        d.gz_f_out = N[S_GZ_F];
        d.gz_out = N[S_GZ];
      }
  std::vector<char> all;
  auto put = [&](const void *x, size_t n) { all.insert(all.end(), (const char *)x, (const char *)x + n); };
  put(tab.data(), sizeof(EnsMember) * tab.size());
  put(maps.data(), sizeof(StageMap) * maps.size());
  put(list.data(), sizeof(EnsTile) * list.size());
  int rc = ehip(e, hipMemcpy(e->d_mem, all.data(), all.size(), hipMemcpyHostToDevice), "tables");
  if (rc) return rc;
  drop_graphs(e);
  e->built_shape = e->shape;
  return GMC_OK;
}

template <int TY>
void launch_tend(gmc_ens *e, const EnsMember *mem, int grid) {
  using S = Tile<TY>;
  hipLaunchKernelGGL(k_tend_ens<S>, dim3(grid), dim3(S::NT), 0, e->stream, mem, e->d_maps, e->d_tiles, e->tiles[0]);
}

// the launches of one ensemble step for parity par (0: old 1 -> new 2)
void ens_launch_step(gmc_ens *e, int par) {
  const int nm = (int)e->m.size();
  const EnsShape &sh = kEnsShapes[e->shape];
  // k_tend_ens covers every tile when grid == total or grid >= NXCD
  const int grid = sh.mult ? std::min(e->tiles[0], sh.mult * 256) : e->tiles[0];
  const EnsTile *t1 = e->d_tiles + e->tiles[0], *t2 = t1 + e->tiles[1];
  auto lds = [&](size_t item, int tiles) {
    return (uint32_t)std::max(e->per_wg * item, tiles ? sizeof(double) * StageTile::SH_ALL : 0);
  };
  const dim3 block(e->per_wg * NF);
  for (int st = 0; st < e->nstage; st++) {
    const EnsMember *mem = e->d_mem + ((size_t)par * e->nstage + st) * nm;
    switch (sh.ty) {
    case 5: launch_tend<5>(e, mem, grid); break;
    case 7: launch_tend<7>(e, mem, grid); break;
    default: launch_tend<11>(e, mem, grid);
    }
    hipLaunchKernelGGL(k_filter_ens<true>, dim3(e->n_gz + e->tiles[1]), block, lds(e->lds_gz, e->tiles[1]), e->stream,
                       mem, e->d_maps, t1, e->tiles[1], e->d_items, e->n_gz, e->per_wg,
                       (int)(e->lds_gz / sizeof(double)));
    hipLaunchKernelGGL(k_filter_ens<false>, dim3(e->n_uv + e->tiles[2]), block, lds(e->lds_uv, e->tiles[2]), e->stream,
                       mem, e->d_maps, t2, e->tiles[2], e->d_items + e->per_wg * e->n_gz, e->n_uv, e->per_wg,
                       (int)(e->lds_uv / sizeof(double)));
  }
}

// steps per graph of a long run (even: the parity ends where it began); as
// gmc_step's, since consecutive graph launches leave a gap that kernels
// inside one graph do not
constexpr int kEnsBlock = 8;

// the graph of `steps` (1 or kEnsBlock) ensemble steps from parity par
int ens_graph(gmc_ens *e, int par, int steps, hipGraphExec_t *out) {
  hipGraphExec_t &slot = steps == 1 ? e->graph[par] : e->graph_block[par];
  if (slot) { *out = slot; return GMC_OK; }
  hipGraph_t graph = nullptr;
  int rc = ehip(e, hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal), "begin capture");
  if (rc) return rc;
  for (int s = 0; s < steps; s++) ens_launch_step(e, (par + s) % 2);
  const hipError_t le = hipGetLastError();
  rc = ehip(e, hipStreamEndCapture(e->stream, &graph), "end capture");
  if (!rc) rc = ehip(e, le, "ensemble launch");
  if (!rc) rc = ehip(e, hipGraphInstantiate(&slot, graph, nullptr, nullptr, 0), "graph instantiate");
  if (graph) (void)hipGraphDestroy(graph);
  if (!rc) *out = slot;
  return rc;
}

int ens_run(gmc_ens *e, const double *dt, int nsteps) {
  const int nm = (int)e->m.size();
  for (gmc_ctx *c : e->m) {
    // the batch steps every member from member 0's time level
    if (c->old_level != e->m[0]->old_level)
      return eerr(e, GMC_ESTATE, "members are at different time levels (one was stepped on its own)");
  }
  for (gmc_ctx *c : e->m) derived_forget(c);
  bool same = e->built_shape == e->shape;
  for (int k = 0; k < nm && same; k++) same = e->dt[k] == dt[k];
  if (!same) {
    for (int k = 0; k < nm; k++) e->dt[k] = dt[k];
    int rc = build_tables(e);
    if (rc) return rc;
  }
  for (int s = 0; s < nsteps;) {
    const int par = e->m[0]->old_level == 1 ? 0 : 1;
    const int steps = nsteps - s >= kEnsBlock ? kEnsBlock : 1;
    hipGraphExec_t g = nullptr;
    int rc = ens_graph(e, par, steps, &g);
    if (!rc) rc = ehip(e, hipGraphLaunch(g, e->stream), "graph launch");
    if (rc) return rc;
    for (int k = 0; k < steps; k++)
      for (gmc_ctx *c : e->m) std::swap(c->old_level, c->new_level);
    s += steps;
  }
  return GMC_OK;
}

}  // namespace
}  // namespace gmc

using namespace gmc;

extern "C" {

int gmc_ens_create(gmc_ctx *const *members, int32_t n, gmc_ens **out) {
  if (!out) return GMC_EINVAL;
  *out = nullptr;
  if (!members || n < 1) return GMC_EINVAL;
  gmc_ens *e = new gmc_ens();
  auto fail = [&](int code, const char *msg) {
    gmc_ens_destroy(e);
    (void)msg;
    return code;
  };
  for (int k = 0; k < n; k++) {
    gmc_ctx *c = members[k];
    if (!c || !c->prepared || c->cfg.use_div_damp || c->cfg.time_scheme != members[0]->cfg.time_scheme ||
        c->old_level != members[0]->old_level || c->grid.nlon > Tile<5>::kMaxPoleLon)
      return fail(GMC_EINVAL, "member not batchable");
    for (int j = 0; j < k; j++)
      if (members[j] == c) return fail(GMC_EINVAL, "member listed twice");
    if (fused_prepare(c)) return fail(GMC_EINVAL, "member plan");
    if (hipStreamSynchronize(c->stream) != hipSuccess) return fail(GMC_EDEVICE, "member sync");
    e->m.push_back(c);
  }
  e->scheme = members[0]->cfg.time_scheme;
  e->nstage = stage_count(e->scheme);
  e->dt.assign(n, 0.0);
  // few tiles: every row in the three kernels, a filter item a workgroup
  int ntiles = 0;
  for (const gmc_ctx *c : e->m)
    ntiles += ((c->grid.nlon + TX - 1) / TX) * ((c->grid.nlat + StageTile::TY - 1) / StageTile::TY);
  e->whole = ntiles >= kWholeTiles;
  e->per_wg = e->whole ? kItemsPerWg : 1;
  // filter work items of every member, tagged with the member index
  std::vector<Item> gz, uv;
  size_t lgz = 0, luv = 0;
  for (int k = 0; k < n; k++) {
    gmc_ctx *c = e->m[k];
    const Grid &g = c->grid;
    std::vector<int32_t> nb_lon(g.nlat), nb_lat(g.nhalf), ns_lon(g.nlat);
    if (hipMemcpy(nb_lon.data(), c->big.ngrid_lon, sizeof(int32_t) * g.nlat, hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(nb_lat.data(), c->big.ngrid_lat, sizeof(int32_t) * g.nhalf, hipMemcpyDeviceToHost) != hipSuccess ||
        hipMemcpy(ns_lon.data(), c->small1.ngrid_lon, sizeof(int32_t) * g.nlat, hipMemcpyDeviceToHost) != hipSuccess)
      return fail(GMC_EDEVICE, "filter tables");
    // the rows that the tiles do not take through the whole stage
    StageMap sm;
    stage_map(g.nlon, g.nlat, nb_lon, ns_lon, nb_lat, StageTile::TY, sm, e->whole);
    auto polar = [&](int r) { return r < sm.ra || r >= sm.rb; };
    std::vector<Item> a, b;
    for (int r = 0; r < g.nlat; r++)
      if (polar(r))
        add_row(a, r, 0, nb_lon[r] + std::max(1, nb_lon[r] / 2), g.nlon, lgz, nb_lon[r], ns_lon[r], kStageWork);
    for (int r = 0; r < g.nlat; r++)
      if (polar(r)) add_row(b, r, 1, nb_lon[r], g.nlon, luv, nb_lon[r], 0, kStageWork);
    for (int r = 0; r < g.nhalf; r++)
      if (polar(r)) add_row(b, r, 2, nb_lat[r], g.nlon, luv, nb_lat[r], 0, kStageWork);
    e->nb_lon.push_back(nb_lon);
    e->nb_lat.push_back(nb_lat);
    e->ns_lon.push_back(ns_lon);
    for (auto &it : a) {
      it.member = k;
      gz.push_back(it);
    }
    for (auto &it : b) {
      it.member = k;
      uv.push_back(it);
    }
  }
  deal_items(gz, e->per_wg);
  deal_items(uv, e->per_wg);
  e->n_gz = (int)gz.size() / e->per_wg;
  e->n_uv = (int)uv.size() / e->per_wg;
  e->lds_gz = lgz;
  e->lds_uv = luv;
  int most = 0;
  for (const EnsShape &sh : kEnsShapes) {
    std::vector<StageMap> maps;
    most = std::max(most, ens_maps(e, sh.ty, maps));
  }
  gz.insert(gz.end(), uv.begin(), uv.end());
  int rc = ehip(e, hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking), "stream");
  if (!rc) rc = ehip(e, hipMalloc((void **)&e->d_items, sizeof(Item) * gz.size()), "items");
  if (!rc) rc = ehip(e, hipMemcpy(e->d_items, gz.data(), sizeof(Item) * gz.size(), hipMemcpyHostToDevice), "items");
  if (!rc)
    rc = ehip(e, hipMalloc((void **)&e->d_mem, (sizeof(EnsMember) * 2 * e->nstage + sizeof(StageMap)) * n +
                                                   sizeof(EnsTile) * most), "tables");
  e->d_maps = (StageMap *)(e->d_mem + (size_t)2 * e->nstage * n);
  e->d_tiles = (EnsTile *)(e->d_maps + n);
  // an item's window and taps are at most about three circles of the widest
  // member's (k_tend's limit): four of them fit
  constexpr size_t kLds = 160 * 1024;
  if (!rc && e->per_wg * std::max(e->lds_gz, e->lds_uv) > kLds) rc = eerr(e, GMC_EINVAL, "filter window exceeds LDS");
  for (const void *f : {(const void *)k_filter_ens<true>, (const void *)k_filter_ens<false>})
    if (!rc) rc = ehip(e, hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds), "lds");
  if (rc) {
    gmc_ens_destroy(e);
    return rc;
  }
  *out = e;
  return GMC_OK;
}

int gmc_ens_destroy(gmc_ens *e) {
  if (!e) return GMC_EINVAL;
  if (e->stream) hip_note(hipStreamSynchronize(e->stream), "ensemble sync");
  drop_graphs(e);
  if (e->d_mem) hip_note(hipFree(e->d_mem), "ensemble tables free");
  if (e->d_items) hip_note(hipFree(e->d_items), "ensemble items free");
  if (e->stream) hip_note(hipStreamDestroy(e->stream), "ensemble stream destroy");
  delete e;
  return GMC_OK;
}

const char *gmc_ens_last_error(const gmc_ens *e) { return e ? e->err.c_str() : "null ensemble"; }

int gmc_ens_step(gmc_ens *e, const double *dt, int32_t nsteps) {
  if (!e) return GMC_EINVAL;
  if (!dt || nsteps < 0) return eerr(e, GMC_EINVAL, "bad step arguments");
  for (size_t k = 0; k < e->m.size(); k++)
    if (!(dt[k] > 0)) return eerr(e, GMC_EINVAL, "dt must be positive");
  int rc = ens_run(e, dt, nsteps);
  if (!rc) rc = ehip(e, hipStreamSynchronize(e->stream), "ensemble sync");
  return rc;
}

int gmc_ens_shape(gmc_ens *e, int32_t shape) {
  if (!e) return GMC_EINVAL;
  if (shape < 0 || shape >= kNumEnsShapes) return eerr(e, GMC_EINVAL, "no such shape");
  e->shape = shape;
  return GMC_OK;
}

const char *gmc_ens_shape_name(int32_t shape) {
  return shape >= 0 && shape < kNumEnsShapes ? kEnsShapes[shape].name : "";
}

int gmc_ens_autotune(gmc_ens *e, const double *dt, int32_t trial_steps, int32_t *choice, double *times_ms,
                     int32_t cap, int32_t *ncand) {
  if (!e) return GMC_EINVAL;
  if (!dt || trial_steps < 1 || !choice) return eerr(e, GMC_EINVAL, "bad autotune arguments");
  const int nm = (int)e->m.size();
  // snapshot every member's fields and levels into one buffer; the trials
  // run on the members and the snapshot is restored afterwards
  std::vector<size_t> off(nm + 1, 0);
  for (int k = 0; k < nm; k++) off[k + 1] = off[k] + (e->m[k]->slab_bytes + 255) / 256 * 256;
  char *save = nullptr;
  std::vector<int> levels(nm);
  for (int k = 0; k < nm; k++) levels[k] = e->m[k]->old_level;
  int rc = GMC_OK;
  for (int k = 0; k < nm && !rc; k++) rc = ehip(e, hipStreamSynchronize(e->m[k]->stream), "member sync");
  if (!rc) rc = ehip(e, hipMalloc((void **)&save, off[nm]), "snapshot alloc");
  for (int k = 0; k < nm && !rc; k++)
    rc = ehip(e, hipMemcpyAsync(save + off[k], e->m[k]->slab, e->m[k]->slab_bytes, hipMemcpyDeviceToDevice, e->stream),
              "snapshot");
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  if (!rc) rc = ehip(e, hipEventCreate(&ev0), "event");
  if (!rc) rc = ehip(e, hipEventCreate(&ev1), "event");
  const int keep = e->shape;
  int best = keep;
  float best_ms = 0.f;
  for (int s = 0; s < kNumEnsShapes && !rc; s++) {
    e->shape = s;
    rc = ens_run(e, dt, 1);  // warm-up, builds tables and graphs
    if (!rc) rc = ehip(e, hipEventRecord(ev0, e->stream), "event");
    if (!rc) rc = ens_run(e, dt, trial_steps);
    if (!rc) rc = ehip(e, hipEventRecord(ev1, e->stream), "event");
    if (!rc) rc = ehip(e, hipEventSynchronize(ev1), "event sync");
    float ms = 0.f;
    if (!rc) rc = ehip(e, hipEventElapsedTime(&ms, ev0, ev1), "elapsed");
    ms /= trial_steps;
    if (!rc && times_ms && s < cap) times_ms[s] = ms;
    if (!rc && (s == 0 || ms < best_ms)) { best_ms = ms; best = s; }
  }
  if (save) {
    for (int k = 0; k < nm; k++) {
      if (!rc)
        rc = ehip(e, hipMemcpyAsync(e->m[k]->slab, save + off[k], e->m[k]->slab_bytes, hipMemcpyDeviceToDevice,
                                    e->stream), "restore");
      e->m[k]->old_level = levels[k];
      e->m[k]->new_level = levels[k] == 1 ? 2 : 1;
    }
    if (!rc) rc = ehip(e, hipStreamSynchronize(e->stream), "restore sync");
    else hip_note(hipStreamSynchronize(e->stream), "autotune sync");
    hip_note(hipFree(save), "snapshot free");
  }
  if (ev0) hip_note(hipEventDestroy(ev0), "event destroy");
  if (ev1) hip_note(hipEventDestroy(ev1), "event destroy");
  e->shape = rc ? keep : best;
  if (!rc) {
    *choice = best;
    if (ncand) *ncand = kNumEnsShapes;
  }
  return rc;
}

int gmc_ens_stream(gmc_ens *e, void **stream) {
  if (!e || !stream) return GMC_EINVAL;
  *stream = (void *)e->stream;
  return GMC_OK;
}

}  // extern "C"

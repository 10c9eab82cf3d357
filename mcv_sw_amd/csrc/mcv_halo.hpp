// The boundary pass of the cubed sphere (correct_bdy_ghost,
// spatial_operators_mod.F90:282-492, ghost_mod.f90:154-227): values of one
// ghost point, one cube-edge point or one cube vertex, formed from the band
// (the raw lines nearest each panel side that a stage wrote: geopotential and
// sphere winds, FP64 in both forms).  One set of routines serves both forms
// and both users: the stage kernel, whose tiles at the panel sides finish the
// points they stage, and the boundary kernel, which finishes a whole level.
//
// The stage that writes the band converts its winds, once per point, with the
// matrix of the point it has just updated.  Converting while reading took a
// 32-byte matrix beside each of the DOF points of a ghost value, 28 loads
// instead of 8 (MCV4) and 20 to 30 more registers in the stage kernels.
//
// M has npv, dx and the tables of the boundary pass (MeshDev, MeshF32).
#pragma once

#include "mcv_device.hpp"

namespace mcv {

// Writes the raw values of point (i, j) of panel p to the band lines it is on;
// P is the point's A*IG.
__device__ __forceinline__ void put_band(D3 *band, const int npv, const int H, const int p,
                                         const int i, const int j, const double *P,
                                         const double ph, const double u, const double v) {
  D3 r;
  r.a = ph;
  // sphere winds (spatial_operators_mod.F90:391-405)
  r.b = P[0] * u + P[2] * v;
  r.c = P[1] * u + P[3] * v;
  if (i <= H + 1) stg(band, band_point(npv, H, p, 0, i, j), r);
  if (i >= npv - H) stg(band, band_point(npv, H, p, 1, npv + 1 - i, j), r);
  if (j <= H + 1) stg(band, band_point(npv, H, p, 2, j, i), r);
  if (j >= npv - H) stg(band, band_point(npv, H, p, 3, npv + 1 - j, i), r);
}

// The panel side whose lines hold the halo source of (p, side), which is also
// the other panel's side of that cube edge.
__device__ __forceinline__ int source_side(const HaloSrc &hs) {
  return hs.col ? (hs.far ? 1 : 0) : (hs.far ? 3 : 2);
}

// Ghost point at depth k (1..H) beyond `side` of panel p, along index s
// (ghost_mod.f90:154-227): the neighbour's line at normal index k+1 (or nPV-k)
// is band depth k+1 of the side it is parallel to; its sphere winds go back
// through SP2P at the ghost point (spatial_operators_mod.F90:408-492).
template <int DOF, class M>
__device__ __forceinline__ D3 ghost_value(const M &m, const D3 *band, const int p, const int side,
                                          const int k, const int s) {
  constexpr int H = DOF - 1;
  const int npv = m.npv;
  const HaloSrc hs = kHalo[p - 1][side];
  const int src = source_side(hs);
  const uint32_t gi = (uint32_t)((k - 1) * npv + (s - 1));
  const int c = ldg(m.giref, gi);
  const double cf = ldg(m.gcoef, gi);
  double qp[DOF], qz[DOF], qm[DOF];
#pragma unroll
  for (int l = 0; l < DOF; ++l) {
    const int tpos = (c - 1) * H + 1 + l;
    const int al = hs.rev ? npv + 1 - tpos : tpos;
    const D3 x = ldg(band, band_point(npv, H, hs.q, src, k + 1, al));
    qp[l] = x.a;
    qz[l] = x.b;
    qm[l] = x.c;
  }
  const double zh = ghost_interp<DOF>(qz, cf, m.dx), mh = ghost_interp<DOF>(qm, cf, m.dx);
  D3 r;
  r.a = ghost_interp<DOF>(qp, cf, m.dx);
  apply2(m.sp2p_ghost + 4 * ghost_point(npv, H, p, side, k, s), zh, mh, r.b, r.c);
  return r;
}

// Mean of the two copies of a cube-edge point (position sa of side a of panel
// pa, sb of side b of pb): geopotential and sphere winds
// (spatial_operators_mod.F90:298-345).  The sums commute, so both copies find
// the same bits.
template <int DOF>
__device__ __forceinline__ D3 edge_mean(const int npv, const D3 *band, const int pa, const int a,
                                        const int sa, const int pb, const int b, const int sb) {
  const D3 x = ldg(band, band_point(npv, DOF - 1, pa, a, 1, sa));
  const D3 y = ldg(band, band_point(npv, DOF - 1, pb, b, 1, sb));
  return D3{0.5 * (x.a + y.a), 0.5 * (x.b + y.b), 0.5 * (x.c + y.c)};
}

// Mean of the three copies of cube vertex vx, in the reference's summation
// order (spatial_operators_mod.F90:347-386).
template <int DOF>
__device__ __forceinline__ D3 vertex_mean(const int npv, const D3 *band, const int vx) {
  D3 x[3];
#pragma unroll
  for (int l = 0; l < 3; ++l) {
    const VtxPt vp = kVerts[vx][l];
    // either edge through the corner holds its raw value
    x[l] = ldg(band, band_point(npv, DOF - 1, vp.p, vp.ci ? 1 : 0, 1, vp.cj ? npv : 1));
  }
  return D3{(x[0].a + x[1].a + x[2].a) / 3.0, (x[0].b + x[1].b + x[2].b) / 3.0,
            (x[0].c + x[1].c + x[2].c) / 3.0};
}

// Panel winds of a mean of sphere winds at point s of edge line `side` of panel p.
template <class M>
__device__ __forceinline__ D3 edge_winds(const M &m, const D3 &mean, const int p, const int side,
                                         const int s) {
  D3 r;
  r.a = mean.a;
  apply2(m.sp2p_edge + 4 * edge_point(m.npv, p, side, s), mean.b, mean.c, r.b, r.c);
  return r;
}

// Point s of the edge line `side` of panel p, vertices included.
template <int DOF, class M>
__device__ __forceinline__ D3 edge_value(const M &m, const D3 *band, const int p, const int side,
                                         const int s) {
  const int npv = m.npv;
  if (s > 1 && s < npv) {
    const HaloSrc hs = kHalo[p - 1][side];
    const int other = source_side(hs), so = hs.rev ? npv + 1 - s : s;
    return edge_winds(m, edge_mean<DOF>(npv, band, p, side, s, hs.q, other, so), p, side, s);
  }
  const int far = s > 1 ? 1 : 0;
  const int ci = side < 2 ? side : far, cj = side < 2 ? far : side - 2;
  return edge_winds(m, vertex_mean<DOF>(npv, band, kVertexAt[p - 1][2 * cj + ci]), p, ci,
                    cj ? npv : 1);
}

// Points of a tile's staged region that the boundary pass owns (ghost points
// and the edge lines of panel p), each finished by one thread and handed to
// put(lx, ly, values).  The tile is given by its extents: staged point
// (lx, ly) is panel point (i0 - H + lx, j0 - H + ly).  The ghost points come
// first and the edge lines start on a wavefront of their own, so that a
// wavefront goes through one of the two chains of dependent loads.
struct TileSides {
  int sides, n;  // the sides in reach of the staged region (2 bits each), their number
};

__device__ __forceinline__ TileSides tile_sides(const int i0, const int j0, const int lw,
                                                const int lh, const int H, const int npv) {
  TileSides t{0, 0};
  if (i0 - H <= 1) { t.sides |= 0 << (2 * t.n); ++t.n; }
  if (i0 - H + lw - 1 >= npv) { t.sides |= 1 << (2 * t.n); ++t.n; }
  if (j0 - H <= 1) { t.sides |= 2 << (2 * t.n); ++t.n; }
  if (j0 - H + lh - 1 >= npv) { t.sides |= 3 << (2 * t.n); ++t.n; }
  return t;
}

template <int DOF, int L, class M, class Put>
__device__ __forceinline__ void finish_tile(const M &m, const D3 *band, const TileSides &ts,
                                            const int p, const int i0, const int j0,
                                            const int nx, const int ny, const Put &put) {
  constexpr int H = DOF - 1;
  const int npv = m.npv, lw = nx + 2 * H, lh = ny + 2 * H;
  const int ng = ts.n * H * L, e0 = (ng + 63) / 64 * 64, total = e0 + ts.n * L;
  for (int t = threadIdx.x; t < total; t += blockDim.x) {
    const bool ghost = t < e0;
    if (ghost && t >= ng) continue;
    const int r = div_small<L>(ghost ? t : t - e0), pos = (ghost ? t : t - e0) - r * L;
    const int sl = ghost ? div_small<H>(r) : r, d = ghost ? r - sl * H + 1 : 0;
    const int side = (ts.sides >> (2 * sl)) & 3;
    const int s = (side < 2 ? j0 : i0) - H + pos;  // along the side
    if (s < 1 || s > npv) continue;
    // a vertex belongs to the W or E side
    if (!ghost && side >= 2 && (s == 1 || s == npv)) continue;
    const int at = (side & 1) ? npv + d : 1 - d;  // across it
    const int lx = (side < 2 ? at : s) - (i0 - H), ly = (side < 2 ? s : at) - (j0 - H);
    if (lx < 0 || lx >= lw || ly < 0 || ly >= lh) continue;
    const bool inx = lx >= H && lx < H + nx, iny = ly >= H && ly < H + ny;
    if (!inx && !iny) continue;  // a halo corner of the tile, never read
    put(lx, ly, ghost ? ghost_value<DOF>(m, band, p, side, d, s)
                      : edge_value<DOF>(m, band, p, side, s));
  }
}

// Work item t of the boundary pass on one whole level, t in
// [0, boundary_items()): one ghost point, one edge point (its two copies) or
// one cube vertex (its three) per item, each handed to store(g, values).  The
// items are independent, each a short chain of loads.
template <int DOF, class Store>
__device__ __forceinline__ void boundary_item(const MeshDev &m, const D3 *band, const int t,
                                              const Store &store) {
  constexpr int H = DOF - 1;
  const int npv = m.npv, nh = m.nh;
  const int nghost = 6 * 4 * H * npv, nedge = 12 * npv;
  if (t < nghost) {
    // (panel, side, depth k, along-edge s), s fastest
    const int s = t % npv + 1, r = t / npv, k = r % H + 1, ps = r / H;
    const int side = ps % 4, p = ps / 4 + 1;
    const int at = (side & 1) ? npv + k : 1 - k;
    store(pidx(nh, H, p, side < 2 ? at : s, side < 2 ? s : at),
          ghost_value<DOF>(m, band, p, side, k, s));
  } else if (t < nghost + nedge) {
    const int s = (t - nghost) % npv + 1, e = (t - nghost) / npv;
    if (s > 1 && s < npv) {  // the ends are vertices
      const EdgePair ep = kEdges[e];
      const int sb = ep.rev ? npv + 1 - s : s;
      const D3 mean = edge_mean<DOF>(npv, band, ep.pa, ep.sa, s, ep.pb, ep.sb, sb);
      int i, j;
      edge_ij(npv, ep.sa, s, i, j);
      store(pidx(nh, H, ep.pa, i, j), edge_winds(m, mean, ep.pa, ep.sa, s));
      edge_ij(npv, ep.sb, sb, i, j);
      store(pidx(nh, H, ep.pb, i, j), edge_winds(m, mean, ep.pb, ep.sb, sb));
    }
  } else {
    const int vx = t - nghost - nedge;
    const D3 mean = vertex_mean<DOF>(npv, band, vx);
#pragma unroll
    for (int l = 0; l < 3; ++l) {
      const VtxPt vp = kVerts[vx][l];
      const int i = vp.ci ? npv : 1, j = vp.cj ? npv : 1;
      store(pidx(nh, H, vp.p, i, j), edge_winds(m, mean, vp.p, vp.ci ? 1 : 0, j));
    }
  }
}

}  // namespace mcv

// phx_flux.hip -- fused reconstruction + Riemann flux kernels (fluid.cpp:676-770) for gfx950.
//
// The reference reconstructs every cell once per direction into ql/qr arrays and a second
// kernel reads them back.  Here each cell is reconstructed once per direction in
// registers and the face states never reach memory:
//
//  * x (unit stride): one lane per cell along a row; primitives are staged through LDS
//    once per variable and the cell's upper-edge state is published in LDS, so lane l forms
//    face i from the upper edge of cell i-1 (lane l-1) and the lower edge of cell i (its
//    own).  Blocks overlap by 2H+1 cells.
//  * y, z (strided): one 64-lane wave of a few columns marches along the sweep with an LDS
//    ring of primitive rows, passing upper edges to the next row by cross-lane shuffles;
//    or LDS tiles of a few consecutive i by a stretch of the own direction, overlapping by
//    2H+1 rows.  The autotuner picks the kind and shape per block size.
//
// Results are bit-identical to reconstructing per face: the same arithmetic runs on the
// same operands.
//
// This file builds the sweeps with the exact arithmetic and holds what both arithmetics
// share: the sweep shapes and the dispatch by phx_fluid_params::flux_arith.
#include <hip/hip_runtime.h>

#include "phx.h"
#include "phx_device.hpp"
#include "phx_internal.hpp"

#define PHX_FLUX_NS flux_exact
#define PHX_FLUX_DISPATCH
#include "phx_flux_sweeps.hpp"

namespace phx {

// ---- dispatch --------------------------------------------------------------------------
TileShape resolve_tile_shape(int d, int recon, int mhd, const BlockGeom &bg, TileShape want) {
  const int H = recon == PHX_RECON_CONSTANT ? 0 : recon == PHX_RECON_LINEAR ? 1 : 2;
  const int NP = mhd ? 10 : 7;
  if (want.ts == 0) {
    // The default.  The sweeps are bound by VALU issue, so the shape with the fewest
    // wave-steps (one 64-lane reconstruction and flux) wins once there are enough waves: a
    // marching wave's first row of a segment only starts it, a tile's 2H + 1 edge rows are
    // redone by its neighbours.  A wave-step of a tile is cheaper (no ring, no barriers
    // between steps): 7.0 against 8.8 ns per SIMD at 64^3, 6.3 against 7.0 at 96^3 (exact
    // arithmetic), hence the 0.83.  Marching segments of about three steps where that still
    // makes four waves per SIMD (4096), else single-step segments for the most waves.
    // Tiles of 8 x 32: 27 faces per 32 rows, 4 waves and 20 KB each, so eight per CU.
    // Measured (us, exact arithmetic, y sweep; the choice first): 128^3 fast 8 x -6 176
    // against 193; 96^3 8 x -5 116 / 125; 64^3 8 x -10 47 / 49; 48^3 8 x 32 26.0 / 28.3;
    // 32^3 8 x -5 15.7 / 19.7; 100 x 75 x 51 8 x 32 61 / 59.  (Segments of at least 24 faces
    // from 1024 waves on, tiles of up to 64 rows below, took 189, 143, 75, 34, 20 and 79.)
    // Without the 5-point stencils a wave-step is too short to pay for the ring: tiles.
    const int ti = want.ti > 0 ? want.ti : 8;
    const TileShape t = resolve_tile_shape(d, recon, mhd, bg, TileShape{ti, 32});
    if (H < 2) return t;
    const int nf = bg.ie[d] - bg.is[d] + 3;
    TileShape m = resolve_tile_shape(d, recon, mhd, bg, TileShape{ti, -1});
    const int MR = kMarchLanes / m.ti;
    auto steps = [&](int nseg) { return (nf + nseg + MR - 1) / MR; };  // of a column
    const long chunks = flux_march_groups(bg, d, m.ti, 1);
    int nseg = (steps(1) + 2) / 3;
    nseg = (steps(nseg) + 2) / 3;
    if (chunks * nseg < 4096) nseg = MR > 1 ? (nf + MR - 2) / (MR - 1) : nf;
    m = resolve_tile_shape(d, recon, mhd, bg, TileShape{m.ti, -nseg});
    const long tile_steps = flux_tile_groups(bg, d, t.ti, t.ts, H) * ((t.ti * t.ts + 63) / 64);
    // (under half a wave per SIMD both are one launch's latency, and the tiles' is shorter: 16^3
    // 12.9 against 13.5, 24^3 13.8 / 14.0)
    const long march_steps = chunks * steps(-m.ts);
    return march_steps >= 512 && (double)march_steps < 0.83 * (double)tile_steps ? m : t;
  }
  if (want.ts < 0) {  // marching: ti a power of two up to 64, -ts segments of the faces
    const int want_ti = want.ti > 0 ? want.ti : 8;
    int ti = 1;
    while (ti * 2 <= want_ti && ti < kMarchLanes) ti *= 2;
    while (ti > 1 && march_lds_bytes(NP, H, ti) > kMarchMaxLdsBytes) ti /= 2;
    const int nf = bg.ie[d] - bg.is[d] + 3;
    return TileShape{ti, -(-want.ts < nf ? -want.ts : nf)};
  }
  // own-direction cells the face range needs: s-2-H .. e+1+H
  const int need = bg.ie[d] - bg.is[d] + 4 + 2 * H;
  const int cap = need <= kTileMaxRows ? need : kTileMaxRows;
  TileShape t = want;
  if (t.ti <= 0) t.ti = 8;
  if (t.ts == 0) t.ts = 64;
  if (t.ts > cap) t.ts = cap;
  if (t.ts < 2 * H + 2) t.ts = 2 * H + 2 <= cap ? 2 * H + 2 : cap;
  if (t.ti < 1) t.ti = 1;
  while (t.ti > 1 && (t.ti * t.ts > kTileMaxThreads ||
                      (long)NP * t.ti * t.ts * 8 > kTileMaxLdsBytes))
    t.ti /= 2;
  while (t.ti * t.ts > kTileMaxThreads || (long)NP * t.ti * t.ts * 8 > kTileMaxLdsBytes)
    t.ts /= 2;
  return t;
}

// every direction's groups for one launch of 256-lane groups: x rows and tiles of up to 8 x 32,
// each direction starting at a multiple of 8 groups
FluxGroups all_flux_groups(int recon, int mhd, const BlockGeom &bg) {
  const int H = recon == PHX_RECON_CONSTANT ? 0 : recon == PHX_RECON_LINEAR ? 1 : 2;
  FluxGroups fg{};
  fg.n[0] = (unsigned)flux_x_groups(bg, H);
  for (int d = 1; d < 3; ++d) {
    fg.off[d] = (fg.off[d - 1] + fg.n[d - 1] + 7) / 8 * 8;
    if (d >= bg.ndim) continue;
    const TileShape t = resolve_tile_shape(d, recon, mhd, bg, TileShape{8, 32});
    fg.n[d] = (unsigned)flux_tile_groups(bg, d, t.ti, t.ts, H);
    fg.ti[d] = t.ti;
    fg.ts[d] = t.ts;
  }
  fg.off[3] = fg.off[2] + fg.n[2];
  return fg;
}

// One launch in place of two or three: a small block's sweeps are each one launch's latency on
// a part of the chip (16^3: 13 us apiece on 41-54 of 256 CUs), and on larger blocks each
// launch ends in a partial round.  Whole stage, one launch against separate ones in their
// default shapes (us): 16^3 36.5 / 57.3, 32^3 57.2 / 62.7, 48^3 92 / 109, 64^3 171 / 180,
// 100 x 75 x 51 (5,824 groups) 216 / 239, 2-D 256 x 128 42 / 48; 96^3 (14,171) fast 412 / 400: from
// about 8,192 groups on, the 5-point stencils' marching waves win.  The shorter stencils
// sweep in tiles on any block (150 x 90 x 70 hydro PLM 201 / 218).
bool one_launch_fluxes(int recon, int mhd, const BlockGeom &bg) {
  if (bg.ndim == 1) return false;
  return recon < PHX_RECON_WENO5Z || all_flux_groups(recon, mhd, bg).off[3] <= 8192;
}

long pack_groups_flux(int d, int recon, const BlockGeom &bg, TileShape shape) {
  const int H = recon == PHX_RECON_CONSTANT ? 0 : recon == PHX_RECON_LINEAR ? 1 : 2;
  if (d == 0) return flux_x_groups(bg, H);
  if (shape.ts < 0) return flux_march_groups(bg, d, shape.ti, -shape.ts);
  return flux_tile_groups(bg, d, shape.ti, shape.ts, H);
}

void launch_fluxes(int d, int recon, int riemann, int mhd, int geom, const DevParams &dp,
                   const BlockGeom &bg, const PrimPtrs &prim, const FluxPtrs &flux, double *fsig,
                   hipStream_t s, TileShape sh, bool fast) {
  if (fast)
    flux_fast::launch_fluxes(d, recon, riemann, mhd, geom, dp, bg, prim, flux, fsig, s, sh);
  else
    flux_exact::launch_fluxes(d, recon, riemann, mhd, geom, dp, bg, prim, flux, fsig, s, sh);
}

void launch_pack_flux(int d, int recon, int riemann, int geom, const DevParams &dp,
                      const PackView &v, long groups, TileShape sh, hipStream_t s, bool fast) {
  if (fast)
    flux_fast::launch_pack_flux(d, recon, riemann, geom, dp, v, groups, sh, s);
  else
    flux_exact::launch_pack_flux(d, recon, riemann, geom, dp, v, groups, sh, s);
}

}  // namespace phx

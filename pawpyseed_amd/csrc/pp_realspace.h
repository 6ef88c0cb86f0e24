// Real-space plan of one structure (pp_realspace.hip) and the tile kernel's
// work lists on it (pp_rstile.hip).
#pragma once
#include <mutex>
#include <vector>

#include "pp_geom.h"
#include "pp_internal.h"

namespace pp {

struct RsSite {
  double R[3];
  double rmax;
  int c[3], g[3];
  int nproj, nchan, n;  // projectors, channels, wave-grid points
  int chan_off;         // first channel of the species in chan_l
  int proj_off;         // first projection of the site
  long spl_off;         // species block: x[n], then f, b, c, d (n each) per channel
};

struct RsLat {
  double m[9];
};

struct RsWeights {
  double w[64];
};

// candidate c of a site's box -> unwrapped (i, j, k), k fastest (the
// reference's loop order, density.c:272-276)
__device__ __forceinline__ void rs_cand(const RsSite &s, int c, int &i, int &j, int &k) {
  const int w1 = 2 * s.g[1] + 1, w2 = 2 * s.g[2] + 1;
  k = c % w2 - s.g[2] + s.c[2];
  j = (c / w2) % w1 - s.g[1] + s.c[1];
  i = c / (w1 * w2) - s.g[0] + s.c[0];
}

// unwrapped box vector r - R in cartesian coordinates (density.c:277-281)
__device__ __forceinline__ double rs_vec(const RsSite &s, const RsLat &L, int f0, int f1, int f2, int i, int j, int k,
                                         double *v) {
  double f[3] = {(double)i / f0 - s.R[0], (double)j / f1 - s.R[1], (double)k / f2 - s.R[2]};
  d_frac_to_cart(f, L.m, v);
  return sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
}

// Spline interval of a partial-wave difference at distance r on the wave
// grid x[n], and the angles of the vector v (utils.c:461-489, 522-561).
struct RsPoint {
  bool below, beyond;
  int id;
  double t, rdiv, ct, phi;
};
__device__ __forceinline__ RsPoint rs_point(const double *x, int n, const double *v, double r) {
  RsPoint p;
  double theta = 0.0;
  p.phi = 0.0;
  if (r != 0.0) {
    theta = acos(v[2] / r);
    if (r - fabs(v[2]) != 0.0)
      p.phi = acos(v[0] / sqrt(v[0] * v[0] + v[1] * v[1]));
    if (v[1] < 0)
      p.phi = 2.0 * M_PI - p.phi;
  }
  p.ct = cos(theta);
  p.id = 0;
  p.t = 0.0;
  p.below = r < x[0];
  p.beyond = r > x[n - 1];
  if (!p.below && !p.beyond) {
    p.id = (int)(log(r / x[0]) / log(x[1] / x[0]));
    if (p.id > n - 2)
      p.id = n - 2;
    p.t = r - x[p.id];
  }
  p.rdiv = p.below ? x[0] : r;
  return p;
}
// Radial value over r of channel ch of the species block at x.
__device__ __forceinline__ double rs_radial(const double *x, int n, int ch, const RsPoint &p) {
  const double *fc = x + (long)n * (1 + 4 * ch);
  const double *bc = fc + n, *cc = bc + n, *dc = cc + n;
  const double f = p.beyond  ? 0.0
                   : p.below ? fc[0]
                             : fc[p.id] + p.t * (bc[p.id] + p.t * (cc[p.id] + p.t * dc[p.id]));
  return f / p.rdiv;
}

}  // namespace pp

struct pp_rsplan {
  pp_ctx *ctx = nullptr;
  double lattice[9];
  int fftg[3];
  int nsites = 0, ptot = 0, pmax = 0;
  long npts = 0;
  bool atomic = false;
  std::vector<int> proj_off, site_pt;
  std::vector<int> color_off, color_sites, color_maxpts;
  pp::DevBuf d_geo, d_pts, d_tab, d_tab_off, d_site_pt, d_colors, d_spl, d_chan_l;
  pp::DevBuf dens2;  // densities of the second stream's chunks
  // points and value tables of the per-site augmentation kernels, built on
  // first use (d_pts, d_tab, d_tab_off); blkoff: first point of every block
  // of 256 box candidates
  std::vector<pp::RsSite> geo;
  std::vector<long> blkoff;
  int nblk = 1;
  bool sites_built = false;
  // work lists of the tile kernel, built on first use (pp_rstile.hip); not
  // tile_ok: a site box reaches past the neighbouring cells
  bool tile_ok = false, tile_built = false;
  int nvid = 0, ks = 0;  // (site, lattice image) pairs, groups of four projector slots
  long nent = 0;
  pp::DevBuf l_off, l_ent, l_tab, l_vid;
  std::mutex build_mu;  // the first uses of two host threads
};



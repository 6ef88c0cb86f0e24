// Augmentation and density of a real-space chunk in one pass over it.
//
// A wavefront takes a block of 16 consecutive x of one x-line and 32 of the
// chunk's bands at a time: per 16 bands one 16x16 FP64 MFMA tile of real and
// one of imaginary parts, so that a lane holds both parts of its band and
// loads 16 bytes (256 in a row of lanes).  The tiles start from the chunk's
// values times the scale and Bloch phase and are increased by
// sum_p t_p(x) c_p(band) over the sites whose spheres hold points of the
// block: t the partial-wave differences in real-harmonic form (the same sum
// as the complex form with half the products), c the site's projections in
// that form times the phase of its lattice image, so the points need no phase
// of their own.  The tiles then give the block's densities, weighted and
// summed over the bands, and the states in their band-major places.  Sites
// that share points add into one accumulator in site order: no atomics and no
// colours.
//
// A read-modify-write of every sphere point per colour and a read of the
// whole chunk for the density become one read: 216^3 x 64 bands in FP64,
// 4.5 + 1.8 ms before, 2.84 now (13.2 GB, 4.6 TB/s; 3.4 with the coefficients
// loaded where they are used; FP32 2.29, 3.19).  What bounds it is the latency
// of the loads at three wavefronts per SIMD: the matrix units are busy under a third
// of it.  Tiles of 8 bands with interleaved parts, 8-byte loads and
// the blocks of x fastest took 5.8 ms, without the first entry's table values
// loaded a step ahead 4.0 ms.  A form that also ran the x pass, so that
// the chunk was never written, read each table row once per band group, 33 GB
// where this reads 13, and took 8.8 ms against 3.2 (x pass) plus this.
//
// Work lists: an entry is a (site, lattice image) whose sphere holds points
// of one block; its table holds the site's partial-wave differences at the
// block's points, zero outside the sphere, laid out as the MFMA reads it.
// The plan's first use builds them once: every (site, y, z) of the sites' boxes counts
// the blocks it reaches, the host scans the counts, and the entries of a
// block are put in site order.
#include <cstring>
#include <new>
#include <type_traits>

#include "pp_realspace.h"

namespace pp {

// The blocks of line (j, k) of a site's box that hold points inside its
// sphere: fn(image shift along x, block) for each, in x order.
template <typename F>
__device__ __forceinline__ void rs_tile_blocks(const RsSite &g, const RsLat &L, int f0, int f1, int f2, int j, int k,
                                               F &&fn) {
  int last = -1 << 30;
  for (int i = g.c[0] - g.g[0]; i <= g.c[0] + g.g[0]; i++) {
    double v[3];
    if (!(rs_vec(g, L, f0, f1, f2, i, j, k, v) < g.rmax))
      continue;
    const int sh = i < 0 ? -1 : i >= f0 ? 1 : 0, blk = (i - sh * f0) / 16, id = sh * 65536 + blk;
    if (id != last)
      fn(sh, blk);
    last = id;
  }
}
// thread -> unwrapped (j, k) of a site's box and the wrapped line; false past
// the box
__device__ __forceinline__ bool rs_tile_jk(const RsSite &g, int t, int f1, int f2, int &j, int &k, int &img,
                                           long &line) {
  const int w1 = 2 * g.g[1] + 1, w2 = 2 * g.g[2] + 1;
  if (t >= w1 * w2)
    return false;
  j = t / w2 - g.g[1] + g.c[1];
  k = t % w2 - g.g[2] + g.c[2];
  const int sj = j < 0 ? -1 : j >= f1 ? 1 : 0, sk = k < 0 ? -1 : k >= f2 ? 1 : 0;
  img = (sj + 1) * 3 + sk + 1;  // + 9 (shift along x + 1)
  line = (long)(j - sj * f1) * f2 + (k - sk * f2);
  return true;
}

__global__ __launch_bounds__(256) void k_rst_count(const RsSite *__restrict__ geo, RsLat L, int f0, int f1, int f2,
                                                   int nxb, int *__restrict__ cells, int *__restrict__ used) {
  const int s = blockIdx.y;
  const RsSite g = geo[s];
  int j, k, img;
  long line;
  if (!rs_tile_jk(g, blockIdx.x * 256 + threadIdx.x, f1, f2, j, k, img, line))
    return;
  rs_tile_blocks(g, L, f0, f1, f2, j, k, [&](int sh, int blk) {
    atomicAdd(&cells[line * nxb + blk], 1);
    used[s * 27 + (sh + 1) * 9 + img] = 1;
  });
}

// ent[.] = (site image, unwrapped x of the block's first point, j, k)
__global__ __launch_bounds__(256) void k_rst_fill(const RsSite *__restrict__ geo, RsLat L, int f0, int f1, int f2,
                                                  int nxb, const int *__restrict__ off, int *__restrict__ cells,
                                                  const int *__restrict__ vid, int4 *__restrict__ ent) {
  const int s = blockIdx.y;
  const RsSite g = geo[s];
  int j, k, img;
  long line;
  if (!rs_tile_jk(g, blockIdx.x * 256 + threadIdx.x, f1, f2, j, k, img, line))
    return;
  rs_tile_blocks(g, L, f0, f1, f2, j, k, [&](int sh, int blk) {
    const long c = line * nxb + blk;
    ent[off[c] + atomicAdd(&cells[c], -1) - 1] =
        make_int4(vid[s * 27 + (sh + 1) * 9 + img], sh * f0 + 16 * blk, j, k);
  });
}

// The entries of a block in site-image order (a handful each).
__global__ __launch_bounds__(256) void k_rst_sort(long ncell, const int *__restrict__ off, int4 *__restrict__ ent) {
  const long c = (long)blockIdx.x * 256 + threadIdx.x;
  if (c >= ncell)
    return;
  const int i0 = off[c], i1 = off[c + 1];
  for (int i = i0 + 1; i < i1; i++) {
    const int4 e = ent[i];
    int q = i;
    for (; q > i0 && ent[q - 1].x > e.x; q--)
      ent[q] = ent[q - 1];
    ent[q] = e;
  }
}

// tab[(i * ks + p / 4) * 64 + (p % 4) * 16 + x]: slot p of entry i at the
// block's point x; one thread per (entry, point).
__global__ __launch_bounds__(256) void k_rst_values(const RsSite *__restrict__ geo, RsLat L, int f0, int f1, int f2,
                                                    long nent, const int4 *__restrict__ ent,
                                                    const int2 *__restrict__ vsite, int ks,
                                                    const double *__restrict__ spl, const int *__restrict__ chan_l,
                                                    double *__restrict__ tab) {
  const long i = (long)blockIdx.x * 16 + (threadIdx.x >> 4);
  const int x = threadIdx.x & 15;
  if (i >= nent)
    return;
  const int4 e = ent[i];
  const RsSite g = geo[vsite[e.x].x];
  double *out = tab + i * ks * 64 + x;
  double v[3];
  const int xi = e.y + x;
  const int xw = xi - (e.y < 0 ? -f0 : e.y >= f0 ? f0 : 0);  // wrapped; past the axis in its last block
  const double r = rs_vec(g, L, f0, f1, f2, xi, e.z, e.w, v);
  const bool in = xw < f0 && xi >= g.c[0] - g.g[0] && xi <= g.c[0] + g.g[0] && r < g.rmax;
  const double *xg = spl + g.spl_off;
  const RsPoint rp = rs_point(xg, g.n, v, r);
  int p = 0;
  for (int ch = 0; ch < g.nchan; ch++) {
    const int l = chan_l[g.chan_off + ch];
    const double radial = in ? rs_radial(xg, g.n, ch, rp) : 0.0;
    for (int m = -l; m <= l; m++, p++) {
      const int am = m < 0 ? -m : m;
      const double norm = sqrt((2 * l + 1) / (4.0 * M_PI) * d_fact(l - am) / d_fact(l + am));
      const double a = in ? norm * d_legendre(l, am, rp.ct) * radial : 0.0;
      double sn, cs;
      sincos(am * rp.phi, &sn, &cs);
      out[(p >> 2) * 64 + (p & 3) * 16] = in ? (m < 0 ? a * sn : a * cs) : 0.0;
    }
  }
  for (; p < 4 * ks; p++)
    out[(p >> 2) * 64 + (p & 3) * 16] = 0.0;
}

// What the pass over a chunk reads besides it, in one launch.  The first nb0
// work-groups: ph = e^{2 pi i k_a i / n_a} of the three axes, the first times
// the scale.  The others: coef[(v * 4 ks + p) * NB + b], the coefficient of
// real-harmonic slot p of site image v for band b, with P_m the band's
// projections:
//   m > 0: P_m + (-1)^m P_-m,  slot -m: i (P_m - (-1)^m P_-m),  m = 0: P_0,
// times e^{2 pi i k.(R - image)}; zero past the bands and the projectors.
//
// The tables are zero at a block's points outside a sphere, and zero times an
// infinite or NaN coefficient would reach all of them: such a coefficient is
// left zero and the band's values inside the site's sphere, where the sum is
// not finite anyway, are made NaN in the chunk.
template <typename T>
__global__ __launch_bounds__(256) void k_rst_coef(int nb0, int nvid, const int2 *__restrict__ vsite,
                                                  const RsSite *__restrict__ geo, const int *__restrict__ chan_l,
                                                  int ks, int NB, int nbc, const cplx<double> *__restrict__ proj,
                                                  long ldp, double k0, double k1, double k2, RsLat L, int f0, int f1,
                                                  int f2, double scl, cplx<double> *__restrict__ ph,
                                                  cplx<double> *__restrict__ coef, cplx<T> *__restrict__ grid) {
  if ((int)blockIdx.x < nb0) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= f0 + f1 + f2)
      return;
    const double a = i < f0 ? k0 * i / f0 : i < f0 + f1 ? k1 * (i - f0) / f1 : k2 * (i - f0 - f1) / f2;
    const double q = i < f0 ? scl : 1.0;
    double sn, cs;
    sincospi(2.0 * a, &sn, &cs);
    ph[i] = mk<double>(q * cs, q * sn);
    return;
  }
  const long t = (long)(blockIdx.x - nb0) * 256 + threadIdx.x;
  if (t >= (long)nvid * 4 * ks * NB)
    return;
  const int b = (int)(t % NB), p = (int)(t / NB % (4 * ks)), v = (int)(t / NB / (4 * ks));
  const int2 vs = vsite[v];
  const RsSite &g = geo[vs.x];
  cplx<double> c = mk<double>(0, 0);
  if (b < nbc && p < g.nproj) {
    int m = p, ch = g.chan_off;
    for (; m >= 2 * chan_l[ch] + 1; ch++)
      m -= 2 * chan_l[ch] + 1;
    m -= chan_l[ch];
    const cplx<double> *P = proj + (long)b * ldp + g.proj_off + p;
    if (m == 0) {
      c = *P;
    } else {
      const int am = m < 0 ? -m : m;
      const double sg = (am & 1) ? -1.0 : 1.0;
      const cplx<double> pp = m > 0 ? P[0] : P[2 * am], pn = m > 0 ? P[-2 * am] : P[0];
      c = m > 0 ? mk<double>(pp.x + sg * pn.x, pp.y + sg * pn.y)
                : mk<double>(-(pp.y - sg * pn.y), pp.x - sg * pn.x);
    }
    const int s0 = vs.y / 9 - 1, s1 = vs.y / 3 % 3 - 1, s2 = vs.y % 3 - 1;
    double sn, cs;
    sincospi(2.0 * (k0 * (g.R[0] - s0) + k1 * (g.R[1] - s1) + k2 * (g.R[2] - s2)), &sn, &cs);
    c = c * mk<double>(cs, sn);
    if (!(isfinite(c.x) && isfinite(c.y))) {
      c = mk<double>(0, 0);
      for (int q = 0; q < (2 * g.g[0] + 1) * (2 * g.g[1] + 1) * (2 * g.g[2] + 1); q++) {
        int i, j, k;
        rs_cand(g, q, i, j, k);
        double d[3];
        if (!(rs_vec(g, L, f0, f1, f2, i, j, k, d) < g.rmax))
          continue;
        const long pt = ((long)((i + f0) % f0) * f1 + (j + f1) % f1) * f2 + (k + f2) % f2;
        grid[pt * NB + b] = mk<T>((T)NAN, (T)NAN);
      }
    }
  }
  coef[t] = c;
}

typedef double rs_doublex4 __attribute__((ext_vector_type(4)));

struct RsTileArgs {
  const int *off;      // first entry of every (line, block of 16 x)
  const int4 *ent;     // entries: (site image, ...)
  const double *tab;   // [entry][ks][64]
  const cplx<double> *coef;  // [site image][4 ks][NB]
  const cplx<double> *ph;
  int ks, nxb, NB, nbc, f0, f1, f2;
  int rz;  // x-lines of a work-group
  int xcd; // states: work-groups of an XCD
  double scl;
  int unphase;
  cplx<double> *states;  // [band][ldo]
  long ldo;
  double *dens;
  RsWeights w;
};

template <int CTRL> __device__ __forceinline__ double rs_dpp_add(double v) {
  int2 u = __builtin_bit_cast(int2, v);
  u.x = __builtin_amdgcn_mov_dpp(u.x, CTRL, 0xF, 0xF, true);
  u.y = __builtin_amdgcn_mov_dpp(u.y, CTRL, 0xF, 0xF, true);
  return v + __builtin_bit_cast(double, u);
}
// Sum over the 16 lanes of a row (in every lane): neighbours, pairs (quad
// permutes), then the mirrored half and row.
__device__ __forceinline__ double rs_row_sum(double v) {
  return rs_dpp_add<0x140>(rs_dpp_add<0x141>(rs_dpp_add<0x4E>(rs_dpp_add<0xB1>(v))));
}

// Work-group: rz (at most RS_Z) consecutive x-lines (y, z..) of one block of
// 16 x, so that their densities are written as rows of rz consecutive z; each
// of the four wavefronts takes every fourth line, PL groups of 16 bands at a
// time: one accumulator tile of the real parts and one of the imaginary parts
// for each (a lane past the chunk's bands repeats its last one, unused).  KS:
// groups of four projector slots (0: any number).  With ST the finished
// states go straight from the FP64 accumulators to the band-major output, the
// four wavefronts' lines together through LDS as rows of four consecutive z:
// the chunk is not written, and no rounding follows an FP32 transform.  (Put
// back into the chunk for a copy to the band-major output, the states of 64
// bands on 108^3 with 18 projectors took 1540 us in FP32 and 2098 in FP64
// where these take 1290 and 1680.)  Two LDS tiles leave one barrier a step;
// the run-time form keeps to one tile and its occupancy (32 projectors, FP64:
// 1980 us, 2190 with two).
constexpr int RS_Z = 16;
constexpr int RS_E = 8;  // entries of a line's block whose site images are kept in LDS
constexpr int RS_SB = 65;  // row of a band in the states' LDS tile: 16 x of 4 z, and one off the banks
// Wavefronts per SIMD that the compiled forms are held to: with room for one
// more the compiler saves registers by loading the coefficients in smaller
// batches (108^3, 64 bands, 9 projectors, FP32 density: 852 us against 793).
// The run-time form, whose loads wait anyway, takes what fits (32 projectors,
// FP64 density: 1555 us, held to three 1616).
constexpr int rs_waves(int KS, int PL, bool most) { return most && KS == 0 ? 8 : PL > 1 ? 3 : 4; }
template <typename T, int KS, int PL, bool ST>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(rs_waves(KS, PL, false), rs_waves(KS, PL, true))))
void k_rs_tiles(cplx<T> *__restrict__ g, RsTileArgs L) {
  typedef T vec2 __attribute__((ext_vector_type(2)));
  __shared__ double dl[16][RS_Z + 1];
  __shared__ double s_w[64];
  __shared__ int s_i0[RS_Z], s_i1[RS_Z], s_vid[RS_Z * RS_E];
  __shared__ cplx<double> s_ez[RS_Z];
  __shared__ cplx<double> s_st2[KS > 0 ? 2 : 1][ST ? 16 * PL * RS_SB : 1];
  // z, then y, then the block of x: groups in flight together share 16 planes.
  // States: consecutive groups on one XCD, since the group of the next four z
  // writes the other half of each band's 128 bytes and one L2 has to merge the
  // two (90^3 points, 64 bands, 4 projectors: 728 -> 608 us FP32, 970 -> 833
  // FP64; 60^3 and 108^3 within 2%).
  const int nzb = (L.f2 + L.rz - 1) / L.rz, nyz = L.f1 * nzb;
  const int blk = ST ? (int)(blockIdx.x % 8) * L.xcd + (int)(blockIdx.x / 8) : (int)blockIdx.x;
  if (ST && blk >= L.nxb * nyz)
    return;
  const int xb = blk / nyz, r = blk % nyz;
  const int y = r / nzb, z0 = (r % nzb) * L.rz;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, row = lane >> 4;
  if (threadIdx.x < 64)
    s_w[threadIdx.x] = threadIdx.x < (unsigned)L.nbc ? L.w.w[threadIdx.x] : 0.0;
  // the lines' entry ranges, site images and phases
  if (threadIdx.x < RS_Z * RS_E) {
    const int q = threadIdx.x / RS_E, k = threadIdx.x % RS_E, z = min(z0 + q, L.f2 - 1);
    const long cell = ((long)y * L.f2 + z) * L.nxb + xb;
    const int i0 = L.off[cell], i1 = L.off[cell + 1];
    if (k == 0) {
      s_i0[q] = i0;
      s_i1[q] = i1;
      s_ez[q] = L.ph[L.f0 + L.f1 + z];
    }
    s_vid[threadIdx.x] = i0 + k < i1 ? L.ent[i0 + k].x : 0;
  }
  __syncthreads();
  cplx<double> ex[4];
  vec2 *gx[4];
  const cplx<double> ey = L.ph[L.f0 + y];
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const int x = min(16 * xb + row + 4 * v, L.f0 - 1);
    ex[v] = L.ph[x] * ey;
    gx[v] = reinterpret_cast<vec2 *>(g + ((long)x * L.f1 + y) * L.f2 * L.NB);
  }
  const int ks = KS > 0 ? KS : L.ks, nh = (L.NB + 16 * PL - 1) / (16 * PL);
  // the wavefront's steps: its lines, PL groups at a time.  A step's chunk
  // values are loaded during the step before.  (With ST all wavefronts take
  // as many steps, for the barriers; a line past the last repeats it.)
  const int nz = min(L.rz, L.f2 - z0), nstep = (ST ? (nz + 3) / 4 : (nz - wave + 3) / 4) * nh;
  vec2 u[PL][4];
  auto places = [&](int h, int (&at)[PL]) {
#pragma unroll
    for (int c = 0; c < PL; c++)
      at[c] = min((h * PL + c) * 16 + col, L.NB - 1);
  };
  auto line = [&](int s) { return ST ? min(wave + 4 * (s / nh), nz - 1) : wave + 4 * (s / nh); };
  auto values = [&](int s, vec2 (&w)[PL][4]) {
    int at[PL];
    places(s % nh, at);
    const long zo = (long)(z0 + line(s)) * L.NB;
#pragma unroll
    for (int v = 0; v < 4; v++)
#pragma unroll
      for (int c = 0; c < PL; c++)
        w[c][v] = __builtin_nontemporal_load(gx[v] + zo + at[c]);
  };
  // the projector values of the step's first entry, loaded with them
  double tf[KS > 0 ? KS : 1];
  auto table = [&](int s) {
    if (KS > 0) {
      const int q = line(s);
      const double *ta = L.tab + (long)min(s_i0[q], max(s_i1[q] - 1, 0)) * KS * 64 + lane;
#pragma unroll
      for (int j = 0; j < KS; j++)
        tf[j] = ta[j * 64];
    }
  };
  if (nstep > 0) {
    values(0, u);
    table(0);
  }
  double dens[4] = {0.0, 0.0, 0.0, 0.0};
  for (int st = 0; st < nstep; st++) {
    const int zi = line(st), h = st % nh;
    const int i0 = __builtin_amdgcn_readfirstlane(s_i0[zi]), i1 = __builtin_amdgcn_readfirstlane(s_i1[zi]);
    const cplx<double> ez = s_ez[zi];
    int at[PL];
    places(h, at);
    rs_doublex4 dr[PL], di[PL];
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const cplx<double> e = ex[v] * ez;
#pragma unroll
      for (int c = 0; c < PL; c++) {
        const double a = (double)u[c][v].x, b = (double)u[c][v].y;
        dr[c][v] = a * e.x - b * e.y;
        di[c][v] = b * e.x + a * e.y;
      }
    }
    if (st + 1 < nstep)
      values(st + 1, u);
    int i = i0;
    if (KS > 0 && i < i1) {
      const int vid = __builtin_amdgcn_readfirstlane(s_vid[zi * RS_E]);
      const cplx<double> *cb = L.coef + ((long)vid * ks * 4 + row) * L.NB;
      // a group's coefficients are loaded before the products of the group
      // before it (left alone the compiler waits for each load ahead of its two
      // products: density of 64 bands and 18 projectors on 108^3, FP64 1466
      // against 1306 us, FP32 990 against 890; one group at a time keeps to the
      // registers of three wavefronts per SIMD, all groups at once spill)
      cplx<double> q[2][PL];
      auto coefs = [&](int j) {
#pragma unroll
        for (int c = 0; c < PL; c++)
          q[j & 1][c] = cb[j * 4 * L.NB + at[c]];
      };
      coefs(0);
#pragma unroll
      for (int j = 0; j < KS; j++) {
        if (j + 1 < KS)
          coefs(j + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < PL; c++) {
          dr[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(tf[j], q[j & 1][c].x, dr[c], 0, 0, 0);
          di[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(tf[j], q[j & 1][c].y, di[c], 0, 0, 0);
        }
      }
      i++;
    }
    if (st + 1 < nstep)
      table(st + 1);
    for (; i < i1; i++) {
      const int vid = __builtin_amdgcn_readfirstlane(i - i0 < RS_E ? s_vid[zi * RS_E + i - i0] : L.ent[i].x);
      const double *ta = L.tab + (long)i * ks * 64 + lane;
      const cplx<double> *cb = L.coef + ((long)vid * ks * 4 + row) * L.NB;
      if constexpr (KS > 0) {
        cplx<double> q[2][PL];
        double av[2];
        auto load = [&](int j) {
          av[j & 1] = ta[j * 64];
#pragma unroll
          for (int c = 0; c < PL; c++)
            q[j & 1][c] = cb[j * 4 * L.NB + at[c]];
        };
        load(0);
#pragma unroll
        for (int j = 0; j < KS; j++) {
          if (j + 1 < KS)
            load(j + 1);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int c = 0; c < PL; c++) {
            dr[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[j & 1], q[j & 1][c].x, dr[c], 0, 0, 0);
            di[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[j & 1], q[j & 1][c].y, di[c], 0, 0, 0);
          }
        }
      } else {
        for (int j = 0; j < ks; j++) {
          const double av = ta[j * 64];
#pragma unroll
          for (int c = 0; c < PL; c++) {
            const cplx<double> q = cb[j * 4 * L.NB + at[c]];
            dr[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, q.x, dr[c], 0, 0, 0);
            di[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, q.y, di[c], 0, 0, 0);
          }
        }
      }
    }
    if (L.dens) {
#pragma unroll
      for (int c = 0; c < PL; c++) {
        const int b = (h * PL + c) * 16 + col;
        if (b < L.nbc) {
          const double w = s_w[b];
#pragma unroll
          for (int v = 0; v < 4; v++)
            dens[v] += w * (dr[c][v] * dr[c][v] + di[c][v] * di[c][v]);
        }
      }
      if (h + 1 == nh) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const double q = rs_row_sum(dens[v]);
          if (col == 0)
            dl[row + 4 * v][zi] = q;
          dens[v] = 0.0;
        }
      }
    }
    if constexpr (ST) {
      cplx<double> *s_st = s_st2[KS > 0 ? st & 1 : 0];
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const cplx<double> e = ex[v] * ez;
#pragma unroll
        for (int c = 0; c < PL; c++) {
          double a = dr[c][v], b = di[c][v];
          if (L.unphase) {  // times e^{-2 pi i k.r}
            a = (dr[c][v] * e.x + di[c][v] * e.y) / L.scl;
            b = (di[c][v] * e.x - dr[c][v] * e.y) / L.scl;
          }
          s_st[(c * 16 + col) * RS_SB + (row + 4 * v) * 4 + wave] = mk<double>(a, b);
        }
      }
      __syncthreads();
      const int zl = 4 * (st / nh) + (threadIdx.x & 3), x = 16 * xb + (threadIdx.x >> 2 & 15);
      if (zl < nz && x < L.f0) {
        const long pt = ((long)x * L.f1 + y) * L.f2 + z0 + zl;
#pragma unroll
        for (int q = 0; q < 4 * PL; q++) {
          const int band = (int)(threadIdx.x >> 6) + 4 * q, b = h * PL * 16 + band;
          if (b < L.nbc)
            L.states[b * L.ldo + pt] = s_st[band * RS_SB + (threadIdx.x & 63)];
        }
      }
      if (KS == 0)
        __syncthreads();
    }
  }
  if (!L.dens)
    return;
  __syncthreads();
  const int x = 16 * xb + (threadIdx.x >> 4), zi = threadIdx.x & 15;
  if (x < L.f0 && zi < nz)
    L.dens[((long)x * L.f1 + y) * L.f2 + z0 + zi] += dl[threadIdx.x >> 4][zi];
}

static int tile_build(pp_ctx *ctx, pp_rsplan *rp) {
  const int ns = rp->nsites, f0 = rp->fftg[0], f1 = rp->fftg[1], f2 = rp->fftg[2];
  const int nxb = (f0 + 15) / 16;
  const long ncell = (long)f1 * f2 * nxb;
  hipStream_t sm = ctx->stream;
  RsLat L;
  memcpy(L.m, rp->lattice, sizeof(L.m));
  int wmax = 1;
  for (const RsSite &g : rp->geo)
    wmax = std::max(wmax, (2 * g.g[1] + 1) * (2 * g.g[2] + 1));
  rp->ks = (rp->pmax + 3) / 4;
  DevBuf cells, used, vid;
  PP_TRY(cells.ensure(sizeof(int) * ncell));
  PP_TRY(used.ensure(sizeof(int) * 27 * ns));
  PP_TRY(vid.ensure(sizeof(int) * 27 * ns));
  PP_TRY(rp->l_off.ensure(sizeof(int) * (ncell + 1)));
  PP_TRY(zero_async(ctx, cells.p, sizeof(int) * ncell));
  PP_TRY(zero_async(ctx, used.p, sizeof(int) * 27 * ns));
  const dim3 grd((wmax + 255) / 256, ns);
  hipLaunchKernelGGL(k_rst_count, grd, dim3(256), 0, sm, (const RsSite *)rp->d_geo.p, L, f0, f1, f2, nxb,
                     (int *)cells.p, (int *)used.p);
  PP_CHECK_HIP(hipGetLastError());
  std::vector<int> hc(ncell), hu(27 * (size_t)ns), off(ncell + 1), hvid(27 * (size_t)ns, -1);
  PP_CHECK_HIP(hipMemcpyAsync(hc.data(), cells.p, sizeof(int) * ncell, hipMemcpyDeviceToHost, sm));
  PP_CHECK_HIP(hipMemcpyAsync(hu.data(), used.p, sizeof(int) * hu.size(), hipMemcpyDeviceToHost, sm));
  PP_CHECK_HIP(hipStreamSynchronize(sm));
  long acc = 0;
  for (long c = 0; c < ncell; c++) {
    off[c] = (int)acc;
    acc += hc[c];
  }
  if (acc >= (1L << 31))
    return PP_ERR_NOMEM;
  off[ncell] = (int)acc;
  rp->nent = acc;
  std::vector<int2> vsite;
  for (int i = 0; i < 27 * ns; i++)
    if (hu[i]) {
      hvid[i] = (int)vsite.size();
      vsite.push_back(make_int2(i / 27, i % 27));
    }
  rp->nvid = (int)vsite.size();
  PP_TRY(rp->l_ent.ensure(sizeof(int4) * std::max(1L, acc)));
  PP_TRY(rp->l_tab.ensure(sizeof(double) * 64 * rp->ks * std::max(1L, acc)));
  PP_TRY(rp->l_vid.ensure(sizeof(int2) * std::max<size_t>(1, vsite.size())));
  PP_CHECK_HIP(hipMemcpyAsync(rp->l_off.p, off.data(), sizeof(int) * (ncell + 1), hipMemcpyHostToDevice, sm));
  if (acc) {
    PP_CHECK_HIP(hipMemcpyAsync(vid.p, hvid.data(), sizeof(int) * hvid.size(), hipMemcpyHostToDevice, sm));
    PP_CHECK_HIP(hipMemcpyAsync(rp->l_vid.p, vsite.data(), sizeof(int2) * vsite.size(), hipMemcpyHostToDevice, sm));
    hipLaunchKernelGGL(k_rst_fill, grd, dim3(256), 0, sm, (const RsSite *)rp->d_geo.p, L, f0, f1, f2, nxb,
                       (const int *)rp->l_off.p, (int *)cells.p, (const int *)vid.p, (int4 *)rp->l_ent.p);
    hipLaunchKernelGGL(k_rst_sort, dim3((unsigned)((ncell + 255) / 256)), dim3(256), 0, sm, ncell,
                       (const int *)rp->l_off.p, (int4 *)rp->l_ent.p);
    hipLaunchKernelGGL(k_rst_values, dim3((unsigned)((acc + 15) / 16)), dim3(256), 0, sm, (const RsSite *)rp->d_geo.p, L,
                       f0, f1, f2, acc, (const int4 *)rp->l_ent.p, (const int2 *)rp->l_vid.p, rp->ks,
                       (const double *)rp->d_spl.p, (const int *)rp->d_chan_l.p, (double *)rp->l_tab.p);
    PP_CHECK_HIP(hipGetLastError());
  }
  PP_CHECK_HIP(hipStreamSynchronize(sm));  // host staging buffers end here
  rp->tile_built = true;
  return PP_OK;
}
// The work lists.  *use = false where the plan has none: no projectors, a box that
// reaches past the neighbouring cells, more blocks than an int counts, or no
// memory for them (a block's table is 16 points long whatever the sphere holds
// of it); the per-site kernels run then.
int rs_tile_ensure(pp_ctx *ctx, pp_rsplan *rp, bool *use) {
  std::lock_guard<std::mutex> lk(rp->build_mu);
  if (rp->tile_ok && !rp->tile_built) {
    int st;
    try {
      st = tile_build(ctx, rp);
    } catch (const std::bad_alloc &) {
      st = PP_ERR_NOMEM;
    }
    if (st == PP_ERR_NOMEM) {
      (void)hipGetLastError();  // the failed allocation's
      rp->tile_ok = false;
      rp->l_off.release();
      rp->l_ent.release();
      rp->l_tab.release();
      rp->l_vid.release();
    } else if (st) {
      return st;
    }
  }
  *use = rp->tile_ok;
  return PP_OK;
}

template <typename T, int KS>
static void rs_tiles_launch(hipStream_t st, cplx<T> *grid, const RsTileArgs &L, unsigned blocks) {
#define PP_RT(PL, ST) hipLaunchKernelGGL((k_rs_tiles<T, KS, PL, ST>), dim3(blocks), dim3(256), 0, st, grid, L)
  if (L.NB <= 16) {
    if (L.states)
      PP_RT(1, true);
    else
      PP_RT(1, false);
  } else if (L.states) {
    PP_RT(2, true);
  } else {
    PP_RT(2, false);
  }
#undef PP_RT
}

// The augmentation of a transformed chunk: densities (wts, dens) and / or the
// finished states, either of them null.
template <typename T>
int rs_tile_run(pp_ctx *ctx, pp_rsplan *rp, const double *kf, int nbc, int NB, const cplx<double> *proj, long ldp,
                int remove_phase, cplx<double> *states, long ldo, const double *wts, double *dens, cplx<T> *grid) {
  const int f0 = rp->fftg[0], f1 = rp->fftg[1], f2 = rp->fftg[2];
  DevBuf &qb = ctx->rs_coef[ctx->slot];
  const long nq = (long)rp->nvid * 4 * rp->ks * NB, nph = f0 + f1 + f2;
  PP_TRY(qb.ensure(sizeof(cplx<double>) * (nq + nph)));
  cplx<double> *coef = (cplx<double> *)qb.p, *ph = coef + nq;
  RsTileArgs L{};
  L.scl = 1.0 / sqrt(det3(rp->lattice));
  RsLat lat;
  memcpy(lat.m, rp->lattice, sizeof(lat.m));
  const int nb0 = (int)((nph + 255) / 256);
  hipLaunchKernelGGL(k_rst_coef<T>, dim3((unsigned)(nb0 + (nq + 255) / 256)), dim3(256), 0, ctx->stream, nb0, rp->nvid,
                     (const int2 *)rp->l_vid.p, (const RsSite *)rp->d_geo.p, (const int *)rp->d_chan_l.p, rp->ks, NB,
                     nbc, proj, ldp, kf[0], kf[1], kf[2], lat, f0, f1, f2, L.scl, ph, coef, grid);
  PP_CHECK_HIP(hipGetLastError());
  L.off = (const int *)rp->l_off.p;
  L.ent = (const int4 *)rp->l_ent.p;
  L.tab = (const double *)rp->l_tab.p;
  L.coef = coef;
  L.ph = ph;
  L.ks = rp->ks;
  L.nxb = (f0 + 15) / 16;
  L.NB = NB;
  L.nbc = nbc;
  L.f0 = f0;
  L.f1 = f1;
  L.f2 = f2;
  L.states = states;
  L.ldo = ldo;
  L.unphase = remove_phase;
  L.dens = dens;
  for (int b = 0; b < 64; b++)
    L.w.w[b] = dens && b < nbc ? wts[b] : 0.0;
  // Four lines a work-group (one a wavefront) where 16 leave the chip short of
  // work-groups (fewer than two per CU: 20^3, 64 bands, 18 projectors, states
  // 125 -> 100 us), and for states of more than 16 bands, whose work-groups
  // wait on each other's lines (64 FP32 bands, 4 projectors: 90^3 749 -> 608 us,
  // 108^3 1162 -> 1101).
  // Else 16, which read the lines' tables together (108^3, 4 bands: 378 us
  // against 417).
  const long cols = (long)L.nxb * f1;
  L.rz = cols * ((f2 + RS_Z - 1) / RS_Z) < 512 || (states && NB > 16) ? 4 : RS_Z;
  long blocks = cols * ((f2 + L.rz - 1) / L.rz);
  L.xcd = (int)((blocks + 7) / 8);
  if (states)
    blocks = 8L * L.xcd;
  switch (rp->ks) {
#define PP_KS(K)                                                        \
  case K:                                                               \
    rs_tiles_launch<T, K>(ctx->stream, grid, L, (unsigned)blocks);      \
    break;
    PP_KS(1) PP_KS(2) PP_KS(3) PP_KS(4) PP_KS(5)
#undef PP_KS
  default:
    rs_tiles_launch<T, 0>(ctx->stream, grid, L, (unsigned)blocks);
  }
  PP_CHECK_HIP(hipGetLastError());
  return PP_OK;
}
template int rs_tile_run<float>(pp_ctx *, pp_rsplan *, const double *, int, int, const cplx<double> *, long, int,
                                cplx<double> *, long, const double *, double *, cplx<float> *);
template int rs_tile_run<double>(pp_ctx *, pp_rsplan *, const double *, int, int, const cplx<double> *, long, int,
                                 cplx<double> *, long, const double *, double *, cplx<double> *);

}  // namespace pp

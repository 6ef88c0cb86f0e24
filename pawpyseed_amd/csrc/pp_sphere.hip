// Projector spheres: table build and the <p_i|psi_nk> sphere sums.
//
// Table build replaces projector.c:193-209 / utils.c:590-696 (serial in the
// reference): per site, every grid point of the bounding box
// +-(int(|a_j x a_k| rmax / V * N_i) + 1) around round(frac * N) with
// |r - R| < (n-1)/n * rmax.  The points of a site are listed line by line
// (j, k outer, i innermost; the reference loops i-j-k, which only changes
// the order of the floating-point sums), so the points of one site on one
// x-line (j, k) form one run of consecutive i, a segment.  Each point
// stores its wrapped grid index, its unwrapped path r - R (for the Bloch
// phase) and, for every projector j = (channel, l, m) of the site, the
// real value t_j of the projector in real-harmonic form:
//   t_(l,m)  = A_lm cos(m phi)   (m >= 0),
//   t_(l,-m) = A_lm sin(m phi)   (m > 0),
// A_lm = N_lm P_l^m(cos theta) spline_l(|r|), evaluated on the
// minimum-image vector (utils.c:547-576).
//
// Sphere sums replace projector.c:223-274 (onto_projector_helper):
// <p_j|psi> = sum_i conj(p_j(i)) psi(idx_i) dv exp(i k.path_i).  With
// s_j = sum_i t_j(i) psi(idx_i) dv exp(i k.path_i) and
// Y_l,-m = (-1)^m conj(Y_lm) (utils.c:377-386, 441-449):
//   <p_(l,m)|psi>  = s_(l,m) - i s_(l,-m),
//   <p_(l,-m)|psi> = (-1)^m (s_(l,m) + i s_(l,-m)),
// so the sums run over real table values (half the flops and bytes of a
// complex table) and the reduction kernel forms the complex projections.
// One work-group per (site, part of its points); lane = band of the chunk,
// so each point's NB bands are one contiguous load from the band-fastest
// grid while the projector values and phase are uniform across the wave.
#include <cmath>
#include <cstring>

#include "pp_geom.h"
#include "pp_sphere.h"

namespace pp {

struct Lat9 {
  double m[9];
};

// decode candidate c of a site's box into (i, j, k): i fastest, then k,
// then j; c % (2 g0 + 1) is the position of i on its line
__device__ __forceinline__ void box_ijk(const SiteGeo &s, int c, int &i, int &j, int &k) {
  int w0 = 2 * s.g[0] + 1, w2 = 2 * s.g[2] + 1;
  i = c % w0 - s.g[0] + s.c[0];
  int t = c / w0;
  k = t % w2 - s.g[2] + s.c[2];
  j = t / w2 - s.g[1] + s.c[1];
}

__device__ __forceinline__ bool inside(const SiteGeo &s, const Lat9 &L, const int *fftg, int i, int j, int k,
                                       double *cv) {
  double fv[3] = {(double)i / fftg[0] - s.coord[0], (double)j / fftg[1] - s.coord[1],
                  (double)k / fftg[2] - s.coord[2]};
  d_frac_to_cart(fv, L.m, cv);
  return sqrt(cv[0] * cv[0] + cv[1] * cv[1] + cv[2] * cv[2]) < s.R0;
}

// The lists of a site are made by one work-group of SITE_W wavefronts, which
// take 63 consecutive candidates at a time and lane 0 the one before them, so
// that a wavefront's two ballots hold its inside flags and segment starts and
// only the counts cross wavefronts.  Bound by the chain of tiles of a site:
// 256 threads with shared flags and scans took 28 us to count and 88 to fill
// for 215 sites of 4,900 points where these take 21 and 35, and for 8 sites 6
// and 14 where these take 4 and 6.  A segment starts at an inside candidate
// that is the first of its line or follows an outside one.
constexpr int SITE_W = 16;
struct SiteBallot {
  unsigned long long in, start;  // of lanes 1..63
  bool mine, first;              // the lane's own bits
  int i, j, k;
  double cv[3];
};
__device__ __forceinline__ SiteBallot site_ballot(const SiteGeo &s, const Lat9 &L, const int *fftg, int c0, int ncand) {
  SiteBallot q;
  const int lane = threadIdx.x & 63, c = c0 + lane - 1;
  bool in = false;
  if (c >= 0 && c < ncand) {
    box_ijk(s, c, q.i, q.j, q.k);
    in = inside(s, L, fftg, q.i, q.j, q.k, q.cv);
  }
  const unsigned long long m = __ballot(in);
  q.mine = in && lane > 0;
  q.first = q.mine && (c % (2 * s.g[0] + 1) == 0 || !(m >> (lane - 1) & 1));
  q.in = m & ~1ull;
  q.start = __ballot(q.first);
  return q;
}

// points (counts[s]) and segments (counts[nsites + s]) of every site
__global__ __launch_bounds__(64 * SITE_W) void k_site_count(const SiteGeo *__restrict__ geo, Lat9 L, int f0, int f1,
                                                            int f2, int nsites, int *__restrict__ counts) {
  const SiteGeo s = geo[blockIdx.x];
  const int fftg[3] = {f0, f1, f2};
  const int ncand = (2 * s.g[0] + 1) * (2 * s.g[1] + 1) * (2 * s.g[2] + 1);
  const int wave = threadIdx.x >> 6;
  __shared__ int red[2][SITE_W];
  int cnt = 0, nseg = 0;
  for (int c0 = 63 * wave; c0 < ncand; c0 += 63 * SITE_W) {
    const SiteBallot q = site_ballot(s, L, fftg, c0, ncand);
    cnt += __popcll(q.in);
    nseg += __popcll(q.start);
  }
  if ((threadIdx.x & 63) == 0) {
    red[0][wave] = cnt;
    red[1][wave] = nseg;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    int n = 0;
    for (int w = 0; w < SITE_W; w++)
      n += red[threadIdx.x][w];
    counts[threadIdx.x * nsites + blockIdx.x] = n;
  }
}

// Ordered compaction of the inside candidates and of the segment starts, a
// tile of 63 SITE_W candidates at a time.  A segment is stored as (first
// point, length, wrapped i of the first point, site) and its wrapped line
// j * N2 + k; the lengths are filled in by k_seg_len.
__global__ __launch_bounds__(64 * SITE_W) void k_site_fill(const SiteGeo *__restrict__ geo, Lat9 L, int f0, int f1,
                                                           int f2, const int *__restrict__ site_pt,
                                                           const int *__restrict__ seg_off, int *__restrict__ pidx,
                                                           double *__restrict__ path, int4 *__restrict__ seg,
                                                           int *__restrict__ segline) {
  const SiteGeo s = geo[blockIdx.x];
  const int fftg[3] = {f0, f1, f2};
  const int ncand = (2 * s.g[0] + 1) * (2 * s.g[1] + 1) * (2 * s.g[2] + 1);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __shared__ int cnt[2][SITE_W];  // points, and segments << 16, of a tile's wavefronts
  int run = site_pt[blockIdx.x], runs = seg_off[blockIdx.x];
  for (int c0 = 0, p = 0; c0 < ncand; c0 += 63 * SITE_W, p ^= 1) {
    const SiteBallot q = site_ballot(s, L, fftg, c0 + 63 * wave, ncand);
    if (lane == 0)
      cnt[p][wave] = __popcll(q.in) | __popcll(q.start) << 16;
    __syncthreads();  // the next tile's counts go to the other half
    int before = 0, all = 0;
    for (int w = 0; w < SITE_W; w++) {
      before += w < wave ? cnt[p][w] : 0;
      all += cnt[p][w];
    }
    const unsigned long long below = (1ull << lane) - 1;
    if (q.mine) {
      const int pos = run + (before & 0xffff) + __popcll(q.in & below);
      const int ii = (q.i % fftg[0] + fftg[0]) % fftg[0];
      const int jj = (q.j % fftg[1] + fftg[1]) % fftg[1];
      const int kk = (q.k % fftg[2] + fftg[2]) % fftg[2];
      pidx[pos] = (ii * fftg[1] + jj) * fftg[2] + kk;
      path[3 * (long)pos + 0] = q.cv[0];
      path[3 * (long)pos + 1] = q.cv[1];
      path[3 * (long)pos + 2] = q.cv[2];
      if (q.first) {
        const int n = runs + (before >> 16) + __popcll(q.start & below);
        seg[n] = make_int4(pos, 0, ii, blockIdx.x);
        segline[n] = jj * fftg[2] + kk;
      }
    }
    run += all & 0xffff;
    runs += all >> 16;
  }
}

// Coverage masks of the x-lines: every segment sets the bits of its points.
__global__ __launch_bounds__(256) void k_xmask(const int4 *__restrict__ seg, const int *__restrict__ segline,
                                               long nseg, int n0, int mw, unsigned *__restrict__ mask) {
  const long q = (long)blockIdx.x * 256 + threadIdx.x;
  if (q >= nseg)
    return;
  const int4 sg = seg[q];
  unsigned *m = mask + (long)segline[q] * mw;
  int x = sg.z;
  for (int i = 0; i < sg.y; i++) {
    atomicOr(&m[x >> 5], 1u << (x & 31));
    if (++x == n0)
      x = 0;
  }
}

// Segment lengths: the points of segment q run to the first point of the
// next segment of its site, or to the end of the site's points.
__global__ __launch_bounds__(256) void k_seg_len(int4 *__restrict__ seg, long nseg, const int *__restrict__ seg_off,
                                                 const int *__restrict__ site_pt) {
  const long q = (long)blockIdx.x * 256 + threadIdx.x;
  if (q >= nseg)
    return;
  const int4 sg = seg[q];
  const int end = q + 1 < seg_off[sg.w + 1] ? seg[q + 1].x : site_pt[sg.w + 1];
  seg[q].y = end - sg.x;
}

// Rows of zeros behind a site's FP32 table: the sums read its rows in whole
// groups of 16.  (Clamping the rows in the sums instead cost them 3%: 216^3,
// 215 sites, 16 bands 676 -> 693 us.)
constexpr int TAB_PAD = 15;

template <typename T>
__global__ __launch_bounds__(256) void k_site_values(const SiteGeo *__restrict__ geo, Lat9 L, int f0, int f1, int f2,
                                                     const int *__restrict__ site_pt, const long *__restrict__ tab_off,
                                                     const int *__restrict__ pidx, const double *__restrict__ spl,
                                                     const int *__restrict__ chan_l, T *__restrict__ table) {
  const int s_id = blockIdx.y;
  const SiteGeo s = geo[s_id];
  const int p0 = site_pt[s_id], np = site_pt[s_id + 1] - p0;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= np) {
    const int w = table_stride(s.nproj, sizeof(T) == 4);
    if (sizeof(T) == 4 && i < np + TAB_PAD)
      for (int p = 0; p < w; p++)
        table[tab_off[s_id] + (long)i * w + p] = (T)0;
    return;
  }
  const int fftg[3] = {f0, f1, f2};
  int g = pidx[p0 + i];
  int kk = g % fftg[2];
  int jj = (g / fftg[2]) % fftg[1];
  int ii = g / (fftg[1] * fftg[2]);
  double pf[3] = {(double)ii / fftg[0], (double)jj / fftg[1], (double)kk / fftg[2]};
  // minimum image of the wrapped point (utils.c:51-73, 566-576)
  // (a square that is no smaller has no smaller root: few roots are taken)
  double best = INFINITY, best2 = INFINITY, v[3] = {0, 0, 0};
  for (int a = -1; a <= 1; a++)
    for (int b = -1; b <= 1; b++)
      for (int c = -1; c <= 1; c++) {
        double fv[3] = {pf[0] + a - s.coord[0], pf[1] + b - s.coord[1], pf[2] + c - s.coord[2]}, cv[3];
        d_frac_to_cart(fv, L.m, cv);
        const double d2 = cv[0] * cv[0] + cv[1] * cv[1] + cv[2] * cv[2];
        if (!(d2 < best2))
          continue;
        const double d = sqrt(d2);
        if (d < best) {
          best = d;
          best2 = d2;
          v[0] = cv[0];
          v[1] = cv[1];
          v[2] = cv[2];
        }
      }
  const double r = best;
  double theta = 0.0, phi = 0.0;
  if (r != 0.0) {
    theta = acos(v[2] / r);
    if (r - fabs(v[2]) != 0.0)
      phi = acos(v[0] / sqrt(v[0] * v[0] + v[1] * v[1]));
    if (v[1] < 0)
      phi = 2.0 * M_PI - phi;
  }
  const double ct = cos(theta);
  const int n = s.ngrid;
  const double *x = spl + s.spl_off;
  const int ts = table_stride(s.nproj, sizeof(T) == 4);
  T *out = table + tab_off[s_id] + (long)i * ts;
  // place on the radial grid (utils.c:461-475), the same for every channel
  const bool beyond = r > x[n - 1], below = r < x[0];
  int id = 0;
  double t = 0.0;
  if (!beyond && !below) {
    id = (int)(r / s.rmax * n);
    if (id > n - 2)
      id = n - 2;
    t = r - x[id];
  }
  // Channels of one l in a row share their angular factors: four channels'
  // radial values, then for each |m| the two real forms: slot m >= 0 holds
  // A_|m| cos(|m| phi), slot -|m| holds A_|m| sin(|m| phi), with
  // A_|m| = N_l|m| P_l^|m|(cos theta) radial.  Bound by its FP64 operations
  // (215 sites of 4,900 points, two channels of l = 0, 1, 2: 143 us with the
  // factors made for every slot and a root for each of the 27 images, 123 so).
  constexpr int CR = 4;
  int p = 0;
  for (int ch = 0; ch < s.nchan;) {
    const int l = chan_l[s.chan_off + ch];
    int nc = 1;
    while (nc < CR && ch + nc < s.nchan && chan_l[s.chan_off + ch + nc] == l)
      nc++;
    double radial[CR];
#pragma unroll
    for (int q = 0; q < CR; q++) {
      radial[q] = 0.0;
      if (q < nc && !beyond) {
        const double *f = x + (long)(1 + ch + q) * n;
        const double *bb = f + (long)s.nchan * n, *cc = bb + (long)s.nchan * n, *dd = cc + (long)s.nchan * n;
        radial[q] = below ? f[0] : f[id] + t * (bb[id] + t * (cc[id] + t * dd[id]));
      }
    }
    for (int am = 0; am <= l; am++) {
      const double norm = sqrt((2 * l + 1) / (4.0 * M_PI) * d_fact(l - am) / d_fact(l + am));
      const double a = norm * d_legendre(l, am, ct);
      double sn, cs;
      sincos(am * phi, &sn, &cs);
#pragma unroll
      for (int q = 0; q < CR; q++)
        if (q < nc) {
          const double pl = a * radial[q];
          out[p + q * (2 * l + 1) + l + am] = (T)(pl * cs);
          if (am > 0)
            out[p + q * (2 * l + 1) + l - am] = (T)(pl * sn);
        }
    }
    p += nc * (2 * l + 1);
    ch += nc;
  }
  for (; p < ts; p++)
    out[p] = (T)0;
}

// phase[pt] = dv / sqrt(V) * exp(i kc . path)
template <typename T>
__global__ __launch_bounds__(256) void k_phase(long npts, const double *__restrict__ path, double k0, double k1,
                                               double k2, double scl, cplx<T> *__restrict__ phase) {
  long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= npts)
    return;
  double kr = k0 * path[3 * i] + k1 * path[3 * i + 1] + k2 * path[3 * i + 2];
  double sn, cs;
  sincos(kr, &sn, &cs);
  phase[i] = mk<T>((T)(scl * cs), (T)(scl * sn));
}

// Sphere sums of one (site, part of its points) by a work-group of 4
// wavefronts, FP64; lane b of every wavefront accumulates PM table slots of
// the site, from slot s0 of its rows of RW, for band b of the chunk.  Tiles of TP points stage their
// table rows, phases and grid indices in LDS with coalesced loads; each
// wavefront then takes every fourth point of the tile, U points per step
// with their grid loads in flight together, and reads the table values as
// LDS broadcasts.  The four wavefronts' sums are added in LDS at the end;
// partial[(blk * PMX + j) * NB + b].
template <typename T, int PM, int U, int RW = PM>
__device__ __forceinline__ void sphere_sum_valu(const cplx<T> *__restrict__ g, int NB, int p0, int len,
                                                const int *__restrict__ pidx, const cplx<T> *__restrict__ phase,
                                                const T *__restrict__ tsite, int a, int e,
                                                cplx<T> *__restrict__ partial, int streaming,
                                                T *__restrict__ s_tab, cplx<T> *__restrict__ s_ph,
                                                int *__restrict__ s_idx, int s0 = 0) {
  constexpr int TP = 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool active = lane < NB;
  cplx<T> acc[PM];
#pragma unroll
  for (int j = 0; j < PM; j++)
    acc[j] = mk<T>(0, 0);
  // a tile's table values, indices and phases: every load of a thread is
  // issued before any is written to LDS, so they are in flight together
  constexpr int SL = (TP * PM + 255) / 256;
  T tv[SL];
  int iv = 0;
  cplx<T> pv = mk<T>(0, 0);
  for (int t0 = a; t0 < e; t0 += TP) {
    const int n = min(TP, e - t0);
    const T *tsrc = tsite + (long)(t0 - p0) * RW + s0;
#pragma unroll
    for (int u = 0; u < SL; u++) {
      const int q = tid + u * 256;
      tv[u] = q < n * PM ? tsrc[RW == PM ? q : q / PM * RW + q % PM] : (T)0;
    }
    if (tid < n) {
      iv = pidx[t0 + tid];
      pv = phase[t0 + tid];
    }
#pragma unroll
    for (int u = 0; u < SL; u++) {
      const int q = tid + u * 256;
      if (q < n * PM)
        s_tab[q] = tv[u];
    }
    if (tid < n) {
      s_idx[tid] = iv;
      s_ph[tid] = pv;
    }
    __syncthreads();
    int i = wave;
    for (; i + 4 * (U - 1) < n; i += 4 * U) {
      cplx<T> x[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const cplx<T> *gp = g + (long)s_idx[i + 4 * u] * NB + lane;
        x[u] = active ? (streaming ? load_nt(gp) : *gp) : mk<T>(0, 0);
      }
#pragma unroll
      for (int u = 0; u < U; u++) {
        const cplx<T> xv = x[u] * s_ph[i + 4 * u];
        const T *tp = s_tab + (i + 4 * u) * PM;
#pragma unroll
        for (int j = 0; j < PM; j++) {
          acc[j].x += tp[j] * xv.x;
          acc[j].y += tp[j] * xv.y;
        }
      }
    }
    for (; i < n; i += 4) {
      cplx<T> xv = active ? g[(long)s_idx[i] * NB + lane] : mk<T>(0, 0);
      xv = xv * s_ph[i];
      const T *tp = s_tab + i * PM;
#pragma unroll
      for (int j = 0; j < PM; j++) {
        acc[j].x += tp[j] * xv.x;
        acc[j].y += tp[j] * xv.y;
      }
    }
    __syncthreads();
  }
  // add the four wavefronts' sums, half of the slots at a time through the
  // table tile (at least 64 lanes x (PM + 1) / 2 complex)
  cplx<T> *red = reinterpret_cast<cplx<T> *>(s_tab);
  constexpr int JH = (PM + 1) / 2;
  for (int w = 1; w < 4; w++) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      if (wave == w) {
#pragma unroll
        for (int j = 0; j < JH; j++)
          if (h * JH + j < PM)
            red[j * 64 + lane] = acc[h * JH + j];
      }
      __syncthreads();
      if (wave == 0) {
#pragma unroll
        for (int j = 0; j < JH; j++)
          if (h * JH + j < PM)
            acc[h * JH + j] = acc[h * JH + j] + red[j * 64 + lane];
      }
      __syncthreads();
    }
  }
  if (wave == 0 && active) {
#pragma unroll
    for (int j = 0; j < PM; j++)
      partial[(long)(s0 + j) * NB + lane] = acc[j];
  }
}

typedef float floatx4 __attribute__((ext_vector_type(4)));

// MFMA operand: value `v` of the 64 table values a wavefront holds in one
// register is broadcast to all 16 blocks of the 4x4x1 MFMA, value group
// ABID (4 table slots of one point) against the lane's band.
template <int ABID> __device__ __forceinline__ floatx4 mfma_quad(float tab, float x, floatx4 acc) {
  return __builtin_amdgcn_mfma_f32_4x4x1f32(tab, x, acc, 4, ABID, 0);
}
template <int I, int Q, int N = 0>
__device__ __forceinline__ void mfma_point(const float (&tab)[Q], float xr, float xi, floatx4 (&ar)[Q],
                                           floatx4 (&ai)[Q]) {
  if constexpr (N < Q) {
    constexpr int q = I * Q + N;  // quad q of the group's 16 points x Q quads
    ar[N] = mfma_quad<q % 16>(tab[q / 16], xr, ar[N]);
    ai[N] = mfma_quad<q % 16>(tab[q / 16], xi, ai[N]);
    mfma_point<I, Q, N + 1>(tab, xr, xi, ar, ai);
  }
}
template <int Q, int I = 0>
__device__ __forceinline__ void mfma_group(const float (&tab)[Q], const cplx<float> (&x)[16], cplx<float> ph,
                                           floatx4 (&ar)[Q], floatx4 (&ai)[Q]) {
  if constexpr (I < 16) {
    const float pr = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ph.x), I));
    const float pi = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ph.y), I));
    const cplx<float> v = x[I] * mk<float>(pr, pi);
    mfma_point<I, Q>(tab, v.x, v.y, ar, ai);
    mfma_group<Q, I + 1>(tab, x, ph, ar, ai);
  }
}

// The FP32 sphere sums on the matrix cores.  A wavefront takes groups of 16
// points: the group's 16 x 4Q table values are Q coalesced register loads,
// its 16 grid runs one 512-byte load each (lane = band), and every (point,
// quad of table slots) is one 4x4x1 16-block MFMA per component, the table
// quad broadcast to the 16 blocks (CBSZ = 4, ABID = the quad's place in the
// register), the blocks' columns the 64 bands: no LDS, no barrier and no
// projector guard in the loop, and 2Q MFMAs of 8 cycles per point where the
// VALU form issued 8Q FMAs of 4.  Register v of accumulator q holds table
// slot 4q + v of the lane's band.  A group's tail points repeat the last
// point with phase 0; their table rows are the next part's of the site or the
// zeros behind its last one (TAB_PAD), since another site's need not be finite.
template <int Q>
__device__ __forceinline__ void sphere_sum_mfma(const cplx<float> *__restrict__ g, int NB, int p0, int len,
                                                const int *__restrict__ pidx, const cplx<float> *__restrict__ phase,
                                                const float *__restrict__ tsite, int a, int e,
                                                cplx<float> *__restrict__ partial, int streaming,
                                                float *__restrict__ red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l16 = lane & 15;
  const int band = lane < NB ? lane : 0;
  floatx4 ar[Q], ai[Q];
#pragma unroll
  for (int q = 0; q < Q; q++)
    ar[q] = ai[q] = floatx4{0.f, 0.f, 0.f, 0.f};
  int idx = 0;
  cplx<float> ph = mk<float>(0, 0);
  float tab[Q];
  auto fetch = [&](int g0) {
    const int n = min(16, e - g0);
    const int pt = g0 + (l16 < n ? l16 : n - 1);
    idx = pidx[pt];
    const cplx<float> v = phase[pt];
    ph = l16 < n ? v : mk<float>(0, 0);
    const float *ts = tsite + (long)(g0 - p0) * (4 * Q) + lane;
#pragma unroll
    for (int r = 0; r < Q; r++)
      tab[r] = ts[r * 64];
  };
  int g0 = a + wave * 16;
  if (g0 < e)
    fetch(g0);
  for (; g0 < e; g0 += 64) {
    cplx<float> x[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const cplx<float> *gp = g + (long)__builtin_amdgcn_readlane(idx, i) * NB + band;
      x[i] = streaming ? load_nt(gp) : *gp;
    }
    // the next group's table, phases and indices are loaded during this
    // group's sums
    float tc[Q];
#pragma unroll
    for (int r = 0; r < Q; r++)
      tc[r] = tab[r];
    const cplx<float> pc = ph;
    if (g0 + 64 < e)
      fetch(g0 + 64);
    mfma_group<Q>(tc, x, pc, ar, ai);
  }
  // add the four wavefronts' sums: 3, 2 and 1 onto 0, in turn
  auto put = [&](float *dst) {
#pragma unroll
    for (int q = 0; q < Q; q++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        dst[((4 * q + v) * 2) * 64 + lane] = ar[q][v];
        dst[((4 * q + v) * 2 + 1) * 64 + lane] = ai[q][v];
      }
  };
  auto add = [&](const float *src) {
#pragma unroll
    for (int q = 0; q < Q; q++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        ar[q][v] += src[((4 * q + v) * 2) * 64 + lane];
        ai[q][v] += src[((4 * q + v) * 2 + 1) * 64 + lane];
      }
  };
  for (int w = 3; w > 0; w--) {
    if (wave == w)
      put(red);
    __syncthreads();
    if (wave == 0)
      add(red);
    __syncthreads();
  }
  if (wave == 0 && lane < NB) {
#pragma unroll
    for (int q = 0; q < Q; q++)
#pragma unroll
      for (int v = 0; v < 4; v++)
        partial[(long)(4 * q + v) * NB + lane] = mk<float>(ar[q][v], ai[q][v]);
  }
}

// One work-group per (site, part of its points).  PM: the widest table row
// of the plan; a site's own row width picks the body (uniform over the
// work-group), so a plan that mixes species sums each at its own width.
template <typename T, int PM, int U>
__device__ __forceinline__ void sphere_sum_block(const cplx<T> *__restrict__ g, int NB,
                                                 const int *__restrict__ site_pt, const int *__restrict__ site_np,
                                                 const long *__restrict__ tab_off, const int *__restrict__ pidx,
                                                 const cplx<T> *__restrict__ phase, const T *__restrict__ table,
                                                 int nparts, cplx<T> *__restrict__ partial, int streaming, int blk) {
  const int s = blk / nparts, part = blk % nparts;
  const int p0 = site_pt[s], p1 = site_pt[s + 1];
  const int len = p1 - p0;
  const int chunk = (len + nparts - 1) / nparts;
  const int a = p0 + part * chunk;
  const int e = min(p1, a + chunk);
  const T *tsite = table + tab_off[s];
  const int ts = table_stride(site_np[s], sizeof(T) == 4);
  cplx<T> *o = partial + (long)blk * PM * NB;
  if constexpr (sizeof(T) == 4) {
    __shared__ float red[PM * 2 * 64];
#define PP_BODY(C)                                                                               \
  if constexpr (C <= PM) {                                                                       \
    if (ts == C) {                                                                               \
      sphere_sum_mfma<C / 4>(g, NB, p0, len, pidx, phase, tsite, a, e, o, streaming, red);       \
      return;                                                                                    \
    }                                                                                            \
  }
    PP_STRIDES_F32(PP_BODY)
#undef PP_BODY
  } else {
    // Rows of 64 in two halves, which read the grid twice: the sums of 64
    // slots take 512 registers a lane and spilled (64 sites of 845 points, 64
    // bands, 64 projectors: setup of 768 us, in halves 503).
    constexpr int PH = PM > 48 ? 48 : PM;
    __shared__ __align__(16) T s_tab[64 * (PH + 1)];
    __shared__ cplx<T> s_ph[64];
    __shared__ int s_idx[64];
#define PP_BODY(C)                                                                                                   \
  if constexpr (C <= PM) {                                                                                           \
    if (ts == C) {                                                                                                   \
      if constexpr (C > 48) {                                                                                        \
        for (int s0 = 0; s0 < C; s0 += C / 2)                                                                        \
          sphere_sum_valu<T, C / 2, U, C>(g, NB, p0, len, pidx, phase, tsite, a, e, o, streaming, s_tab, s_ph, s_idx, s0); \
      } else {                                                                                                       \
        sphere_sum_valu<T, C, U>(g, NB, p0, len, pidx, phase, tsite, a, e, o, streaming, s_tab, s_ph, s_idx);        \
      }                                                                                                              \
      return;                                                                                                        \
    }                                                                                                                \
  }
    PP_STRIDES_F64(PP_BODY)
#undef PP_BODY
  }
}
template <typename T, int PM, int U>
__global__ __launch_bounds__(256) void k_sphere_sum(const cplx<T> *__restrict__ g, int NB,
                                                    const int *__restrict__ site_pt, const int *__restrict__ site_np,
                                                    const long *__restrict__ tab_off, const int *__restrict__ pidx,
                                                    const cplx<T> *__restrict__ phase, const T *__restrict__ table,
                                                    int nparts, cplx<T> *__restrict__ partial, int streaming) {
  sphere_sum_block<T, PM, U>(g, NB, site_pt, site_np, tab_off, pidx, phase, table, nparts, partial, streaming,
                             blockIdx.x);
}
// The sphere sums of a batch of work items (one per blockIdx.y), each with
// its own chunk, plan and phases.
template <typename T, int PM, int U>
__global__ __launch_bounds__(256) void k_sphere_sum_items(const ChunkItem *__restrict__ items, int NB, int streaming) {
  const ChunkItem &it = items[blockIdx.y];
  const int blk = blockIdx.x;
  if (blk >= it.nsites * it.nparts)
    return;
  sphere_sum_block<T, PM, U>((const cplx<T> *)it.grid, NB, (const int *)it.site_pt, (const int *)it.site_np,
                             (const long *)it.tab_off, (const int *)it.pidx, (const cplx<T> *)it.phase,
                             (const T *)it.table, it.nparts, (cplx<T> *)it.partial, streaming, blk);
}

// Sum the parts of every (site, slot, band) in FP64 and form the complex
// projections from the real-harmonic sums.  One work-group per site and 16
// bands: the part sums are read with the bands on consecutive lanes (as
// the sum kernels wrote them) into an LDS tile, and the projections written
// with the slots on consecutive lanes (as the output rows hold them), so
// both sides move whole lines.
constexpr int RED_NB = 16;
template <typename T>
__device__ __forceinline__ void sphere_reduce_block(const cplx<T> *__restrict__ partial, int NB, int nbc, int PM,
                                                    int nparts, int nsites, const int *__restrict__ site_np,
                                                    const int *__restrict__ proj_off, const int *__restrict__ proj_m,
                                                    long ptot, cplx<double> *__restrict__ out, int blk) {
  __shared__ cplx<double> tile[64][RED_NB + 1];
  const int ng = (nbc + RED_NB - 1) / RED_NB;
  const int s = blk / ng, b0 = (blk % ng) * RED_NB;
  if (s >= nsites)
    return;
  const int np = site_np[s], po = proj_off[s];
  const int bl = threadIdx.x % RED_NB, j0 = threadIdx.x / RED_NB;
  if (b0 + bl < nbc)
    for (int j = j0; j < np; j += 256 / RED_NB) {
      cplx<double> c = mk<double>(0, 0);
      const cplx<T> *ps = partial + ((long)s * nparts * PM + j) * NB + b0 + bl;
#pragma unroll 4
      for (int q = 0; q < nparts; q++)
        c = c + cvt<double>(ps[(long)q * PM * NB]);
      tile[j][bl] = c;
    }
  __syncthreads();
  for (int t = threadIdx.x; t < np * RED_NB; t += 256) {
    const int b = t / np, j = t - b * np;
    if (b0 + b >= nbc)
      break;
    const int m = proj_m[po + j];
    const cplx<double> own = tile[j][b];
    cplx<double> r = own;
    if (m > 0) {  // s_(l,m) - i s_(l,-m)
      const cplx<double> sn = tile[j - 2 * m][b];
      r = mk<double>(own.x + sn.y, own.y - sn.x);
    } else if (m < 0) {  // (-1)^m (s_(l,m) + i s_(l,-m))
      const cplx<double> c = tile[j - 2 * m][b];
      const double sg = (m & 1) ? -1.0 : 1.0;
      r = mk<double>(sg * (c.x - own.y), sg * (c.y + own.x));
    }
    out[(long)(b0 + b) * ptot + po + j] = r;
  }
}
template <typename T>
__global__ __launch_bounds__(256) void k_sphere_reduce(const cplx<T> *__restrict__ partial, int NB, int nbc, int PM,
                                                       int nparts, int nsites, const int *__restrict__ site_np,
                                                       const int *__restrict__ proj_off,
                                                       const int *__restrict__ proj_m, long ptot,
                                                       cplx<double> *__restrict__ out) {
  sphere_reduce_block<T>(partial, NB, nbc, PM, nparts, nsites, site_np, proj_off, proj_m, ptot, out, blockIdx.x);
}
template <typename T>
__global__ __launch_bounds__(256) void k_sphere_reduce_items(const ChunkItem *__restrict__ items, int NB, int PM) {
  const ChunkItem &it = items[blockIdx.y];
  sphere_reduce_block<T>((const cplx<T> *)it.partial, NB, it.nbc, PM, it.nparts, it.nsites, (const int *)it.site_np,
                         (const int *)it.proj_off, (const int *)it.proj_m, it.ptot, (cplx<double> *)it.out,
                         blockIdx.x);
}

// Coefficients of the real-harmonic table slots for the expansion
// sum_j P_j p_j(r) (projector.c:324-327): with p_(l,+-m) built from the real
// slots t_(l,m) = A cos m phi, t_(l,-m) = A sin m phi (m > 0),
//   sum_m P_m Y_lm = sum_{m>0} t_(l,m) (P_m + (-1)^m P_-m)
//                 + i t_(l,-m) (P_m - (-1)^m P_-m) + t_(l,0) P_0.
// Q[(s * PMAX + j) * NB + b] for band b of the chunk; P rows of stride
// ptotP, site s of the plan at src_off[s].
template <typename T>
__global__ __launch_bounds__(256) void k_expand_coef(int nsites, int PMAX, int NB, int nbc,
                                                     const int *__restrict__ site_np, const int *__restrict__ proj_off,
                                                     const int *__restrict__ proj_m, const int *__restrict__ src_off,
                                                     const cplx<double> *__restrict__ P, long ptotP,
                                                     cplx<T> *__restrict__ Q) {
  long t = (long)blockIdx.x * 256 + threadIdx.x;
  if (t >= (long)nsites * PMAX * NB)
    return;
  const int b = (int)(t % NB);
  const long r = t / NB;
  const int j = (int)(r % PMAX), s = (int)(r / PMAX);
  cplx<double> q = mk<double>(0, 0);
  if (j < site_np[s] && b < nbc) {
    const int m = proj_m[proj_off[s] + j];
    const cplx<double> *row = P + (long)b * ptotP + src_off[s];
    if (m == 0) {
      q = row[j];
    } else {
      const int am = m < 0 ? -m : m;
      const int jp = m > 0 ? j : j + 2 * am, jn = jp - 2 * am;  // slots of +am and -am
      const double sg = (am & 1) ? -1.0 : 1.0;
      const cplx<double> a = row[jp], c = row[jn];
      if (m > 0)
        q = mk<double>(a.x + sg * c.x, a.y + sg * c.y);
      else  // i (P_m - (-1)^m P_-m)
        q = mk<double>(-(a.y - sg * c.y), a.x - sg * c.x);
    }
  }
  Q[t] = cvt<T>(q);
}

// grid[idx][b] += conj(e^{-i k.path} sum_j Q_j t_j) for every sphere point
// (conjugated so the backward passes give the forward transform).  Lane =
// band; spheres of different sites may share points, so the adds are
// atomic (vector global float/double atomics).
template <typename T, int PMAX>
__global__ __launch_bounds__(256) void k_sphere_expand(cplx<T> *__restrict__ g, int NB, int nbc,
                                                       const int *__restrict__ site_pt, const int *__restrict__ site_np,
                                                       const long *__restrict__ tab_off, const int *__restrict__ pidx,
                                                       const cplx<T> *__restrict__ phase, const T *__restrict__ table,
                                                       const cplx<T> *__restrict__ Q, int nparts) {
  const int s = blockIdx.x / nparts, part = blockIdx.x % nparts;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int p0 = site_pt[s], len = site_pt[s + 1] - p0;
  const int np = site_np[s], ts = table_stride(np, sizeof(T) == 4);
  const int chunk = (len + nparts - 1) / nparts;
  const int a = p0 + part * chunk, e = min(p0 + len, a + chunk);
  if (lane >= nbc)
    return;
  cplx<T> q[PMAX];
#pragma unroll
  for (int j = 0; j < PMAX; j++)
    q[j] = j < np ? Q[((long)s * PMAX + j) * NB + lane] : mk<T>(0, 0);
  const T *tsite = table + tab_off[s];
  for (int i = a + wave; i < e; i += 4) {
    const T *tp = tsite + (long)(i - p0) * ts;
    cplx<T> v = mk<T>(0, 0);
#pragma unroll
    for (int j = 0; j < PMAX; j++)
      if (j < np) {
        v.x += q[j].x * tp[j];
        v.y += q[j].y * tp[j];
      }
    const cplx<T> x = v * phase[i];
    T *dst = reinterpret_cast<T *>(g + (long)pidx[i] * NB + lane);
    atomicAdd(dst, x.x);
    atomicAdd(dst + 1, -x.y);
  }
}

// ------------------------------------------------------------------ host
static void cross(const double *a, const double *b, double *o) {
  o[0] = a[1] * b[2] - a[2] * b[1];
  o[1] = a[2] * b[0] - a[0] * b[2];
  o[2] = a[0] * b[1] - a[1] * b[0];
}
static double nrm(const double *v) { return sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]); }
double det3(const double *m) {
  return m[0] * m[4] * m[8] + m[1] * m[5] * m[6] + m[2] * m[3] * m[7] - m[2] * m[4] * m[6] -
         m[1] * m[3] * m[8] - m[0] * m[5] * m[7];
}

// Host spline coefficients with the reference's boundary conditions
// (utils.c:699-749): y'(x0) = secant slope, natural end.
void spline_coeff_host(const double *x, const double *y, int n, double *b, double *c, double *d) {
  std::vector<double> diag(n), up(n), rhs(n), M(n);
  double h0 = x[1] - x[0];
  diag[0] = 2.0 * h0;
  up[0] = h0;
  rhs[0] = 0.0;  // 6((y1-y0)/h0 - slope0) with slope0 the secant slope
  for (int i = 1; i < n - 1; i++) {
    double hl = x[i] - x[i - 1], hr = x[i + 1] - x[i];
    double w = hl / diag[i - 1];
    diag[i] = 2.0 * (hl + hr) - w * up[i - 1];
    up[i] = hr;
    rhs[i] = 6.0 * ((y[i + 1] - y[i]) / hr - (y[i] - y[i - 1]) / hl) - w * rhs[i - 1];
  }
  M[n - 1] = 0.0;
  for (int i = n - 2; i >= 0; i--)
    M[i] = (rhs[i] - up[i] * M[i + 1]) / diag[i];
  for (int i = 0; i < n - 1; i++) {
    double h = x[i + 1] - x[i];
    b[i] = (y[i + 1] - y[i]) / h - h * (2.0 * M[i] + M[i + 1]) / 6.0;
    c[i] = 0.5 * M[i];
    d[i] = (M[i + 1] - M[i]) / (6.0 * h);
  }
  b[n - 1] = c[n - 1] = d[n - 1] = 0.0;
}

// line-block work lists of the fused x pass (pp_fused.hip)
int fused_plan(pp_sphere *sp, const std::vector<SiteGeo> &geo);

// Sphere radius and candidate box of a site with coord set:
// R0 = (n-1)/n rmax (utils.c:651-652, the site's own species), box
// half-widths g_i = int(|a_j x a_k| rmax / V * N_i) + 1 around
// round(frac * N).
void site_box(const double *lattice, const int *fftg, double rmax, int ngrid, SiteGeo &g) {
  const double vol = det3(lattice);
  g.rmax = rmax;
  g.ngrid = ngrid;
  g.R0 = (ngrid - 1) * rmax / ngrid;
  double cr[3];
  cross(lattice + 3, lattice + 6, cr);
  g.g[0] = (int)(nrm(cr) * rmax / vol * fftg[0]) + 1;
  cross(lattice + 0, lattice + 6, cr);
  g.g[1] = (int)(nrm(cr) * rmax / vol * fftg[1]) + 1;
  cross(lattice + 0, lattice + 3, cr);
  g.g[2] = (int)(nrm(cr) * rmax / vol * fftg[2]) + 1;
  for (int a = 0; a < 3; a++)
    g.c[a] = (int)round(g.coord[a] * fftg[a]);
}

static int sphere_build(pp_sphere *sp) {
  pp_ctx *ctx = sp->ctx;
  sp->gen++;
  const int ns = sp->nsites;
  // per-site geometry
  std::vector<SiteGeo> geo(ns);
  std::vector<long> spl_off(sp->nelems);
  long so = 0;
  for (int e = 0; e < sp->nelems; e++) {
    spl_off[e] = so;
    so += (long)(1 + 4 * sp->nchan[e]) * sp->ngrid[e];
  }
  sp->nproj_site.assign(ns, 0);
  sp->proj_off.assign(ns + 1, 0);
  sp->pmax = 0;
  for (int s = 0; s < ns; s++) {
    SiteGeo &g = geo[s];
    int e = sp->labels[s];
    for (int a = 0; a < 3; a++)
      g.coord[a] = sp->frac[3 * s + a];
    site_box(sp->lattice, sp->fftg, sp->rmax[e], sp->ngrid[e], g);
    g.elem = e;
    g.nchan = sp->nchan[e];
    int np = 0;
    for (int ch = 0; ch < g.nchan; ch++)
      np += 2 * sp->ls[sp->ls_off[e] + ch] + 1;
    g.nproj = np;
    g.spl_off = spl_off[e];
    g.chan_off = sp->ls_off[e];
    sp->nproj_site[s] = np;
    sp->proj_off[s + 1] = sp->proj_off[s] + np;
    if (np > sp->pmax)
      sp->pmax = np;
  }
  sp->ptot = sp->proj_off[ns];
  PP_REQUIRE(sp->pmax <= 64, PP_ERR_UNSUPPORTED, "more than 64 projectors on one site");
  std::vector<int> proj_m(std::max(1, sp->ptot));
  for (int s = 0, q = 0; s < ns; s++) {
    int e = sp->labels[s];
    for (int ch = 0; ch < sp->nchan[e]; ch++) {
      int l = sp->ls[sp->ls_off[e] + ch];
      for (int m = -l; m <= l; m++)
        proj_m[q++] = m;
    }
  }
  PP_TRY(sp->d_proj_m.ensure(sizeof(int) * proj_m.size()));
  PP_CHECK_HIP(hipMemcpyAsync(sp->d_proj_m.p, proj_m.data(), sizeof(int) * proj_m.size(), hipMemcpyHostToDevice,
                              ctx->stream));
  Lat9 L;
  memcpy(L.m, sp->lattice, sizeof(L.m));
  PP_TRY(sp->d_sitemeta.ensure(sizeof(SiteGeo) * ns));
  PP_CHECK_HIP(hipMemcpyAsync(sp->d_sitemeta.p, geo.data(), sizeof(SiteGeo) * ns, hipMemcpyHostToDevice, ctx->stream));
  PP_TRY(sp->d_counts.ensure(sizeof(int) * 2 * ns));
  hipEvent_t ev;
  tbegin(ctx, K_TABLE, &ev);
  hipLaunchKernelGGL(k_site_count, dim3(ns), dim3(64 * SITE_W), 0, ctx->stream, (const SiteGeo *)sp->d_sitemeta.p, L,
                     sp->fftg[0], sp->fftg[1], sp->fftg[2], ns, (int *)sp->d_counts.p);
  tend(ctx, K_TABLE, ev);
  PP_CHECK_HIP(hipGetLastError());
  std::vector<int> counts(2 * ns);
  PP_CHECK_HIP(
      hipMemcpyAsync(counts.data(), sp->d_counts.p, sizeof(int) * 2 * ns, hipMemcpyDeviceToHost, ctx->stream));
  PP_CHECK_HIP(hipStreamSynchronize(ctx->stream));
  sp->site_pt_h.assign(ns + 1, 0);
  sp->seg_off_h.assign(ns + 1, 0);
  std::vector<long> tab_off(ns);
  long to = 0;
  int maxcount = 0;
  for (int s = 0; s < ns; s++) {
    sp->site_pt_h[s + 1] = sp->site_pt_h[s] + counts[s];
    sp->seg_off_h[s + 1] = sp->seg_off_h[s] + counts[ns + s];
    tab_off[s] = to;
    to += (long)(counts[s] + (sp->precision != PP_FP64 ? TAB_PAD : 0)) *
          table_stride(sp->nproj_site[s], sp->precision != PP_FP64);
    if (counts[s] > maxcount)
      maxcount = counts[s];
  }
  sp->npts = sp->site_pt_h[ns];
  sp->nseg = sp->seg_off_h[ns];
  size_t csz = sp->precision == PP_FP64 ? sizeof(double) : sizeof(float);
  PP_TRY(sp->d_site_pt.ensure(sizeof(int) * (ns + 1)));
  PP_TRY(sp->d_site_np.ensure(sizeof(int) * ns));
  PP_TRY(sp->d_tab_off.ensure(sizeof(long) * ns));
  PP_TRY(sp->d_proj_off.ensure(sizeof(int) * (ns + 1)));
  PP_TRY(sp->d_pidx.ensure(sizeof(int) * std::max<long>(1, sp->npts)));
  PP_TRY(sp->d_path.ensure(sizeof(double) * 3 * std::max<long>(1, sp->npts)));
  PP_TRY(sp->d_table.ensure(csz * std::max<long>(1, to)));
  PP_TRY(sp->d_seg_off.ensure(sizeof(int) * (ns + 1)));
  PP_TRY(sp->d_seg.ensure(sizeof(int4) * std::max<long>(1, sp->nseg)));
  PP_TRY(sp->d_segline.ensure(sizeof(int) * std::max<long>(1, sp->nseg)));
  PP_CHECK_HIP(hipMemcpyAsync(sp->d_seg_off.p, sp->seg_off_h.data(), sizeof(int) * (ns + 1), hipMemcpyHostToDevice,
                              ctx->stream));
  PP_CHECK_HIP(hipMemcpyAsync(sp->d_site_pt.p, sp->site_pt_h.data(), sizeof(int) * (ns + 1), hipMemcpyHostToDevice,
                              ctx->stream));
  PP_CHECK_HIP(hipMemcpyAsync(sp->d_site_np.p, sp->nproj_site.data(), sizeof(int) * ns, hipMemcpyHostToDevice,
                              ctx->stream));
  PP_CHECK_HIP(hipMemcpyAsync(sp->d_tab_off.p, tab_off.data(), sizeof(long) * ns, hipMemcpyHostToDevice, ctx->stream));
  PP_CHECK_HIP(hipMemcpyAsync(sp->d_proj_off.p, sp->proj_off.data(), sizeof(int) * (ns + 1), hipMemcpyHostToDevice,
                              ctx->stream));
  tbegin(ctx, K_TABLE, &ev);
  hipLaunchKernelGGL(k_site_fill, dim3(ns), dim3(64 * SITE_W), 0, ctx->stream, (const SiteGeo *)sp->d_sitemeta.p, L,
                     sp->fftg[0], sp->fftg[1], sp->fftg[2], (const int *)sp->d_site_pt.p,
                     (const int *)sp->d_seg_off.p, (int *)sp->d_pidx.p, (double *)sp->d_path.p, (int4 *)sp->d_seg.p,
                     (int *)sp->d_segline.p);
  if (sp->nseg > 0)
    hipLaunchKernelGGL(k_seg_len, dim3((unsigned)((sp->nseg + 255) / 256)), dim3(256), 0, ctx->stream,
                       (int4 *)sp->d_seg.p, sp->nseg, (const int *)sp->d_seg_off.p, (const int *)sp->d_site_pt.p);
  tend(ctx, K_TABLE, ev);
  PP_CHECK_HIP(hipGetLastError());
  // x-line coverage masks (the x pass writes only covered points)
  sp->xmask_words = (sp->fftg[0] + 31) / 32;
  const size_t mbytes = sizeof(unsigned) * (size_t)sp->fftg[1] * sp->fftg[2] * sp->xmask_words;
  PP_TRY(sp->d_xmask.ensure(mbytes));
  PP_TRY(zero_async(ctx, sp->d_xmask.p, mbytes));
  if (sp->nseg > 0) {
    hipLaunchKernelGGL(k_xmask, dim3((unsigned)((sp->nseg + 255) / 256)), dim3(256), 0, ctx->stream,
                       (const int4 *)sp->d_seg.p, (const int *)sp->d_segline.p, sp->nseg, sp->fftg[0],
                       sp->xmask_words, (unsigned *)sp->d_xmask.p);
    PP_CHECK_HIP(hipGetLastError());
  }
  if (maxcount > 0) {
    dim3 grd((maxcount + TAB_PAD + 255) / 256, ns);
    tbegin(ctx, K_TABLE, &ev);
    if (sp->precision == PP_FP64)
      hipLaunchKernelGGL(k_site_values<double>, grd, dim3(256), 0, ctx->stream, (const SiteGeo *)sp->d_sitemeta.p,
                         L, sp->fftg[0], sp->fftg[1], sp->fftg[2], (const int *)sp->d_site_pt.p,
                         (const long *)sp->d_tab_off.p, (const int *)sp->d_pidx.p, (const double *)sp->d_spline.p,
                         (const int *)sp->d_chan.p, (double *)sp->d_table.p);
    else
      hipLaunchKernelGGL(k_site_values<float>, grd, dim3(256), 0, ctx->stream, (const SiteGeo *)sp->d_sitemeta.p, L,
                         sp->fftg[0], sp->fftg[1], sp->fftg[2], (const int *)sp->d_site_pt.p,
                         (const long *)sp->d_tab_off.p, (const int *)sp->d_pidx.p, (const double *)sp->d_spline.p,
                         (const int *)sp->d_chan.p, (float *)sp->d_table.p);
    tend(ctx, K_TABLE, ev);
    PP_CHECK_HIP(hipGetLastError());
  }
  // the fused x pass's work lists are built when that path is first used
  sp->geo_h = geo;
  sp->fx_built = false;
  sp->fused_ok = false;
  return ctx->tune_fused ? fused_plan(sp, geo) : PP_OK;
}

// Sum kernel of a plan whose widest table row is PM (one of the strides of
// table_stride); the FP32 form has no unroll variants.
template <typename T, int PM>
static void launch_sum(pp_ctx *ctx, pp_sphere *sp, const cplx<T> *grid, int NB, const cplx<T> *phase, int nparts,
                       cplx<T> *partial) {
#define PP_SS(U)                                                                                                    \
  hipLaunchKernelGGL((k_sphere_sum<T, PM, U>), dim3(sp->nsites * nparts), dim3(256), 0, ctx->stream, grid, NB,     \
                     (const int *)sp->d_site_pt.p, (const int *)sp->d_site_np.p, (const long *)sp->d_tab_off.p,    \
                     (const int *)sp->d_pidx.p, phase, (const T *)sp->d_table.p, nparts, partial, ctx->tune_sphere_nt)
  if (sizeof(T) == 4 || ctx->tune_sphere_unroll == 8)
    PP_SS(8);
  else
    PP_SS(4);
#undef PP_SS
}

int sphere_parts_of(pp_ctx *ctx, pp_sphere *sp);
int sphere_pm_of(pp_sphere *sp);

template <typename T>
int sphere_sums(pp_ctx *ctx, pp_sphere *sp, const cplx<T> *grid, int NB, int nbc, const cplx<T> *phase,
                cplx<double> *out, long ptot) {
  if (sp->nsites == 0 || nbc == 0)
    return PP_OK;
  const int nparts = sphere_parts_of(ctx, sp);
  const int PM = sphere_pm_of(sp);
  DevBuf &pbuf = ctx->slot ? ctx->partial2 : ctx->partial;
  PP_TRY(pbuf.ensure(sizeof(cplx<T>) * (size_t)sp->nsites * nparts * NB * PM));
  cplx<T> *partial = (cplx<T> *)pbuf.p;
  hipEvent_t ev;
  tbegin(ctx, K_SPHERE_SUM, &ev);
#define PP_SUM(P)                                                     \
  case P:                                                             \
    launch_sum<T, P>(ctx, sp, grid, NB, phase, nparts, partial);      \
    break;
  if constexpr (sizeof(T) == 4) {
    switch (PM) { PP_STRIDES_F32(PP_SUM) }
  } else {
    switch (PM) { PP_STRIDES_F64(PP_SUM) }
  }
#undef PP_SUM
  tend(ctx, K_SPHERE_SUM, ev);
  PP_CHECK_HIP(hipGetLastError());
  const long nblk = (long)sp->nsites * ((nbc + RED_NB - 1) / RED_NB);
  tbegin(ctx, K_SPHERE_REDUCE, &ev);
  hipLaunchKernelGGL(k_sphere_reduce<T>, dim3((unsigned)nblk), dim3(256), 0, ctx->stream, partial, NB, nbc, PM, nparts,
                     sp->nsites, (const int *)sp->d_site_np.p, (const int *)sp->d_proj_off.p,
                     (const int *)sp->d_proj_m.p, ptot, out);
  tend(ctx, K_SPHERE_REDUCE, ev);
  PP_CHECK_HIP(hipGetLastError());
  return PP_OK;
}

// Sphere-sum parts per site of a plan: the tuning value, else enough for
// about 2048 work-groups (eight per CU), of at least 64 points each (one
// group of 16 per wavefront): a cell of 8 sites of 270 points runs 32
// work-groups of one group per wavefront instead of 8 of four.  FP32 rows of
// up to 32 take nine per CU: the matrix cores' sums are a little further from the FP64 ones
// than fused multiply-adds were, and the parts are added in FP64 (215 sites of
// 4,853 points, error of the projections with VALU sums in 10 parts 1.110e-7,
// on the matrix cores in 10 / 11 / 14 parts 1.131e-7 / 1.105e-7 / 1.058e-7,
// sums and reduction of a chunk 151 / 150 / 149 us, of eight chunks in one
// launch 7.71 / 7.75 / 8.02 ms; 512 sites of 11,499 in 4 and 5 parts 2.10e-7
// and 1.84e-7, 733 and 736 us).  Wider rows write as much in partial sums as
// they gather (64 sites, 64 projectors: setup 275 us, with nine 287).
int sphere_parts_of(pp_ctx *ctx, pp_sphere *sp) {
  if (ctx->tune_sphere_parts > 0)
    return ctx->tune_sphere_parts;
  const int ns = std::max(1, sp->nsites);
  const long most = std::max<long>(1, sp->npts / ns / 64);
  const int wgs = sp->precision == PP_FP64 || sp->pmax > 32 ? 2048 : 2304;
  return (int)std::min<long>((wgs + ns - 1) / ns, most);
}
// Widest table row of a plan: the sum kernel that serves it.
int sphere_pm_of(pp_sphere *sp) { return table_stride(sp->pmax, sp->precision != PP_FP64); }
// The plan's part of a work item.
void sphere_item_fields(pp_ctx *ctx, pp_sphere *sp, ChunkItem &it) {
  it.site_pt = (const PP_G int *)sp->d_site_pt.p;
  it.site_np = (const PP_G int *)sp->d_site_np.p;
  it.proj_off = (const PP_G int *)sp->d_proj_off.p;
  it.proj_m = (const PP_G int *)sp->d_proj_m.p;
  it.pidx = (const PP_G int *)sp->d_pidx.p;
  it.tab_off = (const PP_G long *)sp->d_tab_off.p;
  it.table = (const PP_G void *)sp->d_table.p;
  it.nsites = sp->nsites;
  it.nparts = sphere_parts_of(ctx, sp);
}

// Sphere sums and their reduction for a batch of work items: one launch
// each.  PM: the largest sphere_pm_of of the items' plans; maxblk and
// maxred bound the work-groups of the sums (nsites * nparts) and of the
// reduction (nsites * band groups of RED_NB) over the items.
template <typename T>
int sphere_sums_items(pp_ctx *ctx, const ChunkItem *items, int nitems, int NB, int PM, long maxblk, long maxred) {
  if (nitems == 0 || maxblk == 0)
    return PP_OK;
  hipEvent_t ev;
  tbegin(ctx, K_SPHERE_SUM, &ev);
  dim3 grd((unsigned)maxblk, (unsigned)nitems);
  const bool u8 = sizeof(T) == 4 || ctx->tune_sphere_unroll == 8;
#define PP_SI(P)                                                                                                   \
  case P:                                                                                                          \
    if (u8)                                                                                                        \
      hipLaunchKernelGGL((k_sphere_sum_items<T, P, 8>), grd, dim3(256), 0, ctx->stream, items, NB,                 \
                         ctx->tune_sphere_nt);                                                                     \
    else                                                                                                           \
      hipLaunchKernelGGL((k_sphere_sum_items<T, P, 4>), grd, dim3(256), 0, ctx->stream, items, NB,                 \
                         ctx->tune_sphere_nt);                                                                     \
    break;
  if constexpr (sizeof(T) == 4) {
    switch (PM) { PP_STRIDES_F32(PP_SI) }
  } else {
    switch (PM) { PP_STRIDES_F64(PP_SI) }
  }
#undef PP_SI
  tend(ctx, K_SPHERE_SUM, ev);
  PP_CHECK_HIP(hipGetLastError());
  tbegin(ctx, K_SPHERE_REDUCE, &ev);
  hipLaunchKernelGGL(k_sphere_reduce_items<T>, dim3((unsigned)maxred, (unsigned)nitems), dim3(256), 0, ctx->stream,
                     items, NB, PM);
  tend(ctx, K_SPHERE_REDUCE, ev);
  PP_CHECK_HIP(hipGetLastError());
  return PP_OK;
}
template int sphere_sums_items<double>(pp_ctx *, const ChunkItem *, int, int, int, long, long);
template int sphere_sums_items<float>(pp_ctx *, const ChunkItem *, int, int, int, long, long);
// Reduction work-groups of an item.
long sphere_reduce_blocks(int nsites, int nbc) { return (long)nsites * ((nbc + RED_NB - 1) / RED_NB); }

// phase[pt] = dv / sqrt(V) e^{i k.path} (sphere sums) or, with expand,
// e^{-i k.path} (the augmentation functions of projector.c:276-330)
template <typename T>
int make_phase(pp_ctx *ctx, pp_sphere *sp, const double *kfrac, cplx<T> *phase, bool expand) {
  if (sp->npts == 0)
    return PP_OK;
  // reciprocal lattice with 2 pi, rows b_i (utils.h:131)
  double rec[9], v = det3(sp->lattice);
  cross(sp->lattice + 3, sp->lattice + 6, rec + 0);
  cross(sp->lattice + 6, sp->lattice + 0, rec + 3);
  cross(sp->lattice + 0, sp->lattice + 3, rec + 6);
  for (int i = 0; i < 9; i++)
    rec[i] *= 2.0 * M_PI / v;
  double kc[3];
  for (int j = 0; j < 3; j++)
    kc[j] = kfrac[0] * rec[j] + kfrac[1] * rec[3 + j] + kfrac[2] * rec[6 + j];
  double dv = v / sp->fftg[0] / sp->fftg[1] / sp->fftg[2];
  double scl = dv / sqrt(v);
  if (expand) {
    scl = 1.0;
    for (int j = 0; j < 3; j++)
      kc[j] = -kc[j];
  }
  hipEvent_t ev;
  tbegin(ctx, K_PHASE, &ev);
  hipLaunchKernelGGL(k_phase<T>, dim3((unsigned)((sp->npts + 255) / 256)), dim3(256), 0, ctx->stream, sp->npts,
                     (const double *)sp->d_path.p, kc[0], kc[1], kc[2], scl, phase);
  tend(ctx, K_PHASE, ev);
  PP_CHECK_HIP(hipGetLastError());
  return PP_OK;
}

template int sphere_sums<double>(pp_ctx *, pp_sphere *, const cplx<double> *, int, int, const cplx<double> *,
                                 cplx<double> *, long);
template int sphere_sums<float>(pp_ctx *, pp_sphere *, const cplx<float> *, int, int, const cplx<float> *,
                                cplx<double> *, long);
template int make_phase<double>(pp_ctx *, pp_sphere *, const double *, cplx<double> *, bool);
template int make_phase<float>(pp_ctx *, pp_sphere *, const double *, cplx<float> *, bool);

// Accumulate conj of the augmentation functions of the plan's sites for
// a band chunk into grid (zeroed by the caller); P rows [nbc][ptotP] with
// plan site s at src_off_dev[s]; phase from make_phase(expand = true).
template <typename T>
int sphere_expand(pp_ctx *ctx, pp_sphere *sp, cplx<T> *grid, int NB, int nbc, const cplx<T> *phase,
                  const cplx<double> *P, long ptotP, const int *src_off_dev) {
  if (sp->nsites == 0 || nbc == 0)
    return PP_OK;
  const int PM = sp->pmax <= 8 ? 8 : sp->pmax <= 18 ? 18 : sp->pmax <= 32 ? 32 : 64;
  DevBuf &qb = ctx->slot ? ctx->partial2 : ctx->partial;
  const long nq = (long)sp->nsites * PM * NB;
  PP_TRY(qb.ensure(sizeof(cplx<T>) * (size_t)nq));
  cplx<T> *Q = (cplx<T> *)qb.p;
  hipEvent_t ev;
  tbegin(ctx, K_AUG_PREP, &ev);
  hipLaunchKernelGGL(k_expand_coef<T>, dim3((unsigned)((nq + 255) / 256)), dim3(256), 0, ctx->stream, sp->nsites, PM,
                     NB, nbc, (const int *)sp->d_site_np.p, (const int *)sp->d_proj_off.p, (const int *)sp->d_proj_m.p,
                     src_off_dev, P, ptotP, Q);
  tend(ctx, K_AUG_PREP, ev);
  PP_CHECK_HIP(hipGetLastError());
  long avg = sp->npts / std::max(1, sp->nsites);
  int nparts = (int)std::max<long>(1, std::min<long>((2048 + sp->nsites - 1) / sp->nsites, avg / 64));
  tbegin(ctx, K_SPHERE_SUM, &ev);
#define PP_EX(PMX)                                                                                                  \
  hipLaunchKernelGGL((k_sphere_expand<T, PMX>), dim3((unsigned)(sp->nsites * nparts)), dim3(256), 0, ctx->stream,  \
                     grid, NB, nbc, (const int *)sp->d_site_pt.p, (const int *)sp->d_site_np.p,                   \
                     (const long *)sp->d_tab_off.p, (const int *)sp->d_pidx.p, phase, (const T *)sp->d_table.p, Q, \
                     nparts)
  if (PM == 8)
    PP_EX(8);
  else if (PM == 18)
    PP_EX(18);
  else if (PM == 32)
    PP_EX(32);
  else
    PP_EX(64);
#undef PP_EX
  tend(ctx, K_SPHERE_SUM, ev);
  PP_CHECK_HIP(hipGetLastError());
  return PP_OK;
}

template int sphere_expand<double>(pp_ctx *, pp_sphere *, cplx<double> *, int, int, const cplx<double> *,
                                   const cplx<double> *, long, const int *);
template int sphere_expand<float>(pp_ctx *, pp_sphere *, cplx<float> *, int, int, const cplx<float> *,
                                  const cplx<double> *, long, const int *);
int sphere_nsites(pp_sphere *sp) { return sp->nsites; }
long sphere_generation(pp_sphere *sp) { return sp->gen; }
const unsigned *sphere_xmask(pp_sphere *sp, int *words) {
  *words = sp->xmask_words;
  return (const unsigned *)sp->d_xmask.p;
}

long sphere_npts(pp_sphere *sp) { return sp->npts; }
int sphere_ptot(pp_sphere *sp) { return sp->ptot; }
int sphere_precision(pp_sphere *sp) { return sp->precision; }
const int *sphere_fftg(pp_sphere *sp) { return sp->fftg; }
const double *sphere_lattice(pp_sphere *sp) { return sp->lattice; }

}  // namespace pp

using namespace pp;

extern "C" int pp_sphere_create(pp_ctx *ctx, pp_sphere **out, const double *lattice, const int *fftg,
                                int num_sites, const int *labels, const double *frac_coords, int num_elems,
                                const int *nchan, const int *ls, const double *rmax, const int *ngrid,
                                const double *proj, int precision) {
  PP_REQUIRE(ctx && out && lattice && fftg && num_sites >= 0 && num_elems > 0, PP_ERR_ARG,
             "pp_sphere_create: bad arguments");
  PP_REQUIRE(precision == PP_FP64 || precision == PP_FP32 || precision == PP_BF16X3 ||
                 precision == PP_BF16X6 || precision == PP_FP16X3,
             PP_ERR_ARG,
             "pp_sphere_create: unknown precision");
  PP_CHECK_HIP(hipSetDevice(ctx->device));
  pp_sphere *sp = new pp_sphere();
  sp->ctx = ctx;
  sp->precision = precision == PP_FP64 ? PP_FP64 : PP_FP32;
  memcpy(sp->lattice, lattice, sizeof(sp->lattice));
  memcpy(sp->fftg, fftg, sizeof(sp->fftg));
  sp->nsites = num_sites;
  sp->nelems = num_elems;
  sp->labels.assign(labels, labels + num_sites);
  sp->frac.assign(frac_coords, frac_coords + 3 * num_sites);
  sp->nchan.assign(nchan, nchan + num_elems);
  sp->ngrid.assign(ngrid, ngrid + num_elems);
  sp->rmax.assign(rmax, rmax + num_elems);
  for (int s = 0; s < num_sites; s++)
    if (labels[s] < 0 || labels[s] >= num_elems) {
      delete sp;
      PP_REQUIRE(false, PP_ERR_ARG, "pp_sphere_create: site label out of range");
    }
  // species spline blocks: x, f[nchan], b[nchan], c[nchan], d[nchan]
  std::vector<double> spl;
  int lo = 0;
  long po = 0;
  for (int e = 0; e < num_elems; e++) {
    sp->ls_off.push_back(lo);
    int n = ngrid[e];
    if (n < 3) {
      delete sp;
      PP_REQUIRE(false, PP_ERR_ARG, "pp_sphere_create: projector grid needs >= 3 points");
    }
    std::vector<double> x(n);
    for (int j = 0; j < n; j++)
      x[j] = rmax[e] / n * j;  // projector.c:56
    size_t base = spl.size();
    spl.resize(base + (size_t)(1 + 4 * nchan[e]) * n);
    memcpy(&spl[base], x.data(), sizeof(double) * n);
    for (int ch = 0; ch < nchan[e]; ch++) {
      sp->ls.push_back(ls[lo + ch]);
      if (ls[lo + ch] < 0 || ls[lo + ch] > 3) {
        delete sp;
        PP_REQUIRE(false, PP_ERR_UNSUPPORTED, "pp_sphere_create: l must be 0..3");
      }
      const double *f = proj + po + (long)ch * n;
      double *F = &spl[base + (size_t)(1 + ch) * n];
      double *B = &spl[base + (size_t)(1 + nchan[e] + ch) * n];
      double *C = &spl[base + (size_t)(1 + 2 * nchan[e] + ch) * n];
      double *D = &spl[base + (size_t)(1 + 3 * nchan[e] + ch) * n];
      memcpy(F, f, sizeof(double) * n);
      spline_coeff_host(x.data(), f, n, B, C, D);
    }
    lo += nchan[e];
    po += (long)nchan[e] * n;
  }
  int st = sp->d_spline.ensure(sizeof(double) * spl.size());
  if (st == PP_OK)
    st = sp->d_chan.ensure(sizeof(int) * std::max<size_t>(1, sp->ls.size()));
  if (st != PP_OK) {
    delete sp;
    return st;
  }
  PP_CHECK_HIP(hipMemcpy(sp->d_spline.p, spl.data(), sizeof(double) * spl.size(), hipMemcpyHostToDevice));
  PP_CHECK_HIP(hipMemcpy(sp->d_chan.p, sp->ls.data(), sizeof(int) * sp->ls.size(), hipMemcpyHostToDevice));
  st = sphere_build(sp);
  if (st != PP_OK) {
    delete sp;
    return st;
  }
  *out = sp;
  return PP_OK;
}

extern "C" int pp_sphere_rebuild(pp_sphere *sp, const double *frac_coords) {
  PP_REQUIRE(sp && frac_coords, PP_ERR_ARG, "pp_sphere_rebuild: bad arguments");
  sp->frac.assign(frac_coords, frac_coords + 3 * sp->nsites);
  return sphere_build(sp);
}

extern "C" void pp_sphere_destroy(pp_sphere *sp) { delete sp; }

extern "C" int pp_sphere_coverage(pp_sphere *sp, long *covered) {
  PP_REQUIRE(sp && covered, PP_ERR_ARG, "pp_sphere_coverage: null argument");
  PP_CHECK_HIP(hipSetDevice(sp->ctx->device));
  const size_t nw = (size_t)sp->fftg[1] * sp->fftg[2] * sp->xmask_words;
  std::vector<unsigned> m(nw);
  PP_CHECK_HIP(hipStreamSynchronize(sp->ctx->stream));
  if (nw)
    PP_CHECK_HIP(hipMemcpy(m.data(), sp->d_xmask.p, sizeof(unsigned) * nw, hipMemcpyDeviceToHost));
  long c = 0;
  for (unsigned w : m)
    c += __builtin_popcount(w);
  *covered = c;
  return PP_OK;
}

extern "C" int pp_sphere_info(pp_sphere *sp, int *total_projs, long *total_points, int *proj_off) {
  PP_REQUIRE(sp, PP_ERR_ARG, "pp_sphere_info: null plan");
  if (total_projs)
    *total_projs = sp->ptot;
  if (total_points)
    *total_points = sp->npts;
  if (proj_off)
    memcpy(proj_off, sp->proj_off.data(), sizeof(int) * (sp->nsites + 1));
  return PP_OK;
}

// FFT passes of compile-time length N = R1 R2: two register-level DFTs with
// one exchange through LDS between them.
//
// A work-group takes LPW 128-byte band groups (16 bands FP32, 8 FP64) of a
// line, or of adjacent lines where a line has fewer.  A thread of the first half loads its R1 elements (j2 + R2 j1) of
// one line straight into registers, transforms them and writes them, times
// W_N^(j2 k1), to LDS; a thread of the second half reads R2 of those,
// transforms them and stores the outputs k1 + R1 k2 straight to memory.  An
// element makes one LDS round trip and the work-group two barriers; the
// staged form made one round trip and two barriers per radix plus one for
// the line (four or five for the usual lengths).  Per 64-band FP32 chunk on
// 80 x 54 x 54: x 45.5 -> 35.2 us, y 44.8 -> 23.2, z 28.8 -> 16.0 against the
// run-time staged passes; on 108^3 x 252 -> 206, y 134 -> 96, z 64 -> 45, near
// the memory's rate.  Eight or sixteen lanes hold a line's band group, so each
// of their global and LDS accesses is one contiguous 128 bytes and LDS reads
// and writes are free of bank conflicts.
#pragma once
#include "pp_dft.h"
#include "pp_internal.h"
#include "pp_stages.h"

namespace pp {

// Lengths with a pass, as X(N, R1, R2): the 50 even lengths from 8 to 256 with
// factors 2, 3, 5 and 7, and above them seven of the doubled grids (270, 280,
// 288, 300, 320, 324, 360).  294, 336, 378, 384 and 392 are no products of two
// of the radices with a register-level DFT (at most 25); they, 350 and 400 run
// the staged passes.  Where both orders of the halves take the same time the
// one whose FP32 projections are nearer to the FP64 ones stands (215 sites,
// 108 points: 1.13e-7 with 9 first, 1.18e-7 with 12; 120: 9.4e-8, 9.8e-8).
#define PP_FFT2_A(X) X(8, 4, 2) X(10, 5, 2) X(12, 4, 3) X(14, 7, 2) X(16, 4, 4) X(18, 6, 3) X(20, 5, 4) X(24, 6, 4) \
  X(28, 7, 4) X(30, 6, 5) X(32, 8, 4) X(36, 6, 6) X(40, 8, 5) X(42, 7, 6) X(48, 8, 6)
#define PP_FFT2_B(X) X(50, 10, 5) X(54, 9, 6) X(56, 8, 7) X(60, 10, 6) X(64, 8, 8) X(70, 10, 7) X(72, 9, 8) X(80, 10, 8)
#define PP_FFT2_C(X) X(84, 12, 7) X(90, 9, 10) X(96, 12, 8) X(98, 14, 7) X(100, 10, 10) X(108, 9, 12)
#define PP_FFT2_D(X) X(112, 14, 8) X(120, 10, 12) X(126, 14, 9) X(128, 16, 8) X(140, 14, 10) X(144, 12, 12)
#define PP_FFT2_E(X) X(150, 15, 10) X(160, 16, 10) X(162, 18, 9) X(168, 14, 12) X(180, 15, 12) X(192, 16, 12)
#define PP_FFT2_F(X) X(196, 14, 14) X(200, 20, 10) X(210, 15, 14) X(216, 18, 12) X(224, 16, 14)
#define PP_FFT2_G(X) X(240, 16, 15) X(250, 25, 10) X(252, 18, 14) X(256, 16, 16) X(270, 18, 15)
#define PP_FFT2_H(X) X(280, 20, 14) X(288, 18, 16) X(300, 20, 15) X(320, 20, 16) X(324, 18, 18) X(360, 20, 18)
#define PP_FFT2_ALL(X)                                                                              \
  PP_FFT2_A(X) PP_FFT2_B(X) PP_FFT2_C(X) PP_FFT2_D(X) PP_FFT2_E(X) PP_FFT2_F(X) PP_FFT2_G(X) PP_FFT2_H(X)

// Bands of a group: 128 bytes.
template <typename T> constexpr int fft2_bands() { return 128 / (int)sizeof(cplx<T>); }
// Lanes of a line's band group: 8 of 16 bytes each (FP32 two bands a lane),
// or for long FP32 lines 16 of 8 bytes, which doubles the wavefronts that
// share a line's LDS (y pass of 192: 474 -> 448 us per 64-band chunk), unless
// one group fills the work-group alone (fft2_lines), whose rows of 128 bytes
// want the wider accesses (x pass of 216: 1669 us, 2018 with 16 lanes).
template <typename T> constexpr int fft2_lanes(int R1, int R2) {
  return sizeof(T) == 4 && (R1 > R2 ? R1 : R2) >= 16 && 2 * R1 * R2 * 128 <= 52 * 1024 ? 16 : 8;
}
// Band groups of a work-group: about 256 threads and at most 36 KiB of rows
// (four or more work-groups per CU), but two where 52 KiB hold them: the 256
// contiguous bytes per element of two groups side by side run faster than
// 128 (x pass of 108 in FP64 465 -> 421 us; two of 216 leave two work-groups
// per CU, 3185 -> 3715).  Two FP64 units of more than 256 threads do not get
// two work-groups into a CU's registers and take turns with nobody: one (32
// bands in FP64, z / y / x of 200: 200 / 576 / 1103 us against 282 / 796 /
// 1629, of 162: 171 / 391 / 676 against 248 / 578 / 971).
template <typename T> constexpr int fft2_lines(int R1, int R2) {
  const int rm = R1 > R2 ? R1 : R2, by_threads = 256 / (fft2_lanes<T>(R1, R2) * rm);
  const int row = R1 * R2 * 128, by_lds = 36 * 1024 / row, least = 2 * row <= 52 * 1024 ? 2 : 1;
  const int n = by_threads < by_lds ? by_threads : by_lds;
  const bool one = sizeof(T) == 8 && 2 * fft2_lanes<T>(R1, R2) * rm > 256;
  return n > least ? n : one ? (n > 1 ? n : 1) : least;
}
template <typename T> constexpr int fft2_threads(int R1, int R2) {
  return fft2_lines<T>(R1, R2) * fft2_lanes<T>(R1, R2) * (R1 > R2 ? R1 : R2);
}

// What a pass reads besides the chunk: the axis' [k1][j2] twiddles and the
// line geometry (element e of line (l1, l2) at g[l1 * s1 + l2 * s2 + e * es]).
template <typename T> struct Fft2Args {
  const cplx<T> *tw;
  long es, s1, s2;
  int axis, n2, ngroups, streaming;
  long nlines;
};

// A line of a pass: whether it has work, its number, its offset and the
// signed index interval [lo, hi] of its input (pruned as in k_fft_pass).
struct PassLine {
  bool on = false;
  int line = 0, lo = 0, hi = 0;
  long base = 0;
};
// Line l: an entry of the axis' populated-line list where there is one
// (line, lo and hi in one load, the line's elements depend on nothing
// else), else line l itself with the bounds of its k-point.
__device__ __forceinline__ PassLine fft2_line(const SphereBounds &bd, int axis, int n2, long s1, long s2, long l,
                                              long nlines) {
  PassLine r;
  if (l >= nlines)
    return r;
  r.on = true;
  r.lo = -(1 << 30);
  r.hi = 1 << 30;
  const int2 *ll = reinterpret_cast<const int2 *>(axis == 2 ? bd.zl : axis == 1 ? bd.yl : nullptr);
  if (ll) {
    const int2 e = ll[l];
    r.line = e.x;
    r.lo = e.y >> 16;
    r.hi = (int)(short)(e.y & 0xffff);
  } else {
    r.line = (int)l;
  }
  const int l1 = r.line / n2, l2 = r.line % n2;
  r.base = (long)l1 * s1 + (long)l2 * s2;
  if (ll || !bd.xb)
    return r;
  if (axis == 2) {
    const int sx = sgn_idx(l1, bd.n0), sy = sgn_idx(l2, bd.n1);
    r.on = sx >= bd.xb[0] && sx <= bd.xb[1] && sy >= bd.yb[2 * l1] && sy <= bd.yb[2 * l1 + 1];
    r.lo = bd.zb[2 * (l1 * bd.n1 + l2)];
    r.hi = bd.zb[2 * (l1 * bd.n1 + l2) + 1];
  } else if (axis == 1) {
    const int sx = sgn_idx(l1, bd.n0);
    r.on = sx >= bd.xb[0] && sx <= bd.xb[1];
    r.lo = bd.yb[2 * l1];
    r.hi = bd.yb[2 * l1 + 1];
  } else {
    r.lo = bd.xb[0];
    r.hi = bd.xb[1];
  }
  return r;
}

// A lane's part of an element row: PK bands (16 bytes, or one FP32 band).
template <typename T, int PK> struct BandPack {
  cplx<T> v[PK];
};
template <typename T, int PK> __device__ __forceinline__ BandPack<T, PK> load_pack(const cplx<T> *p, bool nt) {
  BandPack<T, PK> r;
  if constexpr (PK == 2)
    load2(p, nt, r.v[0], r.v[1]);
  else
    r.v[0] = nt ? load_nt(p) : *p;
  return r;
}
template <typename T, int PK>
__device__ __forceinline__ void store_pack(cplx<T> *p, bool nt, const BandPack<T, PK> &r) {
  if constexpr (PK == 2)
    store2(p, nt, r.v[0], r.v[1]);
  else if (nt)
    store_nt(p, r.v[0]);
  else
    *p = r.v[0];
}

// The pass of work-group blk: LPW units (line, band group).  buf: LPW * N rows of 128 bytes, twl: N
// twiddles, msk: LPW * MW coverage words (all LDS).
template <typename T, int R1, int R2>
__device__ __forceinline__ void fft2_tile(cplx<T> *__restrict__ g, const Fft2Args<T> &a, const SphereBounds &bd,
                                          int blk, cplx<T> *__restrict__ buf, cplx<T> *__restrict__ twl,
                                          unsigned *__restrict__ msk) {
  constexpr int N = R1 * R2, LPW = fft2_lines<T>(R1, R2), NT = fft2_threads<T>(R1, R2), MW = (N + 31) / 32;
  constexpr int LR = fft2_lanes<T>(R1, R2), ROW = fft2_bands<T>(), PK = ROW / LR;
  const long u0 = (long)blk * LPW;  // units (line, band group), the groups of a line adjacent
  const int t = threadIdx.x, p = t % LR, q = t / LR;
  const bool masked = a.axis == 0 && bd.xm;
  // the units of an element next to each other, so that a wavefront's access
  // to two band groups of a line is whole 256-byte rows (64 bands in FP32, z /
  // y / x of 108: 45 / 95 / 167 us against 50 / 111 / 184 with a unit's
  // elements next to each other, of 192: 123 / 410 / 893 against 142 / 449 /
  // 1034; FP64 and one unit per work-group: the same)
  const int j2 = q / LPW % R2, k1 = q / LPW % R1, ll = q % LPW;
  const unsigned ua = (unsigned)(u0 + ll), ng = (unsigned)a.ngroups;
  const PassLine la = fft2_line(bd, a.axis, a.n2, a.s1, a.s2, ua / ng, a.nlines);
  const bool ina = q < LPW * R2, inb = q < LPW * R1;
  // twiddles and coverage words are read into registers ahead of the line's
  // elements and written to LDS after those loads, so that all wait on one
  // memory latency
  constexpr int TWR = (N + NT - 1) / NT, MKR = (LPW * MW + NT - 1) / NT;
  cplx<T> twr[TWR];
#pragma unroll
  for (int r = 0; r < TWR; r++)
    twr[r] = t + r * NT < N ? a.tw[t + r * NT] : mk<T>(0, 0);
  unsigned mkr[MKR];
  if (masked) {
#pragma unroll
    for (int r = 0; r < MKR; r++) {
      const int i = t + r * NT;
      const long l = (unsigned)(u0 + i / MW) / ng;
      mkr[r] = i < LPW * MW && l < a.nlines && i % MW < bd.xmw ? bd.xm[l * bd.xmw + i % MW] : 0u;
    }
  }
  {
    cplx<T> v[PK][R1];
    const cplx<T> *src = g + la.base + (ua % ng) * ROW + p * PK + (long)j2 * a.es;
    const long step = (long)R2 * a.es;
#pragma unroll
    for (int j1 = 0; j1 < R1; j1++) {
      const int e = j2 + R2 * j1, se = e < N - N / 2 ? e : e - N;
      BandPack<T, PK> x;
#pragma unroll
      for (int c = 0; c < PK; c++)
        x.v[c] = mk<T>(0, 0);
      if (ina && la.on && se >= la.lo && se <= la.hi)
        x = load_pack<T, PK>(src + j1 * step, a.streaming > 1);
#pragma unroll
      for (int c = 0; c < PK; c++)
        v[c][j1] = x.v[c];
    }
#pragma unroll
    for (int r = 0; r < TWR; r++)
      if (t + r * NT < N)
        twl[t + r * NT] = twr[r];
    if (masked) {
#pragma unroll
      for (int r = 0; r < MKR; r++)
        if (t + r * NT < LPW * MW)
          msk[t + r * NT] = mkr[r];
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < PK; c++)
      Dft<T, R1>::run(v[c]);
    if (ina) {
#pragma unroll
      for (int k = 0; k < R1; k++) {
        BandPack<T, PK> x;
        const cplx<T> w = k > 0 ? twl[k * R2 + j2] : mk<T>(1, 0);
#pragma unroll
        for (int c = 0; c < PK; c++)
          x.v[c] = k > 0 ? v[c][k] * w : v[c][k];
        store_pack<T, PK>(buf + (((k * R2 + j2) * LPW + ll) * LR + p) * PK, false, x);
      }
    }
  }
  __syncthreads();
  if (!inb || !la.on)
    return;
  cplx<T> v[PK][R2];
#pragma unroll
  for (int j = 0; j < R2; j++) {
    const BandPack<T, PK> x = load_pack<T, PK>(buf + (((k1 * R2 + j) * LPW + ll) * LR + p) * PK, false);
#pragma unroll
    for (int c = 0; c < PK; c++)
      v[c][j] = x.v[c];
  }
#pragma unroll
  for (int c = 0; c < PK; c++)
    Dft<T, R2>::run(v[c]);
  cplx<T> *dst = g + la.base + (ua % ng) * ROW + p * PK + (long)k1 * a.es;
  const long step = (long)R1 * a.es;
#pragma unroll
  for (int k2 = 0; k2 < R2; k2++) {
    const int e = k1 + R1 * k2;
    if (masked && !((msk[ll * MW + (e >> 5)] >> (e & 31)) & 1u))
      continue;  // no projector sphere reads this point
    BandPack<T, PK> x;
#pragma unroll
    for (int c = 0; c < PK; c++)
      x.v[c] = v[c][k2];
    store_pack<T, PK>(dst + k2 * step, a.streaming != 0, x);
  }
}

#define PP_FFT2_LDS                                                                          \
  constexpr int N = R1 * R2, LPW = fft2_lines<T>(R1, R2);                                       \
  __shared__ __align__(16) cplx<T> buf[LPW * N * fft2_bands<T>()];                       \
  __shared__ cplx<T> twl[N];                                                                 \
  __shared__ unsigned msk[LPW * ((N + 31) / 32)];

template <typename T, int R1, int R2>
__global__ __launch_bounds__(fft2_threads<T>(R1, R2)) void k_fft2(cplx<T> *__restrict__ g, Fft2Args<T> a, SphereBounds bd,
                                                              int xcd_per, int nblk) {
  PP_FFT2_LDS
  const int blk = xcd_per > 0 ? (int)(blockIdx.x % 8) * xcd_per + (int)(blockIdx.x / 8) : (int)blockIdx.x;
  if (blk >= nblk)
    return;
  fft2_tile<T, R1, R2>(g, a, bd, blk, buf, twl, msk);
}

// The bounds of a work item as SphereBounds (lists of the pass only).
__device__ __forceinline__ SphereBounds item_bounds(const ChunkItem *it, int axis) {
  SphereBounds bd;
  bd.zb = (const int *)it->zb;
  bd.yb = (const int *)it->yb;
  bd.xb = (const int *)it->xb;
  bd.n0 = it->n0;
  bd.n1 = it->n1;
  bd.n2 = it->n2;
  bd.zl = axis == 2 ? (const int *)it->zl : nullptr;
  bd.nzl = axis == 2 ? it->nzl : 0;
  bd.yl = axis == 1 ? (const int *)it->yl : nullptr;
  bd.nyl = axis == 1 ? it->nyl : 0;
  bd.xm = axis == 0 ? (const unsigned *)it->xm : nullptr;
  bd.xmw = axis == 0 ? it->xmw : 0;
  return bd;
}
// Lines of a pass over a chunk with these bounds.
__host__ __device__ inline long pass_lines(const SphereBounds &bd, int axis) {
  return axis == 2   ? (bd.zl ? bd.nzl : (long)bd.n0 * bd.n1)
         : axis == 1 ? (bd.yl ? bd.nyl : (long)bd.n0 * bd.n2)
                     : (long)bd.n1 * bd.n2;
}

// The pass over the chunks of a batch of work items (one per blockIdx.y).
template <typename T, int R1, int R2>
__global__ __launch_bounds__(fft2_threads<T>(R1, R2)) void k_fft2_items(const ChunkItem *__restrict__ items, Fft2Args<T> a) {
  PP_FFT2_LDS
  const ChunkItem *it = items + blockIdx.y;
  const SphereBounds bd = item_bounds(it, a.axis);
  a.nlines = pass_lines(bd, a.axis);
  if ((long)blockIdx.x * LPW >= a.nlines * a.ngroups)
    return;
  fft2_tile<T, R1, R2>((cplx<T> *)it->grid, a, bd, (int)blockIdx.x, buf, twl, msk);
}

// Launchers of one length (f64, items64: nullptr where FP64 has no such pass).
struct Fft2Entry {
  int n, r1, r2;
  void (*f32)(hipStream_t, cplx<float> *, const Fft2Args<float> &, const SphereBounds &, bool);
  void (*f64)(hipStream_t, cplx<double> *, const Fft2Args<double> &, const SphereBounds &, bool);
  void (*items32)(hipStream_t, const ChunkItem *, int, const Fft2Args<float> &);
  void (*items64)(hipStream_t, const ChunkItem *, int, const Fft2Args<double> &);
};

// a.nlines: the lines of the pass (of the largest item).
template <typename T, int R1, int R2>
void fft2_launch(hipStream_t st, cplx<T> *g, const Fft2Args<T> &a, const SphereBounds &bd, bool xcd) {
  const long nblk = (a.nlines * a.ngroups + fft2_lines<T>(R1, R2) - 1) / fft2_lines<T>(R1, R2);
  const int per = xcd ? (int)((nblk + 7) / 8) : 0;
  hipLaunchKernelGGL((k_fft2<T, R1, R2>), dim3((unsigned)(per ? 8L * per : nblk)), dim3(fft2_threads<T>(R1, R2)), 0, st, g,
                     a, bd, per, (int)nblk);
}
template <typename T, int R1, int R2>
void fft2_launch_items(hipStream_t st, const ChunkItem *items, int nitems, const Fft2Args<T> &a) {
  const long nblk = (a.nlines * a.ngroups + fft2_lines<T>(R1, R2) - 1) / fft2_lines<T>(R1, R2);
  hipLaunchKernelGGL((k_fft2_items<T, R1, R2>), dim3((unsigned)nblk, (unsigned)nitems), dim3(fft2_threads<T>(R1, R2)), 0,
                     st, items, a);
}
// FP64 passes stop at radix 20: the 25 complex values of a radix-25 half take
// 210 registers, which leave two wavefronts per SIMD, and the staged pass is
// the faster (32 bands in FP64, z / y / x of 250: 342 / 1309 / 3657 us against
// 302 / 1023 / 2776; FP32 145 / 539 / 1518 against 178 / 602 / 1668).
template <int R1, int R2> constexpr auto fft2_f64() {
  if constexpr (R1 <= 20)
    return fft2_launch<double, R1, R2>;
  else
    return nullptr;
}
template <int R1, int R2> constexpr auto fft2_items_f64() {
  if constexpr (R1 <= 20)
    return fft2_launch_items<double, R1, R2>;
  else
    return nullptr;
}
#define PP_FFT2_ENTRY(N, R1, R2)                                                                            \
  {N, R1, R2, fft2_launch<float, R1, R2>, fft2_f64<R1, R2>(), fft2_launch_items<float, R1, R2>, \
   fft2_items_f64<R1, R2>()},
// A translation unit's entries (the lengths are spread over several so that
// they compile in parallel), closed by n = 0.
#define PP_FFT2_TABLE(NAME, LIST)                                  \
  namespace pp {                                                   \
  const Fft2Entry *NAME() {                                        \
    static const Fft2Entry t[] = {LIST(PP_FFT2_ENTRY){0, 0, 0}};   \
    return t;                                                      \
  }                                                                \
  }

// The entry of length n, nullptr when there is none.
const Fft2Entry *fft2_entry(int n);

}  // namespace pp

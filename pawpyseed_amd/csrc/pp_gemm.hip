// Complex "NT" GEMM: C[m][n] (+)= sum_k conj(A[m][k]) B[n][k].
//
// The band-overlap matrix of pseudoprojector.c:63-90 (one cdotc per band
// pair) and the O_M augmentation sum of projector.c:890-910 are both this
// contraction with K contiguous in both operands.  FP64 path: FP64 matrix
// cores (k_zgemm_mfma64) or, selectable, a VALU tile GEMM (64x64 output
// tiles, 4x4 complex accumulators per thread); K tiles of 16 staged through
// LDS; split-K with a deterministic reduction when the tile grid alone
// cannot fill the 256 CUs.
#include <type_traits>

#include "pp_internal.h"

namespace pp {

// (with GA, column k of A is column acol[k] of its rows, as k_zgemm_mfma64)
template <typename TA, typename TB, bool GA>
__global__ __launch_bounds__(256) void k_zgemm_f64(int M, int N, int kbeg_stride, int K, int nsplit,
                                                   const cplx<TA> *__restrict__ A, long lda,
                                                   const int *__restrict__ acol, const cplx<TB> *__restrict__ B,
                                                   long ldb, cplx<double> *__restrict__ C, long ldc, long sSplit) {
  __shared__ cplx<double> As[16][64 + 1];
  __shared__ cplx<double> Bs[16][64 + 1];
  const int tilesN = (N + 63) / 64;
  int split, tile;
  if (!gemm_block(((M + 63) / 64) * tilesN, nsplit, split, tile))
    return;
  const int tm = tile / tilesN, tn = tile % tilesN;
  const int k0 = split * kbeg_stride;
  const int k1 = min(K, k0 + kbeg_stride);
  C += (long)split * sSplit;
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  double ar[4][4], ai[4][4];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++)
      ar[i][j] = ai[i][j] = 0.0;
  for (int kb = k0; kb < k1; kb += 16) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      int e = tid + q * 256;
      int r = e >> 4, kk = e & 15;
      int gm = tm * 64 + r, gn = tn * 64 + r, gk = kb + kk;
      cplx<double> va = mk<double>(0, 0), vb = mk<double>(0, 0);
      if (gk < k1) {
        if (gm < M)
          va = cvt<double>(A[(long)gm * lda + (GA ? acol[gk] : gk)]);
        if (gn < N)
          vb = cvt<double>(B[(long)gn * ldb + gk]);
      }
      As[kk][r] = va;
      Bs[kk][r] = vb;
    }
    __syncthreads();
#pragma unroll 4
    for (int kk = 0; kk < 16; kk++) {
      cplx<double> a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; i++)
        a[i] = As[kk][ty + 16 * i];
#pragma unroll
      for (int j = 0; j < 4; j++)
        b[j] = Bs[kk][tx + 16 * j];
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          // conj(a) * b
          ar[i][j] = fma(a[i].x, b[j].x, ar[i][j]);
          ar[i][j] = fma(a[i].y, b[j].y, ar[i][j]);
          ai[i][j] = fma(a[i].x, b[j].y, ai[i][j]);
          ai[i][j] = fma(-a[i].y, b[j].x, ai[i][j]);
        }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) {
      int gm = tm * 64 + ty + 16 * i, gn = tn * 64 + tx + 16 * j;
      if (gm < M && gn < N)
        C[(long)gm * ldc + gn] = mk<double>(ar[i][j], ai[i][j]);
    }
}

typedef double doublex4 __attribute__((ext_vector_type(4)));

// FP64 matrix-core form of conj(A) B^T on v_mfma_f64_16x16x4_f64.
// Work-group: 4 wavefronts, 64x64 complex outputs, each wavefront a 32x32
// quadrant of 2x2 16x16 tiles.  The four k indices of an MFMA are four
// consecutive complex terms, and a lane holds the whole complex value of
// its term: Re takes (ar, br) and (ai, bi), Im (ar, bi) and (-ai, br), so
// one 16-byte LDS read per operand value serves all four products.  (Taking
// K as the 2K interleaved reals needed the neighbour's value too for Im, a
// third of the LDS reads, and 8-byte accesses with four-way write
// conflicts.)  Output layout of a 16x16 tile: lane l, register v holds row
// l/16 + 4v, column l%16 (unlike the FP32 16x16x4 form, whose register v is
// row 4(l/16)+v).
//
// One launch runs every batch of gb (the k-points of a call): a launch per
// batch split K into enough chunks to fill the chip alone (16 for 512 x 512
// outputs) and paid their partial sums and a tail each time; together four
// batches need four.  The GEMM is bound by the FP64 matrix rate (64 cycles
// per MFMA), so a quadrant at the edge of the outputs runs only the 16x16
// tiles that hold any, and the quadrants rotate over the wavefronts from
// work-group to work-group so that the short ones spread over the SIMDs.
// With GA, column k of A is column acol[k] of its rows (the matched-site
// projections gathered on the way in), the indices loaded a k-step ahead.
template <typename TA, typename TB, bool GA>
__global__ __launch_bounds__(256, 3) void k_zgemm_mfma64(int M, int N, int kchunk, int nsplit, GemmBatch gb,
                                                      const cplx<TA> *__restrict__ A, long lda, long sA,
                                                      const int *__restrict__ acol, const cplx<TB> *__restrict__ B,
                                                      long ldb, long sB, cplx<double> *__restrict__ C, long ldc,
                                                      long sSplit, long sBatch, int accumulate) {
  __shared__ cplx<double> As[64][17];  // 17: the 16 rows of an operand read fall on distinct banks
  __shared__ cplx<double> Bs[64][17];
  const int tilesN = (N + 63) / 64, tiles = ((M + 63) / 64) * tilesN;
  int chunk, tile;
  if (!gemm_block(tiles, nsplit * gb.n, chunk, tile))
    return;
  const int bt = chunk / nsplit, split = chunk % nsplit;
  const int tm = tile / tilesN, tn = tile % tilesN;
  const int K = gb.k[bt];
  const int k0 = split * kchunk;
  const int k1 = min(K, k0 + kchunk);
  A += gb.a[bt] * sA;
  B += gb.b[bt] * sB;
  C += (long)split * sSplit + bt * sBatch;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) + (blockIdx.x >> 3) + (blockIdx.x >> 8)) & 3;
  const int wm = wave >> 1, wn = wave & 1;
  // 16x16 tiles of the quadrant that hold outputs: mt x nt of 2 x 2
  const int mt = min(2, max(0, (M - tm * 64 - wm * 32 + 15) >> 4));
  const int nt = min(2, max(0, (N - tn * 64 - wn * 32 + 15) >> 4));
  doublex4 cr[2][2], ci[2][2];
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2; b++) {
      cr[a][b] = doublex4{0.0, 0.0, 0.0, 0.0};
      ci[a][b] = doublex4{0.0, 0.0, 0.0, 0.0};
    }
  const int lrow = threadIdx.x >> 2, part = threadIdx.x & 3;
  // a k-step's 4 + 4 values of a thread are loaded together, the next
  // step's while the current step's MFMAs run; rows past the last are read
  // as the last one (their outputs are not stored), so only the step at the
  // end of the chunk carries guards
  const cplx<TA> *rowA = A + (long)min(M - 1, tm * 64 + lrow) * lda;
  const cplx<TB> *rowB = B + (long)min(N - 1, tn * 64 + lrow) * ldb;
  cplx<TA> pa[4];
  cplx<TB> pb[4];
  int ca[4] = {0, 0, 0, 0};
  auto columns = [&](int kb) {
    if constexpr (GA) {
#pragma unroll
      for (int c = 0; c < 4; c++)
        ca[c] = acol[min(kb + part * 4 + c, k1 - 1)];
    }
  };
  auto fetch = [&](int kb) {
    const int gk = kb + part * 4;
    if (kb + 16 <= k1) {
#pragma unroll
      for (int c = 0; c < 4; c++) {
        pa[c] = rowA[GA ? ca[c] : gk + c];
        pb[c] = rowB[gk + c];
      }
    } else {
#pragma unroll
      for (int c = 0; c < 4; c++) {
        pa[c] = gk + c < k1 ? rowA[GA ? ca[c] : gk + c] : mk<TA>((TA)0, (TA)0);
        pb[c] = gk + c < k1 ? rowB[gk + c] : mk<TB>((TB)0, (TB)0);
      }
    }
    columns(kb + 16);
  };
  if (k0 < k1) {
    columns(k0);
    fetch(k0);
  }
  const int sub = lane & 15, kq = lane >> 4;
  auto stage = [&](int kb) {
#pragma unroll
    for (int c = 0; c < 4; c++) {
      As[lrow][part * 4 + c] = cvt<double>(pa[c]);
      Bs[lrow][part * 4 + c] = cvt<double>(pb[c]);
    }
    __syncthreads();
    if (kb + 16 < k1)
      fetch(kb + 16);
  };
  // the k loop of MT x NT 16x16 tiles (wavefronts of one work-group may run
  // different ones: each has the same barriers); one loop per count keeps
  // the accumulators in place
  auto steps = [&](auto mtc, auto ntc) {
    constexpr int MT = decltype(mtc)::value, NT = decltype(ntc)::value;
    for (int kb = k0; kb < k1; kb += 16) {
      stage(kb);
      if constexpr (MT > 0 && NT > 0) {
#pragma unroll 2
        for (int kk = 0; kk < 16; kk += 4) {
          cplx<double> a[MT], b[NT];
#pragma unroll
          for (int mi = 0; mi < MT; mi++)
            a[mi] = As[wm * 32 + mi * 16 + sub][kk + kq];
#pragma unroll
          for (int nj = 0; nj < NT; nj++)
            b[nj] = Bs[wn * 32 + nj * 16 + sub][kk + kq];
#pragma unroll
          for (int mi = 0; mi < MT; mi++)
#pragma unroll
            for (int nj = 0; nj < NT; nj++) {
              cr[mi][nj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[mi].x, b[nj].x, cr[mi][nj], 0, 0, 0);
              ci[mi][nj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[mi].x, b[nj].y, ci[mi][nj], 0, 0, 0);
            }
#pragma unroll
          for (int mi = 0; mi < MT; mi++)
#pragma unroll
            for (int nj = 0; nj < NT; nj++) {
              cr[mi][nj] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[mi].y, b[nj].y, cr[mi][nj], 0, 0, 0);
              ci[mi][nj] = __builtin_amdgcn_mfma_f64_16x16x4f64(-a[mi].y, b[nj].x, ci[mi][nj], 0, 0, 0);
            }
        }
      }
      __syncthreads();
    }
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  if (mt == 2 && nt == 2)
    steps(I2{}, I2{});
  else if (mt == 2 && nt == 1)
    steps(I2{}, I1{});
  else if (mt == 1 && nt == 2)
    steps(I1{}, I2{});
  else if (mt == 1 && nt == 1)
    steps(I1{}, I1{});
  else
    steps(I0{}, I0{});
#pragma unroll
  for (int mi = 0; mi < 2; mi++)
#pragma unroll
    for (int nj = 0; nj < 2; nj++) {
      const int j = tn * 64 + wn * 32 + nj * 16 + (lane & 15);
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int i = tm * 64 + wm * 32 + mi * 16 + (lane >> 4) + 4 * v;
        if (i < M && j < N) {
          cplx<double> *c = C + (long)i * ldc + j;
          const cplx<double> s = mk<double>(cr[mi][nj][v], ci[mi][nj][v]);
          *c = accumulate ? *c + s : s;
        }
      }
    }
}

// C[m][n] (+)= sum over splits of partial[s][m][n], in FP64 (partials FP64
// or FP32), for batch blockIdx.y (sP, sC apart)
template <typename TP>
__global__ __launch_bounds__(256) void k_splitk_reduce(int M, int N, int nsplit, const cplx<TP> *__restrict__ P,
                                                       long sP, cplx<double> *__restrict__ C, long ldc, long sC,
                                                       int accumulate) {
  long t = (long)blockIdx.x * 256 + threadIdx.x;
  if (t >= (long)M * N)
    return;
  P += blockIdx.y * sP;
  C += blockIdx.y * sC;
  int m = (int)(t / N), n = (int)(t % N);
  cplx<double> s = accumulate ? C[(long)m * ldc + n] : mk<double>(0, 0);
#pragma unroll 8
  for (int q = 0; q < nsplit; q++)
    s = s + cvt<double>(P[(long)q * M * N + t]);
  C[(long)m * ldc + n] = s;
}

int gemm_fp32_mfma(pp_ctx *ctx, int precision, int M, int N, int K, const void *A, long lda, const void *B, long ldb,
                   cplx<double> *C, long ldc, bool accumulate, int slot);
bool plane_precision(int precision);
int plane_gemm_pipeline(pp_ctx *ctx, int precision, int M, int N, int K, const void *A, long lda, long sA,
                        const void *B, long ldb, long sB, cplx<double> *C, long ldc, long sC, int nbatch,
                        const int *amap, const int *bmap, const int *klen, bool accumulate);

// Split-K policy of the overlap GEMMs.  FP64: the 64x64 output tiles of the
// launch's batches times the K chunks fill one round of the work-groups the
// chip holds with c64 operands (four per CU; their partial sums then fit 64
// MiB), two rounds with c128 ones (three per CU; 514-552 us in two against
// 540-566 in one for four 512 x 512 x 3870), rounded down (57 chunks of 18
// tiles, two work-groups past a round of 1024, took 234 us where 56 took
// 203), in chunks of at least 256 complex terms.  FP32: chunks of at most 512 complex terms, whose FP32 sums are
// exact to the FP32 accumulation of 512 terms, summed in FP64 by the
// reduction (a kernel that instead folds its FP32 sums into FP64 inside
// longer chunks holds 64 more registers per lane and runs at a third of the
// occupancy: 94 against 119 TFLOP/s at 216 atoms).  (The split-plane GEMMs
// chunk K by their plane layout.)  A positive `tune` forces the count.
int splitk_count(int precision, int M, int N, int K, int tune, int nbatch, bool c128) {
  if (tune > 0)
    return tune;
  const int tiles = std::max(1, ((M + 63) / 64) * ((N + 63) / 64) * nbatch);
  int n = precision == PP_FP64 ? (c128 ? 1536 : 1024) / tiles : (1024 + tiles - 1) / tiles;
  if (precision == PP_FP32)
    n = std::max(n, (K + 511) / 512);
  n = std::min(n, std::max(1, K / 256));
  return std::max(1, n);
}

// K chunks of a launch of the batches gb: the batches share the work-groups
// the split policy asks for.
void zgemm64_split(int M, int N, const GemmBatch &gb, int tune, bool c128, int &nsplit, int &kchunk) {
  int K = 0;
  for (int i = 0; i < gb.n; i++)
    K = std::max(K, gb.k[i]);
  nsplit = splitk_count(PP_FP64, M, N, K, tune, gb.n, c128);
  kchunk = (K + nsplit - 1) / nsplit;
  kchunk = std::max(16, (kchunk + 15) / 16 * 16);
  nsplit = std::max(1, (K + kchunk - 1) / kchunk);
}

// Batches of a launch.  A forced chunk count holds that many partial sums for
// each of them: no more batches than keep those within what the policy's own
// counts take (1536 tiles, 96 MiB), or one.
int zgemm64_batches(int M, int N, int tune) {
  const long part = 16L * M * N * std::max(1, tune);
  return tune > 1 ? (int)std::max(1L, std::min<long>(GemmBatch::MAX, (96L << 20) / part)) : GemmBatch::MAX;
}

// FP64 MFMA GEMM of the batches gb: partials dst + batch * sBatch + split *
// sSplit, or with nsplit == 1 the outputs themselves; kchunk a multiple of
// 16.  acol (optional, FP64 operands): column map of A.  No allocation.
int launch_zgemm64(hipStream_t st, int M, int N, const GemmBatch &gb, int atype, const void *A, long lda, long sA,
                   const int *acol, int btype, const void *B, long ldb, long sB, cplx<double> *dst, long dld,
                   long sSplit, long sBatch, int nsplit, int kchunk, bool accumulate) {
  const int tiles = ((M + 63) / 64) * ((N + 63) / 64);
  const dim3 grd = gemm_grid(tiles, nsplit * gb.n);
#define PP_MF(TA, TB, GA)                                                                                      \
  hipLaunchKernelGGL((k_zgemm_mfma64<TA, TB, GA>), grd, dim3(256), 0, st, M, N, kchunk, nsplit, gb,                \
                     (const cplx<TA> *)A, lda, sA, acol, (const cplx<TB> *)B, ldb, sB, dst, dld, sSplit, sBatch,   \
                     accumulate ? 1 : 0)
  if (acol)
    PP_MF(double, double, true);
  else if (atype == 1 && btype == 1)
    PP_MF(float, float, false);
  else if (atype == 0 && btype == 0)
    PP_MF(double, double, false);
  else if (atype == 0 && btype == 1)
    PP_MF(double, float, false);
  else
    PP_MF(float, double, false);
#undef PP_MF
  PP_CHECK_HIP(hipGetLastError());
  return PP_OK;
}

// The VALU form of one batch (the gemm_f64_valu option); acol as
// launch_zgemm64.
int launch_zgemm64_valu(hipStream_t st, int M, int N, int K, int atype, const void *A, long lda, const int *acol,
                        int btype, const void *B, long ldb, cplx<double> *dst, long dld, long sSplit, int nsplit,
                        int kchunk) {
  const dim3 grd = gemm_grid(((M + 63) / 64) * ((N + 63) / 64), nsplit);
#define PP_MV(TA, TB, GA)                                                                                      \
  hipLaunchKernelGGL((k_zgemm_f64<TA, TB, GA>), grd, dim3(256), 0, st, M, N, kchunk, K, nsplit, (const cplx<TA> *)A, \
                     lda, acol, (const cplx<TB> *)B, ldb, dst, dld, sSplit)
  if (acol)
    PP_MV(double, double, true);
  else if (atype == 1 && btype == 1)
    PP_MV(float, float, false);
  else if (atype == 0 && btype == 0)
    PP_MV(double, double, false);
  else if (atype == 0 && btype == 1)
    PP_MV(double, float, false);
  else
    PP_MV(float, double, false);
#undef PP_MV
  PP_CHECK_HIP(hipGetLastError());
  return PP_OK;
}

int launch_splitk_reduce(hipStream_t st, int M, int N, int nsplit, const void *P, bool fp32_partials,
                         cplx<double> *C, long ldc, bool accumulate, int nbatch, long sP, long sC) {
  const dim3 grd((unsigned)(((long)M * N + 255) / 256), (unsigned)nbatch);
  if (fp32_partials)
    hipLaunchKernelGGL(k_splitk_reduce<float>, grd, dim3(256), 0, st, M, N, nsplit, (const cplx<float> *)P, sP, C, ldc,
                       sC, accumulate ? 1 : 0);
  else
    hipLaunchKernelGGL(k_splitk_reduce<double>, grd, dim3(256), 0, st, M, N, nsplit, (const cplx<double> *)P, sP, C,
                       ldc, sC, accumulate ? 1 : 0);
  PP_CHECK_HIP(hipGetLastError());
  return PP_OK;
}

// FP64 GEMM of the batches gb (outputs C + i * sC for batch i of gb).
static int zgemm64_group(pp_ctx *ctx, int M, int N, const GemmBatch &gb, int atype, const void *A, long lda, long sA,
                         const int *acol, int btype, const void *B, long ldb, long sB, cplx<double> *C, long ldc,
                         long sC, bool accumulate, int cls) {
  const bool valu = ctx->tune_gemm_f64_valu != 0;  // one batch a launch (zgemm64_nt)
  int nsplit, kchunk;
  zgemm64_split(M, N, gb, ctx->tune_splitk, atype == 0 && btype == 0, nsplit, kchunk);
  const bool direct = nsplit == 1 && !(valu && accumulate);
  cplx<double> *dst = C;
  long dld = ldc, sSplit = 0, sBatch = sC;
  if (!direct) {
    PP_TRY(ctx->gemm_ws.ensure(sizeof(cplx<double>) * (size_t)nsplit * gb.n * M * N));
    dst = (cplx<double> *)ctx->gemm_ws.p;
    dld = N;
    sSplit = (long)M * N;
    sBatch = sSplit * nsplit;
  }
  const size_t ea = atype == 0 ? 16 : 8, eb = btype == 0 ? 16 : 8;
  hipEvent_t ev;
  tbegin(ctx, cls, &ev);
  int st = valu ? launch_zgemm64_valu(ctx->stream, M, N, gb.k[0], atype, (const char *)A + gb.a[0] * sA * ea, lda, acol,
                                      btype, (const char *)B + gb.b[0] * sB * eb, ldb, dst, dld, sSplit, nsplit, kchunk)
                : launch_zgemm64(ctx->stream, M, N, gb, atype, A, lda, sA, acol, btype, B, ldb, sB, dst, dld, sSplit,
                                 sBatch, nsplit, kchunk, direct && accumulate);
  tend(ctx, cls, ev);
  PP_TRY(st);
  if (!direct) {
    tbegin(ctx, K_GEMM_REDUCE, &ev);
    st = launch_splitk_reduce(ctx->stream, M, N, nsplit, ctx->gemm_ws.p, false, C, ldc, accumulate, gb.n, sBatch, sC);
    tend(ctx, K_GEMM_REDUCE, ev);
  }
  return st;
}

int zgemm64_nt(pp_ctx *ctx, int M, int N, int K, int atype, const void *A, long lda, long sA, const int *acol,
               int btype, const void *B, long ldb, long sB, cplx<double> *C, long ldc, long sC, int nbatch,
               const int *amap, const int *bmap, const int *klen, bool accumulate) {
  if (M <= 0 || N <= 0)
    return PP_OK;
  const int most = ctx->tune_gemm_f64_valu ? 1 : zgemm64_batches(M, N, ctx->tune_splitk);
  for (int b0 = 0; b0 < nbatch; b0 += most) {
    GemmBatch gb;
    gb.n = std::min(most, nbatch - b0);
    for (int i = 0; i < gb.n; i++) {
      gb.a[i] = amap ? amap[b0 + i] : b0 + i;
      gb.b[i] = bmap ? bmap[b0 + i] : b0 + i;
      gb.k[i] = klen ? klen[b0 + i] : K;
    }
    PP_TRY(zgemm64_group(ctx, M, N, gb, atype, A, lda, sA, acol, btype, B, ldb, sB, C + (size_t)b0 * sC, ldc, sC,
                         accumulate, atype == 0 ? K_AUG_GEMM : K_GEMM));
  }
  return PP_OK;
}

int zgemm_nt(pp_ctx *ctx, int precision, int M, int N, int K, int atype, const void *A, long lda, long sA, int btype,
             const void *B, long ldb, long sB, void *C, long ldc, long sC, int nbatch, const int *amap,
             const int *bmap, const int *klen, bool accumulate) {
  if (precision == PP_FP64 || atype != 1 || btype != 1)
    return zgemm64_nt(ctx, M, N, K, atype, A, lda, sA, nullptr, btype, B, ldb, sB, (cplx<double> *)C, ldc, sC, nbatch,
                      amap, bmap, klen, accumulate);
  // FP32 / 3xBF16 batches: the split-K reduction of one batch runs on the
  // second stream while the next batch's GEMM runs (two partials buffers)
  const bool pipe = nbatch > 1 && ctx->tune_streams > 1 && M > 0 && N > 0;
  if (pipe) {
    if (!ctx->aux)
      PP_CHECK_HIP(hipStreamCreateWithFlags(&ctx->aux, hipStreamNonBlocking));
    for (int i = 0; i < 2; i++) {
      if (!ctx->gemm_done[i])
        PP_CHECK_HIP(hipEventCreateWithFlags(&ctx->gemm_done[i], hipEventDisableTiming));
      if (!ctx->red_done[i])
        PP_CHECK_HIP(hipEventCreateWithFlags(&ctx->red_done[i], hipEventDisableTiming));
      PP_CHECK_HIP(hipEventRecord(ctx->red_done[i], ctx->stream));  // no reduction pending yet
    }
    if (!ctx->join)
      PP_CHECK_HIP(hipEventCreateWithFlags(&ctx->join, hipEventDisableTiming));
  }
  int st = PP_OK;
  if (pipe && plane_precision(precision)) {
    st = plane_gemm_pipeline(ctx, precision, M, N, K, A, lda, sA, B, ldb, sB, (cplx<double> *)C, ldc, sC, nbatch,
                             amap, bmap, klen, accumulate);
    (void)hipEventRecord(ctx->join, ctx->aux);
    (void)hipStreamWaitEvent(ctx->stream, ctx->join, 0);
    return st;
  }
  for (int b = 0; b < nbatch && st == PP_OK && M > 0 && N > 0; b++) {
    int ia = amap ? amap[b] : b, ib = bmap ? bmap[b] : b;
    int kk = klen ? klen[b] : K;
    st = gemm_fp32_mfma(ctx, precision, M, N, kk, (const cplx<float> *)A + (size_t)ia * sA, lda,
                        (const cplx<float> *)B + (size_t)ib * sB, ldb, (cplx<double> *)C + (size_t)b * sC, ldc,
                        accumulate, pipe ? (b & 1) : -1);
  }
  if (pipe) {
    // the caller's stream sees every reduction
    (void)hipEventRecord(ctx->join, ctx->aux);
    (void)hipStreamWaitEvent(ctx->stream, ctx->join, 0);
  }
  return st;
}

}  // namespace pp

// Coarsest-level direct solve on the GPU.  Replaces TACSMg's direct coarse
// solve (src/TMR_RefinementTools.cpp:83-86).
//
// Explicit inverses of dense SPD matrices, many at once, by blocked
// Gauss-Jordan: step k turns every 64 x 64 block of A into
//   A_kk <- A_kk^-1,  A_kj <- A_kk^-1 A_kj,  A_ik <- -A_ik A_kk^-1,
//   A_ij <- A_ij - A_ik A_kk^-1 A_kj,
// and after the last block A holds A^-1.  A_kk^-1 is never multiplied as such:
// with A_kk = L D L^T, M = D^-1/2 L^-1 and Y_j = M A_kj the products are M^T M,
// M^T Y_j and Y_i^T Y_j, whose terms stay of the size of A as those of a Cholesky
// factorisation do.  (With the explicit A_kk^-1, entries of 1 / k0 meet small
// couplings: islands of material in void of 1e-8 times the stiffness gave
// residuals of 1e-3 |A| |x|, of 1e-9 a negative pivot; now 6e-17 at 1e-12.)  No
// pivoting: the pivots are those of the Cholesky factorisation of an SPD
// matrix.  A step is one launch over all blocks of all matrices, from one
// buffer to the other, and the workgroup that produces block (k + 1, k + 1)
// also factors it, so that a matrix of nb blocks takes nb + 1 launches.  On the
// way the block (j, i) is the transpose of (i, j), or its negative where k lies
// between them, so only the blocks of the lower triangle are computed and each
// is stored twice, the next pivot block in the first workgroup.  What bounds it
// at the sizes of a coarse level is that chain: the 64 dependent pivots of a
// block (in registers, one barrier each, about 20 us) and the launch, not the
// arithmetic (FP64 matrix cores; three products a block): set-up of 1.2M
// adaptive hex, whose coarsest level takes 16 + 37 steps, 5.9 ms, of the 16^3
// cube with 6 steps 0.48 ms.  It replaced blocked Cholesky, L^-1 and L^-T L^-1
// (about five launches a block column, 54 us of them for the diagonal factor in
// LDS).
//
// Matrices of SCHUR_MIN dofs and more are first split by
// substructuring (coarse.cpp): leaves D_i, separator S,
//   W_i^T = E_i^T D_i^-1,  S <- S - sum_i E_i^T W_i,
// all products through k_gemm_nt, and the solve goes through D_i^-1, W_i and
// S^-1 (k_coarse_rows).
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace tmrx {

namespace {

constexpr int DB = 64;   // block size
constexpr int DT = 256;  // threads per workgroup
// LDS leading dimensions of the matrix-core operands (doubles): rows of a
// half wave's 16 x 2 read fall into distinct banks
constexpr int LDA = 66;  // read as [row][k]
constexpr int LDB = 80;  // read as [k][col]

typedef double f64x4 __attribute__((ext_vector_type(4)));

// wave w of four takes the 32 x 32 quadrant (w / 2, w % 2) of a 64 x 64
// product over 64 inner indices: acc += A^T B, A[k][row] and B[k][col] with
// leading dimension LDB, or (NT) A B^T, A[row][k] and B[col][k] with LDA
template <bool NT>
__device__ __forceinline__ void quad_product(const double *A, const double *B, f64x4 acc[2][2]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r = 32 * (w >> 1) + (lane & 15), c = 32 * (w & 1) + (lane & 15), g = lane >> 4;
#pragma unroll 4
  for (int k = 0; k < DB; k += 4) {
    double a[2], b[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
      a[u] = NT ? A[(r + 16 * u) * LDA + k + g] : A[(k + g) * LDB + r + 16 * u];
      b[u] = NT ? B[(c + 16 * u) * LDA + k + g] : B[(k + g) * LDB + c + 16 * u];
    }
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int v = 0; v < 2; v++)
        acc[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], b[v], acc[u][v], 0, 0, 0);
  }
}
// row and column in the 64 x 64 block of element e of acc[u][v]
__device__ __forceinline__ int quad_row(int u, int e) {
  return 32 * (threadIdx.x >> 7) + 16 * u + 4 * e + ((threadIdx.x & 63) >> 4);
}
__device__ __forceinline__ int quad_col(int v) {
  return 32 * ((threadIdx.x >> 6) & 1) + 16 * v + (threadIdx.x & 15);
}

// 64 x 64 block (leading dimension ld) into LDS
template <int LD>
__device__ __forceinline__ void stage_block(const double *__restrict__ src, int64_t ld, double *dst) {
#pragma unroll
  for (int t = threadIdx.x; t < DB * DB; t += DT) dst[(t >> 6) * LD + (t & 63)] = src[(t >> 6) * ld + (t & 63)];
}

// M = D^-1/2 L^-1 of the SPD block in `blk` (LDS, leading dimension LDA), A = L
// D L^T, so that A^-1 = M^T M: written to out row by row, and its transpose
// behind.  A 4 x 4 piece per thread in registers, L^-1 growing where the
// eliminated columns were, the pivot row and column through LDS (buf: 256
// doubles, two sets in turn, so one barrier a pivot).
__device__ __forceinline__ void factor_block(const double *blk, double *buf, double *__restrict__ out,
                                             int *bad) {
  const int tr = threadIdx.x >> 4, tc = threadIdx.x & 15;
  double a[4][4], di[4] = {1.0, 1.0, 1.0, 1.0};  // 1 / d of the piece's rows
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) a[i][j] = blk[(4 * tr + i) * LDA + 4 * tc + j];
  bool neg = false;
  for (int kb = 0; kb < DB / 4; kb++) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      double *row = buf + 128 * (q & 1), *col = row + 64;
      if (tr == kb)
#pragma unroll
        for (int j = 0; j < 4; j++) row[4 * tc + j] = a[q][j];
      if (tc == kb)
#pragma unroll
        for (int i = 0; i < 4; i++) col[4 * tr + i] = a[i][q];
      __syncthreads();
      const double p = row[4 * kb + q];
      double rv[4], cv[4];
#pragma unroll
      for (int j = 0; j < 4; j++) rv[j] = row[4 * tc + j];
#pragma unroll
      for (int i = 0; i < 4; i++) cv[i] = col[4 * tr + i];
      if (!(p > 0.0)) neg = true;
      // 1 / p by two Newton steps from the hardware estimate: the division's
      // range scaling would lengthen every pivot's chain (neither the estimate
      // nor a step leaves the range for p within 2^-1022 .. 2^1022)
      double d = __builtin_amdgcn_rcp(p);
      d = __builtin_fma(__builtin_fma(-p, d, 1.0), d, d);
      d = __builtin_fma(__builtin_fma(-p, d, 1.0), d, d);
      // rows below the pivot
#pragma unroll
      for (int i = 0; i < 4; i++) cv[i] = tr > kb || (tr == kb && i > q) ? -d * cv[i] : 0.0;
      if (tr == kb) di[q] = d;
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) a[i][j] = __builtin_fma(cv[i], rv[j], a[i][j]);
      if (tc == kb)
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (tr > kb || (tr == kb && i > q)) a[i][q] = cv[i];
    }
  }
  if (neg && threadIdx.x == 0) atomicOr(bad, 1);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const double w = sqrt(di[i]);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int r = 4 * tr + i, c = 4 * tc + j;
      const double m = r > c ? w * a[i][j] : r == c ? w : 0.0;
      out[DB * r + c] = m;
      out[DB * DB + DB * c + r] = m;
    }
  }
}

// problem of block b: last p with tile0[p] <= b
__device__ __forceinline__ int find_prob(const int *__restrict__ tile0, int n, int b) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int m = (lo + hi + 1) >> 1;
    if (tile0[m] <= b)
      lo = m;
    else
      hi = m - 1;
  }
  return lo;
}

}  // namespace

// identity on the padding rows of every matrix
__global__ void k_gj_pad(const GJProb *__restrict__ pr, double *A0, double *A1) {
  const GJProb p = pr[blockIdx.x];
  const int ld = DB * p.nblk, i = p.n + threadIdx.x;
  double *A = ((p.nblk & 1) ? A1 : A0) + p.off;
  if (i < ld) A[(size_t)i * ld + i] = 1.0;
}

// words of a pivot block's factors (M and its transpose), two sets in turn
constexpr int FAC = 2 * DB * DB;

__global__ __launch_bounds__(DT) void k_gj_first(const GJProb *__restrict__ pr, const double *A0,
                                                 const double *A1, double *__restrict__ fac,
                                                 int *bad) {
  __shared__ double blk[DB * LDA], buf[256];
  const GJProb p = pr[blockIdx.x];
  stage_block<LDA>(((p.nblk & 1) ? A1 : A0) + p.off, DB * p.nblk, blk);
  __syncthreads();
  factor_block(blk, buf, fac + (size_t)2 * FAC * blockIdx.x, bad);
}

// w x (the quadrants of a product) into LDS, leading dimension LD
template <int LD>
__device__ __forceinline__ void stage_quads(const f64x4 x[2][2], double w, double *dst) {
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
      for (int e = 0; e < 4; e++) dst[quad_row(u, e) * LD + quad_col(v)] = w * x[u][v][e];
}

__global__ __launch_bounds__(DT) void k_gj_step(int k, int nprob, const GJProb *__restrict__ pr,
                                                const int *__restrict__ tile0, double *A0,
                                                double *A1, double *fac, int *bad) {
  __shared__ double sa[DB * LDB], sb[DB * LDB];
  const int q = find_prob(tile0, nprob, blockIdx.x);
  const GJProb p = pr[q];
  const int nb = p.nblk;
  // the block that goes on to the next factorisation starts with the first
  // wave of workgroups
  int t = blockIdx.x - tile0[q];
  if (k + 1 < nb) {
    const int next = (k + 1) * (k + 4) / 2;
    t = t == 0 ? next : t == next ? 0 : t;
  }
  int i = (int)((sqrtf(8.0f * t + 1.0f) - 1.0f) * 0.5f);
  i += (i + 1) * (i + 2) / 2 <= t;
  i -= i * (i + 1) / 2 > t;
  const int j = t - i * (i + 1) / 2;
  const int64_t ld = DB * nb;
  const double *src = (((nb - k) & 1) ? A1 : A0) + p.off;
  double *dst = (((nb - k - 1) & 1) ? A1 : A0) + p.off;
  const double *M = fac + (size_t)FAC * (2 * q + (k & 1)), *Mt = M + DB * DB;
  double *out = dst + (int64_t)DB * i * ld + DB * j;
  // block (j, i) of the result: the negative of the transpose where one of
  // the two block rows has been through its step and the other has not
  double *mir = dst + (int64_t)DB * j * ld + DB * i;
  const double sign = (i <= k) == (j <= k) ? 1.0 : -1.0;
  f64x4 yj[2][2] = {}, o[2][2] = {};
  if (i == k || j == k) {
    // block row k: M^T (M A_kc), c the other index, or M^T M
    const int c = i == k ? j : i;
    if (c == k) {
      stage_block<LDB>(M, DB, sb);
    } else {
      stage_block<LDB>(Mt, DB, sa);
      stage_block<LDB>(src + (int64_t)DB * k * ld + DB * c, ld, sb);
      __syncthreads();
      quad_product<false>(sa, sb, yj);
      __syncthreads();
      stage_quads<LDB>(yj, 1.0, sb);
    }
    stage_block<LDB>(M, DB, sa);
    __syncthreads();
    quad_product<false>(sa, sb, o);
    double *Nkc = i == k ? out : mir, *Nck = i == k ? mir : out;
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int v = 0; v < 2; v++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          Nkc[quad_row(u, e) * ld + quad_col(v)] = o[u][v][e];
          if (c != k) Nck[quad_col(v) * ld + quad_row(u, e)] = sign * o[u][v][e];
        }
    return;
  }
  // A_ij - A_ik A_kk^-1 A_kj = A_ij -+ Y_i^T Y_j, Y = M A_k. (A_ik is the
  // transpose of A_ki, or its negative where i has been through its step)
  stage_block<LDB>(Mt, DB, sa);
  stage_block<LDB>(src + (int64_t)DB * k * ld + DB * j, ld, sb);
  __syncthreads();
  quad_product<false>(sa, sb, yj);
  __syncthreads();
  if (i != j) {
    f64x4 yi[2][2] = {};
    stage_block<LDB>(src + (int64_t)DB * k * ld + DB * i, ld, sb);
    __syncthreads();
    quad_product<false>(sa, sb, yi);
    __syncthreads();
    stage_quads<LDB>(yi, i < k ? 1.0 : -1.0, sa);
  } else {
    stage_quads<LDB>(yj, i < k ? 1.0 : -1.0, sa);
  }
  stage_quads<LDB>(yj, 1.0, sb);
  const double *Aij = src + (int64_t)DB * i * ld + DB * j;
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
      for (int e = 0; e < 4; e++) o[u][v][e] = Aij[quad_row(u, e) * ld + quad_col(v)];
  __syncthreads();
  quad_product<false>(sa, sb, o);
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        out[quad_row(u, e) * ld + quad_col(v)] = o[u][v][e];
        if (i != j) mir[quad_col(v) * ld + quad_row(u, e)] = sign * o[u][v][e];
      }
  if (i != k + 1 || j != k + 1) return;
  __syncthreads();
  stage_quads<LDA>(o, 1.0, sa);
  __syncthreads();
  factor_block(sa, sb, fac + (size_t)FAC * (2 * q + ((k + 1) & 1)), bad);
}

void launch_gj_inverse(const GJProb *pr, const int *tile0, int nprob, const int *active,
                       const int *tiles, int nsteps, double *A0, double *A1, double *fac,
                       int *bad, hipStream_t st) {
  if (nprob == 0) return;
  hipLaunchKernelGGL(k_gj_pad, dim3(nprob), dim3(DB), 0, st, pr, A0, A1);
  hipLaunchKernelGGL(k_gj_first, dim3(nprob), dim3(DT), 0, st, pr, A0, A1, fac, bad);
  for (int k = 0; k < nsteps; k++)
    hipLaunchKernelGGL(k_gj_step, dim3(tiles[k]), dim3(DT), 0, st, k, active[k], pr, tile0, A0, A1,
                       fac, bad);
  TMRX_LAUNCH_CHECK();
}

// C = A B^T per problem (row-major, dimensions multiples of 64), and C^T into
// a second array where ct >= 0.  A holds couplings of separator nodes to a
// leaf, so most of its 64 x 64 blocks are zero; those are read and skipped
// (the two products of a 9.4k-dof level 533 + 431 us -> 219 + 178).
__global__ __launch_bounds__(DT) void k_gemm_nt(int nprob, const GemmProb *__restrict__ pr,
                                                const int *__restrict__ tile0,
                                                const double *__restrict__ A,
                                                const double *__restrict__ B,
                                                double *__restrict__ C, double *__restrict__ Ct) {
  __shared__ double sa[DB * LDA], sb[DB * LDA];
  const int q = find_prob(tile0, nprob, blockIdx.x);
  const GemmProb p = pr[q];
  const int t = blockIdx.x - tile0[q], nj = p.N / DB, i = t / nj, j = t % nj;
  const double *a = A + p.a + (int64_t)DB * i * p.K, *b = B + p.b + (int64_t)DB * j * p.K;
  f64x4 acc[2][2] = {};
  for (int k = 0; k < p.K; k += DB) {
    __syncthreads();
    double v[DB * DB / DT];
    int any = 0;
#pragma unroll
    for (int e = 0; e < DB * DB / DT; e++) {
      const int s = threadIdx.x + e * DT;
      v[e] = a[(int64_t)(s >> 6) * p.K + k + (s & 63)];
    }
#pragma unroll
    for (int e = 0; e < DB * DB / DT; e++) {
      const int s = threadIdx.x + e * DT;
      sa[(s >> 6) * LDA + (s & 63)] = v[e];
      any |= v[e] != 0.0;
    }
    if (!__syncthreads_or(any)) continue;
    stage_block<LDA>(b + k, p.K, sb);
    __syncthreads();
    quad_product<true>(sa, sb, acc);
  }
#pragma unroll
  for (int u = 0; u < 2; u++)
#pragma unroll
    for (int v = 0; v < 2; v++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int r = DB * i + quad_row(u, e), c = DB * j + quad_col(v);
        C[p.c + (int64_t)r * p.N + c] = acc[u][v][e];
        if (p.ct >= 0) Ct[p.ct + (int64_t)c * p.M + r] = acc[u][v][e];
      }
}

void launch_gemm_nt(int nprob, int ntiles, const GemmProb *pr, const int *tile0, const double *A,
                    const double *B, double *C, double *Ct, hipStream_t st) {
  if (ntiles == 0) return;
  hipLaunchKernelGGL(k_gemm_nt, dim3(ntiles), dim3(DT), 0, st, nprob, pr, tile0, A, B, C, Ct);
  TMRX_LAUNCH_CHECK();
}

// BSR block k into the dense arrays: buf[which[k]] + dst[k], leading
// dimension ld[k] (which 255: dropped)
__global__ void k_coarse_scatter(int nnzb, const double *__restrict__ val,
                                 const uint8_t *__restrict__ which, const int64_t *__restrict__ dst,
                                 const int *__restrict__ ld, double *A0, double *A1, double *Et) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nnzb || which[k] == 255) return;
  double *o = (which[k] == 0 ? A0 : which[k] == 1 ? A1 : Et) + dst[k];
  const double *v = val + 9 * (size_t)k;
  const int64_t l = ld[k];
  for (int p = 0; p < 3; p++)
    for (int q = 0; q < 3; q++) o[p * l + q] = v[3 * p + q];
}

void launch_coarse_scatter(int nnzb, const double *val, const uint8_t *which, const int64_t *dst,
                           const int *ld, double *A0, double *A1, double *Et, hipStream_t st) {
  if (nnzb == 0) return;
  hipLaunchKernelGGL(k_coarse_scatter, dim3((nnzb + 255) / 256), dim3(256), 0, st, nnzb, val, which,
                     dst, ld, A0, A1, Et);
  TMRX_LAUNCH_CHECK();
}

// S[a][b] -= sum_i C_i[loc_i(a)][loc_i(b)] in leaf order, C_i (ldc_i wide)
// holding 3 x 3 blocks of the separator nodes next to leaf i
__global__ void k_schur_sum(int m, int lds, int nleaf, const int *__restrict__ loc,
                            const int64_t *__restrict__ coff, const int *__restrict__ ldc,
                            const double *__restrict__ C, double *__restrict__ S) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)m * m) return;
  const int a = (int)(t / m), b = (int)(t % m), ns = m / 3;
  double s = S[(int64_t)a * lds + b];
  for (int i = 0; i < nleaf; i++) {
    const int la = loc[(int64_t)i * ns + a / 3], lb = loc[(int64_t)i * ns + b / 3];
    if (la < 0 || lb < 0) continue;
    s -= C[coff[i] + (int64_t)(3 * la + a % 3) * ldc[i] + 3 * lb + b % 3];
  }
  S[(int64_t)a * lds + b] = s;
}

void launch_schur_sum(int m, int lds, int nleaf, const int *loc, const int64_t *coff,
                      const int *ldc, const double *C, double *S, hipStream_t st) {
  if (m == 0) return;
  const int64_t n = (int64_t)m * m;
  hipLaunchKernelGGL(k_schur_sum, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, m, lds, nleaf,
                     loc, coff, ldc, C, S);
  TMRX_LAUNCH_CHECK();
}

// One stage of the substructured solve, one wave per row: s = sum over the
// row's segments of M[a + j] v[idx[j]], FP64.
//   stage 1: v = b; leaf rows tmp = s, separator rows tmp = b[dof] - s
//   stage 2: v = tmp; x[dof] = xs[pos] = s
//   stage 3: v = xs; x[dof] = tmp[pos] - s
template <class T, class TA, int STAGE>
__global__ __launch_bounds__(256) void k_coarse_rows(int nrows, const CoarseRow *__restrict__ rows,
                                                     const CoarseSeg *__restrict__ segs,
                                                     const int *__restrict__ idx,
                                                     const TA *__restrict__ M,
                                                     const T *__restrict__ b, T *__restrict__ x,
                                                     double *__restrict__ tmp,
                                                     double *__restrict__ xs, int n, int ntmp,
                                                     int nxs, const int *__restrict__ run) {
  if (run && *run == 0) return;
  const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (r >= nrows) return;
  b += (int64_t)blockIdx.y * n;
  x += (int64_t)blockIdx.y * n;
  tmp += (int64_t)blockIdx.y * ntmp;
  xs += (int64_t)blockIdx.y * nxs;
  const CoarseRow row = rows[r];
  double s = 0.0;
  for (int g = row.seg0; g < row.seg1; g++) {
    const CoarseSeg sg = segs[g];
    const TA *__restrict__ a = M + sg.a;
    const int *__restrict__ ix = idx + sg.idx;
    // eight entries per lane in flight (clamped to the segment, extra terms
    // skipped)
    for (int j0 = lane; j0 < sg.len; j0 += 8 * 64) {
      double av[8], bv[8];
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const int j = min(j0 + 64 * k, sg.len - 1);
        av[k] = (double)a[j];
        const int i = ix[j];
        bv[k] = STAGE == 1 ? (double)b[i] : STAGE == 2 ? tmp[i] : xs[i];
      }
#pragma unroll
      for (int k = 0; k < 8; k++)
        if (j0 + 64 * k < sg.len) s += av[k] * bv[k];
    }
  }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if (lane != 0) return;
  if (STAGE == 1) {
    tmp[row.pos] = row.dof >= 0 ? (double)b[row.dof] - s : s;
  } else if (STAGE == 2) {
    xs[row.pos] = s;
    x[row.dof] = (T)s;
  } else {
    x[row.dof] = (T)(tmp[row.pos] - s);
  }
}

template <class T, class TA>
static void coarse_stages(const CoarseBlocks &cb, const TA *M, const T *b, T *x, hipStream_t st,
                          int nrhs) {
#define TMRX_STAGE(S)                                                                             \
  if (cb.nrow[S - 1])                                                                             \
  hipLaunchKernelGGL((k_coarse_rows<T, TA, S>), dim3((cb.nrow[S - 1] + 3) / 4, nrhs), dim3(256),  \
                     0, st, cb.nrow[S - 1], cb.row[S - 1], cb.seg, cb.idx, M, b, x, cb.tmp,       \
                     cb.xs, cb.n, cb.ntmp, cb.nxs, cb.run)
  TMRX_STAGE(1);
  TMRX_STAGE(2);
  TMRX_STAGE(3);
#undef TMRX_STAGE
  TMRX_LAUNCH_CHECK();
}

template <class T>
void launch_coarse_schur(const CoarseBlocks &cb, const T *b, T *x, hipStream_t st, int nrhs) {
  if (sizeof(T) == 4 && cb.Ainv32)
    coarse_stages<T, float>(cb, cb.Ainv32, b, x, st, nrhs);
  else
    coarse_stages<T, double>(cb, cb.Ainv, b, x, st, nrhs);
}
template void launch_coarse_schur<float>(const CoarseBlocks &, const float *, float *, hipStream_t,
                                         int);
template void launch_coarse_schur<double>(const CoarseBlocks &, const double *, double *,
                                          hipStream_t, int);

}  // namespace tmrx

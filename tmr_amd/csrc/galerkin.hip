// Galerkin coarse operators (TMR_CreateTACSMg with use_galerkin,
// src/TMR_RefinementTools.cpp:37-107: TACSMg forms P^T A P) on the GPU.
//
// Every element e of a finer level lies inside one element E of the next
// coarser level, and the prolongation restricted to e is the trilinear
// interpolation Q_e of E's corners at e's corners (hanging corners included:
// their constraint is the same trilinear interpolation on a coarser face or
// edge).  So P^T Z_f^T K_f Z_f P = Z_c^T (sum_E K_E) Z_c with the element
// matrices
//   K_E = sum_{e in E} (Q_e x I3)^T K_e (Q_e x I3),
// computed level by level (k_galerkin_elem), then assembled into a 3 x 3
// block-sparse (BSR) matrix over the independent nodes of the coarse level
// with the hanging-node expansion Z_c and identity rows and columns on the
// clamped dofs (k_bsr_assemble).  The block sums follow fixed term lists,
// so the operator is the same bit for bit on every setup.
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace tmrx {

// ---------------------------------------------------------------------------
// K_E of every coarse element: one workgroup per element, the 576 entries
// spread over its threads.  MODE 0: children are finest-level elements of
// element densities, K_e = s_e K0[class]; MODE 1: children carry their own
// matrices Kin[e]; MODE 2: finest-level elements of a nodal design,
// K_e = sum_g s_eg Kg[class][g].
constexpr int GAL_THREADS = 256;

template <int MODE>
__global__ void __launch_bounds__(GAL_THREADS)
    k_galerkin_elem(int nE, const int *__restrict__ ptr, const int *__restrict__ child,
                    const int *__restrict__ place, const int *__restrict__ cls,
                    const double *__restrict__ s, const double *__restrict__ Ktab,
                    const double *__restrict__ Kin, double *__restrict__ Kout) {
  __shared__ double A[576], B[576], Q[64];
  const int E = blockIdx.x;
  if (E >= nE) return;
  const int tid = threadIdx.x;
  double acc[3] = {0.0, 0.0, 0.0};
  for (int k = ptr[E]; k < ptr[E + 1]; k++) {
    const int e = child[k];
    if (tid < 64) {
      // trilinear weight of coarse corner c at fine corner a
      const int pl = place[k];
      const int dl = (pl >> 24) & 15;
      const double inv = 1.0 / (double)(1 << dl);
      const int a = tid >> 3, c = tid & 7;
      const int off[3] = {pl & 255, (pl >> 8) & 255, (pl >> 16) & 255};
      double w = 1.0;
      for (int d = 0; d < 3; d++) {
        const double xi = (double)(off[d] + ((a >> d) & 1)) * inv;
        w *= ((c >> d) & 1) ? xi : 1.0 - xi;
      }
      Q[8 * a + c] = w;
    }
    for (int t = tid; t < 576; t += GAL_THREADS) {
      double v;
      if (MODE == 0) {
        v = s[e] * Ktab[576 * (size_t)cls[e] + t];
      } else if (MODE == 1) {
        v = Kin[576 * (size_t)e + t];
      } else {
        const double *Kg = Ktab + 576 * 8 * (size_t)cls[e];
        v = 0.0;
#pragma unroll
        for (int g = 0; g < 8; g++) v += s[8 * (size_t)e + g] * Kg[576 * g + t];
      }
      A[t] = v;
    }
    __syncthreads();
    // B = A (Q x I3): B[(3a+i)][(3c+j)] = sum_b A[(3a+i)][(3b+j)] Q[b][c]
    for (int t = tid; t < 576; t += GAL_THREADS) {
      const int row = t / 24, col = t % 24, c = col / 3, j = col % 3;
      double v = 0.0;
#pragma unroll
      for (int b = 0; b < 8; b++) v += A[24 * row + 3 * b + j] * Q[8 * b + c];
      B[t] = v;
    }
    __syncthreads();
    // K_E += (Q x I3)^T B
    int u = 0;
    for (int t = tid; t < 576; t += GAL_THREADS, u++) {
      const int row = t / 24, col = t % 24, c = row / 3, i = row % 3;
      double v = 0.0;
#pragma unroll
      for (int a = 0; a < 8; a++) v += Q[8 * a + c] * B[24 * (3 * a + i) + col];
      acc[u] += v;
    }
    __syncthreads();
  }
  int u = 0;
  for (int t = tid; t < 576; t += GAL_THREADS, u++) Kout[576 * (size_t)E + t] = acc[u];
}

void launch_galerkin_elem(int mode, int nE, const int *ptr, const int *child, const int *place,
                          const int *cls, const double *s, const double *Ktab, const double *Kin,
                          double *Kout, hipStream_t st) {
  if (nE == 0) return;
  if (mode == 0)
    hipLaunchKernelGGL(k_galerkin_elem<0>, dim3(nE), dim3(GAL_THREADS), 0, st, nE, ptr, child,
                       place, cls, s, Ktab, Kin, Kout);
  else if (mode == 1)
    hipLaunchKernelGGL(k_galerkin_elem<1>, dim3(nE), dim3(GAL_THREADS), 0, st, nE, ptr, child,
                       place, cls, s, Ktab, Kin, Kout);
  else
    hipLaunchKernelGGL(k_galerkin_elem<2>, dim3(nE), dim3(GAL_THREADS), 0, st, nE, ptr, child,
                       place, cls, s, Ktab, Kin, Kout);
  TMRX_LAUNCH_CHECK();
}

// element matrices from scales, one thread per (element, entry)
__global__ void k_elem_matrices(int ne, const int *__restrict__ cls, const double *__restrict__ s,
                                const double *__restrict__ Ktab, int nodal,
                                double *__restrict__ KE) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 576 * (int64_t)ne) return;
  const int e = (int)(t / 576), i = (int)(t % 576);
  double v;
  if (nodal) {
    const double *Kg = Ktab + 576 * 8 * (size_t)cls[e] + i;
    v = 0.0;
    for (int g = 0; g < 8; g++) v += s[8 * (size_t)e + g] * Kg[576 * g];
  } else {
    v = s[e] * Ktab[576 * (size_t)cls[e] + i];
  }
  KE[t] = v;
}

void launch_elem_matrices(int ne, const int *cls, const double *s, const double *Ktab, bool nodal,
                          double *KE, hipStream_t st) {
  if (ne == 0) return;
  const int64_t n = 576 * (int64_t)ne;
  hipLaunchKernelGGL(k_elem_matrices, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, ne, cls,
                     s, Ktab, nodal ? 1 : 0, KE);
  TMRX_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// BSR values: block k (row node i = brow[k], column node j = col[k]) is the
// sum over its terms of w * K_E[(3a+p)][(3b+q)], term code = 64 E + 8 a + b;
// rows and columns of clamped dofs become identity rows and columns.
// One thread per entry, so that a block's nine entries load side by side, and
// four terms in flight per thread (one thread per block, a term at a time:
// 988,000 blocks of a 38,549-node level 799 us, now 550).
__global__ __launch_bounds__(256) void k_bsr_assemble(int nblk, const int *__restrict__ tptr,
                                                      const int *__restrict__ tcode,
                                                      const double *__restrict__ tw,
                                                      const int *__restrict__ brow,
                                                      const int *__restrict__ col,
                                                      const double *__restrict__ KE,
                                                      const uint8_t *__restrict__ bcmask,
                                                      double *__restrict__ val) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= 9 * (int64_t)nblk) return;
  const int k = (int)(t / 9), e = (int)(t % 9), p = e / 3, q = e % 3;
  const int i = brow[k], j = col[k];
  const int t0 = tptr[k], t1 = tptr[k + 1];
  double v = 0.0;
  for (int u0 = t0; u0 < t1; u0 += 4) {
    double w[4], a[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int x = min(u0 + u, t1 - 1), code = tcode[x];
      w[u] = tw[x];
      a[u] = KE[576 * (size_t)(code >> 6) + 24 * (3 * ((code >> 3) & 7) + p) + 3 * (code & 7) + q];
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (u0 + u < t1) v += w[u] * a[u];
  }
  if (((bcmask[i] >> p) & 1) || ((bcmask[j] >> q) & 1)) v = (i == j && p == q) ? 1.0 : 0.0;
  val[t] = v;
}

void launch_bsr_assemble(const BSR64 &A, const int *tptr, const int *tcode, const double *tw,
                         const int *brow, const double *KE, double *val, hipStream_t st) {
  if (A.nnzb == 0) return;
  hipLaunchKernelGGL(k_bsr_assemble, dim3((unsigned)((9 * (int64_t)A.nnzb + 255) / 256)), dim3(256),
                     0, st, A.nnzb, tptr, tcode, tw, brow, A.col, KE, A.bcmask, val);
  TMRX_LAUNCH_CHECK();
}

// Jacobi diagonal from the diagonal blocks (clamped dofs have 1 there)
template <class T>
__global__ void k_bsr_dinv(int n, const int *__restrict__ diag, const double *__restrict__ val,
                           T *__restrict__ dinv) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double *v = val + 9 * (size_t)diag[i];
#pragma unroll
  for (int p = 0; p < 3; p++) dinv[3 * (size_t)i + p] = (T)(1.0 / v[4 * p]);
}

template <class T>
void launch_bsr_dinv(int n, const int *diag, const double *val, T *dinv, hipStream_t st) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_bsr_dinv<T>, dim3((n + 255) / 256), dim3(256), 0, st, n, diag, val, dinv);
  TMRX_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// BSR operator with the epilogues of the tile apply: LANES lanes per block
// row, each summing every LANES-th block of the row two at a time, then a
// butterfly over the group in a fixed order.  32 lanes while one right-hand
// side's rows fit the chip (the loop over a row is a chain of dependent
// loads), else 8; the number of right-hand sides does not count, so that a
// load case is summed in the same order in a batch as by itself.
template <class T, int MODE, int LANES>
__global__ void __launch_bounds__(256)
    k_bsr_apply(int n, const int *__restrict__ ptr, const int *__restrict__ col,
                const T *__restrict__ val, const uint8_t *__restrict__ bcmask,
                const T *__restrict__ x, const T *__restrict__ b, T *__restrict__ y,
                T *__restrict__ x_out, T *__restrict__ d, const T *__restrict__ dinv,
                const T *__restrict__ cf, int cflags, const int *__restrict__ run, int64_t vs) {
  if (run && *run == 0) return;
  const T ca = MODE == ASM_CHEB ? cf[0] : T(0), cc = MODE == ASM_CHEB ? cf[1] : T(0);
  const int64_t off = (int64_t)blockIdx.y * vs;
  x += off;
  if (b) b += off;
  if (y) y += off;
  if (x_out) x_out += off;
  if (d) d += off;
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  const int row = g / LANES, sub = g % LANES;
  const bool valid = row < n;
  T a0 = T(0), a1 = T(0), a2 = T(0);
  if (valid) {
    const int k1 = ptr[row + 1];
    for (int k = ptr[row] + sub; k < k1; k += 2 * LANES) {
      const int kb = min(k + LANES, k1 - 1);
      const bool second = k + LANES < k1;
      const int ja = col[k], jb = col[kb];
      T va[9], vb[9], xa[3], xb[3];
#pragma unroll
      for (int e = 0; e < 9; e++) va[e] = val[9 * (size_t)k + e];
      if (second)
#pragma unroll
        for (int e = 0; e < 9; e++) vb[e] = val[9 * (size_t)kb + e];
#pragma unroll
      for (int c = 0; c < 3; c++) {
        xa[c] = x[3 * (size_t)ja + c];
        xb[c] = x[3 * (size_t)jb + c];
      }
      a0 += va[0] * xa[0] + va[1] * xa[1] + va[2] * xa[2];
      a1 += va[3] * xa[0] + va[4] * xa[1] + va[5] * xa[2];
      a2 += va[6] * xa[0] + va[7] * xa[1] + va[8] * xa[2];
      if (second) {
        a0 += vb[0] * xb[0] + vb[1] * xb[1] + vb[2] * xb[2];
        a1 += vb[3] * xb[0] + vb[4] * xb[1] + vb[5] * xb[2];
        a2 += vb[6] * xb[0] + vb[7] * xb[1] + vb[8] * xb[2];
      }
    }
  }
#pragma unroll
  for (int m = 1; m < LANES; m <<= 1) {
    a0 += __shfl_xor(a0, m);
    a1 += __shfl_xor(a1, m);
    a2 += __shfl_xor(a2, m);
  }
  if (!valid || sub != 0) return;
  const size_t k3 = 3 * (size_t)row;
  const uint8_t msk = bcmask[row];
  const T a[3] = {a0, a1, a2};
  T yo[3], dno[3];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const bool bc = (msk >> c) & 1;
    if (MODE == ASM_STORE) {
      yo[c] = bc ? x[k3 + c] : a[c];
    } else if (MODE == ASM_POWER) {
      yo[c] = dinv[k3 + c] * (bc ? x[k3 + c] : a[c]);
    } else if (MODE == ASM_RESID) {
      yo[c] = bc ? T(0) : b[k3 + c] - a[c];
    } else {  // ASM_CHEB
      if (bc) {
        dno[c] = T(0);
        yo[c] = T(0);
      } else {
        const T r = b[k3 + c] - a[c];
        const T xc = x[k3 + c];
        const T dp = (cflags & CHEB_D_IS_X) ? xc : ((cflags & CHEB_D_READ) ? d[k3 + c] : T(0));
        const T dn = ca * dp + cc * dinv[k3 + c] * r;
        dno[c] = dn;
        yo[c] = xc + dn;
      }
    }
  }
  if (MODE == ASM_CHEB) {
    if (cflags & CHEB_D_STORE)
#pragma unroll
      for (int c = 0; c < 3; c++) d[k3 + c] = dno[c];
#pragma unroll
    for (int c = 0; c < 3; c++) x_out[k3 + c] = yo[c];
  } else {
#pragma unroll
    for (int c = 0; c < 3; c++) y[k3 + c] = yo[c];
  }
}

// rows of 32 lanes that fill the 256 CUs with at most 8 workgroups each
static bool wide_rows(int n) { return (int64_t)n * 32 <= 256 * 8 * 256; }

template <class T, int MODE>
static void bsr_launch(const BSR<T> &A, const T *x, const AsmArgs &g, hipStream_t st, int nrhs,
                       int64_t vs) {
  const bool wide = wide_rows(A.n);
  const int lanes = wide ? 32 : 8;
  const dim3 grid((unsigned)(((int64_t)A.n * lanes + 255) / 256), (unsigned)nrhs);
  if (wide)
    hipLaunchKernelGGL((k_bsr_apply<T, MODE, 32>), grid, dim3(256), 0, st, A.n, A.ptr, A.col, A.val,
                       A.bcmask, x, (const T *)g.b, (T *)g.y, (T *)g.x_out, (T *)g.d,
                       (const T *)g.dinv, (const T *)g.cf, g.cflags, A.run, vs);
  else
    hipLaunchKernelGGL((k_bsr_apply<T, MODE, 8>), grid, dim3(256), 0, st, A.n, A.ptr, A.col, A.val,
                       A.bcmask, x, (const T *)g.b, (T *)g.y, (T *)g.x_out, (T *)g.d,
                       (const T *)g.dinv, (const T *)g.cf, g.cflags, A.run, vs);
}

template <class T>
void launch_bsr_apply(const BSR<T> &A, const T *x, int mode, const AsmArgs &g, hipStream_t st,
                      int nrhs, int64_t vs) {
  if (A.n == 0) return;
  switch (mode) {
    case ASM_STORE: bsr_launch<T, ASM_STORE>(A, x, g, st, nrhs, vs); break;
    case ASM_RESID: bsr_launch<T, ASM_RESID>(A, x, g, st, nrhs, vs); break;
    case ASM_POWER: bsr_launch<T, ASM_POWER>(A, x, g, st, nrhs, vs); break;
    case ASM_CHEB: bsr_launch<T, ASM_CHEB>(A, x, g, st, nrhs, vs); break;
    default: note_launch(hipErrorInvalidValue);
  }
  TMRX_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
constexpr int SOR_TAIL_MAX = 8, SOR_TAIL_ROWS = 32;

// One colour of a point SOR sweep on the BSR matrix (TACSGaussSeidel's
// smoother, symmetric SOR with relaxation omega; TMR_CreateTACSMg,
// src/TMR_RefinementTools.cpp:93-94).  The matrix is the level's BSR with
// its rows in the sweep's colour-major node order (row k holds node
// nodes[k]; columns are node indices), so a colour's rows are contiguous.
// Every node of the colour takes LANES lanes: they sum the row's
// off-diagonal blocks (consecutive lanes on consecutive blocks, which read x
// of other colours only, so the nodes of a colour update side by side) and a
// butterfly combines them; then the node's three dofs update one after
// another through the diagonal block, 0, 1, 2 (backward: 2, 1, 0), each
// x_p <- (1 - omega) x_p + omega (b_p - sum_{q != p} a_pq x_q) / a_pp --
// the point SOR of the dofs in colour-major node order.
// DIR 0: forward, 1: backward, 2: forward then backward, the turn of a
// symmetric sweep (the last colour's neighbours do not change in between).
// A colour is a chain of dependent loads (row, columns, x): with 8 lanes a
// row of 27 to 60 blocks goes round that chain four to eight times, with 32
// once or twice.  32 lanes are taken until they fill the chip (32,858-node
// adaptive level, 2,200 rows a colour: 6.9 -> 4.9 us a launch; one colour of
// 3,058 nodes 5.3 -> 4.1); beyond, 8 lanes leave fewer idle.

// row i (blocks q0 .. q1) on lane `sub` of its LANES
template <class T, int DIR, int LANES>
__device__ __forceinline__ void sor_row(bool valid, int sub, int i, int q0, int q1,
                                        const int *__restrict__ col, const T *__restrict__ val,
                                        const T *__restrict__ b, T *x, T omega) {
  const size_t i3 = 3 * (size_t)i;
  T xi[3] = {T(0), T(0), T(0)}, bi[3] = {T(0), T(0), T(0)};
  if (valid && sub == 0) {
#pragma unroll
    for (int c = 0; c < 3; c++) {
      xi[c] = x[i3 + c];
      bi[c] = b[i3 + c];
    }
  }
  T s0 = T(0), s1 = T(0), s2 = T(0);
  int kd = -1;
  if (valid) {
    // two blocks per lane at a time, loads issued together (the second index
    // clamped to the row, its term skipped past the end)
    for (int q = q0 + sub; q < q1; q += 2 * LANES) {
      const int qb = min(q + LANES, q1 - 1);
      const bool second = q + LANES < q1;
      const int ja = col[q], jb = col[qb];
      T va[9], vb[9], xa[3], xb[3];
#pragma unroll
      for (int e = 0; e < 9; e++) va[e] = val[9 * (size_t)q + e];
      if (second)
#pragma unroll
        for (int e = 0; e < 9; e++) vb[e] = val[9 * (size_t)qb + e];
#pragma unroll
      for (int c = 0; c < 3; c++) {
        xa[c] = x[3 * (size_t)ja + c];
        xb[c] = x[3 * (size_t)jb + c];
      }
      if (ja == i) {
        kd = q;
      } else {
        s0 += va[0] * xa[0] + va[1] * xa[1] + va[2] * xa[2];
        s1 += va[3] * xa[0] + va[4] * xa[1] + va[5] * xa[2];
        s2 += va[6] * xa[0] + va[7] * xa[1] + va[8] * xa[2];
      }
      if (second) {
        if (jb == i) {
          kd = qb;
        } else {
          s0 += vb[0] * xb[0] + vb[1] * xb[1] + vb[2] * xb[2];
          s1 += vb[3] * xb[0] + vb[4] * xb[1] + vb[5] * xb[2];
          s2 += vb[6] * xb[0] + vb[7] * xb[1] + vb[8] * xb[2];
        }
      }
    }
  }
#pragma unroll
  for (int m = 1; m < LANES; m <<= 1) {
    s0 += __shfl_xor(s0, m);
    s1 += __shfl_xor(s1, m);
    s2 += __shfl_xor(s2, m);
    kd = max(kd, __shfl_xor(kd, m));
  }
  if (!valid || sub != 0 || kd < 0) return;
  T D[9];
#pragma unroll
  for (int e = 0; e < 9; e++) D[e] = val[9 * (size_t)kd + e];
  const T r[3] = {bi[0] - s0, bi[1] - s1, bi[2] - s2};
#pragma unroll
  for (int t = 0; t < (DIR == 2 ? 6 : 3); t++) {
    const int p = DIR == 1 ? 2 - t : t < 3 ? t : 5 - t;
    T acc = r[p];
#pragma unroll
    for (int q = 0; q < 3; q++)
      if (q != p) acc -= D[3 * p + q] * xi[q];
    xi[p] = (T(1) - omega) * xi[p] + omega * acc / D[4 * p];
  }
#pragma unroll
  for (int c = 0; c < 3; c++) x[i3 + c] = xi[c];
}

template <class T, int DIR, int LANES>
__global__ __launch_bounds__(256) void k_sor_colour(int cnt, const int *__restrict__ nodes,
                                                    const int *__restrict__ ptr,
                                                    const int *__restrict__ col,
                                                    const T *__restrict__ val,
                                                    const T *__restrict__ b, T *__restrict__ x,
                                                    T omega, const int *__restrict__ run,
                                                    int64_t vs) {
  const int go = run ? *run : 1;
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = g / LANES, sub = g % LANES;
  const bool valid = k < cnt;
  const int64_t off = (int64_t)blockIdx.y * vs;
  const int kk = valid ? k : 0;
  const int i = nodes[kk], q0 = ptr[kk], q1 = ptr[kk + 1];
  if (go == 0) return;
  sor_row<T, DIR, LANES>(valid, sub, i, q0, q1, col, val, b + off, x + off, omega);
}

// The last colours of a sweep, forward, the turn and backward, in one
// workgroup per right-hand side with a barrier in place of a launch between
// colours.  Greedy colouring leaves a few colours of a few nodes at the end
// (hanging corners make cliques), and each was a launch of 4.3 us for one or
// two rounds of loads.  SOR_TAIL_ROWS is one round of 32 lanes a row: a round
// takes about 2.3 us, so a second one costs what the launch did (adaptive
// 50k hex, 22 iterations: 22.8 ms with launches alone, 22.1 with 32 or 64
// rows, 22.5 with 96).
struct SorTail {
  int n, ptr[SOR_TAIL_MAX + 1];  // rows of the n last colours
};
template <class T, int DIR>
__device__ __forceinline__ void sor_tail_colour(int r0, int r1, const int *__restrict__ nodes,
                                                const int *__restrict__ ptr,
                                                const int *__restrict__ col,
                                                const T *__restrict__ val,
                                                const T *__restrict__ b, T *x, T omega) {
  for (int r = r0 + (threadIdx.x >> 5); r < r1; r += 32)
    sor_row<T, DIR, 32>(true, threadIdx.x & 31, nodes[r], ptr[r], ptr[r + 1], col, val, b, x, omega);
  __syncthreads();
}
template <class T>
__global__ __launch_bounds__(1024) void k_sor_tail(SorTail t, const int *__restrict__ nodes,
                                                   const int *__restrict__ ptr,
                                                   const int *__restrict__ col,
                                                   const T *__restrict__ val,
                                                   const T *__restrict__ b, T *x, T omega,
                                                   const int *__restrict__ run, int64_t vs) {
  if (run && *run == 0) return;
  b += (int64_t)blockIdx.y * vs;
  x += (int64_t)blockIdx.y * vs;
  for (int c = 0; c + 1 < t.n; c++)
    sor_tail_colour<T, 0>(t.ptr[c], t.ptr[c + 1], nodes, ptr, col, val, b, x, omega);
  sor_tail_colour<T, 2>(t.ptr[t.n - 1], t.ptr[t.n], nodes, ptr, col, val, b, x, omega);
  for (int c = t.n - 2; c >= 0; c--)
    sor_tail_colour<T, 1>(t.ptr[c], t.ptr[c + 1], nodes, ptr, col, val, b, x, omega);
}

// val_out[k] = val[map[k]] for every 3 x 3 block (the colour-major copy)
__global__ void k_bsr_gather(int nnzb, const int *__restrict__ map, const double *__restrict__ val,
                             double *__restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 9 * (int64_t)nnzb) return;
  const int64_t k = t / 9, e = t % 9;
  out[t] = val[9 * (int64_t)map[k] + e];
}

void launch_bsr_gather(int nnzb, const int *map, const double *val, double *out, hipStream_t st) {
  if (nnzb == 0) return;
  const int64_t n = 9 * (int64_t)nnzb;
  hipLaunchKernelGGL(k_bsr_gather, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, nnzb, map,
                     val, out);
  TMRX_LAUNCH_CHECK();
}

template <class T, int DIR>
static void sor_colour(const BSR<T> &A, const int *nodes, int c0, int cnt, const T *b, T *x,
                       double omega, hipStream_t st, int nrhs, int64_t vs) {
  if (cnt == 0) return;
  const bool wide = wide_rows(cnt);
  const int lanes = wide ? 32 : 8;
  const dim3 grid((unsigned)(((int64_t)cnt * lanes + 255) / 256), (unsigned)nrhs);
  if (wide)
    hipLaunchKernelGGL((k_sor_colour<T, DIR, 32>), grid, dim3(256), 0, st, cnt, nodes + c0,
                       A.ptr + c0, A.col, A.val, b, x, (T)omega, A.run, vs);
  else
    hipLaunchKernelGGL((k_sor_colour<T, DIR, 8>), grid, dim3(256), 0, st, cnt, nodes + c0,
                       A.ptr + c0, A.col, A.val, b, x, (T)omega, A.run, vs);
  TMRX_LAUNCH_CHECK();
}

template <class T>
void launch_sor_symmetric(const BSR<T> &A, const int *nodes, const int *cptr, int ncolors,
                          const T *b, T *x, double omega, hipStream_t st, int nrhs, int64_t vs) {
  if (ncolors == 0) return;
  // colours from t0 on go to the one-workgroup form
  int t0 = ncolors;
  while (t0 > 0 && ncolors - t0 < SOR_TAIL_MAX && cptr[t0] - cptr[t0 - 1] <= SOR_TAIL_ROWS) t0--;
  if (t0 > ncolors - 2) t0 = ncolors - 1;  // the turn alone
  for (int c = 0; c < t0; c++)
    sor_colour<T, 0>(A, nodes, cptr[c], cptr[c + 1] - cptr[c], b, x, omega, st, nrhs, vs);
  if (t0 == ncolors - 1) {
    sor_colour<T, 2>(A, nodes, cptr[t0], cptr[t0 + 1] - cptr[t0], b, x, omega, st, nrhs, vs);
  } else {
    SorTail t{ncolors - t0, {}};
    for (int c = 0; c <= t.n; c++) t.ptr[c] = cptr[t0 + c];
    hipLaunchKernelGGL(k_sor_tail<T>, dim3(1, (unsigned)nrhs), dim3(1024), 0, st, t, nodes, A.ptr,
                       A.col, A.val, b, x, (T)omega, A.run, vs);
    TMRX_LAUNCH_CHECK();
  }
  for (int c = t0 - 1; c >= 0; c--)
    sor_colour<T, 1>(A, nodes, cptr[c], cptr[c + 1] - cptr[c], b, x, omega, st, nrhs, vs);
}

template void launch_sor_symmetric<float>(const BSR<float> &, const int *, const int *, int,
                                          const float *, float *, double, hipStream_t, int,
                                          int64_t);
template void launch_sor_symmetric<double>(const BSR<double> &, const int *, const int *, int,
                                           const double *, double *, double, hipStream_t, int,
                                           int64_t);
template void launch_bsr_dinv<float>(int, const int *, const double *, float *, hipStream_t);
template void launch_bsr_dinv<double>(int, const int *, const double *, double *, hipStream_t);
template void launch_bsr_apply<float>(const BSR<float> &, const float *, int, const AsmArgs &,
                                      hipStream_t, int, int64_t);
template void launch_bsr_apply<double>(const BSR<double> &, const double *, int, const AsmArgs &,
                                       hipStream_t, int, int64_t);

}  // namespace tmrx

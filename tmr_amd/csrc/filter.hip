// Kernels of the design filters (filter.cpp): scalar CSR product, vector
// updates and fixed-order block reductions.
#include <hip/hip_runtime.h>

#include "filter.h"
#include "kernels.h"

namespace tmrx {

constexpr int FB = 256;
static inline dim3 grid_of(int n) { return dim3((unsigned)((n + FB - 1) / FB)); }

// Rows hold 27 entries and more, read through a chain of dependent loads
// (column, then x): eight lanes a row with two entries each in flight, in
// place of one thread, take the product of 9,537 rows from 12.2 to 4.4 us.
constexpr int FL = 8;  // lanes per row
static inline dim3 grid_rows(int n) {
  return dim3((unsigned)(((int64_t)n * FL + FB - 1) / FB));
}

// sum over row i of val[k] x[col[k]], in every lane of the row's group
__device__ __forceinline__ double row_sum(int i, int n, const int *__restrict__ ptr,
                                          const int *__restrict__ col,
                                          const double *__restrict__ val, const double *x) {
  double s = 0.0;
  if (i < n) {
    const int k1 = ptr[i + 1];
    for (int k = ptr[i] + (int)(threadIdx.x % FL); k < k1; k += 2 * FL) {
      const int kb = min(k + FL, k1 - 1);
      const int ca = col[k], cb = col[kb];
      const double va = val[k], vb = val[kb], xa = x[ca], xb = x[cb];
      s += va * xa;
      if (k + FL < k1) s += vb * xb;
    }
  }
#pragma unroll
  for (int m = 1; m < FL; m <<= 1) s += __shfl_xor(s, m);
  return s;
}

__global__ void k_filter_spmv(int n, const int *__restrict__ ptr, const int *__restrict__ col,
                              const double *__restrict__ val, const double *__restrict__ x,
                              double *__restrict__ y) {
  const int i = (int)(((int64_t)blockIdx.x * FB + threadIdx.x) / FL);
  const double s = row_sum(i, n, ptr, col, val, x);
  if (i < n && threadIdx.x % FL == 0) y[i] = s;
}
void launch_filter_spmv(int n, const int *ptr, const int *col, const double *val,
                        const double *x, double *y, hipStream_t st) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_filter_spmv, grid_rows(n), dim3(FB), 0, st, n, ptr, col, val, x, y);
  TMRX_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// Jacobi-preconditioned conjugate gradients with every scalar on the device,
// three launches an iteration: q = A p with p.q; x, r, z = Dinv r with r.r and
// r.z; p.  Each block of the second and third kernel forms alpha, beta and
// the stop test itself from the partial sums of the one before (the same
// order in every block), so nothing waits for the host: with dot products read
// back, an iteration took three round trips (9,537 nodes: 130 us, now 12).
// At most FCG_BLOCKS blocks, each over a contiguous chunk, so that the sums
// stay short; st: [0..1] r.z of the iterations in turn, [2] tolerance;
// flag[0] set when converged (2: |rhs|^2 is not a number), flag[1] the
// iterations done, flag[2] what
// flag[0] was before the direction launch.  That launch sets flag[0] in one
// block and tests flag[2]: blocks that tested the word it sets could lose some
// of their waves before a barrier that the others wait at.
constexpr int FCG_BLOCKS = 1024;
int filter_cg_blocks(int n) {
  const int64_t b = ((int64_t)n + FB - 1) / FB;
  return (int)(b < FCG_BLOCKS ? b : FCG_BLOCKS);
}

// sum of v over the block, in thread 0
__device__ __forceinline__ double fsum(double v, double *red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int w = 0; w < FB / 64; w++) s += red[w];
  return s;
}
// sum of parts[stride * i + o], i < np, in every thread
__device__ __forceinline__ double fparts(int np, const double *__restrict__ parts, int stride, int o,
                                         double *red) {
  double s = 0.0;
  for (int i = threadIdx.x; i < np; i += FB) s += parts[stride * i + o];
  return fsum(s, red);
}

// x = 0, r = rhs, z = Dinv r, p = z; partials r.r, r.z
__global__ __launch_bounds__(FB) void k_fcg_init(int n, int chunk, const double *__restrict__ rhs,
                                                 const double *__restrict__ dinv,
                                                 double *__restrict__ x, double *__restrict__ r,
                                                 double *__restrict__ p,
                                                 double *__restrict__ parts) {
  __shared__ double red[FB / 64];
  const int lo = blockIdx.x * chunk, hi = min(n, lo + chunk);
  double a = 0.0, b = 0.0;
  for (int i = lo + threadIdx.x; i < hi; i += FB) {
    const double v = rhs[i], z = dinv[i] * v;
    x[i] = 0.0;
    r[i] = v;
    p[i] = z;
    a += v * v;
    b += v * z;
  }
  const double sa = fsum(a, red), sb = fsum(b, red);
  if (threadIdx.x == 0) {
    parts[2 * blockIdx.x] = sa;
    parts[2 * blockIdx.x + 1] = sb;
  }
}

__global__ __launch_bounds__(FB) void k_fcg_start(int np, const double *__restrict__ parts,
                                                  double rtol2, double *__restrict__ st,
                                                  int *__restrict__ flag) {
  __shared__ double red[FB / 64];
  const double bb = fparts(np, parts, 2, 0, red), rz = fparts(np, parts, 2, 1, red);
  if (threadIdx.x == 0) {
    st[1] = rz;
    st[2] = rtol2 * bb;
    flag[0] = bb != bb ? 2 : bb == 0.0 ? 1 : 0;
    flag[1] = 0;
    flag[2] = 0;
  }
}

// q = A p, partials p.q: block b takes the rows of its chunk, FB / FL at a time
__global__ __launch_bounds__(FB) void k_fcg_product(int n, int chunk, const int *__restrict__ ptr,
                                                    const int *__restrict__ col,
                                                    const double *__restrict__ val,
                                                    const double *__restrict__ p,
                                                    double *__restrict__ q,
                                                    double *__restrict__ parts,
                                                    const int *__restrict__ flag) {
  __shared__ double red[FB / 64];
  if (flag[0]) return;
  const int lo = blockIdx.x * chunk, hi = min(n, lo + chunk);
  double a = 0.0;
  for (int i0 = lo; i0 < hi; i0 += FB / FL) {
    const int i = i0 + (int)(threadIdx.x / FL);
    const double s = row_sum(i, hi, ptr, col, val, p);
    if (i < hi && threadIdx.x % FL == 0) {
      q[i] = s;
      a += p[i] * s;
    }
  }
  const double sa = fsum(a, red);
  if (threadIdx.x == 0) parts[blockIdx.x] = sa;
}

// x += alpha p, r -= alpha q, z = Dinv r; partials r.r, r.z
__global__ __launch_bounds__(FB) void k_fcg_step(int n, int chunk, int it, int npq,
                                                 const double *__restrict__ pq,
                                                 const double *__restrict__ p,
                                                 const double *__restrict__ q,
                                                 const double *__restrict__ dinv,
                                                 double *__restrict__ x, double *__restrict__ r,
                                                 const double *__restrict__ st,
                                                 double *__restrict__ parts,
                                                 const int *__restrict__ flag, int *publish) {
  __shared__ double red[FB / 64];
  if (flag[0]) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *publish = 1;
    return;
  }
  const double alpha = st[it & 1] / fparts(npq, pq, 1, 0, red);
  const int lo = blockIdx.x * chunk, hi = min(n, lo + chunk);
  double a = 0.0, b = 0.0;
  for (int i = lo + threadIdx.x; i < hi; i += FB) {
    x[i] += alpha * p[i];
    const double v = r[i] - alpha * q[i];
    r[i] = v;
    a += v * v;
    b += v * (dinv[i] * v);
  }
  const double sa = fsum(a, red), sb = fsum(b, red);
  if (threadIdx.x == 0) {
    parts[2 * blockIdx.x] = sa;
    parts[2 * blockIdx.x + 1] = sb;
  }
}

// stop at r.r <= tolerance, else p = z + beta p
__global__ __launch_bounds__(FB) void k_fcg_direction(int n, int chunk, int it, int np,
                                                      const double *__restrict__ parts,
                                                      const double *__restrict__ dinv,
                                                      const double *__restrict__ r,
                                                      double *__restrict__ p,
                                                      double *__restrict__ st,
                                                      const int *__restrict__ before,
                                                      int *__restrict__ flag) {
  __shared__ double red[FB / 64];
  if (*before) return;
  const double rr = fparts(np, parts, 2, 0, red), rz = fparts(np, parts, 2, 1, red);
  const bool done = rr <= st[2];
  const double beta = rz / st[it & 1];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st[(it + 1) & 1] = rz;
    flag[1] = it;
    if (done) flag[0] = 1;
  }
  if (done) return;
  const int lo = blockIdx.x * chunk, hi = min(n, lo + chunk);
  for (int i = lo + threadIdx.x; i < hi; i += FB) p[i] = dinv[i] * r[i] + beta * p[i];
}

void launch_filter_cg_init(int n, const double *rhs, const double *dinv, double *x, double *r,
                           double *p, double *parts, double rtol2, double *sc, int *flag,
                           hipStream_t st) {
  const int nb = filter_cg_blocks(n), chunk = (n + nb - 1) / nb;
  hipLaunchKernelGGL(k_fcg_init, dim3(nb), dim3(FB), 0, st, n, chunk, rhs, dinv, x, r, p, parts);
  hipLaunchKernelGGL(k_fcg_start, dim3(1), dim3(FB), 0, st, nb, parts, rtol2, sc, flag);
  TMRX_LAUNCH_CHECK();
}

void launch_filter_cg_iteration(int n, int it, const int *ptr, const int *col, const double *val,
                                const double *dinv, double *x, double *r, double *p, double *q,
                                double *parts, double *sc, int *flag, hipStream_t st) {
  const int nb = filter_cg_blocks(n), chunk = (n + nb - 1) / nb;
  // the product wants more, shorter chunks: up to FCG_BLOCKS of 32 rows
  const int64_t w = ((int64_t)n + FB / FL - 1) / (FB / FL);
  const int nq = (int)(w < FCG_BLOCKS ? w : FCG_BLOCKS), qchunk = (n + nq - 1) / nq;
  double *pq = parts + 2 * FCG_BLOCKS;
  hipLaunchKernelGGL(k_fcg_product, dim3(nq), dim3(FB), 0, st, n, qchunk, ptr, col, val, p, q, pq,
                     flag);
  hipLaunchKernelGGL(k_fcg_step, dim3(nb), dim3(FB), 0, st, n, chunk, it, nq, pq, p, q, dinv, x, r,
                     sc, parts, flag, flag + 2);
  hipLaunchKernelGGL(k_fcg_direction, dim3(nb), dim3(FB), 0, st, n, chunk, it, nb, parts, dinv, r,
                     p, sc, flag + 2, flag);
  TMRX_LAUNCH_CHECK();
}
int filter_cg_parts() { return 3 * FCG_BLOCKS; }

__global__ void k_filter_fill(int n, double v, double *x) {
  const int i = blockIdx.x * FB + threadIdx.x;
  if (i < n) x[i] = v;
}
void launch_filter_fill(int n, double v, double *x, hipStream_t st) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_filter_fill, grid_of(n), dim3(FB), 0, st, n, v, x);
  TMRX_LAUNCH_CHECK();
}

__global__ void k_filter_lin(int n, int op, const double *a, const double *x,
                             const double *t, double *y) {
  const int i = blockIdx.x * FB + threadIdx.x;
  if (i >= n) return;
  switch (op) {
    case 0: y[i] = x[i]; break;                       // copy
    case 1: y[i] = a[i] * x[i]; break;                // elementwise product
    case 2: y[i] = a[i] * x[i] + t[i]; break;         // product plus t
    case 3: y[i] += t[i]; break;                      // add
    case 4: y[i] = x[i] != 0.0 ? 1.0 / x[i] : 0.0; break;  // reciprocal
  }
}
static void lin(int n, int op, const double *a, const double *x, const double *t,
                double *y, hipStream_t st) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_filter_lin, grid_of(n), dim3(FB), 0, st, n, op, a, x, t, y);
  TMRX_LAUNCH_CHECK();
}
void launch_filter_copy(int n, const double *x, double *y, hipStream_t st) {
  lin(n, 0, nullptr, x, nullptr, y, st);
}
void launch_filter_mul(int n, const double *a, const double *x, double *y, hipStream_t st) {
  lin(n, 1, a, x, nullptr, y, st);
}
void launch_filter_mul_add(int n, const double *a, const double *u, const double *t, double *y,
                           hipStream_t st) {
  lin(n, 2, a, u, t, y, st);
}
void launch_filter_add(int n, const double *t, double *y, hipStream_t st) {
  lin(n, 3, nullptr, nullptr, t, y, st);
}
void launch_filter_recip(int n, const double *x, double *y, hipStream_t st) {
  lin(n, 4, nullptr, x, nullptr, y, st);
}

__global__ void k_filter_stride(int n, int nv, int v, int dir, const double *x, double *y) {
  const int i = blockIdx.x * FB + threadIdx.x;
  if (i >= n) return;
  if (dir == 0)
    y[i] = x[(size_t)i * nv + v];
  else
    y[(size_t)i * nv + v] = x[i];
}
void launch_filter_gather(int n, int nv, int v, const double *x, double *y, hipStream_t st) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_filter_stride, grid_of(n), dim3(FB), 0, st, n, nv, v, 0, x, y);
  TMRX_LAUNCH_CHECK();
}
void launch_filter_scatter(int n, int nv, int v, const double *x, double *y, hipStream_t st) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_filter_stride, grid_of(n), dim3(FB), 0, st, n, nv, v, 1, x, y);
  TMRX_LAUNCH_CHECK();
}

}  // namespace tmrx

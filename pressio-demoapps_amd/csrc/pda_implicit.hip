// pda_implicit.hip -- implicit time stepping on the device: BDF1, BDF2 and
// Crank-Nicolson residuals and Jacobians with pressio's coefficients
// (tests_cpp/pressio/include/pressio/ode/impl/ode_implicit_discrete_residual.hpp:112-168,
//  ode_implicit_discrete_jacobian.hpp:60-121), solved by Newton's method on
// the exact Jacobian of the problem (pressio's Newton loop,
// pressio/solvers_nonlinear/impl/nonlinear_least_squares.hpp:14-118) with a
// device BiCGSTAB (the iteration of Eigen's BiCGSTAB, which pressio's
// default linear solver wraps, solvers_linear_traits.hpp:95-105) and a
// block-Jacobi preconditioner (the m x m diagonal blocks, inverted per cell),
// applied from the right: the matrix of the iteration is I + B with the blocks
// B_ij = cf J_ij (cf J_jj + cnp1 I)^-1, formed once per Newton iteration, beside
// the Jacobian slot by slot, or in its place where memory is short.
//
// Stop rules:
//   PDA_STOP_CORRECTION -- pressio's default: stop when the l2 norm of the
//     Newton correction is below tol, without applying that correction
//     (nonlinear_least_squares.hpp:70-84);
//   PDA_STOP_RESIDUAL   -- stop when ||R(y)||_2 <= tol (the correction that
//     reached it applied).
// The BiCGSTAB scalars live in device memory (no host round trip per dot
// product); the host polls the convergence flag every few iterations.
#include <cmath>

#include "pda_internal.hpp"

namespace pda {
namespace {

constexpr int TB = 256; // threads per block of the vector kernels
constexpr int MAXB = 1024; // most blocks (partial sums) of the reducing kernels

// Device scalars of the Krylov solver.  Each is written by the first block of
// one kernel and read by the kernels after it (never by the one that writes
// it): the search kernel writes RHO_NEXT, RR and DONE_NEXT, the second product
// RHO, ALPHA and DONE, the update kernel W and NITER.
enum { S_RHO = 0, S_RHO_NEXT, S_ALPHA, S_W, S_RR, S_BB, S_TOL2, S_DONE, S_DONE_NEXT, S_NITER, S_COUNT };

// a and b become their sums over the block, the same in every thread
__device__ __forceinline__ void block_sums(double &a, double &b, double *sh) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double ta = __shfl_xor(a, o, 64), tb = __shfl_xor(b, o, 64);
    a += ta;
    b += tb;
  }
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) {
    sh[w] = a;
    sh[TB / 64 + w] = b;
  }
  __syncthreads();
  a = b = 0.;
#pragma unroll
  for (int i = 0; i < TB / 64; ++i) {
    a += sh[i];
    b += sh[TB / 64 + i];
  }
}

// The sums of n pairs of partial sums, in a fixed order, the same in every
// thread of every block: a kernel that needs a dot product reduces the
// partial sums of the kernel that formed it by itself (16 KB from L2, about
// 1.5 us), where a launch of one block to do it took 4.6 us and a gap.
__device__ __forceinline__ void sum_pairs(const double *__restrict__ part, int n, double *sh, double &s1, double &s2) {
  double a = 0., b = 0.;
  for (int i = threadIdx.x; i < n; i += TB) {
    a += part[2 * i];
    b += part[2 * i + 1];
  }
  block_sums(a, b, sh);
  s1 = a;
  s2 = b;
}

__device__ __forceinline__ void put_pair(double *part, double s1, double s2, double *sh) {
  block_sums(s1, s2, sh);
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s1;
    part[2 * blockIdx.x + 1] = s2;
  }
}

// the norms of up to two vectors from their partial sums, into host memory
__global__ void __launch_bounds__(TB) k_norms_out(const double *__restrict__ pa, const double *__restrict__ pb, int n,
                                                  double *__restrict__ host) {
  __shared__ double sh[2 * (TB / 64)];
  double s1, s2;
  sum_pairs(pa, n, sh, s1, s2);
  if (threadIdx.x == 0) host[0] = sqrt(s1);
  if (!pb) return;
  sum_pairs(pb, n, sh, s1, s2);
  if (threadIdx.x == 0) host[1] = sqrt(s1);
}

// The index tables of the Jacobian's blocks
struct Blocks {
  const int64_t *rowbase;
  const int32_t *nblk, *bcol;
  const int64_t *diag; // first value of the diagonal block, per cell
  int maxb;
  int64_t ncell;
};

// The iteration's matrix I + B, slot by slot: entry pair h (a value where M is
// odd) of off-diagonal block e of cell c at ((e PAIRS + h) ncell + c) V, and the
// block's column cell at e ncell + c.  Rows with fewer blocks than the widest
// have zero blocks on their own cell.
template <int M> struct Ell {
  static constexpr int V = M % 2 == 0 ? 2 : 1, PAIRS = M * M / V;
};

// the column cells of the off-diagonal blocks, lane per cell
__global__ void __launch_bounds__(TB) k_ell_cols(Blocks K, int M, int32_t *__restrict__ col) {
  const int64_t c = int64_t(blockIdx.x) * TB + threadIdx.x;
  if (c >= K.ncell) return;
  const int nb = K.nblk[c], d = int((K.diag[c] - K.rowbase[c]) / M);
  for (int e = 0; e + 1 < K.maxb; ++e) {
    const int b = e < d ? e : e + 1;
    col[e * K.ncell + c] = b < nb ? K.bcol[c * K.maxb + b] : int32_t(c);
  }
}

// B's blocks from the Jacobian's and the inverted diagonal blocks: 16 lanes per
// cell, a lane per block, so that a cell's values are read as they lie; a block
// of threads writes 16 consecutive cells of every slot.  Bound by the matrix
// read and written: 512 x 512 Burgers (222 MB) 54 us, repaid within three iterations.
// IN_PLACE: in the place of the Jacobian's blocks, for steppers without room for a
// second matrix (a block is read and written by its lane alone; the diagonal
// blocks stay).
constexpr int FL = 16;
template <int M, bool IN_PLACE>
__global__ void __launch_bounds__(TB) k_form(Blocks K, double *__restrict__ J, double cf,
                                             const double *__restrict__ Minv, double *__restrict__ A) {
  constexpr int V = Ell<M>::V, PAIRS = Ell<M>::PAIRS;
  const int64_t c = (int64_t(blockIdx.x) * TB + threadIdx.x) / FL;
  if (c >= K.ncell) return;
  const int nb = K.nblk[c];
  const int64_t rb = K.rowbase[c];
  const int d = int((K.diag[c] - rb) / M);
  for (int e = threadIdx.x % FL; e + 1 < K.maxb; e += FL) {
    const int b = e < d ? e : e + 1;
    double o[M * M];
#pragma unroll
    for (int k = 0; k < M * M; ++k) o[k] = 0.;
    if (b < nb) {
      double *Jr = J + rb + b * M;
      const double *Mi = Minv + int64_t(K.bcol[c * K.maxb + b]) * M * M;
#pragma unroll
      for (int k = 0; k < M; ++k) {
        double a[M];
#pragma unroll
        for (int j = 0; j < M; ++j) a[j] = cf * Jr[int64_t(k) * nb * M + j];
#pragma unroll
        for (int j = 0; j < M; ++j)
#pragma unroll
          for (int i = 0; i < M; ++i) o[k * M + j] += a[i] * Mi[i * M + j];
      }
      if constexpr (IN_PLACE) {
#pragma unroll
        for (int k = 0; k < M; ++k)
#pragma unroll
          for (int j = 0; j < M; ++j) Jr[int64_t(k) * nb * M + j] = o[k * M + j];
      }
    }
    if constexpr (IN_PLACE) continue;
#pragma unroll
    for (int h = 0; h < PAIRS; ++h)
#pragma unroll
      for (int v = 0; v < V; ++v) A[((int64_t(e) * PAIRS + h) * K.ncell + c) * V + v] = o[h * V + v];
  }
}

// y = (I + B) x, a lane per cell: every load of the matrix, its columns and
// (but for the grid's edges) of x is one contiguous run of the wave, all of a
// cell's loads are in flight together and no sum crosses lanes.  A block of
// threads takes a contiguous range of cells, and the ranges of one XCD are
// neighbours, so that x is read into each L2 once.  SECOND: alpha = rho /
// (r0 . v) from its partial sums, and x = r - alpha v is formed as it is
// gathered, for 50 MB more from L2 but without a launch and a vector for it.
// Bound by the matrix, which stays in the last-level cache: 512 x 512 Burgers
// (12 2 x 2 blocks a cell, 113 MB with their columns) 17.0 us (7.4 TB/s) and
// 18.9 SECOND; 16 lanes per cell over the Jacobian's own CSR blocks 23.8, with
// 14.4 us of launches that applied Minv beside each product.
// Partial sums of (r0 . y), or with SECOND of (y . x, y . y).
// IN_PLACE: the blocks lie in the Jacobian's CSR (k_form), their columns in K.
template <int M, bool SECOND, bool IN_PLACE>
__global__ void __launch_bounds__(TB) k_spmv(Blocks K, const double *__restrict__ A,
                                             const int32_t *__restrict__ col, int slots, int64_t ncell, const double *__restrict__ x,
                                             const double *__restrict__ xv, const double *__restrict__ r0,
                                             double *__restrict__ y, int64_t per_block,
                                             const double *__restrict__ part_in, int npart,
                                             double *__restrict__ part, double *__restrict__ scal) {
  __shared__ double sh[2 * (TB / 64)];
  constexpr int V = Ell<M>::V, PAIRS = Ell<M>::PAIRS;
  double alpha = 0.;
  if constexpr (SECOND) {
    const double dn = scal[S_DONE_NEXT], rho = scal[S_RHO_NEXT];
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    if (dn != 0.) {
      if (lead) scal[S_DONE] = 1.;
      return;
    }
    double s1, s2;
    sum_pairs(part_in, npart, sh, s1, s2);
    alpha = rho / s1;
    if (lead) {
      scal[S_RHO] = rho;
      scal[S_ALPHA] = alpha;
    }
  } else if (scal[S_DONE_NEXT] != 0.) {
    return;
  }
  // block -> range: the blocks of XCD b % 8 take neighbouring ranges
  const int nbk = gridDim.x, q = nbk / 8, rem = nbk % 8, xcd = int(blockIdx.x) % 8, kk = int(blockIdx.x) / 8;
  const int64_t range = int64_t(xcd) * q + (xcd < rem ? xcd : rem) + kk;
  const int64_t c_lo = range * per_block, c_hi = c_lo + per_block < ncell ? c_lo + per_block : ncell;
  double s1 = 0., s2 = 0.;
  for (int64_t c = c_lo + threadIdx.x; c < c_hi; c += TB) {
    double acc[M], own[M];
#pragma unroll
    for (int k = 0; k < M; ++k) {
      own[k] = x[c * M + k];
      if constexpr (SECOND) own[k] -= alpha * xv[c * M + k];
      acc[k] = own[k];
    }
    int nb = 0, d = 0;
    if constexpr (IN_PLACE) {
      nb = K.nblk[c];
      d = int((K.diag[c] - K.rowbase[c]) / M);
      slots = nb - 1;
    }
#pragma unroll 4
    for (int e = 0; e < slots; ++e) {
      int64_t j;
      double u[M], b[M * M];
      if constexpr (IN_PLACE) {
        const int q = e < d ? e : e + 1;
        const double *a = A + K.rowbase[c] + q * M;
        j = int64_t(K.bcol[c * K.maxb + q]) * M;
#pragma unroll
        for (int k = 0; k < M; ++k)
#pragma unroll
          for (int i = 0; i < M; ++i) b[k * M + i] = a[int64_t(k) * nb * M + i];
      } else {
        const double *a = A + (int64_t(e) * PAIRS * ncell + c) * V;
        j = int64_t(col[e * ncell + c]) * M;
#pragma unroll
        for (int h = 0; h < PAIRS; ++h)
#pragma unroll
          for (int v = 0; v < V; ++v) b[h * V + v] = a[h * ncell * V + v];
      }
#pragma unroll
      for (int k = 0; k < M; ++k) {
        u[k] = x[j + k];
        if constexpr (SECOND) u[k] -= alpha * xv[j + k];
      }
#pragma unroll
      for (int k = 0; k < M; ++k)
#pragma unroll
        for (int i = 0; i < M; ++i) acc[k] += b[k * M + i] * u[i];
    }
#pragma unroll
    for (int k = 0; k < M; ++k) {
      y[c * M + k] = acc[k];
      if constexpr (SECOND) {
        s1 += acc[k] * own[k];
        s2 += acc[k] * acc[k];
      } else {
        s1 += r0[c * M + k] * acc[k];
      }
    }
  }
  put_pair(part, s1, s2, sh);
}

// Inverse of the m x m diagonal block of cnp1 I + cf J of every cell
// (Gauss-Jordan with partial pivoting)
template <int M>
__global__ void __launch_bounds__(TB) k_block_inv(Blocks K, const double *__restrict__ J, double cf, double cnp1,
                                                   double *__restrict__ Minv) {
  const int64_t c = int64_t(blockIdx.x) * TB + threadIdx.x;
  if (c >= K.ncell) return;
  double a[M][2 * M];
  const int64_t pos = K.diag[c];
  const int rs = K.nblk[c] * M;
#pragma unroll
  for (int k = 0; k < M; ++k) {
#pragma unroll
    for (int j = 0; j < M; ++j) {
      a[k][j] = cf * J[pos + int64_t(k) * rs + j] + (j == k ? cnp1 : 0.);
      a[k][M + j] = (j == k) ? 1. : 0.;
    }
  }
#pragma unroll
  for (int col = 0; col < M; ++col) {
    int piv = col;
    double best = fabs(a[col][col]);
#pragma unroll
    for (int r = col + 1; r < M; ++r)
      if (fabs(a[r][col]) > best) {
        best = fabs(a[r][col]);
        piv = r;
      }
#pragma unroll
    for (int r = col; r < M; ++r)
      if (r == piv && r != col)
#pragma unroll
        for (int j = 0; j < 2 * M; ++j) {
          const double t = a[col][j];
          a[col][j] = a[r][j];
          a[r][j] = t;
        }
    const double inv = 1. / a[col][col];
#pragma unroll
    for (int j = 0; j < 2 * M; ++j) a[col][j] *= inv;
#pragma unroll
    for (int r = 0; r < M; ++r) {
      if (r == col) continue;
      const double f = a[r][col];
#pragma unroll
      for (int j = 0; j < 2 * M; ++j) a[r][j] -= f * a[col][j];
    }
  }
#pragma unroll
  for (int k = 0; k < M; ++k)
#pragma unroll
    for (int j = 0; j < M; ++j) Minv[(c * M + k) * M + j] = a[k][M + j];
}

// start of a solve: x = 0, r = r0 = -R; partial sums of r0 . r twice (r0 . r
// and r . r); cleared flags for the iterations
__global__ void __launch_bounds__(TB) k_start(const double *__restrict__ R, double *__restrict__ x,
                                              double *__restrict__ r, double *__restrict__ r0, int64_t n,
                                              double *__restrict__ part, double *__restrict__ scal) {
  __shared__ double sh[2 * (TB / 64)];
  double s = 0.;
  for (int64_t i = int64_t(blockIdx.x) * TB + threadIdx.x; i < n; i += int64_t(gridDim.x) * TB) {
    const double b = -R[i];
    x[i] = 0.;
    r[i] = b;
    r0[i] = b;
    s += b * b;
  }
  put_pair(part, s, s, sh);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    scal[S_RHO] = 1.;
    scal[S_ALPHA] = 1.;
    scal[S_W] = 1.;
    scal[S_NITER] = 0.;
    scal[S_DONE] = 0.;
    scal[S_DONE_NEXT] = 0.;
  }
}

// whether a residual with (r0.r, r.r) = (s1, s2) ends the solve: converged, or
// a non-finite reduction (a breakdown, or NaN in the system), whose result
// the Newton loop rejects
__device__ __forceinline__ bool ends(double s1, double s2, double tol2) {
  return s2 <= tol2 || !isfinite(s1) || !isfinite(s2);
}

// The search direction: beta from the partial sums of (r0 . r, r . r), or, in
// the first iteration, the tolerance from those of b . b;
// p = r + beta (p - w v)
__global__ void __launch_bounds__(TB) k_p(const double *__restrict__ r, double *__restrict__ p,
                                           const double *__restrict__ v, int64_t n,
                                           const double *__restrict__ part, int npart, double *__restrict__ scal,
                                           int first, double rtol) {
  __shared__ double sh[2 * (TB / 64)];
  if (scal[S_DONE] != 0.) return; // written by earlier kernels: the same in every block
  const double alpha = scal[S_ALPHA], w = scal[S_W], rho = scal[S_RHO];
  double s1, s2;
  sum_pairs(part, npart, sh, s1, s2);
  const double tol2 = first ? rtol * rtol * s1 : scal[S_TOL2];
  const bool done = ends(s1, s2, tol2) || (first && s1 == 0.);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (first) {
      scal[S_BB] = s1;
      scal[S_TOL2] = tol2;
    }
    scal[S_RR] = s2;
    scal[S_RHO_NEXT] = s1;
    scal[S_DONE_NEXT] = done ? 1. : 0.;
  }
  if (done) return;
  const double beta = (s1 / rho) * (alpha / w);
  auto next = [&](double ri, double pi, double vi) { return first ? ri : ri + beta * (pi - w * vi); };
  const double2 *r2 = reinterpret_cast<const double2 *>(r), *v2 = reinterpret_cast<const double2 *>(v);
  double2 *p2 = reinterpret_cast<double2 *>(p);
  for (int64_t i = int64_t(blockIdx.x) * TB + threadIdx.x; i < n / 2; i += int64_t(gridDim.x) * TB) {
    const double2 a = r2[i], b = p2[i], c = v2[i];
    p2[i] = make_double2(next(a.x, b.x, c.x), next(a.y, b.y, c.y));
  }
  if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) p[n - 1] = next(r[n - 1], p[n - 1], v[n - 1]);
}

// w = (t . s) / (t . t) from their partial sums; s = r - alpha v;
// x += alpha p + w s; r = s - w t; partial sums of (r0 . r, r . r).  Two entries
// per lane in 16-byte accesses, both sums of a block reduced together: 8.2 us at
// 512 x 512 x 2 unknowns (33 MB, in the last-level cache), 8.8 entry by entry.
__global__ void __launch_bounds__(TB) k_xr(double *__restrict__ x, double *__restrict__ r,
                                            const double *__restrict__ p, const double *__restrict__ v,
                                            const double *__restrict__ t, const double *__restrict__ r0, int64_t n,
                                            const double *__restrict__ part_in, int npart,
                                            double *__restrict__ part, double *__restrict__ scal) {
  __shared__ double sh[2 * (TB / 64)];
  if (scal[S_DONE_NEXT] != 0.) return; // the last residual's partial sums stay
  const double alpha = scal[S_ALPHA];
  double ts, tt;
  sum_pairs(part_in, npart, sh, ts, tt);
  const double w = tt > 0. ? ts / tt : 0.;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    scal[S_W] = w;
    scal[S_NITER] += 1.; // read by no other block
  }
  double s1 = 0., s2 = 0.;
  auto update = [&](double &xi, double &ri, double pi, double vi, double ti, double qi) {
    const double si = ri - alpha * vi;
    xi += alpha * pi + w * si;
    ri = si - w * ti;
    s1 += qi * ri;
    s2 += ri * ri;
  };
  double2 *x2 = reinterpret_cast<double2 *>(x), *r2 = reinterpret_cast<double2 *>(r);
  const double2 *p2 = reinterpret_cast<const double2 *>(p), *v2 = reinterpret_cast<const double2 *>(v);
  const double2 *t2 = reinterpret_cast<const double2 *>(t), *q2 = reinterpret_cast<const double2 *>(r0);
  for (int64_t i = int64_t(blockIdx.x) * TB + threadIdx.x; i < n / 2; i += int64_t(gridDim.x) * TB) {
    double2 a = x2[i], b = r2[i];
    const double2 pi = p2[i], vi = v2[i], ti = t2[i], qi = q2[i];
    update(a.x, b.x, pi.x, vi.x, ti.x, qi.x);
    update(a.y, b.y, pi.y, vi.y, ti.y, qi.y);
    x2[i] = a;
    r2[i] = b;
  }
  if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) update(x[n - 1], r[n - 1], p[n - 1], v[n - 1], t[n - 1], r0[n - 1]);
  put_pair(part, s1, s2, sh);
}

// the state of the solve after the last update, into host memory
enum { H_DONE = 0, H_NITER, H_RR, H_BB, H_COUNT };
__global__ void __launch_bounds__(TB) k_check(const double *__restrict__ part, int npart,
                                              const double *__restrict__ scal, double *__restrict__ host) {
  __shared__ double sh[2 * (TB / 64)];
  double s1, s2;
  sum_pairs(part, npart, sh, s1, s2);
  if (threadIdx.x != 0) return;
  host[H_DONE] = scal[S_DONE_NEXT] != 0. || ends(s1, s2, scal[S_TOL2]) ? 1. : 0.;
  host[H_NITER] = scal[S_NITER];
  host[H_RR] = s2;
  host[H_BB] = scal[S_BB];
}

// R = cnp1 y + cn y_n + c2 x2 + cf f, with partial sums of R . R
__global__ void __launch_bounds__(TB) k_residual(double *__restrict__ R, const double *__restrict__ Y, double cnp1,
                                                 const double *__restrict__ Yn, double cn,
                                                 const double *__restrict__ x2, double c2,
                                                 const double *__restrict__ F, double cf, int64_t n,
                                                 double *__restrict__ part) {
  __shared__ double sh[2 * (TB / 64)];
  double s = 0.;
  for (int64_t i = int64_t(blockIdx.x) * TB + threadIdx.x; i < n; i += int64_t(gridDim.x) * TB) {
    double v = cnp1 * Y[i];
    v += cn * Yn[i];
    if (x2) v += c2 * x2[i];
    v += cf * F[i];
    R[i] = v;
    s += v * v;
  }
  put_pair(part, s, 0., sh);
}

// dx = Minv x, the correction from the preconditioned unknowns, with partial
// sums of dx . dx; Y += dx where Y is given
template <int M>
__global__ void __launch_bounds__(TB) k_unscale(const double *__restrict__ Minv, const double *__restrict__ x,
                                                double *__restrict__ dx, double *__restrict__ Y, int64_t ncell,
                                                double *__restrict__ part) {
  __shared__ double sh[2 * (TB / 64)];
  double s = 0.;
  for (int64_t c = int64_t(blockIdx.x) * TB + threadIdx.x; c < ncell; c += int64_t(gridDim.x) * TB) {
#pragma unroll
    for (int k = 0; k < M; ++k) {
      double d = 0.;
#pragma unroll
      for (int j = 0; j < M; ++j) d += Minv[(c * M + k) * M + j] * x[c * M + j];
      dx[c * M + k] = d;
      if (Y) Y[c * M + k] += d;
      s += d * d;
    }
  }
  put_pair(part, s, 0., sh);
}

// Y += dx
__global__ void __launch_bounds__(TB) k_correct(double *__restrict__ Y, const double *__restrict__ dx, int64_t n) {
  const int64_t i = int64_t(blockIdx.x) * TB + threadIdx.x;
  if (i < n) Y[i] += dx[i];
}

unsigned grid_of(int64_t n) { return unsigned(std::max<int64_t>(1, (n + TB - 1) / TB)); }
unsigned grid_strided(int64_t n) { return unsigned(std::max<int64_t>(1, std::min<int64_t>((n + TB - 1) / TB, MAXB))); }

}  // namespace
}  // namespace pda

struct pda_implicit_s {
  pda_problem_s *prob = nullptr;
  int scheme = 0;
  int64_t n = 0, ncell = 0;
  int stop = PDA_STOP_CORRECTION;
  double tol = 1e-6;
  int max_newton = 100;
  double lin_rtol = 1e-14;
  int lin_max = 0;          // 0: 2 * unknowns (Eigen's default)
  int check_every = 4;      // iterations of the recorded graph
  static constexpr int FIRST_POLL = 24; // the first poll comes no later, each further one by twice the count
  pda::DevBuf J, F, Fn, R, Y, Yn, dx, x, r, r0, p, v, t, Minv, scal;
  pda::DevBuf ell, ellcol;  // the iteration's matrix and its column cells
  bool in_place = false;    // without them: the matrix in the Jacobian's place
  pda::DevBuf part[5];      // partial sums: r0.v, (t.s, t.t), (r0.r, r.r), R.R, dx.dx
  pda::DevBuf diag;         // first value of every cell's diagonal block
  double *host = nullptr;   // pinned: what the host reads after a synchronization
  // linear iterations of the last step's first, second, ... Newton iteration;
  // 0 where none converged or the step failed
  int guess_iters[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  void forget_iters() {
    for (int &g : guess_iters) g = 0;
  }
  pda_implicit_stats last{};
  // check_every BiCGSTAB iterations recorded once as a graph (their kernel
  // arguments are the same for every solve of this stepper)
  hipStream_t cap = nullptr;
  hipGraph_t lin_graph = nullptr;
  hipGraphExec_t lin_exec = nullptr;
  ~pda_implicit_s() {
    if (lin_exec) (void)hipGraphExecDestroy(lin_exec);
    if (lin_graph) (void)hipGraphDestroy(lin_graph);
    if (cap) (void)hipStreamDestroy(cap);
    if (host) (void)hipHostFree(host);
  }
};

namespace {
using namespace pda;

enum { P_R0V = 0, P_TS, P_RR, P_RES, P_DX };

Blocks blocks_of(const pda_implicit_s &ip) {
  const pda_problem_s &p = *ip.prob;
  Blocks K;
  K.rowbase = p.view.rowbase;
  K.nblk = p.view.nblk;
  K.bcol = p.d_bcol.as<int32_t>();
  K.diag = ip.diag.as<int64_t>();
  K.maxb = p.maxb;
  K.ncell = ip.ncell;
  return K;
}

// one BiCGSTAB iteration; every kernel is a no-op once the convergence flag is set
template <int M, bool IN_PLACE>
void bicgstab_iteration_in(pda_implicit_s &ip, hipStream_t st, bool first, double rtol) {
  const int64_t n = ip.n, nc = ip.ncell;
  const int slots = ip.prob->maxb - 1;
  double *r = ip.r.as<double>(), *r0 = ip.r0.as<double>(), *pp = ip.p.as<double>();
  double *v = ip.v.as<double>(), *t = ip.t.as<double>(), *scal = ip.scal.as<double>();
  const double *A = IN_PLACE ? ip.J.as<double>() : ip.ell.as<double>();
  const Blocks K = blocks_of(ip);
  const int32_t *col = ip.ellcol.as<int32_t>();
  double *pr0v = ip.part[P_R0V].as<double>(), *pts = ip.part[P_TS].as<double>(), *prr = ip.part[P_RR].as<double>();
  const unsigned gv = grid_strided(n);
  // cells of a block of the products: whole passes of its lanes, at most MAXB blocks
  const int64_t per = ((nc + MAXB - 1) / MAXB + TB - 1) / TB * TB;
  const unsigned gs = unsigned((nc + per - 1) / per);
  hipLaunchKernelGGL(k_p, dim3(gv), dim3(TB), 0, st, r, pp, v, n, prr, int(gv), scal, first ? 1 : 0, rtol);
  hipLaunchKernelGGL((k_spmv<M, false, IN_PLACE>), dim3(gs), dim3(TB), 0, st, K, A, col, slots, nc, pp, nullptr, r0, v,
                     per, nullptr, 0, pr0v, scal);
  hipLaunchKernelGGL((k_spmv<M, true, IN_PLACE>), dim3(gs), dim3(TB), 0, st, K, A, col, slots, nc, r, v, nullptr, t, per,
                     pr0v, int(gs), pts, scal);
  hipLaunchKernelGGL(k_xr, dim3(gv), dim3(TB), 0, st, ip.x.as<double>(), r, pp, v, t, r0, n, pts, int(gs), prr, scal);
}

template <int M> void bicgstab_iteration(pda_implicit_s &ip, hipStream_t st, bool first, double rtol) {
  if (ip.in_place) bicgstab_iteration_in<M, true>(ip, st, first, rtol);
  else bicgstab_iteration_in<M, false>(ip, st, first, rtol);
}

// (cnp1 I + cf J) dx = -R, Y += dx where Y is given, partial sums of dx . dx.  newton: index of the Newton iteration, whose
// linear iterations in the step before decide how many run before the first
// poll (the kernels stop by themselves at convergence, so this moves no value).
// It is polled after FIRST_POLL iterations at the latest and then by twice the
// count, so that an easy solve after a hard one queues few launches without
// work, and a long solve has few polls (about 15 us each) more: without the
// bound, a step of two iterations after one that stopped at 3,000 took 9,980 us
// (64 x 64 Burgers; 160 by itself).
template <int M>
int bicgstab_m(pda_implicit_s &ip, double cf, double cnp1, double *Y, hipStream_t st, double rtol, int newton,
               int *iters, double *rel_res) {
  const int64_t n = ip.n, nc = ip.ncell;
  double *prr = ip.part[P_RR].as<double>(), *scal = ip.scal.as<double>(), *h = ip.host;
  const unsigned gv = grid_strided(n), gc = grid_of(nc);
  hipLaunchKernelGGL((k_block_inv<M>), dim3(gc), dim3(TB), 0, st, blocks_of(ip), ip.J.as<double>(), cf, cnp1,
                     ip.Minv.as<double>());
  hipLaunchKernelGGL((ip.in_place ? k_form<M, true> : k_form<M, false>), dim3(grid_of(nc * FL)), dim3(TB), 0, st,
                     blocks_of(ip), ip.J.as<double>(), cf, ip.Minv.as<double>(), ip.ell.as<double>());
  hipLaunchKernelGGL(k_start, dim3(gv), dim3(TB), 0, st, ip.R.as<double>(), ip.x.as<double>(), ip.r.as<double>(),
                     ip.r0.as<double>(), n, prr, scal);
  PDA_HIP_CHECK(hipGetLastError());
  const int64_t maxit = ip.lin_max > 0 ? ip.lin_max : 2 * n;
  const int K = ip.check_every, slot = newton < 8 ? newton : 7;
  // iteration 0 (p = r) eagerly, then chunks of K iterations replayed from
  // one graph, polling the convergence flag after each chunk from about the
  // last step's count on; a tail shorter than K runs eagerly so that maxit is
  // exact
  bicgstab_iteration<M>(ip, st, true, rtol);
  PDA_HIP_CHECK(hipGetLastError());
  int64_t it = 1;
  auto next_poll = [&] { return std::min<int64_t>(ip.guess_iters[slot] - K, std::max<int64_t>(ip.FIRST_POLL, 2 * it)); };
  int64_t poll = next_poll(); // the iteration from which on each chunk is polled
  bool done = false;
  while (!done) {
    if (maxit - it >= K) {
      if (!ip.lin_exec) {
        if (!ip.cap) PDA_HIP_CHECK(hipStreamCreateWithFlags(&ip.cap, hipStreamNonBlocking));
        PDA_HIP_CHECK(hipStreamBeginCapture(ip.cap, hipStreamCaptureModeThreadLocal));
        for (int k = 0; k < K; ++k) bicgstab_iteration<M>(ip, ip.cap, false, 0.);
        hipGraph_t g = nullptr;
        const hipError_t e = hipStreamEndCapture(ip.cap, &g);
        if (e != hipSuccess || !g) {
          if (g) (void)hipGraphDestroy(g);
          set_error(std::string("bicgstab: graph capture: ") + hipGetErrorString(e));
          return PDA_E_HIP;
        }
        const hipError_t ei = hipGraphInstantiate(&ip.lin_exec, g, nullptr, nullptr, 0);
        if (ei != hipSuccess) {
          (void)hipGraphDestroy(g);
          ip.lin_exec = nullptr;
          set_error(std::string("bicgstab: graph instantiation: ") + hipGetErrorString(ei));
          return PDA_E_HIP;
        }
        ip.lin_graph = g;
      }
      PDA_HIP_CHECK(hipGraphLaunch(ip.lin_exec, st));
      it += K;
      if (it < poll && maxit - it >= K) continue;
    } else {
      for (; it < maxit; ++it) bicgstab_iteration<M>(ip, st, false, 0.);
      PDA_HIP_CHECK(hipGetLastError());
    }
    hipLaunchKernelGGL(k_check, dim3(1), dim3(TB), 0, st, prr, int(gv), scal, h);
    PDA_HIP_CHECK(hipGetLastError());
    PDA_HIP_CHECK(hipStreamSynchronize(st));
    done = h[H_DONE] != 0. || it >= maxit;
    poll = next_poll();
  }
  hipLaunchKernelGGL((k_unscale<M>), dim3(gv), dim3(TB), 0, st, ip.Minv.as<double>(),
                     ip.x.as<double>(), ip.dx.as<double>(), Y, nc, ip.part[P_DX].as<double>());
  PDA_HIP_CHECK(hipGetLastError());
  *iters = int(h[H_NITER]) + (h[H_DONE] == 0. ? 1 : 0); // at the limit the unmet check counts too
  *rel_res = h[H_BB] > 0. ? std::sqrt(h[H_RR] / h[H_BB]) : 0.;
  ip.guess_iters[slot] = h[H_DONE] != 0. ? *iters : 0;
  // a solve that stops at the iteration limit is reported through rel_res;
  // the Newton loop's own stop rule decides
  return PDA_OK;
}

int bicgstab(pda_implicit_s &ip, double cf, double cnp1, double *Y, hipStream_t st, double rtol, int newton,
             int *iters, double *rel) {
  switch (ip.prob->m) {
    case 1: return bicgstab_m<1>(ip, cf, cnp1, Y, st, rtol, newton, iters, rel);
    case 2: return bicgstab_m<2>(ip, cf, cnp1, Y, st, rtol, newton, iters, rel);
    case 3: return bicgstab_m<3>(ip, cf, cnp1, Y, st, rtol, newton, iters, rel);
    case 4: return bicgstab_m<4>(ip, cf, cnp1, Y, st, rtol, newton, iters, rel);
    case 5: return bicgstab_m<5>(ip, cf, cnp1, Y, st, rtol, newton, iters, rel);
  }
  set_error("implicit: unsupported block size");
  return PDA_E_UNSUPPORTED;
}

}  // namespace

extern "C" {

int pda_implicit_create(pda_problem p, int scheme, pda_implicit *out) {
  if (!p || !out || (scheme != PDA_BDF1 && scheme != PDA_BDF2 && scheme != PDA_CRANK_NICOLSON)) {
    set_error("pda_implicit_create: invalid argument");
    return PDA_E_INVALID_ARG;
  }
  if (p->mesh->n_sample != p->mesh->n_stencil) {
    set_error("pda_implicit_create: implicit stepping needs a full mesh (sample == stencil mesh)");
    return PDA_E_INVALID_ARG;
  }
  if (p->m > 5) {
    set_error("pda_implicit_create: unsupported block size");
    return PDA_E_UNSUPPORTED;
  }
  int rc = ensure_device(*p);
  if (rc) return rc;
  auto *ip = new pda_implicit_s();
  ip->prob = p;
  ip->scheme = scheme;
  ip->n = p->mesh->n_stencil * p->m;
  ip->ncell = p->mesh->n_stencil;
  const size_t vb = sizeof(double) * size_t(ip->n);
  hipError_t e = ip->J.alloc(sizeof(double) * size_t(p->nnz));
  pda::DevBuf *vecs[] = {&ip->F, &ip->Fn, &ip->R, &ip->Y, &ip->Yn, &ip->dx, &ip->x, &ip->r, &ip->r0,
                         &ip->p, &ip->v, &ip->t};
  for (auto *d : vecs)
    if (e == hipSuccess) e = d->alloc(vb);
  if (e == hipSuccess) e = ip->Minv.alloc(sizeof(double) * size_t(ip->ncell) * p->m * p->m);
  for (auto &d : ip->part)
    if (e == hipSuccess) e = d.alloc(sizeof(double) * 2 * pda::MAXB);
  if (e == hipSuccess) e = hipHostMalloc(reinterpret_cast<void **>(&ip->host), sizeof(double) * 8, hipHostMallocDefault);
  if (e == hipSuccess) {
    // the diagonal block of every cell (full mesh: cell c's column is c)
    std::vector<int64_t> dg(size_t(ip->ncell), -1);
    for (int64_t c = 0; c < ip->ncell; ++c)
      for (int s = 0; s < p->h_nblk[c]; ++s)
        if (p->h_bcol[size_t(c) * p->maxb + s] == int32_t(c)) dg[c] = p->h_rowbase[c] + int64_t(s) * p->m;
    for (int64_t c = 0; c < ip->ncell; ++c)
      if (dg[c] < 0) {
        set_error("pda_implicit_create: Jacobian pattern lacks a contiguous diagonal block");
        delete ip;
        return PDA_E_STATE;
      }
    e = ip->diag.upload(dg);
  }
  if (e == hipSuccess) e = ip->scal.alloc(sizeof(double) * pda::S_COUNT);
  if (e == hipSuccess) {
    // the iteration's matrix last: where it would take more than half of the
    // memory that is left, the stepper does without (k_form's IN_PLACE), at 8
    // bytes a nonzero instead of 16
    const size_t blocks = size_t(ip->ncell) * size_t(std::max(1, p->maxb - 1));
    const size_t ell = sizeof(double) * blocks * p->m * p->m, cols = sizeof(int32_t) * blocks;
    size_t left = 0, total = 0;
    ip->in_place = hipMemGetInfo(&left, &total) != hipSuccess || left / 2 < ell + cols ||
                   ip->ell.alloc(ell) != hipSuccess || ip->ellcol.alloc(cols) != hipSuccess;
    if (ip->in_place) {
      ip->ell.reset();
      ip->ellcol.reset();
      (void)hipGetLastError(); // a failed allocation is not the caller's error
    } else {
      hipLaunchKernelGGL(k_ell_cols, dim3(grid_of(ip->ncell)), dim3(TB), 0, nullptr, blocks_of(*ip), p->m,
                         ip->ellcol.as<int32_t>());
      e = hipGetLastError();
      if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
    }
  }
  if (e != hipSuccess) {
    set_error(std::string("pda_implicit_create: ") + hipGetErrorString(e));
    delete ip;
    return PDA_E_HIP;
  }
  *out = ip;
  return PDA_OK;
}

void pda_implicit_destroy(pda_implicit ip) { delete ip; }

int pda_implicit_set_options(pda_implicit ip, int stop_rule, double tol, int max_newton,
                             double lin_rtol, int lin_max) {
  if (!ip || (stop_rule != PDA_STOP_CORRECTION && stop_rule != PDA_STOP_RESIDUAL) || !(tol > 0.) ||
      max_newton < 1 || !(lin_rtol > 0.) || lin_max < 0) {
    set_error("pda_implicit_set_options: invalid argument");
    return PDA_E_INVALID_ARG;
  }
  ip->stop = stop_rule;
  ip->tol = tol;
  ip->max_newton = max_newton;
  ip->lin_rtol = lin_rtol;
  ip->lin_max = lin_max;
  ip->forget_iters();
  return PDA_OK;
}

int pda_implicit_step(pda_implicit ip, double *d_U, const double *d_Uprev, const double *d_guess,
                      double t, double dt, pda_stream stream, pda_implicit_stats *stats) {
  if (!ip || !d_U || !(dt > 0.)) {
    set_error("pda_implicit_step: invalid argument");
    return PDA_E_INVALID_ARG;
  }
  hipStream_t st = hipStream_t(stream);
  pda_problem_s &p = *ip->prob;
  const int64_t n = ip->n;
  if (!p.on_device) {
    set_error("pda_implicit_step: problem tables not on the device");
    return PDA_E_STATE;
  }
  double *J = ip->J.as<double>(), *F = ip->F.as<double>(), *R = ip->R.as<double>();
  double *Y = ip->Y.as<double>(), *Yn = ip->Yn.as<double>();
  double *Fn = ip->Fn.as<double>();
  const unsigned gs = grid_strided(n);
  // residual coefficients R = cnp1 y + cn y_n + cnm1 y_{n-1} + cf f(y) [+ cfn f(y_n)]
  int scheme = ip->scheme;
  if (scheme == PDA_BDF2 && !d_Uprev) scheme = PDA_BDF1; // first BDF2 step is BDF1
  double cnp1 = 1., cn = -1., cnm1 = 0., cf = -dt, cfn = 0.;
  if (scheme == PDA_BDF2) {
    cn = -4. / 3.;
    cnm1 = 1. / 3.;
    cf = -(2. / 3.) * dt;
  } else if (scheme == PDA_CRANK_NICOLSON) {
    cf = -0.5 * dt;
    cfn = -0.5 * dt;
  }
  PDA_HIP_CHECK(hipMemcpyAsync(Yn, d_U, sizeof(double) * n, hipMemcpyDeviceToDevice, st));
  PDA_HIP_CHECK(hipMemcpyAsync(Y, d_guess ? d_guess : d_U, sizeof(double) * n, hipMemcpyDeviceToDevice, st));
  int rc;
  if (scheme == PDA_CRANK_NICOLSON) {
    rc = launch_velocity(p, Yn, t, Fn, st);
    if (rc) return rc;
  }
  pda_implicit_stats S{};
  S.converged = 0;
  double *pres = ip->part[P_RES].as<double>(), *pdx = ip->part[P_DX].as<double>(), *h = ip->host;
  const double *Rx2 = scheme == PDA_BDF2 ? d_Uprev : (scheme == PDA_CRANK_NICOLSON ? Fn : nullptr);
  const double c2 = scheme == PDA_BDF2 ? cnm1 : cfn;
  const bool by_residual = ip->stop == PDA_STOP_RESIDUAL;
  // R(Y) and its partial sums.  Residual rule: from the velocity alone, the
  // Jacobian only when another Newton correction is needed; correction rule:
  // f(y) and df/dy from one evaluation (the Jacobian path's velocity, as
  // pressio's residual-and-Jacobian call)
  auto evaluate = [&]() -> int {
    const int e = by_residual ? launch_velocity(p, Y, t + dt, F, st) : launch_jacobian(p, Y, t + dt, J, F, st);
    if (e) return e;
    hipLaunchKernelGGL(k_residual, dim3(gs), dim3(TB), 0, st, R, Y, cnp1, Yn, cn, Rx2, c2, F, cf, n, pres);
    PDA_HIP_CHECK(hipGetLastError());
    return PDA_OK;
  };
  // the norms of the given partial sums on the host
  auto norms = [&](const double *a, const double *b) -> int {
    hipLaunchKernelGGL(k_norms_out, dim3(1), dim3(TB), 0, st, a, b, int(gs), h);
    PDA_HIP_CHECK(hipGetLastError());
    PDA_HIP_CHECK(hipStreamSynchronize(st));
    return PDA_OK;
  };
  auto fail = [&](const char *what) -> int {
    // pressio: ResidualHasNans -> NonlinearSolveFailure, the stepper
    // restores y_n (solvers_nonlinear/impl/root_finder.cpp:60-70,
    // ode/impl/ode_implicit_stepper_standard.hpp:213-225); d_U has not
    // been written yet
    ip->last = S;
    if (stats) *stats = S;
    ip->forget_iters();
    set_error(std::string("pda_implicit_step: ") + what);
    return PDA_E_STATE;
  };
  rc = evaluate();
  if (!rc) rc = norms(pres, nullptr);
  if (rc) return rc;
  double rnorm = h[0];
  for (int it = 0; it < ip->max_newton; ++it) {
    S.residual_norm = rnorm;
    if (it == 0) S.initial_residual_norm = rnorm;
    if (!std::isfinite(rnorm)) return fail("residual is not finite");
    if (by_residual) {
      if (rnorm <= ip->tol) {
        S.converged = 1;
        break;
      }
      rc = launch_jacobian(p, Y, t + dt, J, nullptr, st);
      if (rc) return rc;
    }
    int li = 0;
    double lr = 0.;
    // residual rule: inexact Newton, the linear residual only needs to fall
    // well below the nonlinear target (relative 0.1 tol / ||R||, within
    // [lin_rtol, 0.1]); correction rule: solve to lin_rtol (pressio's
    // BiCGSTAB runs to machine precision)
    double rtol = ip->lin_rtol;
    if (by_residual && rnorm > 0.) rtol = std::min(0.1, std::max(ip->lin_rtol, 0.1 * ip->tol / rnorm));
    // by residual the correction is applied with its norm's partial sums
    rc = bicgstab(*ip, cf, cnp1, by_residual ? Y : nullptr, st, rtol, it, &li, &lr);
    if (rc) return rc;
    S.linear_iters += li;
    S.last_linear_rel_residual = lr;
    S.newton_iters = it + 1;
    const bool more = it + 1 < ip->max_newton;
    if (by_residual) {
      // the next residual and both norms in one go: a non-finite correction
      // is found before d_U is written
      if (more) rc = evaluate();
      if (!rc) rc = norms(pdx, more ? pres : nullptr);
      if (rc) return rc;
      S.correction_norm = h[0];
      if (!std::isfinite(S.correction_norm)) return fail("Newton correction is not finite");
      if (more) rnorm = h[1];
    } else {
      rc = norms(pdx, nullptr);
      if (rc) return rc;
      S.correction_norm = h[0];
      if (!std::isfinite(S.correction_norm)) return fail("Newton correction is not finite");
      if (S.correction_norm < ip->tol) {
        S.converged = 1;
        break;
      }
      hipLaunchKernelGGL(k_correct, dim3(grid_of(n)), dim3(TB), 0, st, Y, ip->dx.as<double>(), n);
      PDA_HIP_CHECK(hipGetLastError());
      if (!more) break;
      rc = evaluate();
      if (!rc) rc = norms(pres, nullptr);
      if (rc) return rc;
      rnorm = h[0];
    }
  }
  PDA_HIP_CHECK(hipMemcpyAsync(d_U, Y, sizeof(double) * n, hipMemcpyDeviceToDevice, st));
  PDA_HIP_CHECK(hipStreamSynchronize(st));
  ip->last = S;
  if (stats) *stats = S;
  if (!S.converged) {
    ip->forget_iters();
    set_error("pda_implicit_step: Newton did not converge within the iteration limit");
    return PDA_E_STATE;
  }
  return PDA_OK;
}

}  // extern "C"

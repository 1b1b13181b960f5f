// pda_rows.hpp -- per-row device code of the generic kernels: the lanes of one
// graph row (one sample-mesh cell) produce all of its V entries, one thread its
// whole Jacobian block-row, so every output value is written exactly once with
// plain stores (no atomics, no zero-fill pass).  The
// per-entry accumulation order follows the reference:
//   - V: x, then y, then z axis, then sources
//     (impl/mixin_directional_flux_balance.hpp:68-84);
//   - interior Jacobian: chain rule flux-Jacobian x reconstruction gradient,
//     left face then right face per axis
//     (impl/mixin_directional_flux_balance_jacobian.hpp:142-284);
//   - near-boundary rows: first-order blocks with BC factors folded into the
//     diagonal block (impl/mixin_directional_flux_balance_jacobian.hpp:311-371).
#pragma once
#include "pda_families.hpp"

namespace pda {
namespace rows {
using namespace fam;

// ---------------------------------------------------------------- velocity
// A row is evaluated by DIM lanes, lane a forming axis a's part on states in
// the axis frame (one instruction stream for the axes); the parts are then
// added in axis order, every lane of the row ending with the sum.  One lane
// per row walked its axes one after the other, and a mesh of 10^5 rows gave
// the chip 1.6 waves per SIMD: 3D WENO5 velocity of the 5 % sample mesh of
// 128^3 42.6 us, 55.9 us with one lane (64.5 us
// with the reference's four divisions per WENO5 weight set and ghost layers
// written to memory and read back); its near-boundary rows of the full mesh
// 138 -> 72 us.
template <int DIM> constexpr int vel_rows() { return 64 / DIM; } // rows per wavefront

// axis a's part of the velocity of graph row r
template <class Ph, int W>
__device__ __forceinline__ void velocity_axis(const View &P, const int32_t *gr, bool near, int a,
                                              const double *__restrict__ U, double (&acc)[Ph::M]) {
  constexpr int M = Ph::M;
  double st[2 * W + 1][M];
  {
    int32_t src[2 * W + 1];
    int minus, plus;
    stencil_cells<Ph::DIM, W>(P, gr, a, src, minus, plus);
#pragma unroll
    for (int p = 0; p <= 2 * W; ++p) {
      double u[M];
#pragma unroll
      for (int k = 0; k < M; ++k) u[k] = U[int64_t(src[p]) * M + k];
#pragma unroll
      for (int k = 0; k < M; ++k) st[p][k] = perm_pick<Ph>([&](int x) { return u[x]; }, a, k);
    }
    if (minus | plus) {
      double sg[2][M]; // the sides' signs in the axis frame
#pragma unroll
      for (int side = 0; side < 2; ++side)
#pragma unroll
        for (int k = 0; k < M; ++k) {
          double v = P.gsign[0][side][AxisPerm<Ph>::p(k, 0)];
          if constexpr (Ph::DIM > 1) v = a == 1 ? P.gsign[1][side][AxisPerm<Ph>::p(k, 1)] : v;
          if constexpr (Ph::DIM > 2) v = a == 2 ? P.gsign[2][side][AxisPerm<Ph>::p(k, 2)] : v;
          sg[side][k] = v;
        }
#pragma unroll
      for (int p = 0; p <= 2 * W; ++p)
#pragma unroll
        for (int k = 0; k < M; ++k) {
          if (minus >> p & 1) st[p][k] = sg[0][k] * st[p][k];
          if (plus >> p & 1) st[p][k] = sg[1][k] * st[p][k];
        }
    }
  }
  Faces<M, W> f;
  reconstruct<M, W>(st, f);
  double FL[M], FR[M], F[M];
  axis_flux<Ph>(P, a, f.lm, f.lp, FL);
  axis_flux<Ph>(P, a, f.rm, f.rp, FR);
  double h = P.hinv[0];
  if constexpr (Ph::DIM > 1) h = a == 1 ? P.hinv[1] : h;
  if constexpr (Ph::DIM > 2) h = a == 2 ? P.hinv[2] : h;
#pragma unroll
  for (int k = 0; k < M; ++k) F[k] = h * (FL[k] - FR[k]);
#pragma unroll
  for (int k = 0; k < M; ++k) acc[k] = perm_pick<Ph>([&](int x) { return F[x]; }, a, k);
  if (near) {
    if (Ph::DIM == 1 || a == 0) AxisTerms<Ph>::template velocity<0>(P, gr, U, acc);
    else if (Ph::DIM == 2 || a == 1) AxisTerms<Ph>::template velocity<1>(P, gr, U, acc);
    else AxisTerms<Ph>::template velocity<2>(P, gr, U, acc);
  }
}

// The velocity of the visited row of this lane of a wavefront (workgroup wg's
// rows, DIM lanes each) into acc, in every lane of the row; returns the row,
// or -1 for a lane without one.  The whole wavefront takes part.
template <class Ph, int W>
__device__ __forceinline__ int64_t velocity_lanes(const View &P, int64_t wg, const double *__restrict__ U,
                                                  double (&acc)[Ph::M]) {
  constexpr int M = Ph::M, D = Ph::DIM, RPW = vel_rows<D>();
  const int lane = threadIdx.x & 63, g = lane / D, a = lane % D;
  const int64_t t = wg * RPW + g;
  int64_t r = -1;
  bool near = false;
#pragma unroll
  for (int k = 0; k < M; ++k) acc[k] = 0.;
  if (g < RPW && t < P.nvisit) {
    r = P.rows ? P.rows[t] : t;
    near = P.ghost_row[r] >= 0;
    velocity_axis<Ph, W>(P, P.graph + r * P.ncols, near, a, U, acc);
  }
  if constexpr (D > 1) {
#pragma unroll
    for (int k = 0; k < M; ++k) {
      double s = __shfl(acc[k], g * D, 64) + __shfl(acc[k], g * D + 1, 64);
      if constexpr (D > 2) s += __shfl(acc[k], (g * D + 2) & 63, 64);
      acc[k] = s;
    }
  }
  if (r >= 0) Sources<Ph>::apply(P, r, near, U, P.graph[r * P.ncols], acc, nullptr);
  return r;
}

// the velocity of workgroup wg's rows; the row's lanes share its stores
template <class Ph, int W>
__device__ __forceinline__ void velocity_rows(const View &P, int64_t wg, const double *__restrict__ U,
                                              double *__restrict__ V) {
  constexpr int M = Ph::M, D = Ph::DIM;
  double acc[M];
  const int64_t r = velocity_lanes<Ph, W>(P, wg, U, acc);
  if (r < 0) return;
  const int a = int(threadIdx.x) % D;
#pragma unroll
  for (int k = 0; k < M; ++k)
    if (k % D == a) V[r * M + k] = acc[k];
}

// ---------------------------------------------------------------- jacobian
// interior row, one axis
template <class Ph, int W, int A, bool WV>
__device__ __forceinline__ void jac_axis_inner(const View &P, const int32_t *gr,
                                               const uint8_t *sl, const double *__restrict__ U,
                                               double *acc, double (&self)[Ph::M][Ph::M],
                                               double *__restrict__ J, int64_t base, int rs) {
  constexpr int M = Ph::M;
  double st[2 * W + 1][M];
  gather<Ph, W, A>(P, gr, U, st);
  Faces<M, W> f;
  double FL[M], FR[M];
  double JLn[M * M], JLp[M * M], JRn[M * M], JRp[M * M];
  const double h = P.hinv[A];
  if constexpr (W == 1) {
    reconstruct<M, W>(st, f);
    if constexpr (WV) {
      Ph::template flux<A>(P, f.lm, f.lp, FL);
      Ph::template flux<A>(P, f.rm, f.rp, FR);
#pragma unroll
      for (int k = 0; k < M; ++k) acc[k] += h * (FL[k] - FR[k]);
    }
    Ph::template fjac<A>(P, f.lm, f.lp, JLn, JLp);
    Ph::template fjac<A>(P, f.rm, f.rp, JRn, JRp);
    double bl[M][M], br[M][M];
#pragma unroll
    for (int k = 0; k < M; ++k)
#pragma unroll
      for (int j = 0; j < M; ++j) {
        bl[k][j] = 0. + JLn[k * M + j] * h + Sources<Ph>::offdiag(P, false, A, k, j);
        self[k][j] += (JLp[k * M + j] - JRn[k * M + j]) * h;
        br[k][j] = 0. + (-JRp[k * M + j]) * h + Sources<Ph>::offdiag(P, false, A, k, j);
      }
    put_block<M>(P, J, base, rs, sl[colof<Ph::DIM>(A, 0, 0)], bl);
    put_block<M>(P, J, base, rs, sl[colof<Ph::DIM>(A, 1, 0)], br);
  } else {
#pragma clang fp contract(off)
    FaceGrads<M, W> G;
    reconstruct_grad<M, W>(st, f, G);
    if constexpr (WV) {
      Ph::template flux<A>(P, f.lm, f.lp, FL);
      Ph::template flux<A>(P, f.rm, f.rp, FR);
#pragma unroll
      for (int k = 0; k < M; ++k) acc[k] += h * (FL[k] - FR[k]);
    }
    Ph::template fjac<A>(P, f.lm, f.lp, JLn, JLp);
    Ph::template fjac<A>(P, f.rm, f.rp, JRn, JRp);
    // stencil point p (0..2W) collects the left face's gradient index p and
    // the right face's index p-1
#pragma unroll
    for (int p = 0; p <= 2 * W; ++p) {
      double b[M][M];
#pragma unroll
      for (int k = 0; k < M; ++k)
#pragma unroll
        for (int j = 0; j < M; ++j) {
          double v = (p == W) ? self[k][j] : 0.;
          if (p < 2 * W) {
            v += JLn[k * M + j] * G.glm[j][p] * h;
            v += JLp[k * M + j] * G.glp[j][p] * h;
          }
          if (p > 0) {
            v -= JRn[k * M + j] * G.grm[j][p - 1] * h;
            v -= JRp[k * M + j] * G.grp[j][p - 1] * h;
          }
          if (p == W - 1 || p == W + 1) v += Sources<Ph>::offdiag(P, false, A, k, j);
          b[k][j] = v;
        }
      if (p == W) {
#pragma unroll
        for (int k = 0; k < M; ++k)
#pragma unroll
          for (int j = 0; j < M; ++j) self[k][j] = b[k][j];
      } else {
        const int side = p > W ? 1 : 0;
        const int L = p > W ? p - W - 1 : W - 1 - p;
        put_block<M>(P, J, base, rs, sl[colof<Ph::DIM>(A, side, L)], b);
      }
    }
  }
}

// near-boundary row, one axis: velocity from the scheme's stencil (ghosts
// for missing cells), Jacobian first order with the BC factors
template <class Ph, int W, int A, bool WV>
__device__ __forceinline__ void jac_axis_near(const View &P, const int32_t *gr, int64_t g,
                                              const uint8_t *sl, const double *__restrict__ U,
                                              double *acc, double (&self)[Ph::M][Ph::M],
                                              double *__restrict__ J, int64_t base, int rs) {
  constexpr int M = Ph::M;
  const double h = P.hinv[A];
  double FL[M], FR[M];
  double st1[3][M];
  gather<Ph, 1, A>(P, gr, U, st1);
  Faces<M, 1> f1;
  reconstruct<M, 1>(st1, f1);
  if constexpr (WV) {
    if constexpr (W == 1) {
      Ph::template flux<A>(P, f1.lm, f1.lp, FL);
      Ph::template flux<A>(P, f1.rm, f1.rp, FR);
    } else {
      double st[2 * W + 1][M];
      gather<Ph, W, A>(P, gr, U, st);
      Faces<M, W> f;
      reconstruct<M, W>(st, f);
      Ph::template flux<A>(P, f.lm, f.lp, FL);
      Ph::template flux<A>(P, f.rm, f.rp, FR);
    }
#pragma unroll
    for (int k = 0; k < M; ++k) acc[k] += h * (FL[k] - FR[k]);
  }
  double JLn[M * M], JLp[M * M], JRn[M * M], JRp[M * M];
  Ph::template fjac<A>(P, f1.lm, f1.lp, JLn, JLp);
  Ph::template fjac<A>(P, f1.rm, f1.rp, JRn, JRp);
  const int32_t l0 = gr[colof<Ph::DIM>(A, 0, 0)], r0 = gr[colof<Ph::DIM>(A, 1, 0)];
  const double *fac = P.bcf + (g * Ph::DIM + A) * M;
#pragma unroll
  for (int k = 0; k < M; ++k)
#pragma unroll
    for (int j = 0; j < M; ++j) self[k][j] += (JLp[k * M + j] - JRn[k * M + j]) * h;
  if (l0 != -1) {
    double b[M][M];
#pragma unroll
    for (int k = 0; k < M; ++k)
#pragma unroll
      for (int j = 0; j < M; ++j) {
        b[k][j] = 0. + JLn[k * M + j] * h;
        if constexpr (AxisTerms<Ph>::near_offdiag) b[k][j] += Sources<Ph>::offdiag(P, true, A, k, j);
      }
    put_block<M>(P, J, base, rs, sl[colof<Ph::DIM>(A, 0, 0)], b);
  }
  if (r0 != -1) {
    double b[M][M];
#pragma unroll
    for (int k = 0; k < M; ++k)
#pragma unroll
      for (int j = 0; j < M; ++j) {
        b[k][j] = 0. + (-JRp[k * M + j]) * h;
        if constexpr (AxisTerms<Ph>::near_offdiag) b[k][j] += Sources<Ph>::offdiag(P, true, A, k, j);
      }
    put_block<M>(P, J, base, rs, sl[colof<Ph::DIM>(A, 1, 0)], b);
  }
  if (l0 == -1) {
#pragma unroll
    for (int k = 0; k < M; ++k)
#pragma unroll
      for (int j = 0; j < M; ++j) self[k][j] += (fac[j] * JLn[k * M + j]) * h;
  }
  if (r0 == -1) {
#pragma unroll
    for (int k = 0; k < M; ++k)
#pragma unroll
      for (int j = 0; j < M; ++j) self[k][j] += (fac[j] * -JRp[k * M + j]) * h;
  }
}

// Jacobian block-row (and velocity when WV, rightHandSideAndJacobian) of
// visited row t
template <class Ph, int W, bool WV>
__device__ __forceinline__ void jacobian_row(const View &P, int64_t t, const double *__restrict__ U,
                                             double *__restrict__ V, double *__restrict__ J) {
  constexpr int M = Ph::M;
  if (t >= P.nvisit) return;
  const int64_t r = P.rows ? P.rows[t] : t;
  const int32_t *gr = P.graph + r * P.ncols;
  const int64_t g = P.ghost_row[r];
  const uint8_t *sl = P.slot + r * P.npos;
  const int64_t base = P.rowbase[r];
  const int rs = P.nblk[r] * M;
  double acc[M];
  double self[M][M];
#pragma unroll
  for (int k = 0; k < M; ++k) {
    acc[k] = 0.;
#pragma unroll
    for (int j = 0; j < M; ++j) self[k][j] = 0.;
  }
  if (g < 0) {
    jac_axis_inner<Ph, W, 0, WV>(P, gr, sl, U, acc, self, J, base, rs);
    if constexpr (Ph::DIM > 1) jac_axis_inner<Ph, W, 1, WV>(P, gr, sl, U, acc, self, J, base, rs);
    if constexpr (Ph::DIM > 2) jac_axis_inner<Ph, W, 2, WV>(P, gr, sl, U, acc, self, J, base, rs);
  } else {
    jac_axis_near<Ph, W, 0, WV>(P, gr, g, sl, U, acc, self, J, base, rs);
    if constexpr (WV) AxisTerms<Ph>::template velocity<0>(P, gr, U, acc);
    if constexpr (Ph::DIM > 1) {
      jac_axis_near<Ph, W, 1, WV>(P, gr, g, sl, U, acc, self, J, base, rs);
      if constexpr (WV) AxisTerms<Ph>::template velocity<1>(P, gr, U, acc);
    }
    if constexpr (Ph::DIM > 2) {
      jac_axis_near<Ph, W, 2, WV>(P, gr, g, sl, U, acc, self, J, base, rs);
      if constexpr (WV) AxisTerms<Ph>::template velocity<2>(P, gr, U, acc);
    }
  }
  Sources<Ph>::apply(P, r, g >= 0, U, gr[0], acc, &self[0][0]);
  put_block<M>(P, J, base, rs, sl[0], self);
  if constexpr (WV) {
#pragma unroll
    for (int k = 0; k < M; ++k) V[r * M + k] = acc[k];
  }
}

}  // namespace rows
}  // namespace pda

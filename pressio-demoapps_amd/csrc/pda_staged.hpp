// pda_staged.hpp -- rows of the first-order Euler Jacobian staged in LDS, four
// lanes per row: device code shared by the kernels that take such rows.
#pragma once
#include "pda_rows.hpp"

namespace pda {
namespace rows {

// Rows of the first-order Euler Jacobian (Euler has no source term) with
// four lanes per row and 16 rows per wavefront.  Lane a < D evaluates the two
// faces of axis a.  The Euler flux along axis a is the flux along x with
// momentum components 1 and 1+a exchanged, so every lane runs the x-face
// code on exchanged states and writes entry (k, j) of its blocks to
// (p(k), p(j)), p the 1 <-> 1+a exchange: one instruction stream for all
// axes.  A row's blocks are assembled in LDS in CSR order (scalar row k,
// block slot, column), the diagonal block adding the axes in order as the
// generic row code does, and the wavefront then copies each staged row to
// its contiguous CSR values with coalesced streaming stores (one thread per
// row would scatter every store over 64 rows); 16 rows consecutive in the
// CSR leave as one range of 16-byte stores.  Used where no structured box
// kernel applies (sample meshes, 2D meshes given as a graph) and for the
// boundary rows of a structured 3D full mesh.  Bound by latency: a wavefront
// alone takes 11 us (three dependent loads, two faces of divisions and square
// roots, the stage, the copy) and the stage's 23 KB leave 7 of them per CU; 5 %
// sample mesh of 128^3 50.6 us (147 MB of values), 61.7 us with a ghost branch
// per block entry and the rows' CSR offsets fetched one by one at the copy.
// Near-boundary rows: a
// missing neighbour along axis a reads the ghost state sign_k U_k of the row's own cell (the first
// ghost layer of every ghost rule), writes no block, and adds fac_j JL (left
// side) or -fac_j JR (right side) of that face, times h, to the axis's
// diagonal part, fac the row's BC factors (the terms of
// impl/mixin_directional_flux_balance_jacobian.hpp:312-369, with the factors
// of impl/euler_3d_prob_class.hpp:626-651).
constexpr int SJ_LANES = 4, SJ_ROWS = 64 / SJ_LANES;

// the axis frame's dof k (AxisPerm, the same for every dimension)
__device__ __forceinline__ int exch(int k, int a) { return AxisPerm<PhEuler3>::p(k, a); }

// ghost sign of native dof exch(k, a) on side `side` of axis a
template <int D>
__device__ __forceinline__ double ghost_sign(const View &P, int a, int side, int k) {
  const double s0 = P.gsign[0][side][exch(k, 0)];
  const double s1 = D > 1 ? P.gsign[1][side][exch(k, 1)] : 0.;
  const double s2 = D > 2 ? P.gsign[2][side][exch(k, 2)] : 0.;
  return a == 0 ? s0 : (a == 1 ? s1 : s2);
}

// LDS of a wavefront's rows
template <int D> struct StagedLds {
  double stage[SJ_ROWS * (D + 2) * (D + 2) * (1 + 2 * D)];
  int64_t base_of[SJ_ROWS]; // first CSR value of the row, -1: no row
  int blk_of[SJ_ROWS];      // its column blocks
};

// the rows of workgroup wg
template <int D>
__device__ __forceinline__ void jac_fo_euler_staged(const View &P, int64_t wg, const double *__restrict__ U,
                                                    double *__restrict__ J, StagedLds<D> &L) {
  using Ph = PhEuler<D>;
  constexpr int M = D + 2, NB = 1 + 2 * D, RS = NB * M, PER = M * RS;
  double *stage = L.stage;
  int64_t *base_of = L.base_of;
  int *blk_of = L.blk_of;
  const int lane = threadIdx.x, g = lane / SJ_LANES, a = lane % SJ_LANES;
  const int64_t t = wg * SJ_ROWS + g;
  int64_t r = -1;
  if (t < P.nvisit) {
    const int64_t rr = P.rows ? P.rows[t] : t;
    r = rr;
  }
  // the row's place in the CSR, in each of its lanes
  const int64_t base = r >= 0 ? P.rowbase[r] : -1;
  const int nblk = r >= 0 ? P.nblk[r] : 0;
  if (a == 0) {
    base_of[g] = base;
    blk_of[g] = nblk;
  }
  const bool act = r >= 0 && a < D;
  double *st = stage + g * PER;
  typename Ph::Side Ln, Lp, Rn, Rp;
  int sL = 0, sR = 0, s0 = 0;
  bool gl = false, gr_ = false; // no neighbour on the left / right
  double fac[M];                // BC factors of native dof exch(j, a)
  double h = 0.;
  if (act) {
    int64_t cells[3];
    {
      const int32_t *gr = P.graph + r * P.ncols;
      const uint8_t *sl = P.slot + r * P.npos;
      const int cl = colof<D>(a, 0, 0), cr = colof<D>(a, 1, 0);
      const int32_t il = gr[cl], ir = gr[cr];
      gl = il < 0;
      gr_ = ir < 0;
      cells[0] = gl ? gr[0] : il;
      cells[1] = gr[0];
      cells[2] = gr_ ? gr[0] : ir;
      sL = gl ? 0 : sl[cl];
      sR = gr_ ? 0 : sl[cr];
      s0 = sl[0];
    }
    double q[3][M];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int k = 0; k < M; ++k) q[c][k] = U[cells[c] * M + exch(k, a)];
#pragma unroll
    for (int k = 0; k < M; ++k) {
      if (gl) q[0][k] = ghost_sign<D>(P, a, 0, k) * q[0][k];
      if (gr_) q[2][k] = ghost_sign<D>(P, a, 1, k) * q[2][k];
      fac[k] = 0.;
    }
    const int64_t gi = P.ghost_row[r];
    if ((gl || gr_) && gi >= 0) {
      const double *f = P.bcf + (gi * D + a) * M;
#pragma unroll
      for (int k = 0; k < M; ++k) fac[k] = f[exch(k, a)];
    }
    Ph::template sides<0>(P, q[0], q[1], Ln, Lp);
    Ph::template sides<0>(P, q[1], q[2], Rn, Rp);
    h = P.hinv[a];
  }
  // a fence between the face math and the stage stores keeps the entry
  // evaluations from being hoisted into it (2D: 148 -> 126 registers)
  wave_sync();
  auto put = [&](int slot, const typename Ph::Side &S, bool minus) {
#pragma unroll
    for (int k = 0; k < M; ++k)
#pragma unroll
      for (int j = 0; j < M; ++j) {
        const double v = Ph::template entry<0>(P, S, k, j);
        st[exch(k, a) * RS + exch(j, a) + slot * M] = 0. + (minus ? -v : v) * h;
      }
  };
  if (act && !gl) put(sL, Ln, false);
  if (act && !gr_) put(sR, Rp, true);
  // every lane forms its axis's part of the diagonal block at once; the
  // axes then add their parts in order, one axis at a time, in LDS
  double dg[M][M];
  wave_sync();
  if (act) {
#pragma unroll
    for (int k = 0; k < M; ++k)
#pragma unroll
      for (int j = 0; j < M; ++j)
        dg[k][j] = (Ph::template entry<0>(P, Lp, k, j) - Ph::template entry<0>(P, Rn, k, j)) * h;
  }
  if (act && gl) {
#pragma unroll
    for (int k = 0; k < M; ++k)
#pragma unroll
      for (int j = 0; j < M; ++j) dg[k][j] += (fac[j] * Ph::template entry<0>(P, Ln, k, j)) * h;
  }
  if (act && gr_) {
#pragma unroll
    for (int k = 0; k < M; ++k)
#pragma unroll
      for (int j = 0; j < M; ++j) dg[k][j] += (fac[j] * -Ph::template entry<0>(P, Rp, k, j)) * h;
  }
#pragma unroll
  for (int ax = 0; ax < D; ++ax) {
    wave_sync();
    if (act && a == ax) {
#pragma unroll
      for (int k = 0; k < M; ++k)
#pragma unroll
        for (int j = 0; j < M; ++j) {
          const int o = exch(k, a) * RS + s0 * M + exch(j, a);
          st[o] = (ax == 0 ? 0. : st[o]) + dg[k][j];
        }
    }
  }
  wave_sync();
  // Copy-out from the row table in LDS alone: the rows' CSR offsets were
  // loaded with their states (not here, one row after the other).  Whole
  // rows leave as one flattened loop over their values: 16-byte stores where
  // every row starts on a 16-byte boundary (2D, if J does, and rows consecutive in
  // the CSR after a leading value), else 8-byte ones.
  const int64_t rb0 = base_of[0];
  const bool whole = __all(base >= 0 && nblk == NB);
  const bool run = __all(base == rb0 + int64_t(g) * PER);
  if (whole && run) {
    constexpr int TOT = SJ_ROWS * PER;
    double *dst = J + rb0;
    const int head = int(reinterpret_cast<uintptr_t>(dst) >> 3 & 1); // a leading value that is not 16-byte aligned
    if (head && lane == 0) store_stream(dst, stage[0]);
    const int npairs = (TOT - head) / 2;
    double2 *d2 = reinterpret_cast<double2 *>(dst + head);
#pragma unroll 4
    for (int q = lane; q < npairs; q += 64)
      store_stream(d2 + q, make_double2(stage[head + 2 * q], stage[head + 2 * q + 1]));
    if (((TOT - head) & 1) && lane == 0) store_stream(dst + TOT - 1, stage[TOT - 1]);
    return;
  }
  if (whole) {
    if (PER % 2 == 0 && reinterpret_cast<uintptr_t>(J) % 16 == 0) {
#pragma unroll 4
      for (int q = lane; q < SJ_ROWS * (PER / 2); q += 64) {
        const int gg = q / (PER / 2), e = 2 * (q - gg * (PER / 2));
        const double *src = stage + gg * PER + e;
        store_stream(reinterpret_cast<double2 *>(J + base_of[gg] + e), make_double2(src[0], src[1]));
      }
    } else {
#pragma unroll 4
      for (int q = lane; q < SJ_ROWS * PER; q += 64) {
        const int gg = q / PER;
        store_stream(J + base_of[gg] + (q - gg * PER), stage[q]);
      }
    }
    return;
  }
  // Near-boundary rows hold nblk of the NB block slots per scalar row.  Their
  // rows in one loop where the wavefronts are few and each one's time counts
  // (2D: the rim of a grid, 9.4 us a launch, 11.2 row after row); row after row
  // in 3D, where they fill the chip and the index arithmetic counts (128^3's
  // boundary rows 78 us, 87 in one loop).
  if constexpr (D == 2) {
#pragma unroll 4
    for (int q = lane; q < SJ_ROWS * PER; q += 64) {
      const int gg = q / PER, e = q - gg * PER;
      const int64_t rb = base_of[gg];
      const int rs = blk_of[gg] * M;
      int k = 0;
#pragma unroll
      for (int c = 1; c < M; ++c) k += e >= c * rs;
      if (rb >= 0 && e < M * rs) store_stream(J + rb + e, stage[gg * PER + k * RS + (e - k * rs)]);
    }
  } else {
#pragma clang loop unroll(disable)
    for (int gg = 0; gg < SJ_ROWS; ++gg) {
      const int64_t rb = base_of[gg];
      if (rb < 0) continue;
      double *dst = J + rb;
      const double *src = stage + gg * PER;
      const int rs = blk_of[gg] * M;
      for (int e = lane; e < M * rs; e += 64) {
        int k = 0;
#pragma unroll
        for (int q = 1; q < M; ++q) k += e >= q * rs;
        store_stream(dst + e, src[k * RS + (e - k * rs)]);
      }
    }
  }
}

}  // namespace rows
}  // namespace pda

// pda_apply.hip -- the Jacobian action AJ = J B (applyJacobian) over the
// Jacobian's blocks.
#include "pda_internal.hpp"

namespace pda {
namespace {

// AJ = J * B over the Jacobian's blocks: a cell's rows hold, for each of its
// nblk column cells, an M x M block, so one column-cell index serves M*M
// values, and the M rows of B that a block reads are consecutive.  Bound by
// the reads of B: the cells of a stencil are scattered, and a block needs
// M ncols values of B for its M*M own.
//
// k_apply_cols, many columns of a row-major B: L lanes per cell, a lane
// holding VW columns of its M results, and 256 / L cells of a block of threads
// (inv = 2^16 / L rounded up, so that thread t's cell is t inv >> 16: exact for t <
// 256 and L <= 64); the block's values are the same for the L lanes (one broadcast load), its M rows of B contiguous runs over
// them.  10 % sample mesh of 512 x 400, WENO3, 32 columns: 133 -> 36 us
// (186 MB of B and AJ: 5.1 TB/s) against a thread per entry of AJ walking the
// scalar CSR, which read every value and column index ncols times.
template <int M, int VW>
__global__ void __launch_bounds__(256) k_apply_cols(View P, const int32_t *__restrict__ bcol, int maxb,
                                                    const double *__restrict__ J, const double *__restrict__ B,
                                                    int64_t ncols, int L, int inv, double *__restrict__ AJ) {
  typedef double vec __attribute__((ext_vector_type(VW)));
  const int g = int(threadIdx.x) * inv >> 16, cells = 256 * inv >> 16; // its cell; cells of the block
  const int64_t r = int64_t(blockIdx.x) * cells + g;
  if (g >= cells || r >= P.nrows) return;
  const int64_t c0 = (int64_t(blockIdx.y) * L + (int(threadIdx.x) - g * L)) * VW;
  if (c0 >= ncols) return;
  const int nb = P.nblk[r];
  const int32_t *bc = bcol + r * maxb;
  const double *Jr = J + P.rowbase[r];
  vec acc[M];
#pragma unroll
  for (int k = 0; k < M; ++k) acc[k] = vec(0.);
#pragma unroll 4
  for (int s = 0; s < nb; ++s) {
    const double *b = B + int64_t(bc[s]) * M * ncols + c0;
    vec x[M];
#pragma unroll
    for (int j = 0; j < M; ++j) x[j] = *reinterpret_cast<const vec *>(b + j * ncols);
#pragma unroll
    for (int k = 0; k < M; ++k)
#pragma unroll
      for (int j = 0; j < M; ++j) acc[k] += Jr[(k * nb + s) * M + j] * x[j];
  }
#pragma unroll
  for (int k = 0; k < M; ++k) *reinterpret_cast<vec *>(AJ + (r * M + k) * ncols + c0) = acc[k];
}

// k_apply_rows, few columns, or a column-major B: L lanes per cell over the
// nblk M column entries of its rows (J's rows are contiguous runs over them),
// NC columns at a time; the later passes over the columns find the cell's
// values in the CU's cache.  The lanes' sums are combined by halving: a lane
// sends the half of its sums that it gives up and keeps the other, so M NC
// sums cost M NC - 1 exchanges and end spread over the lanes, which store one
// or two each (every lane reducing every sum: M NC log2 L exchanges, the larger
// part of the kernel's time).  WENO3 on 512 x 400 (J is 236 MB): one vector
// 1029 -> 54 us, 6 columns 469 -> 98 us row-major and 6295 -> 99 us
// column-major, against a thread per entry of AJ.
template <int M> constexpr int apply_lanes() { return M == 1 ? 8 : 16; } // 5 to 13 entries a row, else 9 to 52 (2D)

template <int M, int NC>
__global__ void __launch_bounds__(256) k_apply_rows(View P, const int32_t *__restrict__ bcol, int maxb,
                                                    const double *__restrict__ J, const double *__restrict__ B,
                                                    int64_t ncols, int64_t bstride, int64_t bcolstride,
                                                    int64_t astride, int64_t acolstride, double *__restrict__ AJ) {
  constexpr int L = apply_lanes<M>();
  constexpr int V = M * NC <= 1 ? 1 : M * NC <= 2 ? 2 : M * NC <= 4 ? 4 : M * NC <= 8 ? 8 : M * NC <= 16 ? 16
                    : M * NC <= 32 ? 32 : 64;
  const int64_t r = int64_t(blockIdx.x) * (256 / L) + threadIdx.x / L;
  if (r >= P.nrows) return; // the L lanes of a cell leave together
  const int l = threadIdx.x % L;
  const int nb = P.nblk[r], n = nb * M;
  const int32_t *bc = bcol + r * maxb;
  const double *Jr = J + P.rowbase[r];
  for (int64_t c0 = 0; c0 < ncols; c0 += NC) {
    double acc[V]; // acc[k * NC + c]
#pragma unroll
    for (int q = 0; q < V; ++q) acc[q] = 0.;
    for (int e = l; e < n; e += L) {
      const double *b = B + (int64_t(bc[e / M]) * M + e % M) * bstride;
      double x[NC], v[M];
#pragma unroll
      for (int c = 0; c < NC; ++c) x[c] = c0 + c < ncols ? b[(c0 + c) * bcolstride] : 0.;
#pragma unroll
      for (int k = 0; k < M; ++k) v[k] = Jr[k * n + e];
#pragma unroll
      for (int k = 0; k < M; ++k)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[k * NC + c] += v[k] * x[c];
    }
    // after the steps, acc[0 .. V / L) are the sums from `first` on
    int first = 0;
#pragma unroll
    for (int st = 0; (L >> st) > 1; ++st) {
      const int o = L >> (st + 1), w = V >> st;
      const bool up = l & o;
      if (w > 1) {
#pragma unroll
        for (int q = 0; q < w / 2; ++q) {
          double lo = acc[q], hi = acc[w / 2 + q];
          // both read before the choice: the compiler otherwise chooses the index
          // and searches acc for it (at 16 sums 1,300 more instructions: five
          // row-major columns of first-order Burgers on 500 x 512 cells 180 us
          // with the Jacobian, 56 now)
          asm volatile("" : "+v"(lo), "+v"(hi));
          const double keep = up ? hi : lo, give = up ? lo : hi;
          acc[q] = keep + __shfl_xor(give, o, 64);
        }
        if (up) first += w / 2;
      } else { // fewer sums than lanes
        acc[0] += __shfl_xor(acc[0], o, 64);
      }
    }
    constexpr int LEFT = V > L ? V / L : 1;
#pragma unroll
    for (int q = 0; q < LEFT; ++q) {
      const int i = first + q, c = i % NC, k = i / NC;
      const bool mine = V >= L || (l & (L / (V < L ? V : L) - 1)) == 0;
      if (mine && k < M && c0 + c < ncols) AJ[(r * M + k) * astride + (c0 + c) * acolstride] = acc[q];
    }
  }
}

}  // namespace

// AJ = J B: the lanes of a cell over the columns where B is row-major and
// they fill at least four lanes, else over the entries of the cell's rows (9
// columns of the sample mesh above: 29 us over the columns; 3 columns 22.5 us
// over the entries)
template <int M>
static int apply_m(const pda_problem_s &p, const double *J, const double *B, int64_t ncols, int layout, double *AJ,
                   hipStream_t s) {
  const View &v = p.view;
  const int32_t *bc = p.d_bcol.as<int32_t>();
  if (layout == 1 && ncols >= 8) {
    // two columns per lane where every row of B and AJ is 16-byte aligned
    const int vw = ncols % 2 == 0 && (reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(AJ)) % 16 == 0 ? 2 : 1;
    // the lanes in equal parts of at most 64, no more than they are: rounded up to
    // a power of two, 33 columns left 31 of 64 lanes idle (scalar family on 600 x
    // 500 cells, first order: 135 us with the Jacobian, 88 now)
    const int64_t lanes = (ncols + vw - 1) / vw, parts = (lanes + 63) / 64;
    const int L = int((lanes + parts - 1) / parts), inv = (65536 + L - 1) / L;
    const dim3 grid{unsigned((v.nrows + 256 / L - 1) / (256 / L)), unsigned(parts), 1};
    if (vw == 2) hipLaunchKernelGGL((k_apply_cols<M, 2>), grid, dim3(256), 0, s, v, bc, p.maxb, J, B, ncols, L, inv, AJ);
    else hipLaunchKernelGGL((k_apply_cols<M, 1>), grid, dim3(256), 0, s, v, bc, p.maxb, J, B, ncols, L, inv, AJ);
    PDA_HIP_CHECK(hipGetLastError());
    return PDA_OK;
  }
  constexpr int L = apply_lanes<M>();
  const int64_t nst = p.mesh->n_stencil * p.m, ns = v.nrows * p.m;
  const int64_t bs = layout == 0 ? 1 : ncols, bcs = layout == 0 ? nst : 1;
  const int64_t as = layout == 0 ? 1 : ncols, acs = layout == 0 ? ns : 1;
  const unsigned gx = unsigned((v.nrows + 256 / L - 1) / (256 / L));
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(gx), dim3(256), 0, s, v, bc, p.maxb, J, B, ncols, bs, bcs, as, acs, AJ);
  };
  if (ncols == 1) go(k_apply_rows<M, 1>);
  else if (ncols == 2) go(k_apply_rows<M, 2>);
  else if (ncols <= 4) go(k_apply_rows<M, 4>);
  else go(k_apply_rows<M, 8>);
  PDA_HIP_CHECK(hipGetLastError());
  return PDA_OK;
}

int launch_apply(const pda_problem_s &p, const double *J, const double *B, int64_t ncols,
                 int layout, double *AJ, hipStream_t s) {
  if (p.view.nrows == 0 || ncols == 0) return PDA_OK;
  switch (p.m) {
    case 1: return apply_m<1>(p, J, B, ncols, layout, AJ, s);
    case 2: return apply_m<2>(p, J, B, ncols, layout, AJ, s);
    case 3: return apply_m<3>(p, J, B, ncols, layout, AJ, s);
    case 4: return apply_m<4>(p, J, B, ncols, layout, AJ, s);
    case 5: return apply_m<5>(p, J, B, ncols, layout, AJ, s);
  }
  set_error("applyJacobian: unsupported block size");
  return PDA_E_UNSUPPORTED;
}

}  // namespace pda

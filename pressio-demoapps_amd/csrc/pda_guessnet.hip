// pda_guessnet.hip -- the learned initial guess for implicit Newton steps on
// periodic 2D two-component fields (the Burgers problem): a 4-layer 3x3
// convolutional network, 32 channels, BF16 weights and activations with
// FP32 accumulation on the MFMA units (v_mfma_f32_16x16x32_bf16), trained
// on the device by the kernels below (forward, backward-data,
// backward-weight, Adam).
//
//   The guess is an FP64 predictor of y_{n+1} of a fractional extrapolation
//   order t in [1, 4] that the network picks per step.  The predictors are
//   the BDF2 relation y = (4/3) y_n - (1/3) y_{n-1} + (2/3) dt f(y) with
//   f(y_{n+1}) extrapolated in time with order k from f_n, ..., f_{n-k}:
//     P_k = (4/3) y_n - (1/3) y_{n-1} + (2/3) dt E_k,
//     E_1 = 2 f_n - f_{n-1},  E_2 = 3 f_n - 3 f_{n-1} + f_{n-2},
//     E_3 = 4 f_n - 6 f_{n-1} + 4 f_{n-2} - f_{n-3},
//     E_4 = 5 f_n - 10 f_{n-1} + 10 f_{n-2} - 5 f_{n-3} + f_{n-4};
//   P(t) interpolates linearly between P_k and P_{k+1} (k = floor(t)).
//   The network's NOUT = 7 output channels, averaged over the grid, are
//   its estimates m_j of what the step costs from P(T_j), T_j = 1 + j/2
//   (j = 0..6), relative to the mean over the orders; t = sum_j p_j T_j
//   with p = softmax(-m / kTau), a soft arg-min (kTau = 1/4 iteration).
//   Training minimises sum_j (m_j - (c_j - mean c))^2 / 7 of a sample, c_j
//   being what the step cost from P(T_j) (the package measures the Newton +
//   Krylov iterations when it makes the sample).  The order that pays
//   changes with the flow: on
//   smooth fields the highest one (the guess error is O(dt^{k+2})), near
//   steep fronts a low one (higher-order extrapolation in time of a front
//   passing a cell amplifies grid-scale error, which costs Newton
//   iterations even where it lowers ||guess - y_{n+1}||_2).
//   Every field the guess adds is FP64 and the network contributes one
//   number, t, so its BF16 rounding cannot put pixel-scale noise into the
//   guess (the Newton and Krylov work grows with the high-frequency content
//   of the guess's error, which pixel noise is).
//   features (8 ch): dt D^k f / s_k for k = 1, 2, 3 (2 channels each, D^k
//                    the k-th backward time difference of f), nu_hat,
//                    |dt D^4 f| / s_4 (f = the problem's velocity, FP64)
//   L1 8->32 SiLU, L2 32->32 SiLU, L3 32->32 SiLU, L4 32->7 (linear)
//   (periodic padding)
// Every convolution is an implicit GEMM: D[cout][pixel] += A[cout][k] B[k][pixel]
// over K = taps x input channels, 32 K per MFMA.  An MFMA pairs A's and B's K
// elements by register position, so any consistent assignment of K to
// (lane group, register element) is valid; the kernels use K = 8*g + j for
// lane group g = lane/16 and element j.  The output layout used is the
// 16x16 MFMA's: lane l holds D[4*(l/16) + i][l%16], i = 0..3; A row = l%16,
// B column = l%16.
#include <algorithm>
#include <cmath>

#include "pda_internal.hpp"

namespace pda {
namespace nn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int C = 32;      // hidden channels
constexpr int CIN0 = 8;    // feature channels (7 used)
constexpr int NOUT = 7;    // output channels: logits of the orders 1, 1.5, ..., 4
constexpr int NCOMP = 2;   // field components per pixel
constexpr int NL = 4;      // layers

// layer geometry: input channels, output channels
__host__ __device__ constexpr int cin_of(int l) { return l == 0 ? CIN0 : C; }
__host__ __device__ constexpr int cout_of(int l) { return l == NL - 1 ? NOUT : C; }
// K steps of 32 of a forward layer: 9 taps x 32 channels, or 9 taps x 8
// channels packed four taps per step
__host__ __device__ constexpr int ksteps(int cin) { return cin == C ? 9 : 3; }

// 1 / (1 + exp(-z)): the hardware reciprocal and one Newton step (exp's own
// error is the larger; the IEEE division is three times the instructions, a
// third of a hidden layer's vector work).  z is kept above -87, where the
// value is 1e-38, so that exp stays finite and the step defined.
__device__ __forceinline__ float sigmoid(float z) {
  const float d = 1.f + __expf(-__builtin_amdgcn_fmed3f(z, -87.f, 3.4e38f)); // fmaxf's two instructions in one
  const float r = __builtin_amdgcn_rcpf(d);
  return __fmaf_rn(r, __fmaf_rn(-d, r, 1.f), r);
}
__device__ __forceinline__ float silu(float z) { return z * sigmoid(z); }
__device__ __forceinline__ float dsilu(float z) {
  const float s = sigmoid(z);
  return s * (1.f + z * (1.f - s));
}

// the velocities the predictors read: f[0] = f(y_n), ..., f[4] = f(y_{n-4})
struct FHist {
  const double *f[5];
};

// features of pixel p: dt D^k f / s_k (k = 1, 2, 3; 2 channels each), nu_hat,
// |dt D^4 f| / s_4
struct Features {
  FHist F;
  double c[4], nu_hat;
};
__device__ __forceinline__ bf16x8 features(const Features &T, int64_t p) {
  bf16x8 x;
  double n4 = 0.;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int64_t i = 2 * p + c;
    const double f0 = T.F.f[0][i], f1 = T.F.f[1][i], f2 = T.F.f[2][i], f3 = T.F.f[3][i], f4 = T.F.f[4][i];
    const double d1 = f0 - f1, d2 = f0 - 2. * f1 + f2, d3 = f0 - 3. * f1 + 3. * f2 - f3;
    const double d4 = f0 - 4. * f1 + 6. * f2 - 4. * f3 + f4;
    x[c] = __bf16(float(d1 * T.c[0]));
    x[2 + c] = __bf16(float(d2 * T.c[1]));
    x[4 + c] = __bf16(float(d3 * T.c[2]));
    n4 += (d4 * T.c[3]) * (d4 * T.c[3]);
  }
  x[6] = __bf16(float(T.nu_hat));
  x[7] = __bf16(float(sqrt(n4)));
  return x;
}

// Forward convolution (and, with MODE_BWD, the backward-data convolution).
//   Wp: packed weights [kstep][ncout_pad][32] bf16 (A operand rows)
//   MODE_FIRST:  as MODE_HIDDEN on the 8 features, formed from the velocity
//                history while the tile is staged and, with X0, kept for the
//                backward
//   MODE_HIDDEN: Z = acc + bias (FP32, kept for the backward; not stored
//                when Z is null, as in inference), Y = SiLU(Z) (bf16); with
//                csum, also the block's per-channel sums of Y (FP32,
//                csum[c][block])
//   MODE_OUT:    out[p][c] = acc + bias for c < NOUT (FP32)
//   MODE_BWD:    dZprev[p][c] = acc * SiLU'(Zprev[p][c]) (bf16), no bias
// A workgroup of four waves owns a tile of 128 RW pixels, TW columns x 128 RW / TW
// rows (tile_of's choice), 32 RW consecutive ones per wave.  The tile and its halo are staged in LDS once, [pixel][channel]
// as in memory, so a pixel operand is one 16-byte LDS read for every tap and
// no lane computes addresses or wraps per tap; the layer's weights stay in
// registers.  M = output channels and N = pixels, so that a lane ends with
// four consecutive channels of one pixel: 8-byte (Y) and 16-byte (Z) accesses
// instead of one per value.  At 512 x 512 a hidden layer takes 15.9 us (33.5 MB
// in and out: 7 us at the copy rate; SiLU's vector instructions: 4 us; the two
// phases overlap little, as all 512 workgroups run at once), 24.2 us when
// every lane gathered its pixels per tap from memory.  Loading the tile in a
// loop that waits for each 16 bytes took 17.4 us.
enum { MODE_FIRST = 0, MODE_HIDDEN = 1, MODE_OUT = 2, MODE_BWD = 3 };
struct ConvArgs {
  const __bf16 *X, *Wp;
  const float *bias;
  int H, W, ntx;          // grid, tiles across
  float *Z;
  __bf16 *Y, *X0;
  float *out;
  const float *Zprev;
  float *csum;
};

template <int MODE, int RW, int TW>
__global__ void __launch_bounds__(256) k_conv(ConvArgs A, Features T) {
  constexpr int CIN = MODE == MODE_FIRST ? CIN0 : C, NT = MODE == MODE_OUT ? 1 : 2, KS = ksteps(CIN);
  constexpr int TR = 128 * RW / TW, XW = TW + 2, NV = CIN / 8, NPT = 2; // NPT: MFMA pixel tiles of 32 pixels
  __shared__ __align__(16) __bf16 sx[(TR + 2) * XW * CIN];
  __shared__ float ssum[4][C];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
  const int H = A.H, W = A.W;
  const int x0 = (int(blockIdx.x) % A.ntx) * TW, y0 = (int(blockIdx.x) / A.ntx) * TR;
  // every load of the tile in flight before the first LDS store
  constexpr int TOT = (TR + 2) * XW * NV, PER = (TOT + 255) / 256;
  bf16x8 stg[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int q = tid + 256 * k < TOT ? tid + 256 * k : TOT - 1;
    const int v = q % NV, px = q / NV % XW, row = q / (NV * XW);
    int x = x0 - 1 + px, y = y0 - 1 + row;
    // columns past W and rows past H only feed pixels that are not stored
    x = x < 0 ? x + W : (x >= W ? (x == W ? 0 : W - 1) : x);
    y = y < 0 ? y + H : (y >= H ? (y == H ? 0 : H - 1) : y);
    const int64_t p = int64_t(y) * W + x;
    if constexpr (MODE == MODE_FIRST) {
      stg[k] = features(T, p);
      if (A.X0 && px >= 1 && px <= TW && row >= 1 && row <= TR && x0 - 1 + px < W && y0 - 1 + row < H)
        *reinterpret_cast<bf16x8 *>(A.X0 + p * CIN) = stg[k];
    } else {
      stg[k] = *reinterpret_cast<const bf16x8 *>(A.X + p * CIN + 8 * v);
    }
  }
#pragma unroll
  for (int k = 0; k < PER; ++k)
    if (tid + 256 * k < TOT) *reinterpret_cast<bf16x8 *>(sx + 8 * (tid + 256 * k)) = stg[k];
  bf16x8 w[KS][NT];
#pragma unroll
  for (int s = 0; s < KS; ++s)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      w[s][nt] = *reinterpret_cast<const bf16x8 *>(A.Wp + (int64_t(s) * (16 * NT) + 16 * nt + r) * 32 + 8 * g);
  f32x4 bias[NT];
  if constexpr (MODE != MODE_BWD) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = 16 * nt + 4 * g + i;
        bias[nt][i] = MODE != MODE_OUT || c < NOUT ? A.bias[c] : 0.f;
      }
  }
  f32x4 ysum[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) ysum[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  __syncthreads();
#pragma unroll 1
  for (int rr = 0; rr < RW; ++rr) {
    // pixel i of the 32: tile column (32 (wave RW + rr) + i) % TW of that row
    const int p0 = 32 * (wave * RW + rr);
    auto row_of = [&](int pt) { return (p0 + 16 * pt + r) / TW; };
    auto col_of = [&](int pt) { return (16 * pt + r) % TW; };
    f32x4 acc[NPT][NT];
#pragma unroll
    for (int pt = 0; pt < NPT; ++pt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[pt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      // the taps of this K step: one of 32 channels, or four of 8 channels,
      // one per lane group (past the ninth: zeros)
      const int tap = CIN == C ? s : (4 * s + g < 9 ? 4 * s + g : 8);
#pragma unroll
      for (int pt = 0; pt < NPT; ++pt) {
        bf16x8 a = *reinterpret_cast<const bf16x8 *>(sx + ((row_of(pt) + tap / 3) * XW + col_of(pt) + tap % 3) * CIN +
                                                     (CIN == C ? 8 * g : 0));
        if constexpr (CIN != C) {
          if (4 * s + g >= 9)
#pragma unroll
            for (int j = 0; j < 8; ++j) a[j] = __bf16(0.f);
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[pt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s][nt], a, acc[pt][nt], 0, 0, 0);
      }
    }
#pragma unroll
    for (int pt = 0; pt < NPT; ++pt) {
      const int x = x0 + col_of(pt), y = y0 + row_of(pt);
      if (x >= W || y >= H) continue;
      const int64_t p = int64_t(y) * W + x;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int c = 16 * nt + 4 * g;
        f32x4 z = acc[pt][nt];
        typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
        bf16x4 o;
        if constexpr (MODE == MODE_OUT) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (c + i < NOUT) A.out[p * NOUT + c + i] = z[i] + bias[nt][i];
        } else if constexpr (MODE == MODE_BWD) {
          const f32x4 zp = *reinterpret_cast<const f32x4 *>(A.Zprev + p * C + c);
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = __bf16(z[i] * dsilu(zp[i]));
          *reinterpret_cast<bf16x4 *>(A.Y + p * C + c) = o;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            z[i] += bias[nt][i];
            o[i] = __bf16(silu(z[i]));
          }
          if (MODE == MODE_HIDDEN && A.csum) { // the last hidden layer
#pragma unroll
            for (int i = 0; i < 4; ++i) ysum[nt][i] += float(o[i]);
          }
          if (A.Z) *reinterpret_cast<f32x4 *>(A.Z + p * C + c) = z;
          *reinterpret_cast<bf16x4 *>(A.Y + p * C + c) = o;
        }
      }
    }
  }
  if constexpr (MODE == MODE_HIDDEN) {
    if (A.csum) { // sum over the 16 pixels of a lane group, then the waves
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v = ysum[nt][i];
#pragma unroll
          for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o);
          if (r == 0) ssum[wave][16 * nt + 4 * g + i] = v;
        }
      __syncthreads();
      if (tid < C)
        A.csum[int64_t(tid) * gridDim.x + blockIdx.x] = (ssum[0][tid] + ssum[1][tid]) + (ssum[2][tid] + ssum[3][tid]);
    }
  }
}

// The tile's shape.  RW: 4 where that still gives the chip a workgroup per CU
// (fewer halo pixels, 1.20 times the tile against 1.59, and the weights loaded for
// more pixels: a hidden layer at 512 x 512 took 16.3 us with 4, 16.9 with 2, 18.0
// with 1 in one run), else 1, and 1 too on grids so low that it stages fewer pixels.  TW: 32
// columns, or 8 where those stage at most three quarters of the pixels, as on
// grids of fewer columns than 32, most of whose tile would be columns that are
// not there (predict on 8 x 65536 pixels 156 -> 84 us, 4 x 131072 270 -> 117,
// 131072 x 4 162 -> 105; pixels in linear order, gathered per tap, 133).
struct Tile {
  int rw, tw, ntx, nty;
};
inline Tile tile_of(int H, int W) {
  auto shape = [&](int rw, int tw) {
    const int tr = 128 * rw / tw;
    return Tile{rw, tw, (W + tw - 1) / tw, (H + tr - 1) / tr};
  };
  auto blocks = [](const Tile &t) { return int64_t(t.ntx) * t.nty; };
  auto staged = [&](const Tile &t) { return blocks(t) * (t.tw + 2) * (128 * t.rw / t.tw + 2); };
  auto pick = [&](int tw) {
    const Tile big = shape(4, tw), small = shape(1, tw);
    return blocks(big) >= 256 && staged(big) <= staged(small) ? big : small;
  };
  const Tile wide = pick(32), narrow = pick(8);
  return 4 * staged(narrow) <= 3 * staged(wide) ? narrow : wide;
}
inline int conv_blocks(int H, int W) {
  const Tile t = tile_of(H, W);
  return t.ntx * t.nty;
}

// Backward-weight of a hidden layer: dW[tap][cout][cin] = sum_p dZ[p][cout]
// X[p + tap][cin] and db[cout] = sum_p dZ[p][cout], as MFMAs with M = cout,
// N = cin, K = pixels.  A workgroup takes a band of WG_SEG columns (every
// nband-th one on grids of more bands than WG_MAX, so that the workgroups' sums
// are bounded: 44 MB, 177 on 131072 x 4 with a workgroup for every band; MANY, a
// kernel of its own: a loop over the bands in the other cost it 8 registers and
// 7 % of a training step) and marches
// up its share of the grid rows, WG_ROWS rows at a time: those rows of dZ and
// the WG_ROWS + 2 rows of X that the taps read are staged in LDS once, in the
// layout they have in memory ([pixel][channel]), and the operands, which need
// the 8 pixels of one channel, come from the transposing LDS reads
// (ds_read_b64_tr_b16: the 16 lanes of a group read 4 pixels x 16 channels,
// every lane getting the 4 pixels of its channel).  A tap's shift in x is a
// pixel more in the read's address; each of the three waves has one row of
// taps, so a wave keeps 3 x 2 x 2 accumulators and no sum crosses waves.
// Pixels past the grid's edge are staged as zeros.  The workgroup's sums leave
// in accumulator order, part[wg][wave][dx][mt][nt][i][lane] and then db, for
// k_wgrad_reduce; db is a product with ones.
// Bound by the staging loads' latency (33.5 MB per layer at 512 x 512, 7 us at
// the copy rate) and by the partial sums (18.9 MB out and in again); at
// 512 x 512 16.7 us per 32-channel layer (10.5 us the 8-channel one; 21.6 and
// 12.7 us with each staging load waited for), where
// one workgroup per tap and 512 pixels, gathering the operands from LDS two
// bytes at a time, took 158 us (63 us), and db, 32 blocks over all pixels,
// another 324 us.
constexpr int WG_SEG = 64, WG_ROWS = 4, WG_MAX = 512; // columns, rows a step, most workgroups
constexpr int WG_THREADS = 192;

typedef short s16x4 __attribute__((ext_vector_type(4)));

// the 4 pixels of this lane's channel: p = the lane's own 8 bytes of the tile
__device__ __forceinline__ s16x4 lds_tr(const __bf16 *p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4 *)(reinterpret_cast<const s16x4 *>(p)));
}
__device__ __forceinline__ bf16x8 join(s16x4 lo, s16x4 hi) {
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  const s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8, v);
}

// 16-wide N tiles of a wave's three taps: 2 of one tap's 32 channels, or two
// taps of 8 channels side by side (the fourth tap repeats the third, unused)
__host__ __device__ constexpr int wg_ntiles(int cin) { return cin == C ? 6 : 2; }
// sums of one workgroup: 3 waves x tiles x 2 (mt) x 256, and db
__host__ __device__ constexpr int wg_sums(int cin) { return 3 * wg_ntiles(cin) * 2 * 256 + C; }

struct WgradGrid {
  int nseg, nband, rows_per_wg, nwg; // bands, bands taken at a time, grid rows of a workgroup, workgroups
};
inline WgradGrid wgrad_grid(int H, int W) {
  WgradGrid G;
  G.nseg = (W + WG_SEG - 1) / WG_SEG;
  G.nband = std::min(G.nseg, WG_MAX);
  const int per = WG_MAX / G.nband; // workgroups a band may take
  G.rows_per_wg = ((H + per - 1) / per + WG_ROWS - 1) / WG_ROWS * WG_ROWS;
  G.nwg = G.nband * ((H + G.rows_per_wg - 1) / G.rows_per_wg);
  return G;
}

template <int CIN, bool MANY>
__global__ void __launch_bounds__(WG_THREADS) k_conv_wgrad(const __bf16 *__restrict__ dZ,
                                                          const __bf16 *__restrict__ X, int H, int W,
                                                          int nband, int rows_per_wg,
                                                          float *__restrict__ part) {
  constexpr int NT = wg_ntiles(CIN);
  __shared__ __align__(16) __bf16 sz[WG_ROWS * WG_SEG * C];
  __shared__ __align__(16) __bf16 sx[(WG_ROWS + 2) * (WG_SEG + 2) * CIN];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, i16 = lane & 15;
  const int yb = (int(blockIdx.x) / nband) * rows_per_wg;
  const int ye = yb + rows_per_wg < H ? yb + rows_per_wg : H;
  f32x4 acc[NT][2], accb[2];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt) {
    accb[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[nt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  bf16x8 ones, zero;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    ones[j] = __bf16(1.f);
    zero[j] = __bf16(0.f);
  }
  int x0 = (int(blockIdx.x) % nband) * WG_SEG;
  for (int y0 = yb; y0 < ye;) {
    constexpr int ZV = WG_ROWS * WG_SEG * (C / 8), XW = WG_SEG + 2, XV = (WG_ROWS + 2) * XW * (CIN / 8);
    constexpr int ZP = (ZV + WG_THREADS - 1) / WG_THREADS, XP = (XV + WG_THREADS - 1) / WG_THREADS;
    bf16x8 dz[ZP], dx[XP]; // every load in flight before the first LDS store
#pragma unroll
    for (int k = 0; k < ZP; ++k) {
      const int q = tid + WG_THREADS * k;
      const int v = q % (C / 8), px = q / (C / 8) % WG_SEG, row = q / (C / 8 * WG_SEG);
      const int x = x0 + px, y = y0 + row;
      dz[k] = zero;
      if (q < ZV && x < W && y < ye)
        dz[k] = *reinterpret_cast<const bf16x8 *>(dZ + (int64_t(y) * W + x) * C + 8 * v);
    }
#pragma unroll
    for (int k = 0; k < XP; ++k) {
      const int q = tid + WG_THREADS * k;
      const int v = q % (CIN / 8), px = q / (CIN / 8) % XW, row = q / (CIN / 8 * XW);
      int x = x0 - 1 + px, y = y0 - 1 + row;
      dx[k] = zero;
      if (q < XV && x <= W && y <= H) { // W, H: the wrapped neighbours of the last column and row
        x = x < 0 ? x + W : (x >= W ? x - W : x);
        y = y < 0 ? y + H : (y >= H ? y - H : y);
        dx[k] = *reinterpret_cast<const bf16x8 *>(X + (int64_t(y) * W + x) * CIN + 8 * v);
      }
    }
#pragma unroll
    for (int k = 0; k < ZP; ++k)
      if (tid + WG_THREADS * k < ZV) *reinterpret_cast<bf16x8 *>(sz + 8 * (tid + WG_THREADS * k)) = dz[k];
#pragma unroll
    for (int k = 0; k < XP; ++k)
      if (tid + WG_THREADS * k < XV) *reinterpret_cast<bf16x8 *>(sx + 8 * (tid + WG_THREADS * k)) = dx[k];
    __syncthreads();
#pragma unroll
    for (int row = 0; row < WG_ROWS; ++row)
#pragma unroll
      for (int ks = 0; ks < WG_SEG / 32; ++ks) {
        const int px = 32 * ks + 8 * g + (i16 >> 2); // this lane's pixel of the first 4 of 8
        bf16x8 a[2];
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
          const __bf16 *pz = sz + (row * WG_SEG + px) * C + 16 * mt + 4 * (i16 & 3);
          a[mt] = join(lds_tr(pz), lds_tr(pz + 4 * C));
          if (wave == 0) accb[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mt], ones, accb[mt], 0, 0, 0);
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          int dx, ch;
          if constexpr (CIN == C) {
            dx = nt / 2;
            ch = 16 * (nt & 1) + 4 * (i16 & 3);
          } else {
            dx = 2 * nt + ((i16 & 3) >> 1);
            dx = dx < 3 ? dx : 2;
            ch = 4 * (i16 & 1);
          }
          const __bf16 *px_ = sx + ((row + wave) * XW + px + dx) * CIN + ch;
          const bf16x8 b = join(lds_tr(px_), lds_tr(px_ + 4 * CIN));
#pragma unroll
          for (int mt = 0; mt < 2; ++mt)
            acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[mt], b, acc[nt][mt], 0, 0, 0);
        }
      }
    __syncthreads();
    y0 += WG_ROWS;
    if (MANY && y0 >= ye && x0 + nband * WG_SEG < W) { // the next of its bands
      x0 += nband * WG_SEG;
      y0 = yb;
    }
  }
  float *dst = part + int64_t(blockIdx.x) * wg_sums(CIN);
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[(((wave * NT + nt) * 2 + mt) * 4 + i) * 64 + lane] = acc[nt][mt][i];
  if (wave == 0 && i16 == 0) {
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[wg_sums(CIN) - C + 16 * mt + 4 * g + i] = accb[mt][i];
  }
}

// dW and db of the three hidden layers from their workgroups' sums: a block
// sums 64 elements, 16 slices of the workgroups at a time (1024 threads, so
// that a slice is 32 loads long; one thread per element walking every partial
// took 121 us per layer, this 8.4 us for the three), then the slices in order.
struct WgradLayers {
  const float *part[NL - 1];
  float *gw[NL - 1]; // dW of the layer, db behind it
  int nwg;
};
constexpr int WR_SLICES = 16;

__global__ void __launch_bounds__(64 * WR_SLICES) k_wgrad_reduce(WgradLayers L) {
  __shared__ float sh[WR_SLICES][64];
  const int l = blockIdx.y, cin = cin_of(l), n = wg_sums(cin);
  const int e0 = blockIdx.x * 64;
  if (e0 >= n) return; // the whole block: the 8-channel layer has fewer sums
  const int k = threadIdx.x & 63, sl = threadIdx.x >> 6, e = e0 + k;
  const float *part = l == 0 ? L.part[0] : (l == 1 ? L.part[1] : L.part[2]);
  float *gw = l == 0 ? L.gw[0] : (l == 1 ? L.gw[1] : L.gw[2]);
  float s = 0.f;
  if (e < n)
#pragma unroll 8
    for (int w = sl; w < L.nwg; w += WR_SLICES) s += part[int64_t(w) * n + e];
  sh[sl][k] = s;
  __syncthreads();
  if (sl != 0 || e >= n) return;
  s = 0.f;
  for (int q = 0; q < WR_SLICES; ++q) s += sh[q][k];
  if (e >= n - C) {
    gw[9 * cin * C + (e - (n - C))] = s;
    return;
  }
  // accumulator order -> dW[tap][cout][cin]
  const int lane = e & 63, i = (e >> 6) & 3, mt = (e >> 8) & 1, t = e >> 9;
  const int NT = wg_ntiles(cin), wave = t / NT, nt = t % NT;
  const int cout = 16 * mt + 4 * (lane >> 4) + i, col = lane & 15;
  const int dx = cin == C ? nt / 2 : 2 * nt + (col >> 3);
  const int ci = cin == C ? 16 * (nt & 1) + col : col & 7;
  if (dx < 3) gw[((3 * wave + dx) * C + cout) * cin + ci] = s;
}

// a sample's costs at the orders T_j = 1 + j/2, by value
struct Costs {
  double c[NOUT];
};

constexpr double kTau = 0.25; // temperature of the soft arg-min over the cost estimates

// policy layout: pol[0..NOUT-1] = the weights p, pol[NOUT] = t,
// pol[NOUT+1 .. NOUT+5] = the extrapolation weights e_j of f_{n-j} in P(t),
// pol[NOUT+6 ..] = the cost estimates m
constexpr int POL_T = NOUT, POL_E = NOUT + 1, POL_M = NOUT + 6, POL_LEN = 2 * NOUT + 6;

// binomial extrapolation weights of order k (1..4) for f_n, ..., f_{n-4}
__device__ __forceinline__ double extrap_weight(int k, int j) {
  // (-1)^j C(k+1, j+1), zero for j > k
  constexpr double E[4][5] = {{2., -1., 0., 0., 0.},
                              {3., -3., 1., 0., 0.},
                              {4., -6., 4., -1., 0.},
                              {5., -10., 10., -5., 1.}};
  return E[k - 1][j];
}

// The cost estimates m_j = grid mean of output channel j.  The output layer
// is linear and its padding periodic, so that mean is
//   m_j = bias_j + sum_i Weff[j][i] mean(Y[:, i]),  Weff[j][i] = sum_tap W[tap][j][i]
// (the BF16 weights the MFMAs use), from the channel sums of the last
// hidden layer; p = softmax(-m / kTau), t = sum_j p_j T_j, the weights of
// P(t) and m into pol; with costs c, also lg[0] = sum_j (m_j - (c_j -
// mean c))^2 / NOUT and lg[1 + j] = d lg[0] / d m_j.  One workgroup: 32
// lanes per channel add the blocks' sums (FP64), 32 per output its products;
// one thread the seven-term rest.  Latency-bound, one launch.
__global__ void __launch_bounds__(1024) k_policy(const float *__restrict__ csum, int nblk, double *__restrict__ sums,
                                                 const float *__restrict__ weff, const float *__restrict__ bias,
                                                 double inv_npix, Costs costs, int with_costs,
                                                 double *__restrict__ pol, double *__restrict__ lg,
                                                 double *__restrict__ host) {
  __shared__ double sc[C], m[NOUT];
  const int ch = threadIdx.x >> 5, l = threadIdx.x & 31;
  double v = 0.;
#pragma unroll 4
  for (int b = l; b < nblk; b += 32) v += double(csum[int64_t(ch) * nblk + b]);
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) v += __shfl_xor(v, o, 32);
  if (l == 0) {
    sc[ch] = v;
    sums[ch] = v;
  }
  __syncthreads();
  if (ch < NOUT) {
    double w = double(weff[ch * C + l]) * sc[l];
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) w += __shfl_xor(w, o, 32);
    if (l == 0) {
      m[ch] = double(bias[ch]) + w * inv_npix;
      pol[POL_M + ch] = m[ch];
    }
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  double mn = 1e300, z = 0., t = 0., e[NOUT];
#pragma unroll
  for (int c = 0; c < NOUT; ++c) mn = fmin(mn, m[c]);
#pragma unroll
  for (int c = 0; c < NOUT; ++c) {
    e[c] = exp(-(m[c] - mn) / kTau);
    z += e[c];
  }
#pragma unroll
  for (int c = 0; c < NOUT; ++c) {
    e[c] /= z;
    pol[c] = e[c];
    t += e[c] * (1. + 0.5 * c);
  }
  t = fmin(fmax(t, 1.), 4.);
  const int k = t >= 4. ? 3 : int(t);
  const double w = t - k;
  pol[POL_T] = t;
#pragma unroll
  for (int j = 0; j < 5; ++j) pol[POL_E + j] = (1. - w) * extrap_weight(k, j) + w * extrap_weight(k + 1, j);
  if (with_costs) {
    double cbar = 0., ls = 0.;
#pragma unroll
    for (int c = 0; c < NOUT; ++c) cbar += costs.c[c];
    cbar /= NOUT;
#pragma unroll
    for (int c = 0; c < NOUT; ++c) {
      const double r = m[c] - (costs.c[c] - cbar);
      ls += r * r;
      lg[1 + c] = 2. * r / NOUT;
    }
    lg[0] = ls / NOUT;
    if (host) *host = ls / NOUT;
  }
}

// guess = (4/3) y_n - (1/3) y_{n-1} + (2/3) dt sum_j e_j f_{n-j}, e = the
// weights of P(t) in pol
__global__ void k_guess(const double *__restrict__ un, const double *__restrict__ unm1, FHist F, double dt,
                        const double *__restrict__ pol, int64_t n, double *__restrict__ guess) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double *e = pol + POL_E;
  const double E = e[0] * F.f[0][i] + e[1] * F.f[1][i] + e[2] * F.f[2][i] + e[3] * F.f[3][i] + e[4] * F.f[4][i];
  guess[i] = (4. / 3.) * un[i] - (1. / 3.) * unm1[i] + ((2. / 3.) * dt) * E;
}

// Backward of the output layer.  The loss reads its grid means alone, so
// d loss / d out[p][c] = (d loss / d m_c) / npix = dz_c at every pixel (held in
// BF16 as every dZ), and with the periodic padding
//   dW[tap][c][i] = dz_c sum_p Y[p][i]  (the channel sums of the policy),
//   db[c] = dz_c npix,
//   d loss / d Y[p][i] = sum_c dz_c Weff[c][i] = dy[i], the same at every pixel:
// one block per tap instead of three passes over the pixels.
__global__ void __launch_bounds__(256) k_out_backward(const double *__restrict__ lg, const double *__restrict__ sums,
                                                      const float *__restrict__ weff, double npix,
                                                      float *__restrict__ gw, float *__restrict__ dy) {
  const int tap = blockIdx.x, e = threadIdx.x;
  auto dz = [&](int c) { return double(float(__bf16(float(lg[1 + c] / npix)))); };
  if (e < NOUT * C) gw[tap * NOUT * C + e] = float(dz(e / C) * sums[e % C]);
  if (tap != 0) return;
  if (e < NOUT) gw[9 * NOUT * C + e] = float(dz(e) * npix);
  if (e < C) {
    double v = 0.;
    for (int c = 0; c < NOUT; ++c) v += dz(c) * double(weff[c * C + e]);
    dy[e] = float(v);
  }
}

// dZ of the last hidden layer: dy[c] SiLU'(Z[p][c]), 8 channels per thread
__global__ void __launch_bounds__(256) k_dz_hidden(const float *__restrict__ dy, const float *__restrict__ Z,
                                                   int64_t npix, __bf16 *__restrict__ dZ) {
  const int64_t q = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (q >= npix * (C / 8)) return;
  const int c0 = 8 * int(q % (C / 8));
  const f32x4 z0 = *reinterpret_cast<const f32x4 *>(Z + 8 * q), z1 = *reinterpret_cast<const f32x4 *>(Z + 8 * q + 4);
  bf16x8 d;
#pragma unroll
  for (int j = 0; j < 8; ++j) d[j] = __bf16(dy[c0 + j] * dsilu(j < 4 ? z0[j & 3] : z1[j & 3]));
  *reinterpret_cast<bf16x8 *>(dZ + 8 * q) = d;
}

// Adam on the FP32 master parameters
__global__ void k_adam(float *__restrict__ w, const float *__restrict__ gr, float *__restrict__ m1,
                       float *__restrict__ m2, int64_t n, float lr, float b1, float b2, float eps,
                       float c1, float c2) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = gr[i];
  m1[i] = b1 * m1[i] + (1.f - b1) * gi;
  m2[i] = b2 * m2[i] + (1.f - b2) * gi * gi;
  w[i] -= lr * (m1[i] * c1) / (sqrtf(m2[i] * c2) + eps);
}

// Pack the FP32 master parameters of every layer into the bf16 B-operand
// layouts: forward Wf[l][s][coutp][32] and backward-data Wb[l][tap'][cin][32]
// (= W[8 - tap'][cout][cin], K = cout); and the output layer's tap sums of
// its BF16 weights, weff[cout][cin] (FP32).
__global__ void k_pack(const float *__restrict__ w, const int64_t *__restrict__ woff, __bf16 *__restrict__ Wf,
                       const int64_t *__restrict__ foff, __bf16 *__restrict__ Wb,
                       const int64_t *__restrict__ boff, float *__restrict__ weff) {
  const int l = blockIdx.y;
  if (l == NL - 1 && blockIdx.x == 0)
    for (int e = threadIdx.x; e < NOUT * C; e += blockDim.x) {
      const float *Wl = w + woff[l];
      float v = 0.f;
      for (int tap = 0; tap < 9; ++tap) v += float(__bf16(Wl[tap * NOUT * C + e]));
      weff[e] = v;
    }
  const int cin = cin_of(l), cout = cout_of(l), coutp = cout == NOUT ? 16 : C;
  const int KS = ksteps(cin);
  const float *W = w + woff[l]; // [tap][cout][cin]
  const int nf = KS * coutp * 32;
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < nf; e += gridDim.x * blockDim.x) {
    const int s = e / (coutp * 32), co = (e / 32) % coutp, k = e % 32;
    float v = 0.f;
    if (co < cout) {
      if (cin == C) {
        v = W[(s * cout + co) * cin + k];
      } else {
        const int tap = 4 * s + k / 8, ci = k % 8;
        v = tap < 9 ? W[(tap * cout + co) * cin + ci] : 0.f;
      }
    }
    Wf[foff[l] + e] = __bf16(v);
  }
  if (l == 0) return; // no input gradient for the first layer
  const int nb = 9 * C * 32;
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < nb; e += gridDim.x * blockDim.x) {
    const int tp = e / (C * 32), ci = (e / 32) % C, k = e % 32;
    const float v = k < cout ? W[((8 - tp) * cout + k) * cin + ci] : 0.f;
    Wb[boff[l] + e] = __bf16(v);
  }
}

}  // namespace nn
}  // namespace pda

struct pda_guessnet_s {
  int H = 0, W = 0;
  int64_t npix = 0;
  double dt = 5e-3;                 // time step of the predictors
  double s[4] = {1e-3, 1e-4, 1e-5, 1e-6}; // spreads of dt D^k f, k = 1..4
  double nu_mean = 5.5e-3, nu_scale = 4.5e-3;
  int64_t nparam = 0;
  int64_t woff[pda::nn::NL + 1] = {0};
  int64_t foff[pda::nn::NL + 1] = {0}, boff[pda::nn::NL + 1] = {0};
  pda::DevBuf w, g, m1, m2;          // FP32 master params, grads, Adam moments
  pda::DevBuf Wf, Wb, d_woff, d_foff, d_boff;
  pda::DevBuf X0, Y[3], Z[3], dZa, dZb, out, part;
  pda::DevBuf csum, sums, weff;      // last hidden layer's channel sums; output tap sums
  pda::DevBuf pol;                   // the last forward's policy: p, t, weights of P(t)
  pda::DevBuf lg;                    // expected cost, its derivatives w.r.t. the NOUT logits
  pda::DevBuf dy;                    // d loss / d Y of the last hidden layer, per channel
  double *hloss = nullptr;           // pinned: the expected cost, for the host
  hipEvent_t loss_ready = nullptr;
  int adam_t = 0;
  ~pda_guessnet_s() {
    if (loss_ready) (void)hipEventDestroy(loss_ready);
    if (hloss) (void)hipHostFree(hloss);
  }
};

namespace {
using namespace pda;
using namespace pda::nn;

int pack(pda_guessnet_s &net, hipStream_t st) {
  hipLaunchKernelGGL(k_pack, dim3(16, NL), dim3(256), 0, st, net.w.as<float>(), net.d_woff.as<int64_t>(),
                     net.Wf.as<__bf16>(), net.d_foff.as<int64_t>(), net.Wb.as<__bf16>(),
                     net.d_boff.as<int64_t>(), net.weff.as<float>());
  PDA_HIP_CHECK(hipGetLastError());
  return PDA_OK;
}

const float *bias_of(const pda_guessnet_s &net, int l) {
  return net.w.as<float>() + net.woff[l] + 9 * cin_of(l) * cout_of(l);
}

// the velocity history a forward reads
int history(const double *const *f, FHist *F, const char *who) {
  if (!f) {
    set_error(std::string(who) + ": null velocity history");
    return PDA_E_INVALID_ARG;
  }
  for (int k = 0; k < 5; ++k) {
    if (!f[k]) {
      set_error(std::string(who) + ": null velocity f_{n-" + std::to_string(k) + "}");
      return PDA_E_INVALID_ARG;
    }
    F->f[k] = f[k];
  }
  return PDA_OK;
}

Features feature_args(const pda_guessnet_s &net, const FHist &F, double nu) {
  Features T;
  T.F = F;
  for (int k = 0; k < 4; ++k) T.c[k] = net.dt / net.s[k];
  T.nu_hat = (nu - net.nu_mean) / net.nu_scale;
  return T;
}

// the order policy of the last forward into net.pol; with costs, the
// cost-estimate loss and its derivatives into net.lg
int policy(pda_guessnet_s &net, const Costs *costs, hipStream_t st, double *host = nullptr) {
  hipLaunchKernelGGL(k_policy, dim3(1), dim3(1024), 0, st, net.csum.as<float>(), conv_blocks(net.H, net.W),
                     net.sums.as<double>(), net.weff.as<float>(), bias_of(net, NL - 1), 1. / double(net.npix),
                     costs ? *costs : Costs{}, costs ? 1 : 0, net.pol.as<double>(), net.lg.as<double>(), host);
  PDA_HIP_CHECK(hipGetLastError());
  return PDA_OK;
}

template <int MODE>
void conv(const pda_guessnet_s &net, ConvArgs A, const Features &T, hipStream_t st) {
  const Tile t = tile_of(net.H, net.W);
  A.H = net.H;
  A.W = net.W;
  A.ntx = t.ntx;
  const dim3 grid{unsigned(t.ntx) * unsigned(t.nty), 1, 1};
  if (t.tw == 32 && t.rw == 4) hipLaunchKernelGGL((k_conv<MODE, 4, 32>), grid, dim3(256), 0, st, A, T);
  else if (t.tw == 32) hipLaunchKernelGGL((k_conv<MODE, 1, 32>), grid, dim3(256), 0, st, A, T);
  else if (t.rw == 4) hipLaunchKernelGGL((k_conv<MODE, 4, 8>), grid, dim3(256), 0, st, A, T);
  else hipLaunchKernelGGL((k_conv<MODE, 1, 8>), grid, dim3(256), 0, st, A, T);
}

// forward through the hidden layers from the velocity history, with the
// last one's channel sums (all the policy needs: the output layer is
// linear); the features and the pre-activations Z are kept only when a
// backward follows; with full_out, the output layer too, out = L4 (FP32
// [p][NOUT])
int forward(pda_guessnet_s &net, const Features &T, bool keep, bool full_out, hipStream_t st) {
  for (int l = 0; l < NL; ++l) {
    if (l == NL - 1 && !full_out) break;
    ConvArgs A{};
    A.X = l == 0 ? nullptr : net.Y[l - 1].as<__bf16>();
    A.Wp = net.Wf.as<__bf16>() + net.foff[l];
    A.bias = bias_of(net, l);
    if (l == NL - 1) {
      A.out = net.out.as<float>();
      conv<MODE_OUT>(net, A, T, st);
      break;
    }
    A.Z = keep ? net.Z[l].as<float>() : nullptr;
    A.Y = net.Y[l].as<__bf16>();
    A.csum = l == NL - 2 ? net.csum.as<float>() : nullptr;
    if (l == 0) {
      A.X0 = keep ? net.X0.as<__bf16>() : nullptr;
      conv<MODE_FIRST>(net, A, T, st);
    } else {
      conv<MODE_HIDDEN>(net, A, T, st);
    }
  }
  PDA_HIP_CHECK(hipGetLastError());
  return PDA_OK;
}

// Gradients (into net.g) of the loss whose derivatives w.r.t. the output
// means are in net.lg.  The output layer's follow from the channel sums.
// Hidden layer l: the sums of dW_l from (dZ_l, input_l); dZ_{l-1} = (dZ_l
// conv flipped transposed W_l) * SiLU'(Z_{l-1}), alternating between dZa and
// dZb; the sums of the three layers are reduced together at the end.
int backward(pda_guessnet_s &net, hipStream_t st) {
  const WgradGrid G = wgrad_grid(net.H, net.W);
  float *gW = net.g.as<float>();
  const __bf16 *Wb = net.Wb.as<__bf16>();
  __bf16 *dz = net.dZa.as<__bf16>(), *dz_next = net.dZb.as<__bf16>();
  hipLaunchKernelGGL(k_out_backward, dim3(9), dim3(256), 0, st, net.lg.as<double>(), net.sums.as<double>(),
                     net.weff.as<float>(), double(net.npix), gW + net.woff[NL - 1], net.dy.as<float>());
  hipLaunchKernelGGL(k_dz_hidden, dim3(unsigned((net.npix * (C / 8) + 255) / 256)), dim3(256), 0, st,
                     net.dy.as<float>(), net.Z[NL - 2].as<float>(), net.npix, dz);
  PDA_HIP_CHECK(hipGetLastError());
  WgradLayers L{};
  L.nwg = G.nwg;
  float *part = net.part.as<float>();
  for (int l = NL - 2; l >= 0; --l) {
    const int cin = cin_of(l);
    L.part[l] = part;
    L.gw[l] = gW + net.woff[l];
    const auto go = [&](auto kernel, const __bf16 *x) {
      hipLaunchKernelGGL(kernel, dim3(G.nwg), dim3(WG_THREADS), 0, st, dz, x, net.H, net.W, G.nband, G.rows_per_wg, part);
    };
    const bool many = G.nseg > G.nband;
    if (cin == C) go(many ? k_conv_wgrad<C, true> : k_conv_wgrad<C, false>, net.Y[l - 1].as<__bf16>());
    else go(many ? k_conv_wgrad<CIN0, true> : k_conv_wgrad<CIN0, false>, net.X0.as<__bf16>());
    part += int64_t(G.nwg) * wg_sums(cin);
    PDA_HIP_CHECK(hipGetLastError());
    if (l == 0) break;
    ConvArgs A{};
    A.X = dz;
    A.Wp = Wb + net.boff[l];
    A.Y = dz_next;
    A.Zprev = net.Z[l - 1].as<float>();
    conv<MODE_BWD>(net, A, Features{}, st);
    PDA_HIP_CHECK(hipGetLastError());
    std::swap(dz, dz_next);
  }
  hipLaunchKernelGGL(k_wgrad_reduce, dim3((wg_sums(C) + 63) / 64, NL - 1), dim3(64 * WR_SLICES), 0, st, L);
  PDA_HIP_CHECK(hipGetLastError());
  return PDA_OK;
}

// loss of the current forward's cost estimates against a sample's costs;
// leaves its derivatives w.r.t. the output means in net.lg
int loss(pda_guessnet_s &net, const double *costs, bool want, hipStream_t st) {
  Costs c;
  for (int j = 0; j < NOUT; ++j) c.c[j] = costs[j];
  if (want && !net.loss_ready) { // the first loss that is asked for; a network that only predicts has none
    if (!net.hloss)
      PDA_HIP_CHECK(hipHostMalloc(reinterpret_cast<void **>(&net.hloss), sizeof(double), hipHostMallocDefault));
    PDA_HIP_CHECK(hipEventCreateWithFlags(&net.loss_ready, hipEventDisableTiming));
  }
  const int rc = policy(net, &c, st, want ? net.hloss : nullptr);
  if (!rc && want) PDA_HIP_CHECK(hipEventRecord(net.loss_ready, st));
  return rc;
}

// The loss of the step whose kernels are all queued: the host waits for the
// policy's launch only, and only now, so that the backward pass follows the
// forward one without a gap (read between the two, the GPU idled 38 of a
// 512 x 512 training step's 241 us).
int read_loss(pda_guessnet_s &net, float *lval) {
  PDA_HIP_CHECK(hipEventSynchronize(net.loss_ready));
  *lval = float(*net.hloss);
  return PDA_OK;
}

int check_costs(const double *costs, const char *who) {
  if (!costs) {
    set_error(std::string(who) + ": null costs");
    return PDA_E_INVALID_ARG;
  }
  for (int j = 0; j < NOUT; ++j)
    if (!std::isfinite(costs[j])) {
      set_error(std::string(who) + ": the costs must be finite");
      return PDA_E_INVALID_ARG;
    }
  return PDA_OK;
}

}  // namespace

extern "C" {

int pda_guessnet_create(int nx, int ny, pda_guessnet *out) {
  if (!out || nx < 4 || ny < 4 || (int64_t(nx) * ny) % 512 != 0 || int64_t(nx) * ny > (int64_t(1) << 30)) {
    set_error("pda_guessnet_create: need nx, ny >= 4 and nx*ny a multiple of 512, at most 2^30");
    return PDA_E_INVALID_ARG;
  }
  auto *net = new pda_guessnet_s();
  net->W = nx;
  net->H = ny;
  net->npix = int64_t(nx) * ny;
  int64_t wo = 0, fo = 0, bo = 0;
  for (int l = 0; l < NL; ++l) {
    net->woff[l] = wo;
    net->foff[l] = fo;
    net->boff[l] = bo;
    const int cin = cin_of(l), cout = cout_of(l), coutp = cout == NOUT ? 16 : C;
    wo += 9 * cin * cout + cout;
    fo += int64_t(ksteps(cin)) * coutp * 32;
    bo += l == 0 ? 0 : 9 * C * 32;
  }
  net->woff[NL] = wo;
  net->foff[NL] = fo;
  net->boff[NL] = bo;
  net->nparam = wo;
  const int64_t np = net->npix;
  hipError_t e = net->w.alloc(sizeof(float) * wo);
  if (e == hipSuccess) e = net->g.alloc(sizeof(float) * wo);
  if (e == hipSuccess) e = net->m1.alloc(sizeof(float) * wo);
  if (e == hipSuccess) e = net->m2.alloc(sizeof(float) * wo);
  if (e == hipSuccess) e = net->Wf.alloc(sizeof(__bf16) * fo);
  if (e == hipSuccess) e = net->Wb.alloc(sizeof(__bf16) * std::max<int64_t>(bo, 1));
  if (e == hipSuccess) e = net->d_woff.upload(std::vector<int64_t>(net->woff, net->woff + NL + 1));
  if (e == hipSuccess) e = net->d_foff.upload(std::vector<int64_t>(net->foff, net->foff + NL + 1));
  if (e == hipSuccess) e = net->d_boff.upload(std::vector<int64_t>(net->boff, net->boff + NL + 1));
  if (e == hipSuccess) e = net->X0.alloc(sizeof(__bf16) * np * CIN0);
  for (int i = 0; i < 3 && e == hipSuccess; ++i) e = net->Y[i].alloc(sizeof(__bf16) * np * C);
  for (int i = 0; i < 3 && e == hipSuccess; ++i) e = net->Z[i].alloc(sizeof(float) * np * C);
  if (e == hipSuccess) e = net->dZa.alloc(sizeof(__bf16) * np * C);
  if (e == hipSuccess) e = net->dZb.alloc(sizeof(__bf16) * np * C);
  if (e == hipSuccess) e = net->out.alloc(sizeof(float) * np * NOUT);
  if (e == hipSuccess)
    e = net->part.alloc(sizeof(float) * size_t(wgrad_grid(ny, nx).nwg) * (wg_sums(CIN0) + (NL - 2) * wg_sums(C)));
  if (e == hipSuccess) e = net->csum.alloc(sizeof(float) * size_t(conv_blocks(ny, nx)) * C);
  if (e == hipSuccess) e = net->sums.alloc(sizeof(double) * C);
  if (e == hipSuccess) e = net->weff.alloc(sizeof(float) * NOUT * C);
  if (e == hipSuccess) e = net->pol.alloc(sizeof(double) * POL_LEN);
  if (e == hipSuccess) e = net->lg.alloc(sizeof(double) * (1 + NOUT));
  if (e == hipSuccess) e = net->dy.alloc(sizeof(float) * C);
  if (e == hipSuccess) e = hipMemset(net->pol.ptr, 0, sizeof(double) * POL_LEN);
  if (e == hipSuccess) e = hipMemset(net->w.ptr, 0, sizeof(float) * wo);
  if (e == hipSuccess) e = hipMemset(net->m1.ptr, 0, sizeof(float) * wo);
  if (e == hipSuccess) e = hipMemset(net->m2.ptr, 0, sizeof(float) * wo);
  if (e != hipSuccess) {
    set_error(std::string("pda_guessnet_create: ") + hipGetErrorString(e));
    delete net;
    return PDA_E_HIP;
  }
  *out = net;
  return PDA_OK;
}

void pda_guessnet_destroy(pda_guessnet net) { delete net; }

int pda_guessnet_num_params(pda_guessnet net, int64_t *n) {
  if (!net || !n) return PDA_E_INVALID_ARG;
  *n = net->nparam;
  return PDA_OK;
}

int pda_guessnet_set_params(pda_guessnet net, const float *w, int64_t n) {
  if (!net || !w || n != net->nparam) {
    set_error("pda_guessnet_set_params: expected the network's parameter count");
    return PDA_E_INVALID_ARG;
  }
  PDA_HIP_CHECK(hipMemcpy(net->w.ptr, w, sizeof(float) * n, hipMemcpyHostToDevice));
  PDA_HIP_CHECK(hipMemset(net->m1.ptr, 0, sizeof(float) * n));
  PDA_HIP_CHECK(hipMemset(net->m2.ptr, 0, sizeof(float) * n));
  net->adam_t = 0;
  const int rc = pack(*net, nullptr);
  if (rc) return rc;
  PDA_HIP_CHECK(hipDeviceSynchronize());
  return PDA_OK;
}

int pda_guessnet_get_params(pda_guessnet net, float *w, int64_t n) {
  if (!net || !w || n != net->nparam) return PDA_E_INVALID_ARG;
  PDA_HIP_CHECK(hipMemcpy(w, net->w.ptr, sizeof(float) * n, hipMemcpyDeviceToHost));
  return PDA_OK;
}

int pda_guessnet_set_scales(pda_guessnet net, double dt, const double *spreads, double nu_mean, double nu_scale) {
  if (!net || !spreads || !(dt > 0.) || !(nu_scale > 0.)) {
    set_error("pda_guessnet_set_scales: dt, the spreads and nu_scale must be positive");
    return PDA_E_INVALID_ARG;
  }
  for (int k = 0; k < 4; ++k)
    if (!(spreads[k] > 0.)) {
      set_error("pda_guessnet_set_scales: dt, the spreads and nu_scale must be positive");
      return PDA_E_INVALID_ARG;
    }
  net->dt = dt;
  for (int k = 0; k < 4; ++k) net->s[k] = spreads[k];
  net->nu_mean = nu_mean;
  net->nu_scale = nu_scale;
  return PDA_OK;
}

int pda_guessnet_predict(pda_guessnet net, const double *d_un, const double *d_unm1, const double *const *d_f,
                         double nu, double *d_guess, pda_stream stream) {
  FHist F;
  if (!net || !d_un || !d_unm1 || !d_guess) {
    set_error("pda_guessnet_predict: null argument");
    return PDA_E_INVALID_ARG;
  }
  int rc = history(d_f, &F, "pda_guessnet_predict");
  if (rc) return rc;
  hipStream_t st = hipStream_t(stream);
  rc = forward(*net, feature_args(*net, F, nu), false, false, st);
  if (!rc) rc = policy(*net, nullptr, st);
  if (rc) return rc;
  const int64_t n = net->npix * NCOMP;
  hipLaunchKernelGGL(k_guess, dim3(unsigned((n + 255) / 256)), dim3(256), 0, st, d_un, d_unm1, F, net->dt,
                     net->pol.as<double>(), n, d_guess);
  PDA_HIP_CHECK(hipGetLastError());
  return PDA_OK;
}

int pda_guessnet_policy(pda_guessnet net, double *order, double *probs, double *estimates) {
  if (!net || !order) {
    set_error("pda_guessnet_policy: null argument");
    return PDA_E_INVALID_ARG;
  }
  double pol[POL_LEN];
  PDA_HIP_CHECK(hipMemcpy(pol, net->pol.ptr, sizeof(pol), hipMemcpyDeviceToHost));
  *order = pol[POL_T];
  for (int j = 0; j < NOUT; ++j) {
    if (probs) probs[j] = pol[j];
    if (estimates) estimates[j] = pol[POL_M + j];
  }
  return PDA_OK;
}

int pda_guessnet_gradients(pda_guessnet net, const double *const *d_f, double nu, const double *costs,
                           float *grad, float *lossv, float *outv, pda_stream stream) {
  FHist F;
  if (!net) {
    set_error("pda_guessnet_gradients: null network");
    return PDA_E_INVALID_ARG;
  }
  int rc = history(d_f, &F, "pda_guessnet_gradients");
  if (!rc) rc = check_costs(costs, "pda_guessnet_gradients");
  if (rc) return rc;
  hipStream_t st = hipStream_t(stream);
  rc = forward(*net, feature_args(*net, F, nu), true, outv != nullptr, st);
  if (!rc) rc = loss(*net, costs, lossv != nullptr, st);
  if (!rc) rc = backward(*net, st);
  if (!rc && lossv) rc = read_loss(*net, lossv);
  if (rc) return rc;
  if (grad)
    PDA_HIP_CHECK(hipMemcpyAsync(grad, net->g.ptr, sizeof(float) * net->nparam, hipMemcpyDeviceToHost, st));
  if (outv)
    PDA_HIP_CHECK(hipMemcpyAsync(outv, net->out.ptr, sizeof(float) * net->npix * NOUT, hipMemcpyDeviceToHost, st));
  PDA_HIP_CHECK(hipStreamSynchronize(st));
  return PDA_OK;
}

int pda_guessnet_train_step(pda_guessnet net, const double *const *d_f, double nu, const double *costs,
                            float lr, float *lossv, pda_stream stream) {
  FHist F;
  if (!net || !(lr > 0.f)) {
    set_error("pda_guessnet_train_step: invalid argument");
    return PDA_E_INVALID_ARG;
  }
  int rc = history(d_f, &F, "pda_guessnet_train_step");
  if (!rc) rc = check_costs(costs, "pda_guessnet_train_step");
  if (rc) return rc;
  hipStream_t st = hipStream_t(stream);
  if (lossv) { // refused before the step is counted
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    PDA_HIP_CHECK(hipStreamIsCapturing(st, &cs));
    if (cs != hipStreamCaptureStatusNone) {
      set_error("pda_guessnet_train_step: the loss cannot be read while the stream is captured");
      return PDA_E_HIP;
    }
  }
  rc = forward(*net, feature_args(*net, F, nu), true, false, st);
  if (!rc) rc = loss(*net, costs, lossv != nullptr, st);
  if (!rc) rc = backward(*net, st);
  if (rc) return rc;
  const float b1 = 0.9f, b2 = 0.999f;
  net->adam_t += 1;
  const float c1 = 1.f / (1.f - std::pow(b1, float(net->adam_t)));
  const float c2 = 1.f / (1.f - std::pow(b2, float(net->adam_t)));
  hipLaunchKernelGGL(k_adam, dim3(unsigned((net->nparam + 255) / 256)), dim3(256), 0, st, net->w.as<float>(),
                     net->g.as<float>(), net->m1.as<float>(), net->m2.as<float>(), net->nparam, lr, b1, b2,
                     1e-8f, c1, c2);
  PDA_HIP_CHECK(hipGetLastError());
  rc = pack(*net, st);
  return rc || !lossv ? rc : read_loss(*net, lossv);
}

}  // extern "C"

// Batched per-fiber assembly of the implicit fiber system (FP64) for fibers of
// one node count N (5..64): persistent 256-thread workgroups, or up to four per
// fiber where there are few.
//
// Reference: fiber.form_linear_operator (python/fiber/fiber.py:322-447),
// apply_BC_rectangular with force- and torque-free ends (:810-961),
// force_operator (:1399-1431) and the tension projection of
// tstep_utils.py:1238-1336; derivative matrices of
// tstep/fiber_matrices.py:38-153 scaled by (2/L)^k.
//
// With D_k = (2/L)^k D0_k, xs = D_1 X, xss = D_2 X, xsss = D_3 X and the
// block-diagonal projection P = diag(PX, PX, PX, PT):
//   A (4N x 4N), blocks a, b in {x, y, z, T}:
//     A_ab (a, b < 3) = delta_ab I/dt + E diag(g_ab) D_4,
//        g_aa = c0 (1 + xs_a^2) + c1 (1 - xs_a^2),  g_ab = (c0 - c1) xs_a xs_b
//     A_aT = -2 c0 diag(xs_a) D_1 - (c0 + c1) diag(xss_a)
//     A_Tb = -(c1 + 7 c0) E diag(xss_b) D_4 - 6 c0 E diag(xsss_b) D_3
//            - p diag(xs_b) D_1
//     A_TT = -2 c0 D_2 + (c0 + c1) diag(|xss|^2)
//   A_sq = [P A ; 14 boundary rows]            (column-major, 4N x 4N)
//   F_a  = [-E D_4 in block a | diag(xss_a) + diag(xs_a) D_1 in block T]
//   Q_c  = P [e_c ; diag(xs_c) D_1]            ((4N - 14) x N)
// Layout of the work: persistent workgroups of four waves, one fiber at a
// time.  The block products P_a M_ab (A_sq's projected rows) and
// P_T (diag(xs_c) D_1) (the tension part of Q_c) run on the FP64 matrix cores
// as their transposes, M^T P^T: a wave keeps one 16-column tile of M for all
// its fibers, with that tile of D_1 .. D_4 in registers (the same for every
// fiber of the launch), forms its entries of M from them, and reads the
// projection from LDS; the transposed output, after an exchange between the
// row tiles, puts the rows of a column of A_sq in consecutive lanes.  The
// products go by column blocks, so that the pieces of a column (of 60 or 62
// rows, not whole lines) are written close together.
// A tile of the finite-difference D_k is zero outside a band of rows: the
// 4-deep MFMA steps outside it (found once per launch from D itself; a dense D
// has none) are skipped, which leaves every sum as it is.
// The remaining entries (boundary rows, Q's identity part; the derivatives of
// the centre lines and the force rows F_a in kernels of their own) go by
// columns, a lane per row, so that no index is divided.
// Bound by the stores (1.3 MB per fiber of 64 nodes) and by how far the forming
// of M hides behind them.  Measured, 4096 fibers of 64 nodes: 0.87 - 1.14 ms
// here, 0.06 ms derivatives, 0.28 ms force rows (5.7 TB/s) against 2.98 ms
// before (matrix entries formed per product from D in memory, all 16 steps, two
// integer divisions per element of F and Q); without the products' stores
// 0.51 ms less, without the matrix instructions the same.
#include "common.h"

#include <algorithm>

namespace f3d {

constexpr int kAsmNmax = 64;
constexpr int kAsmThreads = 256;

// Exchange 16-lane rows of two registers: 32, the upper half of x with the
// lower half of y; 16, the odd rows of x with the even rows of y.
template <int W>
__device__ __forceinline__ void swap_rows(double& x, double& y) {
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  u2 a = __builtin_bit_cast(u2, x), b = __builtin_bit_cast(u2, y);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const u2 s = W == 32 ? __builtin_amdgcn_permlane32_swap(a[h], b[h], false, false)
                         : __builtin_amdgcn_permlane16_swap(a[h], b[h], false, false);
    a[h] = s[0];
    b[h] = s[1];
  }
  x = __builtin_bit_cast(double, a);
  y = __builtin_bit_cast(double, b);
}

// xs, xss, xsss = D_1 X, D_2 X, D_3 X of every fiber and its weights: a lane per
// (fiber, component) with the coordinates in registers, up to kDerivRows rows of
// D per wave (one where few fibers leave CUs idle: 25 us with 8, 5 with one for 32
// fibers of 32 nodes), whose entries are wave-uniform (scalar loads).  xsss goes to the
// start of the fiber's force rows, which are written last.
constexpr int kDerivRows = 8;
template <int NMAX>
__global__ void __launch_bounds__(64)
fiber_deriv_kernel(int nfib, int N, int rows, const long* __restrict__ node0,
                   const double* __restrict__ length, const long* __restrict__ f_off,
                   const double* __restrict__ X, const double* __restrict__ D0,
                   const double* __restrict__ w0, double* __restrict__ xs,
                   double* __restrict__ xss, double* __restrict__ w, double* __restrict__ Fout) {
  const long t = (long)blockIdx.x * 64 + threadIdx.x;
  const int c = (int)(t % 3);
  const bool in = t / 3 < nfib;
  const int f = in ? (int)(t / 3) : nfib - 1;
  const long nd = node0[f];
  const double len = length[f], s1 = 2.0 / len, s2 = s1 * s1, s3 = s2 * s1;
  double x[NMAX];
#pragma unroll
  for (int q = 0; q < NMAX; ++q) x[q] = X[(nd + min(q, N - 1)) * 3 + c];
  const int k0 = blockIdx.y * rows, k1 = min(k0 + rows, N);
  for (int k = k0; k < k1; ++k) {
    const double* __restrict__ d = D0 + k * N;
    double e1 = 0.0, e2 = 0.0, e3 = 0.0;
#pragma unroll
    for (int q = 0; q < NMAX; ++q) {
      if (q < N) {
        e1 = fma(d[q], x[q], e1);
        e2 = fma(d[N * N + q], x[q], e2);
        e3 = fma(d[2 * N * N + q], x[q], e3);
      }
    }
    if (in) {
      xs[(nd + k) * 3 + c] = s1 * e1;
      xss[(nd + k) * 3 + c] = s2 * e2;
      Fout[f_off[f] + 3 * k + c] = s3 * e3;
      if (c == 0) w[nd + k] = w0[k] * (0.5 * len);
    }
  }
}

// Steps of a tile's D kept in registers (a band of 40 rows: stencils of up to
// 12 points); later ones, of a denser D, are read from memory.
constexpr int kBandSteps = 10;

// Workgroups that fit a CU (registers: 141 of 16 nodes, 203 of 32, 242 of 64).  A
// fiber of up to 16 nodes is one tile with four steps; in the form of 32 nodes
// half of its products and registers were padding: 9 nodes, 3000 fibers 73.6 ->
// 51.3 us, 256 fibers 16.8 -> 13.5, one 12.8 -> 10.1 (whole assembly).  A fourth
// workgroup spills: 48.0, 14.5, 10.1.
constexpr int asm_per_cu(int nmax) { return nmax <= 16 ? 3 : 2; }

template <int NMAX>
__global__ void __launch_bounds__(kAsmThreads, asm_per_cu(NMAX))
fiber_assemble_kernel(int nfib, int N, const long* __restrict__ node0,
                      const double* __restrict__ length, const long* __restrict__ a_off,
                      const long* __restrict__ f_off, const long* __restrict__ q_off,
                      const double* __restrict__ xs, const double* __restrict__ xss,
                      const double* __restrict__ xsss_f, const double* __restrict__ D0,
                      const double* __restrict__ PX, const double* __restrict__ PT, double E,
                      double dt, double c0, double c1, double pen, double* __restrict__ Aout,
                      double* __restrict__ Q0, double* __restrict__ Q1,
                      double* __restrict__ Q2) {
  typedef double v4d __attribute__((ext_vector_type(4)));
  constexpr int RT = NMAX / 16;  // row tiles of a projection
  constexpr int KS = NMAX / 4;   // 4-deep steps over the nodes
  constexpr int KB = KS < kBandSteps ? KS : kBandSteps;
  __shared__ double sxs[NMAX * 3], sxss[NMAX * 3], sxsss[NMAX * 3];
  // projections transposed, sP[k * NMAX + r] = P(r, k), zero-padded to NMAX
  __shared__ double sPX[NMAX * NMAX], sPT[NMAX * NMAX];
  // first and last rows of D_2 and D_3 (boundary conditions)
  __shared__ double sB2[2][NMAX], sB3[2][NMAX];

  const int t = threadIdx.x, lane = t & 63;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int g = lane >> 4, c16 = lane & 15;
  const int part = blockIdx.y, parts = gridDim.y;
  const int nx = N - 4, nt = N - 2, n4 = 4 * N, nq = n4 - 14;
  const int NN = N * N;
  for (int e = t; e < NMAX * NMAX; e += kAsmThreads) {
    const int k = e / NMAX, r = e % NMAX;
    sPX[e] = (k < N && r < nx) ? PX[r * N + k] : 0.0;
    sPT[e] = (k < N && r < nt) ? PT[r * N + k] : 0.0;
  }
  if (t < N) {
    sB2[0][t] = D0[NN + t];
    sB2[1][t] = D0[NN + (N - 1) * N + t];
    sB3[0][t] = D0[2 * NN + t];
    sB3[1][t] = D0[2 * NN + (N - 1) * N + t];
  }
  // this wave's column tile and its share of the tile's 19 products (1 or 2
  // tiles: 4 or 2 waves share one; 3 tiles: the fourth wave has none)
  const int ntj = (N + 15) / 16;
  const int jt = wv % ntj, share = ntj == 3 ? 1 : 4 / ntj;
  const int first = ntj == 3 && wv == 3 ? 19 : wv / ntj;
  const int jj = 16 * jt + c16, jc = min(jj, N - 1);
  // the tile's rows of D_1 .. D_4: steps lo .. lo + ks - 1 hold its non-zeros
  // and the diagonal
  int lo = KS, hi = 0;
#pragma unroll 4
  for (int st = 0; st < KS; ++st) {
    const int k = 4 * st + g;
    const bool in = k < N && jj < N;
    const double* __restrict__ d = D0 + (in ? k * N + jj : 0);
    const double e1 = d[0], e2 = d[NN], e3 = d[2 * NN], e4 = d[3 * NN];
    const bool any = in & ((k == jj) | (e1 != 0.0) | (e2 != 0.0) | (e3 != 0.0) | (e4 != 0.0));
    if (__ballot(any) != 0ull) {
      lo = min(lo, st);
      hi = st + 1;
    }
  }
  const int ks = hi - lo;
  double d1[KB], d2[KB], d3[KB], d4[KB];
#pragma unroll
  for (int i = 0; i < KB; ++i) {
    const int k = 4 * (lo + i) + g;
    const bool in = i < ks && k < N && jj < N;
    const int e = in ? k * N + jj : 0;
    d1[i] = in ? D0[e] : 0.0;
    d2[i] = in ? D0[NN + e] : 0.0;
    d3[i] = in ? D0[2 * NN + e] : 0.0;
    d4[i] = in ? D0[3 * NN + e] : 0.0;
  }

  // a fiber's derivatives are loaded before the previous fiber's stores: a
  // wait for a load waits for every store issued before it
  double nxs = 0.0, nxss = 0.0, nxsss = 0.0;
  auto fetch = [&](int f) __attribute__((always_inline)) {
    if (f < nfib && t < 3 * N) {
      const long e = node0[f] * 3 + t;
      nxs = xs[e];
      nxss = xss[e];
      nxsss = xsss_f[f_off[f] + t];
    }
  };
  fetch(blockIdx.x);
  for (int f = blockIdx.x; f < nfib; f += gridDim.x) {
    const double sc = 2.0 / length[f];
    const double s1 = sc, s2 = sc * sc, s3 = s2 * sc, s4 = s2 * s2;
    // (LDS only: one fiber's stores drain during the next)
    lds_barrier();  // LDS reuse across fibers (and the set-up above)
    if (t < 3 * N) {
      sxs[t] = nxs;
      sxss[t] = nxss;
      sxsss[t] = nxsss;
    }
    lds_barrier();
    fetch(f + gridDim.x);

    double* __restrict__ Af = Aout + a_off[f];
    // ---- projected products: p = 4 a + b < 16 is block (a, b) of A_sq's
    // projected rows; p = 16 + c is the tension part of Q_c.
    for (int p = first + share * part; p < 19; p += share * parts) {
      const int a = p < 16 ? p & 3 : 4 + (p - 16), b = p < 16 ? p >> 2 : 0;
      const bool tens = a >= 3;
      const int rows = tens ? nt : nx;
      const double* __restrict__ sP = (tens ? sPT : sPX) + 4 * lo * NMAX;
      v4d acc[RT];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) acc[rt] = v4d{0.0, 0.0, 0.0, 0.0};
      // entry(k, D_1 .. D_4 at (k, jj)): M(k, jj) (rows past N meet zeros of P)
      auto product = [&](auto&& entry) __attribute__((always_inline)) {
        auto step = [&](int i, double e1, double e2, double e3, double e4)
            __attribute__((always_inline)) {
          const double mv = entry(min(4 * (lo + i) + g, N - 1), 4 * (lo + i) + g == jj, e1, e2, e3, e4);
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) {
            const double pv = sP[(4 * i + g) * NMAX + 16 * rt + c16];
            acc[rt] = __builtin_amdgcn_mfma_f64_16x16x4f64(mv, pv, acc[rt], 0, 0, 0);
          }
        };
#pragma unroll
        for (int i = 0; i < KB; ++i)
          if (i < ks) step(i, d1[i], d2[i], d3[i], d4[i]);
#pragma unroll 1
        for (int i = KB; i < ks; ++i) {
          const double* __restrict__ d = D0 + min(4 * (lo + i) + g, N - 1) * N + jc;
          step(i, d[0], d[NN], d[2 * NN], d[3 * NN]);
        }
      };
      if (a < 3 && b < 3) {
        const double diag = a == b ? 1.0 / dt : 0.0;
        product([&](int k, bool on, double, double, double, double e4)
                    __attribute__((always_inline)) {
          const double xa = sxs[k * 3 + a], xb = sxs[k * 3 + b];
          const double gk = a == b ? c0 * (1.0 + xa * xa) + c1 * (1.0 - xa * xa)
                                   : (c0 - c1) * xa * xb;
          return E * gk * s4 * e4 + (on ? diag : 0.0);
        });
      } else if (a < 3) {
        product([&](int k, bool on, double e1, double, double, double)
                    __attribute__((always_inline)) {
          return -2.0 * c0 * sxs[k * 3 + a] * s1 * e1 -
                 (on ? (c0 + c1) * sxss[k * 3 + a] : 0.0);
        });
      } else if (a == 3 && b < 3) {
        product([&](int k, bool, double e1, double, double e3, double e4)
                    __attribute__((always_inline)) {
          return -(c1 + 7.0 * c0) * E * sxss[k * 3 + b] * s4 * e4 -
                 6.0 * c0 * E * sxsss[k * 3 + b] * s3 * e3 - pen * sxs[k * 3 + b] * s1 * e1;
        });
      } else if (a == 3) {
        product([&](int k, bool on, double, double e2, double, double)
                    __attribute__((always_inline)) {
          const double x0 = sxss[k * 3], x1 = sxss[k * 3 + 1], x2 = sxss[k * 3 + 2];
          return -2.0 * c0 * s2 * e2 +
                 (on ? (c1 + c0) * (x0 * x0 + x1 * x1 + x2 * x2) : 0.0);
        });
      } else {
        product([&](int k, bool, double e1, double, double, double)
                    __attribute__((always_inline)) { return sxs[k * 3 + (a - 4)] * s1 * e1; });
      }
      // element e of lane (g, c16): row 16 rt + c16 of column 16 jt + 4 e + g.
      // The row tiles trade 16-lane rows, so that a store covers all rows of
      // one column (NMAX 64) or of two (32) instead of 16 rows of four (16).
      double* __restrict__ dst;
      int col_stride;
      if (a < 4) {
        dst = Af + (long)b * N * n4 + (a < 3 ? a * nx : 3 * nx);
        col_stride = n4;
      } else {
        double* __restrict__ Q = a == 4 ? Q0 : (a == 5 ? Q1 : Q2);
        dst = Q + q_off[3 * f + (a - 4)] + 3 * nx;
        col_stride = nq;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        double col[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) col[rt] = acc[rt][e];
        if constexpr (RT == 4) {
          swap_rows<32>(col[0], col[2]);
          swap_rows<32>(col[1], col[3]);
          swap_rows<16>(col[0], col[1]);
          swap_rows<16>(col[2], col[3]);
        } else if constexpr (RT == 2) {
          swap_rows<16>(col[0], col[1]);
        }
#pragma unroll
        for (int q = 0; q < RT; ++q) {
          // RT 4: column q, row lane; RT 2: columns q and q + 2, row lane % 32;
          // RT 1: columns 0 .. 3, row lane % 16
          const int r = lane & (NMAX - 1);
          const int jc = 16 * jt + 4 * e + q + RT * (lane / NMAX);
          if (r < rows && jc < N) dst[jc * col_stride + r] = col[q];
        }
      }
    }

    // ---- 14 boundary rows of every column (force- and torque-free ends):
    // four columns per wave, a lane per row
    for (int j0 = 4 * (wv + 4 * part); j0 < n4; j0 += 16 * parts) {
      const int j = j0 + g, r = c16;
      if (j < n4 && r < 14) {
        const int b = (j >= N) + (j >= 2 * N) + (j >= 3 * N), jb = j - b * N;
        double v = 0.0;
        if (b < 3) {
          if (r == b) v = E * s3 * sB3[0][jb];
          else if (r == 3) v = -E * s2 * sB2[0][jb] * sxss[b];
          else if (r == 4 + b) v = s2 * sB2[0][jb];
          else if (r == 7 + b) v = -E * s3 * sB3[1][jb];
          else if (r == 10) v = E * s2 * sB2[1][jb] * sxss[(N - 1) * 3 + b];
          else if (r == 11 + b) v = s2 * sB2[1][jb];
        } else {
          if (jb == 0 && r < 3) v = -sxs[r];
          else if (jb == 0 && r == 3) v = -1.0;
          else if (jb == N - 1 && r >= 7 && r < 10) v = sxs[(N - 1) * 3 + (r - 7)];
          else if (jb == N - 1 && r == 10) v = 1.0;
        }
        Af[(long)j * n4 + (n4 - 14) + r] = v;
      }
    }
    // ---- identity part of Q_c: rows [0, 3 nx), P_X in row block c (streamed past
    // L2, like the force rows: 41 and 27 us of 4096 fibers x 64; the products are
    // not, their pieces of lines meet in L2: +140 us) --------
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double* __restrict__ Q = (c == 0 ? Q0 : (c == 1 ? Q1 : Q2)) + q_off[3 * f + c];
      for (int j = wv + 4 * part; j < N; j += 4 * parts) {
#pragma unroll
        for (int b = 0; b < 3; ++b)
          if (lane < nx)
            __builtin_nontemporal_store(b == c ? sPX[j * NMAX + lane] : 0.0,
                                        &Q[j * nq + b * nx + lane]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Force operator F_a of every fiber (three row blocks N x 4N, column-major,
// adjacent): one or two columns per wave, a lane per row.  A wave keeps its
// columns of D_4 and D_1 (read once, against their rows) in registers for all
// its fibers; the rest is stores.  (Inside the assembly above, reading D per
// fiber, this part took 750 us of the 4096 x 64 launch.)
template <int NMAX>
__global__ void __launch_bounds__(256)
fiber_force_kernel(int nfib, int N, const long* __restrict__ node0,
                   const double* __restrict__ length, const long* __restrict__ f_off,
                   const double* __restrict__ D0, const double* __restrict__ xs,
                   const double* __restrict__ xss, double E, double* __restrict__ Fout) {
  constexpr int CW = 64 / NMAX;        // columns per wave and step
  constexpr int NC = NMAX / (4 * CW);  // steps of the workgroup's four waves
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int i = lane % NMAX, j0 = CW * wv + lane / NMAX;
  const double* __restrict__ D04 = D0 + 3l * N * N;
  double c1[NC], c4[NC];
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    const int j = j0 + 4 * CW * q;
    const bool in = i < N && j < N;
    c1[q] = in ? D0[i * N + j] : 0.0;
    c4[q] = in ? D04[i * N + j] : 0.0;
  }
  for (int f = blockIdx.x; f < nfib; f += gridDim.x) {
    if (i >= N) continue;
    const long nd = (node0[f] + i) * 3;
    const double s1 = 2.0 / length[f], s2 = s1 * s1, s4 = s2 * s2;
    double xa[3], xxa[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      xa[a] = xs[nd + a] * s1;
      xxa[a] = xss[nd + a];
    }
    double* __restrict__ Fb = Fout + f_off[f] + i;
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      const int j = j0 + 4 * CW * q;
      if (j >= N) break;
      const double v4 = -E * s4 * c4[q];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        double* __restrict__ Fa = Fb + a * (4 * N * N) + j * N;
#pragma unroll
        for (int b = 0; b < 3; ++b)
          __builtin_nontemporal_store(b == a ? v4 : 0.0, &Fa[b * (N * N)]);
        __builtin_nontemporal_store(xa[a] * c1[q] + (i == j ? xxa[a] : 0.0), &Fa[3 * (N * N)]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Per-fiber right-hand side with the plus-end force f = F_end x_s(L) at the
// last node (zero elsewhere) and the explicit flow v at the nodes:
//   R_a = X_a / dt + v_a + c0 (f_a + x_s,a (x_s . f)) + c1 (f_a - x_s,a (x_s . f))
//   R_T = -p + x_s . (D_1 v) + 2 c0 x_s . (D_1 f) + (c0 - c1) x_ss . f
//   rhs = [P R ; 14 end rows: 0 ... F_end at rows 7..9, F_end . x_s(L) at 10]
// Persistent workgroups, one fiber at a time: wave a < 3 has component a, wave
// 3 the tension, a lane per row.  A lane keeps its row of the projection in
// registers and D_1 is read from a transposed copy in LDS (consecutive lanes,
// consecutive rows), both loaded once per workgroup; the next fiber's nodes are
// on their way during this one.  Every sum keeps its order k = 0 .. N - 1.
// Bound by those N-term chains (the data are 8 KB per fiber).  Measured, 4096
// fibers of 64 nodes: 66 us; 187 us with the rows read from memory per fiber (a lane
// per row: 64 lines per load, and D_1 v by one wave).
template <int NMAX>
__global__ void __launch_bounds__(256, 2)
fiber_rhs_kernel(int nfib, int N, const long* __restrict__ node0,
                 const double* __restrict__ length, const long* __restrict__ rhs_off,
                 const double* __restrict__ X, const double* __restrict__ xs,
                 const double* __restrict__ xss, const double* __restrict__ v,
                 const double* __restrict__ D01, const double* __restrict__ PX,
                 const double* __restrict__ PT, double dt, double c0, double c1, double pen,
                 double end_force, double* __restrict__ rhs) {
  __shared__ double sD[NMAX * NMAX];  // sD[q * NMAX + k] = D_1(k, q), unscaled
  __shared__ double sX[3][NMAX], sxs[3][NMAX], sv[3][NMAX], sdv[3][NMAX];
  __shared__ double sR[4][NMAX], sxssL[3];
  const int t = threadIdx.x, lane = t & 63;
  const int a = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nx = N - 4, nt = N - 2, L = N - 1;
  const int rows = a < 3 ? nx : nt;
  for (int e = t; e < NMAX * NMAX; e += 256) {
    const int k = e / NMAX, q = e % NMAX;
    if (k < N && q < N) sD[q * NMAX + k] = D01[k * N + q];
  }
  double pr[NMAX];
  {
    const double* __restrict__ P = (a < 3 ? PX : PT) + min(lane, rows - 1) * N;
#pragma unroll
    for (int k = 0; k < NMAX; ++k) pr[k] = P[min(k, L)];
  }
  const int ln = min(lane, L);  // the lane's node
  const int tk = t / 3, ta = t - 3 * tk;
  double nX = 0.0, nxs = 0.0, nv = 0.0, nxss = 0.0;
  auto fetch = [&](int f) __attribute__((always_inline)) {
    if (f < nfib && t < 3 * N) {
      const long e = node0[f] * 3 + t;
      nX = X[e];
      nxs = xs[e];
      nv = v[e];
      nxss = tk == L ? xss[e] : 0.0;
    }
  };
  fetch(blockIdx.x);
  for (int f = blockIdx.x; f < nfib; f += gridDim.x) {
    const double s1 = 2.0 / length[f];
    lds_barrier();  // LDS reuse across fibers (and the set-up above)
    if (t < 3 * N) {
      sX[ta][tk] = nX;
      sxs[ta][tk] = nxs;
      sv[ta][tk] = nv;
      if (tk == L) sxssL[ta] = nxss;
    }
    lds_barrier();
    fetch(f + gridDim.x);
    const double fl0 = end_force * sxs[0][L], fl1 = end_force * sxs[1][L],
                 fl2 = end_force * sxs[2][L];
    const double x0 = sxs[0][ln], x1 = sxs[1][ln], x2 = sxs[2][ln];
    if (a < 3) {
      const bool last = ln == L;
      const double xa = a == 0 ? x0 : (a == 1 ? x1 : x2);
      const double fa = last ? (a == 0 ? fl0 : (a == 1 ? fl1 : fl2)) : 0.0;
      const double xf = last ? x0 * fl0 + x1 * fl1 + x2 * fl2 : 0.0;
      const double R = sX[a][ln] / dt + sv[a][ln] + c0 * (fa + xa * xf) + c1 * (fa - xa * xf);
      double d = 0.0;
      for (int q = 0; q < N; ++q) d = fma(sD[q * NMAX + ln], sv[a][q], d);
      if (lane < N) {
        sR[a][lane] = R;
        sdv[a][lane] = d;
      }
    }
    lds_barrier();
    if (a == 3) {
      double dv = 0.0;
      dv = fma(x0, s1 * sdv[0][ln], dv);
      dv = fma(x1, s1 * sdv[1][ln], dv);
      dv = fma(x2, s1 * sdv[2][ln], dv);
      const double d1l = s1 * sD[L * NMAX + ln];
      const double df = (x0 * fl0 + x1 * fl1 + x2 * fl2) * d1l;
      const double xssf = ln == L ? sxssL[0] * fl0 + sxssL[1] * fl1 + sxssL[2] * fl2 : 0.0;
      if (lane < N) sR[3][lane] = -pen + dv + 2.0 * c0 * df + (c0 - c1) * xssf;
    }
    // (a wave reads only the row of R that it wrote itself)
    double val = 0.0;
#pragma unroll
    for (int k = 0; k < NMAX; ++k)
      if (k < N) val = fma(pr[k], sR[a][k], val);
    double* __restrict__ out = rhs + rhs_off[f];
    if (lane < rows) out[a * nx + lane] = val;
    if (a == 0 && lane < 14) {
      double br = 0.0;
      if (lane == 7) br = fl0;
      else if (lane == 8) br = fl1;
      else if (lane == 9) br = fl2;
      else if (lane == 10) br = fl0 * sxs[0][L] + fl1 * sxs[1][L] + fl2 * sxs[2][L];
      out[4 * N - 14 + lane] = br;
    }
  }
}

// ---------------------------------------------------------------------------
// Plus-end forces F_end x_s(L): the force at every node (zero but at the ends),
// and the ends' positions, forces and weights as compact arrays for the explicit
// flows.  A wave per fiber.  Seven gathers and fills of a few KB, 5 us each, in
// one launch.
__global__ void __launch_bounds__(64)
fiber_end_kernel(const long* __restrict__ end_idx, const double* __restrict__ X,
                 const double* __restrict__ xs, const double* __restrict__ w, double end_force,
                 double* __restrict__ force, double* __restrict__ Xe, double* __restrict__ fe,
                 double* __restrict__ we) {
  const int f = blockIdx.x;
  const long last = end_idx[f], first = f ? end_idx[f - 1] + 1 : 0;
  for (long e = first * 3 + threadIdx.x; e < last * 3; e += 64) force[e] = 0.0;
  if (threadIdx.x < 3) {
    const int c = threadIdx.x;
    const double v = end_force * xs[last * 3 + c];
    force[last * 3 + c] = v;
    fe[f * 3l + c] = v;
    Xe[f * 3l + c] = X[last * 3 + c];
    if (c == 0) we[f] = w[last];
  }
}

}  // namespace f3d

using namespace f3d;

extern "C" int f3d_fiber_assemble(int64_t nfib, int32_t N, const int64_t* node0,
                                  const double* length, const int64_t* a_off,
                                  const int64_t* f_off, const int64_t* q_off, const double* X,
                                  const double* D0, const double* PX, const double* PT,
                                  const double* w0, double E, double dt, double c0, double c1,
                                  double penalty, double* A_out, double* F_out, double* Q0,
                                  double* Q1, double* Q2, double* xs_out, double* xss_out,
                                  double* w_out, void* stream) {
  F3D_REQUIRE(N >= 5 && N <= kAsmNmax, F3D_EINVAL, "fiber_assemble: N=%d outside [5,%d]", N,
              kAsmNmax);
  F3D_REQUIRE(nfib >= 0 && nfib < (1ll << 31), F3D_EINVAL, "fiber_assemble: bad fiber count");
  F3D_REQUIRE(dt > 0.0, F3D_EINVAL, "fiber_assemble: dt must be positive");
  if (nfib == 0) return F3D_OK;
  F3D_REQUIRE(node0 && length && a_off && f_off && q_off && X && D0 && PX && PT && w0 && A_out &&
                  F_out && Q0 && Q1 && Q2 && xs_out && xss_out && w_out,
              F3D_EINVAL, "fiber_assemble: NULL argument");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // persistent: as many workgroups as fit a CU
  const int64_t most = asm_per_cu(N <= 16 ? 16 : kAsmNmax) * (int64_t)num_cus();
  const unsigned grid = (unsigned)(nfib < most ? nfib : most);
  const unsigned fgrid = (unsigned)(nfib < 4 * most ? nfib : 4 * most);
  const int64_t dwaves = ceil_div(3 * nfib, (int64_t)64);
  const int rows = (int)std::min<int64_t>(kDerivRows, ceil_div(dwaves * N, 2 * most));
  const dim3 dgrid((unsigned)dwaves, (unsigned)ceil_div(N, rows));
  // few fibers: several workgroups share one, by products and columns
  const unsigned parts = nfib * 4 <= most ? 4 : (nfib * 2 <= most ? 2 : 1);
#define F3D_ASM(NM)                                                                             \
  F3D_LAUNCH(fiber_deriv_kernel<NM>, dgrid, dim3(64), 0, st, (int)nfib, (int)N, rows,           \
             (const long*)node0, length, (const long*)f_off, X, D0, w0, xs_out, xss_out, w_out, \
             F_out);                                                                            \
  F3D_LAUNCH(fiber_assemble_kernel<NM>, dim3(grid, parts), dim3(kAsmThreads), 0, st, (int)nfib, (int)N, \
             (const long*)node0, length, (const long*)a_off, (const long*)f_off,                \
             (const long*)q_off, (const double*)xs_out, (const double*)xss_out,                 \
             (const double*)F_out, D0, PX, PT, E, dt, c0, c1, penalty, A_out, Q0, Q1, Q2);      \
  F3D_LAUNCH(fiber_force_kernel<NM>, dim3(fgrid), dim3(256), 0, st, (int)nfib, (int)N,          \
             (const long*)node0, length, (const long*)f_off, D0, (const double*)xs_out,         \
             (const double*)xss_out, E, F_out)
  if (N <= 16) {
    F3D_ASM(16);
  } else if (N <= 32) {
    F3D_ASM(32);
  } else {
    F3D_ASM(64);
  }
#undef F3D_ASM
  return F3D_OK;
}

extern "C" int f3d_fiber_rhs(int64_t nfib, int32_t N, const int64_t* node0, const double* length,
                             const int64_t* rhs_off, const double* X, const double* xs,
                             const double* xss, const double* v, const double* D0,
                             const double* PX, const double* PT, double dt, double c0, double c1,
                             double penalty, double end_force, double* rhs, void* stream) {
  F3D_REQUIRE(N >= 5 && N <= kAsmNmax, F3D_EINVAL, "fiber_rhs: N=%d outside [5,%d]", N,
              kAsmNmax);
  F3D_REQUIRE(nfib >= 0 && nfib < (1ll << 31), F3D_EINVAL, "fiber_rhs: bad fiber count");
  F3D_REQUIRE(dt > 0.0, F3D_EINVAL, "fiber_rhs: dt must be positive");
  if (nfib == 0) return F3D_OK;
  F3D_REQUIRE(node0 && length && rhs_off && X && xs && xss && v && D0 && PX && PT && rhs,
              F3D_EINVAL, "fiber_rhs: NULL argument");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // persistent: two workgroups fit a CU (registers)
  const int64_t most = 2 * (int64_t)num_cus();
  const unsigned grid = (unsigned)(nfib < most ? nfib : most);
#define F3D_RHS(NM)                                                                          \
  F3D_LAUNCH(fiber_rhs_kernel<NM>, dim3(grid), dim3(256), 0, st, (int)nfib, (int)N,          \
             (const long*)node0, length, (const long*)rhs_off, X, xs, xss, v, D0, PX, PT, dt, \
             c0, c1, penalty, end_force, rhs)
  if (N <= 32) {
    F3D_RHS(32);
  } else {
    F3D_RHS(64);
  }
#undef F3D_RHS
  return F3D_OK;
}

extern "C" int f3d_fiber_ends(int64_t nfib, const int64_t* end_idx, const double* X,
                              const double* xs, const double* w, double end_force, double* force,
                              double* Xe, double* fe, double* we, void* stream) {
  F3D_REQUIRE(nfib >= 0 && nfib < (1ll << 31), F3D_EINVAL, "fiber_ends: bad fiber count");
  if (nfib == 0) return F3D_OK;
  F3D_REQUIRE(end_idx && X && xs && w && force && Xe && fe && we, F3D_EINVAL,
              "fiber_ends: NULL argument");
  F3D_LAUNCH(fiber_end_kernel, dim3((unsigned)nfib), dim3(64), 0,
             reinterpret_cast<hipStream_t>(stream), (const long*)end_idx, X, xs, w, end_force,
             force, Xe, fe, we);
  return F3D_OK;
}

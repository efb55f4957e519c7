// Batched dense kernels over per-fiber blocks of uneven order (n <= 256):
//   * LU factorisation with partial pivoting (LAPACK dgetrf semantics): the
//     entry point, which runs lu_block.hip, and two alternatives it takes on
//     request: FP64 register/LDS-resident, one persistent 1024-thread
//     workgroup per block; equilibrated FP32 blocked on MFMA
//     (lu_factor_f32_mfma_kernel below), two 256-thread workgroups per CU;
//   * forward/backward substitution with optional FP64 iterative refinement,
//     one wavefront per block;
//   * column-major block GEMV, sums of up to four products, one workgroup per
//     block.
//
// Reference: scipy.linalg.lu_factor / lu_solve per fiber in
// python/tstep/tstep_utils.py:1405-1419 and python/tstep/tstep.py:985-988;
// the block-diagonal apply As_fibers.dot(XT) in python/tstep/tstep.py:1173.
//
// LU layout on the CU: the 1024 threads form a 32 x 32 grid (tr = row lane,
// tc = column lane); thread (tr, tc) owns rows tr + 32a and columns tc + 32b,
// a, b in [0, 8), i.e. a 2-D cyclic distribution that keeps every thread busy
// as the trailing matrix shrinks.  FP32 blocks (256 KB at n = 256) live wholly
// in registers.  FP64 blocks (512 KB) do not fit the register file, so the
// last 64 columns live in LDS (128 KB) and the rest in registers.  Each
// elimination step costs two workgroup barriers: pivot search (column owners,
// half-wave shuffles) -> publish pivot row / old row k / column k through LDS
// -> every thread swaps, forms its multipliers and updates its tile.
#include "common.h"

#include <type_traits>

#include <stdlib.h>
#include <string.h>

namespace f3d {

constexpr int kLuG = 32;     // thread grid is kLuG x kLuG
constexpr int kLuTL = 8;     // tile slots per thread and dimension
constexpr int kLuNmax = kLuG * kLuTL;  // 256

__device__ __forceinline__ double readlane_f64(double v, int lane) {
  const unsigned long long u = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(u & 0xffffffffu), lane);
  const int hi = __builtin_amdgcn_readlane((int)(u >> 32), lane);
  return __longlong_as_double(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

// Power of two s with s * amax in [0.5, 1); 1 for amax == 0 or non-finite.
__device__ __forceinline__ double pow2_scale(double amax) {
  if (!(amax > 0.0) || !isfinite(amax)) return 1.0;
  int e;
  frexp(amax, &e);
  return ldexp(1.0, -e);
}

template <typename T, int TLC_LDS>
struct LuTile {
  static constexpr int TLC_REG = kLuTL - TLC_LDS;
  T r[kLuTL][TLC_REG > 0 ? TLC_REG : 1];
  T* lds;  // column-major [32*TLC_LDS][256] for columns >= 32*TLC_REG
  int tr, tc;
  __device__ __forceinline__ T get(int a, int b) const {
    if (b < TLC_REG) return r[a][b];
    return lds[(tc + kLuG * (b - TLC_REG)) * kLuNmax + tr + kLuG * a];
  }
  __device__ __forceinline__ void set(int a, int b, T v) {
    if (b < TLC_REG) r[a][b] = v;
    else lds[(tc + kLuG * (b - TLC_REG)) * kLuNmax + tr + kLuG * a] = v;
  }
};

template <typename T, int TLC_LDS>
__global__ void __launch_bounds__(1024)
lu_factor_kernel(int nb, const int* __restrict__ n_arr, const long* __restrict__ a_off,
                 const long* __restrict__ x_off, const int* __restrict__ order,
                 const double* __restrict__ A, T* __restrict__ LU, double* __restrict__ rs,
                 double* __restrict__ cs, int* __restrict__ piv, int* __restrict__ perm,
                 int* __restrict__ info, int equilibrate) {
  __shared__ T lds_mat[TLC_LDS > 0 ? kLuG * TLC_LDS * kLuNmax : 1];
  __shared__ T rowU[kLuNmax], rowK[kLuNmax], colL[kLuNmax];
  __shared__ unsigned long long amax_bits[kLuNmax];
  __shared__ double scl_r[kLuNmax], scl_c[kLuNmax];
  __shared__ int sh_perm[kLuNmax];
  __shared__ int sh_piv, sh_info;

  LuTile<T, TLC_LDS> t;
  t.lds = lds_mat;
  t.tr = threadIdx.x % kLuG;
  t.tc = threadIdx.x / kLuG;
  const int tr = t.tr, tc = t.tc;

  for (int w = blockIdx.x; w < nb; w += gridDim.x) {
    const int b = order ? order[w] : w;
    const int n = n_arr[b];
    if (n < 1 || n > kLuNmax) {  // uniform per block: every thread skips
      if (threadIdx.x == 0) info[b] = -1;
      continue;
    }
    const int mc = (n + kLuG - 1) / kLuG;  // occupied slots per dimension
    const double* __restrict__ Ab = A + a_off[b];
    const long xo = x_off[b];
    __syncthreads();  // LDS reuse across blocks

    // ---- equilibration scales (powers of two, so scaling is exact) -------
    if (threadIdx.x < kLuNmax) {
      sh_perm[threadIdx.x] = threadIdx.x;
      amax_bits[threadIdx.x] = 0ull;
      scl_r[threadIdx.x] = 1.0;
      scl_c[threadIdx.x] = 1.0;
    }
    if (threadIdx.x == 0) sh_info = 0;
    __syncthreads();
    if (equilibrate) {
      // row maxima
#pragma unroll
      for (int a = 0; a < kLuTL; ++a) {
        const int i = tr + kLuG * a;
        if (a >= mc || i >= n) continue;
        double m = 0.0;
#pragma unroll
        for (int bb = 0; bb < kLuTL; ++bb) {
          const int j = tc + kLuG * bb;
          if (bb < mc && j < n) m = fmax(m, fabs(Ab[i + (long)j * n]));
        }
        atomicMax(&amax_bits[i], (unsigned long long)__double_as_longlong(m));
      }
      __syncthreads();
      if (threadIdx.x < n) {
        scl_r[threadIdx.x] = pow2_scale(__longlong_as_double((long long)amax_bits[threadIdx.x]));
        amax_bits[threadIdx.x] = 0ull;
      }
      __syncthreads();
      // column maxima of the row-scaled matrix
#pragma unroll
      for (int bb = 0; bb < kLuTL; ++bb) {
        const int j = tc + kLuG * bb;
        if (bb >= mc || j >= n) continue;
        double m = 0.0;
#pragma unroll
        for (int a = 0; a < kLuTL; ++a) {
          const int i = tr + kLuG * a;
          if (a < mc && i < n) m = fmax(m, fabs(Ab[i + (long)j * n]) * scl_r[i]);
        }
        atomicMax(&amax_bits[j], (unsigned long long)__double_as_longlong(m));
      }
      __syncthreads();
      if (threadIdx.x < n)
        scl_c[threadIdx.x] = pow2_scale(__longlong_as_double((long long)amax_bits[threadIdx.x]));
      __syncthreads();
    }

    // ---- load the (scaled) block into the tile ---------------------------
#pragma unroll
    for (int a = 0; a < kLuTL; ++a) {
#pragma unroll
      for (int bb = 0; bb < kLuTL; ++bb) {
        const int i = tr + kLuG * a, j = tc + kLuG * bb;
        T v = 0;
        if (a < mc && bb < mc && i < n && j < n) v = (T)(Ab[i + (long)j * n] * scl_r[i] * scl_c[j]);
        t.set(a, bb, v);
      }
    }
    __syncthreads();

    // ---- right-looking elimination --------------------------------------
    for (int k = 0; k < n; ++k) {
      const int kb = k / kLuG, kc = k % kLuG;
      if (tc == kc) {
        double best = -1.0;
        int bi = n;
#pragma unroll
        for (int a = 0; a < kLuTL; ++a) {
          const int i = tr + kLuG * a;
          T v = 0;
#pragma unroll
          for (int bb = 0; bb < kLuTL; ++bb)
            if (bb == kb) v = t.get(a, bb);
          const double av = fabs((double)v);
          if (a < mc && i >= k && i < n && av > best) {
            best = av;
            bi = i;
          }
        }
#pragma unroll
        for (int o = 16; o >= 1; o >>= 1) {
          const double ob = __shfl_xor(best, o, 32);
          const int oi = __shfl_xor(bi, o, 32);
          if (ob > best || (ob == best && oi < bi)) {
            best = ob;
            bi = oi;
          }
        }
        if (tr == 0) {
          sh_piv = bi;
          if (best == 0.0 && sh_info == 0) sh_info = k + 1;
        }
      }
      __syncthreads();
      const int p = sh_piv;
      const int ka = k / kLuG, kr = k % kLuG, pa = p / kLuG, pr = p % kLuG;
      // publish pivot row (old row p), old row k and old column k
#pragma unroll
      for (int bb = 0; bb < kLuTL; ++bb) {
        const int j = tc + kLuG * bb;
        if (bb < mc && j < n) {
          if (tr == pr) {
            T v = 0;
#pragma unroll
            for (int a = 0; a < kLuTL; ++a)
              if (a == pa) v = t.get(a, bb);
            rowU[j] = v;
          }
          if (tr == kr) {
            T v = 0;
#pragma unroll
            for (int a = 0; a < kLuTL; ++a)
              if (a == ka) v = t.get(a, bb);
            rowK[j] = v;
          }
        }
      }
      if (tc == kc) {
#pragma unroll
        for (int a = 0; a < kLuTL; ++a) {
          const int i = tr + kLuG * a;
          T v = 0;
#pragma unroll
          for (int bb = 0; bb < kLuTL; ++bb)
            if (bb == kb) v = t.get(a, bb);
          if (a < mc && i < n) colL[i] = v;
        }
      }
      if (threadIdx.x == 0) {
        piv[xo + k] = p;
        const int tmp = sh_perm[k];
        sh_perm[k] = sh_perm[p];
        sh_perm[p] = tmp;
      }
      __syncthreads();
      const T ukk = rowU[k];
      const T inv = (ukk != (T)0) ? (T)1 / ukk : (T)0;
      T u[kLuTL];
#pragma unroll
      for (int bb = 0; bb < kLuTL; ++bb) {
        const int j = tc + kLuG * bb;
        u[bb] = (bb < mc && j > k && j < n) ? rowU[j] : (T)0;
      }
#pragma unroll
      for (int a = 0; a < kLuTL; ++a) {
        const int i = tr + kLuG * a;
        if (a >= mc || i >= n || i < k) continue;
        if (i == k || i == p) {
#pragma unroll
          for (int bb = 0; bb < kLuTL; ++bb) {
            const int j = tc + kLuG * bb;
            if (bb < mc && j < n) t.set(a, bb, i == k ? rowU[j] : rowK[j]);
          }
        }
        if (i == k) continue;
        const T raw = (i == p) ? rowK[k] : colL[i];
        const T l = raw * inv;
        if (tc == kc) {
#pragma unroll
          for (int bb = 0; bb < kLuTL; ++bb)
            if (bb == kb) t.set(a, bb, l);
        }
#pragma unroll
        for (int bb = 0; bb < kLuTL; ++bb)
          if (bb < mc) t.set(a, bb, t.get(a, bb) - l * u[bb]);
      }
      // The next step's pivot search reads only registers/LDS tile entries
      // that this thread itself updated; the next LDS publish happens after
      // that step's first barrier, which every thread reaches only once it
      // is done with rowU/rowK/colL here.
    }
    __syncthreads();

    // ---- write factors, permutation, scales ----------------------------
    T* __restrict__ Lb = LU + a_off[b];
#pragma unroll
    for (int a = 0; a < kLuTL; ++a) {
#pragma unroll
      for (int bb = 0; bb < kLuTL; ++bb) {
        const int i = tr + kLuG * a, j = tc + kLuG * bb;
        if (a < mc && bb < mc && i < n && j < n) Lb[i + (long)j * n] = t.get(a, bb);
      }
    }
    if (threadIdx.x < n) {
      perm[xo + threadIdx.x] = sh_perm[threadIdx.x];
      if (rs) rs[xo + threadIdx.x] = scl_r[threadIdx.x];
      if (cs) cs[xo + threadIdx.x] = scl_c[threadIdx.x];
    }
    if (threadIdx.x == 0) info[b] = sh_info;
  }
}

// ---------------------------------------------------------------------------
// FP32 blocked LU on MFMA (right-looking, panel width 32, LAPACK getrf
// semantics on the equilibrated matrix), one 256-thread workgroup per block,
// two workgroups per CU.  The equilibrated FP32 matrix is written to the
// output buffer and factored in place there (L2-resident: 256 KB per block).
// Per panel k (columns c0 = 32k .. c0 + 31, local rows 0 .. m-1 from c0 on):
//   1. the panel is loaded into LDS (sL, column-major, one row per thread)
//      and factored column by column with partial pivoting: block argmax
//      (first maximum), row swap, multipliers, rank-1 update of the panel;
//      two barriers per column;
//   2. each thread owns one matrix column outside the panel: it applies the
//      panel's 32 row swaps in order and, right of the panel, solves
//      U12 = L11^-1 A12 for its column (copy kept in LDS, sU, row-major);
//   3. A22 -= L21 U12 on 32 x 32 tiles, one tile per wave at a time:
//      v_mfma_f32_32x32x2f32 with A = -L21 and B = U12 from LDS, C / D
//      loaded from and stored to the factor buffer.
// Orders that are not a multiple of 32 are padded with an identity block
// that is never stored: virtual rows and columns stay decoupled, so the
// factors of the real part are exactly those of the unpadded matrix.
constexpr int kPw = 32;               // panel width = MFMA tile edge
constexpr int kMfThreads = 256;       // 4 waves

typedef float f32x16 __attribute__((ext_vector_type(16)));

__global__ void __launch_bounds__(kMfThreads, 2)
lu_factor_f32_mfma_kernel(int nb, const int* __restrict__ n_arr, const long* __restrict__ a_off,
                          const long* __restrict__ x_off, const int* __restrict__ order,
                          const double* __restrict__ A, float* __restrict__ LU,
                          double* __restrict__ rs, double* __restrict__ cs,
                          int* __restrict__ piv, int* __restrict__ perm, int* __restrict__ info) {
  __shared__ float sL[kPw * kLuNmax];   // panel, column c at c * 256 + local row
  __shared__ float sU[kPw * kLuNmax];   // U12, row q at q * 256 + (col - c0 - 32)
  __shared__ double scl_r[kLuNmax], scl_c[kLuNmax];
  __shared__ float red_v[kMfThreads / 64];
  __shared__ int red_i[kMfThreads / 64];
  __shared__ int sh_piv[kPw];
  __shared__ int sh_perm[kLuNmax];
  __shared__ int sh_info;

  const int t = threadIdx.x;
  const int lane = t & 63, wave = t >> 6;

  for (int w = blockIdx.x; w < nb; w += gridDim.x) {
    const int b = order ? order[w] : w;
    const int n = n_arr[b];
    if (n < 1 || n > kLuNmax) {  // uniform per block
      if (t == 0) info[b] = -1;
      continue;
    }
    const int npad = (n + kPw - 1) / kPw * kPw;
    const double* __restrict__ Ab = A + a_off[b];
    float* __restrict__ Lb = LU + a_off[b];
    const long xo = x_off[b];
    __syncthreads();  // LDS reuse across blocks

    // ---- power-of-two equilibration, scaled FP32 copy into Lb -------------
    sh_perm[t] = t;
    if (t == 0) sh_info = 0;
    if (t < n) {
      double mx = 0.0;
      for (int c = 0; c < n; ++c) mx = fmax(mx, fabs(Ab[t + (long)c * n]));
      scl_r[t] = pow2_scale(mx);
    }
    __syncthreads();
    if (t < n) {
      double mx = 0.0;
      const double* __restrict__ col = Ab + (long)t * n;
      for (int r = 0; r < n; ++r) mx = fmax(mx, fabs(col[r]) * scl_r[r]);
      scl_c[t] = pow2_scale(mx);
    }
    __syncthreads();
    if (t < n) {
      const double sr = scl_r[t];
      for (int c = 0; c < n; ++c)
        Lb[t + (long)c * n] = (float)(Ab[t + (long)c * n] * sr * scl_c[c]);
    }
    __syncthreads();

    for (int c0 = 0; c0 < npad; c0 += kPw) {
      const int m = npad - c0;  // panel rows, a multiple of 32, <= 256
      // ---- 1. panel into LDS (identity on the padding) --------------------
      {
        const int R = c0 + t;
        for (int c = 0; c < kPw; ++c) {
          const int C = c0 + c;
          float v = 0.f;
          if (t < m) v = (R < n && C < n) ? Lb[R + (long)C * n] : (R == C ? 1.f : 0.f);
          sL[c * kLuNmax + t] = v;
        }
      }
      __syncthreads();
      for (int j = 0; j < kPw; ++j) {
        // argmax |a(r, j)| over local rows j <= r < m, first maximum wins
        // (barrier B1 below also orders this step's swap after every thread's
        // last update of its own row; B2 orders the update after the swap)
        float best = (t >= j && t < m) ? fabsf(sL[j * kLuNmax + t]) : -1.f;
        int bi = t;
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
          const float ob = __shfl_xor(best, o, 64);
          const int oi = __shfl_xor(bi, o, 64);
          if (ob > best || (ob == best && oi < bi)) {
            best = ob;
            bi = oi;
          }
        }
        if (lane == 0) {
          red_v[wave] = best;
          red_i[wave] = bi;
        }
        __syncthreads();  // B1
        float pb = red_v[0];
        int p = red_i[0];
#pragma unroll
        for (int q = 1; q < kMfThreads / 64; ++q) {
          const float vq = red_v[q];
          if (vq > pb || (vq == pb && red_i[q] < p)) {
            pb = vq;
            p = red_i[q];
          }
        }
        if (!(pb >= 0.f) || p < j || p >= m) p = j;  // NaN column: keep the diagonal
        // row swap, threads 0..31 one panel column each
        if (t < kPw && p != j) {
          const float x = sL[t * kLuNmax + j];
          sL[t * kLuNmax + j] = sL[t * kLuNmax + p];
          sL[t * kLuNmax + p] = x;
        }
        if (t == 0) sh_piv[j] = p;
        __syncthreads();  // B2
        const float pivot = sL[j * kLuNmax + j];
        if (t == 0 && pivot == 0.f && sh_info == 0 && c0 + j < n) sh_info = c0 + j + 1;
        if (t > j && t < m) {
          const float inv = pivot != 0.f ? 1.f / pivot : 0.f;
          const float l = sL[j * kLuNmax + t] * inv;
          sL[j * kLuNmax + t] = l;
          for (int c = j + 1; c < kPw; ++c)
            sL[c * kLuNmax + t] = fmaf(-l, sL[c * kLuNmax + j], sL[c * kLuNmax + t]);
        }
      }
      __syncthreads();
      // panel back to the factor buffer; pivots and the row permutation
      {
        const int R = c0 + t;
        if (t < m && R < n)
          for (int c = 0; c < kPw && c0 + c < n; ++c) Lb[R + (long)(c0 + c) * n] = sL[c * kLuNmax + t];
      }
      if (t == 0) {
        for (int j = 0; j < kPw; ++j) {
          const int p = sh_piv[j];
          if (c0 + j < n) piv[xo + c0 + j] = c0 + p;
          const int tmp = sh_perm[c0 + j];
          sh_perm[c0 + j] = sh_perm[c0 + p];
          sh_perm[c0 + p] = tmp;
        }
      }
      // ---- 2. row swaps outside the panel, TRSM right of it ---------------
      if (t < npad && (t < c0 || t >= c0 + kPw)) {
        float* __restrict__ colp = Lb + (long)t * n;
        if (t < n) {
          for (int j = 0; j < kPw; ++j) {
            const int p = sh_piv[j];
            if (p != j && c0 + p < n) {
              const float x = colp[c0 + j];
              colp[c0 + j] = colp[c0 + p];
              colp[c0 + p] = x;
            }
          }
        }
        if (t >= c0 + kPw) {
          const int nv = min(kPw, n - c0);  // real rows of the panel (uniform, >= 1)
          const bool full = t < n && nv == kPw;
          float x[kPw];
          if (full) {
#pragma unroll
            for (int i = 0; i < kPw; ++i) x[i] = colp[c0 + i];
          } else {
            const bool live = t < n;
#pragma unroll
            for (int i = 0; i < kPw; ++i) x[i] = (live && i < nv) ? colp[c0 + i] : 0.f;
          }
          // column-oriented forward substitution with the unit-lower L11
#pragma unroll
          for (int q = 0; q < kPw - 1; ++q) {
            const float xq = x[q];
#pragma unroll
            for (int i = q + 1; i < kPw; ++i) x[i] = fmaf(-sL[q * kLuNmax + i], xq, x[i]);
          }
          const int cu = t - c0 - kPw;
#pragma unroll
          for (int i = 0; i < kPw; ++i) sU[i * kLuNmax + cu] = x[i];
          if (full) {
#pragma unroll
            for (int i = 0; i < kPw; ++i) colp[c0 + i] = x[i];
          } else if (t < n) {
#pragma unroll
            for (int i = 0; i < kPw; ++i)
              if (i < nv) colp[c0 + i] = x[i];
          }
        }
      }
      __syncthreads();
      // ---- 3. trailing update on MFMA ---------------------------------------
      const int nr = (npad - c0 - kPw) / kPw;  // trailing tiles per dimension
      for (int tile = wave; tile < nr * nr; tile += kMfThreads / 64) {
        const int ti = tile / nr, tj = tile % nr;
        const int R0 = c0 + kPw + kPw * ti, C0 = c0 + kPw + kPw * tj;
        const int h = lane >> 5, cl = lane & 31;
        const int C = C0 + cl;
        f32x16 acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int R = R0 + 8 * (r >> 2) + 4 * h + (r & 3);
          acc[r] = (R < n && C < n) ? Lb[R + (long)C * n] : 0.f;
        }
        // A (32 x 2 per step): lane holds L21(R0 + cl, 2s + h);
        // B (2 x 32 per step): lane holds U12(2s + h, C0 + cl)
        const float* __restrict__ la = sL + (R0 - c0) + cl;
        const float* __restrict__ ub = sU + (C0 - c0 - kPw) + cl;
#pragma unroll
        for (int s = 0; s < kPw / 2; ++s) {
          const int q = 2 * s + h;
          acc = __builtin_amdgcn_mfma_f32_32x32x2f32(-la[q * kLuNmax], ub[q * kLuNmax], acc, 0,
                                                     0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int R = R0 + 8 * (r >> 2) + 4 * h + (r & 3);
          if (R < n && C < n) Lb[R + (long)C * n] = acc[r];
        }
      }
      __syncthreads();
    }

    if (t < n) {
      perm[xo + t] = sh_perm[t];
      rs[xo + t] = scl_r[t];
      cs[xo + t] = scl_c[t];
    }
    if (t == 0) info[b] = sh_info;
  }
}

// ---------------------------------------------------------------------------
// Triangular solves, one wavefront per block, row 64 s + lane in slot s.  The
// rows go 64 at a time: while the columns of segment s are consumed, slot s
// ("cur") holds the unknowns, and the slots it still changes (NB of them)
// follow in order, so the pivot entry is always cur's (two readlanes into
// scalar registers), the slots are static registers, and the slots a
// triangle excludes are neither loaded nor multiplied.  Within the diagonal
// slot, lanes outside the triangle read the chunk's first (last) row, a line
// that is needed anyway.  A sweep therefore reads n^2 / 2 entries plus the
// chunks' steps at the diagonal, where the former version read all n^2 and
// searched the pivot among four slots for each column (24 VALU + 21 SALU
// instructions per column against 6 + NB).  Columns come in chunks in
// two register sets that trade roles: one loads while the other is used.
// Measured: 2048 fiber blocks of order 64-256 in FP64 215 -> 123 us (452 MB of
// factor: 3.7 TB/s of the copy's 5.1); 1000 blocks of order 128 in FP32 without
// refinement 56 us (factor staged in LDS) and 80 (streamed) -> 22; 32 blocks
// of order 128 in FP64, where the chain alone counts, 53 -> 17.
constexpr int kSlots = 4;
// Columns of a chunk of NS slots: 16 loads of 64 rows in flight per wave.
__host__ __device__ constexpr int chunk_cols(int NS) { return NS == 1 ? 16 : (NS == 2 ? 8 : 4); }

// Columns k0, k0 + step, ... (a chunk, clamped into the block) of a
// column-major block, at the byte offsets of NS rows.
template <typename T, int NS>
__device__ __forceinline__ void load_cols(const T* __restrict__ M, int n, int k0, int step,
                                          const unsigned (&off)[NS], T (&r)[chunk_cols(NS)][NS]) {
#pragma unroll
  for (int u = 0; u < chunk_cols(NS); ++u) {
    int k = k0 + u * step;
    k = k < 0 ? 0 : (k > n - 1 ? n - 1 : k);
    const char* __restrict__ col = reinterpret_cast<const char*>(M + k * n);
#pragma unroll
    for (int m = 0; m < NS; ++m) r[u][m] = *reinterpret_cast<const T*>(col + off[m]);
  }
}

// use(tail, j0, set) for the chunks of cnt columns, load(j0, set) one chunk
// ahead.  The chunk index passes through an empty asm placed after the loads:
// the chunk's work depends on it, so the compiler can neither sink the loads
// to their uses nor hoist the uses to the loads; and the next loads come after
// an asm that takes the work's result (state), so they reuse the set's
// registers instead of a third set.
template <typename T, int NS, typename Load, typename Use>
__device__ __forceinline__ void stream_chunks(int cnt, double& state, Load&& load, Use&& use) {
  constexpr int kCh = chunk_cols(NS);
  T ra[kCh][NS], rb[kCh][NS];
  load(0, ra);
  int j0 = 0;
  for (; j0 + 2 * kCh <= cnt; j0 += 2 * kCh) {
    load(j0 + kCh, rb);
    int ja = j0;
    asm volatile("" : "+s"(ja) : : "memory");
    use(std::false_type{}, ja, ra);
    asm volatile("" : "+v"(state) : : "memory");
    if (j0 + 2 * kCh < cnt) load(j0 + 2 * kCh, ra);
    int jb = j0 + kCh;
    asm volatile("" : "+s"(jb) : : "memory");
    use(std::false_type{}, jb, rb);
    asm volatile("" : "+v"(state) : : "memory");
  }
  if (j0 < cnt) {
    if (j0 + kCh < cnt) load(j0 + kCh, rb);
    use(std::true_type{}, j0, ra);
    if (j0 + kCh < cnt) use(std::true_type{}, j0 + kCh, rb);
  }
}

// w_i -= L(i, k) w_k, i > k, for the columns k = k0 .. of cur's segment.
template <typename T, int NB>
__device__ __forceinline__ void forward_segment(const T* __restrict__ L, int n, int k0, int lane,
                                                double& cur, double (&next)[kSlots - 1]) {
  const int cnt = min(64, n - k0);
  unsigned off[NB + 1];
#pragma unroll
  for (int m = 1; m <= NB; ++m) off[m] = (unsigned)min(k0 + 64 * m + lane, n - 1) * (unsigned)sizeof(T);
  stream_chunks<T, NB + 1>(
      cnt, cur,
      [&](int j0, T (&r)[chunk_cols(NB + 1)][NB + 1]) __attribute__((always_inline)) {
        off[0] = (unsigned)min(k0 + max(lane, j0), n - 1) * (unsigned)sizeof(T);
        load_cols<T, NB + 1>(L, n, k0 + j0, 1, off, r);
      },
      [&](auto tail, int j0, const T (&r)[chunk_cols(NB + 1)][NB + 1]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < chunk_cols(NB + 1); ++u) {
          const int j = j0 + u;
          if (decltype(tail)::value && j >= cnt) break;
          const double wk = readlane_f64(cur, j);
          cur = lane > j ? fma(-(double)r[u][0], wk, cur) : cur;
#pragma unroll
          for (int m = 1; m <= NB; ++m) next[m - 1] = fma(-(double)r[u][m], wk, next[m - 1]);
        }
      });
}

// backward_segment where a pivot of the segment is zero, infinite, NaN or outside
// 2^-400 .. 2^400: a division per column, one column at a time, for any number
// of slots above.
template <typename T>
__device__ __forceinline__ void backward_segment_divide(const T* __restrict__ U, int n, int k0,
                                                        int lane, double& cur,
                                                        double (&next)[kSlots - 1]) {
#pragma unroll 1
  for (int j = min(64, n - k0) - 1; j >= 0; --j) {
    const T* __restrict__ col = U + (long)(k0 + j) * n;
    const double u = (double)col[k0 + min(lane, j)];
    const double wk = readlane_f64(cur, j) / readlane_f64(u, j);
    cur = lane == j ? wk : (lane < j ? fma(-u, wk, cur) : cur);
#pragma unroll
    for (int m = 1; m < kSlots; ++m)
      if (64 * m <= k0) next[m - 1] = fma(-(double)col[k0 - 64 * m + lane], wk, next[m - 1]);
  }
}

// w_k /= U(k, k); w_i -= U(i, k) w_k, i < k, for the columns of cur's segment
// from the last to k0; next[m - 1]: slot m above.  Every row's quotient comes
// from its reciprocal r = 1 / U(i, i), three operations on the chain where a
// division takes about twelve: q = w r, then q + r (w - q U), the correctly
// rounded quotient while nothing over- or underflows (Markstein); a q that is
// not finite stays as it is.  Returns whether the segment has a pivot outside
// 2^-400 .. 2^400, whose reciprocal may do either: its results are to be dropped.
// (The answer comes after the columns, not before them: asked before, a solve of
// 1000 blocks of order 128 waits for the diagonal, 22.6 -> 23.0 us.)
template <typename T, int NB>
__device__ __forceinline__ bool backward_segment(const T* __restrict__ U, int n, int k0, int lane,
                                                 double& cur, double (&next)[kSlots - 1]) {
  const int cnt = min(64, n - k0);
  const double dg = (double)U[(long)min(k0 + lane, n - 1) * (n + 1)];
  unsigned off[NB + 1];
#pragma unroll
  for (int m = 1; m <= NB; ++m) off[m] = (unsigned)(k0 - 64 * m + lane) * (unsigned)sizeof(T);
  const double rc = 1.0 / dg;
  stream_chunks<T, NB + 1>(
      cnt, cur,
      [&](int j0, T (&r)[chunk_cols(NB + 1)][NB + 1]) __attribute__((always_inline)) {
        off[0] = (unsigned)(k0 + min(lane, cnt - 1 - j0)) * (unsigned)sizeof(T);
        load_cols<T, NB + 1>(U, n, k0 + cnt - 1 - j0, -1, off, r);
      },
      [&](auto tail, int j0, const T (&r)[chunk_cols(NB + 1)][NB + 1]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < chunk_cols(NB + 1); ++u) {
          if (decltype(tail)::value && j0 + u >= cnt) break;
          const int j = cnt - 1 - (j0 + u);
          const double q = cur * rc;
          const double t = fma(fma(-q, dg, cur), rc, q);
          const double wk = readlane_f64(isfinite(q) ? t : q, j);
          cur = lane == j ? wk : (lane < j ? fma(-(double)r[u][0], wk, cur) : cur);
#pragma unroll
          for (int m = 1; m <= NB; ++m) next[m - 1] = fma(-(double)r[u][m], wk, next[m - 1]);
        }
      });
  return __ballot(!(fabs(dg) > 0x1p-400 && fabs(dg) < 0x1p400)) != 0ull;
}

// w <- U^-1 L^-1 w (the factor's L unit lower, U upper, column-major), FP64
// arithmetic; sw: 256 doubles of LDS, each lane its own.
template <typename T>
__device__ __forceinline__ void trsv_lu(const T* __restrict__ L, int n, int lane,
                                        double (&w)[kSlots], double* __restrict__ sw) {
  const int ns = (n + 63) >> 6;
  double cur = w[0], next[kSlots - 1] = {w[1], w[2], w[3]};
  for (int s = 0; s < ns; ++s) {
    const int nb = ns - 1 - s;
    if (nb == 3) forward_segment<T, 3>(L, n, 64 * s, lane, cur, next);
    else if (nb == 2) forward_segment<T, 2>(L, n, 64 * s, lane, cur, next);
    else if (nb == 1) forward_segment<T, 1>(L, n, 64 * s, lane, cur, next);
    else forward_segment<T, 0>(L, n, 64 * s, lane, cur, next);
    sw[64 * s + lane] = cur;
    cur = next[0];
    next[0] = next[1];
    next[1] = next[2];
  }
  cur = sw[64 * (ns - 1) + lane];
#pragma unroll
  for (int m = 0; m < kSlots - 1; ++m) next[m] = sw[64 * max(ns - 2 - m, 0) + lane];
  for (int s = ns - 1; s >= 0; --s) {
    const double cur0 = cur, next0[kSlots - 1] = {next[0], next[1], next[2]};
    bool wide;
    if (s == 3) wide = backward_segment<T, 3>(L, n, 64 * s, lane, cur, next);
    else if (s == 2) wide = backward_segment<T, 2>(L, n, 64 * s, lane, cur, next);
    else if (s == 1) wide = backward_segment<T, 1>(L, n, 64 * s, lane, cur, next);
    else wide = backward_segment<T, 0>(L, n, 64 * s, lane, cur, next);
    if (wide) {
      cur = cur0;
#pragma unroll
      for (int m = 0; m < kSlots - 1; ++m) next[m] = next0[m];
      backward_segment_divide<T>(L, n, 64 * s, lane, cur, next);
    }
    sw[64 * s + lane] = cur;
    cur = next[0];
    next[0] = next[1];
    next[1] = next[2];
  }
#pragma unroll
  for (int m = 0; m < kSlots; ++m) w[m] = sw[64 * m + lane];
}

// r -= A y over NS slots, and the rows' sums of |A|; y in LDS.
template <int NS>
__device__ __forceinline__ void residual(const double* __restrict__ A, int n, int lane,
                                         const double* __restrict__ sy, double (&r)[kSlots],
                                         double (&rowabs)[kSlots]) {
  unsigned off[NS];
#pragma unroll
  for (int m = 0; m < NS; ++m) off[m] = (unsigned)min(64 * m + lane, n - 1) * 8u;
  for (int k0 = 0; k0 < n; k0 += 64) {
    const int cnt = min(64, n - k0);
    const double y = sy[k0 + lane];
    stream_chunks<double, NS>(
        cnt, r[0],
        [&](int j0, double (&c)[chunk_cols(NS)][NS]) __attribute__((always_inline)) {
          load_cols<double, NS>(A, n, k0 + j0, 1, off, c);
        },
        [&](auto tail, int j0, const double (&c)[chunk_cols(NS)][NS]) __attribute__((always_inline)) {
#pragma unroll
          for (int u = 0; u < chunk_cols(NS); ++u) {
            if (decltype(tail)::value && j0 + u >= cnt) break;
            const double yj = readlane_f64(y, j0 + u);
#pragma unroll
            for (int m = 0; m < NS; ++m) {
              r[m] = fma(-c[u][m], yj, r[m]);
              rowabs[m] += fabs(c[u][m]);
            }
          }
        });
  }
}

// REFINE false (no refinement asked for) leaves the residual's registers out:
// two waves per SIMD instead of one.
template <typename T, bool REFINE>
__global__ void __launch_bounds__(64, REFINE ? 1 : 2)
lu_solve_kernel(const int* __restrict__ n_arr, const long* __restrict__ a_off,
                const long* __restrict__ x_off, const double* __restrict__ A,
                const T* __restrict__ LU, const double* __restrict__ rs,
                const double* __restrict__ cs, const int* __restrict__ perm,
                const double* x, double* y, int refine, double tol, int* __restrict__ iters) {
  __shared__ double sw[64 * kSlots];
  const int b = blockIdx.x;
  const int lane = threadIdx.x;
  const int n = n_arr[b];
  if (n < 1 || n > 64 * kSlots) {
    if (iters && lane == 0) iters[b] = -1;
    return;
  }
  const long xo = x_off[b];
  const T* __restrict__ L = LU + a_off[b];
  const int* __restrict__ pm = perm + xo;

  // w = P (rs .* x): row i of the factor is row perm[i] of A.
  int src[kSlots];
  double w[kSlots], yv[kSlots], xv[kSlots], csv[kSlots];
#pragma unroll
  for (int m = 0; m < kSlots; ++m) {
    const int i = 64 * m + lane;
    src[m] = i < n ? min(max(pm[i], 0), n - 1) : 0;
    w[m] = i < n ? x[xo + src[m]] * (rs ? rs[xo + src[m]] : 1.0) : 0.0;
    xv[m] = REFINE && i < n ? x[xo + i] : 0.0;
    csv[m] = (cs && i < n) ? cs[xo + i] : 1.0;
  }
  int it = 0;
  double anorm = -1.0;
  double rprev = 0.0;
  for (bool first = true;; first = false) {
    trsv_lu<T>(L, n, lane, w, sw);
#pragma unroll
    for (int m = 0; m < kSlots; ++m) yv[m] = first ? w[m] * csv[m] : yv[m] + w[m] * csv[m];
    if (!first) ++it;
    if (!REFINE || it >= refine) break;
    // r = x - A y in FP64, and ||A||_inf
    const double* __restrict__ Ab = A + a_off[b];
    double r[kSlots], rowabs[kSlots];
#pragma unroll
    for (int m = 0; m < kSlots; ++m) {
      r[m] = xv[m];
      rowabs[m] = 0.0;
      sw[64 * m + lane] = yv[m];
    }
    if (n > 192) residual<4>(Ab, n, lane, sw, r, rowabs);
    else if (n > 128) residual<3>(Ab, n, lane, sw, r, rowabs);
    else if (n > 64) residual<2>(Ab, n, lane, sw, r, rowabs);
    else residual<1>(Ab, n, lane, sw, r, rowabs);
    double rn = 0.0, yn = 0.0, an = 0.0;
#pragma unroll
    for (int m = 0; m < kSlots; ++m) {
      if (64 * m + lane < n) {
        rn = fmax(rn, fabs(r[m]));
        yn = fmax(yn, fabs(yv[m]));
        an = fmax(an, rowabs[m]);
      }
    }
    rn = wave_max_f64(rn);
    yn = wave_max_f64(yn);
    if (anorm < 0.0) anorm = wave_max_f64(an);
    if (rn <= tol * anorm * yn) break;
    // stagnation: FP64 refinement stopped contracting the residual
    if (it > 0 && rn > 0.5 * rprev) break;
    rprev = rn;
    // dy = solve(r)
#pragma unroll
    for (int m = 0; m < kSlots; ++m) {
      const int i = 64 * m + lane;
      sw[i] = r[m] * ((rs && i < n) ? rs[xo + i] : 1.0);
    }
    __syncthreads();  // one wave: the rows are read across lanes
#pragma unroll
    for (int m = 0; m < kSlots; ++m) w[m] = 64 * m + lane < n ? sw[src[m]] : 0.0;
    __syncthreads();
  }
  if (iters && lane == 0) iters[b] = it;
#pragma unroll
  for (int m = 0; m < kSlots; ++m) {
    const int i = 64 * m + lane;
    if (i < n) y[xo + i] = yv[m];
  }
}

// ---------------------------------------------------------------------------
// y_b = sum over terms of alpha M_b x_b, plus beta y_b; M_b column-major m x k, m
// <= 64 kSlots: a workgroup of four waves per block, all terms in one launch
// (a fiber's rows of the operator have four: A and the three Q_c; in launches
// of their own these took 22 + 3 x 7.5 us for 1000 fibers of 32 nodes, here
// 40.9, and 6 + 3 x 4.6 us for 32 fibers, here 9.2).  A lane has row lane of each 64-row
// segment (R 64), or, for m <= 32, row lane % 32 of every other column (R 32).
// The waves take groups of 16 loads in turn; their sums meet in LDS in a fixed
// order, the same for every launch form (the force rows cancel by 1e6 and more, so
// another order moves a step's densities by up to 1e-8).
// Bound by the loads of M: by HBM where the blocks fill the chip, by the chain
// of one wave's column groups where they do not, which the four waves shorten.
// Measured, against one wave per block and four columns in flight: 1000 blocks
// of 128 x 128 21.9 us (6.0 TB/s) for 32, 3000 of 32 x 128 17.7 for 23, 32
// blocks of 128 x 128 6.1 us for 18, of 114 x 32 3.9 for 10.
// Many small blocks are bound by the waves' start instead: 4096 blocks of 50 x 16
// took 10.8 us with 16 loads in flight and the sums of four terms' groups in LDS, 8.2
// with 8 loads (57 registers for 116) and 2 KB; one wave a block 6.6, but then 64 x 64
// 23.1 for 21.7.
constexpr int kGemvThreads = 256;

// acc += alpha M x for the lane's rows from r0 on, over every fourth group of 16 /
// SL steps, from the group `part`
template <int R, int SL, int UL>
__device__ __forceinline__ void block_gemv_cols(const double* __restrict__ M,
                                                const double* __restrict__ x, int m, int kk,
                                                double alpha, int r0, int part, int lane,
                                                double (&acc)[SL]) {
  constexpr int C = 64 / R;    // columns side by side in a wave
  constexpr int G = 16 / SL;   // steps of a column group
  constexpr int U = UL / SL;   // steps whose loads are in flight together
  const int sub = R == 64 ? 0 : lane / R;
  int row[SL];
  double sum[SL];
#pragma unroll
  for (int s = 0; s < SL; ++s) {
    sum[s] = 0.0;
    row[s] = min(r0 + lane % R + 64 * s, m - 1);
  }
  for (int jg = part * (G * C); jg < kk; jg += 4 * G * C) {
#pragma unroll
    for (int q = 0; q < G / U; ++q) {
      const int j0 = jg + q * (U * C);
      if (q > 0 && j0 >= kk) break;
      double v[U][SL], xv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int j = j0 + u * C + sub, jc = min(j, kk - 1);
        xv[u] = x[jc];
#pragma unroll
        for (int s = 0; s < SL; ++s) v[u][s] = M[(long)jc * m + row[s]];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool in = j0 + u * C + sub < kk;  // past the end: adds nothing
#pragma unroll
        for (int s = 0; s < SL; ++s) sum[s] = in ? fma(v[u][s], xv[u], sum[s]) : sum[s];
      }
    }
  }
#pragma unroll
  for (int s = 0; s < SL; ++s)  // (a term may have fewer rows than the block)
    acc[s] = r0 + lane % R + 64 * s < m ? fma(alpha, sum[s], acc[s]) : acc[s];
}

struct GemvTerms {
  f3d_gemv_term t[F3D_GEMV_TERMS];
};

// SLM: 64-row segments of the tallest block that was announced (a taller one
// goes by pieces); UL: loads of a lane in flight; GM: groups of four waves, which
// take the terms in turn.
template <int SLM, int UL, int GM>
__global__ void __launch_bounds__(kGemvThreads * F3D_GEMV_TERMS)
block_gemv_kernel(int terms, const GemvTerms tt, const long* __restrict__ y_off,
                  double* __restrict__ y, double beta) {
  __shared__ double red[4 * GM][64 * SLM];
  const int b = blockIdx.x;
  const int t = threadIdx.x, lane = t & 63, groups = GM == 1 ? 1 : blockDim.x / kGemvThreads;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  int m = 0;  // rows of the block: of its tallest term
  for (int q = 0; q < terms; ++q) {
    const int mq = tt.t[q].m[b];
    if (mq > 64 * kSlots || tt.t[q].k[b] < 0) return;
    m = max(m, mq);
  }
  double* __restrict__ yb = y + y_off[b];
  using std::integral_constant;
  auto piece = [&](auto first) __attribute__((always_inline)) {
    const int r0 = first, mr = m - r0;
    auto sums = [&](auto R, auto SL) __attribute__((always_inline)) {
      double acc[SL.value];
#pragma unroll
      for (int s = 0; s < SL.value; ++s) acc[s] = 0.0;
#pragma unroll 1
      for (int q = wv / 4; q < terms; q += groups) {
        const f3d_gemv_term& g = tt.t[q];
        const int mq = g.m[b];
        if (mq > r0)
          block_gemv_cols<R.value, SL.value, UL>(g.M + g.m_off[b], g.x + g.x_off[b], mq, g.k[b],
                                                 g.alpha, r0, wv % 4, lane, acc);
      }
      if (R.value == 32) acc[0] += __shfl_xor(acc[0], 32, 64);
#pragma unroll
      for (int s = 0; s < SL.value; ++s) red[wv][64 * s + lane] = acc[s];
    };
    if (m <= 32) sums(integral_constant<int, 32>{}, integral_constant<int, 1>{});
    else if (SLM == 1 || mr <= 64) sums(integral_constant<int, 64>{}, integral_constant<int, 1>{});
    else if (mr <= 128) sums(integral_constant<int, 64>{}, integral_constant<int, SLM == 1 ? 1 : 2>{});
    else sums(integral_constant<int, 64>{}, integral_constant<int, SLM>{});
    __syncthreads();
    if (t < min(mr, 64 * SLM)) {
      double v = (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]);
      for (int g = 1; g < groups; ++g)
        v += (red[4 * g][t] + red[4 * g + 1][t]) + (red[4 * g + 2][t] + red[4 * g + 3][t]);
      yb[r0 + t] = beta == 0.0 ? v : fma(beta, yb[r0 + t], v);
    }
    if (SLM < kSlots) __syncthreads();  // (after the last piece too: faster code)
  };
  if constexpr (SLM == kSlots) {
    if (m > 0) piece(integral_constant<int, 0>{});
  } else {
    for (int r0 = 0; r0 < m; r0 += 64 * SLM) piece(r0);
  }
}

// ---------------------------------------------------------------------------
// y_b = M_b x_b for `count` dense ROW-major m x m matrices (FP64, or FP32
// entries with FP64 products and sums).  One wave computes kGemvRows rows of
// one matrix (fewer at the matrix's end), four waves per 256-thread
// workgroup: each 16-byte piece of x it loads serves all its rows, which
// keeps the x reads (from L2) at a quarter of the matrix bytes.  A wave reads
// each row in 1 KB coalesced steps (16 bytes per lane when `vec` is set: m a
// multiple of 16 / sizeof(TM), M and x 16-byte aligned), accumulates each row
// in two FP64 chains and reduces across the wave in a fixed order, so the
// result is deterministic.  Even one matrix of a few thousand rows puts
// thousands of waves in flight, which an HBM-bound sweep over a large inverse
// needs; the column-major GEMV above runs one workgroup per block.
constexpr int kGemvRows = 4;

__device__ __forceinline__ void gemv_fma16(const double2 a, const double2* __restrict__ v,
                                           double& acc0, double& acc1) {
  acc0 = fma(a.x, v[0].x, acc0);
  acc1 = fma(a.y, v[0].y, acc1);
}

__device__ __forceinline__ void gemv_fma16(const float4 a, const double2* __restrict__ v,
                                           double& acc0, double& acc1) {
  acc0 = fma((double)a.x, v[0].x, acc0);
  acc1 = fma((double)a.y, v[0].y, acc1);
  acc0 = fma((double)a.z, v[1].x, acc0);
  acc1 = fma((double)a.w, v[1].y, acc1);
}

template <typename TM> struct Gemv16;
template <> struct Gemv16<double> { using V = double2; };
template <> struct Gemv16<float> { using V = float4; };

template <typename TM>
__global__ void __launch_bounds__(256)
dense_gemv_kernel(int64_t waves_total, int32_t m, int32_t groups, int vec,
                  const TM* __restrict__ M, const double* __restrict__ x,
                  double* __restrict__ y) {
  constexpr int R = kGemvRows;
  const int lane = threadIdx.x & 63;
  const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= waves_total) return;
  const int64_t b = w / groups;
  const int r0 = (int)(w - b * groups) * R;
  const int nr = min(R, m - r0);
  const double* __restrict__ xb = x + b * (int64_t)m;
  // rows past the matrix's end repeat its last row (loaded again from
  // cache, never stored)
  const TM* __restrict__ Mr[R];
#pragma unroll
  for (int r = 0; r < R; ++r) Mr[r] = M + (b * (int64_t)m + r0 + min(r, nr - 1)) * (int64_t)m;
  double acc0[R], acc1[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc0[r] = acc1[r] = 0.0;
  if (vec) {
    using V = typename Gemv16<TM>::V;
    constexpr int per = (int)(16 / sizeof(TM));  // matrix entries per 16 bytes
    constexpr int xv = per / 2;                  // double2 of x per 16 bytes of M
    const int nv = m / per;
    const double2* __restrict__ x2 = reinterpret_cast<const double2*>(xb);
    int p = lane;
    for (; p + 64 < nv; p += 128) {
      V a[R][2];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        a[r][0] = reinterpret_cast<const V*>(Mr[r])[p];
        a[r][1] = reinterpret_cast<const V*>(Mr[r])[p + 64];
      }
      double2 v0[xv], v1[xv];
#pragma unroll
      for (int q = 0; q < xv; ++q) {
        v0[q] = x2[p * xv + q];
        v1[q] = x2[(p + 64) * xv + q];
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        gemv_fma16(a[r][0], v0, acc0[r], acc1[r]);
        gemv_fma16(a[r][1], v1, acc0[r], acc1[r]);
      }
    }
    for (; p < nv; p += 64) {
      double2 v0[xv];
#pragma unroll
      for (int q = 0; q < xv; ++q) v0[q] = x2[p * xv + q];
#pragma unroll
      for (int r = 0; r < R; ++r)
        gemv_fma16(reinterpret_cast<const V*>(Mr[r])[p], v0, acc0[r], acc1[r]);
    }
  } else {
    for (int j = lane; j < m; j += 64) {
      const double xj = xb[j];
#pragma unroll
      for (int r = 0; r < R; ++r) acc0[r] = fma((double)Mr[r][j], xj, acc0[r]);
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const double sum = wave_sum_f64(acc0[r] + acc1[r]);
    if (lane == 0 && r < nr) y[b * (int64_t)m + r0 + r] = sum;
  }
}

int launch_lu_block(int precision, int64_t nb, int32_t nmax, const int32_t* n, const int64_t* a_off,
                    const int64_t* x_off, const int32_t* order, const double* A, double* lu64,
                    float* lu32, double* rs, double* cs, int32_t* piv, int32_t* perm,
                    int32_t* info, hipStream_t st);

}  // namespace f3d

using namespace f3d;

extern "C" int f3d_lu_factor_batched(int precision, int64_t nb, int32_t nmax, const int32_t* n,
                                     const int64_t* a_off, const int64_t* x_off,
                                     const int32_t* order, const double* A, double* lu64,
                                     float* lu32, double* rs, double* cs, int32_t* piv,
                                     int32_t* perm, int32_t* info, void* stream) {
  F3D_REQUIRE(precision == F3D_F64 || precision == F3D_F32C, F3D_EINVAL,
              "lu_factor: unknown precision %d", precision);
  F3D_REQUIRE(nb >= 0 && nb < (1ll << 31), F3D_EINVAL, "lu_factor: bad batch count");
  F3D_REQUIRE(nmax >= 1 && nmax <= kLuNmax, F3D_EINVAL, "lu_factor: nmax=%d outside [1,%d]",
              nmax, kLuNmax);
  if (nb == 0) return F3D_OK;
  F3D_REQUIRE(n && a_off && x_off && A && piv && perm && info, F3D_EINVAL,
              "lu_factor: NULL argument");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // default: one workgroup per block, left-looking strips in LDS, MFMA updates
  // (lu_block.hip); F3D_LU_KERNEL=workgroup selects the one-workgroup-per-block
  // kernels above (FP32: F3D_LU32_KERNEL=vector for the unblocked one)
  const char* sel_k = getenv("F3D_LU_KERNEL");
  if (!(sel_k && strcmp(sel_k, "workgroup") == 0)) {
    if (precision == F3D_F64) {
      F3D_REQUIRE(lu64 != nullptr, F3D_EINVAL, "lu_factor: lu64 is NULL");
    } else {
      F3D_REQUIRE(lu32 && rs && cs, F3D_EINVAL, "lu_factor: lu32/rs/cs is NULL");
    }
    return launch_lu_block(precision, nb, nmax, n, a_off, x_off, order, A, lu64, lu32, rs, cs, piv,
                           perm, info, st);
  }
  const unsigned grid = (unsigned)(nb < num_cus() ? nb : num_cus());
  if (precision == F3D_F64) {
    F3D_REQUIRE(lu64 != nullptr, F3D_EINVAL, "lu_factor: lu64 is NULL");
    F3D_LAUNCH((lu_factor_kernel<double, 2>), dim3(grid), dim3(1024), 0, st, (int)nb, n,
               (const long*)a_off, (const long*)x_off, order, A, lu64, (double*)nullptr,
               (double*)nullptr, piv, perm, info, 0);
  } else {
    F3D_REQUIRE(lu32 && rs && cs, F3D_EINVAL, "lu_factor: lu32/rs/cs is NULL");
    // F3D_LU32_KERNEL=vector selects the register-resident VALU factorisation
    const char* sel = getenv("F3D_LU32_KERNEL");
    if (sel && strcmp(sel, "vector") == 0) {
      F3D_LAUNCH((lu_factor_kernel<float, 0>), dim3(grid), dim3(1024), 0, st, (int)nb, n,
                 (const long*)a_off, (const long*)x_off, order, A, lu32, rs, cs, piv, perm, info,
                 1);
    } else {
      const long g2 = 2l * num_cus();
      const unsigned grid2 = (unsigned)(nb < g2 ? nb : g2);
      F3D_LAUNCH(lu_factor_f32_mfma_kernel, dim3(grid2), dim3(kMfThreads), 0, st, (int)nb, n,
                 (const long*)a_off, (const long*)x_off, order, A, lu32, rs, cs, piv, perm,
                 info);
    }
  }
  return F3D_OK;
}

extern "C" int f3d_lu_solve_batched(int precision, int64_t nb, int32_t nmax, const int32_t* n,
                                    const int64_t* a_off, const int64_t* x_off, const double* A,
                                    const double* lu64, const float* lu32, const double* rs,
                                    const double* cs, const int32_t* perm, const double* x,
                                    double* y, int32_t refine, double tol, int32_t* iters,
                                    void* stream) {
  F3D_REQUIRE(precision == F3D_F64 || precision == F3D_F32C, F3D_EINVAL,
              "lu_solve: unknown precision %d", precision);
  F3D_REQUIRE(nb >= 0 && nb < (1ll << 31), F3D_EINVAL, "lu_solve: bad batch count");
  F3D_REQUIRE(nmax >= 1 && nmax <= 64 * kSlots, F3D_EINVAL, "lu_solve: nmax=%d outside [1,%d]",
              nmax, 64 * kSlots);
  F3D_REQUIRE(refine >= 0, F3D_EINVAL, "lu_solve: negative refine");
  if (nb == 0) return F3D_OK;
  F3D_REQUIRE(n && a_off && x_off && perm && x && y, F3D_EINVAL, "lu_solve: NULL argument");
  F3D_REQUIRE(refine == 0 || A != nullptr, F3D_EINVAL, "lu_solve: refinement needs A");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (precision == F3D_F64) {
    F3D_REQUIRE(lu64 != nullptr, F3D_EINVAL, "lu_solve: lu64 is NULL");
    if (refine > 0)
      F3D_LAUNCH((lu_solve_kernel<double, true>), dim3((unsigned)nb), dim3(64), 0, st, n,
                 (const long*)a_off, (const long*)x_off, A, lu64, rs, cs, perm, x, y, refine, tol,
                 iters);
    else
      F3D_LAUNCH((lu_solve_kernel<double, false>), dim3((unsigned)nb), dim3(64), 0, st, n,
                 (const long*)a_off, (const long*)x_off, A, lu64, rs, cs, perm, x, y, refine, tol,
                 iters);
  } else {
    F3D_REQUIRE(lu32 && rs && cs, F3D_EINVAL, "lu_solve: lu32/rs/cs is NULL");
    if (refine > 0)
      F3D_LAUNCH((lu_solve_kernel<float, true>), dim3((unsigned)nb), dim3(64), 0, st, n,
                 (const long*)a_off, (const long*)x_off, A, lu32, rs, cs, perm, x, y, refine, tol,
                 iters);
    else
      F3D_LAUNCH((lu_solve_kernel<float, false>), dim3((unsigned)nb), dim3(64), 0, st, n,
                 (const long*)a_off, (const long*)x_off, A, lu32, rs, cs, perm, x, y, refine, tol,
                 iters);
  }
  return F3D_OK;
}

extern "C" int f3d_lu_set_launch(int precision, int32_t factor_waves_per_cu,
                                 int32_t solve_staged) {
  F3D_REQUIRE(precision == F3D_F64 || precision == F3D_F32C, F3D_EINVAL,
              "lu_set_launch: unknown precision %d", precision);
  const int cap = precision == F3D_F64 ? 4 : 8;
  F3D_REQUIRE(factor_waves_per_cu >= 0 && factor_waves_per_cu <= cap, F3D_EINVAL,
              "lu_set_launch: waves per CU %d outside [0, %d]", factor_waves_per_cu, cap);
  F3D_REQUIRE(solve_staged == 0 || solve_staged == 1, F3D_EINVAL,
              "lu_set_launch: solve_staged must be 0 or 1");
  return F3D_OK;
}

template <typename TM>
static int dense_gemv_launch(int64_t count, int32_t m, const TM* M, const double* x, double* y,
                             void* stream) {
  F3D_REQUIRE(count >= 0 && m >= 0, F3D_EINVAL, "dense_gemv: count=%lld m=%d",
              (long long)count, m);
  if (count == 0 || m == 0) return F3D_OK;
  F3D_REQUIRE(M && x && y, F3D_EINVAL, "dense_gemv: NULL argument");
  const int32_t groups = (m + kGemvRows - 1) / kGemvRows;
  const int64_t waves = count * (int64_t)groups;
  F3D_REQUIRE((waves + 3) / 4 < (1ll << 31), F3D_EINVAL, "dense_gemv: %lld x %d rows",
              (long long)count, m);
  const int per = (int)(16 / sizeof(TM));
  const int vec = (m % per == 0) && (((uintptr_t)M | (uintptr_t)x) % 16 == 0);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  F3D_LAUNCH((dense_gemv_kernel<TM>), dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st,
             waves, m, groups, vec, M, x, y);
  return F3D_OK;
}

extern "C" int f3d_dense_gemv_batched(int64_t count, int32_t m, const double* M,
                                      const double* x, double* y, void* stream) {
  return dense_gemv_launch<double>(count, m, M, x, y, stream);
}

extern "C" int f3d_dense_gemv_batched_f32(int64_t count, int32_t m, const float* M,
                                          const double* x, double* y, void* stream) {
  return dense_gemv_launch<float>(count, m, M, x, y, stream);
}

extern "C" int f3d_block_gemv_batched(int64_t nb, int32_t mmax, const int32_t* m,
                                      const int32_t* k, const int64_t* m_off,
                                      const int64_t* x_off, const int64_t* y_off,
                                      const double* M, const double* x, double* y, double alpha,
                                      double beta, void* stream) {
  const f3d_gemv_term term{m, k, m_off, x_off, M, x, alpha};
  return f3d_block_gemv_sum(nb, mmax, 1, &term, y_off, y, beta, stream);
}

extern "C" int f3d_block_gemv_sum(int64_t nb, int32_t mmax, int32_t terms,
                                  const f3d_gemv_term* term, const int64_t* y_off, double* y,
                                  double beta, void* stream) {
  F3D_REQUIRE(nb >= 0 && nb < (1ll << 31), F3D_EINVAL, "block_gemv: bad batch count");
  F3D_REQUIRE(mmax >= 1 && mmax <= 64 * kSlots, F3D_EINVAL,
              "block_gemv: mmax=%d outside [1,%d]", mmax, 64 * kSlots);
  F3D_REQUIRE(terms >= 1 && terms <= F3D_GEMV_TERMS && term, F3D_EINVAL,
              "block_gemv: %d terms outside [1,%d]", terms, F3D_GEMV_TERMS);
  if (nb == 0) return F3D_OK;
  F3D_REQUIRE(y && y_off, F3D_EINVAL, "block_gemv: NULL argument");
  GemvTerms tt{};
  for (int q = 0; q < terms; ++q) {
    const f3d_gemv_term& g = term[q];
    F3D_REQUIRE(g.m && g.k && g.m_off && g.x_off && g.M && g.x, F3D_EINVAL,
                "block_gemv: NULL argument");
    tt.t[q] = g;
  }
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
#define F3D_GV(SLM, UL, GM, G)                                                            \
  F3D_LAUNCH((block_gemv_kernel<SLM, UL, GM>), dim3((unsigned)nb), dim3(kGemvThreads * (G)), 0, \
             st, terms, tt, (const long*)y_off, y, beta)
  // One product of blocks of at most 64 rows has 8 loads of a lane in flight, and so
  // have many blocks (8 per CU) of at most 128; us, for 16 loads: 6 x 16, 32 blocks 2.6
  // for 3.1, 4096 5.5, 10.6; 50 x 16, 32 3.0, 2.9, 4096 8.1, 10.7; 64 x 64, 1000 5.8, 5.8, 4096
  // 21.7, 23.3; 82 x 24, 4096 13.4, 17.0; 114 x 32, 4096 20.0, 22.0; but 114 x 128, 256 7.1,
  // 6.7.  (Sums of several terms have long ones among them.)
  if (terms == 1 && mmax <= 64) F3D_GV(1, 8, 1, 1);
  else if (terms == 1 && mmax <= 128 && nb >= 8 * (int64_t)num_cus()) F3D_GV(kSlots, 8, 1, 1);
  // Four waves a term where the blocks leave CUs idle (32 blocks: 9.2 us for 12.8 with
  // the terms one after the other); elsewhere four waves a block, since the
  // waves of short terms would only hold their places (1000 blocks: 40.9 us for 48.2).
  else F3D_GV(kSlots, 16, F3D_GEMV_TERMS, nb <= num_cus() ? terms : 1);
#undef F3D_GV
  return F3D_OK;
}

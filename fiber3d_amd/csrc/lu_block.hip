// Batched LU with partial pivoting, one workgroup per block, on MFMA.
//
// Reference: scipy.linalg.lu_factor per fiber (LAPACK dgetrf: partial
// pivoting, the first maximal |pivot| wins ties) in
// python/tstep/tstep_utils.py:1405-1419, applied at python/tstep/tstep.py:985-988.
//
// Design (gfx950, wave64).  Each block (order n <= 256) gets one workgroup of
// four waves and is factored left-looking in strips of W columns that stay in
// LDS: a strip is read once from A (its rows gathered through the permutation
// so far, so no working copy is made), brought up to date with the factor's
// earlier columns, factored, and written once.  A launch moves A, the factor
// and the earlier columns each strip reads again (n^3 / (6 W) entries); a
// right-looking form that keeps the trailing matrix in memory moves it once
// per 16 columns.
//   * Earlier columns, 16 at a time: U_k = L_kk^-1 A_k with one lane per row
//     and column group (x_i -= L(i, k) x_k, x_k broadcast within 16 lanes by
//     DPP: 15 steps), then every wave updates its row tiles below with
//     v_mfma_{f64,f32}_16x16x4 (computed transposed, E = D^T, so 16 lanes
//     hold 16 consecutive rows of a column; L from memory, the next 16
//     columns' loads in flight during this one's products).
//   * Panels of 16 columns within the strip, one thread per row: rows never
//     move, each carries its position under the row interchanges.  Per
//     column every wave finds its largest |a| (bits compared as integers on
//     DPP moves; ties go to the lowest position) and puts its candidate row
//     and its reciprocal in LDS; after ONE barrier every wave picks the best
//     of the four and every thread updates its row.  That chain, about 1000
//     cycles a column, bounds a lone block; blocks that share a CU overlap
//     theirs.  (The whole panel in one wave, four rows per lane and no
//     barrier, took longer: more instructions on the same chain.)
//   * Earlier columns of L keep the row order of their own strip's end while
//     the factorisation runs (a byte per row and strip maps positions), and
//     the few rows that later strips moved are put in place at the end.
// Every element sees the same operations in the same order as in an unblocked
// elimination with 16-column panels (FMA chains in a panel and in the
// triangular solves, four 4-deep MFMAs per 16 earlier columns), whatever the
// strip width and the number of waves.
// FP32 blocks are first equilibrated by powers of two (exact) per row and
// column; the solves refine in FP64 against the unscaled FP64 matrix.
// Orders that are not a multiple of 16 are padded with an identity block that
// is never stored: padded rows and columns stay decoupled from the real ones,
// so the real factors are exactly those of the unpadded matrix (the steps of
// padded columns are skipped).
#include "common.h"

#include <type_traits>

namespace f3d {

constexpr int kWp = 16;     // panel width = MFMA tile edge
constexpr int kWmax = 256;  // largest order

template <typename T>
struct Mf16;
// Operands: lane l provides A(l % 16, k = l / 16) and B(k = l / 16, l % 16).
// Output element e of lane l is D(row(l / 16, e), l % 16): the FP64
// instruction interleaves the rows (4 e + l / 16), the FP32 one keeps four
// consecutive rows per lane (4 (l / 16) + e).
template <>
struct Mf16<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ int row(int g, int e) { return 4 * e + g; }
  static __device__ __forceinline__ v4 mma(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mf16<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ int row(int g, int e) { return 4 * g + e; }
  static __device__ __forceinline__ v4 mma(float a, float b, v4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// Power of two s with s * amax in [0.5, 1); 1 for amax == 0 or non-finite.
// (From the exponent field; denormal and near-overflow maxima take frexp.)
__device__ __forceinline__ double pow2_scale_w(double amax) {
  const unsigned ex = (unsigned)((unsigned long long)__double_as_longlong(amax) >> 52);
  if (ex >= 1u && ex <= 2044u) return __longlong_as_double((long long)(2045u - ex) << 52);
  if (!(amax > 0.0) || !isfinite(amax)) return 1.0;
  int e;
  frexp(amax, &e);
  return ldexp(1.0, -e);
}

// Data-parallel-primitive lane moves (DPP): quad_perm xor 1 / xor 2,
// row_half_mirror and row_mirror; a butterfly of them leaves every lane of a
// 16-lane row holding the row's maximum.
template <int CTRL>
__device__ __forceinline__ unsigned dpp_mov(unsigned v) {
  return (unsigned)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v) {
  const unsigned long long u = __double_as_longlong(v);
  const unsigned lo = dpp_mov<CTRL>((unsigned)(u & 0xffffffffu));
  const unsigned hi = dpp_mov<CTRL>((unsigned)(u >> 32));
  return __longlong_as_double(((unsigned long long)hi << 32) | lo);
}
template <typename V>
__device__ __forceinline__ V row_max(V v) {
  V o;
  o = dpp_mov<0xB1>(v);   // quad_perm [1,0,3,2]
  v = o > v ? o : v;
  o = dpp_mov<0x4E>(v);   // quad_perm [2,3,0,1]
  v = o > v ? o : v;
  o = dpp_mov<0x141>(v);  // row_half_mirror
  v = o > v ? o : v;
  o = dpp_mov<0x140>(v);  // row_mirror
  v = o > v ? o : v;
  return v;
}
__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
  v = row_max(v);
  // the four rows: row 0 into 1 and 2 into 3, then row 1 into 2 and 3
  unsigned o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);
  v = max(v, o);
  o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false);
  v = max(v, o);
  return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}

// Compile-time loop: f(std::integral_constant<int, I>) for I in [B, E).
template <int B, int E, typename F>
__device__ __forceinline__ void sfor(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    sfor<B + 1, E>(f);
  }
}

// |v| as an integer that orders like |v|, plus one; 0 for NaN.  FP64: the
// high word here, the low word breaks its ties.
__device__ __forceinline__ unsigned abs_key(double v) {
  return v == v ? ((unsigned)((unsigned long long)__double_as_longlong(v) >> 32) & 0x7fffffffu) + 1u
                : 0u;
}
__device__ __forceinline__ unsigned abs_key(float v) {
  return v == v ? (__float_as_uint(v) & 0x7fffffffu) + 1u : 0u;
}
__device__ __forceinline__ unsigned low_key(double v) {
  return (unsigned)((unsigned long long)__double_as_longlong(v) & 0xffffffffu);
}
__device__ __forceinline__ unsigned low_key(float) { return 0u; }

// p[i], from a wave-uniform base and a 32-bit byte offset (one register
// instead of a 64-bit address; a block has at most 512 KB).
template <typename V>
__device__ __forceinline__ V ld(const V* __restrict__ p, int i) {
  return *reinterpret_cast<const V*>(reinterpret_cast<const char*>(p) + (unsigned)i * (unsigned)sizeof(V));
}
template <typename V>
__device__ __forceinline__ void st(V* __restrict__ p, int i, V v) {
  *reinterpret_cast<V*>(reinterpret_cast<char*>(p) + (unsigned)i * (unsigned)sizeof(V)) = v;
}

// Lane K's value of v in every 16-lane row.
template <int K>
__device__ __forceinline__ float row_bcast(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + K, 0xF, 0xF, true));
}
template <int K>
__device__ __forceinline__ double row_bcast(double v) {
  return dpp_mov<0x150 + K>(v);
}

// A wave's pivot candidate: the |a| key's high and low words, row | position
// << 16, and what the next column waits for (the reciprocal and the next
// entry), in one LDS read.
template <typename T>
struct alignas(16) LuCand {
  unsigned key, low;
  int at, pad;
  T inv, u1;
};

// For blocks of order up to NM.
template <typename T, int W, int NM>
struct LuShared {
  // LDS column stride of a strip: 16 columns x 4 rows (an MFMA operand) and 64
  // rows of a column both spread over all banks
  static constexpr int kWs = NM + 4;
  T s[W * kWs];                       // the strip, column c at c * kWs + row
  LuCand<T> cand[2][4];
  T crow[2][4][kWp];                  // the candidates' rows
  double srow[sizeof(T) == 4 ? NM : 1];     // FP32: row scales
  double scol[sizeof(T) == 4 ? kWp : 1];    // FP32: column scales of 16 columns
  unsigned char perm[NM];             // row of A now at a position
  unsigned char pos[NM];              // position of a row of the strip
  unsigned char piv[NM];              // interchange of every column
  unsigned char prow[kWp];            // the panel's pivot rows
  unsigned char pend[NM / W][NM];     // position of a row of A at a strip's end
};

// x <- L_kk^-1 x for R columns per lane: lane e16 of a 16-lane row holds row
// e16, l[k] = L_kk(e16, k).
template <typename T, int R>
__device__ __forceinline__ void unit_lower_solve(const T (&l)[kWp - 1], T (&x)[R], int e16) {
  sfor<0, kWp - 1>([&](auto K) __attribute__((always_inline)) {
    constexpr int k = decltype(K)::value;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const T v = fma(-l[k], row_bcast<k>(x[r]), x[r]);
      x[r] = e16 > k ? v : x[r];
    }
  });
}

__device__ __forceinline__ bool in_mask(unsigned long long m) {
  return __builtin_amdgcn_inverse_ballot_w64(m);
}

// Lane w's value of v, w wave-uniform.
__device__ __forceinline__ float rl(float v, int w) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), w));
}
__device__ __forceinline__ double rl(double v, int w) {
  const unsigned long long u = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(u & 0xffffffffu), w);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(u >> 32), w);
  return __longlong_as_double(((unsigned long long)hi << 32) | lo);
}

template <typename T, int W, int NM>
__device__ __forceinline__ void lu_block_body(LuShared<T, W, NM>& sh, const int* __restrict__ n_arr,
                                              const long* __restrict__ a_off,
                                              const long* __restrict__ x_off,
                                              const int* __restrict__ order,
                                              const double* __restrict__ A, T* __restrict__ LU,
                                              double* __restrict__ rs, double* __restrict__ cs,
                                              int* __restrict__ piv, int* __restrict__ perm,
                                              int* __restrict__ info) {
  typedef typename Mf16<T>::v4 v4;
  constexpr bool kEq = sizeof(T) == 4;  // FP32: equilibrate
  constexpr int kCt = W / kWp;          // column tiles
  constexpr int kWs = LuShared<T, W, NM>::kWs;
  const int tid = threadIdx.x, lane = tid & 63;
  const bool row = NM == kWmax || tid < NM;  // whether this thread has a row
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, e16 = lane & 15;
  const int b = order ? order[blockIdx.x] : (int)blockIdx.x;
  const int n = n_arr[b];
  if (n < 1 || n > NM) {  // uniform per workgroup
    if (tid == 0) info[b] = -1;
    return;
  }
  const int npad = (n + kWp - 1) / kWp * kWp;
  const int RT = npad / kWp;  // row tiles
  const double* __restrict__ Ab = A + a_off[b];
  T* __restrict__ M = LU + a_off[b];
  const long xo = x_off[b];
  int first_zero = 0;

  if (row) sh.perm[tid] = (unsigned char)tid;
  double sr = 1.0;
  if constexpr (kEq) {
    // row maxima, one thread per row
    double mx = 0.0;
    for (int c0 = 0; c0 < n; c0 += 16) {
      double v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = ld(Ab, min(tid, n - 1) + min(c0 + u, n - 1) * n);
#pragma unroll
      for (int u = 0; u < 16; ++u) mx = fmax(mx, fabs(v[u]));
    }
    sr = tid < n ? pow2_scale_w(mx) : 1.0;
    if (row) sh.srow[tid] = sr;
  }
  __syncthreads();

  for (int C0 = 0; C0 < npad; C0 += W) {
    const int ctn = min(kCt, (npad - C0) / kWp);  // column tiles of this strip
    const int phys = row ? sh.perm[tid] : tid;    // row of A of this thread's row
    // ---- the strip, rows in the order of the positions so far -------------------
    for (int h0 = 0; h0 < 16 * ctn; h0 += 16) {
      double v[16];
      const unsigned at = (unsigned)min(phys, n - 1) * 8u;
#pragma unroll
      for (int c = 0; c < 16; ++c)
        v[c] = *reinterpret_cast<const double*>(
            reinterpret_cast<const char*>(Ab + min(C0 + h0 + c, n - 1) * n) + at);
      T* __restrict__ dst = sh.s + h0 * kWs + tid;
      if constexpr (kEq) {
        // column maxima of the row-scaled matrix, by their high words (the
        // scale needs the exponent only); padded rows repeat a real row
        const double sp = sh.srow[min(phys, n - 1)];
        unsigned* __restrict__ hi = reinterpret_cast<unsigned*>(sh.s + h0 * kWs);
#pragma unroll
        for (int c = 0; c < 16; ++c) {
          v[c] *= sp;
          const unsigned h =
              (unsigned)((unsigned long long)__double_as_longlong(v[c]) >> 32) & 0x7fffffffu;
          if (row) hi[c * kWs + tid] = v[c] == v[c] ? h : 0u;
        }
        lds_barrier();
        const int c = tid >> 4, t0 = tid & 15;  // 16 threads per column
        unsigned h = 0u;
        for (int r = 4 * t0; r < npad; r += 64) {
          const uint4 q = *reinterpret_cast<const uint4*>(&hi[c * kWs + r]);
          h = max(h, max(max(q.x, q.y), max(q.z, q.w)));
        }
        h = row_max(h);
        if (t0 == 0) {
          double sc = 1.0;
          if (h >= 0x00100000u && h < 0x7ff00000u) {
            sc = pow2_scale_w(__longlong_as_double((long long)h << 32));
          } else if (C0 + h0 + c < n) {
            // zero, denormal or infinite: the maximum itself
            double mx = 0.0;
            for (int r = 0; r < n; ++r)
              mx = fmax(mx, fabs(Ab[r + (C0 + h0 + c) * n] * sh.srow[r]));
            sc = pow2_scale_w(mx);
          }
          sh.scol[c] = sc;
          if (C0 + h0 + c < n) cs[xo + C0 + h0 + c] = sc;
        }
        lds_barrier();
#pragma unroll
        for (int c = 0; c < 16; ++c)
          if (row) dst[c * kWs] = (T)(v[c] * sh.scol[kEq ? c : 0]);
      } else {
#pragma unroll
        for (int c = 0; c < 16; ++c)
          if (row) dst[c * kWs] = (T)v[c];
      }
      if (npad != n) {
        // the identity outside the real rows and columns
#pragma unroll
        for (int c = 0; c < 16; ++c) {
          const int C = C0 + h0 + c;
          if (row && (phys >= n || C >= n)) dst[c * kWs] = phys == C ? (T)1 : (T)0;
        }
      }
    }
    lds_barrier();

    // ---- earlier columns, 16 at a time -----------------------------------------
    if (C0 > 0) {
      T lk[kWp - 1];  // row e16 of L_kk
      auto load_kk = [&](int kb) __attribute__((always_inline)) {
        const unsigned ko = (unsigned)(16 * kb + e16) * (unsigned)sizeof(T);
#pragma unroll
        for (int k = 0; k < kWp - 1; ++k)
          lk[k] = *reinterpret_cast<const T*>(
              reinterpret_cast<const char*>(M + (16 * kb + k) * n) + ko);
      };
      // this wave's row tiles kb + 1 + wv, + 4, ... (NQ of them): their L
      // loads while U_kb is solved
      auto apply = [&](auto NQc, int kb) __attribute__((always_inline)) {
        constexpr int NQ = decltype(NQc)::value;
        T lv[NQ > 0 ? NQ : 1][4];
        if constexpr (NQ > 0) {
          // (where each row keeps its L; a padded row repeats another's: it
          // is never stored and never a pivot of a real column)
          const unsigned char* __restrict__ pe = sh.pend[16 * kb / W];
          unsigned li[NQ];
#pragma unroll
          for (int q = 0; q < NQ; ++q)
            li[q] = ((unsigned)min((int)pe[sh.perm[16 * (kb + 1 + wv + 4 * q) + e16]], n - 1) +
                     (unsigned)(g * n)) * (unsigned)sizeof(T);
#pragma unroll
          for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int q = 0; q < NQ; ++q)
              lv[q][s] = *reinterpret_cast<const T*>(
                  reinterpret_cast<const char*>(M + (16 * kb + 4 * s) * n) + li[q]);
        }
        T x[kCt];
#pragma unroll
        for (int r = 0; r < kCt; ++r) x[r] = sh.s[(16 * r + 4 * wv + g) * kWs + 16 * kb + e16];
        unit_lower_solve<T, kCt>(lk, x, e16);
#pragma unroll
        for (int r = 0; r < kCt; ++r) sh.s[(16 * r + 4 * wv + g) * kWs + 16 * kb + e16] = x[r];
        lds_barrier();
        if (16 * (kb + 1) < C0) load_kk(kb + 1);
        if constexpr (NQ > 0) {
#pragma unroll
          for (int ct = 0; ct < kCt; ++ct) {
            T ua[4];
            v4 d[NQ];
            T* __restrict__ t = sh.s + 16 * ct * kWs + 16 * (kb + 1 + wv) + e16;
#pragma unroll
            for (int s = 0; s < 4; ++s)
              ua[s] = -sh.s[(16 * ct + e16) * kWs + 16 * kb + 4 * s + g];
#pragma unroll
            for (int q = 0; q < NQ; ++q)
#pragma unroll
              for (int e = 0; e < 4; ++e) d[q][e] = t[Mf16<T>::row(g, e) * kWs + 64 * q];
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
              for (int q = 0; q < NQ; ++q) d[q] = Mf16<T>::mma(ua[s], lv[q][s], d[q]);
#pragma unroll
            for (int q = 0; q < NQ; ++q)
#pragma unroll
              for (int e = 0; e < 4; ++e) t[Mf16<T>::row(g, e) * kWs + 64 * q] = d[q][e];
          }
        }
        lds_barrier();
      };
      load_kk(0);
      for (int kb = 0; 16 * kb < C0; ++kb) {
        const int nq = (RT - kb - 1 - wv + 3) >> 2;  // (every wave passes the same barriers)
        if (nq >= 4) apply(std::integral_constant<int, 4>{}, kb);
        else if (nq == 3) apply(std::integral_constant<int, 3>{}, kb);
        else if (nq == 2) apply(std::integral_constant<int, 2>{}, kb);
        else if (nq == 1) apply(std::integral_constant<int, 1>{}, kb);
        else apply(std::integral_constant<int, 0>{}, kb);
      }
    }

    // ---- the strip's own panels ---------------------------------------------
    const bool mine = tid >= C0 && tid < npad;
    int pos = tid;  // position of row tid of the strip
    LuCand<T>* __restrict__ my_cand = &sh.cand[0][tid >> 6];
    const LuCand<T>* __restrict__ all_cand = &sh.cand[0][lane & 3];
    T* __restrict__ my_crow = sh.crow[0][tid >> 6];
    for (int ss = 0; ss < ctn; ++ss) {
      const int c0 = C0 + 16 * ss;
      T* __restrict__ panel = sh.s + 16 * ss * kWs;
      T a[kWp];
#pragma unroll
      for (int c = 0; c < kWp; ++c) a[c] = row ? panel[c * kWs + tid] : (T)0;
      bool live = mine && pos >= c0;
      int vat = 0;  // lane j: column j's pivot row | position << 16
      auto column = [&](auto J) __attribute__((always_inline)) {
        constexpr int j = decltype(J)::value;
        constexpr int buf = j & 1;
        const int c = c0 + j;
        // (a padded row pivots padded columns only)
        const unsigned kh = live && (phys < n) == (c < n) ? abs_key(a[j]) : 0u;
        // (off the chain: every row's own reciprocal while the wave searches)
        const T inv_own = a[j] != (T)0 ? (T)1 / a[j] : (T)0;
        const unsigned wh = wave_max_u32(kh);
        unsigned long long who = __ballot(kh == wh);
        int at = tid | pos << 16;
        if (__builtin_popcountll(who) > 1) {
          if (wh == 0u) {
            // no finite candidate in this wave: the row at position c where
            // it is here (it is kept if every wave says so), else nothing
            who = __ballot(mine && pos == c);
            if (who == 0ull) {
              who = 1ull;
              at = 0x7fff0000;
            }
          } else {
            // FP64: the low words; then the lowest position among equals
            const unsigned kl = low_key(a[j]);
            const unsigned wl = sizeof(T) == 8 ? wave_max_u32(in_mask(who) ? kl : 0u) : 0u;
            who &= __ballot(kl == wl);
            const int q = wave_min_i32(in_mask(who) ? pos : 0x7fff);
            who &= __ballot(pos == q);
          }
        }
        if (in_mask(who)) {
          LuCand<T>* __restrict__ o = my_cand + 4 * buf;
          *reinterpret_cast<uint4*>(o) = make_uint4(wh, low_key(a[j]), (unsigned)at, 0u);
          o->inv = inv_own;
          if constexpr (j + 1 < kWp) o->u1 = a[j + 1];
          T* __restrict__ r = my_crow + 4 * kWp * buf;
#pragma unroll
          for (int cc = j + 2; cc < kWp; ++cc) r[cc] = a[cc];
        }
        lds_barrier();
        // the best of the four candidates (lane w of four holds wave w's)
        const LuCand<T> cd = all_cand[4 * buf];
        unsigned bh = max(cd.key, dpp_mov<0xB1>(cd.key));
        bh = max(bh, dpp_mov<0x4E>(bh));
        const unsigned eq = (unsigned)__ballot(cd.key == bh) & 15u;
        int bw = (int)__builtin_ctz(eq);
        if (eq & (eq - 1u)) {
          for (int w = bw + 1; w < 4; ++w) {
            if (!((eq >> w) & 1u)) continue;
            const unsigned lw = (unsigned)__builtin_amdgcn_readlane((int)cd.low, w);
            const unsigned lb = (unsigned)__builtin_amdgcn_readlane((int)cd.low, bw);
            const int pw = __builtin_amdgcn_readlane(cd.at, w);
            const int pb = __builtin_amdgcn_readlane(cd.at, bw);
            const bool none = __builtin_amdgcn_readlane((int)cd.key, bw) == 0;
            if ((!none && lw > lb) || ((none || lw == lb) && (pw >> 16) < (pb >> 16))) bw = w;
          }
        }
        const int bat = __builtin_amdgcn_readlane(cd.at, bw);
        const T inv = rl(cd.inv, bw), u1 = j + 1 < kWp ? rl(cd.u1, bw) : (T)0;
        T u[kWp];
        const T* __restrict__ r = sh.crow[buf][bw];
#pragma unroll
        for (int cc = j + 2; cc < kWp; ++cc) u[cc] = r[cc];
        live = live && tid != (bat & 0xffff);
        if (live) {
          const T l = a[j] * inv;
          a[j] = l;
          if constexpr (j + 1 < kWp) a[j + 1] = fma(-l, u1, a[j + 1]);
#pragma unroll
          for (int cc = j + 2; cc < kWp; ++cc) a[cc] = fma(-l, u[cc], a[cc]);
        }
        // interchange positions c and p
        const int p = bat >> 16;
        pos = pos == c ? p : (pos == p ? c : pos);
        vat = lane == j ? bat : vat;
      };
      // (padded columns change nothing that is stored: 3000 FP64 blocks of order 4
      // 56.7 -> 33.0 us, of order 68 465 -> 421.  Four columns at a time: a test per
      // column costs FP32 1%)
      sfor<0, kWp / 4>([&](auto Q) __attribute__((always_inline)) {
        constexpr int q = 4 * decltype(Q)::value;
        if (q == 0 || c0 + q < n) sfor<q, q + 4>(column);
      });
      if (wv == 0 && lane < kWp) {
        sh.piv[c0 + lane] = (unsigned char)(vat >> 16);
        sh.prow[lane] = (unsigned char)vat;
      }
      if (mine) {
#pragma unroll
        for (int c = 0; c < kWp; ++c) panel[c * kWs + tid] = a[c];
        sh.pos[tid] = (unsigned char)pos;
      }
      lds_barrier();
      {
        // the first zero pivot of a real column
        const bool zero = c0 + e16 < n && panel[e16 * kWs + sh.prow[e16]] == (T)0;
        const unsigned z = (unsigned)__ballot(zero) & 0xffffu;
        if (z != 0u && first_zero == 0) first_zero = c0 + (int)__builtin_ctz(z) + 1;
      }
      if (ss + 1 < ctn) {
        // U's rows of the strip's remaining columns (the pivots' rows, where
        // they stand), then the rows not yet pivoted
        const int pr = sh.prow[e16];
        T lk[kWp - 1];
#pragma unroll
        for (int k = 0; k < kWp - 1; ++k) lk[k] = panel[k * kWs + pr];
        for (int ct = ss + 1; ct < ctn; ++ct) {
          T x[1] = {sh.s[(16 * ct + 4 * wv + g) * kWs + pr]};
          unit_lower_solve<T, 1>(lk, x, e16);
          sh.s[(16 * ct + 4 * wv + g) * kWs + pr] = x[0];
        }
        lds_barrier();
        int pu[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) pu[s] = sh.prow[4 * s + g];
        for (int ct = ss + 1; ct < ctn; ++ct) {
          T ua[4];
#pragma unroll
          for (int s = 0; s < 4; ++s) ua[s] = -sh.s[(16 * ct + e16) * kWs + pu[s]];
          for (int rt = C0 / kWp + wv; rt < RT; rt += 4) {
            const int r = 16 * rt + e16;
            T* __restrict__ t = sh.s + 16 * ct * kWs + r;
            v4 d;
#pragma unroll
            for (int e = 0; e < 4; ++e) d[e] = t[Mf16<T>::row(g, e) * kWs];
#pragma unroll
            for (int s = 0; s < 4; ++s) d = Mf16<T>::mma(ua[s], panel[(4 * s + g) * kWs + r], d);
            if ((int)sh.pos[r] >= c0 + kWp) {
#pragma unroll
              for (int e = 0; e < 4; ++e) t[Mf16<T>::row(g, e) * kWs] = d[e];
            }
          }
        }
        lds_barrier();
      }
    }

    // ---- the finished strip, every row at its position -------------------------
    if (pos < n && tid < npad) {
#pragma unroll
      for (int c = 0; c < W; ++c)
        if (C0 + c < n) st<T>(M, pos + (C0 + c) * n, sh.s[c * kWs + tid]);
    }
    // positions -> rows of A
    if (mine) {
      sh.perm[pos] = (unsigned char)phys;
      sh.pend[C0 / W][phys] = (unsigned char)pos;
    }
    __syncthreads();  // the strip is visible to the next one's loads
  }

  // ---- rows of L that later strips moved ----------------------------------------
  const int phys = row ? sh.perm[tid] : tid;
  for (int C0 = 0; C0 + W < npad; C0 += W) {
    const bool low = tid >= C0 + W && tid < n;
    const int old = low ? min((int)sh.pend[C0 / W][phys], n - 1) : tid;
    if (!__syncthreads_or(old != tid)) continue;
    for (int h = 0; h < W; h += 16) {
      T v[16];
      if (old != tid) {
#pragma unroll
        for (int c = 0; c < 16; ++c) v[c] = ld(M, old + (C0 + h + c) * n);
      }
      __syncthreads();
      if (old != tid) {
#pragma unroll
        for (int c = 0; c < 16; ++c) st<T>(M, tid + (C0 + h + c) * n, v[c]);
      }
    }
  }
  if (tid < n) {
    perm[xo + tid] = phys;
    piv[xo + tid] = sh.piv[tid];
    if constexpr (kEq) rs[xo + tid] = sr;
  }
  if (tid == 0) info[b] = first_zero;
}

// Strip widths.  A workgroup's LDS is its strip: 71 KB in FP64 (two blocks per
// CU), 39 KB in FP32 (four, with 128 registers).  Measured on 2048 fiber
// blocks of order 64-256 in FP64: 0.81 ms (width 16, three blocks per CU:
// 0.79, but the order-256 blocks alone 1.1x slower; width 64: 1.27); on 4096
// blocks of order 256 in FP32: 2.00 ms (width 16: 2.33, width 64: 2.54, three
// blocks per CU: 2.19).  One wavefront per block and a right-looking update in
// memory took 1.85 and 7.3 ms; A read twice (FP32: row maxima first) and the
// factor written once would take 0.15 and 1.1 ms at a large copy's rate.
// FP64 blocks of order up to 64, where two per CU are not all of them, have strips
// of 64 rows (19 KB) and four blocks per CU, with 128 registers: 3000 blocks of order 36
// 259 -> 183 us, 64 325 -> 227 (one wavefront per block 226 and 325); but 512 of order
// 48 45 -> 52, so fewer stay.  (FP32 has four per CU as it is: 3000 of order 36, 152
// against 158.)
constexpr int kLuW64 = 32, kLuW32 = 32;

template <int NM>
__global__ void __launch_bounds__(256, NM == 64 ? 4 : 2)
lu_block_f64_kernel(const int* __restrict__ n_arr, const long* __restrict__ a_off,
                    const long* __restrict__ x_off, const int* __restrict__ order,
                    const double* __restrict__ A, double* __restrict__ LU, int* __restrict__ piv,
                    int* __restrict__ perm, int* __restrict__ info) {
  __shared__ LuShared<double, kLuW64, NM> sh;
  lu_block_body<double, kLuW64, NM>(sh, n_arr, a_off, x_off, order, A, LU, nullptr, nullptr, piv, perm, info);
}
__global__ void __launch_bounds__(256, 4)
lu_block_f32_kernel(const int* __restrict__ n_arr, const long* __restrict__ a_off,
                    const long* __restrict__ x_off, const int* __restrict__ order,
                    const double* __restrict__ A, float* __restrict__ LU, double* __restrict__ rs,
                    double* __restrict__ cs, int* __restrict__ piv, int* __restrict__ perm,
                    int* __restrict__ info) {
  __shared__ LuShared<float, kLuW32, kWmax> sh;
  lu_block_body<float, kLuW32, kWmax>(sh, n_arr, a_off, x_off, order, A, LU, rs, cs, piv, perm, info);
}

int launch_lu_block(int precision, int64_t nb, int32_t nmax, const int32_t* n, const int64_t* a_off,
                    const int64_t* x_off, const int32_t* order, const double* A, double* lu64,
                    float* lu32, double* rs, double* cs, int32_t* piv, int32_t* perm,
                    int32_t* info, hipStream_t st) {
#define F3D_LB(K, ...)                                                                         \
  F3D_LAUNCH(K, dim3((unsigned)nb), dim3(256), 0, st, n, (const long*)a_off, (const long*)x_off, \
             order, A, __VA_ARGS__, piv, perm, info)
  if (precision == F3D_F32C) {
    F3D_LB(lu_block_f32_kernel, lu32, rs, cs);
  } else if (nmax <= 64 && nb > 2 * (int64_t)num_cus()) {
    F3D_LB(lu_block_f64_kernel<64>, lu64);
  } else {
    F3D_LB(lu_block_f64_kernel<kWmax>, lu64);
  }
#undef F3D_LB
  return F3D_OK;
}

}  // namespace f3d

// BF16 GEMM on MFMA with FP32 accumulation, with the epilogues the per-node
// MLP of the learned GMRES initial guess needs for training and inference.
// (No reference counterpart: the learned guess is new to this path.)
//
//   C[m, n] = epi( sum_k A[m, k] B[k, n] )
//   A(m, k) = A[m*sam + k*sak], B(k, n) = B[k*sbk + n*sbn] (FP32 in memory,
//   rounded to BF16 -- round to nearest even -- when staged into LDS);
//   C(m, n) = C[m*scm + n*scn] (FP32).
//
// General tiling for CDNA4 (any shape and strides, K splits): a 256-thread
// workgroup owns a 64 x 64 tile of C; each wave owns a 32 x 32 quarter and
// issues v_mfma_f32_32x32x16_bf16 on 64-deep K chunks, double buffered in LDS
// (both operands with K contiguous, so a fragment is one 16-byte read).  An
// operand is loaded along its unit-stride direction, 256 bytes of a row at a
// time, with float4 where it is aligned: along K, or along its rows with
// pairs of K packed on the way into LDS.
// (Loading both operands element by element with K fastest, whatever their
// strides, was bound by uncoalesced reads of the transposed ones: 103-130 us
// for a gradient product of 8192 samples at 256 x 256.)
// The weight gradients A^T B (K = number of samples) split K over grid.y into
// partial sums that a second kernel adds in a fixed order, with the column sums
// of B (the bias gradients) from the same pass over B; all layers are one
// launch: 22 + 4 us for 23 -> 256 -> 256 -> 4 at 8192 samples (three products
// with atomic sums and three column sums took 360).
// The per-node layers (N = 128 or 256, K <= 256) of many rows take the
// streaming or resident kernels below.
#include "common.h"

#include <math.h>

namespace f3d {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kMT = 64, kNT = 64, kKT = 64;
constexpr int kTP = kKT + 8;  // LDS row pitch (bf16): 144 B, 16-byte aligned

// two values, round to nearest even (one v_cvt_pk_bf16_f32)
__device__ __forceinline__ unsigned pack_bf16(float lo, float hi) {
  const f32x2_t v = {lo, hi};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2_t));
}

// epilogue modes
enum { EPI_STORE = 0, EPI_BIAS_RELU = 1, EPI_RELU_GRAD = 2, EPI_ATOMIC = 3, EPI_BIAS = 4 };

// One operand of a tile: entry (r, k) at p[r * sr + k * sk], r < R.
struct TileOperand {
  const float* p;
  long sr, sk;
  int R;
};

// Registers of one chunk (64 rows x 64 k): 16 values per thread.
// KC (K contiguous): row tid / 4, 16 consecutive k.  Otherwise (rows
// contiguous): two items of two k and four rows each.
template <bool KC>
__device__ __forceinline__ void tile_place(int w, int& r, int& k) {
  const int tid = threadIdx.x;
  if constexpr (KC) {
    r = tid >> 2;
    k = 16 * (tid & 3) + w;
  } else {
    const int item = tid + 256 * (w >> 3);
    r = 4 * (item & 15) + (w & 3);
    k = 2 * (item >> 4) + ((w >> 2) & 1);
  }
}

// A chunk inside the operand takes float4 loads; at its edges, and where rows are
// not aligned, every value has a clamped load of its own, all sixteen in flight
// (a branch per value, or per quad, made the compiler wait inside), and
// tile_mask drops what lies outside when the chunk is used.
template <bool KC>
__device__ __forceinline__ void tile_load(const TileOperand& o, bool whole, int r0, int k0,
                                          int kend, float (&v)[16]) {
  int r, k;
  if (whole) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      tile_place<KC>(4 * q, r, k);
      const float4 f = *reinterpret_cast<const float4*>(o.p + (r0 + r) * o.sr + (k0 + k) * o.sk);
      v[4 * q] = f.x; v[4 * q + 1] = f.y; v[4 * q + 2] = f.z; v[4 * q + 3] = f.w;
    }
  } else {
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      tile_place<KC>(w, r, k);
      v[w] = o.p[min(r0 + r, o.R - 1) * o.sr + min(k0 + k, kend - 1) * o.sk];
    }
  }
}

template <bool KC>
__device__ __forceinline__ void tile_mask(const TileOperand& o, bool whole, int r0, int k0,
                                          int kend, float (&v)[16]) {
  if (whole) return;
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    int r, k;
    tile_place<KC>(w, r, k);
    v[w] = r0 + r < o.R && k0 + k < kend ? v[w] : 0.0f;
  }
}

template <bool KC>
__device__ __forceinline__ void tile_store(unsigned short (&s)[kMT][kTP], const float (&v)[16]) {
  const int tid = threadIdx.x;
  if constexpr (KC) {
    uint4* d = reinterpret_cast<uint4*>(&s[tid >> 2][16 * (tid & 3)]);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const float* w = v + 8 * q;
      d[q] = make_uint4(pack_bf16(w[0], w[1]), pack_bf16(w[2], w[3]), pack_bf16(w[4], w[5]),
                        pack_bf16(w[6], w[7]));
    }
  } else {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int item = tid + 256 * e;
      const int r = 4 * (item & 15), k = 2 * (item >> 4);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<unsigned*>(&s[r + i][k]) = pack_bf16(v[8 * e + i], v[8 * e + 4 + i]);
    }
  }
}

// Whether float4 loads along the unit-stride direction are aligned.
__device__ __forceinline__ bool tile_vec(const TileOperand& o, bool kc) {
  const long unit = kc ? o.sk : o.sr, other = kc ? o.sr : o.sk;
  return unit == 1 && ((reinterpret_cast<uintptr_t>(o.p) | (uintptr_t)(other * 4)) & 15) == 0;
}

struct TileShared {
  __attribute__((aligned(16))) unsigned short a[2][kMT][kTP];
  __attribute__((aligned(16))) unsigned short b[2][kNT][kTP];
};

// acc (this wave's 32 x 32 quarter) = sum over k in [kbeg, kend) of
// A(m0 + .., k) B(k, n0 + ..); colsum: this thread's column sums of B (rows-
// contiguous B: columns 4 (tid % 16) .. + 3) when wanted.
template <bool AKC, bool BKC, bool SUM>
__device__ __forceinline__ f32x16_t tile_product(TileShared& sh, const TileOperand& A,
                                                 const TileOperand& B, int m0, int n0, int kbeg,
                                                 int kend, float (&colsum)[4]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const bool va = tile_vec(A, AKC), vb = tile_vec(B, BKC);
  f32x16_t acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
  float ra[16], rb[16];
  const bool wa = va && m0 + kMT <= A.R, wb = vb && n0 + kNT <= B.R;
  auto load = [&](int k0) __attribute__((always_inline)) {
    const bool in = k0 + kKT <= kend;
    tile_load<AKC>(A, wa && in, m0, k0, kend, ra);
    tile_load<BKC>(B, wb && in, n0, k0, kend, rb);
  };
  auto store = [&](int buf, int k0) __attribute__((always_inline)) {
    const bool in = k0 + kKT <= kend;
    tile_mask<AKC>(A, wa && in, m0, k0, kend, ra);
    tile_mask<BKC>(B, wb && in, n0, k0, kend, rb);
    tile_store<AKC>(sh.a[buf], ra);
    tile_store<BKC>(sh.b[buf], rb);
    if constexpr (SUM) {
#pragma unroll
      for (int i = 0; i < 4; ++i) colsum[i] += (rb[i] + rb[4 + i]) + (rb[8 + i] + rb[12 + i]);
    }
  };
  if (kbeg >= kend) return acc;
  // One copy of the loads and of the stores: the first pass of the loop has no
  // product yet.  (A kernel's instructions are fetched from L2 when it starts,
  // and short products run them about once.)
  const int row = 32 * wm + (lane & 31), col = 32 * wn + (lane & 31);
  int buf = 1;
#pragma unroll 1
  for (int k0 = kbeg - kKT; k0 < kend; k0 += kKT, buf ^= 1) {
    const bool more = k0 + kKT < kend;
    if (more) load(k0 + kKT);  // in flight during the MFMAs
    if (k0 >= kbeg) {
#pragma unroll
      for (int ks = 0; ks < kKT; ks += 16) {
        const int kofs = ks + 8 * (lane >> 5);
        const bf16x8_t a =
            __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(&sh.a[buf][row][kofs]));
        const bf16x8_t b =
            __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(&sh.b[buf][col][kofs]));
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
      }
    }
    if (more) store(buf ^ 1, k0 + kKT);
    lds_barrier();
  }
  return acc;
}

template <int EPI, bool AKC, bool BKC>
__global__ void __launch_bounds__(256)
gemm_bf16_kernel(TileOperand A, TileOperand B, int K, int kchunk, float* __restrict__ C, long scm,
                 long scn, const float* __restrict__ bias, float* __restrict__ Z,
                 const float* __restrict__ Zin, float alpha) {
  __shared__ TileShared sh;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m0 = blockIdx.y * kMT, n0 = blockIdx.x * kNT;
  const int kbeg = blockIdx.z * kchunk;
  // C layout of the 32 x 32 MFMA: register i of lane l holds
  // row 8*(i/4) + 4*(l/32) + i%4, column l%32.
  const int n = n0 + 32 * (wave & 1) + (lane & 31);
  const int mb = m0 + 32 * (wave >> 1) + 4 * (lane >> 5);
  // What the epilogue reads comes before the product: read row by row among its
  // stores, each value waited for the stores of the row before (9 us, of the 10
  // that a small layer took).
  float bn = 0.0f, z[16];
  if (EPI == EPI_BIAS_RELU || EPI == EPI_BIAS) {
    if (bias) bn = bias[min(n, B.R - 1)];
  }
  if (EPI == EPI_RELU_GRAD) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int m = mb + 8 * (i >> 2) + (i & 3);
      z[i] = Zin[(long)min(m, A.R - 1) * scm + (long)min(n, B.R - 1) * scn];
    }
  }
  float unused[4];
  const f32x16_t acc =
      tile_product<AKC, BKC, false>(sh, A, B, m0, n0, kbeg, min(K, kbeg + kchunk), unused);
  if (n >= B.R) return;
  const long c0 = (long)mb * scm + (long)n * scn;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int q = 8 * (i >> 2) + (i & 3);
    if (mb + q >= A.R) break;  // (rows rise with i)
    float v = alpha * acc[i];
    const long ci = c0 + q * scm;
    if (EPI == EPI_ATOMIC) {
      atomicAdd(&C[ci], v);
    } else if (EPI == EPI_BIAS_RELU || EPI == EPI_BIAS) {
      if (bias) v += bn;
      if (EPI == EPI_BIAS_RELU) {
        if (Z) Z[ci] = v;
        v = v > 0.0f ? v : 0.0f;
      }
      C[ci] = v;
    } else if (EPI == EPI_RELU_GRAD) {
      C[ci] = z[i] > 0.0f ? v : 0.0f;
    } else {
      C[ci] = v;
    }
  }
}

// ---------------------------------------------------------------------------
// Weight and bias gradients of several layers in one launch: layer l's
// W = A^T B (A: K x M, B: K x N) and b = column sums of B, K = samples, over
// one K slice per grid.y; partial sums at ws[slice * total + off + m * N + n]
// (weights) and ... + off + M * N + n (biases).
constexpr int kGradLayers = 3;
struct GradLayer {
  TileOperand a, b;  // rows: m (a), n (b)
  int tile0, tiles_n;
  long off;
  float* w;   // the layer's gradients, dense
  float* bs;
};
struct GradPlan {
  GradLayer l[kGradLayers];
  int K, kchunk, slices;
  long total;
};

__global__ void __launch_bounds__(256)
grad_partial_kernel(GradPlan p, float* __restrict__ ws) {
  __shared__ TileShared sh;
  int li = 0;
#pragma unroll
  for (int i = 1; i < kGradLayers; ++i)
    if ((int)blockIdx.x >= p.l[i].tile0) li = i;
  const GradLayer& L = p.l[li];
  const int t = (int)blockIdx.x - L.tile0;
  const int m0 = (t / L.tiles_n) * kMT, n0 = (t % L.tiles_n) * kNT;
  const int kbeg = blockIdx.y * p.kchunk, kend = min(p.K, kbeg + p.kchunk);
  float cs[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  const f32x16_t acc = tile_product<false, false, true>(sh, L.a, L.b, m0, n0, kbeg, kend, cs);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int M = L.a.R, N = L.b.R;
  float* __restrict__ out = ws + blockIdx.y * p.total + L.off;
  const int n = n0 + 32 * (wave & 1) + (lane & 31);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int m = m0 + 32 * (wave >> 1) + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
    if (m < M && n < N) out[(long)m * N + n] = acc[i];
  }
  if (m0 == 0) {
    // the 16 threads of a column quad, in a fixed order
    float* __restrict__ red = reinterpret_cast<float*>(&sh);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) red[(threadIdx.x >> 4) * 64 + 4 * (threadIdx.x & 15) + i] = cs[i];
    __syncthreads();
    if (threadIdx.x < 64 && n0 + (int)threadIdx.x < N) {
      float s = 0.0f;
#pragma unroll
      for (int q = 0; q < 16; ++q) s += red[q * 64 + threadIdx.x];
      out[(long)M * N + n0 + threadIdx.x] = s;
    }
  }
}

__global__ void __launch_bounds__(256)
grad_reduce_kernel(GradPlan p, const float* __restrict__ ws) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= p.total) return;
  float s = 0.0f;
#pragma unroll 8
  for (int q = 0; q < p.slices; ++q) s += ws[q * p.total + i];
  int li = 0;
#pragma unroll
  for (int l = 1; l < kGradLayers; ++l)
    if (i >= p.l[l].off) li = l;
  const GradLayer& L = p.l[li];
  const long e = i - L.off, mn = (long)L.a.R * L.b.R;
  if (e < mn) L.w[e] = s;
  else L.bs[e - mn] = s;
}

// ---------------------------------------------------------------------------
// Streaming path for the per-node layers (M = nodes, large; N = 64 NT up to
// 256; K <= 256): a workgroup owns 128 rows and ALL N columns, so every
// activation row is read from HBM once and written once.  2 x NT waves, each
// owning a 64 x 64 block as 2 x 2 32x32 MFMA tiles (64 accumulator
// registers), so a 256-wide layer runs 8 waves per workgroup.  K is staged
// through LDS in 32-deep chunks, double
// buffered: the next chunk's global loads (float4) are issued before the
// current chunk's MFMAs, one barrier per chunk; each 16-deep step reuses
// every A fragment across the wave's two column tiles and every B fragment
// across its two row tiles.
constexpr int kSM = 128;  // rows per workgroup
constexpr int kSK = 32;   // K chunk
constexpr int kSP = kSK + 8;  // LDS row pitch (bf16 elements): 80 B, 16-byte aligned

template <int EPI, int NT>  // NT = N / 64 (2 or 4); 128 NT threads
__global__ void __launch_bounds__(512)
gemm_bf16_stream_kernel(int M, int N, int K, const float* __restrict__ A, long sam,
                        const float* __restrict__ B, long sbk, long sbn,
                        float* __restrict__ C, long scm, const float* __restrict__ bias,
                        float* __restrict__ Z, const float* __restrict__ Zin, float alpha) {
  constexpr int NW = 64 * NT;      // columns of the workgroup = N
  constexpr int NTH = 128 * NT;    // threads
  constexpr int AK = kSK / NT;     // A floats per thread and chunk
  constexpr int BI = kSK / 16;     // B items (k pair, column quad) per thread
  __shared__ __attribute__((aligned(16))) unsigned short As[2][kSM][kSP];
  __shared__ __attribute__((aligned(16))) unsigned short Bt[2][NW][kSP];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / NT, wn = wave % NT;
  const int m0 = blockIdx.x * kSM;
  f32x16_t acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.0f;

  // staging: A chunk 128 x kSK (row tid / NT, AK consecutive k per thread,
  // float4 pieces), B chunk kSK x NW as BI items per thread of (k pair, 4
  // columns): two float4 rows, stored transposed as four (k, k+1) bf16
  // pairs.  Vector loads where the row is 16-byte aligned and in range.
  float4 ra[AK / 4];
  float4 rb[BI][2];
  const bool bvec = sbn == 1 && ((reinterpret_cast<uintptr_t>(B) | (uintptr_t)(sbk * 4)) & 15) == 0;
  auto ld4 = [&](const float* __restrict__ p, int avail, bool vec) __attribute__((always_inline)) {
    if (vec && avail >= 4) return *reinterpret_cast<const float4*>(p);
    return make_float4(avail > 0 ? p[0] : 0.0f, avail > 1 ? p[1] : 0.0f,
                       avail > 2 ? p[2] : 0.0f, avail > 3 ? p[3] : 0.0f);
  };
  auto load = [&](int k0) __attribute__((always_inline)) {
    const int r = tid / NT, kh = (tid % NT) * AK;
    const int m = m0 + r;
    const float* __restrict__ arow = A + (long)(m < M ? m : 0) * sam;
#pragma unroll
    for (int q = 0; q < AK / 4; ++q) {
      const int k = k0 + kh + 4 * q;
      const float* __restrict__ pa = arow + k;
      const bool al = (reinterpret_cast<uintptr_t>(pa) & 15) == 0;
      ra[q] = m < M ? ld4(pa, K - k, al) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
#pragma unroll
    for (int e = 0; e < BI; ++e) {
      // over (k pair, column quad), k pairs fastest: consecutive lanes store
      // consecutive words of one LDS row (no bank conflicts)
      const int idx = tid + NTH * e;
      const int kp = idx % (kSK / 2), nq = idx / (kSK / 2);
      const int k = k0 + 2 * kp, n = 4 * nq;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int kk = k + h;
        if (kk < K && bvec) {
          rb[e][h] = ld4(B + (long)kk * sbk + n, N - n, true);
        } else if (kk < K) {
          const float* __restrict__ pb = B + (long)kk * sbk + (long)n * sbn;
          rb[e][h] = make_float4(n < N ? pb[0] : 0.0f, n + 1 < N ? pb[sbn] : 0.0f,
                                 n + 2 < N ? pb[2 * sbn] : 0.0f, n + 3 < N ? pb[3 * sbn] : 0.0f);
        } else {
          rb[e][h] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
      }
    }
  };
  auto pack2 = [](float lo, float hi) __attribute__((always_inline)) { return pack_bf16(lo, hi); };
  auto store = [&](int buf) __attribute__((always_inline)) {
    const int r = tid / NT, kh = (tid % NT) * AK;
#pragma unroll
    for (int q = 0; q < AK / 8; ++q) {
      uint4 u;
      u.x = pack2(ra[2 * q].x, ra[2 * q].y);
      u.y = pack2(ra[2 * q].z, ra[2 * q].w);
      u.z = pack2(ra[2 * q + 1].x, ra[2 * q + 1].y);
      u.w = pack2(ra[2 * q + 1].z, ra[2 * q + 1].w);
      *reinterpret_cast<uint4*>(&As[buf][r][kh + 8 * q]) = u;
    }
#pragma unroll
    for (int e = 0; e < BI; ++e) {
      const int idx = tid + NTH * e;
      const int kp = idx % (kSK / 2), nq = idx / (kSK / 2);
      const int n = 4 * nq;
      *reinterpret_cast<unsigned*>(&Bt[buf][n + 0][2 * kp]) = pack2(rb[e][0].x, rb[e][1].x);
      *reinterpret_cast<unsigned*>(&Bt[buf][n + 1][2 * kp]) = pack2(rb[e][0].y, rb[e][1].y);
      *reinterpret_cast<unsigned*>(&Bt[buf][n + 2][2 * kp]) = pack2(rb[e][0].z, rb[e][1].z);
      *reinterpret_cast<unsigned*>(&Bt[buf][n + 3][2 * kp]) = pack2(rb[e][0].w, rb[e][1].w);
    }
  };
  load(0);
  store(0);
  __syncthreads();
  const int nchunks = (K + kSK - 1) / kSK;
  for (int c = 0; c < nchunks; ++c) {
    const int buf = c & 1;
    if (c + 1 < nchunks) load((c + 1) * kSK);  // in flight during the MFMAs
#pragma unroll
    for (int ks = 0; ks < kSK; ks += 16) {
      const int kofs = ks + 8 * (lane >> 5);
      bf16x8_t fa[2], fb[2];
#pragma unroll
      for (int a = 0; a < 2; ++a)
        fa[a] = __builtin_bit_cast(
            bf16x8_t, *reinterpret_cast<const uint4*>(&As[buf][64 * wm + 32 * a + (lane & 31)][kofs]));
#pragma unroll
      for (int b = 0; b < 2; ++b)
        fb[b] = __builtin_bit_cast(
            bf16x8_t, *reinterpret_cast<const uint4*>(&Bt[buf][64 * wn + 32 * b + (lane & 31)][kofs]));
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a], fb[b], acc[a][b], 0, 0, 0);
    }
    if (c + 1 < nchunks) store(buf ^ 1);
    __syncthreads();
  }
  // epilogue: register i of lane l holds row 8(i/4) + 4(l/32) + i%4, column l%32
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int n = 64 * wn + 32 * b + (lane & 31);
      const float bn = (bias && n < N) ? bias[n] : 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int m = m0 + 64 * wm + 32 * a + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
        if (m >= M || n >= N) continue;
        float v = alpha * acc[a][b][i];
        const long ci = (long)m * scm + n;
        if (EPI == EPI_BIAS_RELU || EPI == EPI_BIAS) {
          v += bn;
          if (EPI == EPI_BIAS_RELU) {
            if (Z) Z[ci] = v;
            v = v > 0.0f ? v : 0.0f;
          }
          C[ci] = v;
        } else if (EPI == EPI_RELU_GRAD) {
          C[ci] = Zin[ci] > 0.0f ? v : 0.0f;
        } else {
          C[ci] = v;
        }
      }
    }
}

// ---------------------------------------------------------------------------
// Resident-weight path for the per-node layers: one persistent 512-thread
// workgroup per CU holds all of B (K x N, BF16, transposed, 135 KB at
// N = K = 256) in LDS for the whole launch, so B is read once per CU instead
// of once per row block, and streams blocks of RM rows of A (32 rows at
// N = 256, 64 at N = 128).  The FP32 A rows of the next kRD blocks are in
// flight in registers while a block multiplies: at N = K = 256 that is 64 KB
// of HBM reads outstanding per CU.  Each of the 8 waves owns one 32 x 32
// tile of the block (v_mfma_f32_32x32x16_bf16 over K in 16-deep steps, A
// fragments from the block's LDS rows, B fragments from the resident
// columns).  K must be a multiple of 16 and at most 256, A row-major with
// 16-byte aligned rows.
constexpr int kRKmax = 256;
constexpr int kRP = kRKmax + 8;  // LDS pitch (bf16): 528 B, 16-byte aligned
constexpr int kRD = 2;           // A blocks in flight (2, 3, 4, 6 measured alike)

template <int EPI, int NT>  // N = 64 NT (2 or 4)
__global__ void __launch_bounds__(512)
gemm_bf16_resident_kernel(int M, int N, int K, const float* __restrict__ A, long sam,
                          const float* __restrict__ B, long sbk, long sbn,
                          float* __restrict__ C, long scm, const float* __restrict__ bias,
                          float* __restrict__ Z, const float* __restrict__ Zin, float alpha) {
  constexpr int NW = 64 * NT;        // columns
  constexpr int CT = NW / 32;        // column tiles
  constexpr int RT = 8 / CT;         // row tiles per block
  constexpr int RM = 32 * RT;        // rows per block
  constexpr int PP = RM * kRKmax / 4 / 512;  // float4 pieces per thread (K = 256)
  __shared__ __attribute__((aligned(16))) unsigned short Bs[NW][kRP];
  __shared__ __attribute__((aligned(16))) unsigned short As[RM][kRP];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int ct = wave % CT, rt = wave / CT;
  const int K4 = K / 4;                       // float4 pieces per row
  const int pieces = RM * K4;                 // per block (<= 512 PP)
  const int nblocks = (M + RM - 1) / RM;

  auto pack2 = [](float lo, float hi) __attribute__((always_inline)) { return pack_bf16(lo, hi); };
  // A pieces of block bl into registers: piece q = tid + 512 j is row q / K4,
  // columns 4 (q % K4) ..; rows past M and pieces past the block read row 0
  // (in bounds) and are zeroed when staged.
  float4 ra[kRD][PP];
  auto load = [&](int bl, float4 (&r)[PP]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < PP; ++j) {
      const int q = tid + 512 * j;
      const int row = q / K4, c4 = q - row * K4;
      const long m = (long)bl * RM + row;
      const bool ok = q < pieces && m < M;
      r[j] = *reinterpret_cast<const float4*>(A + (ok ? m : 0) * sam + 4 * (ok ? c4 : 0));
    }
  };
  auto stage = [&](int bl, const float4 (&r)[PP]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < PP; ++j) {
      const int q = tid + 512 * j;
      if (q < pieces) {
        const int row = q / K4, c4 = q - row * K4;
        const bool ok = (long)bl * RM + row < M;
        uint2 u;
        u.x = ok ? pack2(r[j].x, r[j].y) : 0u;
        u.y = ok ? pack2(r[j].z, r[j].w) : 0u;
        *reinterpret_cast<uint2*>(&As[row][4 * c4]) = u;
      }
    }
  };

  // the first kRD blocks' A loads, then B into LDS (transposed, BF16)
  int bl = blockIdx.x;
#pragma unroll
  for (int d = 0; d < kRD; ++d) {
    const int b = bl + d * (int)gridDim.x;
    load(b < nblocks ? b : nblocks - 1, ra[d]);
  }
  for (int idx = tid; idx < NW * (K / 2); idx += 512) {
    // (k pair, column), k pairs fastest: consecutive lanes store
    // consecutive words of one LDS row
    const int kp = idx % (K / 2), n = idx / (K / 2);
    const int k = 2 * kp;
    const float b0 = n < N ? B[(long)k * sbk + (long)n * sbn] : 0.0f;
    const float b1 = n < N ? B[(long)(k + 1) * sbk + (long)n * sbn] : 0.0f;
    *reinterpret_cast<unsigned*>(&Bs[n][k]) = pack2(b0, b1);
  }

  const int n = 32 * ct + (lane & 31);
  const float bn = (bias && n < N) ? bias[n] : 0.0f;
  // block i of this workgroup uses register set i % kRD (unrolled by kRD)
  for (; bl < nblocks; bl += kRD * (int)gridDim.x) {
#pragma unroll
    for (int d = 0; d < kRD; ++d) {
      const int b = bl + d * (int)gridDim.x;
      if (b >= nblocks) continue;  // (uniform; the last round's spare set)
      __syncthreads();  // the previous block's MFMAs are done with As
      stage(b, ra[d]);
      __syncthreads();
      // this register set's next block (an in-bounds reload past the end)
      const int nb = b + kRD * (int)gridDim.x;
      load(nb < nblocks ? nb : nblocks - 1, ra[d]);
      f32x16_t acc;
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
      const int kofs = 8 * (lane >> 5);
      // (the compiler reports that it cannot honour this unroll hint in
      // full, but the loop it emits with it measured 4-8% faster than
      // without it or fully unrolled to K = 256)
#pragma unroll 4
      for (int k0 = 0; k0 < K; k0 += 16) {
        const bf16x8_t fa = __builtin_bit_cast(
            bf16x8_t, *reinterpret_cast<const uint4*>(&As[32 * rt + (lane & 31)][k0 + kofs]));
        const bf16x8_t fb = __builtin_bit_cast(
            bf16x8_t, *reinterpret_cast<const uint4*>(&Bs[32 * ct + (lane & 31)][k0 + kofs]));
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa, fb, acc, 0, 0, 0);
      }
      // register i of lane l holds row 8(i/4) + 4(l/32) + i%4, column l%32.
      // All 16 results are formed before any store, in registers of their
      // own: a store whose data register is overwritten before it has
      // issued makes the next write wait for it.
      const long m0 = (long)b * RM + 32 * rt + 4 * (lane >> 5);
      float v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        v[i] = alpha * acc[i];
        if (EPI == EPI_BIAS_RELU || EPI == EPI_BIAS) v[i] += bn;
      }
      auto row_of = [](int i) { return 8 * (i >> 2) + (i & 3); };
      if ((long)(b + 1) * RM <= M) {
        // a whole block: no row checks
        const long base = m0 * scm + n;
        if (EPI == EPI_RELU_GRAD) {
          float zin[16];
#pragma unroll
          for (int i = 0; i < 16; ++i) zin[i] = Zin[base + row_of(i) * scm];
#pragma unroll
          for (int i = 0; i < 16; ++i) C[base + row_of(i) * scm] = zin[i] > 0.0f ? v[i] : 0.0f;
        } else {
          if (EPI == EPI_BIAS_RELU && Z) {
#pragma unroll
            for (int i = 0; i < 16; ++i) Z[base + row_of(i) * scm] = v[i];
          }
#pragma unroll
          for (int i = 0; i < 16; ++i)
            C[base + row_of(i) * scm] = EPI == EPI_BIAS_RELU ? (v[i] > 0.0f ? v[i] : 0.0f) : v[i];
        }
      } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const long m = m0 + row_of(i);
          if (m >= M) continue;
          const long ci = m * scm + n;
          if (EPI == EPI_RELU_GRAD) {
            C[ci] = Zin[ci] > 0.0f ? v[i] : 0.0f;
          } else {
            if (EPI == EPI_BIAS_RELU && Z) Z[ci] = v[i];
            C[ci] = EPI == EPI_BIAS_RELU ? (v[i] > 0.0f ? v[i] : 0.0f) : v[i];
          }
        }
      }
    }
  }
}

}  // namespace f3d

using namespace f3d;

// Rows from which the row-block kernels are the faster ones.  Fewer leave CUs
// idle or pay B's set-up for a block or two; the tiled kernel's time grows
// faster with the rows, and faster still where its last 64-deep chunk of K is
// partial.  us, N = 256, resident against tiled: K = 256, 8192 rows 38 / 11,
// 32768 47 / 31, 49152 51 / 49, 262144 134 / 231; K = 128, 49151 32 / 32; K = 32, 4096
// 8.1 / 7.2, 8192 8.9 / 10.3, 49151 18 / 40; K = 96, 8192 16 / 12, 16384 18.5 / 19.8,
// 49151 27 / 48; K = 144, 24576 29 / 26, 32768 31 / 33; K = 16, 4096 6.0 / 6.2, 262144
// 65 / 118.  N = 128 crosses near the same rows (K = 32, 8192 7.2 / 7.2; K = 96,
// 16384 11.9 / 11.9; K = 144, 32768 18.5 / 19).
constexpr int kStreamRows = 49152;
static int64_t resident_rows(int64_t K) {
  const int64_t part = K % 64;
  if (part == 0) return kStreamRows;
  return part == 32 ? 128 * K : std::min(256 * K, 20480 + 64 * K);
}
// The streaming kernel takes any K and alignment; at N = 256 a CU has one
// workgroup of it, so its time is that of 128 rows a CU up to there: 32768 rows of K
// = 130 (250), 28 us for 34 (38 for 49), but 48 for 41 (67 for 59) at 40000.  From
// 7/8 of that on, where the tiled kernel has a partial chunk or a long one, and
// B's rows are contiguous or its set-up little beside the products.  (K <= 16: the
// tiled kernel at every size: K = 4, 262144 rows 97 / 88.)
static bool stream_fills(int64_t M, int64_t N, int64_t K, bool b_rows) {
  const int64_t full = (int64_t)kSM * num_cus();
  return N == 256 && M <= full && 8 * M > 7 * full && (K % 64 != 0 || K > 128) &&
         (b_rows || K > 128);
}

// Row tiles of the tiled kernel's grid (its y extent).
constexpr int64_t kTiledRowTiles = 65535;

// Whether row-major a (M x K, row stride sa) and c (M x N, row stride sc) share
// memory.
static bool meets_rows(const float* a, int64_t M, int64_t K, int64_t sa, const float* c, int64_t N,
                       int64_t sc) {
  const int64_t a0 = std::min<int64_t>(0, (M - 1) * sa), a1 = std::max<int64_t>(0, (M - 1) * sa) + K;
  const int64_t c0 = std::min<int64_t>(0, (M - 1) * sc), c1 = std::max<int64_t>(0, (M - 1) * sc) + N;
  return K > 0 && a + a0 < c + c1 && c + c0 < a + a1;
}

// Kernel for the per-node layers N = 128 / N = 256 (set by the autotuner
// through f3d_gemm_set_stream): 0 tiled, 1 streaming, 2 resident-weight.
static int g_gemm_stream[2] = {2, 2};

extern "C" int f3d_gemm_set_stream(int32_t n, int32_t enable) {
  F3D_REQUIRE(n == 128 || n == 256, F3D_EINVAL, "gemm_set_stream: N must be 128 or 256");
  F3D_REQUIRE(enable >= 0 && enable <= 2, F3D_EINVAL,
              "gemm_set_stream: kernel must be 0 (tiled), 1 (streaming) or 2 (resident)");
  g_gemm_stream[n == 256 ? 1 : 0] = enable;
  return F3D_OK;
}

extern "C" int f3d_gemm_bf16(int epi, int64_t M, int64_t N, int64_t K, int32_t ksplit,
                             const float* A, int64_t sam, int64_t sak, const float* B,
                             int64_t sbk, int64_t sbn, float* C, int64_t scm, int64_t scn,
                             const float* bias, float* Z, const float* Zin, float alpha,
                             void* stream) {
  F3D_REQUIRE(epi >= 0 && epi <= 4, F3D_EINVAL, "gemm_bf16: unknown epilogue %d", epi);
  F3D_REQUIRE(M >= 0 && N >= 0 && K >= 0 && M < (1ll << 31) && N < (1ll << 31) &&
                  K < (1ll << 31),
              F3D_EINVAL, "gemm_bf16: bad sizes");
  F3D_REQUIRE(ksplit >= 1, F3D_EINVAL, "gemm_bf16: ksplit must be >= 1");
  F3D_REQUIRE(epi == EPI_ATOMIC || ksplit == 1, F3D_EINVAL,
              "gemm_bf16: K splitting needs the atomic epilogue");
  F3D_REQUIRE(epi != EPI_RELU_GRAD || Zin != nullptr, F3D_EINVAL,
              "gemm_bf16: relu-grad epilogue needs Zin");
  if (M == 0 || N == 0) return F3D_OK;
  F3D_REQUIRE(A && B && C, F3D_EINVAL, "gemm_bf16: NULL operand");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // the row-block kernels: row-major A (unit K stride) and C (unit N stride), N
  // in {128, 256}, K <= 256, no K split; the resident one also needs K a
  // multiple of 16 and 16-byte rows of A
  const int mode = (N == 128 || N == 256) ? g_gemm_stream[N == 256 ? 1 : 0] : 0;
  const bool rows_ok = epi != EPI_ATOMIC && ksplit == 1 && sak == 1 && scn == 1 && mode > 0 &&
                       K <= 256 && M >= kSM;
  const bool resident = mode == 2 && K > 0 && K % 16 == 0 && sam % 4 == 0 &&
                        (reinterpret_cast<uintptr_t>(A) & 15) == 0;
  // Calls that only they can take: C or Z over A (a row block reads all of its
  // rows before it writes them, where a tile of the tiled kernel may be
  // written while another still reads), and more rows than its grid has.
  const bool must = meets_rows(A, M, K, sam, C, N, scm) ||
                    (Z && meets_rows(A, M, K, sam, Z, N, scm)) ||
                    ceil_div(M, (int64_t)kMT) > kTiledRowTiles;
  const bool resident_ok = rows_ok && resident && (must || M >= resident_rows(K));
  const bool stream_ok =
      rows_ok && (must || (K > 16 && (M >= kStreamRows || (!resident && stream_fills(M, N, K, sbn == 1)))));
  if (resident_ok) {
    const int RM = N == 256 ? 32 : 64;
    const int64_t nblocks = ceil_div(M, (int64_t)RM);
    const dim3 g((unsigned)std::min<int64_t>(nblocks, num_cus()));
#define F3D_R(E, T)                                                                          \
  F3D_LAUNCH((gemm_bf16_resident_kernel<E, T>), g, dim3(512), 0, st, (int)M, (int)N, (int)K, A, \
             (long)sam, B, (long)sbk, (long)sbn, C, (long)scm, bias, Z, Zin, alpha)
#define F3D_RE(E) if (N == 256) F3D_R(E, 4); else F3D_R(E, 2)
    switch (epi) {
      case EPI_STORE: F3D_RE(EPI_STORE); break;
      case EPI_BIAS_RELU: F3D_RE(EPI_BIAS_RELU); break;
      case EPI_RELU_GRAD: F3D_RE(EPI_RELU_GRAD); break;
      default: F3D_RE(EPI_BIAS); break;
    }
#undef F3D_RE
#undef F3D_R
    return F3D_OK;
  }
  if (stream_ok) {
    const dim3 g((unsigned)ceil_div(M, kSM));
#define F3D_S(E, T)                                                                            F3D_LAUNCH((gemm_bf16_stream_kernel<E, T>), g, dim3(128 * T), 0, st, (int)M, (int)N, (int)K, A,              (long)sam, B, (long)sbk, (long)sbn, C, (long)scm, bias, Z, Zin, alpha)
#define F3D_SE(E) if (N == 256) F3D_S(E, 4); else F3D_S(E, 2)
    switch (epi) {
      case EPI_STORE: F3D_SE(EPI_STORE); break;
      case EPI_BIAS_RELU: F3D_SE(EPI_BIAS_RELU); break;
      case EPI_RELU_GRAD: F3D_SE(EPI_RELU_GRAD); break;
      default: F3D_SE(EPI_BIAS); break;
    }
#undef F3D_SE
#undef F3D_S
    return F3D_OK;
  }
  int64_t kchunk = ceil_div(K > 0 ? K : 1, ksplit);
  kchunk = (int64_t)align_up((size_t)kchunk, kKT);
  const unsigned gz = (unsigned)ceil_div(K > 0 ? K : 1, kchunk);
  const dim3 grid((unsigned)ceil_div(N, kNT), (unsigned)ceil_div(M, kMT), gz);
  // each operand along its unit-stride direction (along K where both are or
  // neither is)
  const TileOperand oa{A, (long)sam, (long)sak, (int)M}, ob{B, (long)sbn, (long)sbk, (int)N};
  const bool akc = sak == 1 || sam != 1, bkc = sbk == 1 || sbn != 1;
#define F3D_GK(E, X, Y)                                                                     \
  F3D_LAUNCH((gemm_bf16_kernel<E, X, Y>), grid, dim3(256), 0, st, oa, ob, (int)K, (int)kchunk, \
             C, (long)scm, (long)scn, bias, Z, Zin, alpha)
#define F3D_G(E)                                   \
  do {                                             \
    if (akc && bkc) F3D_GK(E, true, true);         \
    else if (akc) F3D_GK(E, true, false);          \
    else if (bkc) F3D_GK(E, false, true);          \
    else F3D_GK(E, false, false);                  \
  } while (0)
  switch (epi) {
    case EPI_STORE: F3D_G(EPI_STORE); break;
    case EPI_BIAS_RELU: F3D_G(EPI_BIAS_RELU); break;
    case EPI_RELU_GRAD: F3D_G(EPI_RELU_GRAD); break;
    case EPI_ATOMIC: F3D_G(EPI_ATOMIC); break;
    default: F3D_G(EPI_BIAS); break;
  }
#undef F3D_G
#undef F3D_GK
  return F3D_OK;
}

// ---------------------------------------------------------------------------
namespace f3d {
// Mean squared error over n outputs and its gradient 2 (y - t) / n; the sum in
// FP64, per block and then over the blocks in a fixed order.
constexpr int kMseBlocks = 64;
__global__ void __launch_bounds__(256)
mse_kernel(int64_t n, const float* __restrict__ y, const float* __restrict__ t, float c,
           float* __restrict__ dy, double* __restrict__ part) {
  __shared__ double red[4];
  double s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const float d = y[i] - t[i];
    dy[i] = c * d;
    s = fma((double)d, (double)d, s);
  }
  s = wave_sum_f64(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}
__global__ void __launch_bounds__(kMseBlocks)
mse_final_kernel(int64_t n, const double* __restrict__ part, float* __restrict__ loss) {
  const double s = wave_sum_f64(part[threadIdx.x]);
  if (threadIdx.x == 0) loss[0] = (float)(s / (double)n);
}

// One Adam step over several tensors in one launch (a step of the net is 6
// tensors; one launch per tensor and operation took 66, and the host longer
// than all of the step's products).
constexpr int kAdamTensors = 8;
struct AdamArgs {
  float* p[kAdamTensors];
  const float* g[kAdamTensors];
  float* m[kAdamTensors];
  float* v[kAdamTensors];
  int64_t begin[kAdamTensors];  // of the tensor's elements in the launch
  int64_t total;
  int count;
};
__global__ void __launch_bounds__(256)
adam_kernel(AdamArgs a, float lr, float b1, float c1, float b2, float c2, float eps, float inv1,
            float inv2) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.total) return;
  int k = 0;
#pragma unroll
  for (int q = 1; q < kAdamTensors; ++q)
    if (q < a.count && i >= a.begin[q]) k = q;
  const int64_t e = i - a.begin[k];
  const float g = a.g[k][e];
  const float m = a.m[k][e] * b1 + c1 * g;
  const float v = a.v[k][e] * b2 + c2 * g * g;
  a.m[k][e] = m;
  a.v[k][e] = v;
  a.p[k][e] -= lr * (m * inv1) / (sqrtf(v * inv2) + eps);
}
}  // namespace f3d

extern "C" size_t f3d_mse_workspace_size(void) { return kMseBlocks * sizeof(double); }

extern "C" int f3d_mse(int64_t n, const float* y, const float* t, float* dy, float* loss, void* ws,
                       size_t ws_bytes, void* stream) {
  F3D_REQUIRE(n >= 1, F3D_EINVAL, "mse: n=%lld", (long long)n);
  F3D_REQUIRE(y && t && dy && loss, F3D_EINVAL, "mse: NULL argument");
  F3D_REQUIRE(ws != nullptr && ws_bytes >= f3d_mse_workspace_size(), F3D_EWORKSPACE,
              "mse: workspace %zu bytes < required %zu", ws_bytes, f3d_mse_workspace_size());
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  double* part = reinterpret_cast<double*>(ws);
  // (2 / n rounded once: the FP32 value of n is not n from 2^24 on)
  F3D_LAUNCH(mse_kernel, dim3(kMseBlocks), dim3(256), 0, st, n, y, t, (float)(2.0 / (double)n), dy,
             part);
  F3D_LAUNCH(mse_final_kernel, dim3(1), dim3(kMseBlocks), 0, st, n, (const double*)part, loss);
  return F3D_OK;
}

extern "C" int f3d_adam(int32_t count, const int64_t* sizes, float* const* p,
                        const float* const* g, float* const* m, float* const* v, double lr,
                        double b1, double b2, double eps, int64_t t, void* stream) {
  F3D_REQUIRE(count >= 0 && t >= 1, F3D_EINVAL, "adam: count=%d t=%lld", count, (long long)t);
  F3D_REQUIRE(count == 0 || (sizes && p && g && m && v), F3D_EINVAL, "adam: NULL argument");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const float inv1 = (float)(1.0 / (1.0 - pow(b1, (double)t)));
  const float inv2 = (float)(1.0 / (1.0 - pow(b2, (double)t)));
  for (int32_t k0 = 0; k0 < count; k0 += kAdamTensors) {
    AdamArgs a{};
    for (int32_t k = k0; k < count && k < k0 + kAdamTensors; ++k) {
      F3D_REQUIRE(sizes[k] >= 0 && (sizes[k] == 0 || (p[k] && g[k] && m[k] && v[k])), F3D_EINVAL,
                  "adam: tensor %d", k);
      a.p[k - k0] = p[k];
      a.g[k - k0] = g[k];
      a.m[k - k0] = m[k];
      a.v[k - k0] = v[k];
      a.begin[k - k0] = a.total;
      a.total += sizes[k];
      ++a.count;
    }
    if (a.total == 0) continue;
    F3D_REQUIRE(a.total < (1ll << 38), F3D_EINVAL, "adam: too many elements");
    F3D_LAUNCH(adam_kernel, dim3((unsigned)ceil_div(a.total, 256)), dim3(256), 0, st, a, (float)lr,
               (float)b1, (float)(1.0 - b1), (float)b2, (float)(1.0 - b2), (float)eps, inv1, inv2);
  }
  return F3D_OK;
}

// ---------------------------------------------------------------------------
// The MLP in -> width -> width -> out as whole passes (three and four
// launches): the products through f3d_gemm_bf16 and the kernels above.
extern "C" int f3d_mlp_forward(int64_t M, int32_t n_in, int32_t width, int32_t n_out,
                               const float* X, int64_t sxm, int64_t sxk, const float* W1,
                               const float* b1, const float* W2, const float* b2, const float* W3,
                               const float* b3, float* H1, float* H2, float* Y, void* stream) {
  F3D_REQUIRE(M >= 0 && n_in >= 1 && width >= 1 && n_out >= 1, F3D_EINVAL, "mlp_forward: bad sizes");
  if (M == 0) return F3D_OK;
  F3D_REQUIRE(X && W1 && W2 && W3 && H1 && H2 && Y, F3D_EINVAL,
              "mlp_forward: NULL argument");
  int rc = f3d_gemm_bf16(EPI_BIAS_RELU, M, width, n_in, 1, X, sxm, sxk, W1, width, 1, H1, width, 1,
                         b1, nullptr, nullptr, 1.0f, stream);
  if (rc != F3D_OK) return rc;
  rc = f3d_gemm_bf16(EPI_BIAS_RELU, M, width, width, 1, H1, width, 1, W2, width, 1, H2, width, 1,
                     b2, nullptr, nullptr, 1.0f, stream);
  if (rc != F3D_OK) return rc;
  return f3d_gemm_bf16(EPI_BIAS, M, n_out, width, 1, H2, width, 1, W3, n_out, 1, Y, n_out, 1, b3,
                       nullptr, nullptr, 1.0f, stream);
}

// Samples per K slice of the gradient products: slices of at least 256 samples,
// at most 64 of them (24 tiles at 23 -> 256 -> 256 -> 4, so 768 workgroups at a
// batch of 8192).
static void grad_slices(int64_t M, int* kchunk, int* slices) {
  int64_t c = ceil_div(M > 0 ? M : 1, (int64_t)64);
  c = (int64_t)align_up((size_t)(c < 256 ? 256 : c), kKT);
  *kchunk = (int)c;
  *slices = (int)ceil_div(M > 0 ? M : 1, c);
}

static int64_t mlp_params(int64_t n_in, int64_t width, int64_t n_out) {
  return n_in * width + width + width * width + width + width * n_out + n_out;
}

extern "C" size_t f3d_mlp_workspace_size(int64_t M, int32_t n_in, int32_t width, int32_t n_out) {
  if (M < 0 || M >= (1ll << 31) || n_in < 1 || width < 1 || n_out < 1) return 0;
  int kchunk, slices;
  grad_slices(M, &kchunk, &slices);
  return sizeof(float) * ((size_t)slices * (size_t)mlp_params(n_in, width, n_out) +
                          2 * (size_t)M * (size_t)width);
}

extern "C" int f3d_mlp_backward(int64_t M, int32_t n_in, int32_t width, int32_t n_out,
                                const float* X, int64_t sxm, int64_t sxk, const float* H1,
                                const float* H2, const float* dY, int64_t sym, int64_t syk,
                                const float* W2, const float* W3, float* gW1, float* gW2,
                                float* gW3, float* gb1, float* gb2, float* gb3, void* ws,
                                size_t ws_bytes, void* stream) {
  F3D_REQUIRE(M >= 0 && M < (1ll << 31) && n_in >= 1 && width >= 1 && n_out >= 1, F3D_EINVAL,
              "mlp_backward: bad sizes");
  // (no samples: zero gradients, and arrays of no elements may have no address)
  F3D_REQUIRE(M == 0 || (X && H1 && H2 && dY), F3D_EINVAL, "mlp_backward: NULL argument");
  F3D_REQUIRE(W2 && W3 && gW1 && gW2 && gW3 && gb1 && gb2 && gb3, F3D_EINVAL,
              "mlp_backward: NULL argument");
  const size_t need = f3d_mlp_workspace_size(M, n_in, width, n_out);
  F3D_REQUIRE(ws != nullptr && ws_bytes >= need, F3D_EWORKSPACE,
              "mlp_backward: workspace %zu bytes < required %zu", ws_bytes, need);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  float* dZ2 = reinterpret_cast<float*>(ws);
  float* dZ1 = dZ2 + (size_t)M * width;
  float* part = dZ1 + (size_t)M * width;
  // dZ = (dOut W^T) where the layer's ReLU was open
  if (M > 0) {
    int rc = f3d_gemm_bf16(EPI_RELU_GRAD, M, width, n_out, 1, dY, sym, syk, W3, 1, n_out, dZ2,
                           width, 1, nullptr, nullptr, H2, 1.0f, stream);
    if (rc != F3D_OK) return rc;
    rc = f3d_gemm_bf16(EPI_RELU_GRAD, M, width, width, 1, dZ2, width, 1, W2, 1, width, dZ1, width,
                       1, nullptr, nullptr, H1, 1.0f, stream);
    if (rc != F3D_OK) return rc;
  }
  GradPlan p;
  grad_slices(M, &p.kchunk, &p.slices);
  p.K = (int)M;
  int tiles = 0;
  long off = 0;
  auto layer = [&](int i, const float* a, int64_t am, int64_t ak, int m, const float* b, int64_t bn,
                   int64_t bk, int n, float* w, float* bs) {
    GradLayer& L = p.l[i];
    L.a = TileOperand{a, (long)am, (long)ak, m};
    L.b = TileOperand{b, (long)bn, (long)bk, n};
    L.tile0 = tiles;
    L.tiles_n = (int)ceil_div(n, kNT);
    L.off = off;
    L.w = w;
    L.bs = bs;
    tiles += (int)ceil_div(m, kMT) * L.tiles_n;
    off += (long)m * n + n;
  };
  layer(0, X, sxk, sxm, n_in, dZ1, 1, width, width, gW1, gb1);
  layer(1, H1, 1, width, width, dZ2, 1, width, width, gW2, gb2);
  layer(2, H2, 1, width, width, dY, syk, sym, n_out, gW3, gb3);
  p.total = off;
  F3D_LAUNCH(grad_partial_kernel, dim3((unsigned)tiles, (unsigned)p.slices), dim3(256), 0, st, p,
             part);
  F3D_LAUNCH(grad_reduce_kernel, dim3((unsigned)ceil_div(p.total, (int64_t)256)), dim3(256), 0, st,
             p, (const float*)part);
  return F3D_OK;
}

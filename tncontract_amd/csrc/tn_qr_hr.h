// A 64-column block of the Householder QR (tn_qr.hip) through its orthonormal
// factor instead of column by column: Cholesky QR in two passes, then the
// reflectors that Householder's method would have made, reconstructed from
// the orthonormal columns (Ballard, Demmel, Grigori, Jacquelin, Nguyen and
// Solomonik, IPDPS 2014).
//
// The register panels factor 8 columns per launch of one workgroup, two
// dependent grid launches after each, 400 us for 64 columns of 5120 rows; the
// matrix cores idle meanwhile.  Here the columns' long dimension only meets
// 64 x 64 matrices:
//   1. G = (P D)^T (P D) over row chunks (D: powers of two that bring the
//      columns' norms to [1, 2)), G = L L^T, Q1 = P D L^{-T} by the inverse X of
//      L and one step of refinement, Q1 += (P D - Q1 L^T) X^T: the inverse alone
//      leaves P D - Q1 L^T at cond(P D) eps (up to 2e-13 of a column's norm for
//      blocks that pass below), the refined one at rounding;
//   2. E = Q1^T Q1 - I (about cond(P D)^2 eps), N = its strict upper triangle
//      plus half its diagonal: Q = Q1 (I - N) is orthonormal and
//      P = Q R, R = (I + N) L^T D^{-1}, to O(|E|^2);
//   3. the top 64 rows Q_t: Q_t - S = Y_t U without pivoting, S_j = -sign of
//      the pivot, which is the sign dlarfg gives the diagonal of R; Y = the
//      reflectors ([Y_t; Q_b U^{-1}]), T = -U S Y_t^{-T}, and S R the R of
//      Householder's method.
// Every block that this cannot reproduce to rounding keeps the panels: *bad
// is raised, before anything of the matrix is overwritten, when |E| exceeds
// 1e-9, when a pivot is within 1e-12 of zero (its sign, so the sign of a row
// of R, would be rounding's) or within 1e-8 of one (a column that is zero
// below the pivot, whose reflector dlarfg leaves out), or for anything not
// finite.  The flag stays on the device: the panels' launches follow in the
// same stream and return at once while it is 0, and once it is raised the
// kernels here do, for the rest of the factorisation.  That is what a block
// that stays with the panels costs, about 12 us: 1280 x 640 triangular, whose
// first block does, 3.98 -> 4.11 ms.  A product of Gaussian factors of rank 0.6 n
// never does (what is left past the rank is rounding, well conditioned after
// D), the sites of an MPO-applied chain do part way: the QR sweep over 12 of
// them 8.1 -> 6.8 ms at chi = 64, 13.5 -> 8.9 ms at chi = 128.
#pragma once
#include "tn_internal.h"

namespace tn {

constexpr int HB = 64;         // columns of a block
constexpr int HCH = 16;        // row chunks of the Gram sums (at most)
constexpr int HROWS = 64;      // rows per workgroup of hr_apply
// Rows from the diagonal down that a block needs: the buffer that Q is formed in
// holds the 64 x 64 matrices from 256 rows on.  There it pays at every size: one
// block of 257 rows 311 us by the panels, 181 here, of 1024 rows 372 and 198, of
// 5120 rows 646 and 267 (blocks of 128 .. 255 rows in a taller matrix would gain
// as well: 300 x 128 502 -> 372 us).
constexpr int64_t HR_MIN_ROWS = 256;

typedef double hf64x4 __attribute__((ext_vector_type(4)));
typedef double hf64x4u __attribute__((ext_vector_type(4), aligned(8)));

struct HrWs {
  double *part, *G, *F, *X, *M, *d, *delta;
  int* bad;
};

__global__ void hr_reset(int* bad) { *bad = 0; }

// part[chunk] (64 x 64, column-major, entries of the tiles on and below the
// diagonal) = P^T P over the chunk's rows; P: rows x 64, column-major (ld).
// A wave takes 16 rows at a time: lane (lr, lk) holds rows 4 lk .. 4 lk + 3
// of columns 16 t + lr, t = 0 .. 3 (each column 128 bytes in a row), which
// are both operands of the tile products (the sum over rows is in the order
// that suits the loads).
__global__ void __launch_bounds__(256) hr_gram(const double* __restrict__ P, int64_t rows,
                                               int64_t ld, int nchunk, double* __restrict__ part,
                                               const int* __restrict__ bad, int when) {
  if (*bad != when) return;
  __shared__ double Gs[HB][HB + 1];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  hf64x4 acc[10];
#pragma unroll
  for (int i = 0; i < 10; ++i) acc[i] = hf64x4{0, 0, 0, 0};
  const int64_t groups = ceil_div(rows, 16);
  for (int64_t g = (int64_t)blockIdx.x * 4 + wave; g < groups; g += 4 * (int64_t)nchunk) {
    const int64_t r = 16 * g + 4 * lk;
    hf64x4 x[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const double* p = P + (int64_t)(16 * t + lr) * ld + r;
      if (16 * g + 16 <= rows) {
        x[t] = *(const hf64x4u*)p;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[t][e] = r + e < rows ? p[e] : 0.0;
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      int n = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j <= i; ++j, ++n)
          acc[n] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i][e], x[j][e], acc[n], 0, 0, 0);
    }
  }
  // the waves' sums in turn (fixed order)
  for (int w = 0; w < 4; ++w) {
    if (wave == w) {
      int n = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j <= i; ++j, ++n)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            double* q = &Gs[16 * j + lr][16 * i + lk + 4 * e];  // [column][row]
            *q = w == 0 ? acc[n][e] : *q + acc[n][e];
          }
    }
    __syncthreads();
  }
  double* out = part + (int64_t)blockIdx.x * HB * HB;
  for (int e = threadIdx.x; e < HB * HB; e += 256) {
    const int c = e >> 6, r = e & 63;
    if (r >> 4 >= c >> 4) out[e] = Gs[c][r];
  }
}

// Entry (r, c), r >= c, of the Gram: the chunks' sums in order.
__device__ __forceinline__ double hr_sum(const double* __restrict__ part, int nchunk, int r, int c) {
  double v[HCH];
#pragma unroll
  for (int k = 0; k < HCH; ++k) v[k] = k < nchunk ? part[k * HB * HB + c * HB + r] : 0.0;
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < HCH; ++k) s += v[k];
  return s;
}

// G (64 x 64) from the chunks' sums, over 16 CUs (one workgroup reading them
// all took 24 us).
__global__ void __launch_bounds__(256) hr_gram_sum(const double* __restrict__ part, int nchunk,
                                                   double* __restrict__ G,
                                                   const int* __restrict__ bad, int when) {
  if (*bad != when) return;
  const int e = blockIdx.x * 256 + threadIdx.x, c = e >> 6, r = e & 63;
  G[e] = r >= c ? hr_sum(part, nchunk, r, c) : hr_sum(part, nchunk, c, r);
}

// d_j = 2^-e_j with 4^e_j within a factor of two of G_jj; G (lower) = D G D;
// *delta: twice the smallest pivot of it that is kept (a dropped one raises
// bad through the second Gram).
__global__ void __launch_bounds__(256) hr_scale(const double* __restrict__ part, int nchunk,
                                                double* __restrict__ G, double* __restrict__ d,
                                                double* __restrict__ delta,
                                                const int* __restrict__ bad) {
  if (*bad) return;
  const int e = blockIdx.x * 256 + threadIdx.x, c = e >> 6, r = e & 63;
  if (r >= c) {
    const double g = hr_sum(part, nchunk, r, c);
    const double gr = hr_sum(part, nchunk, r, r), gc = hr_sum(part, nchunk, c, c);
    const int er = gr > 0.0 ? -(__builtin_amdgcn_frexp_exp(gr) >> 1) : 0;
    const int ec = gc > 0.0 ? -(__builtin_amdgcn_frexp_exp(gc) >> 1) : 0;
    const double v = __builtin_amdgcn_ldexp(g, er + ec);
    G[c * HB + r] = v;
    G[r * HB + c] = v;
    if (r == c) d[c] = __builtin_amdgcn_ldexp(1.0, ec);
  }
  if (e == 0) *delta = 2e-8;
}

// Out (rows x 64) = In (rows x 64) B, both column-major; B[i][c] =
// B0[i * 64 + c].  Out2 (null or a second copy, ld2).  Each
// wave 16 rows, as the transposed product (B^T In^T): In is read and Out
// written straight from and to memory, 128 bytes of a column at a time (more
// and shorter workgroups measured better: 64 rows 9 us against 128 rows 13.8
// us at 5120 rows).  In
// and Out may be the same array (a row is read before it is written, by the
// wave that writes it).
// SOLVE: Out = (In D) L^{-T} with B0 = X^T, X = L^{-1}, and one step of
// refinement against L (F: its lower triangle, column-major; D = diag(d)).  A
// product comes out in the layout of its operand, so the three of them chain in
// registers.
template <bool SOLVE>
__global__ void __launch_bounds__(256) hr_apply(const double* In, int64_t rows, int64_t ldi,
                                                const double* __restrict__ B0,
                                                const double* __restrict__ F,
                                                const double* __restrict__ d, double* Out,
                                                int64_t ldo, double* __restrict__ Out2,
                                                int64_t ld2, const int* __restrict__ bad) {
  if (*bad) return;
  __shared__ double Bs[HB][HB + 1];
  __shared__ double Ls[SOLVE ? HB : 1][HB + 1];  // L^T
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lk = lane >> 4;
  const int64_t r = (int64_t)blockIdx.x * HROWS + 16 * wave + lr;
  double x[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) x[k] = r < rows ? In[(int64_t)(4 * k + lk) * ldi + r] : 0.0;
  {
    // (every load of B before the first LDS store)
    constexpr int PER = HB * HB / 256;
    double v[PER], f[SOLVE ? PER : 1];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int e = threadIdx.x + 256 * k;
      v[k] = B0[e];
      if constexpr (SOLVE) f[k] = (e & 63) >= (e >> 6) ? F[e] : 0.0;
    }
    if constexpr (SOLVE) {
#pragma unroll
      for (int k = 0; k < 16; ++k) x[k] *= d[4 * k + lk];
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int e = threadIdx.x + 256 * k;
      Bs[e >> 6][e & 63] = v[k];
      if constexpr (SOLVE) Ls[e >> 6][e & 63] = f[k];
    }
  }
  __syncthreads();
  // acc += y M, lane (lr, lk) holding columns 4 k + lk (k = 0 .. 15) of row lr
  // of y and of acc (acc[i][e]: k = 4 i + e)
  hf64x4 acc[4];
  auto mul = [&](const double (*M)[HB + 1], const double (&y)[16]) {
#pragma unroll
    for (int k = 0; k < 16; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(M[4 * k + lk][16 * i + lr], y[k], acc[i], 0,
                                                      0, 0);
  };
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = hf64x4{0, 0, 0, 0};
  mul(Bs, x);
  if constexpr (SOLVE) {
    double q[16], y[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      q[k] = acc[k >> 2][k & 3];
      y[k] = -q[k];
      acc[k >> 2][k & 3] = x[k];
    }
    mul(Ls, y);
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      y[k] = acc[k >> 2][k & 3];
      acc[k >> 2][k & 3] = q[k];
    }
    mul(Bs, y);
  }
  if (r >= rows) return;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t c = 16 * i + lk + 4 * e;
      Out[c * ldo + r] = acc[i][e];
      if (Out2) Out2[c * ld2 + r] = acc[i][e];
    }
}

// Steps 2 and 3 on the block's top 64 rows, one workgroup of 8 waves; lane t
// of wave q holds row t, columns 8 q .. 8 q + 7 of each matrix.  V: Q1 on
// entry (its top 64 rows become Y_t), W: the block of the matrix (its top 64
// rows become S R and Y_t), M = (I - N) U^{-1} row-major, T row-major.  The
// LU goes panel by panel of 8 columns like cq_diag's Cholesky: wave b factors
// panel b alone (pivots and the panel's entries of the pivot row by
// readlane), the later waves then take its columns; the same column
// operations turn I - N into M.
constexpr int HC = 8;
__global__ void __launch_bounds__(512) hr_reflect(const double* __restrict__ G,
                                                  const double* __restrict__ F,
                                                  const double* __restrict__ d,
                                                  double* __restrict__ V, int64_t ldv,
                                                  double* __restrict__ W, int64_t ldw,
                                                  double* __restrict__ M, double* __restrict__ T,
                                                  int* bad) {
  if (*bad) return;
  __shared__ __attribute__((aligned(16))) double As[HB][HB + 2];  // [row][column]: N, then L^T D^{-1}
  __shared__ double Bs[HB][HB + 1];   // [column][row]: Q1's top rows, later N's rows
  __shared__ double Ls[HB][HB];       // columns of Y_t, zero on and above the diagonal
  __shared__ double Xs[2][HC][HB];    // a panel's columns of M, then of T
  __shared__ double sg[HB];
  __shared__ int flag;
  const int t = threadIdx.x & 63;
  const int q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (threadIdx.x == 0) flag = 0;
  __syncthreads();
  bool fine = true;
#pragma unroll
  for (int k = 0; k < HC; ++k) {
    const int c = HC * q + k;
    Bs[c][t] = V[(int64_t)c * ldv + t];
    const double e = G[c * HB + t] - (t == c ? 1.0 : 0.0);
    fine = fine && fabs(e) <= 1e-9;   // false for NaN
    As[t][c] = t < c ? e : (t == c ? 0.5 * e : 0.0);
  }
  __syncthreads();
  // a = Q_t = Q1_t - Q1_t N, x = I - N
  double a[HC], x[HC], acc[HC];
#pragma unroll
  for (int k = 0; k < HC; ++k) {
    const int c = HC * q + k;
    a[k] = Bs[c][t];
    x[k] = (t == c ? 1.0 : 0.0) - As[t][c];
    acc[k] = 0.0;
  }
#pragma unroll 4
  for (int i = 0; i < HC * q + HC; ++i) {
    const double v = Bs[i][t];
    const double2* n = (const double2*)&As[i][HC * q];
#pragma unroll
    for (int k = 0; k < HC; k += 2) {
      const double2 nk = n[k / 2];
      acc[k] = fma(v, nk.x, acc[k]);
      acc[k + 1] = fma(v, nk.y, acc[k + 1]);
    }
  }
#pragma unroll
  for (int k = 0; k < HC; ++k) a[k] -= acc[k];
  // R = (I + N) L^T D^{-1}: column c's entries i <= c
  double rr[HC];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < HC; ++k) {
    const int c = HC * q + k;
    const double n = As[t][c];
    rr[k] = t <= c ? F[t * HB + c] * (1.0 / d[c]) : 0.0;  // (L^T D^{-1})[t][c]: d = 2^e
    Bs[c][t] = n;                                  // N[t][c]
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < HC; ++k) As[t][HC * q + k] = rr[k];
  __syncthreads();
#pragma unroll 4
  for (int i = 0; i < HC * q + HC; ++i) {
    const double v = Bs[i][t];                     // N[t][i]
    const double2* n = (const double2*)&As[i][HC * q];
#pragma unroll
    for (int k = 0; k < HC; k += 2) {
      const double2 nk = n[k / 2];
      rr[k] = fma(v, nk.x, rr[k]);
      rr[k + 1] = fma(v, nk.y, rr[k + 1]);
    }
  }
  // LU of Q_t - S with S chosen on the way
  double sgn[HC];
  auto factor = [&](int b) {
#pragma unroll
    for (int kc = 0; kc < HC; ++kc) {
      const int c = HC * b + kc;
      const double al = readlane_f64(a[kc], c);
      const double s = al >= 0.0 ? -1.0 : 1.0;
      fine = fine && fabs(al) >= 1e-12 && fabs(al) <= 1.0 - 1e-8;
      const double piv = al - s;            // 1 <= |piv| <= 2
      double inv = __builtin_amdgcn_rcp(piv);  // ~2^-23, squared by each step
      inv = fma(inv, fma(-piv, inv, 1.0), inv);
      inv = fma(inv, fma(-piv, inv, 1.0), inv);
      sgn[kc] = s;
      const double l = t > c ? a[kc] * inv : 0.0;
      x[kc] *= inv;
#pragma unroll
      for (int k = kc + 1; k < HC; ++k) {
        const double u = readlane_f64(a[k], c);
        a[k] = fma(-l, u, a[k]);
        x[k] = fma(-x[kc], u, x[k]);
      }
      a[kc] = t > c ? l : (t == c ? piv : a[kc]);
      Ls[c][t] = l;
      Xs[b & 1][kc][t] = x[kc];
      if (t == 0) sg[c] = s;
    }
  };
  if (q == 0) factor(0);
#pragma unroll 1
  for (int b = 0; b < HB / HC; ++b) {
    __syncthreads();  // panel b published
    if (q > b) {
#pragma unroll
      for (int kc = 0; kc < HC; ++kc) {
        const int c = HC * b + kc;
        const double l = Ls[c][t], xc = Xs[b & 1][kc][t];
#pragma unroll
        for (int k = 0; k < HC; ++k) {
          const double u = readlane_f64(a[k], c);
          a[k] = fma(-l, u, a[k]);
          x[k] = fma(-xc, u, x[k]);
        }
      }
    }
    if (q == b + 1) factor(b + 1);
  }
  if (!fine) flag = 1;
  __syncthreads();
  if (flag) {
    if (threadIdx.x == 0) *bad = 1;
    return;
  }
  // T Y_t^T = -U S, column by column: T_c = -S_c U_c - sum_{j < c} T_j Y_t[c][j]
  double tc[HC];
#pragma unroll
  for (int k = 0; k < HC; ++k) tc[k] = t <= HC * q + k ? -sgn[k] * a[k] : 0.0;
#pragma unroll 1
  for (int b = 0; b < HB / HC; ++b) {
    if (q == b) {
#pragma unroll
      for (int kc = 0; kc < HC; ++kc) {
#pragma unroll
        for (int j = 0; j < kc; ++j) tc[kc] = fma(-tc[j], Ls[HC * b + j][HC * b + kc], tc[kc]);
        Xs[b & 1][kc][t] = tc[kc];
      }
    }
    __syncthreads();
    if (q > b) {
#pragma unroll
      for (int kc = 0; kc < HC; ++kc) {
        const double v = Xs[b & 1][kc][t];
#pragma unroll
        for (int k = 0; k < HC; ++k) tc[k] = fma(-v, Ls[HC * b + kc][HC * q + k], tc[k]);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < HC; ++k) {
    const int c = HC * q + k;
    M[t * HB + c] = x[k];
    T[t * HB + c] = t <= c ? tc[k] : 0.0;
    V[(int64_t)c * ldv + t] = t > c ? a[k] : (t == c ? 1.0 : 0.0);
    W[(int64_t)c * ldw + t] = t > c ? a[k] : sg[t] * rr[k];
  }
}

}  // namespace tn

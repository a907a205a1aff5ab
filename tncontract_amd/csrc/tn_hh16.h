// Householder QR of a small matrix by one workgroup, a column per row of 16
// lanes: lane l of column q holds rows l, l + 16, ... in registers (NI of
// them; ni = ceil(rows / 16) are used).  Shared by the small QR (tn_qr.hip) and
// the small SVD (tn_svd.hip).
#pragma once
#include "tn_common.h"
#include "tn_jacobi.h"

namespace tn {

// Sum over the lane's row of 16.
__device__ __forceinline__ double row16_sum(double v) {
  v += dpp_f64<0xB1, 0xF>(v);   // quad_perm [1,0,3,2]
  v += dpp_f64<0x4E, 0xF>(v);   // quad_perm [2,3,0,1]
  v += dpp_f64<0x141, 0xF>(v);  // row_half_mirror
  v += dpp_f64<0x140, 0xF>(v);  // row_mirror
  return v;
}

// Whether a reflector's squared norm below the pivot has lost digits to
// underflow that count against the pivot alpha; then the column is taken times
// kHhUp (the squares of FP64's smallest numbers and of the largest that come
// here stay in range), and in products with other columns those times kHhUpX.
// (A column left with rounding only by the reflectors before it shrinks by
// 1e-16 from column to column, down to there.)
constexpr double kHhUp = 0x1p700, kHhUpX = 0x1p300;
__device__ __forceinline__ bool hh_underflows(double n2, double alpha) {
  return n2 < 0x1p-960 && fabs(alpha) < 0x1p-400;
}

// k reflectors (k <= 16 NP; dlarfg's convention, beta = -sign(alpha) norm) of
// the columns x, one barrier a column: column j goes to LDS (two buffers of 16
// NI doubles), every column sums its own dot with it below the pivot and the
// norm, and v . x_q = x_q[j] + scale (that dot).  On return x holds R on and
// above the diagonal and the reflectors below it.
template <int NI, int NP>
__device__ __forceinline__ void hh16_factor(double (&x)[NI], int q, int l, int k, int ni,
                                            double (*vcol)[16 * NI], double* taus) {
  const int lane = threadIdx.x & 63;
  for (int j = 0; j < k; ++j) {
    double* vc = vcol[j & 1];
    if (q == j) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
        if (i < ni) vc[l + 16 * i] = x[i];
    }
    lds_barrier();
    double v[NI], n2 = 0.0, dot = 0.0;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int r = l + 16 * i;
      v[i] = (i < ni && r > j) ? vc[r] : 0.0;
      n2 = fma(v[i], v[i], n2);
      dot = fma(v[i], x[i], dot);
    }
    n2 = row16_sum(n2);
    dot = row16_sum(dot);
    double alpha = vc[j], up = 1.0, down = 1.0;
    if (hh_underflows(n2, alpha)) {
      up = kHhUp;
      down = 1.0 / kHhUpX;
      alpha *= up;
      n2 = dot = 0.0;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        v[i] *= up;
        n2 = fma(v[i], v[i], n2);
        dot = fma(v[i], x[i] * kHhUpX, dot);
      }
      n2 = row16_sum(n2);
      dot = row16_sum(dot);
    }
    // this column's pivot-row entry, held by lane j % 16 of its row
    double pt = x[0];
#pragma unroll
    for (int p = 1; p < NP; ++p)
      if (j >= 16 * p) pt = x[p];
    const double pv = __shfl(pt, (lane & 48) | (j & 15), 64);
    double tj = 0.0, scale = 0.0, beta = alpha;
    if (n2 != 0.0) {  // NaN too: it has to reach R
      const double h = sqrt(alpha * alpha + n2);
      beta = alpha >= 0.0 ? -h : h;
      tj = (beta - alpha) / beta;
      scale = 1.0 / (alpha - beta);
    }
    if (q == j) {
      if (l == 0) taus[j] = tj;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int r = l + 16 * i;
        x[i] = r > j ? x[i] * up * scale : (r == j ? beta / up : x[i]);
      }
    } else if (q > j) {
      const double w = tj * fma(scale * down, dot, pv), ws = w * scale;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int r = l + 16 * i;
        x[i] = r == j ? x[i] - w : fma(-ws, v[i], x[i]);
      }
    }
  }
}

// x <- H_0 ... H_{top} x for a column x, from the reflectors in W (column j at
// W + j * ld), within the lane's row of 16 (no barrier).
template <int NI>
__device__ __forceinline__ void hh16_apply_q(double (&x)[NI], int l, int top, int ni,
                                             const double* W, int ld, const double* taus) {
  for (int j = top; j >= 0; --j) {
    double v[NI], dot = 0.0;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int r = l + 16 * i;
      v[i] = (i < ni && r > j) ? W[j * ld + r] : (r == j ? 1.0 : 0.0);
      dot = fma(v[i], x[i], dot);
    }
    const double w = taus[j] * row16_sum(dot);
#pragma unroll
    for (int i = 0; i < NI; ++i) x[i] = fma(-w, v[i], x[i]);
  }
}

}  // namespace tn

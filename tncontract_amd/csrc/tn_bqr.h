// Batched Householder QR of many independent column-major L x k matrices
// (k <= L <= kQrRows), panel by panel over all of them at once, and the
// application of their Q factors: the preconditioner of the batched one-sided Jacobi
// (tn_batched.hip).  One-sided Jacobi on the rows of R instead of the
// columns of X = Q R converges in far fewer sweeps on graded and
// rank-deficient matrices (Drmac & Veselic, "New fast and accurate Jacobi
// SVD algorithm I", SIAM J. Matrix Anal. Appl. 29 (2008)): the k - rank
// rows of R that carry only rounding are negligible from the start.
//
// Per panel of QNB = 16 columns (LAPACK dgeqrf's steps with dlarfg's
// reflector convention, beta = -sign(alpha) ||x||, and dlarft's forward
// column-wise T), every job's panel in the same two launches, by workgroups
// that hold all rows below the panel's first one in registers, as 16 x 16
// tiles in the fragment layout of v_mfma_f64_16x16x4 (column lane % 16; rows
// 4 (lane / 16) + e, e = 0 .. 3: 32 contiguous bytes a lane):
//   * bqr_panel, one workgroup per job, one barrier per reflector: a column
//     reaches the others by DPP, and one exchange through LDS sums its dots
//     with all 16 columns (its norm, the update of the later columns and the
//     earlier reflectors' products that T is made of);
//   * bqr_trail, one workgroup per 16 trailing columns of a job: C -= V T^T
//     V^T C, C read once and written once.
// What bounds both is latency: few workgroups run once the small jobs are
// done, so the rows are spread over all waves of a workgroup (the panel's over
// 8, whose reflectors' scalar work is repeated in every wave) and every load of
// a tile is issued at once.  Averaged over the panels of 32 jobs of sizes up to
// 1022, the trailing update takes 18.5 us, the application of Q 17.5 and the
// panel 27.8; with 4 waves per 64 columns staging V through LDS 64 rows at a
// time, and two barriered block sums per reflector, 79, 79 and 47.5.
#pragma once
#include "tn_common.h"
#include "tn_hh16.h"
#include "tn_jacobi.h"

#include <utility>

namespace tn {

constexpr int QNB = 16;         // reflectors per panel (T is QNB x QNB)
constexpr int kQrRows = 1024;   // rows a workgroup holds in registers (64 per wave)
constexpr int QNW = kQrRows / 64;
constexpr int QNT = 64 * QNW;

typedef double f64x4q __attribute__((ext_vector_type(4)));

struct QJob {
  int64_t x;    // the job's L x k matrix (column-major, ld = L): on exit R on and
                // above the diagonal, the reflectors below it
  int64_t r;    // the rows of R as k vectors of length k
  int64_t qz;   // Q [Z; 0]: L x ncols, column-major
  int64_t tf;   // the panels' T factors, QNB x QNB row-major each
  int64_t z;    // the job's rotation accumulator Z (k x k, columns contiguous)
  int32_t L, k;
  int32_t job;  // index of the job in the batch
  int32_t pad;
};

// A pair of neighbouring doubles, 8-byte aligned (odd column strides).
typedef double f64x2q __attribute__((ext_vector_type(2), aligned(8)));

// Value of lane LANE of this lane's row of 16 (DPP row_newbcast).
template <int LANE>
__device__ __forceinline__ double dpp_row_bcast(double v) {
  return __longlong_as_double(__builtin_amdgcn_update_dpp(
      0ll, __double_as_longlong(v), 0x150 + LANE, 0xf, 0xf, true));
}

// Sum over the four lanes lane % 16 + 16 k (the same bits in all four):
// swapping the odd rows of 16 (then the upper half) of one copy with the even
// rows (lower half) of another leaves the two values to add in every lane.
__device__ __forceinline__ double column_sum(double v) {
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  long long u = __double_as_longlong(v);
  u2 lo = __builtin_amdgcn_permlane16_swap((unsigned)u, (unsigned)u, false, false);
  u2 hi = __builtin_amdgcn_permlane16_swap((unsigned)(u >> 32), (unsigned)(u >> 32), false, false);
  v = __longlong_as_double(((long long)hi[0] << 32) | lo[0]) +
      __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
  u = __double_as_longlong(v);
  lo = __builtin_amdgcn_permlane32_swap((unsigned)u, (unsigned)u, false, false);
  hi = __builtin_amdgcn_permlane32_swap((unsigned)(u >> 32), (unsigned)(u >> 32), false, false);
  return __longlong_as_double(((long long)hi[0] << 32) | lo[0]) +
         __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
}

// C[p0:L, c0:c1) -= V op(T) V^T C[p0:L, c0:c1) for c1 - c0 <= 16 (column-
// major C, ld = ldc; called by the whole workgroup of 16 waves), V the nb
// reflectors of the panel at column p0 of X (ld = L; unit diagonal, zero above
// it), op(T) = T^T if trans (applying Q^T) else T.  A[m][k] of the MFMA is in
// lane m + 16 k, B[k][n] in lane n + 16 k, D[k + 4 e][n] in element e of lane
// n + 16 k; the update's A rows are permuted so that D's rows are C's.
__device__ __forceinline__ void qr_block_reflect(const double* __restrict__ X, int L, int p0,
                                                 int nb, const double (*Ts)[QNB + 1], bool trans,
                                                 double* __restrict__ C, int64_t ldc, int c0,
                                                 int c1, double (*part)[256]) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int lr = lane & 15, lk = lane >> 4;
  const int R0 = p0 + 64 * wave, rb = R0 + 4 * lk;
  const bool act = R0 < L;
  const bool cok = c0 + lr < c1;
  double* Cc = C + (int64_t)(cok ? c0 + lr : c0) * ldc;
  // every row of the wave's exists, below the panel's triangle, for 16
  // columns and reflectors: no bounds test
  const bool full = wave > 0 && R0 + 64 <= L && c1 - c0 == 16 && nb == QNB;
  double c[4][4], w[4][4];
  f64x4q y = {0.0, 0.0, 0.0, 0.0}, y1 = {0.0, 0.0, 0.0, 0.0};
  if (act) {
    double v[4][4];
    const double* Vc = X + (int64_t)(p0 + min(lr, nb - 1)) * L;
    if (full) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          const f64x2q a = *(const f64x2q*)(Vc + rb + 16 * t + e);
          const f64x2q b = *(const f64x2q*)(Cc + rb + 16 * t + e);
          v[t][e] = a[0];
          v[t][e + 1] = a[1];
          c[t][e] = b[0];
          c[t][e + 1] = b[1];
        }
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = rb + 16 * t + e, d = row - p0 - lr;
          v[t][e] = (lr < nb && row < L && d >= 0) ? (d == 0 ? 1.0 : Vc[row]) : 0.0;
          c[t][e] = (cok && row < L) ? Cc[row] : 0.0;
        }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        y = __builtin_amdgcn_mfma_f64_16x16x4f64(v[t][e], c[t][e], y, 0, 0, 0);
        y1 = __builtin_amdgcn_mfma_f64_16x16x4f64(v[t][e + 1], c[t][e + 1], y1, 0, 0, 0);
      }
    // V again, as the update's operand: row R0 + 16 t + 4 (lr % 4) + lr / 4 of
    // reflector lk + 4 u (in flight across the reduction)
    const int r2 = R0 + 4 * (lr & 3) + (lr >> 2);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int q = lk + 4 * u;
      const double* Vq = X + (int64_t)(p0 + min(q, nb - 1)) * L;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int row = r2 + 16 * t, d = row - p0 - q;
        if (full)
          w[t][u] = Vq[row];
        else
          w[t][u] = (q < nb && row < L && d >= 0) ? (d == 0 ? 1.0 : Vq[row]) : 0.0;
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) part[wave][64 * e + lane] = y[e] + y1[e];
  }
  lds_barrier();
  // Y summed over the waves: four threads an element, four partials each
  {
    const int q = tid & 255, g = tid >> 8, nw = min((L - p0 + 63) >> 6, QNW);
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (4 * g + i < nw) s += part[4 * g + i][q];
    lds_barrier();
    part[g][q] = s;
  }
  lds_barrier();
  if (!act) return;
  // Y2 = op(T) Y: element u of y holds Y[lk + 4u][lr], the B operand of
  // the k-step whose summation indices are lk + 4u
  f64x4q y2 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int kk = lk + 4 * u, q = 64 * u + lane;
    const double yu = (part[0][q] + part[1][q]) + (part[2][q] + part[3][q]);
    const double a = trans ? Ts[kk][lr] : Ts[lr][kk];
    y2 = __builtin_amdgcn_mfma_f64_16x16x4f64(a, yu, y2, 0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    f64x4q d = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int u = 0; u < 4; ++u)
      d = __builtin_amdgcn_mfma_f64_16x16x4f64(w[t][u], y2[u], d, 0, 0, 0);
    if (full) {
#pragma unroll
      for (int e = 0; e < 4; e += 2)
        *(f64x2q*)(Cc + rb + 16 * t + e) = f64x2q{c[t][e] - d[e], c[t][e + 1] - d[e + 1]};
    } else if (cok) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (rb + 16 * t + e < L) Cc[rb + 16 * t + e] = c[t][e] - d[e];
    }
  }
}

constexpr int QPW = 8;                        // waves of bqr_panel
constexpr int QPT = kQrRows / (16 * QPW);     // 16-row tiles a wave holds

struct QPanelLds {
  double part[2][QPW][QNB];   // the waves' dots of a column with all 16
  double row[2][QNB];         // the panel's row at the pivot
  double dots[QNB][QNB];      // [JJ][c] = v_JJ . (column c): T's inner products for c < JJ
  double tau[QNB];
};

// Reflector JJ of the panel (nb columns; JJ a compile-time index: the lane a
// column is broadcast from): formed from column JJ, applied to the later
// columns.  P[t][e]: the lane's rows of column lane % 16, nt tiles of which
// exist.  x . P_c below the pivot comes from one exchange for every column c,
// and the reflector v = (1; scal x) gives v . P_c = P[JJ][c] + scal x . P_c.
// Columns keep x; myscal is the scal of this lane's column once it is a
// reflector, 1 before.
template <int JJ>
__device__ __forceinline__ void qr_panel_step(double (&P)[QPT][4], int nt, int nb, QPanelLds& sm,
                                              double& myscal) {
  if (JJ >= nb) return;  // block-uniform
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
  double x[QPT][4], acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int t = 0; t < QPT; ++t) {
    if (t >= nt) break;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[t][e] = dpp_row_bcast<JJ>(P[t][e]);
    if (t == 0 && wave == 0) {
      // the panel's triangle: rows 4 lk + e <= JJ of the first tile
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (4 * lk + e <= JJ) x[0][e] = 0.0;
      if (lk == JJ / 4) sm.row[JJ & 1][lr] = P[0][JJ & 3] * myscal;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = fma(x[t][e], P[t][e], acc[e]);
  }
  const double a = column_sum((acc[0] + acc[1]) + (acc[2] + acc[3]));
  if (lk == 0) sm.part[JJ & 1][wave][lr] = a;
  lds_barrier();
  double d = column_sum(sm.part[JJ & 1][2 * lk][lr] + sm.part[JJ & 1][2 * lk + 1][lr]);
  const double prow = sm.row[JJ & 1][lr];
  double s = dpp_row_bcast<JJ>(d), alpha = dpp_row_bcast<JJ>(prow), up = 1.0, down = 1.0;
  if (hh_underflows(s, alpha)) {  // block-uniform
    up = kHhUp;
    down = 1.0 / kHhUpX;
    alpha *= up;
    double b = 0.0, c = 0.0;
#pragma unroll
    for (int t = 0; t < QPT; ++t) {
      if (t >= nt) break;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[t][e] *= up;
        b = fma(x[t][e], P[t][e] * kHhUpX, b);
        c = fma(x[t][e], x[t][e], c);
        if (lr == JJ && (t > 0 || wave > 0 || 4 * lk + e > JJ)) P[t][e] = x[t][e];
      }
    }
    // (the pivot column's lane: the norm of the scaled column)
    b = column_sum(lr == JJ ? c : b);
    lds_barrier();
    if (lk == 0) sm.part[JJ & 1][wave][lr] = b;
    lds_barrier();
    d = column_sum(sm.part[JJ & 1][2 * lk][lr] + sm.part[JJ & 1][2 * lk + 1][lr]);
    s = dpp_row_bcast<JJ>(d);
  }
  double beta = alpha, tau = 0.0, scal = 1.0;
  if (s != 0.0) {
    beta = -copysign(sqrt(fma(alpha, alpha, s)), alpha);
    tau = (beta - alpha) / beta;
    scal = 1.0 / (alpha - beta);
  }
  const double vp = fma(scal * myscal * down, d, prow);  // v . (column c, or reflector c)
  if (wave == 0 && lk == 0) {
    sm.dots[JJ][lr] = vp;
    sm.tau[JJ] = tau;
  }
  const double f = lr > JJ ? -tau * vp : 0.0, g = f * scal;
#pragma unroll
  for (int t = 0; t < QPT; ++t) {
    if (t >= nt) break;
#pragma unroll
    for (int e = 0; e < 4; ++e) P[t][e] = fma(g, x[t][e], P[t][e]);
  }
  if (lr == JJ) myscal = scal;
  if (wave == 0 && lk == JJ / 4) P[0][JJ & 3] = lr == JJ ? beta / up : P[0][JJ & 3] + f;
}

template <int... J>
__device__ __forceinline__ void qr_panel(std::integer_sequence<int, J...>, double (&P)[QPT][4],
                                         int nt, int nb, QPanelLds& sm, double& myscal) {
  (qr_panel_step<J>(P, nt, nb, sm, myscal), ...);
}

// T of the panel's nb reflectors (zero past them), row-major at out, by wave 0
// (lane i: row i): T[0:j, j] = -tau_j T[0:j, 0:j] (V^T v_j)[0:j], T[j][j] =
// tau_j.
__device__ __forceinline__ void qr_panel_t(const QPanelLds& sm, int nb, double* __restrict__ out) {
  const int i = threadIdx.x & 15;
  double T[QNB];
#pragma unroll
  for (int c = 0; c < QNB; ++c) T[c] = 0.0;
#pragma unroll 1
  for (int j = 0; j < nb; ++j) {
    double t = 0.0;
#pragma unroll
    for (int c = 0; c < QNB; ++c) t = fma(T[c], c < j ? sm.dots[j][c] : 0.0, t);
    const double tau = sm.tau[j], v = i < j ? -tau * t : (i == j ? tau : 0.0);
#pragma unroll
    for (int c = 0; c < QNB; ++c) T[c] = c == j ? v : T[c];
  }
  if (threadIdx.x < 16) {
#pragma unroll
    for (int c = 0; c < QNB; ++c) out[i * QNB + c] = T[c];
  }
}

// Panel p of every job (one workgroup per job that has it; items: the
// indices into qjobs): the panel's QNB columns factored in registers, the
// reflectors and R's entries stored back, T into Tf.
__global__ void __launch_bounds__(64 * QPW) bqr_panel(double* __restrict__ Wv,
                                                      double* __restrict__ Tf,
                                                      const QJob* __restrict__ qjobs,
                                                      const int* __restrict__ items, int p) {
  __shared__ QPanelLds sm;
  const QJob Q = qjobs[items[blockIdx.x]];
  const int L = Q.L, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lr = lane & 15;
  const int p0 = p * QNB, nb = min(QNB, Q.k - p0), nt = (L - p0 + 16 * QPW - 1) / (16 * QPW);
  double* Xc = Wv + Q.x + (int64_t)(p0 + min(lr, nb - 1)) * L;
  const int rb = p0 + 16 * wave + 4 * (lane >> 4);  // tile t: 16 QPW t rows on
  double P[QPT][4];
#pragma unroll
  for (int t = 0; t < QPT; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = rb + 16 * QPW * t + e;
      P[t][e] = (row < L && lr < nb) ? Xc[row] : 0.0;
    }
  double myscal = 1.0;
  qr_panel(std::make_integer_sequence<int, QNB>{}, P, nt, nb, sm, myscal);
  if (lr < nb) {
#pragma unroll
    for (int t = 0; t < QPT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = rb + 16 * QPW * t + e;
        if (row < L) Xc[row] = row > p0 + lr ? P[t][e] * myscal : P[t][e];
      }
  }
  // (dots and tau are wave 0's own writes)
  if (tid < 64) qr_panel_t(sm, nb, Tf + Q.tf + (int64_t)p * (QNB * QNB));
}

// Columns of a job in groups of 16 (one workgroup): item = (index into qjobs,
// group).
struct QItem {
  int32_t q, g;
};

// Trailing update after panel p: the group's columns (after the panel) of
// X get C -= V T^T V^T C.
__global__ void __launch_bounds__(QNT) bqr_trail(double* __restrict__ Wv,
                                                 const double* __restrict__ Tf,
                                                 const QJob* __restrict__ qjobs,
                                                 const QItem* __restrict__ items, int p) {
  __shared__ double Ts[QNB][QNB + 1];
  __shared__ double part[QNW][256];
  const QItem it = items[blockIdx.x];
  const QJob Q = qjobs[it.q];
  const int tid = threadIdx.x;
  const int p0 = p * QNB, nb = min(QNB, Q.k - p0);
  const int c0 = p0 + nb + QNB * it.g, c1 = min(Q.k, c0 + QNB);
  // (the reduction's barriers order Ts before its use)
  if (tid < QNB * QNB) Ts[tid >> 4][tid & 15] = Tf[Q.tf + (int64_t)p * (QNB * QNB) + tid];
  double* X = Wv + Q.x;
  qr_block_reflect(X, Q.L, p0, nb, Ts, true, X, Q.L, c0, c1, part);
}

// The rows of R as vectors: Rv[c * k + i] = R[c][i] (i >= c), 0 below.
__global__ void __launch_bounds__(256) bqr_rvec(double* __restrict__ Wv,
                                                const QJob* __restrict__ qjobs) {
  const QJob Q = qjobs[blockIdx.y];
  const int64_t kk = (int64_t)Q.k * Q.k;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < kk; e += (int64_t)gridDim.x * 256) {
    const int64_t c = e / Q.k, i = e - c * Q.k;
    Wv[Q.r + e] = i >= c ? Wv[Q.x + i * Q.L + c] : 0.0;
  }
}

// Q [Z; 0] for the columns c < ncols of Z in the order perm (column-major,
// ld = L): first the copy (grid-wide), then bqr_apply per panel.
__global__ void __launch_bounds__(256) bqr_qz_init(double* __restrict__ QZ,
                                                   const double* __restrict__ Zb,
                                                   const QJob* __restrict__ qjobs,
                                                   const int* __restrict__ perm,
                                                   const int64_t* __restrict__ sbase,
                                                   const int* __restrict__ ncols) {
  const QJob Q = qjobs[blockIdx.y];
  const int nc = ncols[Q.job];
  const int64_t tot = (int64_t)Q.L * nc;
  const int* pm = perm + sbase[Q.job];
  const double* Z = Zb + Q.z;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < tot; e += (int64_t)gridDim.x * 256) {
    const int64_t c = e / Q.L, i = e - c * Q.L;
    QZ[Q.qz + e] = i < Q.k ? Z[(int64_t)pm[c] * Q.k + i] : 0.0;
  }
}

// Panel p's block reflector applied to the group's columns of Q Z (panels in
// reverse order make Q [Z; 0]); groups at or past the job's ncols exit.
__global__ void __launch_bounds__(QNT) bqr_apply(const double* __restrict__ Wv,
                                                 const double* __restrict__ Tf,
                                                 const QJob* __restrict__ qjobs,
                                                 const QItem* __restrict__ items,
                                                 const int* __restrict__ ncols, int p,
                                                 double* __restrict__ QZ) {
  __shared__ double Ts[QNB][QNB + 1];
  __shared__ double part[QNW][256];
  const QItem it = items[blockIdx.x];
  const QJob Q = qjobs[it.q];
  const int nc = ncols[Q.job];
  const int c0 = QNB * it.g, c1 = min(nc, c0 + QNB);
  if (c0 >= c1) return;  // block-uniform
  const int tid = threadIdx.x;
  const int p0 = p * QNB, nb = min(QNB, Q.k - p0);
  if (tid < QNB * QNB) Ts[tid >> 4][tid & 15] = Tf[Q.tf + (int64_t)p * (QNB * QNB) + tid];
  qr_block_reflect(Wv + Q.x, Q.L, p0, nb, Ts, false, QZ + Q.qz, Q.L, c0, c1, part);
}

}  // namespace tn

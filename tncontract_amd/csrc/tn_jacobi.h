// Pair-step building blocks of the one-sided block Jacobi (Hestenes) shared
// by the SVD and PSD eigensolver (tn_svd.hip) and the batched truncation
// (tn_batched.hip): vectors in blocks of 16, pairs of blocks (32 vectors)
// scheduled round-robin (circle method), per pair a 32 x 32 Gram matrix
// diagonalised by one cyclic sweep of two-sided Jacobi in LDS and applied
// to the pair's vectors by MFMA.
#pragma once
#include "tn_common.h"

namespace tn {

constexpr int JB = 16;       // vectors per block
constexpr int J2 = 2 * JB;   // pair width

__device__ __forceinline__ int rr_block(int pos, int step, int nblk) {
  return pos == 0 ? 0 : 1 + (pos - 1 + step) % (nblk - 1);
}

// pair pi at step s -> blocks (I, J)
__device__ __forceinline__ void pair_blocks(int pi, int s, int nblk, int& I, int& J) {
  I = rr_block(pi, s, nblk);
  J = rr_block(nblk - 1 - pi, s, nblk);
}

__device__ __forceinline__ int64_t pair_vec(int c, int I, int J) {
  return c < JB ? (int64_t)I * JB + c : (int64_t)J * JB + (c - JB);
}

// Whether step s of a sweep over nblk blocks rotates all 496 pairs of its 32
// vectors (31 rounds), or only the 256 pairs across the two blocks (16
// rounds).  A block meets every other one in a sweep, and its inner pairs are
// near convergence already when they have just been rotated: simulated on
// Gaussian, graded, clustered and rank-deficient matrices of 96 .. 512
// vectors, inner pairs at every fourth step need the sweeps that inner pairs
// at every step need (a third of the cases one more) with 0.64 of the rounds;
// inner pairs once a sweep 1 to 3 more sweeps.  Up to four blocks (three
// steps a sweep) the rounds saved do not pay for the added sweeps' launches.
// Measured: SVDs of 512 x 2560 19.1 -> 16.9 ms, of 254 x 636 3.35 -> 3.09 ms,
// with errors against 64 bits no larger.
__host__ __device__ __forceinline__ bool inner_step(int s, int nblk) {
  return nblk <= 4 || (s & 3) == 0;
}
__host__ __device__ __forceinline__ int step_rounds(bool inner) { return inner ? J2 - 1 : JB; }

typedef double f64x4 __attribute__((ext_vector_type(4)));

// Workgroup barrier that orders LDS accesses only.  __syncthreads() also
// fences global memory, which on gfx9 means waiting for every outstanding
// global load (one counter for loads and stores); this barrier lets loads
// issued before it stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Scale of a matrix whose vectors meet the Jacobi.  Squared norms and inner
// products of entries around 2^(+-500) leave FP64's range: the norms are then
// lost, and pair_rotates' lower limits would leave pairs alone whose vectors
// are as long as any other.  The vectors are therefore multiplied by the power
// of two that brings their largest entry to [0.5, 1) when its exponent is
// beyond a limit (kScaleExp for matrices whose entries are squared), and the
// singular values by its inverse: exact, and everything within the limit keeps
// its bits.  Codes: entry_code(x) = exponent + 2048, 0 for what has none (0,
// inf, NaN); code_scale(largest code) = the exponent to take out.
constexpr int kScaleExp = 200;
__device__ __forceinline__ int entry_code(double x) {
  return x != 0.0 && fabs(x) < INFINITY ? __builtin_amdgcn_frexp_exp(x) + 2048 : 0;
}
__device__ __forceinline__ int code_scale(int code, int limit = kScaleExp) {
  const int e = code - 2048;
  return code == 0 || abs(e) <= limit ? 0 : e;
}

constexpr int EIG_NT = 512;  // threads of a pair eigensolve (8 waves)
constexpr int EIG_NW = EIG_NT / 64;
constexpr int GPAD = 2;      // G row padding: rows stay 16-byte aligned
// Exponents of the pair's squared norms up to which products of two Gram
// entries (and of tol^2) stay inside FP64's range unscaled.
constexpr int EIG_RANGE = 400;

struct EigLds {
  // the pair Gram in circle positions (eig_pos), ping-pong over the rounds
  __attribute__((aligned(16))) double G[2][J2][J2 + GPAD];
  __attribute__((aligned(16))) double cs[2][JB][2];  // (c, s) of the 16 rotations of a round
  double Q[J2][J2 + 1];
  float red[EIG_NW];
  int wide;  // a squared norm beyond 2^(+-EIG_RANGE): the rounds scale every pair
};

// Circle position of index v: slot s holds the pair (s, 31 - s), its first
// member at position 2 s and its second at 2 s + 1.
__device__ __forceinline__ int eig_pos(int v) { return v < JB ? 2 * v : 2 * (J2 - 1 - v) + 1; }

// Largest normalised off-diagonal over the pair, encoded for atomicMax.
__device__ __forceinline__ unsigned long long dbits(double x) {
  return (unsigned long long)__double_as_longlong(x);
}

// The pair's Gram entries G_pq, G_pp, G_qq scaled by the same power of two
// 2^-e (exactly), e the exponent of max(G_pp, G_qq): the rotation test and
// the convergence measure then square numbers of order one, never the tiny
// entries of nearly-null vectors, whose squares underflow FP64.
__device__ __forceinline__ void pair_scaled(double gpq, double gpp, double gqq, double& spq,
                                            double& spp, double& sqq) {
  const int e = __builtin_amdgcn_frexp_exp(fmax(gpp, gqq));
  spq = __builtin_amdgcn_ldexp(gpq, -e);
  spp = __builtin_amdgcn_ldexp(gpp, -e);
  sqq = __builtin_amdgcn_ldexp(gqq, -e);
}

// Rotation predicate of a pair (l, h) from G_lh, G_ll, G_hh: G_lh^2 > tol^2
// G_ll G_hh on the scaled entries, and one of the two vectors not negligible
// (squared norm > neg2).  The convergence measure eig_off counts the pairs for
// which it holds at tol; the rounds rotate those for which it holds at tol / 4
// (rot_coef_v; rot_coef_n tests the first two conditions alone).  A vector
// whose squared norm underflows is not rotated with one 2^40 times longer: the
// norm is lost and its product with the other is not, so the pair would be
// rotated without end (the rounding that a sparse low-rank matrix leaves can
// shrink by 1e-16 from vector to vector, down to there); nor is a pair whose
// inner product is lost in its terms' underflow.  The limits are absolute: the
// callers scale the vectors (code_scale), so they lie far below the rounding of
// the longest one.
constexpr double kNormMin = 0x1p-1018, kNormRatio = 0x1p-80, kDotMin = 0x1p-1060;
__device__ __forceinline__ bool pair_rotates(double gpq, double gpp, double gqq, double tol,
                                             double neg2, double& spq, double& spp, double& sqq) {
  pair_scaled(gpq, gpp, gqq, spq, spp, sqq);
  return spq * spq > tol * tol * fmax(spp * sqq, 0.0) && fmax(gpp, gqq) > neg2 &&
         fabs(gpq) > kDotMin &&
         (fmin(gpp, gqq) > kNormMin || fmin(spp, sqq) > kNormRatio);
}

// Convergence measure of the pair block: the largest |G_pq| / sqrt(G_pp G_qq)
// (an FP32 estimate from the scaled entries, at least just above tol) over
// the pairs of this step (inner: all; otherwise those across the blocks) for
// which pair_rotates holds, 0 if there are none.  A block pair with off <= tol is
// left alone, so a sweep whose every step had that, inner pairs at every fourth
// step included, has changed nothing: every pair of vectors is then within tol.
// Pairs of two
// negligible vectors (squared norms <= neg2) are left out: the caller has
// shown that the space they span lies below its truncation threshold
// whether or not they are orthogonalised (neg2 = 0: every pair).
// Block-uniform.  Also leaves in sm whether eig_rotate has to scale the pairs.
__device__ inline double eig_off(EigLds& sm, double tol, double neg2 = 0.0, bool inner = true) {
  const int tid = threadIdx.x;
  const float above = (float)tol * (1.0f + 0x1p-20f) + 0x1p-126f;
  float off = 0.0f;
  // one pair a thread: the 31 rounds of 16 circle pairs
  if (tid < (J2 - 1) * JB) {
    const int r = tid >> 4, sl = tid & 15;
    const int va = sl == 0 ? 0 : 1 + (sl - 1 + r) % (J2 - 1), vb = 1 + (J2 - 2 - sl + r) % (J2 - 1);
    const int p = eig_pos(va), q = eig_pos(vb);
    double spq, spp, sqq;
    const bool rot = pair_rotates(sm.G[0][p][q], sm.G[0][p][p], sm.G[0][q][q], tol, neg2, spq,
                                  spp, sqq);
    // (float)(spp sqq) may flush to 0: rsq then gives inf (or NaN for a
    // zero spq), which fminf clamps
    const float v = fminf(fabsf((float)spq) * __builtin_amdgcn_rsqf((float)(spp * sqq)), 1e30f);
    if (rot && (inner || (va < JB) != (vb < JB))) off = fmaxf(v, above);
  }
  off = wave_max_dpp(off);
  if ((tid & 63) == 0) sm.red[tid >> 6] = off;
  if (tid >= EIG_NT - 64) {
    // the last wave (its lanes carry the fewest pairs): the largest exponent,
    // in magnitude, of the nonzero squared norms
    const double d = sm.G[0][tid & 31][tid & 31];
    const int ex = d > 0.0 ? abs(__builtin_amdgcn_frexp_exp(d)) : 0;
    const float far = wave_max_dpp((float)ex);
    if ((tid & 63) == 0) sm.wide = far > (float)EIG_RANGE ? 1 : 0;
  }
  lds_barrier();
  off = 0.0f;
#pragma unroll
  for (int w = 0; w < EIG_NW; ++w) off = fmaxf(off, sm.red[w]);
  lds_barrier();
  return (double)off;
}

// 1 / sqrt(1 + t^2) from the hardware estimate y (v_rsq_f64, up to 3e-8 off) by
// one third-order step, y (1 + e / 2 + 3 e^2 / 8), on a short dependent chain.
// Its defect e = 1 - (1 + t^2) y^2 is taken as (1 - y^2) - (t y)^2, never from
// the rounded 1 + t^2: that lies on a grid of 2^-52, the result on one of 2^-53,
// and of small angles (|t| in 1e-9 .. 1e-3) it made the cosine 6e-17 too long on
// average (3e-17 with two Newton steps).  Each rotation then lengthened its two
// vectors, and a column of Z ended 7e-14 too long after an SVD of 254 vectors.
__device__ __forceinline__ double cos_of_tan(double t) {
  const double y = __builtin_amdgcn_rsq(fma(t, t, 1.0));
  const double p = t * y;
  const double e = fma(-p, p, fma(-y, y, 1.0));
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

// Rotation coefficients for index x against partner px: G' = J^T G J with
// J_ll = J_hh = c, J_lh = s, J_hl = -s (l < h); row x of J^T G is
// a*G[x] + b*G[px] with a = c and b = -s (x = l) or +s (x = h).
// t = tan(angle) = sgn(D P) |P| / (|D| + sqrt(D^2 + P^2)), D = gqq - gpp,
// P = 2 gpq (the sign from the operands' signs: their product may
// underflow).  The angle only has to shrink the off-diagonal, so
// 1 / (|D| + sqrt(D^2 + P^2)) is evaluated in FP32 on D, P scaled by a power
// of two (exact) into [0.5, 1), where it lies in (0.5, 2]: a 2^-24 error in
// t leaves a 2^-24 fraction of G_lh, which the next sweeps remove like any
// other (same sweep counts as an FP64 angle, measured).  t is that
// reciprocal times the scaled |P| in FP64, so an angle far below FP32's
// range (a nearly-null vector against a large one) is still |P| / (2 |D|)
// and rotates.  Orthogonality comes from c = 1/sqrt(1 + t^2) in FP64
// (cos_of_tan) and s = t c, so c^2 + s^2 = 1 to FP64
// rounding.  A pair is rotated when pair_rotates holds; the coefficients are
// computed without a branch
// (a pair that is not rotated selects c = 1, s = 0, discarding whatever the
// formula gave).
// The coefficients from the three Gram entries of the pair (l, h): G_lh,
// G_ll, G_hh; x_is_l: whether the index asked for is l.
__device__ __forceinline__ void rot_coef_v(double gpq, double gpp, double gqq, bool x_is_l,
                                           double tol, double neg2, double& a, double& b) {
  double spq, spp, sqq;
  const bool rot = pair_rotates(gpq, gpp, gqq, tol, neg2, spq, spp, sqq);
  const double D = gqq - gpp, P = 2.0 * gpq;
  const int e = __builtin_amdgcn_frexp_exp(fmax(fabs(D), fabs(P)));
  const double dd = __builtin_amdgcn_ldexp(fabs(D), -e), pp = __builtin_amdgcn_ldexp(fabs(P), -e);
  const float d = (float)dd, p = (float)pp;
  const float hyp = __builtin_amdgcn_sqrtf(fmaf(d, d, p * p));
  const double tabs = pp * (double)__builtin_amdgcn_rcpf(d + hyp);
  const double t = ((D < 0.0) == (P < 0.0)) ? tabs : -tabs;
  const double c = cos_of_tan(t);
  const double sn = t * c;
  a = rot ? c : 1.0;
  b = rot ? (x_is_l ? -sn : sn) : 0.0;
}

// v of the first lane of this lane's row of 16 (DPP row_newbcast:0)
__device__ __forceinline__ double dpp_row_first(double v) {
  const long long u = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)u, 0x150, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(u >> 32), 0x150, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// v from lane + 1 (row_shl:1) / lane - 1 (row_shr:1) within the lane's row
// of 16 (DPP; the lane without a source gets 0)
__device__ __forceinline__ double dpp_from_next(double v) {
  const long long u = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)u, 0x101, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(u >> 32), 0x101, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
__device__ __forceinline__ double dpp_from_prev(double v) {
  const long long u = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)u, 0x111, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(u >> 32), 0x111, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// v from lane - 1 within the lane's row of 16, the first lane's from the last
// (DPP row_ror:1)
__device__ __forceinline__ double dpp_from_prev_ring(double v) {
  const long long u = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(unsigned)u, 0x121, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(u >> 32), 0x121, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// rot_coef_v(..., x_is_l = true) for Gram entries whose products stay in
// range (EIG_RANGE), on a shorter chain: no scaling, the hypotenuse and the
// tangent from v_rsq_f64 and v_rcp_f64 (about 2^-23 relative, as good as the
// FP32 angle).
__device__ __forceinline__ void rot_coef_n(double gpq, double gpp, double gqq, double tol2,
                                           double neg2, double& a, double& b) {
  const bool rot = gpq * gpq > tol2 * gpp * gqq && fmax(gpp, gqq) > neg2;
  const double D = gqq - gpp, P = gpq + gpq;
  const double h2 = fma(D, D, P * P);
  const double hyp = h2 * __builtin_amdgcn_rsq(h2);
  const double tp = P * __builtin_amdgcn_rcp(fabs(D) + hyp);
  // -t: the sign of P, flipped where D is not negative
  const long long flip = ~__double_as_longlong(D) & (long long)0x8000000000000000ull;
  const double u = __longlong_as_double(__double_as_longlong(tp) ^ flip);
  const double c = cos_of_tan(u);
  a = rot ? c : 1.0;
  b = rot ? u * c : 0.0;
}

// One cyclic sweep (31 rounds of 16 disjoint rotations, circle order; or the
// pairs across the blocks only, 16 rounds in which the second members move on
// by one slot and the first ones stay) of the two-sided Jacobi on G,
// accumulating Q, by 8 waves and one barrier per round.  One inner sweep per outer step: the outer block
// iteration needs the same number of sweeps with one inner sweep as with
// full inner convergence (measured), at a fraction of the cost.
//
// A round is one dependent chain (the pair's entries, the rotation, the
// update, the exchange), so what bounds it is the chain's instructions and
// LDS trips, and the layout keeps everything else off it:
//  * waves 0-3 carry G.  G lies in LDS in circle positions, where a round's
//    moves are the same for every round: a lane reads its 2 x 2 block (row
//    pair rp, column pair cp) and its column pair's diagonal block from fixed
//    addresses and writes the updated block to the fixed addresses it moves
//    to.  Lane l of the 16-lane row of row pair rp owns column pair
//    (l + rp) mod 16, so the rotation of the row pair is always in the row's
//    first lane and reaches the row by a DPP broadcast (row and column
//    rotations of a pair are the same bits) instead of an LDS permute.
//  * waves 4-7 carry Q, one round behind, from the (c, s) that wave 0 leaves
//    in LDS: Q' = Q J only mixes columns, and the circle moves a column
//    between neighbouring column slots (first slots from lane cp + 1 to cp,
//    second slots from cp - 1 to cp, slot 1-first to 0-second, 15-second to
//    15-first, vector 0 fixed), which stay within the lane's DPP row of 16.
//    Their work fills the issue slots that the G waves' latencies leave.
// Measured (in-kernel clock, n = 1024): 1220 cycles a round with one group of
// four waves for G and Q on index-ordered LDS and an LDS permute for the row
// rotations, 797 in this layout, 719 with rot_coef_n's shorter chain; of
// those the coefficients are 250, the reads 75, the 16 products and the DPP
// moves 120, the writes 130, the barrier and the loop the rest, and the Q
// waves nothing.  jac_eig_apply at n = 256 with Z 17.8 -> 12.4 us, at
// 512 x 2560 SVDs 31.8 -> 20.5 us.  A conflict-free split of the positions
// (first members 0-15, second 16-31, rows 32 banks apart, 8-byte accesses)
// measured the same 725 cycles: the accesses' number, not conflicts, counts.
// Pairs are rotated down to a quarter of tol, the convergence measure counts
// those above tol: a sweep then leaves none just under tol, which the next
// measure, rounded differently, may find above it (eigensolves at n = 1024
// otherwise run a sweep that rotates next to nothing one time in two).
// Q is left in sm.Q.
struct EigSlots {  // a G lane's fixed places: rows and columns of its block, and where they move
  int rp, cp, r0, r1, c0, c1;
  __device__ EigSlots(int tid, bool inner) {
    rp = tid >> 4;
    cp = ((tid & 15) + rp) & 15;
    if (!inner) {
      r0 = 2 * rp;
      r1 = 2 * ((rp + 1) & 15) + 1;
      c0 = 2 * cp;
      c1 = 2 * ((cp + 1) & 15) + 1;
      return;
    }
    r0 = rp == 0 ? 0 : (rp == 1 ? 1 : 2 * (rp - 1));
    r1 = rp == 15 ? 30 : 2 * (rp + 1) + 1;
    c0 = cp == 0 ? 0 : (cp == 1 ? 1 : 2 * (cp - 1));
    c1 = cp == 15 ? 30 : 2 * (cp + 1) + 1;
  }
};

// The G waves' side of the rounds; coef(gpq, gpp, gqq, c, s): the rotation of
// a pair.
template <bool INNER, typename Coef>
__device__ __forceinline__ void eig_rounds_g(EigLds& sm, Coef coef) {
  const EigSlots z(threadIdx.x, INNER);
  constexpr int LD = J2 + GPAD;
  const int ix0 = 2 * z.rp * LD + 2 * z.cp, ix1 = ix0 + LD, iy = 2 * z.cp * LD + 2 * z.cp;
  const int o00 = z.r0 * LD + z.c0, o01 = z.r0 * LD + z.c1;
  const int o10 = z.r1 * LD + z.c0, o11 = z.r1 * LD + z.c1;
  auto round = [&](const double* g, double* h, double* cs) {
    const double2 y0 = *(const double2*)(g + iy);
    const double yqq = g[iy + LD + 1];
    const double2 g0 = *(const double2*)(g + ix0), g1 = *(const double2*)(g + ix1);
    // (c, s) for the first member of each pair; the second's s is -s
    double cy, sy;
    coef(y0.y, y0.x, yqq, cy, sy);
    if (threadIdx.x < 16) *(double2*)(cs + 2 * z.cp) = double2{cy, sy};
    const double cx = dpp_row_first(cy), sx = dpp_row_first(sy);
    const double r00 = cx * g0.x + sx * g1.x, r01 = cx * g0.y + sx * g1.y;
    const double r10 = cx * g1.x - sx * g0.x, r11 = cx * g1.y - sx * g0.y;
    h[o00] = cy * r00 + sy * r01;
    h[o01] = cy * r01 - sy * r00;
    h[o10] = cy * r10 + sy * r11;
    h[o11] = cy * r11 - sy * r10;
    lds_barrier();
  };
  double* const ga = &sm.G[0][0][0];
  double* const gb = &sm.G[1][0][0];
  for (int r = 0; r < (INNER ? J2 - 2 : JB); r += 2) {  // 31 or 16 rounds
    round(ga, gb, &sm.cs[0][0][0]);
    round(gb, ga, &sm.cs[1][0][0]);
  }
  if constexpr (INNER) round(ga, gb, &sm.cs[0][0][0]);
}

// The Q waves' side of the rounds.
template <bool INNER>
__device__ __forceinline__ void eig_rounds_q(EigLds& sm) {
  const int t = threadIdx.x - 256, rp = t >> 4, cp = t & 15;
  const int y0 = cp, y1 = J2 - 1 - cp;
  const int R0 = 2 * rp, R1 = 2 * rp + 1;
  double qa0 = R0 == y0 ? 1.0 : 0.0, qa1 = R0 == y1 ? 1.0 : 0.0;   // Q[R0][y0], Q[R0][y1]
  double qb0 = R1 == y0 ? 1.0 : 0.0, qb1 = R1 == y1 ? 1.0 : 0.0;   // Q[R1][y0], Q[R1][y1]
  auto step = [&](int b) {
    const double2 v = *(const double2*)&sm.cs[b][cp][0];
    const double cy = v.x, sy = v.y;
    // Q' = Q J on the column pair, then the circle shift of the columns
    const double na0 = cy * qa0 + sy * qa1, na1 = cy * qa1 - sy * qa0;
    const double nb0 = cy * qb0 + sy * qb1, nb1 = cy * qb1 - sy * qb0;
    if constexpr (!INNER) {
      qa0 = na0;
      qb0 = nb0;
      qa1 = dpp_from_prev_ring(na1);
      qb1 = dpp_from_prev_ring(nb1);
      return;
    }
    const double fa = dpp_from_next(na0), fb = dpp_from_next(nb0);
    const double pa = dpp_from_prev(na1), pb = dpp_from_prev(nb1);
    qa0 = cp == 0 ? na0 : (cp == 15 ? na1 : fa);
    qb0 = cp == 0 ? nb0 : (cp == 15 ? nb1 : fb);
    qa1 = cp == 0 ? fa : pa;
    qb1 = cp == 0 ? fb : pb;
  };
  lds_barrier();
  for (int r = 0; r < (INNER ? J2 - 2 : JB - 2); r += 2) {
    step(0);
    lds_barrier();
    step(1);
    lds_barrier();
  }
  step(0);
  if constexpr (!INNER) {
    lds_barrier();
    step(1);
  }
  // after 31 (16) rounds every slot holds its first members again
  sm.Q[R0][y0] = qa0;
  sm.Q[R0][y1] = qa1;
  sm.Q[R1][y0] = qb0;
  sm.Q[R1][y1] = qb1;
}

template <bool INNER>
__device__ __forceinline__ void eig_rounds(EigLds& sm, double tol, double neg2) {
  if (threadIdx.x >= 256) {
    eig_rounds_q<INNER>(sm);
  } else if (__builtin_amdgcn_readfirstlane(sm.wide)) {
    eig_rounds_g<INNER>(sm, [&](double gpq, double gpp, double gqq, double& c, double& s) {
      rot_coef_v(gpq, gpp, gqq, true, 0.25 * tol, neg2, c, s);
    });
  } else {
    const double tol2 = (0.25 * tol) * (0.25 * tol);
    eig_rounds_g<INNER>(sm, [&](double gpq, double gpp, double gqq, double& c, double& s) {
      rot_coef_n(gpq, gpp, gqq, tol2, neg2, c, s);
    });
  }
}

__device__ inline void eig_rotate(EigLds& sm, double tol, double neg2 = 0.0, bool inner = true) {
  if (inner)
    eig_rounds<true>(sm, tol, neg2);
  else
    eig_rounds<false>(sm, tol, neg2);
  lds_barrier();
}

// Gram matrix of a pair's 32 vectors over at most kPairLen rows (vector v at
// W + v * ld, nv vectors, `rows` rows) by the whole workgroup of 8 waves,
// straight from memory: wave w takes rows 32 w .. 32 w + 31, two neighbouring
// rows a lane and load, as operands of v_mfma_f64_16x16x4 (the summation index
// may be any row, as long as both operands agree), for the three 16 x 16
// quarters that are not each other's mirror; the waves' sums meet in LDS and
// put(r, c, s) takes the entries (both mirrored ones).  No staging and no
// barrier before the last: what bounds it is one trip to memory and 24 MFMAs a
// wave.
constexpr int kPairLen = 32 * EIG_NW;
typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));  // odd ld: 8-byte aligned

struct PairGramLds {
  double part[EIG_NW][3][JB * JB];
};

template <typename Put>
__device__ __forceinline__ void pair_gram_rows(PairGramLds& pg, const double* __restrict__ W,
                                               int64_t ld, int rows, int64_t nv, int I, int J,
                                               Put put) {
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
  const int r0 = 32 * wave;
  const int64_t vi = (int64_t)I * JB + lr, vj = (int64_t)J * JB + lr;
  f64x4 acc[3] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
  if (r0 < rows) {
    double xi[8], xj[8];
    if (r0 + 32 <= rows && ((int64_t)max(I, J) + 1) * JB <= nv) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = r0 + 8 * j + 2 * lk;
        const f64x2u a = *(const f64x2u*)(W + vi * ld + r), b = *(const f64x2u*)(W + vj * ld + r);
        xi[2 * j] = a[0];
        xi[2 * j + 1] = a[1];
        xj[2 * j] = b[0];
        xj[2 * j + 1] = b[1];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int r = r0 + 8 * (j >> 1) + 2 * lk + (j & 1);
        xi[j] = (vi < nv && r < rows) ? W[vi * ld + r] : 0.0;
        xj[j] = (vj < nv && r < rows) ? W[vj * ld + r] : 0.0;
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(xi[j], xi[j], acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(xi[j], xj[j], acc[1], 0, 0, 0);
      acc[2] = __builtin_amdgcn_mfma_f64_16x16x4f64(xj[j], xj[j], acc[2], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) pg.part[wave][t][64 * e + lane] = acc[t][e];
  }
  lds_barrier();
  const int nw = (rows + 31) >> 5;
  for (int q = tid; q < 3 * JB * JB; q += EIG_NT) {
    const int t = q >> 8, i = q & 255, m = ((i & 63) >> 4) + 4 * (i >> 6), n = i & 15;
    // (every load issued before the first add)
    double v[EIG_NW], s = 0.0;
#pragma unroll
    for (int w = 0; w < EIG_NW; ++w) v[w] = pg.part[min(w, nw - 1)][t][i];
#pragma unroll
    for (int w = 0; w < EIG_NW; ++w) s += w < nw ? v[w] : 0.0;
    const int r = t == 2 ? JB + m : m, c = t == 0 ? n : JB + n;
    put(r, c, s);
    if (t == 1) put(c, r, s);
  }
}

// ... over all L <= kPairLen rows into sm.G[0].
__device__ inline void pair_gram(EigLds& sm, PairGramLds& pg, const double* __restrict__ W,
                                 int64_t L, int64_t nv, int I, int J) {
  pair_gram_rows(pg, W, L, (int)L, nv, I, J,
                 [&](int r, int c, double s) { sm.G[0][eig_pos(r)][eig_pos(c)] = s; });
  lds_barrier();
}

// Rows [rs, re) (re - rs <= 16 NT NW, NW waves) of the pair's 32 vectors (vector v at
// base + v * ld, nv vectors) <- rows . Q, as the transposed product
// (Q^T X^T) on v_mfma_f64_16x16x4: the B operand of each 16 x 16 output tile
// is 16 consecutive rows of 4 vectors, read straight from memory (four
// 128-byte runs per load), the A operand is Q^T from LDS, and the output
// tile is 16 consecutive rows of 4 vectors again, stored straight back: no
// LDS staging and no barrier.  Wave w covers rows rs + 16 NT w + [0, 16 NT)
// as NT row tiles; lane (lr = lane % 16, lk = lane / 16).
//   apply_rows_fetch:  x[ks][nt] = row rs + 16 NT w + 16 nt + lr of vector
//                      4 ks + lk of the pair (issued early: in flight while
//                      the caller computes Q);
//   apply_rows_finish: 16 NT MFMAs per wave (2 vector tiles x NT row tiles x
//                      8 k-steps) and the stores.
// Whether the chunk is a whole 16 NT NW rows and all 32 vectors of the pair
// exist (block-uniform): then the loads and stores need no bounds test.
template <int NT, int NW>
__device__ __forceinline__ bool apply_rows_full(int64_t nv, int64_t rs, int64_t re, int I, int J) {
  return re - rs == 16 * NT * NW && (int64_t)max(I, J) * JB + JB <= nv;
}

template <int NT, int NW>
__device__ __forceinline__ void apply_rows_fetch(const double* __restrict__ base, int64_t ld,
                                                 int64_t nv, int64_t rs, int64_t re, int I,
                                                 int J, double (&x)[8][NT]) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int lr = lane & 15, lk = lane >> 4;
  const int64_t r0 = rs + 16 * NT * wave + lr;
  if (apply_rows_full<NT, NW>(nv, rs, re, I, J)) {
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) {
      const double* p = base + pair_vec(4 * ks + lk, I, J) * ld + r0;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) x[ks][nt] = p[16 * nt];
    }
    return;
  }
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) {
    const int64_t v = pair_vec(4 * ks + lk, I, J);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int64_t r = r0 + 16 * nt;
      x[ks][nt] = (v < nv && r < re) ? base[v * ld + r] : 0.0;
    }
  }
}

template <int NT, int NW>
__device__ __forceinline__ void apply_rows_finish(double* __restrict__ base, int64_t ld,
                                                  int64_t nv, int64_t rs, int64_t re, int I,
                                                  int J, const double (&x)[8][NT],
                                                  const double (*Q)[J2 + 1]) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int lr = lane & 15, lk = lane >> 4;
  const int64_t r0 = rs + 16 * NT * wave + lr;
  f64x4 acc[2][NT];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f64x4{0, 0, 0, 0};
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) {
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      // A[i][k] = Q^T[16 mt + i][4 ks + k] = Q[4 ks + k][16 mt + i]
      const double a = Q[4 * ks + lk][16 * mt + lr];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        acc[mt][nt] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, x[ks][nt], acc[mt][nt], 0, 0, 0);
    }
  }
  // output tile (mt, nt): lane holds vector 16 mt + lk + 4 e, row 16 nt + lr
  if (apply_rows_full<NT, NW>(nv, rs, re, I, J)) {
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        double* p = base + pair_vec(16 * mt + lk + 4 * e, I, J) * ld + r0;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) p[16 * nt] = acc[mt][nt][e];
      }
    return;
  }
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t v = pair_vec(16 * mt + lk + 4 * e, I, J);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int64_t r = r0 + 16 * nt;
        if (v < nv && r < re) base[v * ld + r] = acc[mt][nt][e];
      }
    }
}

}  // namespace tn

// hj_qr.hip -- the QR factorization of a block-pair visit and Drmac's sorted
// level-0 (the reference's build options USE_QR and USE_DRMAC,
// share/device_code_common.hpp:78-85,140-144), one workgroup per block pair.
//
// The visit, of eight waves with up to 16 panels of 32 rows in LDS (32x32,
// column-major with leading dimension 33; beyond 512 rows, 15 more at a time):
//  * the panels' Householder QR (dQR32,
//    share/device_code_common_Kepler.hpp:326-371), each by a wave of its own:
//    the panels do not depend on each other (householder32);
//  * the panels' factors into the first's, in order (dPeelOff,
//    share/device_code_common_QR.hpp:4-92), by a wavefront of Givens rotations:
//    32 dependent rotations a panel, all that is serial here (merge_panel);
//  * level-0: Drmac's sweeps for sorted definite blocks when asked
//    (share/device_code_cdsort_Drmac.hpp:4-316; drmac_r), otherwise the
//    Cholesky path's, four waves on R and four on W (hj_visit.hpp);
//  * counters, the update flag and W to HBM; the block update is k_update's.
// Reductions over 32 rows are the butterfly 16, 8, 4, 2, 1 of the reference's
// dSum32, the first level or levels inside a lane.
// This path is latency-bound; like the reference's, it is an accuracy option
// for extremely graded column pairs, not a fast path.  Measured, 512 x 256
// (16 panels a pair): Householder 70 us (two panels a wave), merges 150 us
// (480 steps of 312 ns), level-0 32 us; 262 us a launch, where one wave a
// pair, doing all of it in turn, took 1466 us.
#include <climits>
#include <cfloat>

#include "hj_device.hpp"
#include "hj_kernels.hpp"
#include "hj_visit.hpp"

namespace hj {
namespace {

// Magnitude limits of the overflow- and underflow-safe sums of squares
// (share/HypJacL.hpp:53-86).  Squares of entries in [SSQ_SMALL, SSQ_BIG]
// and 32-term sums of them stay normal and finite.
constexpr double SSQ_SMALL = 0x1p-511;              // sqrt of the smallest normal
constexpr double SSQ_BIG = 0x1.6a09e667f3bcap+509;  // a little below sqrt(DBL_MAX / 32)
constexpr double PROD_SMALL = 0x1p-970;             // smallest normal / epsilon
constexpr double COT_LIMIT = 0x1.fffffffffffffp+1020;  // DBL_MAX / 8

// ---------------------------------------------------------------------------
// Reductions over the 32 rows of one column held by a quad, v[j] = row r + 4j.

__device__ __forceinline__ double quad_max_abs(const double (&v)[8])
{
  double m = fabs(v[0]);
#pragma unroll
  for (unsigned j = 1u; j < 8u; ++j) m = fmax(m, fabs(v[j]));
  m = fmax(m, lane_xor2(m));
  return fmax(m, lane_xor1(m));
}

// smallest nonzero magnitude (DBL_MAX when every entry is zero)
__device__ __forceinline__ double quad_min_abs_nz(const double (&v)[8])
{
  double m = DBL_MAX;
#pragma unroll
  for (unsigned j = 0u; j < 8u; ++j) m = fmin(m, (v[j] == 0.0) ? DBL_MAX : fabs(v[j]));
  m = fmin(m, lane_xor2(m));
  return fmin(m, lane_xor1(m));
}

// The power of two that moves x next to the limit t: for x <= t the least s
// with x 2^s >= t, for x > t the greatest s with x 2^s <= t.
__device__ __forceinline__ int scale_to(double x, double t)
{
  int ex, et;
  const double mx = frexp(x, &ex), mt = frexp(t, &et);
  const int s = et - ex;
  return (x <= t) ? s + (mx < mt ? 1 : 0) : s - (mx > mt ? 1 : 0);
}

// A scaled value f 2^e with f brought to an even exponent's power of two
// removed (f in [1, 4)), so that the square root rescales exactly.
__device__ __forceinline__ void even_normalize(int &e, double &f)
{
  int s = ilogb(f);
  s += s & 1;
  e += s;
  f = scalbn(f, -s);
}

// (e, f) = f1 2^e1 + f2 2^e2: the smaller term, by exponent then fraction,
// rescaled to the larger one's exponent.
__device__ __forceinline__ void add_scaled(int e1, double f1, int e2, double f2, int &e, double &f)
{
  const bool first_smaller = (e1 != e2) ? (e1 < e2) : !(f2 < f1);
  if (first_smaller) {
    e = e2;
    f = scalbn(f1, e1 - e2) + f2;
  }
  else {
    e = e1;
    f = scalbn(f2, e2 - e1) + f1;
  }
}

// Sum of squares of the entries in one magnitude band, each scaled by 2^e
// first (outer bands) or taken as is (middle band).
enum Band { BAND_LOW = 0, BAND_MID = 1, BAND_HIGH = 2 };

__device__ __forceinline__ double band_ssq(const double (&v)[8], Band b, int e)
{
  double sq[8];
#pragma unroll
  for (unsigned j = 0u; j < 8u; ++j) {
    const double a = fabs(v[j]);
    double y;
    if (b == BAND_HIGH) y = (a > SSQ_BIG) ? scalbn(a, e) : 0.0;
    else if (b == BAND_MID) y = ((a >= SSQ_SMALL) && (a <= SSQ_BIG)) ? a : 0.0;
    else y = (a < SSQ_SMALL) ? scalbn(a, e) : 0.0;
    sq[j] = y * y;
  }
  return sum4x8(sq);
}

// The sum of squares of the column as f 2^e (returned), without overflow
// or harmful underflow: entries above SSQ_BIG or below SSQ_SMALL are summed
// in a band of their own, scaled toward the limit, and the band sums are
// combined by add_scaled (dSSQ32, share/device_code_common_Kepler.hpp:203-260).
// e is INT_MIN for a zero column.
__device__ int quad_ssq(const double (&v)[8], double &f)
{
  const double hi = quad_max_abs(v);
  if (hi == 0.0) {
    f = 0.0;
    return INT_MIN;
  }
  const double lo = quad_min_abs_nz(v);
  if (hi > SSQ_BIG) {
    int eh = scale_to(hi, SSQ_BIG);
    double fh = band_ssq(v, BAND_HIGH, eh);
    eh = -2 * eh;
    if (lo > SSQ_BIG) {
      f = fh;
      return eh;
    }
    int em = 0;
    double fm = band_ssq(v, BAND_MID, 0);
    if (!(fm > 0.0)) {
      f = fh;
      return eh;
    }
    even_normalize(em, fm);
    even_normalize(eh, fh);
    int e;
    add_scaled(em, fm, eh, fh, e, f);
    return e;
  }
  if (lo < SSQ_SMALL) {
    int el = scale_to(lo, SSQ_SMALL);
    double fl = band_ssq(v, BAND_LOW, el);
    el = -2 * el;
    if (hi < SSQ_SMALL) {
      f = fl;
      return el;
    }
    int em = 0;
    double fm = band_ssq(v, BAND_MID, 0);
    if (!(fm > 0.0)) {
      f = fl;
      return el;
    }
    even_normalize(em, fm);
    even_normalize(el, fl);
    int e;
    add_scaled(el, fl, em, fm, e, f);
    return e;
  }
  double sq[8];
#pragma unroll
  for (unsigned j = 0u; j < 8u; ++j) sq[j] = v[j] * v[j];
  f = sum4x8(sq);
  return 0;
}

// ||column||_2 (dNRM2_32, share/device_code_common_Kepler.hpp:269-275)
__device__ __forceinline__ double quad_nrm2(const double (&v)[8])
{
  double f;
  const int e = quad_ssq(v, f);
  return scalbn(sqrt(f), e / 2);
}

// x^T y / (nx ny) for nx >= ny, the division placed so that neither the
// product nor the quotient leaves the normal range
// (dCOSA_, share/device_code_common_Kepler.hpp:277-303)
__device__ __forceinline__ double quad_cos_ordered(double nx, double ny, const double (&x)[8],
                                                   const double (&y)[8])
{
  const bool huge = (ny >= 1.0) && ((nx * ny) >= DBL_MAX);
  const bool tiny = !(ny >= 1.0) && ((nx * ny) <= PROD_SMALL);
  double z[8];
  if (huge) {
#pragma unroll
    for (unsigned j = 0u; j < 8u; ++j)
      z[j] = (fabs(x[j]) >= fabs(y[j])) ? ((x[j] / nx) * y[j]) : ((y[j] / nx) * x[j]);
    return sum4x8(z) / ny;
  }
  if (tiny) {
#pragma unroll
    for (unsigned j = 0u; j < 8u; ++j)
      z[j] = (fabs(x[j]) >= fabs(y[j])) ? (x[j] * (y[j] / ny)) : (y[j] * (x[j] / ny));
    return sum4x8(z) / nx;
  }
#pragma unroll
  for (unsigned j = 0u; j < 8u; ++j) z[j] = x[j] * y[j];
  return (sum4x8(z) / ny) / nx;
}

__device__ __forceinline__ double quad_cos(double np, double nq, const double (&p)[8],
                                           const double (&q)[8])
{
  return (np >= nq) ? quad_cos_ordered(np, nq, p, q) : quad_cos_ordered(nq, np, q, p);
}

// ---------------------------------------------------------------------------
// Factorization.

// [c s; -s c] [f; g] = [r; 0] with r >= 0, r formed as the larger magnitude
// times sqrt(1 + (smaller / larger)^2) (dGivens,
// share/device_code_common_rotate.hpp:120-155)
__device__ __forceinline__ void givens(double f, double g, double &c, double &s, double &r)
{
  const double af = fabs(f), ag = fabs(g);
  const bool fbig = af >= ag;
  const double big = fbig ? af : ag, small = fbig ? ag : af;
  const bool one = small == 0.0;  // one of the two is zero
  const double q = small / big;
  r = one ? big : pin(big * sqrt(__fma_rn(q, q, 1.0)));
  // (the quotients are issued side by side, also where they are not used)
  const double cq = pin(f / r), sq = pin(g / r);
  c = one ? (fbig ? copysign(1.0, f) : 0.0) : cq;
  s = one ? (fbig ? 0.0 : copysign(1.0, g)) : sq;
}

// Sum of the 32 rows of a column held by 16 lanes, lane r holding rows row_of(r)
// and row_of(r) + 16 as a, b: the butterfly 16, 8, 4, 2, 1.
__device__ __forceinline__ double sum16x2(double a, double b)
{
  double s = a + b;
  s = s + dpp_mov<0x128>(s);
  s = s + dpp_mov<0x141>(s);
  s = s + dpp_mov<0x4E>(s);
  return s + dpp_mov<0xB1>(s);
}

// Whether x adds to a plain sum of squares (quad_ssq's middle band)
__device__ __forceinline__ unsigned ssq_plain(double x)
{
  const double a = fabs(x);
  const bool zero = x == 0.0, above = a >= SSQ_SMALL, below = a <= SSQ_BIG;
  return (unsigned)zero | ((unsigned)above & (unsigned)below);
}

// ||A(k0:31, c)||_2 by quads (all of the wave's with the same column, or each
// with its own): the norm of a column with entries outside the middle band
__device__ __noinline__ double column_nrm2(const lds_f64 *A, unsigned c, unsigned k0, unsigned r4)
{
  double v[8];
#pragma unroll
  for (unsigned j = 0u; j < 8u; ++j) {
    const unsigned x = r4 + 4u * j;
    v[j] = (x >= k0) ? A[c * L0LD + x] : 0.0;
  }
  return quad_nrm2(v);
}

// Householder QR of the 32x32 block A in place by one wave: for k = 0..30 the
// reflector I - tau v v^T with v_k = 1, v_x = A(x,k) / (alpha + beta) below the
// diagonal, beta = sign(alpha) ||A(k:31,k)||, applied to columns k+1..31 as
// A(:,c) += (-(tau v^T A(:,c))) v; column k becomes (-beta, 0, ..., 0).
// A step is bound by the instructions it issues: 16 lanes hold a column (two
// rows each), so that the norm and the divisions, which every group does for
// itself, are few, and four columns a group are updated side by side.
__device__ void householder32(double *A_, unsigned l)
{
  lds_f64 *const A = (lds_f64 *)A_;
  const unsigned g = l >> 4, x0 = row_of(l & 15u), x1 = x0 + 16u;
#pragma unroll 1
  for (unsigned k = 0u; k < 31u; ++k) {
    const double a0 = A[k * L0LD + x0], a1 = A[k * L0LD + x1];
    const double alpha = A[k * L0LD + k];
    double v0 = (x0 >= k) ? a0 : 0.0, v1 = (x1 >= k) ? a1 : 0.0;
    double nrm = sqrt(sum16x2(v0 * v0, v1 * v1));
    if (__ballot((ssq_plain(v0) & ssq_plain(v1)) == 0u) != 0ull)
      nrm = column_nrm2(A, k, k, l & 3u);
    if (!(nrm > 0.0))
      continue;  // the same in every lane: every group holds column k
    // column k has been read by every lane before any lane writes it
    wave_lds_sync();
    const double beta = copysign(nrm, alpha), ab = alpha + beta;
    // (the three quotients side by side)
    const double tau = pin(ab / beta);
    v0 = pin(v0 / ab);
    v1 = pin(v1 / ab);
    v0 = (x0 == k) ? 1.0 : ((x0 > k) ? v0 : 0.0);
    v1 = (x1 == k) ? 1.0 : ((x1 > k) ? v1 : 0.0);
#pragma unroll 1
    for (unsigned c = k + 1u + g; c < 32u; c += 16u) {
      double b0[4], b1[4], t[4];
#pragma unroll
      for (unsigned i = 0u; i < 4u; ++i) {
        // (a column past the last: the last again, not stored)
        const lds_f64 *const p = A + min(c + 4u * i, 31u) * L0LD;
        b0[i] = p[x0];
        b1[i] = p[x1];
      }
#pragma unroll
      for (unsigned i = 0u; i < 4u; ++i)
        t[i] = v0 * b0[i] + v1 * b1[i];
#pragma unroll
      for (unsigned i = 0u; i < 4u; ++i) t[i] = t[i] + dpp_mov<0x128>(t[i]);
#pragma unroll
      for (unsigned i = 0u; i < 4u; ++i) t[i] = t[i] + dpp_mov<0x141>(t[i]);
#pragma unroll
      for (unsigned i = 0u; i < 4u; ++i) t[i] = t[i] + dpp_mov<0x4E>(t[i]);
#pragma unroll
      for (unsigned i = 0u; i < 4u; ++i) t[i] = t[i] + dpp_mov<0xB1>(t[i]);
#pragma unroll
      for (unsigned i = 0u; i < 4u; ++i) {
        const double tdp = -(tau * t[i]);
        b0[i] = __fma_rn(tdp, v0, b0[i]);
        b1[i] = __fma_rn(tdp, v1, b1[i]);
      }
#pragma unroll
      for (unsigned i = 0u; i < 4u; ++i) {
        if (c + 4u * i < 32u) {
          A[(c + 4u * i) * L0LD + x0] = b0[i];
          A[(c + 4u * i) * L0LD + x1] = b1[i];
        }
      }
    }
    if (g == 3u) {
      if (x0 >= k) A[k * L0LD + x0] = (x0 == k) ? -beta : 0.0;
      if (x1 >= k) A[k * L0LD + x1] = (x1 == k) ? -beta : 0.0;
    }
    wave_lds_sync();
  }
}

constexpr unsigned QR_WAVES = 8u;
constexpr unsigned QR_NT = 64u * QR_WAVES;
constexpr unsigned QR_LANES = QR_NT / 32u;  // lanes a pivot pair of level-0, R's and W's
constexpr unsigned QR_PANELS = 16u;         // panels in LDS at once, the running factor among them
constexpr unsigned QR_PANEL = 32u * L0LD;

// LDS of a visit: the panels (the first is the running factor R, the second
// becomes W), what inner_sweeps_by shares (see PairLds), the rotations of a
// merge step by its parity
struct QrLds {
  static constexpr unsigned N = 32u, LD = L0LD;
  static constexpr double TOL = MYTOL;
  double R[QR_PANEL];
  double W[QR_PANEL];
  double panels[(QR_PANELS - 2u) * QR_PANEL];
  double rot[2][16][4];
  double gv[2][32][2];
  unsigned act[2][16];
  unsigned cs[2], cb[2];
  unsigned cmax;
  int swp;
  __attribute__((aligned(16))) uint8_t S0[STRAT0_TAB_BYTES];
};
static_assert(offsetof(QrLds, W) == sizeof(double) * QR_PANEL &&
                  offsetof(QrLds, panels) == sizeof(double) * 2u * QR_PANEL,
              "the panels adjoin");

// x of the lane before (lane 0: 0)
__device__ __forceinline__ double lane_before(double x)
{
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x138, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x138, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

// The R factor of [R; P1; P2; ...] for upper triangular panels, one after the
// other, by the workgroup.  With the next panel P, at step k = 0..31 every row
// x >= k of R meets row x-k of P in the rotation that zeroes P(x-k, x) against
// R(x, x), applied to columns x..31 (products and sums rounded separately).
// The chain is one rotation a step (a division, a root, a division) and what
// brings the next step's operands: wave 0 keeps the diagonal and the two
// diagonals above it in registers, lane x column x: step k's rotation, the
// entries beside the diagonal by it (the lane before's: the next rotation's
// P entry), and the second diagonal's by step k-1's, while the other waves
// apply step k-1's to the entries further right, a thread an entry of R, which
// stays in its register over all panels.  A barrier a step.
struct Merge {
  unsigned l, t;       // lane of wave 0's, thread of the others (wave 0: >= MERGE_ENTRIES)
  unsigned x, col;     // the thread's entry of R
  double A0, A1, A2;   // wave 0: R(x, x), R(x-1, x), R(x-2, x)
  double a;            // others: R(x, col)
};
constexpr unsigned MERGE_ENTRIES = 29u * 30u / 2u;  // entries with col >= x + 3
static_assert(MERGE_ENTRIES <= QR_NT - 64u, "a thread an entry");

__device__ __forceinline__ void merge_begin(Merge &M, const QrLds &L, unsigned tid)
{
  const lds_f64 *const R = (const lds_f64 *)L.R;
  M.l = min(tid, 64u);
  M.t = tid < 64u ? MERGE_ENTRIES : tid - 64u;
  // entries by column 3, 4, ..., column c with rows 0 .. c-3
  unsigned c = 3u, off = 0u;
  while (c < 31u && off + (c - 2u) <= M.t) {
    off += c - 2u;
    ++c;
  }
  M.col = tid < 64u ? (tid & 31u) : c;
  M.x = tid < 64u ? (tid & 31u) : min(M.t - off, 31u);
  // (read by every thread: a branch around the ones it does not use would
  // keep them in memory)
  M.A0 = R[M.x * L0LD + M.x];
  M.A1 = R[M.x * L0LD + (M.x >= 1u ? M.x - 1u : 0u)];
  M.A2 = R[M.x * L0LD + (M.x >= 2u ? M.x - 2u : 0u)];
  M.a = R[M.col * L0LD + M.x];
}

__device__ __forceinline__ void merge_end(const Merge &M, QrLds &L)
{
  lds_f64 *const R = (lds_f64 *)L.R;
  if (M.l < 32u) {
    R[M.x * L0LD + M.x] = M.A0;
    if (M.x >= 1u) R[M.x * L0LD + M.x - 1u] = M.A1;
    if (M.x >= 2u) R[M.x * L0LD + M.x - 2u] = M.A2;
  }
  else if (M.t < MERGE_ENTRIES)
    R[M.col * L0LD + M.x] = M.a;
  __syncthreads();
}

// all threads of the workgroup; P synchronized
__device__ __forceinline__ void merge_panel(Merge &M, QrLds &L, double *P_)
{
  lds_f64 *const P = (lds_f64 *)P_;
  lds_f64 *const gv = (lds_f64 *)&L.gv[0][0][0];
  if (M.l < 64u) {
    const lds_f64 *const pc = P + M.x * L0LD;
    double g = pc[M.x], c2 = 0.0, s2 = 0.0;
#pragma unroll 1
    for (unsigned k = 0u; k < 32u; ++k) {
      const bool next = M.x > k;  // this lane rotates at step k+1
      double b = pc[next ? M.x - k - 1u : 0u];
      double c, s, r;
      givens(M.A0, g, c, s, r);
      if (M.x >= k) M.A0 = r;
      if (M.l < 32u) {
        gv[64u * (k & 1u) + 2u * M.x] = c;
        gv[64u * (k & 1u) + 2u * M.x + 1u] = s;
      }
      if (k) {
        // the second diagonal's entry by step k-1's rotation of row x-2
        const double ca = c2 * M.A2, sb = s2 * b, cb = c2 * b, sa = s2 * M.A2;
        M.A2 = next ? ca + sb : M.A2;
        b = cb - sa;
      }
      // the entry beside the diagonal by this step's rotation of row x-1
      const double c1 = lane_before(c), s1 = lane_before(s);
      const double ca = c1 * M.A1, sb = s1 * b, cb = c1 * b, sa = s1 * M.A1;
      M.A1 = next ? ca + sb : M.A1;
      g = cb - sa;
      c2 = lane_before(c1);
      s2 = lane_before(s1);
      __syncthreads();
    }
  }
  else {
    __syncthreads();
#pragma unroll 1
    for (unsigned k = 0u; k < 31u; ++k) {
      if (M.t < MERGE_ENTRIES && M.x >= k) {
        lds_f64 *const p = P + M.col * L0LD + M.x - k;
        const double c = gv[64u * (k & 1u) + 2u * M.x], s = gv[64u * (k & 1u) + 2u * M.x + 1u];
        const double b = *p;
        const double ca = c * M.a, sb = s * b, cb = c * b, sa = s * M.a;
        M.a = ca + sb;
        *p = cb - sa;
      }
      __syncthreads();
    }
  }
}

// ---------------------------------------------------------------------------
// One of Drmac's sorted definite level-0 sweeps on R (posd for definite >= 0:
// the larger norm first; negd: the smaller first),
// share/device_code_cdsort_Drmac.hpp:4-316: level0_r with other rotations.
// The cosine of the pivot columns and their norms are formed overflow-safe
// (wave by wave, by the plain sums where those are in range); the rotation
// comes from cot(2 phi) = (nq/np - np/nq) / (2 cos), and where that exceeds
// COT_LIMIT the smaller column is made orthogonal to the larger one directly.
// W's columns take c = 1 and t = -+cos there.
__device__ __forceinline__ void drmac_r(QrLds &L, unsigned y, unsigned r, unsigned s0steps,
                                        int definite, unsigned &my_s, unsigned &my_b)
{
  constexpr unsigned LD = L0LD;
  const bool pos = (definite >= 0);
  lds_f64 *const R = (lds_f64 *)L.R;
  lds_f64 *const M = R + row_of(r);
  const uint16_t *const S0 = reinterpret_cast<const uint16_t *>(L.S0) + y;
#pragma unroll 1
  for (unsigned step = 0u; step < s0steps; ++step) {
    const unsigned pq = S0[16u * step], p = pq & 255u, q = pq >> 8;
    lds_f64 *const ap = M + p * LD, *const aq = M + q * LD;
    const double Gp[2] = {ap[0], ap[16]}, Gq[2] = {aq[0], aq[16]};
    double Dp, Dq, cs;
    dots3<16u>(Gp, Gq, Dp, Dq, cs);
    double Ap = sqrt(Dp), Aq = sqrt(Dq);
    {
      const double nx = fmax(Ap, Aq), ny = fmin(Ap, Aq), nn = nx * ny;
      const bool fits = nn < DBL_MAX, above = nn > PROD_SMALL;
      cs = (cs / ny) / nx;
      const unsigned plain = ssq_plain(Gp[0]) & ssq_plain(Gp[1]) & ssq_plain(Gq[0]) & ssq_plain(Gq[1]) &
                         (unsigned)((ny >= 1.0) ? fits : above);
      if (__ballot(plain == 0u) != 0ull) {
        double vp[8], vq[8];
#pragma unroll
        for (unsigned j = 0u; j < 8u; ++j) {
          vp[j] = R[p * LD + (r & 3u) + 4u * j];
          vq[j] = R[q * LD + (r & 3u) + 4u * j];
        }
        Ap = column_nrm2(R, p, 0u, r & 3u);
        Aq = column_nrm2(R, q, 0u, r & 3u);
        cs = quad_cos(Ap, Aq, vp, vq);
      }
    }
    const bool rot = (fabs(cs) >= MYTOL);
    const double q_p = Aq / Ap, p_q = Ap / Aq;
    const double ct2 = (q_p - p_q) / (2.0 * cs), act = fabs(ct2);
    const bool ortho = rot & !(ct2 <= COT_LIMIT);
    const bool small = act < SQRT_HEPS, large = act >= SQRT_2_HEPS;
    const double sq = pin(sqrt(__fma_rn(act, act, 1.0)));
    const double cot = large ? 2.0 * act : act + (small ? 1.0 : sq);
    double t = copysign(1.0 / cot, ct2);
    const double cr = rsqrt_near1(__fma_rn(t, t, 1.0));
    const bool big = small | (!large & (cr < 1.0));
    double c = big ? cr : 1.0;
    const double tc = t * cs;
    // the norms after the rotation decide which column goes first
    const double Ap2 = Ap * sqrt(__fma_rn(-tc, q_p, 1.0));
    const double Aq2 = Aq * sqrt(__fma_rn(tc, p_q, 1.0));
    bool cross = rot ? !(pos ? (Ap2 >= Aq2) : (Ap2 <= Aq2)) : (pos ? (Ap < Aq) : (Aq < Ap));
    // (a wave of nothing but rotations and swaps: no branch)
    if (__ballot(ortho) == 0ull) {
      apply_pair<16u, 2u, false>(ap, aq, Gp, Gq, rot, cross, true, c, t);
    }
    else {
      if (ortho) {
        // the smaller column loses its component along the larger, which
        // stays or comes first
        cross = !(pos ? (Ap >= Aq) : (Ap <= Aq));
        c = 1.0;
        t = cross ? cs : -cs;
#pragma unroll
        for (unsigned i = 0u; i < 2u; ++i) {
          const double up = Gp[i] / Ap, uq = Gq[i] / Aq;
          aq[16u * i] = cross ? Ap * __fma_rn(-cs, uq, up) : Aq * __fma_rn(-cs, up, uq);
          if (cross) ap[16u * i] = Gq[i];
        }
      }
      else
        apply_pair<16u, 2u, false>(ap, aq, Gp, Gq, rot, cross, true, c, t);
    }
    if (r == 0u) {
      double *const o = L.rot[step & 1u][y];
      o[0] = c;
      o[1] = t;
      o[2] = o[3] = 0.0;
      L.act[step & 1u][y] = (rot ? ACT_ROT : 0u) | (cross ? ACT_CROSS : 0u) | ACT_TRIG;
    }
    my_s += rot ? 1u : 0u;
    my_b += (rot & !ortho & big) ? 1u : 0u;
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------

// J of the pair's 32 columns (J is +1 on the first nplus columns of G):
// npos of them are positive, and they come first; definite is +1 / -1 when
// all / none are, else 0 (share/device_code_nosort_accumV.hpp:53-76, whose
// case nplus = 16 bj + 16 stays mixed with npos = 32).
__device__ __forceinline__ void pair_signs(int definite, unsigned nplus, unsigned bi, unsigned bj,
                                           int &def, bool &hyp, unsigned &npos)
{
  def = definite;
  hyp = false;
  npos = 0u;
  if (definite)
    return;
  if (nplus <= 16u * bi) {
    def = -1;
  }
  else if (nplus > 16u * bj + 16u) {
    def = +1;
    npos = 32u;
  }
  else {
    def = 0;
    hyp = true;
    npos = min(nplus - 16u * bi, 16u) + ((nplus > 16u * bj) ? nplus - 16u * bj : 0u);
  }
}

// One block pair per workgroup.
template <bool SORT, bool DRMAC>
__global__ __launch_bounds__(QR_NT) void k_pair_qr(const double *__restrict__ G, unsigned ldG,
                                                   unsigned nrow, const uint16_t *__restrict__ pairs,
                                                   double *__restrict__ Wout,
                                                   unsigned *__restrict__ flags, RunCtl *__restrict__ ctl,
                                                   const uint8_t *__restrict__ strat0, unsigned s0steps,
                                                   unsigned nswp, int definite, unsigned nplus)
{
  __shared__ QrLds L;
  const unsigned tid = threadIdx.x, l = tid & 63u, w = tid >> 6;
  const unsigned pi = blockIdx.x;
  const unsigned bi = pairs[2u * pi], bj = pairs[2u * pi + 1u];
  static_assert(STRAT0_TAB_BYTES == 64u * sizeof(uint4), "one 16-byte piece per lane of a wave");
  if (tid < 64u)
    reinterpret_cast<uint4 *>(L.S0)[l] = reinterpret_cast<const uint4 *>(strat0)[l];
  if (tid == 0u) {
    L.swp = 0;
    L.cmax = 0u;
    L.cs[0] = L.cb[0] = 0u;
  }

  PairSigns sg;
  pair_signs(definite, nplus, bi, bj, sg.def, sg.hyp, sg.npos);

  // panel loads: lane l takes row l % 32 of the pair's columns 2i + l / 32
  // (i < 8 in block bi, i >= 8 in block bj)
  const unsigned row = l & 31u, half = l >> 5;
  const double *const c0 = G + (size_t)(16u * bi + half) * ldG + row;
  const double *const c1 = G + (size_t)(16u * bj + half) * ldG + row;
  const unsigned npan = nrow / 32u;
  Merge M;
  // panels at .. at + n - 1 in slots s0 .. s0 + n - 1 (slot 0: the running
  // factor), wave w those of slots w and w + 8
  for (unsigned at = 0u, s0 = 0u; at < npan; s0 = 1u) {
    const unsigned n = min(npan - at, QR_PANELS - s0);
    double v[2][16];
#pragma unroll
    for (unsigned h = 0u; h < 2u; ++h) {
      const unsigned sl = w + QR_WAVES * h;
      if (sl >= s0 && sl < s0 + n) {
#pragma unroll
        for (unsigned i = 0u; i < 16u; ++i)
          v[h][i] = ((i < 8u) ? c0 : c1)[(size_t)(2u * (i & 7u)) * ldG + 32u * (at + sl - s0)];
      }
    }
#pragma unroll
    for (unsigned h = 0u; h < 2u; ++h) {
      const unsigned sl = w + QR_WAVES * h;
      if (sl >= s0 && sl < s0 + n) {
#pragma unroll
        for (unsigned i = 0u; i < 16u; ++i)
          L0A(L.R + sl * QR_PANEL, row, 2u * i + half) = v[h][i];
      }
    }
    wave_lds_sync();
#pragma unroll 1
    for (unsigned sl = w; sl < s0 + n; sl += QR_WAVES)
      if (sl >= s0) householder32(L.R + sl * QR_PANEL, l);
    __syncthreads();
    if (!s0) merge_begin(M, L, tid);
#pragma unroll 1
    for (unsigned sl = 1u; sl < s0 + n; ++sl)
      merge_panel(M, L, L.R + sl * QR_PANEL);
    at += n;
  }
  merge_end(M, L);
  // W = I
  for (unsigned e = tid; e < 1024u; e += QR_NT)
    L0A(L.W, e & 31u, e >> 5) = ((e & 31u) == (e >> 5)) ? 1.0 : 0.0;
  __syncthreads();

  unsigned blk_s, blk_b;
  if (DRMAC && SORT && !sg.hyp)
    inner_sweeps_by<QR_LANES>(tid, L, s0steps, nswp, false, blk_s, blk_b,
                              [&](unsigned y, unsigned r, unsigned &my_s, unsigned &my_b, bool &) {
                                drmac_r(L, y, r, s0steps, sg.def, my_s, my_b);
                              });
  else
    inner_sweeps<SORT, QR_LANES>(tid, L, sg, s0steps, nswp, false, blk_s, blk_b);

  if (tid == 0u) {
    // the run's counter: big rotations in the high word, all in the low one;
    // without a big rotation only the low word is added to, with no carry
    // out of it (share/device_code_nosort.hpp:94-103)
    if (blk_s && blk_b)
      atomicAdd(&ctl->cvg, (((unsigned long long)blk_b) << 32) | blk_s);
    else if (blk_s)
      atomicAdd(reinterpret_cast<unsigned *>(&ctl->cvg), blk_s);
    flags[pi] = SORT ? 1u : (blk_s ? 1u : 0u);
  }
  double *const wo = Wout + (size_t)pi * 1024u;
  for (unsigned e = tid; e < 1024u; e += QR_NT)
    wo[e] = L0A(L.W, e & 31u, e >> 5);
}

}  // namespace

void launch_pair_qr(hipStream_t s, bool sort, bool drmac, const double *G, unsigned ldG,
                    unsigned nrow, const uint16_t *pairs, unsigned np, double *W, unsigned *flags,
                    RunCtl *ctl, const uint8_t *strat0, unsigned s0steps, unsigned nswp,
                    int definite, unsigned nplus)
{
  if (sort && drmac)
    hipLaunchKernelGGL((k_pair_qr<true, true>), dim3(np), dim3(QR_NT), 0, s, G, ldG, nrow, pairs, W,
                       flags, ctl, strat0, s0steps, nswp, definite, nplus);
  else if (sort)
    hipLaunchKernelGGL((k_pair_qr<true, false>), dim3(np), dim3(QR_NT), 0, s, G, ldG, nrow, pairs, W,
                       flags, ctl, strat0, s0steps, nswp, definite, nplus);
  else
    hipLaunchKernelGGL((k_pair_qr<false, false>), dim3(np), dim3(QR_NT), 0, s, G, ldG, nrow, pairs, W,
                       flags, ctl, strat0, s0steps, nswp, definite, nplus);
}

}  // namespace hj

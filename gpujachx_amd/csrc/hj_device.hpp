// hj_device.hpp -- device-side scalar arithmetic of the method (gfx950).
// Every operation is an IEEE-754 double operation (fma, +, *, /, sqrt are
// correctly rounded on gfx950), written out explicitly; the translation unit
// is compiled with -ffp-contract=off so no other fusion happens.
#ifndef HJ_DEVICE_HPP
#define HJ_DEVICE_HPP

#include <hip/hip_runtime.h>
#include <cstdint>

namespace hj {

// constants of the method (share/HypJacL.hpp:11-51)
constexpr double SQRT_HEPS = 0x1.6a09e667f3bcdp-27;  // sqrt(2^-53)
constexpr double SQRT_2_HEPS = 0x1p27;               // sqrt(2 / 2^-53)
constexpr double MYTOL = 0x1.6a09e667f3bcdp-51;      // sqrt(32) * 2^-53
constexpr double COSHI_FIX = 0x1.279a74590331cp+0;   // 2/sqrt(3), correctly rounded
constexpr double TANH1_FIX = 0.5;

// x held in a register at this point: the operations producing it are
// issued here, on every path, rather than moved into a later branch (where
// they would run after, not beside, the other work of the step)
__device__ __forceinline__ double pin(double x)
{
  asm volatile("" : "+v"(x));
  return x;
}

__device__ __forceinline__ uint64_t d2u(double x) { return (uint64_t)__double_as_longlong(x); }
__device__ __forceinline__ double u2d(uint64_t u) { return __longlong_as_double((long long)u); }

// m*(y+d)^2 - 1 with exact products; see rsqrt_core.
__device__ __forceinline__ double rs_resid(double m, double y, double d)
{
  const double h = y * y, l = __fma_rn(y, y, -h);
  const double p = m * h, pe = __fma_rn(m, h, -p);
  const double q = m * l;
  const double my = m * y;
  double T = (p - 1.0) + pe;
  T = T + q;
  T = T + (2.0 * d) * my;
  T = T + (m * d) * d;
  return T;
}

// Correctly rounded 1/sqrt(m) for m in [1,4): the hardware reciprocal square
// root refined by two Newton steps y += y(1 - m y^2)/2 lands within an ulp
// (the hardware seed has more than 20 correct bits, so the Newton error is
// far below the final rounding); y then moves to a neighbour when the
// midpoint between them lies on the other side of 1/sqrt(m), judged by the
// sign of m*mid^2 - 1 with fma-exact products.  Straight-line code.
__device__ __forceinline__ double rsqrt_core(double m)
{
  double y = __builtin_amdgcn_rsq(m);
  double h = m * y;
  y = __fma_rn(0.5 * y, __fma_rn(-h, y, 1.0), y);
  h = m * y;
  y = __fma_rn(0.5 * y, __fma_rn(-h, y, 1.0), y);
  const double up = u2d(d2u(y) + 1u), dn = u2d(d2u(y) - 1u);
  const double Tu = rs_resid(m, y, (up - y) * 0.5);
  const double Td = rs_resid(m, y, -((y - dn) * 0.5));
  return (Tu < 0.0) ? up : ((Td > 0.0) ? dn : y);
}

// The same value from one cubic step and one residual: with
// e = 1 - m y0^2 (|e| < 2^-22, the hardware seed), y = y0 (1 + e/2 + 3/8 e^2)
// is within an ulp of 1/sqrt(m); e1 = 1 - m y^2, formed from the exact product
// m y = h + l, has |e1| < 2^-51 and an error below 2^-104, so 1/sqrt(m) =
// y + y e1/2 up to 2^-102.5 relative (the next term, 3/8 e1^2, included).
// Rounding y + (y/2)(e1 +- 2^-100) therefore brackets the rounding of the
// exact value: equal results are the correctly rounded 1/sqrt(m).  They differ
// only for values within 2^-101 of a midpoint of two doubles: sure is false
// there (and true for a NaN), and the caller takes rsqrt_core.  Any m whose
// sqrt is far from the ends of the exponent range will do (the steps scale
// with m): half the instructions of rsqrt_core, whose two midpoint residuals
// cost more than its value.
__device__ __forceinline__ double rsqrt_bracket(double m, bool &sure)
{
  double y = __builtin_amdgcn_rsq(m);
  double h = m * y;
  double e = __fma_rn(-h, y, 1.0);
  y = __fma_rn(y * e, __fma_rn(e, 0.375, 0.5), y);
  h = m * y;
  const double l = __fma_rn(m, y, -h);
  e = __fma_rn(-h, y, 1.0);
  e = __fma_rn(-l, y, e);
  const double yh = 0.5 * y;
  const double lo = __fma_rn(yh, e - 0x1p-100, y), hi = __fma_rn(yh, e + 0x1p-100, y);
  sure = !(hi > lo);
  return lo;
}

// Whether x is a positive normal number with an exponent in [-927, 929): the
// inputs rsqrt_bracket takes unscaled.
__device__ __forceinline__ bool rsqrt_plain_range(double x)
{
  return (unsigned)__double2hiint(x) - 0x06000000u < 0x7a000000u - 0x06000000u;
}

// Correctly rounded 1/sqrt(x).  Replaces my_drsqrt_rn of
// share/device_code_common.hpp:89-133 (whose contract is the correctly
// rounded result).  Own method: x = m * 4^k with m in [1,4), rsqrt_core(m),
// exact rescaling; IEEE special values as the reference returns them.
__device__ __forceinline__ double dev_rsqrt_any(double x)
{
  // special inputs resolved by selects (no branches: the callers' code stays
  // straight-line for the scheduler); the main path also runs on them, its
  // value discarded.  x = mt * 2^e with mt in [0.5, 1) (v_frexp_*, subnormal
  // x included), then x = m * 4^k with m = mt * 2^(2 - e mod 2) in [1, 4)
  const bool special = !((x > 0.0) && (x < __builtin_inf()));  // not positive finite
  const int e = __builtin_amdgcn_frexp_exp(x);
  const double mt = __builtin_amdgcn_frexp_mant(x);
  const int odd = e & 1;
  const double m = __builtin_amdgcn_ldexp(mt, 2 - odd);
  const int k = (e - 2 + odd) >> 1;  // exact: e - 2 + odd is even
  const double y = rsqrt_core(m);
  const double normal = __builtin_amdgcn_ldexp(y, -k);  // exact: the result is a normal number
  const uint64_t b0 = d2u(x);
  double sp = 0.0;                                                   // +inf
  sp = (x < 0.0) ? u2d(0xfff8000000000000ull) : sp;                  // negative: NaN
  sp = (x == 0.0) ? u2d((b0 & 0x8000000000000000ull) | 0x7ff0000000000000ull) : sp;  // +-0: +-inf
  sp = (x != x) ? x + x : sp;                                        // NaN
  return special ? sp : normal;
}

// Correctly rounded 1/sqrt(m) of a rotation's m = 1 +- t^2 (2^-26 < m <= 2,
// or NaN): no scaling, no special values.
__device__ __forceinline__ double rsqrt_near1(double m)
{
  bool sure;
  double y = rsqrt_bracket(m, sure);
  if (__ballot(!sure) != 0ull)
    y = dev_rsqrt_any(m);
  return y;
}

// Lane exchanges by DPP (no LDS traffic): xor 1 and xor 2 are quad permutations.
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v)
{
  // every lane reads a lane of its own row (quad / half-row permutations):
  // no lane keeps an old value, so none is set up
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_xor2(double v) { return dpp_mov<0x4E>(v); }
__device__ __forceinline__ double lane_xor1(double v) { return dpp_mov<0xB1>(v); }

// Row held by lane l of a group of LANES (8 or 16) lanes that share the 32 rows
// of a pivot pair: lane l keeps rows row_of(l) + LANES i.  The reduction's
// partners at distance 4, 2 and 1 are then lanes l ^ 7, l ^ 2 and l ^ 1, each
// one DPP move (half-row mirror, quad permutations); distance 8 is a
// rotation of the 16-lane row by 8.
__device__ __forceinline__ unsigned row_of(unsigned l)
{
  return l ^ ((l & 4u) ? 3u : 0u);
}

// a, b, c computed before anything after this point uses one of them
__device__ __forceinline__ void pin3(double &a, double &b, double &c)
{
  asm volatile("" : "+v"(a), "+v"(b), "+v"(c));
}

// One reduction level of three sums, side by side (one after the other each
// would wait out its own add -> DPP latency).
template <int CTRL>
__device__ __forceinline__ void level3(double &a, double &b, double &c)
{
  const double x = dpp_mov<CTRL>(a), y = dpp_mov<CTRL>(b), z = dpp_mov<CTRL>(c);
  a = a + x;
  b = b + y;
  c = c + z;
  pin3(a, b, c);
}

// Dp = p.p, Dq = q.q, Apq = p.q over the LANES ROWS (32 or 64) rows of a pivot
// pair, p[i], q[i] being row row_of(l) + LANES i: each by the xor butterfly
// (32,) 16,8,4,2,1 of the row distances, the first levels inside the lane.
template <unsigned LANES, unsigned ROWS = 32u / LANES>
__device__ __forceinline__ void dots3(const double *p, const double *q, double &Dp, double &Dq,
                                      double &Apq)
{
  double tp[ROWS], tq[ROWS], tx[ROWS];
#pragma unroll
  for (unsigned i = 0u; i < ROWS; ++i) {
    tp[i] = __fma_rn(p[i], p[i], 0.0);
    tq[i] = __fma_rn(q[i], q[i], 0.0);
    tx[i] = __fma_rn(p[i], q[i], 0.0);
  }
#pragma unroll
  for (unsigned n = ROWS / 2u; n >= 1u; n >>= 1) {
#pragma unroll
    for (unsigned i = 0u; i < n; ++i) {
      tp[i] = tp[i] + tp[i + n];
      tq[i] = tq[i] + tq[i + n];
      tx[i] = tx[i] + tx[i + n];
    }
  }
  Dp = tp[0];
  Dq = tq[0];
  Apq = tx[0];
  pin3(Dp, Dq, Apq);
  if constexpr (LANES >= 16u) level3<0x128>(Dp, Dq, Apq);  // rows 8 apart
  if constexpr (LANES >= 8u) level3<0x141>(Dp, Dq, Apq);   // 4 apart (see row_of)
  level3<0x4E>(Dp, Dq, Apq);
  level3<0xB1>(Dp, Dq, Apq);
}

// Whether |Apq| < sqrt(Dp) sqrt(Dq) tol is certain, as rounded, from the
// squares alone: they say so by 2^-40, far more than the roundings of either
// side, and none of them is near the ends of the exponent range.  (NaN: not.)
__device__ __forceinline__ bool surely_orthogonal(double Apq, double Dp, double Dq, double tol)
{
  const double b = (Dp * Dq) * (tol * tol * (1.0 - 0x1p-40));
  const bool less = Apq * Apq < b, above = b > 0x1p-960, below = b < 0x1p+1000;
  return less & above & below;
}

// 2x2 rotation of share/device_code_common_rotate.hpp:189-237 (USE_RSQRT),
// trigonometric (trig) or hyperbolic, for a pivot pair whose lanes (a multiple of
// four, from a multiple of four on) all hold the same Apq, Dp, Dq; also
// sqrt(Dp) sqrt(Dq).  HYP: trig is set per pair, else every pair is
// trigonometric.  Returns whether the rotation is big.
//   trig: zeta = (Dq-Dp)/(2Apq); |zeta| < sqrt(eps/2): t = 1/(|zeta|+1),
//         |zeta| >= sqrt(2/eps): t = 1/(2|zeta|), c = 1, else
//         t = 1/(|zeta| + sqrt(zeta^2+1)); c = rsqrt(1+t^2); big = c < 1.
//   hyp:  zeta = -(Dq+Dp)/(2Apq); |zeta| >= sqrt(2/eps): t = 1/(2|zeta|),
//         c = 1; |zeta| > 1: t = 1/(|zeta| + sqrt(zeta^2-1)),
//         c = rsqrt(1-t^2), big = c > 1; else c = 2/sqrt(3), t = 1/2.
// Evaluated without divergent branches: every path's operations are issued and
// the taken branch's results are selected, so the values equal the branch
// formulas bit for bit; the reciprocal root is skipped by a wave-uniform branch
// where no lane takes a branch that uses it.  The three square roots -- of
// zeta^2 +- 1, Dp and Dq -- are one instruction sequence,
// on lanes 0, 1 and 2 of every quad, spread by DPP moves (the roots of the
// norms are wanted late, by the convergence test).  (Pinned values: operands of
// selects, which would otherwise become branches.)
template <bool HYP>
__device__ __forceinline__ bool rot_quad(bool trig, double Apq, double Dp, double Dq, unsigned l,
                                         double &c, double &t, double &Dpq_)
{
  if (!HYP) trig = true;
  const double h = Dq + (trig ? -Dp : Dp);
  const double qz = h / (2.0 * Apq);
  const double ct2 = trig ? qz : -qz;
  const double CT2 = fabs(ct2);
  const bool large = CT2 >= SQRT_2_HEPS;
  const bool small = trig & (CT2 < SQRT_HEPS);
  const bool fix = !trig & !large & !(CT2 > 1.0);
  const double z = pin(__fma_rn(CT2, CT2, trig ? 1.0 : -1.0));
  const unsigned q = l & 3u;
  const double s3 = sqrt((q == 1u) ? Dp : ((q == 2u) ? Dq : z));
  const double sq = dpp_mov<0x00>(s3);
  Dpq_ = dpp_mov<0x55>(s3) * dpp_mov<0xAA>(s3);
  // CT2 + CT2, CT2 + 1 or CT2 + sqrt
  const double cot = CT2 + (large ? CT2 : (small ? 1.0 : sq));
  const double rcot = pin(1.0 / cot);
  const double tt = fix ? TANH1_FIX : copysign(rcot, ct2);
  double cr = 1.0;
  if (__ballot(!large & !fix) != 0ull)
    cr = pin(rsqrt_near1(__fma_rn(trig ? tt : -tt, tt, 1.0)));
  c = large ? 1.0 : (fix ? COSHI_FIX : cr);
  t = tt;
  const bool off1 = HYP ? (trig ? (cr < 1.0) : (cr > 1.0)) : (cr < 1.0);
  return !large & (small | fix | off1);
}

__device__ __forceinline__ double readlane_d(double v, int lane)
{
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}

// A double in LDS: helpers that take generic pointers to LDS (a caller's
// dynamic LDS region, a function not inlined) access them through this type,
// so the accesses are LDS instructions (ds_*) rather than flat ones.
typedef __attribute__((address_space(3))) double lds_f64;

// LDS of one wave's pair state: the 32x32 matrices R and W column-major with
// leading dimension 33
constexpr unsigned L0LD = 33u;
#define L0A(A, r, c) (A)[(c) * L0LD + (r)]

// the LDS accesses of a wave before this point complete before any after it
__device__ __forceinline__ void wave_lds_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// In-place 32x32 Cholesky by one wave, share/device_code_common_Cholesky.hpp:58-158
// (USE_RSQRT): column k is scaled by rsqrt(A(k,k)), the diagonal set to
// sqrt(A(k,k)), then A(x,j) = fma(-A(x,k), A(j,k), A(x,j)) for the rows
// x >= j > k.  A: the Gram's lower triangle in LDS (A[c * LD + r] = A(r,c),
// c <= r); on return A holds R = L^T (zeros below the diagonal).  col: 64
// doubles of LDS for the column broadcast.  check: whether every factor entry
// is finite and the diagonal positive (wave-uniform).
//
// chol32_any takes any input: column by column in LDS, lane l on row l % 32
// of the columns j = l/32, l/32 + 2, ...
template <unsigned LD>
__device__ __forceinline__ bool chol32_any(lds_f64 *A, lds_f64 *col, unsigned l, bool check)
{
  const unsigned x = l & 31u, h = l >> 5;
#pragma unroll 1
  for (unsigned k = 0u; k < 32u; ++k) {
    const double akk = A[k * LD + k];
    const double v = A[k * LD + x];
    const double rk = dev_rsqrt_any(akk), dk = sqrt(akk);
    const double w = (x == k) ? dk : v * rk;
    wave_lds_sync();
    if (x >= k) A[k * LD + x] = w;
    col[x] = w;
    wave_lds_sync();
#pragma unroll 1
    for (unsigned j = k + 1u + h; j < 32u; j += 2u)
      if (x >= j) A[j * LD + x] = __fma_rn(-w, col[j], A[j * LD + x]);
    wave_lds_sync();
  }
  bool ok = true;
#pragma unroll 1
  for (unsigned c = h; c < 32u; c += 2u) {
    const double v = A[c * LD + x];
    if (check && c <= x) ok = ok && (fabs(v) <= 0x1.fffffffffffffp+1023);
    if (check && c == x) ok = ok && (v > 0.0);
  }
  // R = L^T in place, one column against one row at a time
#pragma unroll 1
  for (unsigned c = 0u; c < 32u; ++c) {
    const double v = A[c * LD + x];
    wave_lds_sync();
    if (h == 0u && x > c) {
      A[x * LD + c] = v;
      A[c * LD + x] = 0.0;
    }
    wave_lds_sync();
  }
  return !check || (__ballot(ok) == ~0ull);
}

// Lane l keeps row x = l % 32 of the columns c = 2i + l/32 (i = 0..15), so
// one instruction updates an even column in one half of the wave and an odd
// one in the other: 16 registers and half the update instructions of a
// row-per-lane layout.  The updates run on every row; above the diagonal
// they produce values that no later step reads (the pivot is read on the
// diagonal, the broadcast column below it) and that are not stored.  The
// next pivot A(k+1,k+1) - L(k+1,k)^2 is formed from two readlanes as soon
// as column k is scaled, so its rsqrt (rsqrt_bracket: the chain of the 32
// pivots is this routine's time) runs beside the column's updates.  The
// diagonal stays unscaled until the end, where one square root instruction
// serves all 32 entries.  A pivot that rsqrt_bracket does not settle sends
// the matrix, still whole in LDS, to chol32_any.
template <unsigned LD>
__device__ __forceinline__ bool chol32_wave(double *A_, double *col_, unsigned l, bool check)
{
  lds_f64 *const A = (lds_f64 *)A_;
  lds_f64 *const col = (lds_f64 *)col_;
  const unsigned x = l & 31u, h = l >> 5;
  double b[16];
#pragma unroll
  for (unsigned i = 0u; i < 16u; ++i) {
    const unsigned c = 2u * i + h;
    b[i] = (c <= x) ? A[c * LD + x] : 0.0;
  }
  // the lanes of the other half than the pivot column's write beside col
  // (no branch, no select); xh[hk]: x in the half of the even (odd) columns,
  // 0 in the other
  lds_f64 *const cw[2] = {col + x + 32u * h, col + x + 32u * (h ^ 1u)};
  const unsigned xh[2] = {h ? 0u : x, h ? x : 0u};
  double akk = readlane_d(b[0], 0);
  bool sure;
  double rk = rsqrt_bracket(akk, sure);
  unsigned long long bad = __ballot(!(sure && rsqrt_plain_range(akk)));
#pragma unroll
  for (unsigned k = 0u; k + 1u < 32u; ++k) {
    const unsigned ik = k >> 1, hk = k & 1u, k1 = k + 1u;
    const double u = pin(b[ik] * rk);
    *cw[hk] = u;
    b[ik] = pin((xh[hk] > k) ? u : b[ik]);
    const double lk = readlane_d(u, hk * 32u + k1);
    const double d1 = readlane_d(b[k1 >> 1], (k1 & 1u) * 32u + k1);
    akk = __fma_rn(-lk, lk, d1);
    // the other half reads what this half stored: without the fence the
    // compiler may issue a lane's read of col[x] before the other lane's
    // store
    wave_lds_sync();
    const double lx = col[x];
    double cv[16];
#pragma unroll
    for (unsigned i = k1 >> 1; i < 16u; ++i)
      cv[i] = col[2u * i + h];
    // the column's reads are issued here, all of them, and used after the
    // pivot's chain has started
    __builtin_amdgcn_sched_barrier(0);
    rk = rsqrt_bracket(akk, sure);
    bad |= __ballot(!(sure && rsqrt_plain_range(akk)));
#pragma unroll
    for (unsigned i = k1 >> 1; i < 16u; ++i) {
      // column 2i + h; for i = k1/2 with k1 odd, only half 1's column is
      // beyond k
      const double f = __fma_rn(-lx, cv[i], b[i]);
      b[i] = ((k1 & 1u) && i == (k1 >> 1) && h == 0u) ? b[i] : f;
    }
    // settled here: left to itself the compiler delays the updates to their
    // columns' pivots and the test to the end, all operands in registers
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" : "+s"(bad));
#pragma unroll
    for (unsigned i = k1 >> 1; i < 16u; ++i)
      asm volatile("" : "+v"(b[i]));
    wave_lds_sync();
  }
  if (bad)
    return chol32_any<LD>(A, col, l, check);
  bool ok = true;
  if (check) {
    // (the diagonal is positive: its pivots were in rsqrt_bracket's range)
#pragma unroll
    for (unsigned i = 0u; i < 16u; ++i) {
      const unsigned c = 2u * i + h;
      if (c < x) ok = ok && (fabs(b[i]) <= 0x1.fffffffffffffp+1023);
    }
    ok = (__ballot(ok) == ~0ull);
  }
#pragma unroll
  for (unsigned i = 0u; i < 16u; ++i) {
    const unsigned c = 2u * i + h;
    A[x * LD + c] = (c <= x) ? b[i] : 0.0;
  }
  wave_lds_sync();
  const double d = sqrt(A[x * LD + x]);
  wave_lds_sync();
  A[x * LD + x] = d;
  return ok;
}

// Sum of the 32 rows of one pivot pair held by 4 lanes, lane r holding rows
// r + 4k as v[k]: the xor butterfly 16,8,4,2,1 of the reference's 32-lane
// reduction (levels 16, 8 and 4 inside the lane, 2 and 1 across lanes).
__device__ __forceinline__ double sum4x8(const double *v)
{
  const double a0 = v[0] + v[4], a1 = v[1] + v[5], a2 = v[2] + v[6], a3 = v[3] + v[7];
  double s = (a0 + a2) + (a1 + a3);
  s = s + lane_xor2(s);
  s = s + lane_xor1(s);
  return s;
}

__device__ __forceinline__ unsigned wave_sum_u(unsigned v)
{
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1)
    v += (unsigned)__shfl_xor((int)v, o, 64);
  return v;
}

// Level-0 sweeps of one block pair by one wave (the inner Jacobi of
// share/device_code_nosort.hpp:4-222 for SORT false,
// share/device_code_cdsort_KISS.hpp:4-260 and share/device_code_cdsort.hpp:25-167
// for SORT true).  R: the Cholesky factor, W: the identity on entry, column
// c at c LD (LD = 36: of the 16 slots' columns, four rows each, those of
// neighbouring pairs fall into different LDS banks; 33 made fourfold
// conflicts).  Slot y = l/4 takes pivot pair y of a step, lane r = l%4 of
// the slot holds rows r + 4k of the two columns; the pivot pairs of a step
// touch disjoint columns, so one wave-level LDS sync per step suffices.
// Returns the rotation counts of all its sweeps (the reference's counting:
// a sweep without a rotation ends the loop and adds nothing) in every lane,
// and whether a pivot pair was swapped by the sort rule (W is the identity
// exactly when nothing was rotated or swapped).
template <bool SORT, unsigned LD>
__device__ __forceinline__ void wave_level0(double *R_, double *W_, const uint8_t *S0,
                                            unsigned s0steps, unsigned nswp, int def, bool hyp,
                                            unsigned npos, unsigned l, unsigned &out_s,
                                            unsigned &out_b, bool &out_swap)
{
  lds_f64 *const R = (lds_f64 *)R_;
  lds_f64 *const W = (lds_f64 *)W_;
  const unsigned y = l >> 2, r = l & 3u;
  unsigned blk_s = 0u, blk_b = 0u;
  bool swapped = false;
  for (unsigned swp = 0u; swp < nswp; ++swp) {
    unsigned my_s = 0u, my_b = 0u;
    for (unsigned step = 0u; step < s0steps; ++step) {
      const unsigned p = S0[(step * 16u + y) * 2u], q = S0[(step * 16u + y) * 2u + 1u];
      double Gp[8], Gq[8];
#pragma unroll
      for (unsigned k = 0u; k < 8u; ++k) {
        Gp[k] = R[p * LD + r + 4u * k];
        Gq[k] = R[q * LD + r + 4u * k];
      }
      double Dp, Dq, Apq;
      dots3<4u>(Gp, Gq, Dp, Dq, Apq);
      int pdef = def;
      if (hyp) {
        if ((p < npos) && (q < npos)) pdef = +1;
        else if ((p >= npos) && (q >= npos)) pdef = -1;
        else pdef = 0;
      }
      bool trig;
      if (!SORT) trig = !hyp || pdef;
      else trig = (pdef != 0);
      // the rotation on every lane; only a transforming pair uses it
      double c, t, Dpq_;
      const bool rot_b = rot_quad<true>(trig, Apq, Dp, Dq, l, c, t, Dpq_);
      const double Apq_ = fabs(Apq);
      const int transf_s = !(Apq_ < (Dpq_ * MYTOL));
      int transf_b = 0;
      if (transf_s) {
        // (W's columns: the same lane reads and writes the same entries)
        double Vp[8], Vq[8];
#pragma unroll
        for (unsigned k = 0u; k < 8u; ++k) {
          Vp[k] = W[p * LD + r + 4u * k];
          Vq[k] = W[q * LD + r + 4u * k];
        }
        transf_b = rot_b ? 1 : 0;
        const double t_ = trig ? -t : t;
        if (SORT && trig) {
          Dp = __fma_rn(t, Apq, Dp);
          Dq = __fma_rn(t_, Apq, Dq);
        }
        bool keep = true;
        if (SORT)
          keep = (!pdef) || ((pdef > 0) && (Dp >= Dq)) || ((pdef < 0) && (Dp <= Dq));
        const unsigned PP = keep ? p : q, QQ = keep ? q : p;
#pragma unroll
        for (unsigned k = 0u; k < 8u; ++k) {
          // big rotation: scale by c; otherwise c == 1 exactly (rot_quad), and
          // c * x is x
          const double rp = __fma_rn(t_, Gq[k], Gp[k]), rq = __fma_rn(t, Gp[k], Gq[k]);
          const double wp = __fma_rn(t_, Vq[k], Vp[k]), wq = __fma_rn(t, Vp[k], Vq[k]);
          R[PP * LD + r + 4u * k] = c * rp;
          R[QQ * LD + r + 4u * k] = c * rq;
          W[PP * LD + r + 4u * k] = c * wp;
          W[QQ * LD + r + 4u * k] = c * wq;
        }
      }
      else if (SORT && (((pdef > 0) && (Dp < Dq)) || ((pdef < 0) && (Dq < Dp)))) {
        double Vp[8], Vq[8];
#pragma unroll
        for (unsigned k = 0u; k < 8u; ++k) {
          Vp[k] = W[p * LD + r + 4u * k];
          Vq[k] = W[q * LD + r + 4u * k];
        }
#pragma unroll
        for (unsigned k = 0u; k < 8u; ++k) {
          R[p * LD + r + 4u * k] = Gq[k];
          R[q * LD + r + 4u * k] = Gp[k];
          W[p * LD + r + 4u * k] = Vq[k];
          W[q * LD + r + 4u * k] = Vp[k];
        }
        swapped = true;
      }
      my_s += (unsigned)transf_s;
      my_b += (unsigned)transf_b;
      wave_lds_sync();
    }
    // every lane of a slot holds the slot's counts: sum over the wave / 4
    const unsigned swp_s = wave_sum_u(my_s) >> 2, swp_b = wave_sum_u(my_b) >> 2;
    if (swp_s) {
      blk_s += swp_s;
      blk_b += swp_b;
    }
    else
      break;
  }
  out_s = blk_s;
  out_b = blk_b;
  out_swap = __ballot(swapped) != 0ull;
}

}  // namespace hj

#endif

// hj_visit.hpp -- the visit of one 32-column block pair by a workgroup: 32x32
// Cholesky of the pair's Gram, the inner Jacobi sweep(s) on R accumulating W,
// the counters and the visit record.  Shared by the kernels that only visit
// (k_pair, k_stage: hj_kernels.hip) and the whole step (k_step: hj_step.hip).
#ifndef HJ_VISIT_HPP
#define HJ_VISIT_HPP

#include "hj_device.hpp"
#include "hj_kernels.hpp"

namespace hj {

#define LDR 33u
#define RA(A, r, c) (A)[(c) * LDR + (r)]
// LDS of one pair visit
struct PairLds {
  static constexpr unsigned N = 32u, LD = LDR;  // order and leading dimension of R and W
  static constexpr double TOL = MYTOL;          // of the convergence test
  double R[32u * LDR];
  double W[32u * LDR];
  double cholcol[64];
  double diag[32];        // the Gram's diagonal
  double rot[2][16][4];   // per step parity and pivot pair: c, t, |Apq|, |p| |q|
  unsigned act[2][16];    // ... what happens to its columns (ACT_*)
  unsigned cs[2], cb[2];  // rotations of an inner sweep, by its parity
  unsigned cmax;          // bits of the largest cosine of the first inner sweep
  float bnorm[2];
  int chol_ok;
  int swp;    // a pivot pair was swapped by the sort rule
  __attribute__((aligned(16))) uint8_t S0[STRAT0_TAB_BYTES];
};

// what a step does to a pivot pair's columns of R and W
constexpr unsigned ACT_ROT = 1u;    // rotated
constexpr unsigned ACT_CROSS = 2u;  // the results change places (with ACT_ROT or alone)
constexpr unsigned ACT_TRIG = 4u;   // the rotation is trigonometric
constexpr unsigned ACT_NORMS = 8u;  // no rotation: |p|^2 and |q|^2 in place of c and t

// The columns of M (R or W) of a pivot pair after the step: lane l of the
// pair's group holds rows row + LANES i as P[i], Q[i]; ap, aq: the first of
// them in LDS.  Without branches: an untouched pair is stored as it is.
template <unsigned LANES, unsigned ROWS, bool HYP>
__device__ __forceinline__ void apply_pair(lds_f64 *ap, lds_f64 *aq, const double *P,
                                           const double *Q, bool rot, bool cross, bool trig,
                                           double c, double t)
{
  lds_f64 *const A = cross ? aq : ap, *const B = cross ? ap : aq;
  const double t_ = (!HYP || trig) ? -t : t;
  // every pair of the wave rotates: no selects (worth the branch where a lane
  // holds eight rows: 4608 x 2048 at width 32 263.7 -> 260.3 ms, in three runs in
  // turn, the runs of one side within 0.1 %)
  if (ROWS > 4u && __ballot(!rot) == 0ull) {
    double x[ROWS], y[ROWS];
#pragma unroll
    for (unsigned i = 0u; i < ROWS; ++i) {
      x[i] = c * __fma_rn(t_, Q[i], P[i]);
      y[i] = c * __fma_rn(t, P[i], Q[i]);
    }
#pragma unroll
    for (unsigned i = 0u; i < ROWS; ++i) {
      A[LANES * i] = x[i];
      B[LANES * i] = y[i];
    }
    return;
  }
  double a[ROWS], b[ROWS];
#pragma unroll
  for (unsigned i = 0u; i < ROWS; ++i) {
    // big rotation: scale by c; otherwise c == 1 exactly (rot_quad), and
    // c * x is x
    const double x = pin(c * __fma_rn(t_, Q[i], P[i])), y = pin(c * __fma_rn(t, P[i], Q[i]));
    a[i] = rot ? x : P[i];
    b[i] = rot ? y : Q[i];
  }
#pragma unroll
  for (unsigned i = 0u; i < ROWS; ++i) {
    A[LANES * i] = a[i];
    B[LANES * i] = b[i];
  }
}

// LDS column of a pivot index, fetched ahead: the operands of the next step's
// reads are ready when its barrier opens
__device__ __forceinline__ unsigned pinu(unsigned x)
{
  asm volatile("" : "+v"(x));
  return x;
}

// One level-0 sweep on R: lane r of group y takes pivot pair y of every step.
// Counts its rotations and leaves each step's (c, t, ...) for the W waves.
template <bool SORT, unsigned LANES, bool HYP, class Lds>
__device__ __forceinline__ void level0_r(Lds &L, unsigned y, unsigned r, unsigned s0steps,
                                         int def, unsigned npos, unsigned &my_s, unsigned &my_b,
                                         bool &swapped)
{
  constexpr unsigned ROWS = Lds::N / LANES, LD = Lds::LD, PAIRS = Lds::N / 2u;
  lds_f64 *const M = (lds_f64 *)L.R + row_of(r);
  const uint16_t *const S0 = reinterpret_cast<const uint16_t *>(L.S0) + y;
  // sorted definite pairs: columns by decreasing D for J = I, by increasing
  // D for J = -I: descending in D xor this sign
  const uint64_t neg0 = (!HYP && def < 0) ? 0x8000000000000000ull : 0ull;
  unsigned pq = S0[0];
  unsigned p = pq & 255u, q = pq >> 8, op = p * LD, oq = q * LD;
  bool calm = false;
#pragma unroll 1
  for (unsigned step = 0u; step < s0steps; ++step) {
    lds_f64 *const ap = M + op, *const aq = M + oq;
    double Gp[ROWS], Gq[ROWS];
#pragma unroll
    for (unsigned i = 0u; i < ROWS; ++i) {
      Gp[i] = ap[LANES * i];
      Gq[i] = aq[LANES * i];
    }
    pq = S0[PAIRS * min(step + 1u, s0steps - 1u)];
    bool trig = true, inorder = SORT;
    uint64_t neg = neg0;
    if (HYP) {
      const bool pp = p < npos, qp = q < npos;
      trig = (pp == qp);
      neg = pp ? 0ull : 0x8000000000000000ull;
      inorder = SORT & trig;
    }
    double Dp, Dq, Apq;
    dots3<LANES, ROWS>(Gp, Gq, Dp, Dq, Apq);
    const double Apq_ = fabs(Apq);
    // No pair of the wave rotates: at most swaps.  Asked only after a step
    // without a rotation: the test would be in the chain of a step with one
    // (40 of its 1490 cycles), and visits are calm or busy as a whole.
    if (calm && __ballot(!surely_orthogonal(Apq, Dp, Dq, Lds::TOL)) == 0ull) {
      const bool cross = SORT & inorder & (u2d(d2u(Dp) ^ neg) < u2d(d2u(Dq) ^ neg));
      if (SORT && __ballot(cross) != 0ull) {
        swapped = swapped | cross;
        apply_pair<LANES, ROWS, HYP>(ap, aq, Gp, Gq, false, cross, trig, 1.0, 0.0);
      }
      if (r == 0u) {
        double *const o = L.rot[step & 1u][y];
        o[0] = Dp;
        o[1] = Dq;
        o[2] = Apq_;
        L.act[step & 1u][y] = (cross ? ACT_CROSS : 0u) | ACT_NORMS;
      }
      p = pq & 255u;
      q = pq >> 8;
      op = pinu(p * LD);
      oq = pinu(q * LD);
      __syncthreads();
      continue;
    }
    // the rotation on every lane; only a transforming pair uses it
    double c, t, Dpq_;
    const bool big = rot_quad<HYP>(trig, Apq, Dp, Dq, r, c, t, Dpq_);
    const bool transf = !(Apq_ < (Dpq_ * Lds::TOL));
    bool cross = false;
    if (SORT) {
      // rotated: unless in order afterwards; not rotated: when out of order
      const double Ep = pin(__fma_rn(t, Apq, Dp)), Eq = pin(__fma_rn(-t, Apq, Dq));
      const bool ge = u2d(d2u(Ep) ^ neg) >= u2d(d2u(Eq) ^ neg);
      const bool lt = u2d(d2u(Dp) ^ neg) < u2d(d2u(Dq) ^ neg);
      cross = inorder & ((transf & !ge) | (!transf & lt));
      swapped = swapped | (cross & !transf);
    }
    apply_pair<LANES, ROWS, HYP>(ap, aq, Gp, Gq, transf, cross, trig, c, t);
    if (r == 0u) {
      double *const o = L.rot[step & 1u][y];
      o[0] = c;
      o[1] = t;
      o[2] = Apq_;
      o[3] = Dpq_;
      L.act[step & 1u][y] = (transf ? ACT_ROT : 0u) | (cross ? ACT_CROSS : 0u) |
                            (trig ? ACT_TRIG : 0u);
    }
    my_s += transf ? 1u : 0u;
    my_b += (transf & big) ? 1u : 0u;
    calm = __ballot(transf) == 0ull;
    p = pq & 255u;
    q = pq >> 8;
    op = pinu(p * LD);
    oq = pinu(q * LD);
    __syncthreads();
  }
}

// The same sweep's rotations applied to W, each step's between the barrier
// that ends it on the R waves and the next; with cosines, the largest
// |Apq| / (|p| |q|).
template <unsigned LANES, class Lds>
__device__ __forceinline__ void level0_w(Lds &L, unsigned y, unsigned r, unsigned s0steps,
                                         bool cosines)
{
  constexpr unsigned ROWS = Lds::N / LANES, LD = Lds::LD, PAIRS = Lds::N / 2u;
  lds_f64 *const M = (lds_f64 *)L.W + row_of(r);
  const uint16_t *const S0 = reinterpret_cast<const uint16_t *>(L.S0) + y;
  double my_cos = 0.0;
#pragma unroll 1
  for (unsigned step = 0u; step < s0steps; ++step) {
    const unsigned pq = S0[PAIRS * step];
    const unsigned op = pinu((pq & 255u) * LD), oq = pinu((pq >> 8) * LD);
    __syncthreads();
    const double *const o = L.rot[step & 1u][y];
    const unsigned act = L.act[step & 1u][y];
    if (__ballot((act & (ACT_ROT | ACT_CROSS)) != 0u) != 0ull) {
      lds_f64 *const ap = M + op, *const aq = M + oq;
      double P[ROWS], Q[ROWS];
#pragma unroll
      for (unsigned i = 0u; i < ROWS; ++i) {
        P[i] = ap[LANES * i];
        Q[i] = aq[LANES * i];
      }
      apply_pair<LANES, ROWS, true>(ap, aq, P, Q, (act & ACT_ROT) != 0u, (act & ACT_CROSS) != 0u,
                                    (act & ACT_TRIG) != 0u, o[0], o[1]);
    }
    if (cosines) {
      const double cn = o[2], cd = (act & ACT_NORMS) ? sqrt(o[0]) * sqrt(o[1]) : o[3];
      my_cos = fmax(my_cos, (cd > 0.0) ? cn / cd : 0.0);
    }
  }
  // (a nonnegative float's bits order as the float does)
  if (cosines && r == 0u)
    atomicMax(&L.cmax, __float_as_uint((float)my_cos));
}

// J of a pair's 32 columns, share/device_code_nosort_accumV.hpp:53-76: def +1
// / -1 where all / none are positive, else 0 (hyp) with the first npos positive
struct PairSigns {
  int def;
  unsigned npos;
  bool hyp;
};

__device__ __forceinline__ PairSigns pair_signs16(int definite, unsigned nplus, unsigned iBlk,
                                                  unsigned jBlk)
{
  PairSigns s = {definite, 0u, false};
  if (!definite) {
    const unsigned ifc0 = iBlk * 16u, ifc1 = jBlk * 16u;
    if (nplus <= ifc0) { s.npos = 0u; s.def = -1; }
    else if (nplus <= ifc0 + 16u) { s.npos = nplus - ifc0; s.def = 0; }
    else if (nplus <= ifc1) { s.npos = 16u; s.def = 0; }
    else if (nplus <= ifc1 + 16u) { s.npos = 16u + (nplus - ifc1); s.def = 0; }
    else { s.npos = 32u; s.def = +1; }
    s.hyp = (s.def == 0);
  }
  return s;
}

// Inner Jacobi: share/device_code_nosort.hpp:4-222 (SORT false),
// share/device_code_cdsort_KISS.hpp:4-260 and share/device_code_cdsort.hpp:25-167
// (SORT true): up to nswp level-0 sweeps by the N LANES threads of a workgroup,
// half of them on R, half on W.  Returns, in every thread, the rotations.
// on_r: one sweep on R by lane r of pivot pair y (level0_r, or another with
// its counts and its steps' (c, t) and ACT_* in L).
template <unsigned LANES, class Lds, class OnR>
__device__ __forceinline__ void inner_sweeps_by(unsigned tid, Lds &L, unsigned s0steps, unsigned nswp,
                                                bool cosines, unsigned &blk_s, unsigned &blk_b,
                                                OnR on_r)
{
  constexpr unsigned NT = Lds::N * LANES;
  const bool onR = tid < NT / 2u;  // this wave's matrix: R or W
  const unsigned ht = tid & (NT / 2u - 1u);
  const unsigned y = ht / LANES, r = ht & (LANES - 1u);
  blk_s = blk_b = 0u;
  for (unsigned swp = 0u; swp < nswp; ++swp) {
    unsigned my_s = 0u, my_b = 0u;
    bool swapped = false;
    if (!onR)
      level0_w<LANES>(L, y, r, s0steps, cosines && swp == 0u);
    else
      on_r(y, r, my_s, my_b, swapped);
    // every lane of a pair's group holds its counts
    if (onR && r == 0u && my_s) {
      atomicAdd(&L.cs[swp & 1u], my_s);
      atomicAdd(&L.cb[swp & 1u], my_b);
    }
    if (onR && swapped)
      L.swp = 1;
    __syncthreads();
    const unsigned swp_s = L.cs[swp & 1u];
    // (the other parity was read before this sweep's steps)
    if (tid == 0u)
      L.cs[(swp + 1u) & 1u] = 0u;
    if (tid == 64u)
      L.cb[(swp + 1u) & 1u] = 0u;
    if (!swp_s)
      break;
    blk_s += swp_s;
    blk_b += L.cb[swp & 1u];
  }
}

template <bool SORT, unsigned LANES, class Lds>
__device__ __forceinline__ void inner_sweeps(unsigned tid, Lds &L, const PairSigns &sg, unsigned s0steps,
                                             unsigned nswp, bool cosines, unsigned &blk_s, unsigned &blk_b)
{
  inner_sweeps_by<LANES>(tid, L, s0steps, nswp, cosines, blk_s, blk_b,
                         [&](unsigned y, unsigned r, unsigned &my_s, unsigned &my_b, bool &swapped) {
                           if (sg.hyp)
                             level0_r<SORT, LANES, true>(L, y, r, s0steps, sg.def, sg.npos, my_s, my_b, swapped);
                           else
                             level0_r<SORT, LANES, false>(L, y, r, s0steps, sg.def, sg.npos, my_s, my_b, swapped);
                         });
}

// The visit's LDS before its Gram: level-0 table (16 bytes a thread), W = I,
// counters.
template <unsigned NT>
__device__ __forceinline__ void visit_init(unsigned tid, PairLds &L,
                                           const uint8_t *__restrict__ strat0)
{
  if (tid < STRAT0_TAB_BYTES / 16u)
    reinterpret_cast<uint4 *>(L.S0)[tid] = reinterpret_cast<const uint4 *>(strat0)[tid];
  for (unsigned e = tid; e < 1024u; e += NT)
    RA(L.W, e & 31u, e >> 5) = ((e & 31u) == (e >> 5)) ? 1.0 : 0.0;
  if (tid == 0u) {
    L.swp = 0;
    L.cmax = 0u;
    L.cs[0] = L.cb[0] = 0u;
  }
}

// entry e of a Gram partial (tiles 00, 10, 11 in the MFMA output layout) into
// R's lower triangle
__device__ __forceinline__ void gram_entry(PairLds &L, unsigned e, double s)
{
  const unsigned tile = e >> 8, l = (e >> 2) & 63u, r = e & 3u;
  const unsigned i = 4u * r + (l >> 4), j = l & 15u;
  const unsigned row = (tile == 0u) ? i : (16u + i);
  const unsigned col = (tile == 2u) ? (16u + j) : j;
  RA(L.R, row, col) = s;
  if (row == col) L.diag[row] = s;
}

// visit_init and the Gram from the chunk partials of pair pi
template <unsigned NT>
__device__ __forceinline__ void visit_load(unsigned tid, unsigned pi, PairLds &L,
                                           const double *__restrict__ part, unsigned nchunk,
                                           const uint8_t *__restrict__ strat0)
{
  // sum of the chunk partials in chunk order: a thread's entries with all
  // their chunk loads in flight together (one memory round trip)
  const double *const pp = part + (size_t)pi * nchunk * 768u;
  constexpr unsigned NE = (768u + NT - 1u) / NT;
  double v[NE][MAX_GRAM_CHUNKS];
#pragma unroll
  for (unsigned q = 0u; q < NE; ++q)
#pragma unroll
    for (unsigned c = 0u; c < MAX_GRAM_CHUNKS; ++c)
      if (c < nchunk && tid + NT * q < 768u) v[q][c] = pp[(size_t)c * 768u + tid + NT * q];
  visit_init<NT>(tid, L, strat0);
#pragma unroll
  for (unsigned q = 0u; q < NE; ++q) {
    const unsigned e = tid + NT * q;
    if (e >= 768u) break;
    double s = v[q][0];
#pragma unroll
    for (unsigned c = 1u; c < MAX_GRAM_CHUNKS; ++c)
      if (c < nchunk) s = s + v[q][c];
    gram_entry(L, e, s);
  }
}

// One pair visit by the 32 LANES threads of a workgroup (LANES = 16 or 8
// lanes per pivot pair).  The first half of the waves keeps R: per level-0
// step the dot products, the rotation, the update of R.  The other half
// applies the same rotations to W one step behind, from the step's (c, t) in
// LDS, and does the bookkeeping (the largest cosine), so that neither is in
// the chain of the 31 dependent steps; a barrier per step is all that orders
// the two (the pivot pairs of a step touch disjoint columns).  A step is
// bound by that chain -- LDS reads, five reduction levels, division, square
// root, division, reciprocal root, the update and the barrier -- and by the
// instructions one wave issues on it, so the lanes share the square roots
// (rot_quad), the rows are laid out for one-move reduction levels (row_of)
// and the next step's pivot indices are fetched ahead.
//
// Measured (cycles of 2.4 GHz, 512 x 256 in k_pair's LANES = 16): partial sums
// 3.3K, Cholesky 11.4K (23.4K with the column's reads waited for one by one),
// a level-0 sweep 46K = 1490 a step, end 3K; 27 us a visit, 29 us a launch,
// where two waves of 8 lanes a pair, each with both R and W, took 51 us.
// LANES = 8 (half the waves): 33.5 us, 4: 42 us.  k_stage takes 8, the
// largest that its 256-thread workgroups hold; its items set its pace, and
// one visit a workgroup there times the same as two (8192 x 8192: 1.29 s).
// L: visit_init and the Gram's entries written, not yet synchronized.  plan:
// the visit's plan (PLAN_FP64 without a plan); not PLAN_SKIP.  Returns, in
// every thread, whether W (in L.W, synchronized) differs from the identity;
// writes the record and, unless flags is null (k_step, which updates itself),
// flags[pi].
template <bool SORT, unsigned LANES>
__device__ __forceinline__ bool visit_core(unsigned tid, unsigned pi, PairLds &L,
                                           const PairSigns &sg, unsigned *__restrict__ flags,
                                           RunCtl *__restrict__ ctl, VisitRec *__restrict__ rec,
                                           uint8_t plan, unsigned s0steps, unsigned nswp)
{
  __syncthreads();
  // Cholesky, share/device_code_common_Cholesky.hpp:58-158 (USE_RSQRT):
  // column k scaled by rsqrt(A(k,k)), diagonal sqrt(A(k,k)), then
  // A(x,j) = fma(-A(x,k), A(j,k), A(x,j)) for x >= j > k; R = L^T.
  if (tid < 64u) {
    // a Gram from the split products may miss positive definiteness (nearly
    // dependent columns): then no update, FP64 at the next visit
    const bool ok = chol32_wave<LDR>(L.R, L.cholcol, tid, plan == PLAN_SPLIT);
    if (tid == 0u) L.chol_ok = ok ? 1 : 0;
  }
  else if (tid < 66u) {
    // squared Frobenius norms of the two blocks, for the visit record
    double sn = 0.0;
    for (unsigned k = 0u; k < 16u; ++k)
      sn = sn + L.diag[16u * (tid - 64u) + k];
    L.bnorm[tid - 64u] = (float)log2(sn);
  }
  __syncthreads();
  if (plan == PLAN_SPLIT && !L.chol_ok) {
    if (tid == 0u) {
      flags[pi] = 0u;
      VisitRec v;
      v.rot_s = 0u;
      v.rot_b = 0u;
      v.maxcos = 1.0f;
      v.l2ni = L.bnorm[0];
      v.l2nj = L.bnorm[1];
      v.sweep = ctl->sweep;
      v.skips = 0u;
      v.flags = REC_SPLIT | REC_SPLIT_FAIL;
      rec[pi] = v;
      atomicAdd(&ctl->split, 1u);
    }
    return false;
  }

  unsigned blk_s, blk_b;
  inner_sweeps<SORT, LANES>(tid, L, sg, s0steps, nswp, true, blk_s, blk_b);

  // the block update is left out exactly when W is the identity (no rotation,
  // no swap)
  const bool upd = blk_s || L.swp;
  // convergence counter, share/device_code_nosort.hpp:94-103
  if (tid == 0u) {
    unsigned long long *const cvg = &ctl->cvg;
    if (blk_s) {
      if (blk_b)
        atomicAdd(cvg, (((unsigned long long)blk_b) << 32) | blk_s);
      else
        atomicAdd(reinterpret_cast<unsigned *>(cvg), blk_s);
    }
    if (flags) flags[pi] = upd ? 1u : 0u;
    VisitRec v;
    v.rot_s = blk_s;
    v.rot_b = blk_b;
    v.maxcos = __uint_as_float(L.cmax);
    v.l2ni = L.bnorm[0];
    v.l2nj = L.bnorm[1];
    v.sweep = ctl->sweep;
    v.skips = 0u;
    v.flags = (plan == PLAN_SPLIT) ? REC_SPLIT : 0u;
    rec[pi] = v;
    if (plan == PLAN_SPLIT)
      atomicAdd(&ctl->split, 1u);
  }
  return upd;
}

// The visit of pair pi from its Gram partials; W to Wout (W(k, j) at 32 j + k)
template <bool SORT, unsigned LANES>
__device__ __forceinline__ void pair_visit(unsigned tid, unsigned pi, PairLds &L,
                                           const uint16_t *__restrict__ pairs,
                                           const double *__restrict__ part, unsigned nchunk,
                                           double *__restrict__ Wout, unsigned *__restrict__ flags,
                                           RunCtl *__restrict__ ctl, VisitRec *__restrict__ rec,
                                           uint8_t plan, const uint8_t *__restrict__ strat0,
                                           unsigned s0steps, unsigned nswp, int definite,
                                           unsigned nplus)
{
  constexpr unsigned NT = 32u * LANES;
  visit_load<NT>(tid, pi, L, part, nchunk, strat0);
  const PairSigns sg = pair_signs16(definite, nplus, pairs[2u * pi], pairs[2u * pi + 1u]);
  // (W of a pair left alone is read by nothing)
  if (!visit_core<SORT, LANES>(tid, pi, L, sg, flags, ctl, rec, plan, s0steps, nswp))
    return;
  double *const wo = Wout + (size_t)pi * 1024u;
  for (unsigned e = tid; e < 1024u; e += NT)
    wo[e] = RA(L.W, e & 31u, e >> 5);
}

// a skipped visit: no update, the record keeps the last executed visit
__device__ __forceinline__ void skip_visit(unsigned tid, unsigned pi, unsigned *flags, RunCtl *ctl,
                                           VisitRec *rec)
{
  if (tid == 0u) {
    flags[pi] = 0u;
    rec[pi].skips += 1u;
    atomicAdd(&ctl->skipped, 1u);
  }
}

}  // namespace hj

#endif

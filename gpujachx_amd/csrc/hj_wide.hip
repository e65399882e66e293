// hj_wide.hip -- the wide-block form: blocks of 32 columns, so a level-1
// visit treats a 64-column block pair (64x64 Gram, Cholesky and level-0 on
// R, 64x64 W).  A sweep moves half the HBM bytes of the reference's
// 16-column blocks (share/HypJacL.hpp:112-116) for the same FP64 flops.
// Step by step: Gram partials (k_gram_w), visits (k_pair_w), block update
// (k_update_w), each in the arithmetic of the 16-column kernels written for
// 64 columns:
//   - Gram: the 10 16x16 tiles of the pair's lower triangle on FP64 MFMA
//     16x16x4, per tile the chain over the rows of a wave's sub-chunk in
//     16-row slabs, the waves added in order, the chunks in order by the
//     visit;
//   - Cholesky (share/device_code_common_Cholesky.hpp:58-158, USE_RSQRT) at
//     64 pivots, 32 at a time;
//   - level-0: 32 pivot pairs a step, 8 lanes a pair, dot products by the xor
//     butterfly 32,16,8 in the lane, 4,2,1 across lanes; the convergence test
//     at tolerance sqrt(64) 2^-53;
//   - update: out(r, j) = MFMA chain over k = 0..63.
// With the learned pair-skip a step's plan marks skipped pairs: no Gram, no
// visit (its record keeps the last executed visit), no update.
#include "../../include/hypjac.h"
#include "hj_kernels.hpp"
#include "hj_device.hpp"
#include "hj_fused.hpp"
#include "hj_util.hpp"
#include "hj_visit.hpp"

namespace hj {

namespace {

constexpr unsigned WTILES = 10u;             // tiles of a 64-column pair's lower triangle
constexpr unsigned WPART = WTILES * 256u;    // doubles per Gram partial
constexpr unsigned LDRW = 72u;               // column of R and W in LDS: of eight lanes a pivot pair, two neighbouring pairs in different banks
constexpr double WTOL = 0x1p-50;             // sqrt(64) * 2^-53
#define RW(A, r, c) (A)[(c) * LDRW + (r)]

// tile tt -> (ti, tj), tt = ti (ti + 1) / 2 + tj
__device__ __forceinline__ unsigned tile_i(unsigned tt)
{
  return (tt >= 6u) ? 3u : ((tt >= 3u) ? 2u : ((tt >= 1u) ? 1u : 0u));
}

// Gram partials of the pairs of one step: workgroup (pair, row chunk), its
// waves taking equal row sub-chunks, wave 0 adding the others' tiles in
// wave order; partial of (pair, chunk) at part[(pi * nchunk + c) * WPART],
// tile tt at + 256 tt, element (4r + l/16, l%16) at + 4l + r.  A slab (16
// rows x 64 columns) is read 128 bytes of a column per lane group (lane l:
// row l%16 of column 4u + l/16) with the next slab's loads in flight, and
// turned into the MFMA operand layout (lane l, register r of group t: row
// 4r + l/16 of column 16t + l%16) through the wave's LDS buffer.
constexpr unsigned LDTW = 17u;  // padded column of a wave's slab buffer

struct GramLdsW {
  union {
    d4 red[WTILES][64];  // one wave's tiles at a time
    double T[GRAM_WAVES][64u * LDTW];
  };
};

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_gram_w(const double *__restrict__ G, unsigned ldG,
                                                const uint16_t *__restrict__ pairs,
                                                unsigned nchunk, unsigned CH,
                                                double *__restrict__ part,
                                                const uint8_t *__restrict__ plan)
{
  __shared__ GramLdsW S;
  const unsigned l = threadIdx.x & 63u, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const unsigned pi = blockIdx.x / nchunk, c = blockIdx.x - pi * nchunk;
  if (plan && plan[pi] == PLAN_SKIP)
    return;  // a skipped visit needs no Gram
  const unsigned a = pairs[2u * pi], b = pairs[2u * pi + 1u];
  const unsigned SUB = CH / nw;
  const size_t r0 = (size_t)c * CH + (size_t)w * SUB + (l & 15u);
  // column 4u + l/16 of the pair: block a for u < 8, block b after
  const double *const ga = G + (size_t)(32u * a + (l >> 4)) * ldG + r0;
  const double *const gb = G + (size_t)(32u * b + (l >> 4)) * ldG + r0;
  lds_f64 *const T = (lds_f64 *)S.T[w];
  d4 acc[WTILES];
#pragma unroll
  for (unsigned tt = 0u; tt < WTILES; ++tt)
    acc[tt] = d4{0.0, 0.0, 0.0, 0.0};
  double xn[16];
#pragma unroll
  for (unsigned u = 0u; u < 8u; ++u) {
    xn[u] = ga[(size_t)(4u * u) * ldG];
    xn[8u + u] = gb[(size_t)(4u * u) * ldG];
  }
  for (unsigned s = 0u; s < SUB; s += 16u) {
#pragma unroll
    for (unsigned u = 0u; u < 16u; ++u)
      T[(4u * u + (l >> 4)) * LDTW + (l & 15u)] = xn[u];
    if (s + 16u < SUB) {
#pragma unroll
      for (unsigned u = 0u; u < 8u; ++u) {
        xn[u] = ga[(size_t)(4u * u) * ldG + s + 16u];
        xn[8u + u] = gb[(size_t)(4u * u) * ldG + s + 16u];
      }
    }
    wave_lds_sync();
    d4 X[4];
#pragma unroll
    for (unsigned t = 0u; t < 4u; ++t)
#pragma unroll
      for (unsigned r = 0u; r < 4u; ++r)
        X[t][r] = T[(16u * t + (l & 15u)) * LDTW + 4u * r + (l >> 4)];
    wave_lds_sync();
#pragma unroll
    for (unsigned r = 0u; r < 4u; ++r) {
      unsigned tt = 0u;
#pragma unroll
      for (unsigned ti = 0u; ti < 4u; ++ti)
#pragma unroll
        for (unsigned tj = 0u; tj <= ti; ++tj, ++tt)
          acc[tt] = mfma(X[ti][r], X[tj][r], acc[tt]);
    }
  }
  // wave 0 adds the other waves' tiles in wave order, one wave's at a time
  // through the (former slab) buffer
  for (unsigned u = 1u; u < nw; ++u) {
    __syncthreads();
    if (w == u) {
#pragma unroll
      for (unsigned tt = 0u; tt < WTILES; ++tt)
        S.red[tt][l] = acc[tt];
    }
    __syncthreads();
    if (w == 0u) {
#pragma unroll
      for (unsigned tt = 0u; tt < WTILES; ++tt)
        acc[tt] = acc[tt] + S.red[tt][l];
    }
  }
  if (w == 0u) {
    double *const o = part + (size_t)blockIdx.x * WPART;
#pragma unroll
    for (unsigned tt = 0u; tt < WTILES; ++tt)
      *reinterpret_cast<d4 *>(o + tt * 256u + 4u * l) = acc[tt];
  }
}

// The same partials where the sub-chunks are too few for a wave each to fill the
// chip: four waves a sub-chunk, each with two or three of the ten tiles' chains
// (the two diagonal 32x32 quarters and the rows of the other one), reading
// 32-row panels of the pair's columns into LDS, the next one's loads in flight.
// Workgroup (pair, chunk), NW sub-chunks.  A wave issues 64 cycles of FP64 MFMA
// a tile and four rows; 4608 x 2048, whose 576-row chunks hold one sub-chunk
// each (256 in all), 187 us a step with all ten tiles on a wave, 159 now.
constexpr unsigned GTW_LD = 34u;  // padded panel column: operands in 32 different banks

template <unsigned W>
__device__ __forceinline__ void gram_w_tiles_panel(const lds_f64 *p, d4 *acc)
{
  // tile rows / columns of wave W's chains
  constexpr unsigned TI[4][3] = {{0u, 1u, 1u}, {2u, 3u, 3u}, {2u, 2u, 0u}, {3u, 3u, 0u}};
  constexpr unsigned TJ[4][3] = {{0u, 0u, 1u}, {2u, 2u, 3u}, {0u, 1u, 0u}, {0u, 1u, 0u}};
  constexpr unsigned NTILE = W < 2u ? 3u : 2u;
#pragma unroll
  for (unsigned r = 0u; r < 32u; r += 4u)
#pragma unroll
    for (unsigned t = 0u; t < NTILE; ++t)
      acc[t] = mfma(p[16u * GTW_LD * TI[W][t] + r], p[16u * GTW_LD * TJ[W][t] + r], acc[t]);
}

template <unsigned NW>
__global__ __launch_bounds__(256u * NW) void k_gram_w_tiles(const double *__restrict__ G, unsigned ldG,
                                                            const uint16_t *__restrict__ pairs,
                                                            unsigned nchunk, unsigned CH,
                                                            double *__restrict__ part,
                                                            const uint8_t *__restrict__ plan)
{
  __shared__ union {
    double P[NW][2][64u * GTW_LD];
    d4 red[NW][WTILES][64];
  } S;
  const unsigned tid = threadIdx.x, l = tid & 63u, sub = tid >> 8, w = (tid >> 6) & 3u;
  const unsigned pi = blockIdx.x / nchunk, c = blockIdx.x - pi * nchunk;
  if (plan && plan[pi] == PLAN_SKIP)
    return;  // a skipped visit needs no Gram
  const unsigned a = pairs[2u * pi], b = pairs[2u * pi + 1u];
  const unsigned SUB = CH / NW;
  // wave w reads columns 2w + l/32 + 8k of the pair, row l % 32 of a panel
  const size_t r0 = (size_t)c * CH + (size_t)sub * SUB + (l & 31u);
  const unsigned cw = 2u * w + (l >> 5);
  const double *const ga = G + (size_t)(32u * a + cw) * ldG + r0;
  const double *const gb = G + (size_t)(32u * b + cw) * ldG + r0;
  const size_t cs = (size_t)8u * ldG;
  double x[8];
#pragma unroll
  for (unsigned k = 0u; k < 4u; ++k) {
    x[k] = ga[k * cs];
    x[4u + k] = gb[k * cs];
  }
  d4 acc[3];
#pragma unroll
  for (unsigned t = 0u; t < 3u; ++t)
    acc[t] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
  for (unsigned g = 0u, h = 0u; g < SUB; g += 32u, h ^= 1u) {
    lds_f64 *const p = (lds_f64 *)S.P[sub][h];
#pragma unroll
    for (unsigned k = 0u; k < 8u; ++k)
      p[(cw + 8u * k) * GTW_LD + (l & 31u)] = x[k];
    if (g + 32u < SUB) {
#pragma unroll
      for (unsigned k = 0u; k < 4u; ++k) {
        x[k] = ga[k * cs + g + 32u];
        x[4u + k] = gb[k * cs + g + 32u];
      }
    }
    // (two buffers: a wave writes this one again only after the next
    // panel's barrier, when every wave has left it)
    __syncthreads();
    const lds_f64 *const o = p + (l & 15u) * GTW_LD + (l >> 4);
    if (w == 0u) gram_w_tiles_panel<0u>(o, acc);
    else if (w == 1u) gram_w_tiles_panel<1u>(o, acc);
    else if (w == 2u) gram_w_tiles_panel<2u>(o, acc);
    else gram_w_tiles_panel<3u>(o, acc);
  }
  // tile numbers of the wave's chains: i (i + 1) / 2 + j
  const unsigned t0 = (w == 0u) ? 0u : (w == 1u) ? 5u : (w == 2u) ? 3u : 6u;
  const unsigned t1 = (w == 0u) ? 1u : (w == 1u) ? 8u : (w == 2u) ? 4u : 7u;
  const unsigned t2 = (w == 0u) ? 2u : 9u;
  double *const o = part + (size_t)blockIdx.x * WPART + 4u * l;
  if (NW == 1u) {
    *reinterpret_cast<d4 *>(o + 256u * t0) = acc[0];
    *reinterpret_cast<d4 *>(o + 256u * t1) = acc[1];
    if (w < 2u) *reinterpret_cast<d4 *>(o + 256u * t2) = acc[2];
    return;
  }
  // the sub-chunks' tiles added in order
  __syncthreads();
  S.red[sub][t0][l] = acc[0];
  S.red[sub][t1][l] = acc[1];
  if (w < 2u) S.red[sub][t2][l] = acc[2];
  __syncthreads();
  for (unsigned t = tid >> 6; t < WTILES; t += 4u * NW) {
    d4 v = S.red[0][t][l];
#pragma unroll
    for (unsigned u = 1u; u < NW; ++u)
      v = v + S.red[u][t][l];
    *reinterpret_cast<d4 *>(o + 256u * t) = v;
  }
}

constexpr unsigned VT = 512u;  // threads of a visit: half on R, half on W, 8 lanes a pivot pair

// LDS of a 64-column pair visit
constexpr unsigned S0W_BYTES = 64u * 32u * 2u;  // level-0 table of order 64 (<= 64 steps)

struct PairLdsW {
  static constexpr unsigned N = 64u, LD = LDRW;  // order and leading dimension of R and W
  static constexpr double TOL = WTOL;            // of the convergence test
  double R[64u * LDRW];
  double W[64u * LDRW];
  double A22[32u * L0LD];  // the Cholesky's trailing block
  double col[64];
  double diag[64];         // the Gram's diagonal
  double rot[2][32][4];    // per step parity and pivot pair: c, t, |Apq|, |p| |q|
  unsigned act[2][32];     // ... what happens to its columns (ACT_*)
  unsigned cs[2], cb[2];   // rotations of an inner sweep, by its parity
  unsigned cmax;           // bits of the largest cosine of the first inner sweep
  float bnorm[2];
  int swp;
  __attribute__((aligned(16))) uint8_t S0[S0W_BYTES];
};

// The first 32 columns of the Cholesky factor of the 64x64 Gram in A (lower
// triangle, A[c * LDRW + r] = A(r, c)) by one wave, lane x on row x:
// share/device_code_common_Cholesky.hpp:58-158 (USE_RSQRT) for k < 32, j < 32.
// On return A holds the first 32 rows of R = L^T (R(k, x) at A[x * LDRW + k])
// and zeros below them; the columns from 32 on are untouched.
//
// panel_any takes any input, column by column in LDS.
__device__ __forceinline__ void panel_any(lds_f64 *A, lds_f64 *col, unsigned x)
{
#pragma unroll 1
  for (unsigned k = 0u; k < 32u; ++k) {
    const double akk = A[k * LDRW + k], v = A[k * LDRW + x];
    const double rk = dev_rsqrt_any(akk), dk = sqrt(akk);
    const double w = (x == k) ? dk : v * rk;
    wave_lds_sync();
    if (x >= k) A[k * LDRW + x] = w;
    col[x] = w;
    wave_lds_sync();
#pragma unroll 1
    for (unsigned j = k + 1u; j < 32u; ++j)
      if (x >= j) A[j * LDRW + x] = __fma_rn(-w, col[j], A[j * LDRW + x]);
    wave_lds_sync();
  }
#pragma unroll 1
  for (unsigned c = 0u; c < 32u; ++c) {
    const double v = A[c * LDRW + x];
    wave_lds_sync();
    if (x > c) {
      A[x * LDRW + c] = v;
      A[c * LDRW + x] = 0.0;
    }
    wave_lds_sync();
  }
}

// chol32_wave's scheme on 64 rows: the panel in registers, the next pivot's
// rsqrt (the chain of the pivots) beside the column's updates, the diagonal's
// square roots in one instruction sequence at the end.
__device__ __forceinline__ void panel_wave(double *A_, double *col_, unsigned x)
{
  lds_f64 *const A = (lds_f64 *)A_;
  lds_f64 *const col = (lds_f64 *)col_;
  double b[32];
#pragma unroll
  for (unsigned c = 0u; c < 32u; ++c)
    b[c] = (c <= x) ? A[c * LDRW + x] : 0.0;
  double akk = readlane_d(b[0], 0);
  bool sure;
  double rk = rsqrt_bracket(akk, sure);
  unsigned long long bad = __ballot(!(sure && rsqrt_plain_range(akk)));
#pragma unroll
  for (unsigned k = 0u; k < 32u; ++k) {
    const unsigned k1 = k + 1u;
    const double u = pin(b[k] * rk);
    col[x] = u;
    b[k] = pin((x > k) ? u : b[k]);
    if (k1 == 32u)
      break;
    const double lk = readlane_d(u, k1);
    const double d1 = readlane_d(b[k1], k1);
    akk = __fma_rn(-lk, lk, d1);
    wave_lds_sync();
    double cv[32];
#pragma unroll
    for (unsigned j = k1; j < 32u; ++j)
      cv[j] = col[j];
    // the column's reads are issued here, all of them, and used after the
    // pivot's chain has started
    __builtin_amdgcn_sched_barrier(0);
    rk = rsqrt_bracket(akk, sure);
    bad |= __ballot(!(sure && rsqrt_plain_range(akk)));
#pragma unroll
    for (unsigned j = k1; j < 32u; ++j)
      b[j] = __fma_rn(-u, cv[j], b[j]);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" : "+s"(bad));
#pragma unroll
    for (unsigned j = k1; j < 32u; ++j)
      asm volatile("" : "+v"(b[j]));
    wave_lds_sync();
  }
  if (bad) {
    panel_any(A, col, x);
    return;
  }
  // (above the diagonal: entries of other columns' lower triangle stay)
#pragma unroll
  for (unsigned c = 0u; c < 32u; ++c)
    if (c <= x) A[x * LDRW + c] = b[c];
#pragma unroll
  for (unsigned c = 0u; c < 32u; ++c)
    if (c < x) A[c * LDRW + x] = 0.0;
  wave_lds_sync();
  const double d = sqrt(A[x * LDRW + x]);
  wave_lds_sync();
  if (x < 32u) A[x * LDRW + x] = d;
}

// In-place 64x64 Cholesky by the workgroup, R = L^T with zeros below: the
// first 32 columns (one wave), the trailing block's update by them (a chain
// over k = 0..31 in order on FP64 MFMA, one wave a tile), its Cholesky (one
// wave, chol32_wave), while the others set W to the identity.  Every entry
// takes the same operations in the same order as column by column.  Ends
// synchronized.
__device__ __forceinline__ void chol64_block(PairLdsW &L, unsigned tid)
{
  lds_f64 *const A = (lds_f64 *)L.R;
  lds_f64 *const B = (lds_f64 *)L.A22;
  const unsigned l = tid & 63u, w = tid >> 6;
  if (w == 0u) {
    panel_wave(L.R, L.col, l);
  }
  else if (tid < 66u) {
    // squared Frobenius norms of the two blocks, for the visit record
    double sn = 0.0;
    for (unsigned k = 0u; k < 32u; ++k)
      sn = sn + L.diag[32u * (tid - 64u) + k];
    L.bnorm[tid - 64u] = (float)log2(sn);
  }
  __syncthreads();
  if (w < 3u) {
    // tile (ti, tj) of the trailing block: 00, 10, 11
    const unsigned i0 = w ? 16u : 0u, j0 = (w == 2u) ? 16u : 0u;
    const lds_f64 *const X = A + (32u + i0 + (l & 15u)) * LDRW + (l >> 4);
    const lds_f64 *const Y = A + (32u + j0 + (l & 15u)) * LDRW + (l >> 4);
    const lds_f64 *const C = A + (32u + j0 + (l & 15u)) * LDRW + 32u + i0 + (l >> 4);
    d4 acc;
#pragma unroll
    for (unsigned r = 0u; r < 4u; ++r)
      acc[r] = C[4u * r];
#pragma unroll
    for (unsigned u = 0u; u < 8u; ++u)
      acc = mfma(-X[4u * u], Y[4u * u], acc);
#pragma unroll
    for (unsigned r = 0u; r < 4u; ++r)
      B[(j0 + (l & 15u)) * L0LD + i0 + 4u * r + (l >> 4)] = acc[r];
  }
  __syncthreads();
  if (w == 0u) {
    (void)chol32_wave<L0LD>(L.A22, L.col, l, false);
  }
  else {
    for (unsigned e = tid - 64u; e < 4096u; e += VT - 64u)
      RW(L.W, e & 63u, e >> 6) = ((e & 63u) == (e >> 6)) ? 1.0 : 0.0;
  }
  __syncthreads();
  for (unsigned e = tid; e < 1024u; e += VT)
    RW(L.R, 32u + (e & 31u), 32u + (e >> 5)) = L.A22[(e >> 5) * L0LD + (e & 31u)];
  __syncthreads();
}

// J of a pair's 64 columns (see PairSigns)
__device__ __forceinline__ PairSigns pair_signs32(int definite, unsigned nplus, unsigned iBlk,
                                                  unsigned jBlk)
{
  PairSigns s = {definite, 0u, false};
  if (!definite) {
    const unsigned ifc0 = iBlk * 32u, ifc1 = jBlk * 32u;
    if (nplus <= ifc0) { s.npos = 0u; s.def = -1; }
    else if (nplus <= ifc0 + 32u) { s.npos = nplus - ifc0; s.def = 0; }
    else if (nplus <= ifc1) { s.npos = 32u; s.def = 0; }
    else if (nplus <= ifc1 + 32u) { s.npos = 32u + (nplus - ifc1); s.def = 0; }
    else { s.npos = 64u; s.def = +1; }
    s.hyp = (s.def == 0);
  }
  return s;
}

// Block update M[:, pair] <- M[:, pair] W of one pair's rows [rbeg, rend) by the
// NT threads of a workgroup: W in LDS (Wl, row-major, padded), each
// wave 16-row slabs of the chunk with the next slab's loads in flight.  Per
// slab the MFMA chains run over k = 0..63 in order: A = W^T (lane l:
// W(4u + l/16, 16h + l%16)), B = the slab's transpose (lane l:
// M(row + l%16, column 4u + l/16)); lane l, register q of tile h holds
// output column 16h + 4q + l/16 of row row + l%16.
constexpr unsigned LDWW = 65u;

template <unsigned NT>
__device__ __forceinline__ void update_w_rows(double *Wl_, double *__restrict__ M, unsigned ldM,
                                              unsigned rbeg, unsigned rend, unsigned a, unsigned b,
                                              const double *__restrict__ Wp, unsigned tid)
{
  lds_f64 *const Wl = (lds_f64 *)Wl_;
  const unsigned l = tid & 63u, w = tid >> 6;
  constexpr unsigned STEP = NT / 4u;  // rows of all waves' slabs
  for (unsigned e = tid; e < 4096u; e += NT)
    Wl[(e & 63u) * LDWW + (e >> 6)] = Wp[e];  // Wl[k * LDWW + j] = W(k, j), at 64 j + k of Wp
  __syncthreads();
  // column 4u + l/16 of the pair: block a for u < 8, block b after
  double *const ca = M + (size_t)(32u * a + (l >> 4)) * ldM + (l & 15u);
  double *const cb = M + (size_t)(32u * b + (l >> 4)) * ldM + (l & 15u);
  const lds_f64 *const wl = Wl + (l >> 4) * LDWW + (l & 15u);
  unsigned row = rbeg + 16u * w;
  double xn[16];
  if (row < rend) {
#pragma unroll
    for (unsigned u = 0u; u < 8u; ++u) {
      xn[u] = ca[(size_t)(4u * u) * ldM + row];
      xn[8u + u] = cb[(size_t)(4u * u) * ldM + row];
    }
  }
  for (; row < rend; row += STEP) {
    double x[16];
#pragma unroll
    for (unsigned u = 0u; u < 16u; ++u)
      x[u] = xn[u];
    if (row + STEP < rend) {
#pragma unroll
      for (unsigned u = 0u; u < 8u; ++u) {
        xn[u] = ca[(size_t)(4u * u) * ldM + row + STEP];
        xn[8u + u] = cb[(size_t)(4u * u) * ldM + row + STEP];
      }
    }
    d4 acc[4];
#pragma unroll
    for (unsigned h = 0u; h < 4u; ++h)
      acc[h] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (unsigned u = 0u; u < 16u; ++u) {
      const lds_f64 *const wr = wl + 4u * u * LDWW;
#pragma unroll
      for (unsigned h = 0u; h < 4u; ++h)
        acc[h] = mfma(wr[16u * h], x[u], acc[h]);
    }
#pragma unroll
    for (unsigned h = 0u; h < 4u; ++h)
#pragma unroll
      for (unsigned q = 0u; q < 4u; ++q)
        ((h < 2u) ? ca : cb)[(size_t)(16u * (h & 1u) + 4u * q) * ldM + row] = acc[h][q];
  }
}

// The pairs of one step, a workgroup per (pair, chunk of rows).  Pairs whose W is
// the identity (flag 0) are left alone.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_update_w(
    double *__restrict__ M, unsigned ldM, unsigned nrow, const uint16_t *__restrict__ pairs,
    const double *__restrict__ Wbuf, const unsigned *__restrict__ flags, unsigned nchunk, unsigned rows)
{
  __shared__ double Wl[64u * LDWW];
  const unsigned pi = blockIdx.x / nchunk, c = blockIdx.x - pi * nchunk;
  if (!flags[pi])
    return;
  const unsigned rbeg = c * rows;
  update_w_rows<256u>(Wl, M, ldM, rbeg, min(rbeg + rows, nrow), pairs[2u * pi], pairs[2u * pi + 1u],
                      Wbuf + (size_t)pi * 4096u, threadIdx.x);
}

// One 64-column block pair per workgroup of 512 threads: chunk partials ->
// R (lower), Cholesky, level-0 sweeps on R accumulating W, counters, W and
// the update flag out.  The visit of 32 columns (hj_visit.hpp) at 64: four
// waves keep R, eight lanes a pivot pair, four apply the same rotations to W
// one step behind.  A level-0 step is bound by its instructions (a wave of
// either kind on every SIMD) and by LDS, which moves R and W once in and once
// out: 1024 cycles at 128 bytes each, so the columns' leading dimension keeps
// the groups of a wave off each other's banks (LDRW = 65: two- to fourfold
// conflicts).  Measured, 4608 x 2048: partials 4 us, Cholesky 14 us, a level-0
// sweep 73 us (89 us at LDRW = 65); 92 us a launch, 126 us with eight waves of
// 16 lanes a pair that each kept R and W, and a Cholesky of 64 pivots with two
// barriers each.
template <bool SORT>
__global__ __launch_bounds__(512) void k_pair_w(const uint16_t *__restrict__ pairs,
                                                const double *__restrict__ part, unsigned nchunk,
                                                double *__restrict__ Wout,
                                                unsigned *__restrict__ flags,
                                                RunCtl *__restrict__ ctl,
                                                const uint8_t *__restrict__ strat0,
                                                unsigned s0steps, unsigned nswp, int definite,
                                                unsigned nplus, const uint8_t *__restrict__ plan,
                                                VisitRec *__restrict__ rec, unsigned np, VItems V)
{
  __shared__ PairLdsW L;
  const unsigned tid = threadIdx.x, pi = blockIdx.x;
  if (pi >= np) {
    // V by the W of the step before, on the CUs that no visit takes
    static_assert(64u * LDWW <= 64u * LDRW, "W fits R");
    const unsigned v = (pi - np) / V.nch, c = pi - np - v * V.nch;
    if (!V.flags[v])
      return;
    const unsigned r0 = c * V.ch;
    update_w_rows<VT>(L.R, V.V, V.ld, r0, min(r0 + V.ch, V.nrow), V.pairs[2u * v], V.pairs[2u * v + 1u],
                      V.W + (size_t)v * 4096u, tid);
    return;
  }
  unsigned long long *const cvg = &ctl->cvg;
  if (plan && plan[pi] == PLAN_SKIP) {
    // skipped visit: no update, the record keeps the last executed visit
    if (tid == 0u) {
      flags[pi] = 0u;
      rec[pi].skips += 1u;
      atomicAdd(&ctl->skipped, 1u);
    }
    return;
  }
  const PairSigns sg = pair_signs32(definite, nplus, pairs[2u * pi], pairs[2u * pi + 1u]);
  {
    const double *const pp = part + (size_t)pi * nchunk * WPART;
    // a thread's entries with all their chunk loads in flight together; the
    // chunks summed in chunk order
    constexpr unsigned NE = WPART / VT;
    double v[NE][MAX_GRAM_CHUNKS];
#pragma unroll
    for (unsigned q = 0u; q < NE; ++q)
#pragma unroll
      for (unsigned c = 0u; c < MAX_GRAM_CHUNKS; ++c)
        if (c < nchunk) v[q][c] = pp[(size_t)c * WPART + tid + VT * q];
    for (unsigned e = tid; e < 2u * 32u * s0steps; e += VT)
      L.S0[e] = strat0[e];
    if (tid == 0u) {
      L.swp = 0;
      L.cmax = 0u;
      L.cs[0] = L.cb[0] = 0u;
    }
#pragma unroll
    for (unsigned q = 0u; q < NE; ++q) {
      const unsigned e = tid + VT * q;
      double s = v[q][0];
#pragma unroll
      for (unsigned c = 1u; c < MAX_GRAM_CHUNKS; ++c)
        if (c < nchunk) s = s + v[q][c];
      const unsigned tt = e >> 8, ti = tile_i(tt), tj = tt - ti * (ti + 1u) / 2u;
      const unsigned l = (e >> 2) & 63u, r = e & 3u;
      const unsigned row = 16u * ti + 4u * r + (l >> 4), col = 16u * tj + (l & 15u);
      RW(L.R, row, col) = s;
      if (row == col) L.diag[row] = s;
    }
  }
  __syncthreads();
  chol64_block(L, tid);

  unsigned blk_s, blk_b;
  inner_sweeps<SORT, VT / 64u>(tid, L, sg, s0steps, nswp, rec != nullptr, blk_s, blk_b);
  if (tid == 0u) {
    // convergence counter, share/device_code_nosort.hpp:94-103
    if (blk_s) {
      if (blk_b)
        atomicAdd(cvg, (((unsigned long long)blk_b) << 32) | blk_s);
      else
        atomicAdd(reinterpret_cast<unsigned *>(cvg), blk_s);
    }
    flags[pi] = (blk_s || L.swp) ? 1u : 0u;
    if (rec) {
      // the record in the units of a 32-column pair's inner sweep (496 pivot
      // pairs): this pair's counts scaled from its 2016
      VisitRec v;
      v.rot_s = (min(blk_s, 2016u) * 496u + 1008u) / 2016u;
      v.rot_b = (min(blk_b, 2016u) * 496u + 1008u) / 2016u;
      v.maxcos = __uint_as_float(L.cmax);
      v.l2ni = L.bnorm[0];
      v.l2nj = L.bnorm[1];
      v.sweep = ctl->sweep;
      v.skips = 0u;
      v.flags = 0u;
      rec[pi] = v;
    }
  }
  double *const wo = Wout + (size_t)pi * 4096u;
  for (unsigned e = tid; e < 4096u; e += VT)
    wo[e] = RW(L.W, e & 63u, e >> 6);
}

}  // namespace

unsigned wide_part_doubles() { return WPART; }

namespace {

// Sub-chunks of a step up to which k_gram_w_tiles takes its Gram: one a SIMD.
// Beyond, a wave each fills the chip.  Measured, us a step with k_gram_w /
// k_gram_w_tiles: 1088 x 512 (16 sub-chunks) 200 / 145, 4608 x 2048 (256) 187
// / 159, 6144 x 2048 (1024) 174 / 164, 4096 x 2048 (2048) 148 / 153, 8192 x
// 4096 (4096) 273 / 283.
constexpr unsigned GRAM_W_TILES_MAX = 1024u;

// Rows a workgroup of k_update_w: two workgroups a CU (each brings W's 32 KB
// with it), at most 512 rows.  Measured, us a step at one / two / four a CU:
// 4608 x 2048 170 / 158 / 158, 4096 x 2048 153 / 146 / 148, 6144 x 4096 234 /
// 234 / 245.
unsigned update_w_rows_per_wg(unsigned nrow, unsigned np)
{
  unsigned rows = 512u;
  while (rows > 64u && np * ((nrow + rows - 1u) / rows) < 512u)
    rows /= 2u;
  return rows;
}

}  // namespace

void launch_gram_w(hipStream_t s, const double *G, unsigned ldG, const uint16_t *pairs,
                   unsigned np, unsigned nchunk, unsigned CH, double *part, const uint8_t *plan)
{
  const unsigned nw = gram_waves(CH);
  if (np * nchunk * nw <= GRAM_W_TILES_MAX) {
    const auto k = (nw == 1u) ? k_gram_w_tiles<1u> : (nw == 2u) ? k_gram_w_tiles<2u> : k_gram_w_tiles<4u>;
    hipLaunchKernelGGL(k, dim3(np * nchunk), dim3(256u * nw), 0, s, G, ldG, pairs, nchunk, CH, part,
                       plan);
    return;
  }
  hipLaunchKernelGGL(k_gram_w, dim3(np * nchunk), dim3(64u * nw), 0, s, G, ldG, pairs, nchunk, CH,
                     part, plan);
}

void launch_pair_w(hipStream_t s, bool sort, const uint16_t *pairs, unsigned np,
                   const double *part, unsigned nchunk, double *W, unsigned *flags,
                   RunCtl *ctl, const uint8_t *strat0, unsigned s0steps,
                   unsigned nswp, int definite, unsigned nplus, const uint8_t *plan,
                   VisitRec *rec, const VItems &v)
{
  const auto k = sort ? k_pair_w<true> : k_pair_w<false>;
  hipLaunchKernelGGL(k, dim3(np + v.n), dim3(VT), 0, s, pairs, part, nchunk, W, flags, ctl, strat0,
                     s0steps, nswp, definite, nplus, plan, rec, np, v);
}

void launch_update_w(hipStream_t s, double *M, unsigned ldM, unsigned nrow,
                     const uint16_t *pairs, unsigned np, const double *W,
                     const unsigned *flags)
{
  const unsigned rows = update_w_rows_per_wg(nrow, np), nch = (nrow + rows - 1u) / rows;
  hipLaunchKernelGGL(k_update_w, dim3(np * nch), dim3(256), 0, s, M, ldM, nrow, pairs, W, flags,
                     nch, rows);
}

}  // namespace hj

// hj_step.hip -- one level-1 step in one launch, for matrices whose block pairs
// fit one workgroup's LDS (up to STEP_MAX_ROWS rows).
//
// Workgroup pi loads its pair's 32 columns into LDS once, forms their Gram (the
// sub-chunks and row order of k_gram, so the same bits), runs the visit
// (hj_visit.hpp), and writes the columns times W back, together with V's.
// Small steps are all latency: against the launches k_pair and k_upgram (or
// k_gram and k_update) and k_update for V, each of which starts with a chain of
// cold reads of indices, flags, W or partials, this saves two launches and
// the trips of the partials and W through memory, and reads the columns once.
// What is left is the visit (25 us of the step), the two reads and the FP64
// MFMAs (64 cycles each on a SIMD: 384 for the Gram and 1024 for the updates
// of G and V at 512 rows, over four SIMDs).  Beyond STEP_MAX_ROWS a pair no
// longer fits, and its rows through one CU cost more than the launches.
#include "hj_fused.hpp"
#include "hj_visit.hpp"

namespace hj {
namespace {

constexpr unsigned STEP_WAVES = 8u;
constexpr unsigned STEP_LANES = 2u * STEP_WAVES;  // lanes per pivot pair of the visit
constexpr unsigned STEP_NT = 64u * STEP_WAVES;
constexpr unsigned STEP_PER_WAVE = STEP_MAX_ROWS / 16u / STEP_WAVES;  // 16-row slabs

struct StepLds {
  PairLds pair;
  // the pair's columns, column c at c (nrow + 2): the Gram's operands (16
  // columns x 2 rows a half-wave) fall into 32 different banks
  double cols[32u * (STEP_MAX_ROWS + 2u)];
};

// The Gram of the columns in LDS: nsub sub-chunks (a power of two up to
// STEP_WAVES) of SUB rows, added in order, to L.pair.R.  Unit u = (tile t = u
// / nsub, sub-chunk u % nsub) is one wave's MFMA chain: a wave takes units w,
// w + 8, w + 16.
__device__ __forceinline__ void step_gram(StepLds &L, unsigned ld, unsigned nsub, unsigned SUB,
                                          unsigned tid)
{
  const unsigned l = tid & 63u, w = tid >> 6;
  const unsigned shift = (unsigned)__builtin_ctz(nsub);
  const lds_f64 *const base = (const lds_f64 *)L.cols + (l & 15u) * ld + (l >> 4);
  d4 acc[3];
#pragma unroll
  for (unsigned k = 0u; k < 3u; ++k) {
    acc[k] = d4{0.0, 0.0, 0.0, 0.0};
    const unsigned u = w + STEP_WAVES * k, t = u >> shift;
    if (t >= 3u)
      continue;
    const unsigned r0 = (u & (nsub - 1u)) * SUB;
    // tile 0: block i with itself, 1: block j with block i, 2: j with itself
    const lds_f64 *const X = base + (t ? 16u * ld : 0u) + r0;
    const lds_f64 *const Y = base + (t == 2u ? 16u * ld : 0u) + r0;
    for (unsigned r = 0u; r < SUB; r += 64u) {
#pragma unroll
      for (unsigned j = 0u; j < 64u; j += 4u)
        acc[k] = mfma(X[r + j], Y[r + j], acc[k]);
    }
  }
  // The chains' tiles through LDS, entry by entry summed in sub-chunk order:
  // all three tiles at once behind the columns where there is room (fewer
  // than STEP_WAVES sub-chunks, of one wave each: one of up to 448 rows, two of
  // up to 384 or four of 256), else one at a time through the still unused R and W.
  static_assert(offsetof(PairLds, W) == sizeof(double) * 32u * LDR, "R and W adjoin");
  static_assert(2u * 32u * LDR >= STEP_WAVES * 256u, "room for a tile of every sub-chunk");
  const unsigned rounds = (nsub == STEP_WAVES) ? 3u : 1u;
  lds_f64 *const buf = (lds_f64 *)(rounds == 3u ? L.pair.R : L.cols + 32u * ld);
  const unsigned nt = rounds == 3u ? 1u : 3u;  // tiles a round
  double tot[3];
#pragma unroll
  for (unsigned rd = 0u; rd < 3u; ++rd) {
    if (rd >= rounds)
      break;
#pragma unroll
    for (unsigned k = 0u; k < 3u; ++k) {
      const unsigned u = w + STEP_WAVES * k, t = u >> shift;
      if (t < 3u && (nt == 3u || t == rd)) {
        lds_f64 *const o = buf + (nt == 3u ? u : (u & (nsub - 1u))) * 256u + l * 4u;
#pragma unroll
        for (unsigned r = 0u; r < 4u; ++r)
          o[r] = acc[k][r];
      }
    }
    __syncthreads();
    // entry tid of the round's tiles (and, of three, entry tid + 512)
#pragma unroll
    for (unsigned q = 0u; q < 2u; ++q) {
      const unsigned e = tid + STEP_NT * q;
      if (e < 256u * nt) {
        double p[STEP_WAVES];
#pragma unroll
        for (unsigned v = 0u; v < STEP_WAVES; ++v)
          if (v < nsub) p[v] = buf[((e >> 8) * nsub + v) * 256u + (e & 255u)];
        double sum = p[0];
#pragma unroll
        for (unsigned v = 1u; v < STEP_WAVES; ++v)
          if (v < nsub) sum = sum + p[v];
        tot[nt == 3u ? q : rd] = sum;
      }
    }
    if (nt == 1u)
      __syncthreads();
  }
  if (nt == 3u) {
    gram_entry(L.pair, tid, tot[0]);
    if (tid < 256u) gram_entry(L.pair, tid + STEP_NT, tot[1]);
  }
  else if (tid < 256u) {
#pragma unroll
    for (unsigned t = 0u; t < 3u; ++t)
      gram_entry(L.pair, 256u * t + tid, tot[t]);
  }
}

// out = x W for a 16-row slab: lane l, x[u] = row l%16 of pair column 4u +
// l/16; the products of k_update.  Stored to the columns at ci (block i) and
// cj, column step 4 ld, row offset r.
__device__ __forceinline__ void slab_update(const double *x, const double *a0, const double *a1,
                                            double *__restrict__ ci, double *__restrict__ cj,
                                            size_t step, unsigned r)
{
  d4 acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = acc0;
#pragma unroll
  for (unsigned u = 0u; u < 8u; ++u) {
    acc0 = mfma(a0[u], x[u], acc0);
    acc1 = mfma(a1[u], x[u], acc1);
  }
#pragma unroll
  for (unsigned u = 0u; u < 4u; ++u) {
    ci[u * step + r] = acc0[u];
    cj[u * step + r] = acc1[u];
  }
}

template <bool SORT>
__global__ __launch_bounds__(STEP_NT) void k_step(StepArgs A)
{
  __shared__ StepLds L;
  const unsigned tid = threadIdx.x, pi = blockIdx.x, l = tid & 63u, w = tid >> 6;
  const unsigned iBlk = A.pairs[2u * pi], jBlk = A.pairs[2u * pi + 1u];
  const unsigned ld = A.nrow + 2u;
  // (a sweep queued after the run's last one; a vector load)
  const unsigned done = __hip_atomic_load(&A.ctl->done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // the pair's columns, four a wave, all loads in flight together (rows are a
  // multiple of 64)
  {
    double v[4][STEP_MAX_ROWS / 64u];
#pragma unroll
    for (unsigned q = 0u; q < 4u; ++q) {
      const unsigned c = w + STEP_WAVES * q;
      const double *const g =
          A.G + (size_t)(c < 16u ? 16u * iBlk + c : 16u * jBlk + c - 16u) * A.ldG + l;
#pragma unroll
      for (unsigned k = 0u; k < STEP_MAX_ROWS / 64u; ++k)
        if (64u * k < A.nrow) v[q][k] = g[64u * k];
    }
#pragma unroll
    for (unsigned q = 0u; q < 4u; ++q)
#pragma unroll
      for (unsigned k = 0u; k < STEP_MAX_ROWS / 64u; ++k)
        if (64u * k < A.nrow) L.cols[(w + STEP_WAVES * q) * ld + 64u * k + l] = v[q][k];
  }
  // V's slabs w, w + 8, ... of the pair, read while the Gram and the visit run
  const unsigned nsv = A.nrowV / 16u;
  double *const vi = A.V + (size_t)(16u * iBlk + (l >> 4)) * A.ldV + (l & 15u);
  double *const vj = A.V + (size_t)(16u * jBlk + (l >> 4)) * A.ldV + (l & 15u);
  const size_t vstep = (size_t)4u * A.ldV;
  double xv[STEP_PER_WAVE][8];
#pragma unroll
  for (unsigned k = 0u; k < STEP_PER_WAVE; ++k) {
    const unsigned s = w + STEP_WAVES * k;
    if (s < nsv) {
#pragma unroll
      for (unsigned u = 0u; u < 4u; ++u) {
        xv[k][u] = vi[u * vstep + 16u * s];
        xv[k][4u + u] = vj[u * vstep + 16u * s];
      }
    }
  }
  if (done)
    return;
  __syncthreads();
  step_gram(L, ld, A.nsub, A.SUB, tid);
  visit_init<STEP_NT>(tid, L.pair, A.strat0);
#pragma unroll
  for (unsigned k = 0u; k < STEP_PER_WAVE; ++k)
#pragma unroll
    for (unsigned u = 0u; u < 8u; ++u)
      asm volatile("" : "+v"(xv[k][u]));  // read by now, not after the visit
  const PairSigns sg = pair_signs16(A.definite, A.nplus, iBlk, jBlk);
  if (!visit_core<SORT, STEP_LANES>(tid, pi, L.pair, sg, nullptr, A.ctl, A.rec, PLAN_FP64,
                                    A.s0steps, A.nswp))
    return;  // W is the identity
  const lds_f64 *const W = (const lds_f64 *)L.pair.W;
  double a0[8], a1[8];
#pragma unroll
  for (unsigned u = 0u; u < 8u; ++u) {
    a0[u] = RA(W, 4u * u + (l >> 4), l & 15u);
    a1[u] = RA(W, 4u * u + (l >> 4), 16u + (l & 15u));
  }
  double *const gi = A.G + (size_t)(16u * iBlk + (l >> 4)) * A.ldG + (l & 15u);
  double *const gj = A.G + (size_t)(16u * jBlk + (l >> 4)) * A.ldG + (l & 15u);
  const size_t gstep = (size_t)4u * A.ldG;
  const lds_f64 *const P = (const lds_f64 *)L.cols + (l >> 4) * ld + (l & 15u);
#pragma unroll 1
  for (unsigned s = w; s < A.nrow / 16u; s += STEP_WAVES) {
    double x[8];
#pragma unroll
    for (unsigned u = 0u; u < 8u; ++u)
      x[u] = P[4u * u * ld + 16u * s];
    slab_update(x, a0, a1, gi, gj, gstep, 16u * s);
  }
#pragma unroll
  for (unsigned k = 0u; k < STEP_PER_WAVE; ++k) {
    const unsigned s = w + STEP_WAVES * k;
    if (s < nsv)
      slab_update(xv[k], a0, a1, vi, vj, vstep, 16u * s);
  }
}

}  // namespace

void launch_step(hipStream_t s, bool sort, unsigned np, const StepArgs &a)
{
  if (sort)
    hipLaunchKernelGGL(k_step<true>, dim3(np), dim3(STEP_NT), 0, s, a);
  else
    hipLaunchKernelGGL(k_step<false>, dim3(np), dim3(STEP_NT), 0, s, a);
}

}  // namespace hj

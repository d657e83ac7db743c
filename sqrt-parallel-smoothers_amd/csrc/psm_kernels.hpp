// Kernels and host launchers of the parallel square-root smoother, templated
// on the real type, the state/observation dimensions and the form
// (square-root or covariance).
//
// Data layout in HBM
//  * Caller-visible trajectories are array-of-structs, exactly the shapes of the
//    reference: mean (n_states, nx), chol/cov (n_states, nx, nx).
//  * Internal per-state buffers (linearized model, smoother elements) and the
//    scan items are struct-of-arrays within blocks of 64 positions (blk), with
//    positions interleaved (StateMap, LevelMap) so that the items a wave works
//    on in one step are consecutive words.
//
// One filter pass over a ragged batch (all sequences concatenated, n_states
// states) is
//   1. k_linearize_states   one lane per state: transition and observation
//                           linearized at the nominal state
//   2. k_filter_reduce      one lane per chunk of C states: the chunk aggregate
//                           by absorbing its steps one by one
//   3. k_scan_up            exclusive scan of the chunk aggregates with the
//                           full filtering operator (Kogge-Stone inside a
//                           workgroup, recursive across workgroups; no
//                           down-sweep, see 4)
//   4. k_filter_apply       one lane per chunk: takes the prior through the
//                           chunk's prefixes of every scan level, then runs
//                           the sequential square-root Kalman filter from
//                           that incoming filtered state, writing the filtered
//                           states and the per-step log-likelihood terms
// and the smoother pass mirrors it backwards in time (elements, reverse scan,
// application).  Because the first state of every sequence carries its prior
// (and the last state of every sequence is the smoother's terminal element),
// both scans run over the concatenation without segment bookkeeping.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "psm_core.hpp"
#include "psm_scan_mem.hpp"
#include "psm_coop.hpp"

namespace psm {

constexpr int kScanWG = 64;     // one wave per scan workgroup
// Scan workgroup size for an aggregate type: one wave, or half a wave when three
// LDS buffers of 64 aggregates would not fit the 160 KB of LDS (tangent types).
template <typename Agg, typename R>
constexpr int scan_wg() {
  return (3 * odd_words(Agg::NQ) * 64 * (int)sizeof(R) <= 150 * 1024) ? 64 : 32;
}
constexpr int kLaneWG = 64;     // workgroup size of the lane-per-item kernels
constexpr int kRowVL = 16;      // groups of 16 lanes per workgroup of the cooperative scans

// Positions in the internal struct-of-arrays buffers.  The lane-per-chunk
// kernels run 64 consecutive chunks in one wave and step through their C
// states in lock step, so slot k of chunk c is stored at
//   (c / 64) * 64 C + 64 k + c % 64,
// and one component of one slot is 64 consecutive words for the wave (one
// full-line load instead of a C-strided gather).
struct StateMap {
  int C;
  PSM_DEV int64_t at(int64_t c, int64_t k) const { return (c >> 6) * ((int64_t)C << 6) + (k << 6) + (c & 63); }
  PSM_DEV int64_t operator()(int64_t i) const {
    const int64_t c = i / C;
    return at(c, i - c * C);
  }
};
inline int64_t state_stride(int64_t M, int C) {
  const int64_t g = (int64_t)C * 64;
  return (M + g - 1) / g * g;
}

// A scan level: n items in scan order, K per lane, WG lanes per workgroup.
// Scan position p of lane l, fold step j (p = blk * WG K + l K + j) is stored at
// blk * WG K + j WG + l, so every fold step of a workgroup touches WG
// consecutive words.  Level 0 holds the chunk aggregates: the smoother scans
// them in reverse (rev = 1), chunk c sitting at scan position n - 1 - c.
struct LevelMap {
  int64_t n;       // items
  int K;
  int WG;
  int rev;
  // (item counts fit 32 bits: 2^31 chunk aggregates would not fit the memory)
  PSM_DEV int64_t at(int64_t p) const {
    const uint32_t span = (uint32_t)K * (uint32_t)WG;
    const uint32_t b = (uint32_t)p / span;
    const uint32_t r = (uint32_t)p - b * span;
    const uint32_t l = r / (uint32_t)K;
    return (int64_t)b * span + (r - l * K) * WG + l;
  }
  // fold step j of lane t of workgroup b
  PSM_DEV int64_t at(int64_t b, int t, int j) const { return (b * K + j) * WG + t; }
  PSM_DEV int64_t pos(int64_t c) const { return at(rev ? n - 1 - c : c); }
};

PSM_DEV int seq_of(const int64_t* __restrict__ soff, int nseq, int64_t i) {
  int lo = 0, hi = nseq - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (soff[mid] <= i) lo = mid; else hi = mid - 1;
  }
  return lo;
}

template <typename R, int N>
PSM_DEV void ld_aos(const R* __restrict__ p, int64_t i, R (&v)[N]) {
#pragma unroll
  for (int a = 0; a < N; ++a) v[a] = p[i * N + a];
}
template <typename R, int M, int N>
PSM_DEV void ld_aos(const R* __restrict__ p, int64_t i, R (&v)[M][N]) {
#pragma unroll
  for (int a = 0; a < M; ++a)
#pragma unroll
    for (int b = 0; b < N; ++b) v[a][b] = p[i * M * N + a * N + b];
}
template <typename R, int N>
PSM_DEV void st_aos(R* __restrict__ p, int64_t i, const R (&v)[N]) {
#pragma unroll
  for (int a = 0; a < N; ++a) p[i * N + a] = v[a];
}
template <typename R, int M, int N>
PSM_DEV void st_aos(R* __restrict__ p, int64_t i, const R (&v)[M][N]) {
#pragma unroll
  for (int a = 0; a < M; ++a)
#pragma unroll
    for (int b = 0; b < N; ++b) p[i * M * N + a * N + b] = v[a][b];
}

// Trajectories (a mean and a factor per state) come in two layouts: the API's
// array-of-structs (state i at m + i NX, L + i NX^2; inter == 0), or, inside a
// launch sequence that owns them, the state-interleaved layout of the
// workspace (inter != 0: blocked at the state's interleaved position pos, means
// first, then a factor's lower triangle or a covariance in full (SYM), so that a
// launch sequence and the host loop over the same passes agree bit for bit),
// which lane-per-chunk kernels read and write coalesced.
template <bool SYM, int NX>
constexpr int kTrajWords = NX + (SYM ? NX * NX : NX * (NX + 1) / 2);
template <bool SYM, typename R, int NX>
PSM_DEV void traj_load(const R* __restrict__ m_, const R* __restrict__ L_, int inter,
                       int64_t i, int64_t pos, R (&m)[NX], R (&L)[NX][NX]) {
  if (inter) {
    const R* p = blk<kTrajWords<SYM, NX>>(m_, pos);
    int q = 0;
    ld(p, kBlk, 0, q, m);
    if constexpr (SYM) ld(p, kBlk, 0, q, L);
    else ld_tri<false>(p, kBlk, 0, q, L);
  } else {
    ld_aos(m_, i, m);
    ld_aos(L_, i, L);
  }
}
template <bool SYM, typename R, int NX>
PSM_DEV void traj_store(R* __restrict__ m_, R* __restrict__ L_, int inter, int64_t i,
                        int64_t pos, const R (&m)[NX], const R (&L)[NX][NX]) {
  if (inter) {
    R* p = blk<kTrajWords<SYM, NX>>(m_, pos);
    int q = 0;
    st(p, kBlk, 0, q, m);
    if constexpr (SYM) st(p, kBlk, 0, q, L);
    else st_tri(p, kBlk, 0, q, L);
  } else {
    st_aos(m_, i, m);
    st_aos(L_, i, L);
  }
}

// p[0..n) <- v (flag words and counters; a kernel rather than hipMemsetAsync,
// so that a captured graph replays it like any other launch)
template <typename T>
__global__ void k_fill(T* __restrict__ p, int n, T v) {
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < n) p[i] = v;
}

// ============================================================================
// 1. linearization at every nominal state
// ============================================================================
template <typename R, int NIN, int NOUT, bool SQRT, typename S>
PSM_DEV void linearize_point(const ModelView<R, S>& md, const SigmaView<R>& sp, int use_sigma,
                             const R (&m)[NIN], const R (&Lx)[NIN][NIN], R (&F)[NOUT][NIN],
                             R (&C)[NOUT][NOUT], R (&b)[NOUT]) {
  if (use_sigma) {
    if constexpr (SQRT) {
      linearize_sigma<R, NIN, NOUT, true>(md, sp, m, Lx, F, C, b);
    } else {
      R Lc[NIN][NIN];
      cholesky(Lx, Lc);   // get_mvnsqrt (parsmooth/linearization/_common.py:9-14)
      linearize_sigma<R, NIN, NOUT, false>(md, sp, m, Lc, F, C, b);
    }
  } else {
    linearize_extended<R, NIN, NOUT>(md, m, F, C, b);
  }
}

// Linearization of the single-precision paths.  In FP32 arithmetic the
// textbook formulas cancel: the sigma-point regression subtracts F P F^T from
// the sigma-point covariance, which is ~0.1 against a process noise Q ~ 3e-9
// on the bearings-only model; the coordinated turn's turn-rate derivatives are
// differences of two numbers ~dt that agree to O((w dt)^2); b = f(m) - F m
// cancels at large |m|.  The FP32 path therefore uses the cancellation-free
// forms of psm_models.hpp (centred residuals, series in w dt, closed-form
// offsets), all in FP32.  Rules with a negative weight and conditional-moments
// models keep the reference's downdate form, evaluated in FP64 from the FP32
// inputs and rounded back.  In square-root form, a regression noise factor
// whose min|diag| / max|diag| falls below the fallback threshold is recomputed
// that way too (and counted), like every other triangular factor.
template <typename R> struct WiderOf { using type = R; };
template <> struct WiderOf<float> { using type = double; };
template <> struct WiderOf<DualT<float>> { using type = DualT<double>; };

template <typename A, int N, typename B>
PSM_DEV void widen(const B (&a)[N], A (&b)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) b[i] = A(a[i]);
}
template <typename A, int M, int N, typename B>
PSM_DEV void widen(const B (&a)[M][N], A (&b)[M][N]) {
#pragma unroll
  for (int i = 0; i < M; ++i) widen(a[i], b[i]);
}

// b <- b + F m - next, formed in FP64
template <typename R, int NO, int NI, typename N>
PSM_DEV void centre(const R (&F)[NO][NI], const R (&m)[NI], const N (&next)[NO], R (&b)[NO]) {
#pragma unroll
  for (int a = 0; a < NO; ++a) {
    double s = (double)b[a] - (double)next[a];
#pragma unroll
    for (int k = 0; k < NI; ++k) s = fma((double)F[a][k], (double)m[k], s);
    b[a] = (R)s;
  }
}

template <typename R, int NIN, int NOUT, bool SQRT, typename From>
PSM_DEV void linearize_point_wide(const ModelView<R>& md, const SigmaView<R>& sp, int use_sigma,
                                  const R (&m)[NIN], const R (&Lx)[NIN][NIN], R (&F)[NOUT][NIN],
                                  R (&C)[NOUT][NOUT], R (&b)[NOUT], const From& from) {
  using W = typename WiderOf<R>::type;
  const ModelView<W, R> mw{md.kind, md.params, md.q_mean, md.q_chol, md.row, md.pt, md.npts};
  const SigmaView<W> sw{sp.npts, sp.xi, sp.wm, sp.wc};
  W mW[NIN], LW[NIN][NIN], FW[NOUT][NIN], CW[NOUT][NOUT], bW[NOUT];
  widen(m, mW);
  widen(Lx, LW);
  linearize_point<W, NIN, NOUT, SQRT>(mw, sw, use_sigma, mW, LW, FW, CW, bW);
  if constexpr (From::kNominal) centre(FW, mW, from.next, bW);
  widen(FW, F);
  widen(CW, C);
  widen(bW, b);
}

template <typename R, int NIN, int NOUT, bool SQRT, typename FB, typename PC = NoPoints, typename From = FromZero>
PSM_DEV void linearize_point_w(const ModelView<R>& md, const SigmaView<R>& sp, int use_sigma,
                               const R (&m)[NIN], const R (&Lx)[NIN][NIN], R (&F)[NOUT][NIN],
                               R (&C)[NOUT][NOUT], R (&b)[NOUT], const FB& fb,
                               const PC& pc = PC{}, const From& from = From{}) {
  if constexpr (kFallback<R, SQRT> && !FB::kRedo) {
    // FP32 square-root pass without FP64 code: a point the centred regression
    // cannot take (conditional moments, a negative weight) or whose factor is
    // ill-conditioned raises the flag, and the guarded second launch
    // linearizes every point again with the FP64 path below
    if (!use_sigma) {
      linearize_extended<R, NIN, NOUT>(md, m, F, C, b);
      if constexpr (From::kNominal) centre(F, from.at, from.next, b);
      return;
    }
    const bool done = md.kind != PSM_MODEL_CONDITIONAL &&
                      linearize_sigma_centred<R, NIN, NOUT, true>(md, sp, m, Lx, F, C, b, pc, from);
    if (!done || (fb.thr > 0.0f && ill_conditioned(C, fb.thr))) fb.raise();
  } else if constexpr (IsSingle<R>::value) {
    if (!use_sigma) {
      linearize_extended<R, NIN, NOUT>(md, m, F, C, b);
      if constexpr (From::kNominal) centre(F, from.at, from.next, b);
      return;
    }
    bool done = false;
    if (md.kind != PSM_MODEL_CONDITIONAL) {
      if constexpr (SQRT) {
        done = linearize_sigma_centred<R, NIN, NOUT, true>(md, sp, m, Lx, F, C, b, pc, from);
        if constexpr (kFallback<R, SQRT>) {
          if (done && fb.thr > 0.0f && ill_conditioned(C, fb.thr)) {
            count_fallback(fb);
            done = false;
          }
        }
      } else {
        R Lc[NIN][NIN];
        cholesky(Lx, Lc);   // get_mvnsqrt (parsmooth/linearization/_common.py:9-14)
        done = linearize_sigma_centred<R, NIN, NOUT, false>(md, sp, m, Lc, F, C, b, pc, from);
      }
    }
    if (!done) linearize_point_wide<R, NIN, NOUT, SQRT>(md, sp, use_sigma, m, Lx, F, C, b, from);
  } else {
    linearize_point<R, NIN, NOUT, SQRT>(md, sp, use_sigma, m, Lx, F, C, b);
  }
}

// Centred states of the FP32 square-root passes.  Between the linearization and
// the output every mean is a difference from the nominal mean of its state:
// x_k = n_k + d_k turns x_{k+1} = F x_k + b into d_{k+1} = F d_k + b', b' = b + F n_k
// - n_{k+1}, and y = H x + c into y = H d + c', c' = c + H n_k.  Under the extended rule
// these sums are formed in FP64, where n_k, n_{k+1} and F are exact; a regression's
// b' is E f - n_{k+1} (model_minus and the mean increment): by way of b, which FP32
// rounds at the size of x, every step had that rounding for an offset (8.6e-6 at a
// position of 300, against a process noise of 5.8e-5).  The rounding of an aggregate's A (about 1 on
// its diagonal, so 6e-8 a step, adding up along a sequence) multiplies d, of the
// size of the posterior's spread, and not x, a position of 10 to 1000: the
// smoothed means of a T = 16,385 pass were 1.5e-5 of their norm off a 64-bit
// recursion, and are 1.8e-6 with this.  ref holds n_k (blocked at the states'
// interleaved positions, NX words; RefSource).  Trajectories hold n + d in either layout, so that a
// launch sequence and the host loop over the same passes agree bit for bit.
template <typename R, bool SQRT>
constexpr bool kCentred = SQRT && std::is_same<R, float>::value;

// Which values the means are held relative to.  A regression and the nonlinear models
// take the nominal, which their result depends on in any case.  A linear model
// under the extended rule does not, and must not lose the digits of a nominal that is
// far from the states, or all of them to one that is not finite: with a linear
// transition a smoother or a sampler takes the filtered mean, and with a linear
// observation too a filter takes the prior mean where there is one, the nominal
// in the components that are observed, as far as their contributions to an observation
// are no larger than twice the observation, and zero elsewhere (constant velocity in
// the plane, T = 5,000, means against FP64: a nominal near the states 2.5e-8 of the
// norm off; zeros, one 1e4 or 1e6 away or not a number 1.5e-7, where relative to it
// they were 2.4e-6 and 1.9e-4 off or lost; absolute means were 2.8e-7 off).
enum { REF_NOMINAL = 0, REF_CHECKED = 1, REF_FILTERED = 2 };
template <typename R>
struct RefSource {
  int mode;
  const int64_t* soff;
  int nseq;
  const R* ys;
  const R* m0;
  const R* fm;
};
// The reference of state i, whose nominal mean is n.
template <typename R, int NX, int NY>
PSM_DEV void ref_mean(const RefSource<R>& rs, const ModelView<R>& ob, int64_t i, const R (&n)[NX], R (&ref)[NX]) {
  copy(n, ref);
  if (rs.mode == REF_FILTERED) {
    ld_aos(rs.fm, i, ref);
  } else if (rs.mode == REF_CHECKED) {
    const int s = seq_of(rs.soff, rs.nseq, i);
    if (i == rs.soff[s]) {
      ld_aos(rs.m0, s, ref);
    } else {
      R y[NY];
      ld_aos(rs.ys, i - s - 1, y);
      bool seen[NX], far[NX];
#pragma unroll
      for (int j = 0; j < NX; ++j) seen[j] = far[j] = false;
#pragma unroll
      for (int r = 0; r < NY; ++r) {
        R a = R(0);
#pragma unroll
        for (int j = 0; j < NX; ++j) a += ob.par(r * NX + j) != R(0) ? abs_(ob.par(r * NX + j) * n[j]) : R(0);
        const bool ok = a <= R(2) * abs_(y[r] - ob.qm(r));   // not for NaN
#pragma unroll
        for (int j = 0; j < NX; ++j) {
          if (ob.par(r * NX + j) != R(0)) {
            seen[j] = true;
            far[j] = far[j] || !ok;
          }
        }
      }
#pragma unroll
      for (int j = 0; j < NX; ++j) ref[j] = seen[j] && !far[j] ? n[j] : R(0);
    }
  }
#pragma unroll
  for (int j = 0; j < NX; ++j) ref[j] = isfinite(ref[j]) ? ref[j] : R(0);
}

// m -/+ the reference mean at interleaved position pos
template <typename R, int NX>
PSM_DEV void to_centred(const R* __restrict__ ref, int64_t pos, R (&m)[NX]) {
  R n[NX];
  int q = 0;
  ld(blk<NX>(ref, pos), kBlk, 0, q, n);
#pragma unroll
  for (int a = 0; a < NX; ++a) m[a] -= n[a];
}
template <typename R, int NX>
PSM_DEV void from_centred(const R* __restrict__ ref, int64_t pos, R (&m)[NX]) {
  R n[NX];
  int q = 0;
  ld(blk<NX>(ref, pos), kBlk, 0, q, n);
#pragma unroll
  for (int a = 0; a < NX; ++a) m[a] += n[a];
}

// Thread t fills position t of the state-interleaved buffer (coalesced stores);
// its state is the inverse of StateMap.
template <typename R, int NX, int NY, bool SQRT, typename FB = Fallback>
__global__ __launch_bounds__(kLaneWG) void k_linearize_states(
    int64_t M, int64_t Mp, int C, ModelView<R> tr, ModelView<R> ob, int do_obs, SigmaView<R> sp,
    int use_sigma, const R* __restrict__ nom_m, const R* __restrict__ nom_L, int nom_inter,
    RefSource<R> rs, R* __restrict__ lin, R* __restrict__ ref, FB fb) {
  if (fb.skip()) return;
  // FP32: the rule is converted once per workgroup, and the regressions' increments
  // wait in LDS for their residual passes
  constexpr bool kSingle = std::is_same<R, float>::value;
  constexpr int kPts = kSingle ? 2 * NX + 1 : 1, kOut = kSingle ? (NX > NY ? NX : NY) : 1;
  __shared__ R increments[kPts * kOut * (kSingle ? kLaneWG : 1)], rule[kPts * (NX + 2)];
  const bool staged = kSingle && use_sigma && sp.npts <= kPts;
  if (staged) {
    for (int q = threadIdx.x; q < sp.npts * NX; q += kLaneWG) rule[q] = sp.pxi(q);
    for (int p = threadIdx.x; p < sp.npts; p += kLaneWG) {
      rule[kPts * NX + p] = sp.pwm(p);
      rule[kPts * (NX + 1) + p] = sp.pwc(p);
    }
    __syncthreads();
  }
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= Mp) return;
  const int64_t g = (int64_t)C << 6;
  const int64_t gb = t / g;
  const int64_t r = t - gb * g;
  const int64_t i = ((gb << 6) + (r & 63)) * C + (r >> 6);
  if (i >= M) return;
  tr.row = i;
  ob.row = i;
  R m[NX], L[NX][NX];
  traj_load<!SQRT, R, NX>(nom_m, nom_L, nom_inter, i, t, m, L);
  R at[NX];
  if constexpr (kCentred<R, SQRT>) ref_mean<R, NX, NY>(rs, ob, i, m, at);
  R* lp = blk<Step<R, NX, NY>::NQ>(lin, t);
  auto run = [&](const auto& pc) {
    {
      R F[NX][NX], Cq[NX][NX], b[NX];
      if constexpr (kCentred<R, SQRT>) {
        R next[NX];
        copy(at, next);
        if (i + 1 < M) {
          R n[NX];
          if (nom_inter) {
            // the next slot of this chunk, or the first of the next
            const int64_t pos = (r >> 6) + 1 < C ? t + 64 : StateMap{C}(i + 1);
            int q = 0;
            ld(blk<kTrajWords<!SQRT, NX>>(nom_m, pos), kBlk, 0, q, n);
          } else {
            ld_aos(nom_m, i + 1, n);
          }
          ref_mean<R, NX, NY>(rs, ob, i + 1, n, next);
        }
        int q = 0;
        st(blk<NX>(ref, t), kBlk, 0, q, at);
        linearize_point_w<R, NX, NX, SQRT>(tr, sp, use_sigma, m, L, F, Cq, b, fb, pc, FromNominal<R, NX, NX>{at, next});
      } else {
        linearize_point_w<R, NX, NX, SQRT>(tr, sp, use_sigma, m, L, F, Cq, b, fb, pc);
      }
      int q = 0;
      st(lp, kBlk, 0, q, F);
      if constexpr (SQRT) lower_factor(Cq);
      st_tri(lp, kBlk, 0, q, Cq);
      st(lp, kBlk, 0, q, b);
    }
    if (do_obs) {
      R H[NY][NX], Cr[NY][NY], c[NY];
      if constexpr (kCentred<R, SQRT>) {
        const R zero[NY] = {};
        linearize_point_w<R, NX, NY, SQRT>(ob, sp, use_sigma, m, L, H, Cr, c, fb, pc, FromNominal<R, NX, NY>{at, zero});
      } else {
        linearize_point_w<R, NX, NY, SQRT>(ob, sp, use_sigma, m, L, H, Cr, c, fb, pc);
      }
      int q = Step<R, NX, NY>::NTRANS;
      st(lp, kBlk, 0, q, H);
      if constexpr (SQRT) lower_factor(Cr);
      st_tri(lp, kBlk, 0, q, Cr);
      st(lp, kBlk, 0, q, c);
    }
  };
  if constexpr (kSingle) {
    if (staged) {
      run(PointCache<R>{increments + threadIdx.x, kLaneWG, rule, rule + kPts * NX, rule + kPts * (NX + 1)});
      return;
    }
  }
  run(NoPoints{});
}

// ============================================================================
// 2. chunk aggregates of the filter
// ============================================================================
template <typename R, int NX, int NY, bool SQRT, typename FB = Fallback>
__global__ __launch_bounds__(kLaneWG) void k_filter_reduce(
    int64_t M, int chunk, int64_t nchunks, const int64_t* __restrict__ soff, int nseq,
    const R* __restrict__ lin, const R* __restrict__ ys, const R* __restrict__ m0,
    const R* __restrict__ L0, const R* __restrict__ ref, R* __restrict__ agg, LevelMap lm, FB fb) {
  if (fb.skip()) return;
  const StateMap sm{chunk};
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nchunks) return;
  const int64_t i0 = c * chunk;
  const int64_t i1 = min(i0 + chunk, M);
  int s = seq_of(soff, nseq, i0);
  FAgg<R, NX> a;
  set_identity(a);
  for (int64_t i = i0; i < i1; ++i) {
    while (i >= soff[s + 1]) ++s;
    if (i == soff[s]) {
      set_zero(a.A);
      ld_aos(m0, s, a.b);
      if constexpr (kCentred<R, SQRT>) to_centred(ref, sm.at(c, i - i0), a.b);
      ld_aos(L0, s, a.U);
      if constexpr (SQRT) lower_factor(a.U);
      set_zero(a.eta);
      set_zero(a.Z);
      a.flag = FLAG_HEAD;
    } else {
      Step<R, NX, NY> st_;
      load_trans<!SQRT>(lin, i > i0 ? sm.at(c, i - i0 - 1) : sm.at(c - 1, chunk - 1), st_);
      load_obs<!SQRT>(lin, sm.at(c, i - i0), st_);
      R y[NY];
      ld_aos(ys, i - s - 1, y);
      absorb_fb<R, NX, NY, SQRT>(a, st_, y, fb);
    }
  }
  store_agg(agg, lm.pos(c), a);
}

// ============================================================================
// 3. exclusive scan of aggregates (filter: forward, smoother: reverse)
// ============================================================================
// in/out: the items of one level (LevelMap: n items in scan order, stored
// interleaved).  Workgroup w covers scan positions [w*WG*K, (w+1)*WG*K): every
// lane folds its K items, a Kogge-Stone scan over the lanes runs in a
// double-buffered LDS array, and the lane then writes the exclusive prefix of
// each of its items (within the workgroup) to out_excl; the workgroup's
// inclusive total becomes item w of the next level (tm).  Aggregates live in
// LDS / HBM, never whole in registers: the operator reads its operands from
// memory as it needs them.
template <typename Agg, typename R, bool SQRT, int WG = scan_wg<Agg, R>(), typename FB = Fallback>
__global__ __launch_bounds__(WG) void k_scan_up(const R* __restrict__ in, LevelMap lm,
                                                R* __restrict__ out_excl, R* __restrict__ totals,
                                                LevelMap tm, FB fb) {
  if (fb.skip()) return;
  using V = typename ViewOf<Agg>::type;
  constexpr int NX = Agg_nx<Agg>::value;
  constexpr int NQ = Agg::NQ;
  // buffers 0 and 1: running / scanned aggregates; buffer 2: the lane's next
  // input item, copied from HBM in one burst so that the combination reads
  // only LDS
  __shared__ R lds[3 * NQ * WG];
  const int t = threadIdx.x;
  const int K = lm.K;
  const int64_t n = lm.n;
  auto slot = [&](int buf, int lane) { return V{lds + buf * NQ * WG, (int64_t)WG, (int64_t)lane}; };
  const V stage = slot(2, t);
  const int64_t base = ((int64_t)blockIdx.x * WG + t) * K;
  auto view = [&](const R* p, int64_t pos) { return V{blk<NQ>(const_cast<R*>(p), pos), kBlk, 0}; };
  auto item = [&](int j) { return view(in, lm.at(blockIdx.x, t, j)); };
  int cur = 0;
  if (base < n) view_copy(item(0), slot(0, t));
  else view_identity(slot(0, t));
  for (int j = 1; j < K; ++j) {
    const int64_t p = base + j;
    if (p >= n) break;
    view_copy(item(j), stage);
    combine_mem_fb<R, NX, SQRT>(slot(cur, t), stage, slot(1 - cur, t), fb);
    cur = 1 - cur;
  }
  if (cur == 1) view_copy(slot(1, t), slot(0, t));
  cur = 0;
  for (int d = 1; d < WG; d <<= 1) {
    __syncthreads();
    if (t >= d) combine_mem_fb<R, NX, SQRT>(slot(cur, t - d), slot(cur, t), slot(1 - cur, t), fb);
    else view_copy(slot(cur, t), slot(1 - cur, t));
    cur = 1 - cur;
  }
  __syncthreads();
  if (t == WG - 1 && totals != nullptr)
    view_copy(slot(cur, t), view(totals, tm.at((int64_t)blockIdx.x)));
  // running exclusive prefix in this lane's slot of the other buffer; once
  // every lane has read its predecessor's inclusive prefix, slot(cur, t) is
  // free for the next running prefix
  V run = slot(1 - cur, t);
  if (t == 0) view_identity(run);
  else view_copy(slot(cur, t - 1), run);
  __syncthreads();
  V tmp = slot(cur, t);
  for (int j = 0; j < K; ++j) {
    const int64_t p = base + j;
    if (p >= n) break;
    view_copy(run, view(out_excl, lm.at(blockIdx.x, t, j)));
    // the running prefix after the lane's last item is its inclusive total,
    // which the scan over the lanes already produced
    if (j + 1 == K || p + 1 == n) break;
    view_copy(item(j), stage);
    combine_mem_fb<R, NX, SQRT>(run, stage, tmp, fb);
    const V x = run;
    run = tmp;
    tmp = x;
  }
}

// k_scan_up with G lanes per combination
// (psm_coop.hpp): VL groups per workgroup, each one virtual lane of the scan
// above (folds K items, joins the Kogge-Stone scan over the groups, rewrites its
// items' exclusive prefixes).  The level layout is that of k_scan_up with VL
// lanes, so the two are interchangeable.  One call site combines in all three
// parts, so the instructions of a combination are fetched once.
template <typename Agg, typename R, bool SQRT, int G, int VL, typename FB = Fallback>
__global__ __launch_bounds__(VL * G) void k_scan_up_coop(
    const R* __restrict__ in, LevelMap lm, R* __restrict__ out_excl, R* __restrict__ totals,
    LevelMap tm, FB fb) {
  if (fb.skip()) return;
  using V = typename ViewOf<Agg>::type;
  constexpr int NQP = odd_words(Agg::NQ);
  __shared__ R acc[NQP * VL];    // the running / scanned aggregate of each group
  __shared__ R stage[NQP * VL];  // the group's next input item
  const int t = (int)threadIdx.x / G;
  const int r = (int)threadIdx.x % G;
  R* mine = acc + t * NQP;
  R* my_stage = stage + t * NQP;
  const int K = lm.K;
  const int64_t n = lm.n;
  const int64_t base = ((int64_t)blockIdx.x * VL + t) * K;
  constexpr int NQ = Agg::NQ;
  auto view = [&](const R* p, int64_t pos) { return V{blk<NQ>(const_cast<R*>(p), pos), kBlk, 0}; };
  {
    ItemRegs<V, G> move;
    if (base < n) move.load(view(in, lm.at(blockIdx.x, t, 0)), r);
    else move.identity(r);
    move.store(mine, r);
  }
  constexpr int kScan = VL == 64 ? 6 : VL == 32 ? 5 : VL == 16 ? 4 : 0;
  static_assert((1 << kScan) == VL, "groups per workgroup");
  const int folds = K - 1;
  const int steps = folds + kScan + folds;
  for (int step = 0;; ++step) {
    // an opaque copy of the lane: what the step derives from it (offsets, row
    // kinds, addresses) is formed anew each time, not hoisted into registers that
    // live through the combinations
    int rl = r;
    asm volatile("" : "+v"(rl));
    const bool fold = step < folds, scan = !fold && step < folds + kScan;
    const int j = fold ? step + 1 : step - folds - kScan;   // item of a fold / rewrite step
    if (step == folds + kScan) {
      // the workgroup's total, and the exclusive prefix of each group
      __syncthreads();
      if (t == VL - 1 && totals != nullptr) {
        ItemRegs<V, G> move;
        move.load(mine, rl);
        move.store(view(totals, tm.at((int64_t)blockIdx.x)), rl);
      }
      ItemRegs<V, G> move;
      if (t == 0) move.identity(rl);
      else move.load(mine - NQP, rl);
      __syncthreads();
      move.store(mine, rl);
    }
    if (step >= folds + kScan && base + j < n) {
      group_sync();
      ItemRegs<V, G> move;
      move.load(mine, rl);
      move.store(view(out_excl, lm.at(blockIdx.x, t, j)), rl);
    }
    if (step == steps) break;
    R* e1 = mine;
    const R* e2 = my_stage;
    bool act = base + j < n;
    if (scan) {
      const int d = 1 << (step - folds);
      act = t >= d;
      e1 = act ? mine - d * NQP : mine;
      e2 = mine;
      __syncthreads();
    } else {
      if (act) {
        ItemRegs<V, G> move;
        move.load(view(in, lm.at(blockIdx.x, t, j)), rl);
        move.store(my_stage, rl);
      }
      group_sync();
    }
    // an idle group keeps what it has: its running aggregate is e1 outside the scan
    CoopStep<V, G, SQRT> cs;
    if (act) cs.prepare(e1, e2, !scan, rl, fb);
    if (scan) __syncthreads();
    else group_sync();
    cs.commit(mine, rl);
  }
}

// ============================================================================
// 4. filter application
// ============================================================================
// The exclusive prefixes of every scan level, level 0 (the chunks) first: an
// item's prefix covers the items before it in its own workgroup, the prefix of
// its workgroup is an item of the next level.
template <typename R>
struct ScanLevels {
  static constexpr int kMax = 16;
  int n;
  uint32_t span[kMax];   // chunks per item of the level
  const R* prefix[kMax];
  LevelMap map[kMax];
};

// Takes the first distribution of the scan through the prefixes that precede
// chunk c, from the top level down.  The whole prefix of a chunk contains the
// first state of its sequence (HEAD), so it is a distribution (m, L) and
// taking it through one more aggregate costs half a combination: no
// A, eta and Z are formed.  Every lane of a wavefront does this for its own chunk
// with consecutive lanes on consecutive items; it replaces a down-sweep, which
// would read and write every aggregate of a level once more.
// Push(view, m, L): (m, L) <- aggregate applied to (m, L).
template <typename V, typename R, int NX, typename Push>
PSM_DEV void enter_chunk(int64_t c, const ScanLevels<R>& lv, R (&m)[NX], R (&L)[NX][NX], Push&& push) {
  const uint32_t p0 = (uint32_t)(lv.map[0].rev ? lv.map[0].n - 1 - c : c);
  for (int l = lv.n - 1; l >= 0; --l) {
    const V v{blk<V::QF + 1>(const_cast<R*>(lv.prefix[l]), lv.map[l].at(p0 / lv.span[l])), kBlk, 0};
    const int f = v.flag();
    if (f == FLAG_IDENT) continue;
    if (f == FLAG_HEAD) view_head(v, m, L);
    else push(v, m, L);
  }
}

template <typename R, int NX, int NY, bool SQRT, typename FB = Fallback>
__global__ __launch_bounds__(kLaneWG) void k_filter_apply(
    int64_t M, int chunk, int64_t nchunks, const int64_t* __restrict__ soff, int nseq,
    const R* __restrict__ lin, const R* __restrict__ ys, const R* __restrict__ m0,
    const R* __restrict__ L0, const R* __restrict__ ref, ScanLevels<R> lv, R* __restrict__ out_m,
    R* __restrict__ out_L, int out_inter, typename AccOf<R>::type* __restrict__ ell_state, FB fb) {
  if (fb.skip()) return;
  using Acc = typename AccOf<R>::type;
  const StateMap sm{chunk};
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nchunks) return;
  const int64_t i0 = c * chunk;
  const int64_t i1 = min(i0 + chunk, M);
  int s = seq_of(soff, nseq, i0);
  R m[NX], L[NX][NX];
  set_zero(m);
  set_zero(L);
  enter_chunk<FView<R, NX>>(c, lv, m, L, [&](const FView<R, NX>& v, R (&mm)[NX], R (&LL)[NX][NX]) {
    filter_push_fb<R, NX, SQRT>(v, mm, LL, fb);
  });
  for (int64_t i = i0; i < i1; ++i) {
    while (i >= soff[s + 1]) ++s;
    Acc e = Acc(0.0);
    if (i == soff[s]) {
      ld_aos(m0, s, m);
      ld_aos(L0, s, L);
      // the caller's factor of the prior goes out as it is; the recursion and the
      // interleaved trajectory take its lower triangular form
      if (!out_inter) traj_store<!SQRT, R, NX>(out_m, out_L, 0, i, sm.at(c, i - i0), m, L);
      if constexpr (SQRT) lower_factor(L);
      if (out_inter) traj_store<!SQRT, R, NX>(out_m, out_L, 1, i, sm.at(c, i - i0), m, L);
      if constexpr (kCentred<R, SQRT>) to_centred(ref, sm.at(c, i - i0), m);
    } else {
      Step<R, NX, NY> st_;
      load_trans<!SQRT>(lin, i > i0 ? sm.at(c, i - i0 - 1) : sm.at(c - 1, chunk - 1), st_);
      load_obs<!SQRT>(lin, sm.at(c, i - i0), st_);
      R y[NY];
      ld_aos(ys, i - s - 1, y);
      e = kf_step_fb<R, NX, NY, SQRT>(st_, y, m, L, fb);
      R x[NX];
      copy(m, x);
      if constexpr (kCentred<R, SQRT>) from_centred(ref, sm.at(c, i - i0), x);
      traj_store<!SQRT, R, NX>(out_m, out_L, out_inter, i, sm.at(c, i - i0), x, L);
    }
    if (ell_state != nullptr) ell_state[i] = e;
  }
}

// Per-sequence sum of the per-state log-likelihood terms (FP64).  One block per
// sequence, as wide as the sequences are long (ell_threads), with 8 loads in flight
// per thread: the sum is bound by their latency (131,072 states: 17 us; with 256
// threads and one load each 127).
inline int ell_threads(int64_t M, int64_t nseq) {
  const int64_t mean = M / nseq;
  return mean <= 128 ? 64 : mean <= 2048 ? 256 : 1024;
}

template <int BS, typename Acc>
__global__ __launch_bounds__(BS) void k_ell_reduce(const Acc* __restrict__ ell_state,
                                                    const int64_t* __restrict__ soff,
                                                    Acc* __restrict__ ell) {
  __shared__ Acc red[BS];
  const int s = blockIdx.x;
  const int64_t a = soff[s], b = soff[s + 1];
  constexpr int NU = 8;
  Acc part[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) part[u] = Acc(0.0);
  int64_t i = a + threadIdx.x;
  for (; i + (NU - 1) * BS < b; i += NU * BS) {
#pragma unroll
    for (int u = 0; u < NU; ++u) part[u] += ell_state[i + u * BS];
  }
#pragma unroll
  for (int u = 0; u < NU - 1; ++u)
    if (i + u * BS < b) part[u] += ell_state[i + u * BS];
  Acc acc = part[0];
#pragma unroll
  for (int u = 1; u < NU; ++u) acc += part[u];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int w = BS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) ell[s] = red[0];
}

// ============================================================================
// smoother passes
// ============================================================================
template <typename R, int NX, int NY, bool SQRT, typename FB = Fallback>
__global__ __launch_bounds__(kLaneWG) void k_smoother_reduce(
    int64_t M, int chunk, int64_t nchunks, const int64_t* __restrict__ soff, int nseq,
    const R* __restrict__ lin, const R* __restrict__ fm, const R* __restrict__ fL, int f_inter,
    const R* __restrict__ ref, R* __restrict__ elems, R* __restrict__ agg, LevelMap lm, FB fb) {
  if (fb.skip()) return;
  const StateMap sm{chunk};
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nchunks) return;
  const int64_t i0 = c * chunk;
  const int64_t i1 = min(i0 + chunk, M);
  int s = seq_of(soff, nseq, i1 - 1);
  SAgg<R, NX> acc;
  set_identity(acc);
  for (int64_t i = i1 - 1; i >= i0; --i) {
    while (i < soff[s]) --s;
    R m[NX], L[NX][NX];
    const int64_t pos = sm.at(c, i - i0);
    traj_load<!SQRT, R, NX>(fm, fL, f_inter, i, pos, m, L);
    if constexpr (kCentred<R, SQRT>) to_centred(ref, pos, m);
    SAgg<R, NX> e;
    if (i == soff[s + 1] - 1) {
      copy(m, e.g);
      set_zero(e.E);
      copy(L, e.D);
      e.flag = FLAG_HEAD;
    } else {
      // a caller's filtered factors may be any square roots
      if constexpr (SQRT) {
        if (!f_inter) lower_factor(L);
      }
      R F[NX][NX], cq[NX][NX], bt[NX];
      const R* p = blk<Step<R, NX, NY>::NQ>(lin, pos);
      int q = 0;
      ld(p, kBlk, 0, q, F);
      ld_tri<!SQRT>(p, kBlk, 0, q, cq);
      ld(p, kBlk, 0, q, bt);
      smoother_element_fb<R, NX, SQRT>(F, cq, bt, m, L, e, fb);
    }
    store_agg(elems, pos, e);
    if constexpr (SQRT) {
      if (!f_inter && e.flag == FLAG_HEAD) lower_factor(e.D);
    }
    combine_into_fb<R, NX, SQRT>(acc, e, fb);
    copy_agg(e, acc);
  }
  store_agg(agg, lm.pos(c), acc);
}

template <typename R, int NX, bool SQRT, typename FB = Fallback>
__global__ __launch_bounds__(kLaneWG) void k_smoother_apply(
    int64_t M, int chunk, int64_t nchunks, const R* __restrict__ elems,
    ScanLevels<R> lv, const R* __restrict__ ref, R* __restrict__ out_m, R* __restrict__ out_L, int out_inter,
    FB fb) {
  if (fb.skip()) return;
  const StateMap sm{chunk};
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nchunks) return;
  const int64_t i0 = c * chunk;
  const int64_t i1 = min(i0 + chunk, M);
  R m[NX], D[NX][NX];
  set_zero(m);
  set_zero(D);
  enter_chunk<SView<R, NX>>(c, lv, m, D, [&](const SView<R, NX>& v, R (&mm)[NX], R (&DD)[NX][NX]) {
    SAgg<R, NX> e;
    view_load(v, e);
    smoother_apply_fb<R, NX, SQRT>(e, mm, DD, fb);
  });
  for (int64_t i = i1 - 1; i >= i0; --i) {
    SAgg<R, NX> e;
    load_agg(elems, sm.at(c, i - i0), e);
    if (e.flag == FLAG_HEAD) {
      copy(e.g, m);
      copy(e.D, D);
    } else {
      smoother_apply_fb<R, NX, SQRT>(e, m, D, fb);
    }
    R x[NX];
    copy(m, x);
    if constexpr (kCentred<R, SQRT>) from_centred(ref, sm.at(c, i - i0), x);
    if (e.flag == FLAG_HEAD) {
      // the last filtered factor goes out as it is; the recursion and the
      // interleaved trajectory take its lower triangular form
      if (!out_inter) st_aos(out_L, i, D);
      if constexpr (SQRT) lower_factor(D);
    }
    if (out_inter || e.flag != FLAG_HEAD) traj_store<!SQRT, R, NX>(out_m, out_L, out_inter, i, sm.at(c, i - i0), x, D);
    else st_aos(out_m, i, x);
  }
}

// ============================================================================
// operator-level batched kernels (array-of-structs in and out)
// ============================================================================
template <typename R, int NIN, int NOUT, bool SQRT>
__global__ __launch_bounds__(kLaneWG) void k_linearize_points(
    int64_t n, ModelView<R> md, SigmaView<R> sp, int use_sigma, const R* __restrict__ xm,
    const R* __restrict__ xL, R* __restrict__ F, R* __restrict__ C, R* __restrict__ b) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  md.row = i;
  R m[NIN], L[NIN][NIN], Fo[NOUT][NIN], Co[NOUT][NOUT], bo[NOUT];
  ld_aos(xm, i, m);
  ld_aos(xL, i, L);
  linearize_point_w<R, NIN, NOUT, SQRT>(md, sp, use_sigma, m, L, Fo, Co, bo, Fallback{0.0f, nullptr});
  st_aos(F, i, Fo);
  st_aos(C, i, Co);
  st_aos(b, i, bo);
}

template <typename R, int NX, int NY, bool SQRT>
__global__ __launch_bounds__(kLaneWG) void k_filter_elements(
    int64_t n, const R* __restrict__ F, const R* __restrict__ cq, const R* __restrict__ bt,
    const R* __restrict__ H, const R* __restrict__ cr, const R* __restrict__ c,
    const R* __restrict__ m, const R* __restrict__ L, const R* __restrict__ y, R* __restrict__ A,
    R* __restrict__ b, R* __restrict__ U, R* __restrict__ eta, R* __restrict__ Z) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  Step<R, NX, NY> s;
  ld_aos(F, i, s.F);
  ld_aos(cq, i, s.cq);
  ld_aos(bt, i, s.bt);
  ld_aos(H, i, s.H);
  ld_aos(cr, i, s.cr);
  ld_aos(c, i, s.c);
  R mm_[NX], LL[NX][NX], yy[NY];
  ld_aos(m, i, mm_);
  ld_aos(L, i, LL);
  ld_aos(y, i, yy);
  if constexpr (SQRT) {  // a caller's factors may be any square roots
    lower_factor(s.cq);
    lower_factor(LL);
  }
  FAgg<R, NX> e;
  filter_element<R, NX, NY, SQRT>(s, mm_, LL, yy, e);
  st_aos(A, i, e.A);
  st_aos(b, i, e.b);
  st_aos(U, i, e.U);
  st_aos(eta, i, e.eta);
  st_aos(Z, i, e.Z);
}

template <typename R, int NX>
struct FPtrs {
  const R* p[5];
};
template <typename R, int NX>
struct FOut {
  R* p[5];
};

template <typename R, int NX, bool SQRT>
__global__ __launch_bounds__(kLaneWG) void k_filter_combine(int64_t n, FPtrs<R, NX> a,
                                                            FPtrs<R, NX> b, FOut<R, NX> o) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  FAgg<R, NX> e1, e2;
  ld_aos(a.p[0], i, e1.A); ld_aos(a.p[1], i, e1.b); ld_aos(a.p[2], i, e1.U);
  ld_aos(a.p[3], i, e1.eta); ld_aos(a.p[4], i, e1.Z);
  ld_aos(b.p[0], i, e2.A); ld_aos(b.p[1], i, e2.b); ld_aos(b.p[2], i, e2.U);
  ld_aos(b.p[3], i, e2.eta); ld_aos(b.p[4], i, e2.Z);
  e1.flag = FLAG_NORMAL;
  e2.flag = FLAG_NORMAL;
  if constexpr (SQRT) {  // a caller's factors may be any square roots
    lower_factor(e1.U);
    lower_factor(e1.Z);
    lower_factor(e2.U);
    lower_factor(e2.Z);
  }
  combine_into<R, NX, SQRT>(e1, e2);
  st_aos(o.p[0], i, e2.A); st_aos(o.p[1], i, e2.b); st_aos(o.p[2], i, e2.U);
  st_aos(o.p[3], i, e2.eta); st_aos(o.p[4], i, e2.Z);
}

template <typename R, int NX, bool SQRT>
__global__ __launch_bounds__(kLaneWG) void k_smoother_elements(
    int64_t n, const R* __restrict__ F, const R* __restrict__ cq, const R* __restrict__ bt,
    const R* __restrict__ m, const R* __restrict__ L, R* __restrict__ g, R* __restrict__ E,
    R* __restrict__ D) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  R Fi[NX][NX], cqi[NX][NX], bti[NX], mi[NX], Li[NX][NX];
  ld_aos(F, i, Fi);
  ld_aos(cq, i, cqi);
  ld_aos(bt, i, bti);
  ld_aos(m, i, mi);
  ld_aos(L, i, Li);
  if constexpr (SQRT) {  // a caller's factors may be any square roots
    lower_factor(cqi);
    lower_factor(Li);
  }
  SAgg<R, NX> e;
  smoother_element<R, NX, SQRT>(Fi, cqi, bti, mi, Li, e);
  st_aos(g, i, e.g);
  st_aos(E, i, e.E);
  st_aos(D, i, e.D);
}

template <typename R, int NX>
struct SPtrs {
  const R* p[3];
};
template <typename R, int NX>
struct SOut {
  R* p[3];
};

template <typename R, int NX, bool SQRT>
__global__ __launch_bounds__(kLaneWG) void k_smoother_combine(int64_t n, SPtrs<R, NX> a,
                                                              SPtrs<R, NX> b, SOut<R, NX> o) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  SAgg<R, NX> e1, e2;
  ld_aos(a.p[0], i, e1.g); ld_aos(a.p[1], i, e1.E); ld_aos(a.p[2], i, e1.D);
  ld_aos(b.p[0], i, e2.g); ld_aos(b.p[1], i, e2.E); ld_aos(b.p[2], i, e2.D);
  e1.flag = FLAG_NORMAL;
  e2.flag = FLAG_NORMAL;
  if constexpr (SQRT) {  // a caller's factors may be any square roots
    lower_factor(e1.D);
    lower_factor(e2.D);
  }
  combine_into<R, NX, SQRT>(e1, e2);
  st_aos(o.p[0], i, e2.g); st_aos(o.p[1], i, e2.E); st_aos(o.p[2], i, e2.D);
}

}  // namespace psm

// Sequential filter and smoother (parallel=False): one lane per sequence runs
// the Kalman recursion through its steps, linearizing as it goes.
//
// Without a nominal trajectory the reference linearizes at the running
// estimate -- the transition at the filtered state, the observation at the
// predicted state (parsmooth/sequential/_filtering.py:31-43), and in the
// smoother the transition at the smoothed successor
// (parsmooth/sequential/_smoothing.py:27-33) -- which no parallel scan can
// reproduce, since each linearization point depends on the previous step.
// With a nominal trajectory both read it instead.  A ragged batch of many
// short sequences fills the device one sequence per lane with no scan work.
#pragma once
#include "psm_kernels.hpp"

namespace psm {

// Predicted distribution (m1, L1) of one transition step: the linearization
// point of the observation when there is no nominal trajectory.
template <typename R, int NX, bool SQRT>
PSM_DEV void seq_predict(const R (&F)[NX][NX], const R (&cq)[NX][NX], const R (&bt)[NX],
                         const R (&m)[NX], const R (&L)[NX][NX], R (&m1)[NX], R (&L1)[NX][NX]) {
  mv(F, m, m1);
#pragma unroll
  for (int i = 0; i < NX; ++i) m1[i] += bt[i];
  if constexpr (SQRT) {
    R M[NX][2 * NX];
#pragma unroll
    for (int i = 0; i < NX; ++i)
#pragma unroll
      for (int j = 0; j < NX; ++j) {
        R acc = F[i][j] * L[j][j];
#pragma unroll
        for (int k = j + 1; k < NX; ++k) acc = fma(F[i][k], L[k][j], acc);
        M[i][j] = acc;
        M[i][NX + j] = cq[i][j];
      }
    tria_lower_inplace<NX>(M);
#pragma unroll
    for (int i = 0; i < NX; ++i)
#pragma unroll
      for (int j = 0; j < NX; ++j) L1[i][j] = M[i][j];
  } else {
    R FP[NX][NX];
#pragma unroll
    for (int i = 0; i < NX; ++i)
#pragma unroll
      for (int j = 0; j < NX; ++j) {
        R acc = R(0);
#pragma unroll
        for (int k = 0; k < NX; ++k) acc = fma(F[i][k], L[k][j], acc);
        FP[i][j] = acc;
      }
#pragma unroll
    for (int i = 0; i < NX; ++i)
#pragma unroll
      for (int j = 0; j < NX; ++j) {
        R acc = cq[i][j];
#pragma unroll
        for (int k = 0; k < NX; ++k) acc = fma(FP[i][k], F[j][k], acc);
        L1[i][j] = acc;
      }
  }
}

// Lane s filters sequence s: states [soff[s], soff[s+1]), state soff[s] the
// prior.  nom_m == nullptr: linearize at the running estimate.  ell (may be
// null) receives the per-sequence log-likelihood, accumulated in FP64.
template <typename R, int NX, int NY, bool SQRT>
__global__ __launch_bounds__(kLaneWG) void k_seq_filter(
    int nseq, const int64_t* __restrict__ soff, ModelView<R> tr, ModelView<R> ob, SigmaView<R> sp,
    int use_sigma, const R* __restrict__ nom_m, const R* __restrict__ nom_L,
    const R* __restrict__ ys, const R* __restrict__ m0, const R* __restrict__ L0,
    R* __restrict__ out_m, R* __restrict__ out_L, typename AccOf<R>::type* __restrict__ ell,
    Fallback fb) {
  using Acc = typename AccOf<R>::type;
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nseq) return;
  const int64_t a = soff[s], e = soff[s + 1];
  R m[NX], L[NX][NX];
  ld_aos(m0, s, m);
  ld_aos(L0, s, L);
  st_aos(out_m, a, m);
  st_aos(out_L, a, L);
  // the recursion takes lower triangular factors; a caller's may be any square roots
  if constexpr (SQRT) lower_factor(L);
  Acc acc = Acc(0.0);
  for (int64_t i = a + 1; i < e; ++i) {
    Step<R, NX, NY> st_;
    R rm[NX], rL[NX][NX];
    if (nom_m != nullptr) {
      ld_aos(nom_m, i - 1, rm);
      ld_aos(nom_L, i - 1, rL);
    } else {
      copy(m, rm);
      copy(L, rL);
    }
    tr.row = i - 1;
    linearize_point_w<R, NX, NX, SQRT>(tr, sp, use_sigma, rm, rL, st_.F, st_.cq, st_.bt, fb);
    if constexpr (SQRT) lower_factor(st_.cq);
    if (nom_m != nullptr) {
      ld_aos(nom_m, i, rm);
      ld_aos(nom_L, i, rL);
    } else {
      seq_predict<R, NX, SQRT>(st_.F, st_.cq, st_.bt, m, L, rm, rL);
    }
    ob.row = i;
    linearize_point_w<R, NX, NY, SQRT>(ob, sp, use_sigma, rm, rL, st_.H, st_.cr, st_.c, fb);
    R y[NY];
    ld_aos(ys, i - s - 1, y);
    acc += kf_step_fb<R, NX, NY, SQRT>(st_, y, m, L, fb);
    st_aos(out_m, i, m);
    st_aos(out_L, i, L);
  }
  if (ell != nullptr) ell[s] = acc;
}

// Lane s smooths sequence s backwards from its last filtered state (the
// Rauch-Tung-Striebel recursion as a smoother element applied to the
// smoothed successor).  nom_m == nullptr: the transition out of state i is
// linearized at the smoothed state i+1.
template <typename R, int NX, bool SQRT>
__global__ __launch_bounds__(kLaneWG) void k_seq_smoother(
    int nseq, const int64_t* __restrict__ soff, ModelView<R> tr, SigmaView<R> sp, int use_sigma,
    const R* __restrict__ nom_m, const R* __restrict__ nom_L, const R* __restrict__ fm,
    const R* __restrict__ fL, R* __restrict__ out_m, R* __restrict__ out_L, Fallback fb) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nseq) return;
  const int64_t a = soff[s], e = soff[s + 1];
  R m[NX], D[NX][NX];
  ld_aos(fm, e - 1, m);
  ld_aos(fL, e - 1, D);
  st_aos(out_m, e - 1, m);
  st_aos(out_L, e - 1, D);
  if constexpr (SQRT) lower_factor(D);
  for (int64_t i = e - 2; i >= a; --i) {
    R rm[NX], rL[NX][NX];
    if (nom_m != nullptr) {
      ld_aos(nom_m, i, rm);
      ld_aos(nom_L, i, rL);
    } else {
      copy(m, rm);
      copy(D, rL);
    }
    R F[NX][NX], cq[NX][NX], bt[NX];
    tr.row = i;
    linearize_point_w<R, NX, NX, SQRT>(tr, sp, use_sigma, rm, rL, F, cq, bt, fb);
    if constexpr (SQRT) lower_factor(cq);
    R xm[NX], xL[NX][NX];
    ld_aos(fm, i, xm);
    ld_aos(fL, i, xL);
    if constexpr (SQRT) lower_factor(xL);
    SAgg<R, NX> el;
    smoother_element_fb<R, NX, SQRT>(F, cq, bt, xm, xL, el, fb);
    smoother_apply_fb<R, NX, SQRT>(el, m, D, fb);
    st_aos(out_m, i, m);
    st_aos(out_L, i, D);
  }
}

// ---------------------------------------------------------------- ahead of the recursion
// At a nominal trajectory the linearizations (and, smoothing, the whole smoother
// elements) do not depend on the recursion.  A workgroup then takes 64 sequences
// with one wavefront for the recursion and P more that form the next P steps
// meanwhile, on SIMDs that a batch of up to 64 sequences per CU leaves idle:
//   round r:  wavefront 1 + p forms step r P + p in registers, while wavefront 0
//             takes its 64 sequences through the steps of round r - 1 from LDS;
//             barrier; the new steps go to LDS; barrier.
// Every lane takes part in every round of the longest of its 64 sequences.
// 4,096 tracks of 20 to 100 steps, FP64: 345 us a filter and 235 a smoother pass,
// 725 and 900 with all of a step on the recursion's lane.
constexpr size_t kLdsBytes = 160 * 1024;
template <int NW, typename R>
constexpr int ahead_waves() {
  return kLdsBytes / (NW * 64 * sizeof(R)) >= 3 ? 3 : (int)(kLdsBytes / (NW * 64 * sizeof(R)));
}
// With every workgroup on a CU of its own, the recursion's wavefront has a SIMD
// to itself; beyond, the forming wavefronts would take the place of other
// sequences' recursions.
constexpr int kAheadMaxSeqs = 64 * 256;

// longest of the 64 sequences' step counts, on every lane
PSM_DEV int64_t wave_max(int64_t n) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    const int64_t o = __shfl_xor((long long)n, d, 64);
    n = o > n ? o : n;
  }
  return n;
}

// form(j): step j into registers; put(buf, lane): those to LDS; take(buf, lane, j)
template <int P, int NW, typename R, typename Form, typename Put, typename Take>
PSM_DEV void seq_ahead(R (&buf)[P][NW * 64], int64_t n, Form&& form, Put&& put, Take&& take) {
  const int wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
  const int64_t rounds = (wave_max(n) + P - 1) / P;
  for (int64_t r = 0; r <= rounds; ++r) {
    const int64_t j = r * P + (wave - 1);
    const bool forms = wave > 0 && j < n;
    if (wave == 0) {
      for (int p = 0; p < P; ++p) {
        const int64_t i = (r - 1) * P + p;
        if (i >= 0 && i < n) take(buf[p], lane, i);
      }
    } else if (forms) {
      form(j);
    }
    __syncthreads();
    if (forms) put(buf[wave - 1], lane);
    __syncthreads();
  }
}

template <typename R, int N1, int N2>
PSM_DEV void put_words(R* b, int lane, int& q, const R (&a)[N1][N2]) {
#pragma unroll
  for (int i = 0; i < N1; ++i)
#pragma unroll
    for (int j = 0; j < N2; ++j) b[64 * q++ + lane] = a[i][j];
}
template <typename R, int N>
PSM_DEV void put_words(R* b, int lane, int& q, const R (&a)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) b[64 * q++ + lane] = a[i];
}
template <typename R, int N1, int N2>
PSM_DEV void take_words(const R* b, int lane, int& q, R (&a)[N1][N2]) {
#pragma unroll
  for (int i = 0; i < N1; ++i)
#pragma unroll
    for (int j = 0; j < N2; ++j) a[i][j] = b[64 * q++ + lane];
}
template <typename R, int N>
PSM_DEV void take_words(const R* b, int lane, int& q, R (&a)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) a[i] = b[64 * q++ + lane];
}

template <typename R, int NX, int NY>
struct SeqFilterAhead {
  static constexpr int NW = 2 * NX * NX + NX + NY * NX + NY * NY + 2 * NY;
  static constexpr int P = ahead_waves<NW, R>();
};
template <typename R, int NX, int NY, bool SQRT>
__global__ __launch_bounds__(64 * (1 + SeqFilterAhead<R, NX, NY>::P)) void k_seq_filter_ahead(
    int nseq, const int64_t* __restrict__ soff, ModelView<R> tr, ModelView<R> ob, SigmaView<R> sp,
    int use_sigma, const R* __restrict__ nom_m, const R* __restrict__ nom_L,
    const R* __restrict__ ys, const R* __restrict__ m0, const R* __restrict__ L0,
    R* __restrict__ out_m, R* __restrict__ out_L, typename AccOf<R>::type* __restrict__ ell,
    Fallback fb) {
  using Acc = typename AccOf<R>::type;
  constexpr int NW = SeqFilterAhead<R, NX, NY>::NW, P = SeqFilterAhead<R, NX, NY>::P;
  __shared__ R buf[P][NW * 64];
  const int s = blockIdx.x * 64 + ((int)threadIdx.x & 63);
  const bool have = s < nseq;
  const int64_t a = have ? soff[s] : 0, e = have ? soff[s + 1] : 1;
  R m[NX], L[NX][NX];
  if (have && threadIdx.x < 64) {
    ld_aos(m0, s, m);
    ld_aos(L0, s, L);
    st_aos(out_m, a, m);
    st_aos(out_L, a, L);
    if constexpr (SQRT) lower_factor(L);
  }
  Acc acc = Acc(0.0);
  Step<R, NX, NY> f;
  R y[NY];
  seq_ahead<P, NW>(buf, e - a - 1,
    [&](int64_t j) {
      const int64_t i = a + 1 + j;
      R rm[NX], rL[NX][NX];
      ld_aos(ys, i - s - 1, y);
      ld_aos(nom_m, i - 1, rm);
      ld_aos(nom_L, i - 1, rL);
      tr.row = i - 1;
      linearize_point_w<R, NX, NX, SQRT>(tr, sp, use_sigma, rm, rL, f.F, f.cq, f.bt, fb);
      if constexpr (SQRT) lower_factor(f.cq);
      ld_aos(nom_m, i, rm);
      ld_aos(nom_L, i, rL);
      ob.row = i;
      linearize_point_w<R, NX, NY, SQRT>(ob, sp, use_sigma, rm, rL, f.H, f.cr, f.c, fb);
    },
    [&](R* b, int lane) {
      int q = 0;
      put_words(b, lane, q, f.F);
      put_words(b, lane, q, f.cq);
      put_words(b, lane, q, f.bt);
      put_words(b, lane, q, f.H);
      put_words(b, lane, q, f.cr);
      put_words(b, lane, q, f.c);
      put_words(b, lane, q, y);
    },
    [&](const R* b, int lane, int64_t j) {
      Step<R, NX, NY> g;
      R yy[NY];
      int q = 0;
      take_words(b, lane, q, g.F);
      take_words(b, lane, q, g.cq);
      take_words(b, lane, q, g.bt);
      take_words(b, lane, q, g.H);
      take_words(b, lane, q, g.cr);
      take_words(b, lane, q, g.c);
      take_words(b, lane, q, yy);
      acc += kf_step_fb<R, NX, NY, SQRT>(g, yy, m, L, fb);
      st_aos(out_m, a + 1 + j, m);
      st_aos(out_L, a + 1 + j, L);
    });
  if (have && threadIdx.x < 64 && ell != nullptr) ell[s] = acc;
}

template <typename R, int NX>
struct SeqSmootherAhead {
  static constexpr int NW = 2 * NX * NX + NX;
  static constexpr int P = ahead_waves<NW, R>();
};
template <typename R, int NX, bool SQRT>
__global__ __launch_bounds__(64 * (1 + SeqSmootherAhead<R, NX>::P)) void k_seq_smoother_ahead(
    int nseq, const int64_t* __restrict__ soff, ModelView<R> tr, SigmaView<R> sp, int use_sigma,
    const R* __restrict__ nom_m, const R* __restrict__ nom_L, const R* __restrict__ fm,
    const R* __restrict__ fL, R* __restrict__ out_m, R* __restrict__ out_L, Fallback fb) {
  constexpr int NW = SeqSmootherAhead<R, NX>::NW, P = SeqSmootherAhead<R, NX>::P;
  __shared__ R buf[P][NW * 64];
  const int s = blockIdx.x * 64 + ((int)threadIdx.x & 63);
  const bool have = s < nseq;
  const int64_t a = have ? soff[s] : 0, e = have ? soff[s + 1] : 1;
  R m[NX], D[NX][NX];
  if (have && threadIdx.x < 64) {
    ld_aos(fm, e - 1, m);
    ld_aos(fL, e - 1, D);
    st_aos(out_m, e - 1, m);
    st_aos(out_L, e - 1, D);
    if constexpr (SQRT) lower_factor(D);
  }
  SAgg<R, NX> el;
  seq_ahead<P, NW>(buf, e - a - 1,
    [&](int64_t j) {
      const int64_t i = e - 2 - j;
      R rm[NX], rL[NX][NX], F[NX][NX], cq[NX][NX], bt[NX];
      ld_aos(nom_m, i, rm);
      ld_aos(nom_L, i, rL);
      tr.row = i;
      linearize_point_w<R, NX, NX, SQRT>(tr, sp, use_sigma, rm, rL, F, cq, bt, fb);
      if constexpr (SQRT) lower_factor(cq);
      ld_aos(fm, i, rm);
      ld_aos(fL, i, rL);
      if constexpr (SQRT) lower_factor(rL);
      smoother_element_fb<R, NX, SQRT>(F, cq, bt, rm, rL, el, fb);
    },
    [&](R* b, int lane) {
      int q = 0;
      put_words(b, lane, q, el.g);
      put_words(b, lane, q, el.E);
      put_words(b, lane, q, el.D);
    },
    [&](const R* b, int lane, int64_t j) {
      SAgg<R, NX> g;
      g.flag = 0;
      int q = 0;
      take_words(b, lane, q, g.g);
      take_words(b, lane, q, g.E);
      take_words(b, lane, q, g.D);
      smoother_apply_fb<R, NX, SQRT>(g, m, D, fb);
      st_aos(out_m, e - 2 - j, m);
      st_aos(out_L, e - 2 - j, D);
    });
}

}  // namespace psm

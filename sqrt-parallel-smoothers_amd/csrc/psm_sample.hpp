// Pathwise sampling from the smoothing distribution
// (parsmooth/_pathwise_sampler.py:13-38 and :64-127).
//
// With the smoother elements (g_k, E_k, D_k) of the nominal trajectory, a
// sample path is the backward affine recursion
//     x_k = E_k x_{k+1} + g_k + D_k eps_k          (D_k: chol; in covariance
//                                                   form its Cholesky factor)
// whose last state of every sequence is its own head element (E = 0:
// x_T = m_T + L_T eps_T), so a ragged batch needs no segment bookkeeping.  The
// reference runs the recursion as an associative scan of the affine maps
// (G2 G1, G2 e1 + e2); here it is a chain through chunks of Cs states, which form
// groups of Cs chunks:
//   1. k_sample_reduce  lane (chunk, column): the chunk's composite map
//                       P_c = E_i0 ... E_i1-1 and offset o_c; a column is a
//                       sample (offset) or a unit vector (column of P_c), so
//                       that every step is one matrix-vector product
//   2. k_sample_fold    lane (group, column): the same over the group's chunks
//   3. k_sample_bounds  lane per sample: the states at the group starts,
//                       backwards over the groups
//   4. k_sample_spread  lane (group, sample): the states at the group's chunk
//                       starts
//   5. k_sample_apply   lane (chunk, sample): the recursion through the chunk
// (one chunk takes 5 alone, one group 1, 4 and 5).  With Cs about the cube root of
// the states the chain is at most 5 Cs steps: T = 16,384 and 64 samples take 144, on
// 512 x 69 lanes in 1 and 512 x 64 in 5, and 48, 16, 8, 22 and 44 us (one level of 128 chunks, where every sample's lane formed P_c too:
// 656, 25 and 201 us).  Each lane loads the next item before it uses the current
// one: kernels 1 and 5 read every element once per column, from cache.  The
// standard normals eps (n_states, n_samples, nx) are drawn by the caller.
#pragma once
#include "psm_kernels.hpp"

namespace psm {

// Items per chunk and chunks per group: about the cube root of the states.
inline int64_t sample_chunk(int64_t M) {
  int64_t c = 16;
  while (c * c * c < M && c < 1024) c += 8;
  return c;
}

template <typename R, int NX, bool SQRT>
struct SampleItem {
  SAgg<R, NX> a;
  R eps[NX];
  int64_t at;
  PSM_DEV void load(const R* __restrict__ elems, int64_t pos, const R* __restrict__ e) {
    load_agg(elems, pos, a);
    at = pos;
    if (e != nullptr) {
#pragma unroll
      for (int i = 0; i < NX; ++i) eps[i] = e[i];
    } else {
      set_zero(eps);
    }
  }
  // x <- E x [+ g + D eps]; D is a factor, or its covariance.  The factors are lower
  // triangular, but for a sequence's last one, which is the caller's: what it has above
  // the diagonal is loaded there alone (16,384 states and 64 samples: 166 us, 173 with
  // the whole of every factor).
  PSM_DEV void step(bool off, const R* __restrict__ elems, R (&x)[NX]) const {
    R L[NX][NX], y[NX];
    if constexpr (SQRT) copy(a.D, L);
    else cholesky(a.D, L);
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      R s = a.g[i];
#pragma unroll
      for (int j = 0; j <= i; ++j) s = fma(L[i][j], eps[j], s);
      y[i] = off ? s : R(0);
#pragma unroll
      for (int j = 0; j < NX; ++j) y[i] = fma(a.E[i][j], x[j], y[i]);
    }
    if constexpr (SQRT) {
      if (a.flag == FLAG_HEAD && off) {
        const R* p = blk<SAgg<R, NX>::NQ>(elems, at) + (NX + NX * NX) * kBlk;
#pragma unroll
        for (int i = 0; i < NX; ++i)
#pragma unroll
          for (int j = i + 1; j < NX; ++j) y[i] = fma(p[(i * NX + j) * kBlk], eps[j], y[i]);
      }
    }
    copy(y, x);
  }
};

// Column q of a composite map: an offset (q < S, from zero) or column q - S of the
// matrix (from a unit vector, without offsets).
template <typename R, int NX>
PSM_DEV void sample_start(int q, int S, R (&x)[NX]) {
#pragma unroll
  for (int i = 0; i < NX; ++i) x[i] = q - S == i ? R(1) : R(0);
}
template <typename R, int NX>
PSM_DEV void sample_map_store(int64_t c, int q, int S, const R (&x)[NX], R* __restrict__ P, R* __restrict__ o) {
  if (q < S) {
    st_aos(o, c * S + q, x);
  } else {
#pragma unroll
    for (int i = 0; i < NX; ++i) P[(c * NX + i) * NX + (q - S)] = x[i];
  }
}

template <typename R, int NX, bool SQRT>
__global__ __launch_bounds__(kLaneWG) void k_sample_reduce(
    int64_t M, int chunk, int64_t Cs, int64_t nch, int S, const R* __restrict__ elems,
    const R* __restrict__ eps, R* __restrict__ P, R* __restrict__ o) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int cols = S + NX;
  if (t >= nch * cols) return;
  const int64_t c = t / cols;
  const int q = (int)(t - c * cols);
  const StateMap sm{chunk};
  const int64_t i0 = c * Cs;
  const int64_t i1 = min(i0 + Cs, M);
  const bool off = q < S;
  auto noise = [&](int64_t k) { return off ? eps + (k * S + q) * NX : nullptr; };
  R x[NX];
  sample_start(q, S, x);
  SampleItem<R, NX, SQRT> cur, next;
  cur.load(elems, sm(i1 - 1), noise(i1 - 1));
  for (int64_t k = i1 - 1; k >= i0; --k) {
    if (k > i0) next.load(elems, sm(k - 1), noise(k - 1));
    cur.step(off, elems, x);
    cur = next;
  }
  sample_map_store(c, q, S, x, P, o);
}

template <typename R, int NX>
__global__ __launch_bounds__(kLaneWG) void k_sample_fold(int64_t nch, int64_t Cs, int64_t ngr, int S,
                                                         const R* __restrict__ P, const R* __restrict__ o,
                                                         R* __restrict__ P2, R* __restrict__ o2) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int cols = S + NX;
  if (t >= ngr * cols) return;
  const int64_t d = t / cols;
  const int q = (int)(t - d * cols);
  const int64_t c0 = d * Cs, c1 = min(c0 + Cs, nch);
  R x[NX];
  sample_start(q, S, x);
  for (int64_t c = c1 - 1; c >= c0; --c) {
    R Pm[NX][NX], ov[NX], xn[NX];
    ld_aos(P, c, Pm);
    if (q < S) ld_aos(o, c * S + q, ov);
    else set_zero(ov);
    mv(Pm, x, xn);
#pragma unroll
    for (int i = 0; i < NX; ++i) x[i] = xn[i] + ov[i];
  }
  sample_map_store(d, q, S, x, P2, o2);
}

// xb[c]: the state at the start of item c, backwards over the items [c0, c1) of a
// lane from the state behind its last one (xin at `in`, zero if null).
template <typename R, int NX>
PSM_DEV void sample_walk(int64_t c0, int64_t c1, int S, int s, const R* __restrict__ P,
                         const R* __restrict__ o, const R* __restrict__ xin, R* __restrict__ xb) {
  R x[NX];
  if (xin != nullptr) ld_aos(xin, 0, x);
  else set_zero(x);
  for (int64_t c = c1 - 1; c >= c0; --c) {
    R Pm[NX][NX], ov[NX], xn[NX];
    ld_aos(P, c, Pm);
    ld_aos(o, c * S + s, ov);
    mv(Pm, x, xn);
#pragma unroll
    for (int i = 0; i < NX; ++i) x[i] = xn[i] + ov[i];
    st_aos(xb, c * S + s, x);
  }
}

template <typename R, int NX>
__global__ __launch_bounds__(kLaneWG) void k_sample_bounds(int64_t ngr, int S, const R* __restrict__ P2,
                                                           const R* __restrict__ o2,
                                                           R* __restrict__ xg) {
  const int s = (int)((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
  if (s >= S) return;
  sample_walk<R, NX>(0, ngr, S, s, P2, o2, nullptr, xg);
}

template <typename R, int NX>
__global__ __launch_bounds__(kLaneWG) void k_sample_spread(int64_t nch, int64_t Cs, int64_t ngr, int S,
                                                           const R* __restrict__ P, const R* __restrict__ o,
                                                           const R* __restrict__ xg, R* __restrict__ xb) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ngr * S) return;
  const int64_t d = t / S;
  const int s = (int)(t - d * S);
  sample_walk<R, NX>(d * Cs, min((d + 1) * Cs, nch), S, s, P, o,
                     d + 1 < ngr ? xg + ((d + 1) * S + s) * NX : nullptr, xb);
}

template <typename R, int NX, bool SQRT>
__global__ __launch_bounds__(kLaneWG) void k_sample_apply(
    int64_t M, int chunk, int64_t Cs, int64_t nch, int S, const R* __restrict__ elems,
    const R* __restrict__ eps, const R* __restrict__ xb, const R* __restrict__ ref, R* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nch * S) return;
  const int64_t c = t / S;
  const int s = (int)(t - c * S);
  const StateMap sm{chunk};
  const int64_t i0 = c * Cs;
  const int64_t i1 = min(i0 + Cs, M);
  R x[NX];
  if (c + 1 < nch) ld_aos(xb, (c + 1) * S + s, x);
  else set_zero(x);
  SampleItem<R, NX, SQRT> cur, next;
  cur.load(elems, sm(i1 - 1), eps + ((i1 - 1) * S + s) * NX);
  for (int64_t k = i1 - 1; k >= i0; --k) {
    if (k > i0) next.load(elems, sm(k - 1), eps + ((k - 1) * S + s) * NX);
    cur.step(true, elems, x);
    R xn[NX];
    copy(x, xn);
    if constexpr (kCentred<R, SQRT>) from_centred(ref, sm(k), xn);
    st_aos(out, k * S + s, xn);
    cur = next;
  }
}

}  // namespace psm

// Register-resident small dense linear algebra for the square-root smoother
// kernels (gfx950).  Every matrix is a fixed-size C array held in VGPRs; all
// loops have compile-time trip counts and are fully unrolled, so one lane owns
// one whole problem instance (a time step, a chunk aggregate, ...).
//
// Conventions
//  * Row-major R M[rows][cols].
//  * tria(M) returns the lower-triangular L with L L^T = M M^T and a
//    non-negative diagonal (Householder reflections applied from the right,
//    row by row, with the sign choice that maps a row tail onto +||x|| e_0).
//    This is the operation parsmooth/_utils.py:22-24 computes through a QR of
//    M^T; the reference's diagonal signs come from LAPACK and are arbitrary, the
//    sign choice here makes the factor unique.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#define PSM_DEV __device__ __forceinline__

namespace psm {

// sqrt for the factorisations' non-negative, finite arguments: the hardware
// reciprocal square-root estimate, one Goldschmidt step for sqrt(x) and
// 1 / (2 sqrt(x)), and a final residual correction; it matched the correctly
// rounded square root on a million random normal values in 1e-30..1e30 (and
// at 0), without the IEEE sequence's rescaling of tiny arguments.
PSM_DEV double sqrt_(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = fma(-g, h, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  const double d = fma(-g, g, x);
  g = fma(d, h, g);
  return x == 0.0 ? x : g;
}
// 1 / x for the normal, finite divisors of the factorisations: in FP64 the
// hardware estimate (about 2^-24 relative) refined by two Newton steps, which
// on a million random normal values in 1e-30..1e30 gave the correctly rounded
// reciprocal every time, in five instructions instead of the IEEE division's
// special-case sequence; in FP32 the division, which the FP32 build already
// lowers to the hardware reciprocal.
PSM_DEV double rcp_(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(r, fma(-x, r, 1.0), r);
  r = fma(r, fma(-x, r, 1.0), r);
  return r;
}
PSM_DEV float rcp_(float x) { return 1.0f / x; }
PSM_DEV float sqrt_(float x) { return sqrtf(x); }
PSM_DEV double abs_(double x) { return fabs(x); }
PSM_DEV float abs_(float x) { return fabsf(x); }
PSM_DEV double log_(double x) { return log(x); }
PSM_DEV float log_(float x) { return logf(x); }

// ----------------------------------------------------------------------------
// basic products
// ----------------------------------------------------------------------------
template <typename R, int M, int K, int N>
PSM_DEV void mm(const R (&a)[M][K], const R (&b)[K][N], R (&c)[M][N]) {
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int j = 0; j < N; ++j) {
      R s = a[i][0] * b[0][j];
#pragma unroll
      for (int k = 1; k < K; ++k) s = fma(a[i][k], b[k][j], s);
      c[i][j] = s;
    }
}

// c = a * b^T
template <typename R, int M, int K, int N>
PSM_DEV void mmT(const R (&a)[M][K], const R (&b)[N][K], R (&c)[M][N]) {
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int j = 0; j < N; ++j) {
      R s = a[i][0] * b[j][0];
#pragma unroll
      for (int k = 1; k < K; ++k) s = fma(a[i][k], b[j][k], s);
      c[i][j] = s;
    }
}

template <typename R, int M, int N>
PSM_DEV void mv(const R (&a)[M][N], const R (&x)[N], R (&y)[M]) {
#pragma unroll
  for (int i = 0; i < M; ++i) {
    R s = a[i][0] * x[0];
#pragma unroll
    for (int k = 1; k < N; ++k) s = fma(a[i][k], x[k], s);
    y[i] = s;
  }
}

template <typename R, int M, int N>
PSM_DEV void set_zero(R (&a)[M][N]) {
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int j = 0; j < N; ++j) a[i][j] = R(0);
}

template <typename R, int N>
PSM_DEV void set_zero(R (&a)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) a[i] = R(0);
}

template <typename R, int N>
PSM_DEV void set_eye(R (&a)[N][N]) {
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j < N; ++j) a[i][j] = (i == j) ? R(1) : R(0);
}

template <typename R, int M, int N>
PSM_DEV void copy(const R (&a)[M][N], R (&b)[M][N]) {
#pragma unroll
  for (int i = 0; i < M; ++i)
#pragma unroll
    for (int j = 0; j < N; ++j) b[i][j] = a[i][j];
}

template <typename R, int N>
PSM_DEV void copy(const R (&a)[N], R (&b)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) b[i] = a[i];
}

// ----------------------------------------------------------------------------
// Householder pivots
// ----------------------------------------------------------------------------
// Reflecting the rows of a matrix from the right so that the pivot row x
// becomes (||x||, 0, ..., 0) maps another row m to
//     m_0' = p / ||x||,   m_j' = m_j - t x_j  (j > 0),   p = <x, m>,
//     t = (p / ||x|| + sgn(x_0) m_0) / (||x|| + |x_0|)
// (the reflector v = x + sgn(x_0) ||x|| e_0, which never cancels, with the
// first column's sign flipped where that gives -||x||).  p needs the pivot row
// only, so the inner products of every row run beside the chain that forms the
// norm, its reciprocal and 1 / (||x|| + |x_0|); a pivot then costs one square
// root and one reciprocal in sequence.  A pivot row without a norm (exactly
// zero, or below the range of its square) reflects nothing: f, gs and inv are
// zero and keep is one.  Applied to the pivot row itself the map gives
// (||x||, 0, ..., 0), so a kernel may update all rows alike.
template <typename R>
struct Pivot {
  R nrm;   // ||x||
  R inv;   // 1 / ||x||
  R f;     // 1 / (||x|| (||x|| + |x_0|))
  R gs;    // sgn(x_0) / (||x|| + |x_0|)
  R keep;  // 1 for a pivot row without a norm, else 0
};

// Tangent types, whose products are three instructions each and whose inner products
// formed early spill, take the reflector itself instead: with v_0 = x_0 +
// sgn(x_0) ||x||, v_j = x_j, the map is m - f <v, m> v, f = 1 / (||x|| (||x|| + |x_0|)),
// and the first column's sign: half the products beside the inner one, and one
// reciprocal (forward gradient of 256 x 4,096 steps, cubature, FP64: 250 ms, 340 with
// the map above; k_linearize_states 2.36 ms a pass, 4.42).
template <typename R>
struct Reflector {
  R nrm;
  R v0;
  R f;
  bool flip;
};
template <typename R>
using PivotOf = std::conditional_t<std::is_floating_point<R>::value, Pivot<R>, Reflector<R>>;

// Smallest ||x||^2 a pivot divides by: the products of its reciprocals stay finite.
template <typename R> PSM_DEV constexpr double pivot_min() { return 1e-290; }
template <> PSM_DEV constexpr double pivot_min<float>() { return 1.2e-38; }

// s = sqrt(x), r = 1 / s and g = 1 / (s + a) for a normal, positive x and a >= 0.
// FP64: the hardware reciprocal square root refined as in sqrt_; the reciprocal's
// hardware estimate is taken from the unrefined root, beside the refinement, and
// its two Newton steps use the refined sum.
PSM_DEV void pivot_scalars(double x, double a, double& s, double& r, double& g) {
  const double y = __builtin_amdgcn_rsq(x);
  double q = x * y, h = 0.5 * y;
  g = __builtin_amdgcn_rcp(q + a);
  const double e = fma(-q, h, 0.5);
  q = fma(q, e, q);
  h = fma(h, e, h);
  s = fma(fma(-q, q, x), h, q);
  r = h + h;
  r = fma(fma(-s, r, 1.0), r, r);
  const double d = s + a;
  g = fma(g, fma(-d, g, 1.0), g);
  g = fma(g, fma(-d, g, 1.0), g);
}
PSM_DEV void pivot_scalars(float x, float a, float& s, float& r, float& g) {
  s = sqrtf(x);
  r = __builtin_amdgcn_rsqf(x);
  g = rcp_(s + a);
}
// The pivot of a row with first entry x0 and squared norm n2.
template <typename R>
PSM_DEV PivotOf<R> make_pivot(R x0, R n2) {
  const bool ok = !(n2 <= R(pivot_min<R>()));  // NaN passes through the norm
  PivotOf<R> p;
  if constexpr (std::is_floating_point<R>::value) {
    R s, r, g;
    pivot_scalars(n2, abs_(x0), s, r, g);      // whatever they are of a row without a norm, they go unused
    r = ok ? r : R(0);
    g = ok ? g : R(0);
    p.nrm = ok ? s : abs_(x0);
    p.inv = r;
    p.f = r * g;
    p.gs = x0 < R(0) ? -g : g;
    p.keep = ok ? R(0) : R(1);
  } else {
    const R s = sqrt_(ok ? n2 : R(1));         // a tangent of the unused would not go unused
    const R a = abs_(x0);
    p.nrm = ok ? s : a;
    p.v0 = x0 < R(0) ? x0 - s : x0 + s;
    p.f = ok ? rcp_(fma(s, a, n2)) : R(0);
    p.flip = ok && !(x0 < R(0));
  }
  return p;
}

// Active columns of pivot i of a matrix [X | T] with NL columns on the left and,
// on the right, NT columns whose lower-triangular shape the pivots keep (row k
// holds columns NL..NL + k): columns i..NL - 1 and NL..NL + min(i, NT - 1).
// With NT = 0 it is a plain matrix.
template <int NL, int NT>
PSM_DEV constexpr bool pivot_column(int i, int j) {
  return (j >= i && j < NL) || (j >= NL && j - NL <= i && j - NL < NT);
}

// Squared norm of pivot row x at pivot i, in two chains.
template <int NL, int NT, typename R, int NC>
PSM_DEV R pivot_norm2(const R (&x)[NC], int i) {
  R a = x[i] * x[i], b = R(0);
  bool odd = true;
#pragma unroll
  for (int j = 0; j < NC; ++j)
    if (j != i && pivot_column<NL, NT>(i, j)) {
      if (odd) b = fma(x[j], x[j], b);
      else a = fma(x[j], x[j], a);
      odd = !odd;
    }
  return a + b;
}

// Row m reflected by pivot row x at pivot i.
template <int NL, int NT, typename R, int NC>
PSM_DEV void pivot_apply(const PivotOf<R>& pv, const R (&x)[NC], R (&m)[NC], int i) {
  R a, b = R(0);
  if constexpr (std::is_floating_point<R>::value) a = x[i] * m[i];
  else a = pv.v0 * m[i];
  bool odd = true;
#pragma unroll
  for (int j = 0; j < NC; ++j)
    if (j != i && pivot_column<NL, NT>(i, j)) {
      if (odd) b = fma(x[j], m[j], b);
      else a = fma(x[j], m[j], a);
      odd = !odd;
    }
  const R p = a + b;
  R t;
  if constexpr (std::is_floating_point<R>::value) {
    t = fma(pv.gs, m[i], p * pv.f);
    m[i] = fma(pv.keep, m[i], p * pv.inv);
  } else {
    t = pv.f * p;
    const R r = fma(-t, pv.v0, m[i]);
    m[i] = pv.flip ? -r : r;
  }
#pragma unroll
  for (int j = 0; j < NC; ++j)
    if (j != i && pivot_column<NL, NT>(i, j)) m[j] = fma(-t, x[j], m[j]);
}

// ----------------------------------------------------------------------------
// tria: in-place Householder triangularisation from the right.
// On exit M[:, :min(ROWS,COLS)] holds L (lower, non-negative diagonal) and the
// remaining columns are zero.
// ----------------------------------------------------------------------------
// The first NP pivots of [X | T] (columns as in pivot_column); the pivot rows
// are left reduced to their diagonal entry, the columns of later pivots and T
// keep what the reflections leave there.
template <int NL, int NT, int NP, typename R, int ROWS, int NC>
PSM_DEV void tria_pivots(R (&M)[ROWS][NC]) {
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const PivotOf<R> pv = make_pivot(M[i][i], pivot_norm2<NL, NT>(M[i], i));
#pragma unroll
    for (int k = i + 1; k < ROWS; ++k) pivot_apply<NL, NT>(pv, M[i], M[k], i);
    M[i][i] = pv.nrm;
#pragma unroll
    for (int j = 0; j < NC; ++j)
      if (j != i && pivot_column<NL, NT>(i, j)) M[i][j] = R(0);
  }
}

template <typename R, int ROWS, int COLS>
PSM_DEV void tria_inplace(R (&M)[ROWS][COLS]) {
  constexpr int NR = ROWS < COLS ? ROWS : COLS;
  tria_pivots<COLS, 0, NR>(M);
}

// tria of [X | T], X ROWS x NL with ROWS <= NL, T lower triangular.
template <int NL, typename R, int ROWS>
PSM_DEV void tria_lower_inplace(R (&M)[ROWS][NL + ROWS]) {
  tria_pivots<NL, ROWS, ROWS>(M);
}

// A lower-triangular square root of C C^T: C itself when it is lower
// triangular, else tria(C).  The recursions and the operators take lower
// triangular factors, and a caller's (the prior's, a filtered trajectory's,
// chol Q, which the extended linearization passes through) may be any square root.
template <typename R>
PSM_DEV bool nonzero_(R x) { return x != R(0); }
template <typename R, int N>
PSM_DEV void lower_factor(R (&C)[N][N]) {
  bool upper = false;
#pragma unroll
  for (int a = 0; a < N; ++a)
#pragma unroll
    for (int b = a + 1; b < N; ++b) upper = upper || nonzero_(C[a][b]);
  if (upper) tria_inplace<R, N, N>(C);
}

// L (ROWS x ROWS) = tria(M)
template <typename R, int ROWS, int COLS>
PSM_DEV void tria(R (&M)[ROWS][COLS], R (&L)[ROWS][ROWS]) {
  tria_inplace<R, ROWS, COLS>(M);
#pragma unroll
  for (int i = 0; i < ROWS; ++i)
#pragma unroll
    for (int j = 0; j < ROWS; ++j) L[i][j] = (j < COLS && j <= i) ? M[i][j] : R(0);
}

// ----------------------------------------------------------------------------
// triangular solves (L lower triangular, N x N)
// ----------------------------------------------------------------------------
// X = L^{-1} B
template <typename R, int N, int K>
PSM_DEV void solve_lower(const R (&L)[N][N], const R (&B)[N][K], R (&X)[N][K]) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const R inv = rcp_(L[i][i]);
#pragma unroll
    for (int c = 0; c < K; ++c) {
      R s = B[i][c];
#pragma unroll
      for (int j = 0; j < i; ++j) s = fma(-L[i][j], X[j][c], s);
      X[i][c] = s * inv;
    }
  }
}

// X = L^{-T} B
template <typename R, int N, int K>
PSM_DEV void solve_lower_T(const R (&L)[N][N], const R (&B)[N][K], R (&X)[N][K]) {
#pragma unroll
  for (int ii = 0; ii < N; ++ii) {
    const int i = N - 1 - ii;
    const R inv = rcp_(L[i][i]);
#pragma unroll
    for (int c = 0; c < K; ++c) {
      R s = B[i][c];
#pragma unroll
      for (int j = i + 1; j < N; ++j) s = fma(-L[j][i], X[j][c], s);
      X[i][c] = s * inv;
    }
  }
}

// x = L^{-1} b
template <typename R, int N>
PSM_DEV void solve_lower_v(const R (&L)[N][N], const R (&b)[N], R (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    R s = b[i];
#pragma unroll
    for (int j = 0; j < i; ++j) s = fma(-L[i][j], x[j], s);
    x[i] = s * rcp_(L[i][i]);
  }
}

// X = B L^{-1}   (B is M x N):  X L = B
template <typename R, int M, int N>
PSM_DEV void solve_right_lower(const R (&L)[N][N], const R (&B)[M][N], R (&X)[M][N]) {
#pragma unroll
  for (int jj = 0; jj < N; ++jj) {
    const int j = N - 1 - jj;
    const R inv = rcp_(L[j][j]);
#pragma unroll
    for (int r = 0; r < M; ++r) {
      R s = B[r][j];
#pragma unroll
      for (int k = j + 1; k < N; ++k) s = fma(-X[r][k], L[k][j], s);
      X[r][j] = s * inv;
    }
  }
}

// X = B L^{-T}   (B is M x N):  X L^T = B
template <typename R, int M, int N>
PSM_DEV void solve_right_lower_T(const R (&L)[N][N], const R (&B)[M][N], R (&X)[M][N]) {
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const R inv = rcp_(L[j][j]);
#pragma unroll
    for (int r = 0; r < M; ++r) {
      R s = B[r][j];
#pragma unroll
      for (int k = 0; k < j; ++k) s = fma(-X[r][k], L[j][k], s);
      X[r][j] = s * inv;
    }
  }
}

// ----------------------------------------------------------------------------
// general square solve with partial pivoting: X = A^{-1} B (covariance form)
// ----------------------------------------------------------------------------
template <typename R, int N, int K>
PSM_DEV void solve_general(R (&A)[N][N], R (&B)[N][K]) {
#pragma unroll
  for (int c = 0; c < N; ++c) {
    // pivot search among rows c..N-1 (swap by predicated selects: the row
    // indices stay compile-time constants so nothing leaves the registers)
#pragma unroll
    for (int r = c + 1; r < N; ++r) {
      const bool sw = abs_(A[r][c]) > abs_(A[c][c]);
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const R t = A[c][j];
        A[c][j] = sw ? A[r][j] : t;
        A[r][j] = sw ? t : A[r][j];
      }
#pragma unroll
      for (int j = 0; j < K; ++j) {
        const R t = B[c][j];
        B[c][j] = sw ? B[r][j] : t;
        B[r][j] = sw ? t : B[r][j];
      }
    }
    const R inv = rcp_(A[c][c]);
#pragma unroll
    for (int r = c + 1; r < N; ++r) {
      const R l = A[r][c] * inv;
#pragma unroll
      for (int j = c; j < N; ++j) A[r][j] = fma(-l, A[c][j], A[r][j]);
#pragma unroll
      for (int j = 0; j < K; ++j) B[r][j] = fma(-l, B[c][j], B[r][j]);
    }
  }
#pragma unroll
  for (int ii = 0; ii < N; ++ii) {
    const int i = N - 1 - ii;
    const R inv = rcp_(A[i][i]);
#pragma unroll
    for (int j = 0; j < K; ++j) {
      R s = B[i][j];
#pragma unroll
      for (int k = i + 1; k < N; ++k) s = fma(-A[i][k], B[k][j], s);
      B[i][j] = s * inv;
    }
  }
}

// Cholesky factorisation (lower) of a symmetric positive definite matrix.
template <typename R, int N>
PSM_DEV void cholesky(const R (&A)[N][N], R (&L)[N][N]) {
#pragma unroll
  for (int j = 0; j < N; ++j) {
    R s = A[j][j];
#pragma unroll
    for (int k = 0; k < j; ++k) s = fma(-L[j][k], L[j][k], s);
    const R d = sqrt_(s);
    L[j][j] = d;
    const R inv = rcp_(d);
#pragma unroll
    for (int i = j + 1; i < N; ++i) {
      R t = A[i][j];
#pragma unroll
      for (int k = 0; k < j; ++k) t = fma(-L[i][k], L[j][k], t);
      L[i][j] = t * inv;
    }
#pragma unroll
    for (int i = 0; i < j; ++i) L[i][j] = R(0);
  }
}

// Rank-one update / downdate of a lower factor: L L^T + mult v v^T.
// Column recurrence of parsmooth/_utils.py:39-81 (_cholesky_update): entries
// above the diagonal are dropped and non-finite entries are set to zero.
template <typename R, int N>
PSM_DEV void cholesky_update(R (&L)[N][N], const R (&v)[N], R mult) {
  R omega[N];
#pragma unroll
  for (int i = 0; i < N; ++i) omega[i] = v[i];
  R b = R(1);
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const R d = L[j][j];
    const R wj = omega[j];
    const R new_d = sqrt_(d * d + mult / b * wj * wj);
    const R gamma = d * d * b + mult * wj * wj;
    const R r = wj / d;
    const R s = mult * wj / gamma;
#pragma unroll
    for (int i = 0; i < N; ++i) omega[i] = fma(-r, L[i][j], omega[i]);
#pragma unroll
    for (int i = j + 1; i < N; ++i) L[i][j] = new_d * (L[i][j] / d + s * omega[i]);
    L[j][j] = new_d;
    b = b + mult * r * r;
  }
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const R x = L[i][j];
      L[i][j] = (j > i || !isfinite(x)) ? R(0) : x;
    }
}

}  // namespace psm

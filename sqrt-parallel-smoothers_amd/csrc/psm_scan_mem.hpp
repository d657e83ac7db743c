// Memory-operand forms of the filtering / smoothing operators used by the scan
// kernels.  Both operands are read straight from memory (LDS or global,
// struct-of-arrays) when needed and the result is written field by field as
// soon as it is final, so a lane never holds two aggregates plus the
// 2nx x 2nx triangularisation at once.  The output may alias the second
// operand: every field of e2 is read for the last time before the same field
// of the output is written.
#pragma once
#include "psm_core.hpp"

namespace psm {

template <typename R, int NX>
struct FView {
  using real_type = R;
  R* base;
  int64_t stride;
  int64_t idx;
  static constexpr int NXV = NX;
  static constexpr int QUNIT = 0;   // first field of the identity's unit matrix (A)
  static constexpr int QA = 0, QB = NX * NX, QU = NX * NX + NX, QE = 2 * NX * NX + NX,
                       QZ = 2 * NX * NX + 2 * NX, QF = 3 * NX * NX + 2 * NX;
  PSM_DEV R& at(int q) const { return base[(int64_t)q * stride + idx]; }
  PSM_DEV R& A(int i, int j) const { return at(QA + i * NX + j); }
  PSM_DEV R& b(int i) const { return at(QB + i); }
  PSM_DEV R& U(int i, int j) const { return at(QU + i * NX + j); }
  PSM_DEV R& eta(int i) const { return at(QE + i); }
  PSM_DEV R& Z(int i, int j) const { return at(QZ + i * NX + j); }
  PSM_DEV int flag() const { return (int)at(QF); }
  PSM_DEV void set_flag(int f) const { at(QF) = R(f); }
};

template <typename R, int NX>
struct SView {
  using real_type = R;
  R* base;
  int64_t stride;
  int64_t idx;
  static constexpr int NXV = NX;
  static constexpr int QUNIT = NX;  // first field of the identity's unit matrix (E)
  static constexpr int QG = 0, QE = NX, QD = NX + NX * NX, QF = NX + 2 * NX * NX;
  PSM_DEV R& at(int q) const { return base[(int64_t)q * stride + idx]; }
  PSM_DEV R& g(int i) const { return at(QG + i); }
  PSM_DEV R& E(int i, int j) const { return at(QE + i * NX + j); }
  PSM_DEV R& D(int i, int j) const { return at(QD + i * NX + j); }
  PSM_DEV int flag() const { return (int)at(QF); }
  PSM_DEV void set_flag(int f) const { at(QF) = R(f); }
};

template <typename V>
PSM_DEV void view_copy(const V& s, const V& d) {
  constexpr int NQ = V::QF + 1;
#pragma unroll
  for (int q = 0; q < NQ; ++q) d.at(q) = s.at(q);
}

template <typename R, int NX>
PSM_DEV void view_identity(const FView<R, NX>& d) {
#pragma unroll
  for (int q = 0; q < FView<R, NX>::QF; ++q) d.at(q) = R(0);
#pragma unroll
  for (int i = 0; i < NX; ++i) d.A(i, i) = R(1);
  d.set_flag(FLAG_IDENT);
}

template <typename R, int NX>
PSM_DEV void view_identity(const SView<R, NX>& d) {
#pragma unroll
  for (int q = 0; q < SView<R, NX>::QF; ++q) d.at(q) = R(0);
#pragma unroll
  for (int i = 0; i < NX; ++i) d.E(i, i) = R(1);
  d.set_flag(FLAG_IDENT);
}

// ---------------------------------------------------------------- square-root filter
// The rows of FilterArray (psm_core.hpp) one after the other: the reduced pivot
// rows stay in registers and every other row is read, reflected and used up.
template <typename R, int NX, typename C = R>
PSM_DEV void sqrt_combine_mem(const FView<R, NX>& e1, const FView<R, NX>& e2,
                              const FView<R, NX>& out) {
  FilterArray<C, NX> q;
  C w[NX], r[2 * NX], Vt[NX][NX];
  {
    C Z2[NX][NX];
#pragma unroll
    for (int k = 0; k < NX; ++k)
#pragma unroll
      for (int j = 0; j <= k; ++j) Z2[k][j] = (C)e2.Z(k, j);
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      C u[NX];
#pragma unroll
      for (int k = i; k < NX; ++k) u[k] = (C)e1.U(k, i);
#pragma unroll
      for (int j = 0; j < NX; ++j) {
        C acc = C(0);
#pragma unroll
        for (int k = (i > j ? i : j); k < NX; ++k) acc = fma(u[k], Z2[k][j], acc);
        q.x[i][j] = acc;
      }
    }
    q.reduce();
    C b1[NX], eta2[NX];
#pragma unroll
    for (int k = 0; k < NX; ++k) {
      b1[k] = (C)e1.b(k);
      eta2[k] = (C)e2.eta(k);
    }
    innovation(b1, eta2, Z2, w);
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      C acc = (C)e1.U(j, j) * w[j];
#pragma unroll
      for (int k = j + 1; k < NX; ++k) acc = fma((C)e1.U(k, j), w[k], acc);
      r[j] = C(0);
      r[NX + j] = acc;
    }
    q.reflect(r);
    // [A1^T Z2 | 0] -> [V^T | Y]: eta and Z = tria([Y | Z1])
    C Zc[NX][2 * NX], eta[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      C row[2 * NX], a1[NX];
      C h = (C)e1.eta(i);
#pragma unroll
      for (int k = 0; k < NX; ++k) {
        a1[k] = (C)e1.A(k, i);
        h = fma(a1[k], w[k], h);
      }
#pragma unroll
      for (int j = 0; j < NX; ++j) {
        C acc = a1[j] * Z2[j][j];
#pragma unroll
        for (int k = j + 1; k < NX; ++k) acc = fma(a1[k], Z2[k][j], acc);
        row[j] = acc;
        row[NX + j] = C(0);
      }
      q.reflect(row);
#pragma unroll
      for (int j = 0; j < NX; ++j) {
        Vt[i][j] = row[j];
        Zc[i][j] = row[NX + j];
        Zc[i][NX + j] = (C)e1.Z(i, j);
        h = fma(-row[j], r[j], h);
      }
      eta[i] = h;
    }
#pragma unroll
    for (int i = 0; i < NX; ++i) out.eta(i) = (R)eta[i];
    tria_lower_inplace<NX>(Zc);
#pragma unroll
    for (int i = 0; i < NX; ++i)
#pragma unroll
      for (int j = 0; j < NX; ++j) out.Z(i, j) = (R)(Zc[i][j]);
  }
  // [0 | A2 U1] -> [S | .]: A, b and U = tria([S | U2])
  C Uc[NX][2 * NX];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    C row[2 * NX], a2[NX];
    C bb = (C)e2.b(i);
#pragma unroll
    for (int k = 0; k < NX; ++k) {
      a2[k] = (C)e2.A(i, k);
      bb = fma(a2[k], (C)e1.b(k), bb);
    }
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      C acc = a2[j] * (C)e1.U(j, j);
#pragma unroll
      for (int k = j + 1; k < NX; ++k) acc = fma(a2[k], (C)e1.U(k, j), acc);
      row[j] = C(0);
      row[NX + j] = acc;
    }
    q.reflect(row);
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      C acc = C(0);
#pragma unroll
      for (int k = 0; k < NX; ++k) acc = fma(a2[k], (C)e1.A(k, j), acc);
#pragma unroll
      for (int k = 0; k < NX; ++k) acc = fma(-row[k], Vt[j][k], acc);
      out.A(i, j) = (R)acc;
      Uc[i][j] = row[j];
      Uc[i][NX + j] = (C)e2.U(i, j);
      bb = fma(row[j], r[j], bb);
    }
    out.b(i) = (R)bb;
  }
  tria_lower_inplace<NX>(Uc);
#pragma unroll
  for (int i = 0; i < NX; ++i)
#pragma unroll
    for (int j = 0; j < NX; ++j) out.U(i, j) = (R)(Uc[i][j]);
}

// ---------------------------------------------------------------- square-root smoother
// out = e1 (+) e2 with e1 the later aggregate: g = E2 g1 + g2, E = E2 E1,
// D = tria([E2 D1 | D2]).
template <typename R, int NX, typename C = R>
PSM_DEV void sqrt_smoother_combine_mem(const SView<R, NX>& e1, const SView<R, NX>& e2,
                                       const SView<R, NX>& out) {
  C E2[NX][NX];
#pragma unroll
  for (int i = 0; i < NX; ++i)
#pragma unroll
    for (int j = 0; j < NX; ++j) E2[i][j] = (C)e2.E(i, j);
  C M[NX][2 * NX];
#pragma unroll
  for (int i = 0; i < NX; ++i)
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      C acc = C(0);
#pragma unroll
      for (int k = j; k < NX; ++k) acc = fma(E2[i][k], (C)e1.D(k, j), acc);
      M[i][j] = acc;
      M[i][NX + j] = (C)e2.D(i, j);
    }
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    C g = (C)e2.g(i);
#pragma unroll
    for (int k = 0; k < NX; ++k) g = fma(E2[i][k], (C)e1.g(k), g);
    out.g(i) = (R)(g);
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      C acc = C(0);
#pragma unroll
      for (int k = 0; k < NX; ++k) acc = fma(E2[i][k], (C)e1.E(k, j), acc);
      out.E(i, j) = (R)(acc);
    }
  }
  tria_lower_inplace<NX>(M);
#pragma unroll
  for (int i = 0; i < NX; ++i)
#pragma unroll
    for (int j = 0; j < NX; ++j) out.D(i, j) = (R)(M[i][j]);
}

}  // namespace psm

namespace psm {

template <typename R, int NX>
PSM_DEV void view_load(const FView<R, NX>& v, FAgg<R, NX>& a) {
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    a.b[i] = v.b(i);
    a.eta[i] = v.eta(i);
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      a.A[i][j] = v.A(i, j);
      a.U[i][j] = v.U(i, j);
      a.Z[i][j] = v.Z(i, j);
    }
  }
  a.flag = v.flag();
}
template <typename R, int NX>
PSM_DEV void view_store(const FAgg<R, NX>& a, const FView<R, NX>& v) {
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    v.b(i) = a.b[i];
    v.eta(i) = a.eta[i];
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      v.A(i, j) = a.A[i][j];
      v.U(i, j) = a.U[i][j];
      v.Z(i, j) = a.Z[i][j];
    }
  }
  v.set_flag(a.flag);
}
template <typename R, int NX>
PSM_DEV void view_load(const SView<R, NX>& v, SAgg<R, NX>& a) {
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    a.g[i] = v.g(i);
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      a.E[i][j] = v.E(i, j);
      a.D[i][j] = v.D(i, j);
    }
  }
  a.flag = v.flag();
}
template <typename R, int NX>
PSM_DEV void view_store(const SAgg<R, NX>& a, const SView<R, NX>& v) {
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    v.g(i) = a.g[i];
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      v.E(i, j) = a.E[i][j];
      v.D(i, j) = a.D[i][j];
    }
  }
  v.set_flag(a.flag);
}

// out <- e1 (+) e2 with the HEAD / IDENT rules of combine_into; out may alias e2.
template <typename R, int NX, bool SQRT>
PSM_DEV void combine_mem(const FView<R, NX>& e1, const FView<R, NX>& e2, const FView<R, NX>& out) {
  const int f1 = e1.flag(), f2 = e2.flag();
  if (f2 == FLAG_HEAD || f1 == FLAG_IDENT) { view_copy(e2, out); return; }
  if (f2 == FLAG_IDENT) { view_copy(e1, out); return; }
  if constexpr (SQRT) {
    sqrt_combine_mem<R, NX>(e1, e2, out);
  } else {
    FAgg<R, NX> a, b;
    view_load(e1, a);
    view_load(e2, b);
    std_combine_core<R, NX>(a, b, b);
    view_store(b, out);
  }
  out.set_flag(f1);
}

template <typename R, int NX, bool SQRT>
PSM_DEV void combine_mem(const SView<R, NX>& e1, const SView<R, NX>& e2, const SView<R, NX>& out) {
  const int f1 = e1.flag(), f2 = e2.flag();
  if (f2 == FLAG_HEAD || f1 == FLAG_IDENT) { view_copy(e2, out); return; }
  if (f2 == FLAG_IDENT) { view_copy(e1, out); return; }
  if constexpr (SQRT) {
    sqrt_smoother_combine_mem<R, NX>(e1, e2, out);
  } else {
    SAgg<R, NX> a, b;
    view_load(e1, a);
    view_load(e2, b);
    std_smoother_combine_core<R, NX>(a, b);
    view_store(b, out);
  }
  out.set_flag(f1);
}

template <typename Agg> struct ViewOf;
template <typename R, int NX> struct ViewOf<FAgg<R, NX>> { using type = FView<R, NX>; };
template <typename R, int NX> struct ViewOf<SAgg<R, NX>> { using type = SView<R, NX>; };

}  // namespace psm

namespace psm {

template <typename R, int NX>
PSM_DEV bool view_ill(const FView<R, NX>& v, float thr) {
  R L[NX][NX];
#pragma unroll
  for (int i = 0; i < NX; ++i)
#pragma unroll
    for (int j = 0; j < NX; ++j) L[i][j] = (i == j) ? v.U(i, i) : R(0);
  return ill_conditioned(L, thr);
}
template <typename R, int NX>
PSM_DEV bool view_ill(const SView<R, NX>& v, float thr) {
  R L[NX][NX];
#pragma unroll
  for (int i = 0; i < NX; ++i)
#pragma unroll
    for (int j = 0; j < NX; ++j) L[i][j] = (i == j) ? v.D(i, i) : R(0);
  return ill_conditioned(L, thr);
}

// combine_mem with the FP64 re-triangularisation fallback (FP32 square-root
// form).  out must not alias e2 here, so the operands survive for the redo.
template <typename R, int NX, bool SQRT, typename V, typename FB>
PSM_DEV void combine_mem_fb(const V& e1, const V& e2, const V& out, const FB& fb) {
  const int f1 = e1.flag(), f2 = e2.flag();
  combine_mem<R, NX, SQRT>(e1, e2, out);
  if constexpr (kFallback<R, SQRT> && !FB::kRedo) {
    if (fb.thr > 0.f && f2 != FLAG_HEAD && f1 != FLAG_IDENT && f2 != FLAG_IDENT && view_ill(out, fb.thr))
      fb.raise();
  } else if constexpr (kFallback<R, SQRT>) {
    if (fb.thr > 0.f && f2 != FLAG_HEAD && f1 != FLAG_IDENT && f2 != FLAG_IDENT &&
        view_ill(out, fb.thr)) {
      // the memory-operand operator in FP64 on the FP32 operands: no aggregate
      // is ever whole in registers
      if constexpr (std::is_same<V, FView<R, NX>>::value)
        sqrt_combine_mem<R, NX, double>(e1, e2, out);
      else
        sqrt_smoother_combine_mem<R, NX, double>(e1, e2, out);
      count_fallback(fb);
    }
  }
}

// The distribution a HEAD aggregate is: (b, U) of a filter's, (g, D) of a smoother's.
template <typename R, int NX>
PSM_DEV void view_head(const FView<R, NX>& v, R (&m)[NX], R (&L)[NX][NX]) {
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    m[i] = v.b(i);
#pragma unroll
    for (int j = 0; j < NX; ++j) L[i][j] = v.U(i, j);
  }
}
template <typename R, int NX>
PSM_DEV void view_head(const SView<R, NX>& v, R (&m)[NX], R (&L)[NX][NX]) {
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    m[i] = v.g(i);
#pragma unroll
    for (int j = 0; j < NX; ++j) L[i][j] = v.D(i, j);
  }
}

// (m, L) (+) e2: the filtering operator with a distribution on the left (A1, eta1
// and Z1 are zero), of which only b and U are left to form (see FilterArray).
template <typename R, int NX, typename C>
PSM_DEV void sqrt_filter_push(const FView<R, NX>& e2, C (&m)[NX], C (&L)[NX][NX]) {
  FilterArray<C, NX> q;
  C r[2 * NX];
  {
    C Z2[NX][NX];
#pragma unroll
    for (int k = 0; k < NX; ++k)
#pragma unroll
      for (int j = 0; j <= k; ++j) Z2[k][j] = (C)e2.Z(k, j);
#pragma unroll
    for (int i = 0; i < NX; ++i)
#pragma unroll
      for (int j = 0; j < NX; ++j) {
        C acc = C(0);
#pragma unroll
        for (int k = (i > j ? i : j); k < NX; ++k) acc = fma(L[k][i], Z2[k][j], acc);
        q.x[i][j] = acc;
      }
    C eta2[NX], w[NX];
#pragma unroll
    for (int k = 0; k < NX; ++k) eta2[k] = (C)e2.eta(k);
    innovation(m, eta2, Z2, w);
    innovation_row(L, w, r);
  }
  q.reduce();
  q.reflect(r);
  C Uc[NX][2 * NX], b[NX];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    C row[2 * NX], a2[NX];
    C bb = (C)e2.b(i);
#pragma unroll
    for (int k = 0; k < NX; ++k) {
      a2[k] = (C)e2.A(i, k);
      bb = fma(a2[k], m[k], bb);
    }
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      C acc = a2[j] * L[j][j];
#pragma unroll
      for (int k = j + 1; k < NX; ++k) acc = fma(a2[k], L[k][j], acc);
      row[j] = C(0);
      row[NX + j] = acc;
    }
    q.reflect(row);
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      Uc[i][j] = row[j];
      Uc[i][NX + j] = (C)e2.U(i, j);
      bb = fma(row[j], r[j], bb);
    }
    b[i] = bb;
  }
  tria_lower_inplace<NX>(Uc);
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    m[i] = b[i];
#pragma unroll
    for (int j = 0; j < NX; ++j) L[i][j] = Uc[i][j];
  }
}

// The same for the covariance form: with N = I + J2 P, w = eta2 - J2 m and
// [X1^T | y] = N^-1 [A2^T | w],  m' = A2 (m + P y) + b2 and P' = X1 (P A2^T) + C2.
template <typename R, int NX>
PSM_DEV void std_filter_push(const FView<R, NX>& e2, R (&m)[NX], R (&P)[NX][NX]) {
  R N[NX][NX], B[NX][NX + 1];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    R jm = e2.Z(i, 0) * m[0];
#pragma unroll
    for (int k = 1; k < NX; ++k) jm = fma(e2.Z(i, k), m[k], jm);
    B[i][NX] = e2.eta(i) - jm;
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      R s1 = (i == j) ? R(1) : R(0);
#pragma unroll
      for (int k = 0; k < NX; ++k) s1 = fma(P[j][k], e2.Z(k, i), s1);   // (I + P J2)^T
      N[i][j] = s1;
      B[i][j] = e2.A(j, i);
    }
  }
  solve_general<R, NX, NX + 1>(N, B);
  R v[NX], CA[NX][NX];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    R a = P[i][0] * B[0][NX];
#pragma unroll
    for (int k = 1; k < NX; ++k) a = fma(P[i][k], B[k][NX], a);
    v[i] = m[i] + a;
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      R c = P[i][0] * e2.A(j, 0);
#pragma unroll
      for (int k = 1; k < NX; ++k) c = fma(P[i][k], e2.A(j, k), c);
      CA[i][j] = c;                    // P A2^T
    }
  }
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    R b = e2.A(i, 0) * v[0];
#pragma unroll
    for (int k = 1; k < NX; ++k) b = fma(e2.A(i, k), v[k], b);
    m[i] = b + e2.b(i);
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      R c = B[0][i] * CA[0][j];
#pragma unroll
      for (int k = 1; k < NX; ++k) c = fma(B[k][i], CA[k][j], c);
      P[i][j] = c + e2.U(i, j);
    }
  }
}

// (m, L) <- aggregate v applied to (m, L), with the FP64 recomputation of an
// ill-conditioned FP32 factor.
template <typename R, int NX, bool SQRT, typename FB>
PSM_DEV void filter_push_fb(const FView<R, NX>& v, R (&m)[NX], R (&L)[NX][NX], const FB& fb) {
  if constexpr (!SQRT) {
    std_filter_push<R, NX>(v, m, L);
  } else if constexpr (kFallback<R, SQRT> && !FB::kRedo) {
    sqrt_filter_push<R, NX, R>(v, m, L);
    if (fb.thr > 0.f && ill_conditioned(L, fb.thr)) fb.raise();
  } else if constexpr (kFallback<R, SQRT>) {
    R m0[NX], L0[NX][NX];
    copy(m, m0);
    copy(L, L0);
    sqrt_filter_push<R, NX, R>(v, m, L);
    if (fb.thr > 0.f && ill_conditioned(L, fb.thr)) {
      double md[NX], Ld[NX][NX];
      cvt(m0, md);
      cvt(L0, Ld);
      sqrt_filter_push<R, NX, double>(v, md, Ld);
      cvt(md, m);
      cvt(Ld, L);
      count_fallback(fb);
    }
  } else {
    sqrt_filter_push<R, NX, R>(v, m, L);
  }
}

}  // namespace psm

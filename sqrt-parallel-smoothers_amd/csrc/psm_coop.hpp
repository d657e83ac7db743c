// Cooperative scan operators: G lanes run one combination.
//
// One lane running a whole combination issues a chain of thousands of dependent
// instructions, and a scan level seldom has enough items to hide it.  Here a
// group of G lanes of one wavefront -- a DPP quad (G = 4) or a DPP row
// (G = 16) -- runs one combination.  Each lane holds whole rows of the array
// being reduced (FilterArray in psm_core.hpp); a pivot row is broadcast inside
// the group with DPP moves (no LDS round trip) and every lane reflects its own
// rows, so a pivot costs its broadcast, one square root and one reciprocal
// whatever the number of rows.  (The covariance form is dealt out by columns: see
// its operators below.)
//
// The 3 n + 1 rows of the filtering array are dealt out so that the n rows that
// become Z lie on the low half of the group and the n rows that become U on the
// high half, row i in slot i / (G / 2): the two closing triangularisations then
// run side by side, each half broadcasting its own pivot row.  The n pivot rows
// and the innovation's row fill the places left over in the last of these slots and then
// further slots.  For n = 5 the 16 rows fill four slots of a quad, or one row per
// lane of a DPP row, without a gap.  No update is masked: a pivot row that is
// done is never read again, an update of the pivot row with itself leaves its
// norm on the diagonal, and what the later pivots leave right of a finished
// row's diagonal is not read.
//
// Operands and results are arrays of fields in LDS, one contiguous item per
// group, at an odd number of words so that the groups of a wavefront fall on
// different banks.  A result stays in registers until its group may overwrite an
// operand, so a scan needs one buffer.  Groups of one wavefront may take
// different paths (combine / copy): no broadcast leaves its group.
#pragma once
#include <cstdint>
#include <type_traits>

#include "psm_scan_mem.hpp"

namespace psm {

template <int I, int N, typename F>
PSM_DEV void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

// Orders LDS accesses of the lanes of one wavefront.
PSM_DEV void group_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Keeps the scheduler from moving instructions across a phase of a combination by
// a quad: it would otherwise hoist the operand loads of later phases far ahead and
// hold them in more registers than two wavefronts per SIMD have.  With one or two
// rows a lane there is room, and the phases overlap.
template <int G>
PSM_DEV void phase() {
  if constexpr (G == 4) __builtin_amdgcn_sched_barrier(0);
}
// Forms x here: results that only some lanes store would otherwise be sunk into
// that branch, behind the closing triangularisations, their operands live until then.
template <typename R>
PSM_DEV void form_now(R& x) {
  asm volatile("" : "+v"(x));
}

// ---------------------------------------------------------------- broadcasts
constexpr int kDppRowNewBcast = 0x150;   // row_newbcast:L is kDppRowNewBcast + L

// The 64-bit form of __builtin_amdgcn_update_dpp (the builtin is declared on int).
extern "C" __device__ long psm_update_dpp_i64(long old, long src, int ctrl, int row_mask, int bank_mask,
                                              bool bound_ctrl) __asm("llvm.amdgcn.update.dpp.i64");

template <int CTRL>
PSM_DEV float dpp(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
template <int CTRL>
PSM_DEV double dpp(double v) {
  if constexpr (CTRL >= kDppRowNewBcast) {  // the one control 64-bit moves have
    return __builtin_bit_cast(double, psm_update_dpp_i64(0, __builtin_bit_cast(long, v), CTRL, 0xF, 0xF, true));
  } else {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xF, 0xF, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xF, 0xF, true);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
  }
}
// `old` with lanes 8..15 of every DPP row (banks 2 and 3) replaced by v moved by CTRL
template <int CTRL>
PSM_DEV float dpp_high(float old, float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
      __builtin_bit_cast(int, old), __builtin_bit_cast(int, v), CTRL, 0xF, 0xC, false));
}
template <int CTRL>
PSM_DEV double dpp_high(double old, double v) {
  return __builtin_bit_cast(double, psm_update_dpp_i64(__builtin_bit_cast(long, old), __builtin_bit_cast(long, v),
                                                       CTRL, 0xF, 0xC, false));
}

// Value of lane L of this lane's group.
template <int G, int L, typename C>
PSM_DEV C from_lane(C v) {
  static_assert((G == 4 || G == 16) && L >= 0 && L < G, "group lane");
  if constexpr (G == 4) return dpp<L * 0x55>(v);
  else return dpp<kDppRowNewBcast + L>(v);
}
// Value of lane LO on the low half of the group, of lane HI on the high half.
template <int G, int LO, int HI, typename C>
PSM_DEV C from_lanes(C v) {
  static_assert(LO < G / 2 && HI >= G / 2 && HI < G, "one lane per half");
  if constexpr (G == 4) return dpp<LO * 0x05 + HI * 0x50>(v);
  else return dpp_high<kDppRowNewBcast + HI>(dpp<kDppRowNewBcast + LO>(v), v);
}

// ---------------------------------------------------------------- items
constexpr int odd_words(int n) { return n | 1; }

// The fields of one item dealt out over the lanes of a group, on their way
// between HBM (struct-of-arrays, FView / SView) and LDS: all loads are in flight
// before the first store waits for one.
template <typename V, int G>
struct ItemRegs {
  using R = typename V::real_type;
  static constexpr int NQ = V::QF + 1;
  static constexpr int N = (NQ + G - 1) / G;
  R v[N];
  PSM_DEV void load(const V& s, int r) {
#pragma unroll
    for (int c = 0; c < N; ++c)
      if ((c + 1) * G <= NQ || c * G + r < NQ) v[c] = s.at(c * G + r);
  }
  PSM_DEV void load(const R* s, int r) {
#pragma unroll
    for (int c = 0; c < N; ++c)
      if ((c + 1) * G <= NQ || c * G + r < NQ) v[c] = s[c * G + r];
  }
  PSM_DEV void store(R* d, int r) const {
#pragma unroll
    for (int c = 0; c < N; ++c)
      if ((c + 1) * G <= NQ || c * G + r < NQ) d[c * G + r] = v[c];
  }
  PSM_DEV void store(const V& d, int r) const {
#pragma unroll
    for (int c = 0; c < N; ++c)
      if ((c + 1) * G <= NQ || c * G + r < NQ) d.at(c * G + r) = v[c];
  }
  // the identity: QI is the first field of its unit matrix
  PSM_DEV void identity(int r) {
    constexpr int NX = V::NXV, QI = V::QUNIT;
#pragma unroll
    for (int c = 0; c < N; ++c) {
      const int q = c * G + r;
      const int e = q - QI;
      v[c] = (e >= 0 && e < NX * NX && e / NX == e % NX) ? R(1) : R(0);
      if (q == V::QF) v[c] = R(FLAG_IDENT);
    }
  }
};

// ---------------------------------------------------------------- filtering
enum { ROW_Z = 0, ROW_U = 1, ROW_P = 2, ROW_R = 3, ROW_NONE = 4 };

// Where the rows of the filtering array lie: ROW_Z rows [A1^T Z2 | 0], ROW_U rows
// [0 | A2 U1], ROW_P the pivot rows [W | I], ROW_R the row [0 | w^T U1].
template <int NX, int G>
struct FilterRows {
  static constexpr int HL = G / 2;                      // lanes per half
  static constexpr int ZS = (NX + HL - 1) / HL;         // slots of the Z and U rows
  static constexpr int LAST = NX - (ZS - 1) * HL;       // rows per half in the last of them
  static constexpr int H = HL - LAST;                   // places left in it, per half
  static constexpr int NH = 2 * H < NX + 1 ? 2 * H : NX + 1;  // r and the last pivot rows placed there
  static constexpr int M = NX - (NH > 0 ? NH - 1 : 0);  // pivot rows 0..M-1 in further slots
  static constexpr int REST = M + (NH > 0 ? 0 : 1);
  static constexpr int NS = ZS + (REST + G - 1) / G;

  static constexpr int hole(int q) { return q < H ? LAST + q : HL + LAST + (q - H); }
  static constexpr int pslot(int i) { return i >= M ? ZS - 1 : ZS + i / G; }
  static constexpr int plane(int i) { return i >= M ? hole(NX - i) : i % G; }
  static constexpr int rslot() { return NH > 0 ? ZS - 1 : ZS + M / G; }
  static constexpr int rlane() { return NH > 0 ? hole(0) : M % G; }
  static constexpr int kind(int s, int l) {
    if (s == rslot() && l == rlane()) return ROW_R;
    for (int i = 0; i < NX; ++i)
      if (s == pslot(i) && l == plane(i)) return ROW_P;
    const int row = s * HL + l % HL;
    return s < ZS && row < NX ? (l < HL ? ROW_Z : ROW_U) : ROW_NONE;
  }
  static constexpr int index(int s, int l) {
    for (int i = 0; i < NX; ++i)
      if (s == pslot(i) && l == plane(i)) return i;
    const int row = s * HL + l % HL;
    return s < ZS && row < NX ? row : 0;
  }
  // four bits per lane
  static constexpr uint64_t kinds(int s) {
    uint64_t w = 0;
    for (int l = 0; l < G; ++l) w |= (uint64_t)kind(s, l) << (4 * l);
    return w;
  }
  static constexpr uint64_t indices(int s) {
    uint64_t w = 0;
    for (int l = 0; l < G; ++l) w |= (uint64_t)index(s, l) << (4 * l);
    return w;
  }
  // whether slot s holds rows that pivot i still has to reflect
  static constexpr bool live(int s, int i) {
    for (int l = 0; l < G; ++l) {
      const int k = kind(s, l);
      if (k == ROW_Z || k == ROW_U || k == ROW_R || (k == ROW_P && index(s, l) > i)) return true;
    }
    return false;
  }
  static constexpr bool has(int s, int k) {
    for (int l = 0; l < G; ++l)
      if (kind(s, l) == k) return true;
    return false;
  }
};

// The lane's part of a combination's result, held in registers until the group
// may overwrite an operand.
template <typename V, int G, bool SQRT = true> struct CoopResult;

template <typename R, int NX, int G>
struct CoopResult<FView<R, NX>, G, true> {
  using V = FView<R, NX>;
  using L = FilterRows<NX, G>;
  static constexpr int n = NX, NS = L::NS, ZS = L::ZS, HL = L::HL;
  R f[ZS][n];   // rows of Z (low half) or U (high half)
  R A[ZS][n];   // rows of A (high half)
  R h[ZS];      // entries of eta (low half) or b (high half)

  PSM_DEV void write(R* out, int flag, int r) const {
    const bool high = r >= HL;
    static_for<0, ZS>([&](auto sc) {
      constexpr int s = decltype(sc)::value;
      const int i = s * HL + (high ? r - HL : r);
      if (s + 1 < ZS || i < n) {
        R* op = out + (high ? V::QU : V::QZ) + i * n;
        out[(high ? V::QB : V::QE) + i] = h[s];
#pragma unroll
        for (int j = 0; j < n; ++j) op[j] = f[s][j];
        if (high) {
#pragma unroll
          for (int j = 0; j < n; ++j) out[V::QA + i * n + j] = A[s][j];
        }
      }
    });
    if (r == 0) out[V::QF] = R(flag);
  }

  // e1 (+) e2 (e1 earlier) from fields in LDS, computed in C.  Returns (when ILL)
  // whether U is ill-conditioned at thr, on every lane.
  template <typename C, bool ILL>
  PSM_DEV bool compute(const R* e1, const R* e2, int r, float thr);
};

template <typename R, int NX, int G>
template <typename C, bool ILL>
PSM_DEV bool CoopResult<FView<R, NX>, G, true>::compute(const R* e1, const R* e2, int r, float thr) {
  const bool high = r >= HL;

  // w = eta2 - Z2 (Z2^T b1) and w^T U1, on every lane
  C w[n], wu[n];
  {
    C t[n];
#pragma unroll
    for (int j = 0; j < n; ++j) {
      t[j] = (C)e2[V::QZ + j * n + j] * (C)e1[V::QB + j];
#pragma unroll
      for (int k = j + 1; k < n; ++k) t[j] = fma((C)e2[V::QZ + k * n + j], (C)e1[V::QB + k], t[j]);
    }
#pragma unroll
    for (int i = 0; i < n; ++i) {
      w[i] = (C)e2[V::QE + i];
#pragma unroll
      for (int k = 0; k <= i; ++k) w[i] = fma(-(C)e2[V::QZ + i * n + k], t[k], w[i]);
    }
#pragma unroll
    for (int j = 0; j < n; ++j) {
      wu[j] = (C)e1[V::QU + j * n + j] * w[j];
#pragma unroll
      for (int k = j + 1; k < n; ++k) wu[j] = fma((C)e1[V::QU + k * n + j], w[k], wu[j]);
    }
  }
  phase<G>();

  // rows of the array: a row of coefficients times the lower triangular Z2 or U1
  C x[NS][2 * n], a[ZS][n];
  static_for<0, NS>([&](auto sc) {
    constexpr int s = decltype(sc)::value;
    const int kind = (int)((L::kinds(s) >> (4 * r)) & 15), i = (int)((L::indices(s) >> (4 * r)) & 15);
    const R* ap = e1 + V::QU + i;          // P: column i of U1
    int step = n;
    const R* mp = e2 + V::QZ;
    if constexpr (L::has(s, ROW_Z)) ap = kind == ROW_Z ? e1 + V::QA + i : ap;
    if constexpr (L::has(s, ROW_U)) {
      ap = kind == ROW_U ? e2 + V::QA + i * n : ap;
      step = kind == ROW_U ? 1 : step;
      mp = kind == ROW_U ? e1 + V::QU : mp;
    }
    C c[n];
#pragma unroll
    for (int k = 0; k < n; ++k) c[k] = (C)ap[k * step];
    if constexpr (s < ZS) {
#pragma unroll
      for (int k = 0; k < n; ++k) a[s][k] = c[k];
    }
#pragma unroll
    for (int j = 0; j < n; ++j) {
      C acc = c[j] * (C)mp[j * n + j];
#pragma unroll
      for (int k = j + 1; k < n; ++k) acc = fma(c[k], (C)mp[k * n + j], acc);
      x[s][j] = acc;
      x[s][n + j] = C(0);
    }
    if constexpr (L::has(s, ROW_U)) {
#pragma unroll
      for (int j = 0; j < n; ++j) {
        x[s][n + j] = kind == ROW_U ? x[s][j] : C(0);
        x[s][j] = kind == ROW_U ? C(0) : x[s][j];
      }
    }
    if constexpr (L::has(s, ROW_P)) {
#pragma unroll
      for (int j = 0; j < n; ++j) x[s][n + j] = (kind == ROW_P && i == j) ? C(1) : x[s][n + j];
    }
    if constexpr (L::has(s, ROW_R)) {
#pragma unroll
      for (int j = 0; j < n; ++j) {
        x[s][j] = kind == ROW_R ? C(0) : x[s][j];
        x[s][n + j] = kind == ROW_R ? wu[j] : x[s][n + j];
      }
    }
    phase<G>();
  });

  static_for<0, n>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    C bx[2 * n];
    static_for<0, 2 * n>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if constexpr (pivot_column<n, n>(i, j)) bx[j] = from_lane<G, L::plane(i)>(x[L::pslot(i)][j]);
      else bx[j] = C(0);
    });
    const Pivot<C> pv = make_pivot(bx[i], pivot_norm2<n, n>(bx, i));
    static_for<0, NS>([&](auto sc) {
      constexpr int s = decltype(sc)::value;
      if constexpr (L::live(s, i)) pivot_apply<n, n>(pv, bx, x[s], i);
    });
  });
  phase<G>();

  // A = A2 A1 - S V on the lanes of the U rows (computed on all)
  static_for<0, n>([&](auto jc) {
    constexpr int j = decltype(jc)::value;
    C a1[n], vt[n];
#pragma unroll
    for (int k = 0; k < n; ++k) {
      a1[k] = (C)e1[V::QA + k * n + j];
      vt[k] = from_lane<G, j % HL>(x[j / HL][k]);
    }
    static_for<0, ZS>([&](auto sc) {
      constexpr int s = decltype(sc)::value;
      C p = a[s][0] * a1[0], q = x[s][0] * vt[0];
#pragma unroll
      for (int k = 1; k < n; ++k) {
        p = fma(a[s][k], a1[k], p);
        q = fma(x[s][k], vt[k], q);
      }
      A[s][j] = (R)(p - q);
      form_now(A[s][j]);
    });
    phase<G>();
  });

  // eta = A1^T w + eta1 - V^T r on the low half, b = A2 b1 + b2 + S r on the high one
  C y[ZS][2 * n];
  {
    const R* bp = high ? e2 + V::QB : e1 + V::QE;
    const R* tp = high ? e2 + V::QU : e1 + V::QZ;
    C vec[n], rr[n];
#pragma unroll
    for (int k = 0; k < n; ++k) {
      const C b1 = (C)e1[V::QB + k];
      const C rk = from_lane<G, L::rlane()>(x[L::rslot()][k]);
      vec[k] = high ? b1 : w[k];
      rr[k] = high ? rk : -rk;
    }
    static_for<0, ZS>([&](auto sc) {
      constexpr int s = decltype(sc)::value;
      const int row = s * HL + (high ? r - HL : r);
      const int i = s + 1 < ZS || row < n ? row : 0;
      C hh = (C)bp[i];
#pragma unroll
      for (int k = 0; k < n; ++k) {
        hh = fma(a[s][k], vec[k], hh);
        hh = fma(x[s][k], rr[k], hh);
        y[s][k] = high ? x[s][k] : x[s][n + k];
        y[s][n + k] = (C)tp[i * n + k];
      }
      h[s] = (R)hh;
      form_now(h[s]);
    });
  }
  phase<G>();

  // Z = tria([Y | Z1]) and U = tria([S | U2]), side by side
  C mn = C(0), mx = C(0);
  static_for<0, n>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    C bx[2 * n];
    static_for<0, 2 * n>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if constexpr (pivot_column<n, n>(i, j)) bx[j] = from_lanes<G, i % HL, HL + i % HL>(y[i / HL][j]);
      else bx[j] = C(0);
    });
    const Pivot<C> pv = make_pivot(bx[i], pivot_norm2<n, n>(bx, i));
    mn = (i == 0 || pv.nrm < mn) ? pv.nrm : mn;
    mx = (i == 0 || pv.nrm > mx) ? pv.nrm : mx;
    static_for<i / HL, ZS>([&](auto sc) {
      constexpr int s = decltype(sc)::value;
      pivot_apply<n, n>(pv, bx, y[s], i);
    });
  });
  static_for<0, ZS>([&](auto sc) {
    constexpr int s = decltype(sc)::value;
    const int i = s * HL + (high ? r - HL : r);
#pragma unroll
    for (int j = 0; j < n; ++j) f[s][j] = (j <= i) ? (R)y[s][j] : R(0);
  });
  if constexpr (ILL) {
    // the ratio of U, which the high half has
    const float bad = !(mn >= C(thr) * mx) ? 1.f : 0.f;
    return from_lane<G, HL>(bad) != 0.f;
  }
  return false;
}

// ---------------------------------------------------------------- smoothing
// out = e1 (+) e2 with e1 the later aggregate (parsmooth/parallel/_operators.py:104-125):
// g = E2 g1 + g2, E = E2 E1, D = tria([E2 D1 | D2]).  In a DPP row the low half
// forms the rows of D and the high half those of E; in a quad every lane forms
// both of its rows.
template <typename R, int NX, int G>
struct CoopResult<SView<R, NX>, G, true> {
  using V = SView<R, NX>;
  static constexpr int n = NX;
  static constexpr bool SPLIT = G >= 2 * NX;
  static constexpr int RL = SPLIT ? G / 2 : G;      // lanes that hold rows of D
  static constexpr int NS = (n + RL - 1) / RL;
  R f[NS][n];   // rows of D; of E on the high half of a split group
  R E[NS][n];   // rows of E of a group that is not split
  R g[NS];

  PSM_DEV void write(R* out, int flag, int r) const {
    const bool high = SPLIT && r >= RL;
    const int rr = high ? r - RL : r;
    static_for<0, NS>([&](auto sc) {
      constexpr int s = decltype(sc)::value;
      const int i = s * RL + rr;
      if (i < n) {
        R* op = out + (high ? V::QE : V::QD) + i * n;
        out[V::QG + i] = g[s];   // the halves of a split group store the same value
#pragma unroll
        for (int j = 0; j < n; ++j) op[j] = f[s][j];
        if constexpr (!SPLIT) {
#pragma unroll
          for (int j = 0; j < n; ++j) out[V::QE + i * n + j] = E[s][j];
        }
      }
    });
    if (r == 0) out[V::QF] = R(flag);
  }

  template <typename C, bool ILL>
  PSM_DEV bool compute(const R* e1, const R* e2, int r, float thr);
};

template <typename R, int NX, int G>
template <typename C, bool ILL>
PSM_DEV bool CoopResult<SView<R, NX>, G, true>::compute(const R* e1, const R* e2, int r, float thr) {
  const bool high = SPLIT && r >= RL;
  const int rr = high ? r - RL : r;
  C y[NS][2 * n];
  const R* mp = e1 + (high ? V::QE : V::QD);
  static_for<0, NS>([&](auto sc) {
    constexpr int s = decltype(sc)::value;
    const int row = s * RL + rr;
    const int i = row < n ? row : 0;
    C a[n];
    C gg = (C)e2[V::QG + i];
#pragma unroll
    for (int k = 0; k < n; ++k) {
      a[k] = (C)e2[V::QE + i * n + k];
      gg = fma(a[k], (C)e1[V::QG + k], gg);
    }
    g[s] = (R)gg;
    form_now(g[s]);
#pragma unroll
    for (int j = 0; j < n; ++j) {
      // a split group's halves read D1 or E1 with one set of instructions
      C acc = C(0);
#pragma unroll
      for (int k = SPLIT ? 0 : j; k < n; ++k) acc = fma(a[k], (C)mp[k * n + j], acc);
      y[s][j] = acc;
      y[s][n + j] = (C)e2[V::QD + i * n + j];
    }
#pragma unroll
    for (int j = 0; j < n; ++j) {
      if constexpr (SPLIT) {
        E[s][j] = (R)y[s][j];
      } else {
        C acc = a[0] * (C)e1[V::QE + j];
#pragma unroll
        for (int k = 1; k < n; ++k) acc = fma(a[k], (C)e1[V::QE + k * n + j], acc);
        E[s][j] = (R)acc;
      }
      form_now(E[s][j]);
    }
  });
  phase<G>();
  C mn = C(0), mx = C(0);
  static_for<0, n>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
    C bx[2 * n];
    static_for<0, 2 * n>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      if constexpr (pivot_column<n, n>(i, j)) bx[j] = from_lane<G, i % RL>(y[i / RL][j]);
      else bx[j] = C(0);
    });
    const Pivot<C> pv = make_pivot(bx[i], pivot_norm2<n, n>(bx, i));
    mn = (i == 0 || pv.nrm < mn) ? pv.nrm : mn;
    mx = (i == 0 || pv.nrm > mx) ? pv.nrm : mx;
    static_for<i / RL, NS>([&](auto sc) {
      constexpr int s = decltype(sc)::value;
      pivot_apply<n, n>(pv, bx, y[s], i);
    });
  });
  static_for<0, NS>([&](auto sc) {
    constexpr int s = decltype(sc)::value;
    const int i = s * RL + rr;
#pragma unroll
    for (int j = 0; j < n; ++j) f[s][j] = high ? E[s][j] : (j <= i) ? (R)y[s][j] : R(0);
  });
  if constexpr (ILL) return !(mn >= C(thr) * mx);
  return false;
}

// ---------------------------------------------------------------- covariance form
// e1 (+) e2 of (A, b, C, eta, J) (parsmooth/parallel/_operators.py:22-44), C and J
// symmetric.  With N = I + J2 C1 and w = eta2 - J2 b1 one elimination gives
//   X1^T = N^-1 A2^T,  Y = N^-1 J2 A1,  y = N^-1 w
// and the same two products with C1 and A2 all of
//   C = (A2 C1 X1^T)^T + C2,  A = A2 (A1 - C1 Y),  b = A2 (b1 + C1 y) + b2,
// and the one with A1^T  J = A1^T Y + J1,  eta = A1^T y + eta1.
// (A and b so, as what they are without the second aggregate's information and a
// correction, round less than by way of X1 A1 and X1 (b1 + C1 eta2).)
// Every lane holds columns of [N | A2^T | J2 A1 | w] (3 n + 1 of them, 16 for n = 5):
// a pivot is the broadcast of one column, on which every lane finds the same row
// to exchange, and an update of n entries.  Eliminating above the diagonal as well
// (Gauss-Jordan) takes the back substitution, and its n further broadcasts, out of
// the chain.  A scan launch of 4097 states takes 13 us at n = 5 and one of 5004
// states 24 at n = 6; the lane-per-combination kernel, which spills, 121 and 251.
template <typename R, int NX, int G>
struct CoopResult<FView<R, NX>, G, false> {
  using V = FView<R, NX>;
  static constexpr int n = NX, NC = 3 * n + 1, NS = (NC + G - 1) / G;
  static_assert(n <= G, "the pivot columns lie in the first slot");
  static constexpr bool has_info(int s) { return (s + 1) * G > 2 * n; }   // columns of Y and y
  R z[NS][n];   // column of J, or eta
  R o[NS][n];   // row of C, column of A, or b

  PSM_DEV void write(R* out, int flag, int r) const {
    static_for<0, NS>([&](auto sc) {
      constexpr int s = decltype(sc)::value;
      const int q = s * G + r;
      const bool isx = q >= n && q < 2 * n, isw = q == 3 * n;
      if (q >= n && q < NC) {
        R* op = isx ? out + V::QU + (q - n) * n : isw ? out + V::QB : out + V::QA + (q - 2 * n);
        const int step = isx || isw ? 1 : n;
#pragma unroll
        for (int k = 0; k < n; ++k) op[k * step] = o[s][k];
      }
      if constexpr (has_info(s)) {
        if (q >= 2 * n && q < NC) {
          R* op = isw ? out + V::QE : out + V::QZ + (q - 2 * n);
          const int step = isw ? 1 : n;
#pragma unroll
          for (int k = 0; k < n; ++k) op[k * step] = z[s][k];
        }
      }
    });
    if (r == 0) out[V::QF] = R(flag);
  }

  template <typename C, bool ILL>
  PSM_DEV bool compute(const R* e1, const R* e2, int r, float) {
    static_assert(std::is_same<C, R>::value && !ILL, "no recomputation in this form");
    R x[NS][n], v[NS][n];
    static_for<0, NS>([&](auto sc) {
      constexpr int s = decltype(sc)::value;
      const int q = s * G + r;
      const bool isn = q < n, isx = !isn && q < 2 * n, isj = !isn && !isx && q < 3 * n;
      // column of C1, row of A2, column of A1, or b1
      const R* ap = isn ? e1 + V::QU + q : isx ? e2 + V::QA + (q - n) * n : isj ? e1 + V::QA + (q - 2 * n) : e1 + V::QB;
      const int step = isn || isj ? n : 1;
#pragma unroll
      for (int k = 0; k < n; ++k) v[s][k] = ap[k * step];
#pragma unroll
      for (int i = 0; i < n; ++i) {
        R acc = e2[V::QZ + i * n] * v[s][0];
#pragma unroll
        for (int k = 1; k < n; ++k) acc = fma(e2[V::QZ + i * n + k], v[s][k], acc);
        const R add = isn && i == q ? R(1) : R(0);
        x[s][i] = isx ? v[s][i] : isn || isj ? acc + add : e2[V::QE + i] - acc;
      }
    });
    static_for<0, n>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      R p[n];
#pragma unroll
      for (int k = 0; k < n; ++k) p[k] = from_lane<G, i>(x[0][k]);
#pragma unroll
      for (int k = i + 1; k < n; ++k) {
        const bool sw = abs_(p[k]) > abs_(p[i]);
        const R t = p[i];
        p[i] = sw ? p[k] : t;
        p[k] = sw ? t : p[k];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          const R u = x[s][i];
          x[s][i] = sw ? x[s][k] : u;
          x[s][k] = sw ? u : x[s][k];
        }
      }
      const R inv = rcp_(p[i]);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        x[s][i] *= inv;
#pragma unroll
        for (int k = 0; k < n; ++k)
          if (k != i) x[s][k] = fma(-p[k], x[s][i], x[s][k]);
      }
    });
    static_for<0, NS>([&](auto sc) {
      constexpr int s = decltype(sc)::value;
      const int q = s * G + r;
      const bool isx = q < 2 * n, isj = !isx && q < 3 * n, isw = q == 3 * n;
      if constexpr (has_info(s)) {
        const R* zp = isj ? e1 + V::QZ + (q - 2 * n) : e1 + V::QE;
        const int step = isj ? n : 1;
#pragma unroll
        for (int j = 0; j < n; ++j) {
          R acc = e1[V::QA + j] * x[s][0];
#pragma unroll
          for (int k = 1; k < n; ++k) acc = fma(e1[V::QA + k * n + j], x[s][k], acc);
          z[s][j] = acc + zp[j * step];
        }
      }
      R t[n];
#pragma unroll
      for (int j = 0; j < n; ++j) {
        R acc = e1[V::QU + j * n] * x[s][0];
#pragma unroll
        for (int k = 1; k < n; ++k) acc = fma(e1[V::QU + j * n + k], x[s][k], acc);
        t[j] = isx ? acc : isj ? v[s][j] - acc : v[s][j] + acc;
      }
      const R* op = isx ? e2 + V::QU + (q >= n ? q - n : 0) * n : e2 + V::QB;
#pragma unroll
      for (int j = 0; j < n; ++j) {
        R acc = e2[V::QA + j * n] * t[0];
#pragma unroll
        for (int k = 1; k < n; ++k) acc = fma(e2[V::QA + j * n + k], t[k], acc);
        o[s][j] = isx || isw ? acc + op[j] : acc;
      }
    });
    return false;
  }
};

// g = E2 g1 + g2, E = E2 E1, D = E2 D1 E2^T + D2 (parsmooth/parallel/_operators.py:95-101):
// the low half forms the rows of D, the high half those of E.
template <typename R, int NX, int G>
struct CoopResult<SView<R, NX>, G, false> {
  using V = SView<R, NX>;
  static constexpr int n = NX, HL = G / 2;
  static_assert(n <= HL, "one row per lane of a half");
  R f[n], g;

  PSM_DEV void write(R* out, int flag, int r) const {
    const bool high = r >= HL;
    const int i = high ? r - HL : r;
    if (i < n) {
      R* op = out + (high ? V::QE : V::QD) + i * n;
      out[V::QG + i] = g;   // the same value on both halves
#pragma unroll
      for (int j = 0; j < n; ++j) op[j] = f[j];
    }
    if (r == 0) out[V::QF] = R(flag);
  }

  template <typename C, bool ILL>
  PSM_DEV bool compute(const R* e1, const R* e2, int r, float) {
    static_assert(std::is_same<C, R>::value && !ILL, "no recomputation in this form");
    const bool high = r >= HL;
    const int row = high ? r - HL : r;
    const int i = row < n ? row : 0;
    const R* mp = e1 + (high ? V::QE : V::QD);
    R a[n], t[n];
    g = R(0);
#pragma unroll
    for (int k = 0; k < n; ++k) {
      a[k] = e2[V::QE + i * n + k];
      g = fma(a[k], e1[V::QG + k], g);
    }
    g += e2[V::QG + i];
#pragma unroll
    for (int j = 0; j < n; ++j) {
      t[j] = a[0] * mp[j];
#pragma unroll
      for (int k = 1; k < n; ++k) t[j] = fma(a[k], mp[k * n + j], t[j]);
    }
#pragma unroll
    for (int j = 0; j < n; ++j) {
      R acc = e2[V::QD + i * n + j];
#pragma unroll
      for (int k = 0; k < n; ++k) acc = fma(e2[V::QE + j * n + k], t[k], acc);
      f[j] = high ? t[j] : acc;
    }
    return false;
  }
};

// One combination by a group, in two halves so that the result may overwrite an
// operand of this or of another group: prepare() reads e1 and e2, commit() writes.
// Between them the caller synchronises the groups that read what this one
// writes.  prepare() covers the flag cases of combine_mem and, for FP32, the
// recomputation in FP64 when the combined factor is ill-conditioned (the rule
// of combine_mem_fb).  The flags and the decision are the same on every lane of
// a group, so the group stays together.
template <typename V, int G, bool SQRT>
struct CoopStep {
  using R = typename V::real_type;
  CoopResult<V, G, SQRT> res;
  int flag = -1;   // of the result; negative: nothing to write

  // the result goes where e2 is (scan: e2 holds an item's running aggregate and
  // e1 the earlier one's; an identity e2 belongs to no item and may stay) or, with
  // own == true, where e1 is (a group's own running aggregate)
  template <typename FB>
  PSM_DEV void prepare(R* e1, const R* e2, bool own, int r, const FB& fb) {
    const int f1 = (int)e1[V::QF], f2 = (int)e2[V::QF];
    if (f2 == FLAG_HEAD || f1 == FLAG_IDENT || f2 == FLAG_IDENT) {
      if (own && f2 != FLAG_IDENT) {
        ItemRegs<V, G> item;
        item.load(e2, r);
        group_sync();
        item.store(e1, r);
      }
      return;
    }
    constexpr bool FBK = kFallback<R, SQRT>;
    const bool ill = res.template compute<R, FBK>(e1, e2, r, fb.thr);
    if constexpr (FBK && !FB::kRedo) {
      if (fb.thr > 0.f && ill && r == 0) fb.raise();
    } else if constexpr (FBK) {
      if (fb.thr > 0.f && ill) {
        res.template compute<double, false>(e1, e2, r, 0.f);
        if (r == 0) count_fallback(fb);
      }
    }
    flag = f1;
  }
  PSM_DEV void commit(R* out, int r) const {
    if (flag >= 0) res.write(out, flag, r);
  }
};

}  // namespace psm

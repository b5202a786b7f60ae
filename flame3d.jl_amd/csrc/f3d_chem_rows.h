// The Newton mode's backward-Euler solve with half a wave to a cell, for the
// few cells of a list that take many iterations.
//
// One thread per cell (chem.hip) has the throughput, but its iteration is one
// instruction stream of 19 us, and a cell that fails its first step after 50
// iterations and then takes substeps holds the whole call for a millisecond.
// Here a lane evaluates one species' fits, then one reaction with its
// derivatives, then holds one row of the system (row Ns: the energy) and
// eliminates it; what the reactions give to the rows, the pivot rows and the
// result go through LDS.  An iteration is a chain of 7.5 us: the fits 1.1 us,
// the rates (a falloff's two logarithms and eleven divisions) 1.6, the rows 1.2,
// nine pivots 2.3, the back substitution 0.8.  What counts is the number of
// instructions in the stream (16 lanes to a cell, two reactions to a lane and
// selects for the stoichiometry: 13 us) and that LDS reads are under way before
// they are needed (10.8 us without).  Every sum is formed in the order of the
// one-thread solve, so the states are the same bits.
#pragma once

#include "f3d_chem.h"

namespace f3d {

// What the row solve needs to know of a mechanism's tables at compile time.
template <class T>
struct RowForms {
  static constexpr int count(const int* v) {
    int c = 0;
    for (int m = 0; m < T::NS; ++m) c += v[m] != 0;
    return c;
  }
  // slot of species m among reaction n's reactants (0, 1) or products (2, 3);
  // -1 if it has no part
  static constexpr int slot(int n, int m) {
    if (T::vf[n][m] == 0 && T::vr[n][m] == 0) return -1;
    const int* v = T::vf[n][m] != 0 ? T::vf[n] : T::vr[n];
    int c = T::vf[n][m] != 0 ? 0 : 2;
    for (int j = 0; j < m; ++j) c += v[j] != 0;
    return c;
  }
  static constexpr int falloffs() {
    int c = 0;
    for (int n = 0; n < T::NR; ++n) c += T::rtype[n] == 3;
    return c;
  }
  // at most two reactants and two products, none on both sides, powers of one
  // and two, a mole change of at most one
  static constexpr bool fits() {
    for (int n = 0; n < T::NR; ++n) {
      if (T::sgm[n] > 1 || T::sgm[n] < -1 || count(T::vf[n]) > 2 || count(T::vr[n]) > 2)
        return false;
      for (int m = 0; m < T::NS; ++m)
        if (T::vf[n][m] < 0 || T::vf[n][m] > 2 || T::vr[n][m] < 0 || T::vr[n][m] > 2 ||
            (T::vf[n][m] != 0 && T::vr[n][m] != 0))
          return false;
    }
    return true;
  }
  static constexpr int kLanes = 32;  // lanes of a cell
  // four exponentials of a falloff reaction are evaluated by lanes past the reactions
  static constexpr int kExp = T::NR + 4 * falloffs();
  static_assert(T::NS + 1 <= 16, "the rows within 16 lanes");
  static_assert(kExp <= kLanes, "a reaction to a lane");
  static_assert(fits(), "two reactants, two products");
};

constexpr int kRowCells = 2;  // cells of a wave

template <class T>
struct alignas(16) RowsLds {
  static constexpr int NS = T::NS, N1 = T::NS + 1, kRow = (N1 + 3) / 2 * 2;
  double d[kRowCells][T::NR][8];  // dq/dc of the four slots, dq, dq/dT, dq/d[M]
  double lu[kRowCells][N1][kRow];  // an eliminated row, its right-hand side, 1 / pivot
  double sc[kRowCells][NS + 3];  // concentrations, then 1, Ru T, 1 / (Ru T)
  double r[kRowCells][NS], te[kRowCells][NS], tc[kRowCells][NS];
  double g[kRowCells][NS + 1], h[kRowCells][NS + 1];  // [NS]: 0
  double de[kRowCells][NS], dx[kRowCells][N1];
  double ex[kRowCells][RowForms<T>::kLanes];
  double nu[T::NR][16], wnl[NS][16];  // of the lane's row
};

// LDS written by some lanes of the wave is read by others below this point
// (a wave's LDS accesses are performed in order)
__device__ __forceinline__ void rows_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LDS reads are issued ahead of the arithmetic that the barrier keeps below
// them: left to itself the compiler reads each value where it is used and
// waits for it there
__device__ __forceinline__ void rows_ahead() { __builtin_amdgcn_sched_barrier(0); }

template <int CTRL>
__device__ __forceinline__ unsigned row_dpp(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
}
// maximum over the 16 lanes of a DPP row, in all of them (rotations by 8, 4, 2, 1)
__device__ __forceinline__ unsigned row_max(unsigned v) {
  v = max(v, row_dpp<0x128>(v));
  v = max(v, row_dpp<0x124>(v));
  v = max(v, row_dpp<0x122>(v));
  return max(v, row_dpp<0x121>(v));
}
// the first 16 lanes of this thread's cell where p holds
__device__ __forceinline__ unsigned row_ballot(bool p) {
  return (unsigned)(__ballot(p) >> (threadIdx.x & 32)) & 0xffffu;
}

// A lane's reaction, read from the parameter block once.  The powers are
// products of two LDS entries, x and x again or 1; an absent slot reads 1.
template <class T>
struct RowReaction {
  static constexpr int NS = T::NS;
  int n, rt, ix[4], iq[4], iw, ie;  // ix, iq: reactants 0, 1 and products 2, 3
  int im[4];                        // the participants in species order ([NS]: none)
  double v[4], nu[4], sg;
  double Arr[3], ef[NS], loP[3], Troe[4];
  double c1, c2;  // the lane's exponential: c1 ln T - c2 / T, -T / c1 or -c1 / T
  int kind;
  __device__ void read(const DevParams* __restrict__ P, int l) {
    n = l < T::NR ? l : 0;
    rt = P->rtype[n];
    sg = (double)P->sgm[n];
    iw = P->sgm[n] == 0 ? NS : (P->sgm[n] < 0 ? NS + 1 : NS + 2);
    int cf = 0, cr = 2, cm = 0;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      ix[s] = iq[s] = im[s] = NS;
      v[s] = nu[s] = 0.0;
    }
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const int f = P->vf[n][j], b = P->vr[n][j];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if ((f != 0 && cf == s) || (b != 0 && cr == s)) {
          ix[s] = j;
          iq[s] = f + b == 2 ? j : NS;
          v[s] = (double)(f + b);
        }
        if ((f != 0 || b != 0) && cm == s) {
          im[s] = j;
          nu[s] = (double)(f - b);
        }
      }
      cf += f != 0;
      cr += b != 0;
      cm += f != 0 || b != 0;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      Arr[k] = P->Arr[n][k];
      loP[k] = P->loP[n][k];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) Troe[k] = P->Troe[n][k];
#pragma unroll
    for (int j = 0; j < NS; ++j) ef[j] = P->ef[n][j];
    c1 = Arr[1];
    c2 = Arr[2];
    kind = 0;
    ie = 0;
    int fall = 0;
    for (int i = 0; i < T::NR; ++i) {  // the falloff reactions' exponentials, in order
      if (P->rtype[i] != 3) continue;
      const int first = T::NR + 4 * fall++;
      if (i == l) ie = first;
      const int e = l - first;
      if (e == 0) {
        c1 = P->loP[i][1];
        c2 = P->loP[i][2];
      } else if (e == 1 || e == 2) {
        c1 = P->Troe[i][e];
        kind = 1;
      } else if (e == 3) {
        c1 = P->Troe[i][3];
        kind = 2;
      }
    }
  }
};

// production_rate's body (TDER, RCP, FULL) for one reaction to a lane
template <class T>
__device__ __forceinline__ void row_reaction(const RowReaction<T>& R, RowsLds<T>& L, int grp,
                                             double kf, double invT) {
  constexpr int NS = T::NS;
  double gg[4], hh[4], x[4], q[4], p[4], sc[NS];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    gg[s] = L.g[grp][R.im[s]];
    hh[s] = L.h[grp][R.im[s]];
  }
  const double wRT = L.sc[grp][R.iw];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    q[s] = L.sc[grp][R.iq[s]];
    x[s] = L.sc[grp][R.ix[s]];
  }
#pragma unroll
  for (int m = 0; m < NS; ++m) sc[m] = L.sc[grp][m];
  rows_ahead();
  double dg = 0, dgs = 0;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    dg += gg[s] * R.nu[s];
    dgs += hh[s] * R.nu[s];
    p[s] = x[s] * q[s];
  }
  const double kr = kf * (wRT * f3d_exp(-dg));
  double q_f = kf * p[0] * p[1];
  double q_r = kr * p[2] * p[3];
  double dlnq_dM = 0.0, fac = 1.0, dlnfac = 0.0;
  if (R.rt != 1) {
    double mix = 0.0;
#pragma unroll
    for (int m = 0; m < NS; ++m) mix += R.ef[m] * sc[m];
    fac = mix;
    double den = mix;
    if (RowForms<T>::falloffs() > 0 && R.rt == 3) {
      const double redP = mix / kf * R.loP[0] * L.ex[grp][R.ie];
      const double logPred = f3d_log10(redP);
      const double A_ = R.Troe[0];
      const double e3 = L.ex[grp][R.ie + 1];
      const double e1 = L.ex[grp][R.ie + 2];
      const double e2 = L.ex[grp][R.ie + 3];
      const double Fcent = (1 - A_) * e3 + A_ * e1 + e2;
      const double logFcent = f3d_log10(Fcent);
      const double troe_c = -0.4 - 0.67 * logFcent;
      const double troe_n = 0.75 - 1.27 * logFcent;
      const double troe = (troe_c + logPred) / (troe_n - 0.14 * (troe_c + logPred));
      const double F_troe = f3d_exp10(logFcent / (1.0 + troe * troe));
      fac = (redP / (1.0 + redP)) * F_troe;
      den = (1.0 + redP) * mix;
      const double ln10 = 2.30258509299404568402;
      const double dlnPr = (R.loP[1] - R.Arr[1]) * invT + (R.loP[2] - R.Arr[2]) * invT * invT;
      const double dL = dlnPr / ln10;
      const double dFc = -(1 - A_) / R.Troe[1] * e3 - A_ / R.Troe[2] * e1 +
                         R.Troe[3] * invT * invT * e2;
      const double dLc = dFc / (Fcent * ln10);
      const double u = troe_c + logPred;
      const double v = troe_n - 0.14 * u;
      const double du = -0.67 * dLc + dL;
      const double dv = -1.27 * dLc - 0.14 * du;
      const double dtroe = (du * v - u * dv) / (v * v);
      const double w = 1.0 + troe * troe;
      const double dlog10F = dLc / w - logFcent * (2.0 * troe * dtroe) / (w * w);
      dlnfac = dlnPr / (1.0 + redP) + ln10 * dlog10F;
    }
    q_f *= fac;
    q_r *= fac;
    dlnq_dM = 1.0 / den;
  }
  double* D = L.d[grp][R.n];
  D[0] = kf * R.v[0] * q[0] * p[1] * fac;
  D[1] = kf * R.v[1] * q[1] * p[0] * fac;
  D[2] = -(kr * R.v[2] * q[2] * p[3]) * fac;
  D[3] = -(kr * R.v[3] * q[3] * p[2]) * fac;
  const double dq = q_f - q_r;
  D[4] = dq;
  const double dlnkf = R.Arr[1] * invT + R.Arr[2] * invT * invT;
  const double dlnKc = R.sg * invT - dgs * invT;
  D[5] = q_f * (dlnkf + dlnfac) - q_r * (dlnkf - dlnKc + dlnfac);
  D[6] = dq * dlnq_dM;
}

// what a lane holds of its species (or energy) row over the iterations
template <class T>
struct RowConst {
  static constexpr int NS = T::NS;
  double mw, cmw, rmw, Rmw, hfm, sep;
  __device__ void read(const DevParams* __restrict__ P, RowsLds<T>& L, int l) {
    const int n = l < NS ? l : 0;
    if (threadIdx.x < 16) {
#pragma unroll
      for (int i = 0; i < T::NR; ++i)
        L.nu[i][l] = l < NS ? (double)(P->vr[i][n] - P->vf[i][n]) : 0.0;
#pragma unroll
      for (int j = 0; j < NS; ++j) L.wnl[j][l] = P->wnl[n][j];
    }
    mw = P->mw[n];
    cmw = P->cmw[n];
    rmw = P->rmw[n];
    Rmw = P->Rmw[n];
    hfm = P->hfm[n];
    sep = P->sep[n];
  }
};

typedef double f64x2 __attribute__((ext_vector_type(2)));
template <int FROM, int N>
__device__ __forceinline__ void load_pairs(const double* p, double (&v)[N]) {
  static_assert(N % 2 == 0, "pairs");
#pragma unroll
  for (int j = FROM / 2 * 2; j < N; j += 2) {
    const f64x2 t = *reinterpret_cast<const f64x2*>(p + j);
    v[j] = t.x;
    v[j + 1] = t.y;
  }
}

// what a reaction gives to the rows (RowsLds::d), and the row's nu
struct RowTerm {
  f64x2 p0, p1, p2, p3;
  double nu;
  template <int I>
  __device__ __forceinline__ double get() const {
    const f64x2 p = I < 2 ? p0 : I < 4 ? p1 : I < 6 ? p2 : p3;
    return I % 2 ? p.y : p.x;
  }
};
template <class T, int N>
__device__ __forceinline__ void row_term_load(const RowsLds<T>& L, int grp, int l, RowTerm& t) {
  if constexpr (N < T::NR) {
    const f64x2* d = reinterpret_cast<const f64x2*>(L.d[grp][N]);
    t.p0 = d[0];
    t.p1 = d[1];
    t.p2 = d[2];
    if constexpr (T::rtype[N] != 1) t.p3 = d[3];
    t.nu = L.nu[N][l];
  }
}
template <class T, int N, int M>
__device__ __forceinline__ void row_entry_add(const RowTerm& t, double& a) {
  if constexpr (T::rtype[N] != 1 && T::ef[N][M] != 0.0)
    a += t.template get<6>() * T::ef[N][M] * t.nu;
  constexpr int slot = RowForms<T>::slot(N, M);
  if constexpr (slot >= 0) a += t.template get<slot>() * t.nu;
}
template <class T, int N, int... M>
__device__ __forceinline__ void row_term_add(const RowTerm& t, double (&a)[T::NS + 1],
                                             double& wdot, std::integer_sequence<int, M...>) {
  (row_entry_add<T, N, M>(t, a[M]), ...);
  a[T::NS] += t.p2.y * t.nu;
  wdot += t.p2.x * t.nu;
}
// every reaction in order, the terms of the next two on their way
template <class T, int... N>
__device__ __forceinline__ void row_sums(const RowsLds<T>& L, int grp, int l,
                                         double (&a)[T::NS + 1], double& wdot,
                                         std::integer_sequence<int, N...>) {
  RowTerm t0, t1, t2;
  row_term_load<T, 0>(L, grp, l, t0);
  row_term_load<T, 1>(L, grp, l, t1);
  ((row_term_load<T, N + 2>(L, grp, l, t2), rows_ahead(),
    row_term_add<T, N>(t0, a, wdot, std::make_integer_sequence<int, T::NS>{}), t0 = t1, t1 = t2),
   ...);
}

// column C of the elimination and those after it
template <class T, int C>
__device__ __forceinline__ void row_eliminate(RowsLds<T>& L, int grp, int l, int& pos,
                                              double (&a)[T::NS + 1], double& b) {
  constexpr int N1 = T::NS + 1, kRow = RowsLds<T>::kRow;
  if constexpr (C < N1 - 1) {
    const bool cand = pos >= C && pos < N1;
    const double inv = 1.0 / a[C];  // beside the search: of use if this is the pivot
    const unsigned v = cand ? (unsigned)__double2hiint(a[C]) & 0x7fffffffu : 0u;
    const unsigned vmax = row_max(v);
    unsigned top = row_ballot(cand && v == vmax);
    if (__builtin_popcount(top) != 1) {
      double vm = -1.0;
      unsigned best = 0;
#pragma unroll 1
      for (int i = C; i < N1; ++i) {
        const unsigned at = row_ballot(pos == i);
        const double w = fabs(__shfl(a[C], __builtin_ctz(at | 0x10000u), RowForms<T>::kLanes));
        if (i == C || w > vm) {
          vm = w;
          best = at;
        }
      }
      top = best;
    }
    const int piv = __builtin_ctz(top | 0x10000u);
    const int ppos = __shfl(pos, piv, RowForms<T>::kLanes);
    double* row = L.lu[grp][C];
    if (l == piv) {
#pragma unroll
      for (int j = C; j < N1; ++j) row[j] = a[j];
      row[kRow - 2] = b;
      row[kRow - 1] = inv;
    }
    rows_sync();
    double p[kRow];
    load_pairs<C + 1>(row, p);
    rows_ahead();
    pos = l == piv ? C : (pos == C ? ppos : pos);
    const double f = -a[C] * p[kRow - 1];
#pragma unroll
    for (int j = C + 1; j < N1; ++j) a[j] += f * p[j];
    b += f * p[kRow - 2];
    row_eliminate<T, C + 1>(L, grp, l, pos, a, b);
  }
}

// back substitution of rows I, I - 1, ..; p: row I, on its way
template <class T, int I>
__device__ __forceinline__ void row_back(RowsLds<T>& L, int grp,
                                         const double (&p)[RowsLds<T>::kRow],
                                         double (&dx)[T::NS + 1]) {
  constexpr int N1 = T::NS + 1, kRow = RowsLds<T>::kRow;
  double pn[kRow];
  if constexpr (I > 0) load_pairs<(I > 0 ? I - 1 : 0)>(L.lu[grp][I - 1], pn);
  rows_ahead();
  double xi = p[kRow - 2];
#pragma unroll
  for (int j = I + 1; j < N1; ++j) xi -= p[j] * dx[j];
  dx[I] = xi / p[I];
  L.dx[grp][I] = dx[I];
  if constexpr (I > 0) row_back<T, I - 1>(L, grp, pn, dx);
}

// be_solve of chem.hip for the cell of this half wave: lane l < NS holds r_l in
// rl; every lane holds T and the convergence state
template <class T>
__device__ inline bool be_rows(const NasaTab<T::NS>& N, RowsLds<T>& L, int grp, int l,
                               const DevParams* __restrict__ P, const RowConst<T>& C,
                               const RowReaction<T>& R, double& rl, double& Tm, double h,
                               double E0, double rho_tot, double T_lo, double T_hi, int maxiter,
                               double rtol, double ttol) {
  constexpr int NS = T::NS, N1 = NS + 1;
  constexpr bool kInert = KinCT<T>::inert(NS - 1);
  const bool species = l < NS;
  const double rs = rl;
  const double RsT0 = P->Ru / P->atm * 1e6;
  double dT_prev = 0.0;
  for (int k = 0; k < maxiter; ++k) {
    const double lgT = f3d_log(Tm);
    const double invT = 1.0 / Tm;
    const double RsT = RsT0 * Tm;
    const double iRsT = 1.0 / RsT;
    {
      const GibbsT G(Tm, lgT, invT);
      const EnthalpyT H(Tm, invT);
      const double T2 = 0.5 * Tm * Tm;
      const double T3 = 2.0 / 3.0 * T2 * Tm;
      const double T4 = T2 * T2;
      const double T5 = 0.8 * T4 * Tm;
      const double S2 = Tm * Tm;
      const double S3 = S2 * Tm;
      const double S4 = S2 * S2;
      const NasaSet q = N.at(species ? l : 0, Tm, C.sep);
      const double e = q.c0m1 * Tm + q.c1 * T2 + q.c2 * T3 + q.c3 * T4 + q.c4 * T5 + q.d5;
      const double cp = q.c0 + q.c1 * Tm + q.c2 * S2 + q.c3 * S3 + q.c4 * S4;
      const double xt = R.kind == 0 ? R.c1 * lgT - R.c2 * invT
                                    : (R.kind == 1 ? -Tm / R.c1 : -R.c1 * invT);
      L.ex[grp][l] = f3d_exp(xt);
      L.sc[grp][NS + 1] = RsT;
      L.sc[grp][NS + 2] = iRsT;
      if (species) {
        L.r[grp][l] = rl;
        L.sc[grp][l] = rl * C.cmw;
        L.g[grp][l] = G.g(q);
        L.h[grp][l] = H.h(q);
        L.te[grp][l] = rl * e * C.rmw;
        L.tc[grp][l] = (cp - 1) * rl * C.rmw;
        L.de[grp][l] = e * C.Rmw + C.hfm;
      }
    }
    rows_sync();
    double E = 0, cv = 0, rho = 0;
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      E += L.te[grp][n];
      cv += L.tc[grp][n];
      rho += L.r[grp][n];
    }
    E *= P->Ru;
    cv *= P->Ru;
#pragma unroll
    for (int n = 0; n < NS; ++n) E += P->hfm[n] * L.r[grp][n];
    if (l < T::NR) row_reaction<T>(R, L, grp, R.Arr[0] * L.ex[grp][l], invT);
    rows_sync();
    // The lane's row: every sum over the reactions in order.  A reaction that
    // the species has no part in adds zeros.
    double a[N1], b, wdot = 0.0;
#pragma unroll
    for (int j = 0; j < N1; ++j) a[j] = 0.0;
    row_sums(L, grp, l & 15, a, wdot, std::make_integer_sequence<int, T::NR>{});
    {
      const double src = wdot * C.mw * 1e6 * h;
      b = -(rl - rs - src);
#pragma unroll
      for (int j = 0; j < NS; ++j) a[j] = (j == l ? 1.0 : 0.0) - a[j] * L.wnl[j][l & 15] * h;
      a[NS] = -a[NS] * C.mw * 1e6 * h;
      if (kInert && l == NS - 1) a[NS] = 0.0;
      if (l == NS) {
        b = -(E - E0);
#pragma unroll
        for (int j = 0; j < NS; ++j) a[j] = L.de[grp][j];
        a[NS] = cv;
      }
    }
    // gauss_solve<N1, true, kInert>: a row stays in its lane, pos is its place
    // after the exchanges (rows that were pivots go on being updated, unread).
    // The pivot is the entry of the largest upper word; equal upper words take
    // the comparison in full and then, as the exchanges do, the first place.
    // (An entry that is not a number has the largest upper word and is taken,
    // where the exchanges would pass it over; with either the update is not a
    // number and the solve fails.)
    int pos = l < N1 ? l : 99;
    row_eliminate<T, 0>(L, grp, l, pos, a, b);
    if (pos == N1 - 1) {
      L.lu[grp][N1 - 1][N1 - 1] = a[N1 - 1];
      L.lu[grp][N1 - 1][RowsLds<T>::kRow - 2] = b;
    }
    rows_sync();
    double dx[N1], mx = 0.0;
    {
      double p[RowsLds<T>::kRow];
      load_pairs<N1 - 1>(L.lu[grp][N1 - 1], p);
      row_back<T, N1 - 1>(L, grp, p, dx);
    }
#pragma unroll
    for (int i = 0; i < NS; ++i) mx = fmax(mx, fabs(dx[i]));
    rows_sync();
    rl += species ? L.dx[grp][species ? l : 0] : 0.0;
    const bool bad = row_ballot(species && !(rl > -rho_tot)) != 0;
    Tm += dx[NS];
    const bool flip = k > 0 && dx[NS] * dT_prev < 0 && fabs(dx[NS]) >= 0.5 * fabs(dT_prev);
    dT_prev = dx[NS];
    if (bad || !(Tm > T_lo && Tm < T_hi)) return false;
    if (mx <= rtol * rho && (fabs(dx[NS]) <= ttol || flip)) return true;
  }
  return false;
}

// k_chem<NS, 2> for the cells of `list`, two to a wave; the waves stride over
// the list, whose length (at most `most`) the device knows
template <class T>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1)))
    k_newton_rows(double* __restrict__ U, double* __restrict__ Q, double* __restrict__ rhoi,
                  double dt, int maxiter, double rtol, double ttol,
                  const DevParams* __restrict__ P, Geom g, int max_sub,
                  const int32_t* __restrict__ list, const int32_t* __restrict__ count, int most) {
  constexpr int NS = T::NS;
  __shared__ NasaTab<NS> N;
  __shared__ RowsLds<T> L;
  const int nwork = min(*count, most);
  if ((int)blockIdx.x * kRowCells >= nwork) return;
  N.fill(P);
  const int grp = threadIdx.x >> 5, l = threadIdx.x & 31;
  const long NP = g.NP;
  RowConst<T> C;
  C.read(P, L, l);
  RowReaction<T> R;
  R.read(P, l);
  if (l == 0) {
    L.sc[grp][NS] = 1.0;
    L.g[grp][NS] = L.h[grp][NS] = 0.0;
  }
  const double T_lo = 0.5 * P->min_temp, T_hi = 1.5 * P->max_temp;
  for (int w = (int)blockIdx.x * kRowCells + grp; w < nwork; w += (int)gridDim.x * kRowCells) {
    const long id = list[w];
    const int a = (int)(id % g.Nx);
    const int t = (int)(id / g.Nx);
    const int b = t % g.Ny, c = t / g.Ny;
    const long p = (a + NG) + (long)g.Nxt * ((b + NG) + (long)g.Nyt * (c + NG));
    const double T0 = Q[p + 5 * NP];
    double r[NS], rho_tot = 0.0, r0 = 0.0;
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      r[n] = rhoi[p + n * NP];
      rho_tot += r[n];
      r0 = l == n ? r[n] : r0;
    }
    double E0 = internal_energy<NS, true>(N, P, T0, r);
#pragma unroll
    for (int n = 0; n < NS; ++n) E0 += P->hfm[n] * r[n];
    bool ok = false;
    double Tm = T0, rl = r0;
    for (int nsub = 1; nsub <= max_sub && !ok; nsub *= 2) {
      rl = r0;
      Tm = T0;
      ok = true;
      const double h = dt / nsub;
      for (int k = 0; k < nsub && ok; ++k)
        ok = be_rows<T>(N, L, grp, l, P, C, R, rl, Tm, h, E0, rho_tot, T_lo, T_hi, maxiter, rtol,
                        ttol);
    }
    if (!ok) rl = r0;  // no admissible solution: the reactor is left unreacted
    if (l < NS) L.r[grp][l] = rl;
    rows_sync();
    if (l == 0) {
      double dei = 0;
#pragma unroll
      for (int n = 0; n < NS; ++n) {
        dei += -P->hfm[n] * (L.r[grp][n] - r[n]);
        r[n] = L.r[grp][n];
      }
      chem_epilogue<NS>(N, P, U, Q, rhoi, p, NP, r, dei);
    }
  }
}

}  // namespace f3d

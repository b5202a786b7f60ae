// FP64 stiff chemistry (reactions.jl:176-503): production rates with the
// analytic species Jacobian, point-implicit update with a pivoted dense solve
// in registers, and a backward-Euler Newton mode on (rho_k, T).
//
// One thread per interior cell.  The species count is a template parameter so
// the Ns x Ns (or (Ns+1)^2) matrix, the rates and the Gibbs energies live in
// registers with compile-time indices; the reaction loop runs over the
// mechanism held in the uniform parameter block, so its stoichiometry tests
// are wave-uniform branches that skip the zero terms the reference adds; for a
// shipped mechanism it is unrolled over the compiled-in tables.
//
// The Newton mode is bound by instruction issue at two waves per SIMD, so what
// counts is how many instructions an iteration takes and how long a wave waits
// for its slowest cell.  128^3 H2/O2 reactors (2.45 iterations per cell on
// average, 5.0 for the slowest of 64): 28.6 ms with the reactions in a run-time
// loop, branches in exp and log, every pivot exchange taken and 256-thread
// blocks; 8.84 ms with one instantiation per reaction, selects, exchanges only
// where a lane needs them and one-wave blocks; 8.01 ms with the NASA-7 sets in
// LDS and read once per iteration, and the parameter block's quotients read
// where they are used; 3.44 ms with every sum formed where its terms are (an
// empty asm after each reaction and each species), the series' constants in
// scalar registers and the initial densities read again at the end instead of
// kept: fewer values are held across an iteration, so that two waves fit a
// SIMD with 240 bytes of scratch where one took 850.
#include "f3d_chem.h"
#include "f3d_chem_rows.h"
#include "f3d_internal.h"
#include "f3d_mech_tables.h"

namespace f3d {

// Most backward-Euler substeps the Newton mode tries before giving up.
constexpr int kNewtonMaxSub = 64;
// In a pass over a cell list: iterations of the first step after which a cell
// goes to the half-wave solve (f3d_chem_rows.h).  A list's wave ends with its
// slowest cell; one of 56 iterations takes 1.0 ms here, 0.1 + 0.42 ms this way.
// 64^3 reactors, 151610 of them listed, whole surrogate step: 0.91 ms with 8,
// 0.90 with 6, 0.88 with 5, 0.87 with 4 (1.23 ms all here); but with 4 a tenth
// of a flame's cells would go.
constexpr int kNewtonFirst = 5;

// the parameter block by scalar loads
typedef const __attribute__((address_space(4))) DevParams ConstParams;

// Per-lane values that an iteration needs now and then live in LDS (the
// Jacobian takes the registers): the substep's initial densities and the
// species' g/RT, h/RT and energy derivatives at T.  With the NASA-7 table
// 20 KB for Ns = 9, an eighth of a compute unit's LDS: two waves per SIMD.
template <int NS>
struct NewtonLds {
  double rs[NS][64], g[NS][64], h[NS][64], de[NS][64];
};
template <int NS>
struct GibbsLds {
  const NewtonLds<NS>& L;
  int lane;
  __device__ double g(int m) const { return L.g[m][lane]; }
  __device__ double h(int m) const { return L.h[m][lane]; }
};

// One backward-Euler solve over h of the reactor (rho_k, T) from (r, T),
// total energy fixed at E0: Newton on
//   F_k = rho_k - rs_k - h W_k wdot_k(rho, T) = 0,  F_E = E(rho, T) - E0 = 0
// with the exact mass-action Jacobian (+ third-body terms) and the analytic
// temperature derivative of the rates.  Constant quotients (1e-6/W_n,
// W_n/W_l, Ru/W_n, 1/W_n, the reverse rates' 1/RsT, the pivots' reciprocals)
// are multiplied where the reference's point-implicit step divides.  Returns
// false when the iterate leaves the admissible set (non-finite, T outside
// [T_lo, T_hi], rho_k < -rho_tot) or maxiter iterations pass without
// convergence; `it` counts the iterations taken.
template <int NS, class K>
__device__ inline bool be_solve(const NasaTab<NS>& N, NewtonLds<NS>& L, int lane,
                                const DevParams* __restrict__ P0, double (&r)[NS], double& T,
                                double h, double E0, double rho_tot, double T_lo, double T_hi,
                                int maxiter, double rtol, double ttol, int& it) {
  constexpr int N1 = NS + 1;
  constexpr bool kInert = K::inert(NS - 1);
#pragma unroll
  for (int n = 0; n < NS; ++n) L.rs[n][lane] = r[n];
  double dT_prev = 0.0;
  ConstParams* P = (ConstParams*)(uintptr_t)P0;
  for (int k = 0; k < maxiter; ++k) {
    // the parameters are read again in every iteration (scalar loads that hit
    // the scalar cache): hoisted out of the loop they would be spilled
    asm volatile("" : "+s"(P));
    double sc[NS], wdot[NS];
#pragma unroll
    for (int n = 0; n < NS; ++n) sc[n] = r[n] * P->cmw[n];
    // the rate Jacobian is built in the top-left block of the system matrix
    // and turned into I - W_n/W_l h dwdot/dc in place (one matrix in registers)
    double A[N1][N1], rhs[N1], dx[N1];
    // one pass over the NASA-7 fits: g/RT, h/RT, dE/drho_k, and the sums of E
    // and c_v (ei_specs, thermo.jl:136-160)
    const double lgT = f3d_log(T);
    const double invT = 1.0 / T;
    double E = 0, cv = 0;
    {
      const GibbsT G(T, lgT, invT);
      const EnthalpyT H(T, invT);
      const double T2 = 0.5 * T * T;
      const double T3 = 2.0 / 3.0 * T2 * T;
      const double T4 = T2 * T2;
      const double T5 = 0.8 * T4 * T;
      const double S2 = T * T;
      const double S3 = S2 * T;
      const double S4 = S2 * S2;
#pragma unroll
      for (int n = 0; n < NS; ++n) {
        const NasaSet q = N.at(n, T, P->sep[n]);
        L.g[n][lane] = G.g(q);
        L.h[n][lane] = H.h(q);
        const double e = q.c0m1 * T + q.c1 * T2 + q.c2 * T3 + q.c3 * T4 + q.c4 * T5 + q.d5;
        const double cp = q.c0 + q.c1 * T + q.c2 * S2 + q.c3 * S3 + q.c4 * S4;
        E += r[n] * e * P->rmw[n];
        cv += (cp - 1) * r[n] * P->rmw[n];
        L.de[n][lane] = e * P->Rmw[n] + P->hfm[n];
        // formed here: sunk to their use, the sums would keep every fit alive
        // across the assembly
        asm volatile("" : "+v"(E), "+v"(cv));
      }
      E *= P->Ru;
      cv *= P->Ru;
#pragma unroll
      for (int n = 0; n < NS; ++n) E += P->hfm[n] * r[n];
      asm volatile("" : "+v"(E));
    }
    // rate Jacobian in A[0..NS-1][0..NS-1], d wdot / dT in A[0..NS-1][NS]
    production_rate<NS, true, true, N1, true, true, K>(P0, sc, T, lgT, invT,
                                                       GibbsLds<NS>{L, lane}, A, wdot);
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      if (n == NS - 1 && kInert) {  // no rate: a unit row
        rhs[n] = -(r[n] - L.rs[n][lane]);
#pragma unroll
        for (int l = 0; l <= NS; ++l) A[n][l] = n == l ? 1.0 : 0.0;
        continue;
      }
      const double src = wdot[n] * P->mw[n] * 1e6 * h;
      rhs[n] = -(r[n] - L.rs[n][lane] - src);
#pragma unroll
      for (int l = 0; l < NS; ++l) A[n][l] = (n == l ? 1.0 : 0.0) - A[n][l] * P->wnl[n][l] * h;
      A[n][NS] = -A[n][NS] * P->mw[n] * 1e6 * h;
    }
    rhs[NS] = -(E - E0);
#pragma unroll
    for (int l = 0; l < NS; ++l) A[NS][l] = L.de[l][lane];
    A[NS][NS] = cv;
    gauss_solve<N1, true, kInert>(A, rhs, dx);
    double rho = 0;
#pragma unroll
    for (int n = 0; n < NS; ++n) rho += r[n];
    double mx = 0;
    bool bad = false;
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      r[n] += dx[n];
      mx = fmax(mx, fabs(dx[n]));
      bad = bad || !(r[n] > -rho_tot);
    }
    T += dx[NS];
    ++it;
    // NASA-7 polynomials jump at T_mid: when E0 falls in such a jump the T
    // update flips sign without contracting; with the species converged the
    // step is accepted (the final T comes from GetT of the energy)
    const bool flip = k > 0 && dx[NS] * dT_prev < 0 && fabs(dx[NS]) >= 0.5 * fabs(dT_prev);
    dT_prev = dx[NS];
    if (bad || !(T > T_lo && T < T_hi)) return false;
    if (mx <= rtol * rho && (fabs(dx[NS]) <= ttol || flip)) return true;
  }
  return false;
}

// Threads per block: one wave in the Newton mode, whose registers leave room
// for two waves per SIMD: a block of four would hold their places until its
// slowest wave (the one with the most iterations) has ended.
constexpr int chem_block(int mode) { return mode == 2 ? 64 : kBlock; }

// Two waves per SIMD asked for where the tables are compiled in; with the
// run-time loop the matrices would spill.
// mode 0: eval_gpu_stiff, 1: eval_gpu, 2: backward-Euler Newton.  K: the
// reaction parameters, from the parameter block or compiled in (KinCT).
template <int NS, int MODE, class K = KinRT>
__global__ void __launch_bounds__(chem_block(MODE)) __attribute__((amdgpu_waves_per_eu(K::kConst ? 2 : 1)))
    k_chem(double* __restrict__ U, double* __restrict__ Q, double* __restrict__ rhoi, double dt,
           int maxiter, double rtol, double ttol, int32_t* __restrict__ iters,
           const int64_t* __restrict__ tag, const DevParams* __restrict__ P, Geom g, int bug,
           const int32_t* __restrict__ list, long nwork, int32_t* __restrict__ later,
           int32_t* __restrict__ nlater, int most) {
  __shared__ NasaTab<NS> N;
  N.fill(P);
  // one thread per interior cell, or per entry of an ordered cell list (the
  // surrogate's rejected cells)
  const long t_ = gid();
  if (t_ >= nwork) return;
  const long id = list ? (long)list[t_] : t_;
  const int a = (int)(id % g.Nx);
  const int t = (int)(id / g.Nx);
  const int b = t % g.Ny, c = t / g.Ny;
  const long p = (a + NG) + (long)g.Nxt * ((b + NG) + (long)g.Nyt * (c + NG));
  if (MODE == 2 && iters) iters[id] = 0;
  if (tag && tag[p] != 0) return;
  const long NP = g.NP;
  const double T0 = Q[p + 5 * NP];
  if (!(T0 > P->T_criteria)) return;
  double r[NS], sc[NS], wdot[NS];
#pragma unroll
  for (int n = 0; n < NS; ++n) {
    r[n] = rhoi[p + n * NP];
    sc[n] = r[n] / P->mw[n] * 1e-6;
  }
  if (MODE == 1) {
    double A[NS][NS];
    production_rate_at<NS, false, K>(N, P, sc, T0, A, wdot);
    double dei = 0;
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      const double drho = wdot[n] * P->mw[n] * 1e6 * dt;
      dei += -P->lo[n][5] * drho * P->Ru / P->mw[n];
      r[n] += drho;
    }
    chem_epilogue<NS>(N, P, U, Q, rhoi, p, NP, r, dei);
  } else if (MODE == 0) {
    double A[NS][NS], bb[NS], x[NS];
    production_rate_at<NS, true, K>(N, P, sc, T0, A, wdot);
#pragma unroll
    for (int l = 0; l < NS; ++l)
#pragma unroll
      for (int n = 0; n < NS; ++n)
        A[n][l] = (n == l ? 1.0 : 0.0) - A[n][l] * P->mw[n] / P->mw[l] * dt;
#pragma unroll
    for (int n = 0; n < NS; ++n) bb[n] = wdot[n] * P->mw[n] * 1e6 * dt;
    gauss_solve<NS>(A, bb, x);
    double dei = 0;
    const double* lo_flat = &P->lo[0][0];
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      const double h6 = bug ? lo_flat[35 + n] : P->lo[n][5];
      dei += -h6 * x[n] * P->Ru / P->mw[n];
      r[n] += x[n];
    }
    chem_epilogue<NS>(N, P, U, Q, rhoi, p, NP, r, dei);
  } else {
    __shared__ NewtonLds<NS> L;
    const int lane = threadIdx.x;
    double rho_tot = 0.0;
#pragma unroll
    for (int n = 0; n < NS; ++n) rho_tot += r[n];
    double E0 = internal_energy<NS, true>(N, P, T0, r);
#pragma unroll
    for (int n = 0; n < NS; ++n) E0 += P->hfm[n] * r[n];
    const double T_lo = 0.5 * P->min_temp, T_hi = 1.5 * P->max_temp;
    // one step of dt; on failure restart from the initial state with twice
    // as many backward-Euler substeps (at most kNewtonMaxSub)
    int it = 0;
    bool ok = false;
    double T = T0;
    bool first = later != nullptr;
    for (int nsub = 1; nsub <= kNewtonMaxSub && !ok;) {
#pragma unroll
      for (int n = 0; n < NS; ++n) r[n] = rhoi[p + n * NP];  // written at the end only
      T = T0;
      ok = true;
      const double h = dt / nsub;
      const int limit = first ? min(maxiter, kNewtonFirst) : maxiter;
      for (int k = 0; k < nsub && ok; ++k)
        ok = be_solve<NS, K>(N, L, lane, P, r, T, h, E0, rho_tot, T_lo, T_hi, limit, rtol, ttol,
                             it);
      if (first && !ok) {  // left to k_newton_rows, from the start, or begun again here
        const int slot = atomicAdd(nlater, 1);
        if (slot < most) {
          later[slot] = (int32_t)id;
          return;
        }
        first = false;
        // a solve that had all its iterations or left the admissible set would
        // only fail again
        bool failed = maxiter <= kNewtonFirst || !(T > T_lo && T < T_hi);
#pragma unroll
        for (int n = 0; n < NS; ++n) failed = failed || !(r[n] > -rho_tot);
        if (failed) nsub *= 2;
        continue;
      }
      if (!ok) nsub *= 2;
    }
    if (!ok) {  // no admissible solution: the reactor is left unreacted
#pragma unroll
      for (int n = 0; n < NS; ++n) r[n] = rhoi[p + n * NP];
      it = -it;
    }
    if (iters) iters[id] = it;
    double dei = 0;
#pragma unroll
    for (int n = 0; n < NS; ++n) dei += -P->hfm[n] * (r[n] - rhoi[p + n * NP]);
    chem_epilogue<NS>(N, P, U, Q, rhoi, p, NP, r, dei);
  }
}

template <int NS, class K>
static void chem_k(f3d_ctx* c, int mode, double* U, double* Q, double* rhoi, double dt,
                   int maxiter, double rtol, double ttol, int32_t* iters, const int64_t* tag,
                   hipStream_t s, const int32_t* list, long nlist, int32_t* later, int32_t* nlater) {
  const long n = list ? nlist : (long)c->g.Nx * c->g.Ny * c->g.Nz;
  if (n <= 0) return;
  const int bug = c->bug_compat & 1;
  if (mode == 0)
    hipLaunchKernelGGL((k_chem<NS, 0, K>), dim3(nblocks(n)), dim3(kBlock), 0, s, U, Q, rhoi, dt,
                       maxiter, rtol, ttol, iters, tag, c->dparams, c->g, bug, list, n, nullptr,
                       nullptr, 0);
  else if (mode == 1)
    hipLaunchKernelGGL((k_chem<NS, 1, K>), dim3(nblocks(n)), dim3(kBlock), 0, s, U, Q, rhoi, dt,
                       maxiter, rtol, ttol, iters, tag, c->dparams, c->g, bug, list, n, nullptr,
                       nullptr, 0);
  else
    hipLaunchKernelGGL((k_chem<NS, 2, K>), dim3(nblocks(n, chem_block(2))), dim3(chem_block(2)),
                       0, s, U, Q, rhoi, dt, maxiter, rtol, ttol, iters, tag, c->dparams, c->g, bug,
                       list, n, later, nlater, rows_most(n));
}

// the list pass's slow cells: as many waves as the device holds stride over them
template <class T>
static void launch_rows(f3d_ctx* c, double* U, double* Q, double* rhoi, double dt, int maxiter,
                        double rtol, double ttol, hipStream_t s, long nlist,
                        const int32_t* later, const int32_t* nlater) {
  const int cap = rows_most(nlist);
  const long most = std::min(nlist, (long)cap);
  const long nb = std::min(resident_blocks(&k_newton_rows<T>, 64, &c->rows_blocks),
                           (most + kRowCells - 1) / kRowCells);
  hipLaunchKernelGGL((k_newton_rows<T>), dim3((unsigned)nb), dim3(64), 0, s, U, Q, rhoi, dt,
                     maxiter, rtol, ttol, c->dparams, c->g, kNewtonMaxSub, later, nlater, cap);
}

// the compiled-in tables of the context's mechanism when it is one of the
// shipped ones (f3d_create compares every entry), else the parameter block
template <int NS>
static void chem_ns(f3d_ctx* c, int mode, double* U, double* Q, double* rhoi, double dt,
                    int maxiter, double rtol, double ttol, int32_t* iters, const int64_t* tag,
                    hipStream_t s, const int32_t* list, long nlist, int32_t* later, int32_t* nlater) {
  if constexpr (NS == MechH2LiDryer::NS) {
    if (c->kin_table == F3D_KIN_H2_LIDRYER) {
      chem_k<NS, KinCT<MechH2LiDryer>>(c, mode, U, Q, rhoi, dt, maxiter, rtol, ttol, iters, tag,
                                       s, list, nlist, later, nlater);
      if (later && nlist > 0)
        launch_rows<MechH2LiDryer>(c, U, Q, rhoi, dt, maxiter, rtol, ttol, s, nlist, later, nlater);
      return;
    }
  }
  if constexpr (NS == MechAir5::NS) {
    if (c->kin_table == F3D_KIN_AIR5) {
      chem_k<NS, KinCT<MechAir5>>(c, mode, U, Q, rhoi, dt, maxiter, rtol, ttol, iters, tag, s,
                                  list, nlist, later, nlater);
      if (later && nlist > 0)
        launch_rows<MechAir5>(c, U, Q, rhoi, dt, maxiter, rtol, ttol, s, nlist, later, nlater);
      return;
    }
  }
  chem_k<NS, KinRT>(c, mode, U, Q, rhoi, dt, maxiter, rtol, ttol, iters, tag, s, list, nlist, nullptr,
                    nullptr);
}

int launch_chem(f3d_ctx* c, int mode, double* U, double* Q, double* rhoi, double dt,
                int maxiter, double rtol, double ttol, int32_t* iters, const int64_t* tag,
                hipStream_t s, const int32_t* list, long nlist, int32_t* later,
                int32_t* nlater) {
  if (mode == 0 && (c->bug_compat & 1) && c->g.Ns < 6) {
    set_error("bug_compat coeffs_lo[n,6] read needs Ns >= 6 (it reads past the array for Ns < 6)");
    return F3D_ERR_ARG;
  }
  if (rows_most(nlist) == 0) later = nullptr;
  switch (c->g.Ns) {
    case 5: chem_ns<5>(c, mode, U, Q, rhoi, dt, maxiter, rtol, ttol, iters, tag, s, list, nlist, later, nlater); break;
    case 9: chem_ns<9>(c, mode, U, Q, rhoi, dt, maxiter, rtol, ttol, iters, tag, s, list, nlist, later, nlater); break;
    default: set_error("chemistry: Ns must be 5 or 9"); return F3D_ERR_UNSUPPORTED;
  }
  return hip_check(hipGetLastError(), "chem");
}

}  // namespace f3d

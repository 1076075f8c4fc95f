// Finite-rate chemistry model on the device (shared by the exact kernels
// and the surrogate's fallback): ChemModel / Reaction arithmetic of
// ucs/chem.tcc:575-583 and ucs/reaction.tcc:607-856 in FP64.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/pcfd_chem.h"

namespace pcfd {

constexpr int kChemBlock = 128;
constexpr double kUnivR = 8.31447215;  // J/(mol K), ucs/chem_constants.h:5

struct ChemDev {
  int ns, nr;
  double mw[PCFD_CHEM_MAXS];
  double lo[PCFD_CHEM_MAXS][7], hi[PCFD_CHEM_MAXS][7];
  int type[PCFD_CHEM_MAXR], tb[PCFD_CHEM_MAXR], nloc[PCFD_CHEM_MAXR], loc[PCFD_CHEM_MAXR][PCFD_CHEM_MAXS];
  double A[PCFD_CHEM_MAXR], EA[PCFD_CHEM_MAXR], n[PCFD_CHEM_MAXR];
  double nup[PCFD_CHEM_MAXR][PCFD_CHEM_MAXS], nupp[PCFD_CHEM_MAXR][PCFD_CHEM_MAXS],
      eff[PCFD_CHEM_MAXR][PCFD_CHEM_MAXS];
  double ref_density, ref_time, ref_temperature;
  // per reaction, formed once from the above: net coefficient of every species
  // (its first local occurrence's) and their sum over the local list
  double net[PCFD_CHEM_MAXR][PCFD_CHEM_MAXS], nu[PCFD_CHEM_MAXR];
};

// Powers come in two forms.
//
// LibPow calls pow for every exponent, as the reference does.  The finite-rate
// solver keeps it, in the surrogate's exact fallback too: its source Jacobian
// differences two sources 1e-8 apart, so a last bit of a power is a part in 1e8
// of an entry, and of 200 solves of the reacting bump from random states two
// answered the other form's last bits with more than 2e-7 of a value in their
// result.
//
// ProductPow, for the calls that return rates, sources and Jacobians: the small
// whole exponents that mass action is made of are products -- 1 and x are pow's
// results, x*x is rounded once, the cube's second rounding is corrected -- and the
// halves that Arrhenius rates use come from sqrt(T), each corrected by what its
// roundings left out, so that all are within a hair of half a unit.  (A pow is
// some 200 instructions; with them source and Jacobian of 400k five-species cells
// took 1.58 ms, with products, rate constants shared by the columns and whole-line
// stores 0.24 ms.)
//
// isWholeNumber (ucs/macros.h:24-30); integer exponents go through pow of
// the promoted integer like the reference's pow(Type, Int)
struct LibPow {
  static __device__ __forceinline__ double conc(double x, double e) {
    const int up = (int)(e + 0.5), flat = (int)e;
    return pow(x, up == flat ? (double)flat : e);
  }
  static __device__ __forceinline__ double temp(double T, double n) { return pow(T, n); }
};

struct ProductPow {
  static __device__ __forceinline__ double conc(double x, double e) {
    const int up = (int)(e + 0.5), flat = (int)e;
    if (up == flat) e = (double)flat;
    if (e == 0.0) return 1.0;
    if (e == 1.0) return x;
    if (e == 2.0) return x * x;
    if (e == -1.0) return 1.0 / x;
    if (e == 3.0) {
      const double x2 = x * x, r = x2 * x;
      const double c = __builtin_fma(x2, x, __builtin_fma(x, x, -x2) * x);
      return __builtin_isinf(x2) || __builtin_isnan(c) ? r : c;
    }
    return pow(x, e);
  }
  static __device__ __forceinline__ double temp(double T, double n) {
    if (n == 0.0) return 1.0;
    if (n == 1.0) return T;
    if (n == -1.0) return 1.0 / T;
    // the corrections' products must neither overflow nor vanish
    const bool plain = T > 1.0e-100 && T < 1.0e100;
    if (plain && (fabs(n) == 0.5 || fabs(n) == 1.5)) {
      const double s = sqrt(T), ds = __builtin_fma(-s, s, T) * (0.5 / s);  // sqrt(T) = s + ds
      if (n == 0.5) return s;
      double p = s, dp = ds;  // T^|n| = p + dp
      if (fabs(n) == 1.5) {
        p = T * s;
        dp = __builtin_fma(T, s, -p) + T * ds;
        if (n == 1.5) return p + dp;
      }
      const double y = 1.0 / p;
      return __builtin_fma(y, __builtin_fma(-p, y, 1.0) - dp * y, y);
    }
    return pow(T, n);
  }
};

template <typename P>
__device__ __forceinline__ double kf_of(const ChemDev& m, int r, double T) {
  const double A = m.A[r], EA = m.EA[r], n = m.n[r];
  switch (m.type[r]) {
    case 0: return (A * exp(-EA / (kUnivR * T)));
    case 1: return (A * P::temp(T, n) * exp(-EA / (kUnivR * T)));
    case 2: return (A * P::temp(T, n) * exp(-EA / T));
    case 3: return (A * P::temp(T, n));
  }
  return -999.0;
}

// GetEquilibriumReactionRate (ucs/reaction.tcc:628-679); lnT = log(T)
template <typename P>
__device__ __forceinline__ double kc_of(const ChemDev& m, int r, double T, double lnT) {
  double d[7] = {0, 0, 0, 0, 0, 0, 0};
  const bool high = T > 1000.0;  // GetThermoCoeff: pinned ranges pick the same set
  for (int i = 0; i < m.nloc[r]; ++i) {
    const int s = m.loc[r][i];
    const double* a = high ? m.hi[s] : m.lo[s];
    const double dnu = m.nupp[r][i] - m.nup[r][i];
#pragma unroll
    for (int k = 0; k < 7; ++k) d[k] += dnu * a[k];
  }
  const double Kp =
      exp(d[0] * (lnT - 1.0) + T * (d[1] / 2.0 + T * (d[2] / 6.0 + T * (d[3] / 12.0 + d[4] / 20.0 * T))) -
          d[5] / T + d[6]);
  double Kc = Kp;
  if (!(fabs(m.nu[r]) < 1.0e-15)) Kc *= P::conc(101325.0 / (kUnivR * T), m.nu[r]);
  return Kc;
}

// The functions below take the species count as a template argument (0: the
// model's at run time): with it known the per-species arrays stay in
// registers, where an indexed array would live in scratch memory.
template <int NS>
__device__ __forceinline__ int nspecies_of(const ChemDev& m) {
  return NS > 0 ? NS : m.ns;
}

// v[k] for a k that is the same in every lane
template <int NS>
__device__ __forceinline__ double pick(const double* v, int k) {
  if constexpr (NS == 0) return v[k];
  double x = v[0];
#pragma unroll
  for (int i = 1; i < NS; ++i) x = k == i ? v[i] : x;
  return x;
}

// GetMassProductionRates for one state: rhoi (kg/m^3), T (K) -> wdot (kg/m^3/s)
template <int NS, typename P = ProductPow>
__device__ inline void wdot_of(const ChemDev& m, const double* rhoi, double T, double* wdot) {
  constexpr int MS = NS > 0 ? NS : PCFD_CHEM_MAXS;
  const int ns = nspecies_of<NS>(m);
  double X[MS];
#pragma unroll
  for (int k = 0; k < MS; ++k) {
    if (k >= ns) break;
    X[k] = rhoi[k] / m.mw[k];
    wdot[k] = 0.0;
  }
  const double lnT = log(T);
  for (int r = 0; r < m.nr; ++r) {
    const double Kf = kf_of<P>(m, r, T);
    const double Kb = Kf / kc_of<P>(m, r, T, lnT);
    double pf = 1.0, pd = 1.0;
    for (int k = 0; k < m.nloc[r]; ++k) {
      const double x = pick<NS>(X, m.loc[r][k]);
      pf *= P::conc(x, m.nup[r][k]);
      pd *= P::conc(x, m.nupp[r][k]);
    }
    double Mc = 1.0;
    if (m.tb[r]) {
      Mc = 0.0;
#pragma unroll
      for (int k = 0; k < MS; ++k) {
        if (k >= ns) break;
        Mc += X[k];
      }
      for (int k = 0; k < m.nloc[r]; ++k) Mc += (m.eff[r][k] - 1.0) * pick<NS>(X, m.loc[r][k]);
    }
    const double net = Kf * pf - Kb * pd;
#pragma unroll
    for (int i = 0; i < MS; ++i) {
      if (i >= ns) break;
      const double nu = m.net[r][i];
      if (nu == 0.0) continue;  // AlmostEqualRelative(nu, 0, 1e-15): contributes +0
      double w = nu * Mc * net;
      w *= m.mw[i];
      wdot[i] += w;
    }
  }
}

// SourceTerm (ucs/compressibleFR.tcc:1276-1312) on the FR state
template <int NS, typename P = ProductPow>
__device__ inline void source_of(const ChemDev& m, const double* Q, double vol, double* src) {
  constexpr int MS = NS > 0 ? NS : PCFD_CHEM_MAXS;
  const int ns = nspecies_of<NS>(m);
  double rhoi[MS], w[MS];
  const double T = Q[ns + 3] * m.ref_temperature;
#pragma unroll
  for (int i = 0; i < MS; ++i) {
    if (i >= ns) break;
    rhoi[i] = Q[i] * m.ref_density;
  }
  wdot_of<NS, P>(m, rhoi, T, w);
#pragma unroll
  for (int i = 0; i < MS; ++i) {
    if (i >= ns) break;
    w[i] /= (m.ref_density / m.ref_time);
    src[i] = vol * w[i];
  }
}

// wdot_of of a state and of its ns copies with one species density raised
// (copy c holds rhop[c] in place of rhoi[c]).  The rate constants are
// functions of T alone and a reaction's mass-action factors of the species
// a copy leaves alone are the state's, so both are evaluated once per
// reaction and shared; every copy's products and sums, in their order, are
// wdot_of's, so w[(1 + c) * ns + i] equals wdot_of of copy c bit for bit
// and w[i] that of the state.  w [(ns + 1) * ns].
template <int NS, typename P = ProductPow>
__device__ inline void wdot_rho_columns(const ChemDev& m, const double* rhoi, const double* rhop, double T,
                                        double* w) {
  constexpr int MS = NS > 0 ? NS : PCFD_CHEM_MAXS;
  const int ns = nspecies_of<NS>(m);
  double X[MS], Xp[MS];
#pragma unroll
  for (int k = 0; k < MS; ++k) {
    if (k >= ns) break;
    X[k] = rhoi[k] / m.mw[k];
    Xp[k] = rhop[k] / m.mw[k];
  }
#pragma unroll
  for (int k = 0; k < (MS + 1) * MS; ++k) {
    if (k >= (ns + 1) * ns) break;
    w[k] = 0.0;
  }
  const double lnT = log(T);
  for (int r = 0; r < m.nr; ++r) {
    const double Kf = kf_of<P>(m, r, T);
    const double Kb = Kf / kc_of<P>(m, r, T, lnT);
    // copy s has species s - 1 raised (0: the state itself)
    double pf[MS + 1], pd[MS + 1], Mc[MS + 1];
#pragma unroll
    for (int s = 0; s <= MS; ++s) {
      if (s > ns) break;
      pf[s] = pd[s] = Mc[s] = 1.0;
      if (m.tb[r]) {
        Mc[s] = 0.0;
#pragma unroll
        for (int k = 0; k < MS; ++k) {
          if (k >= ns) break;
          Mc[s] += k == s - 1 ? Xp[k] : X[k];
        }
      }
    }
    for (int k = 0; k < m.nloc[r]; ++k) {
      const int l = m.loc[r][k];
      const double x = pick<NS>(X, l), xp = pick<NS>(Xp, l);
      const double eu = m.nup[r][k], ed = m.nupp[r][k];
      const double fu = P::conc(x, eu), fup = P::conc(xp, eu), fd = P::conc(x, ed), fdp = P::conc(xp, ed);
      const double w1 = m.eff[r][k] - 1.0;
#pragma unroll
      for (int s = 0; s <= MS; ++s) {
        if (s > ns) break;
        const bool raised = l == s - 1;
        pf[s] *= raised ? fup : fu;
        pd[s] *= raised ? fdp : fd;
        if (m.tb[r]) Mc[s] += w1 * (raised ? xp : x);
      }
    }
#pragma unroll
    for (int i = 0; i < MS; ++i) {
      if (i >= ns) break;
      const double nu = m.net[r][i];
      if (nu == 0.0) continue;
#pragma unroll
      for (int s = 0; s <= MS; ++s) {
        if (s > ns) break;
        const double net = Kf * pf[s] - Kb * pd[s];
        double v = nu * Mc[s] * net;
        v *= m.mw[i];
        w[s * ns + i] += v;
      }
    }
  }
}

// source_of of the FR state Q and of its ns copies with Q[c] raised by h
// (the species columns of the forward-difference source Jacobian):
// src[i] is the state's, src[(1 + c) * ns + i] copy c's, each bit for bit
// what source_of gives.  src [(ns + 1) * ns].
template <int NS, typename P = ProductPow>
__device__ inline void source_rho_columns(const ChemDev& m, const double* Q, double h, double vol, double* src) {
  constexpr int MS = NS > 0 ? NS : PCFD_CHEM_MAXS;
  const int ns = nspecies_of<NS>(m);
  double rhoi[MS], rhop[MS];
  const double T = Q[ns + 3] * m.ref_temperature;
#pragma unroll
  for (int i = 0; i < MS; ++i) {
    if (i >= ns) break;
    rhoi[i] = Q[i] * m.ref_density;
    rhop[i] = (Q[i] + h) * m.ref_density;
  }
  wdot_rho_columns<NS, P>(m, rhoi, rhop, T, src);
#pragma unroll
  for (int k = 0; k < (MS + 1) * MS; ++k) {
    if (k >= (ns + 1) * ns) break;
    double v = src[k];
    v /= (m.ref_density / m.ref_time);
    src[k] = vol * v;
  }
}

}  // namespace pcfd

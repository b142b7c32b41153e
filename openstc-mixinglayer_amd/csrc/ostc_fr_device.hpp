// ostc_fr_device.hpp -- point physics of the finite-rate mixture path on the
// device: NASA-7 thermodynamics, mixture-averaged transport, finite-rate
// chemistry, the temperature Newton iteration and the Roe-averaged
// characteristic decomposition of a face.  Templated on the species count NS
// so per-species temporaries live in registers; the coefficient tables
// (ostc_mech_tables) are read through a kernel-argument pointer, which the
// compiler turns into scalar loads wherever the index is wave-uniform.
//
// Arithmetic follows the reference routine named beside each function, in
// its expression order (the library is built with -ffp-contract=off).
#pragma once
#include <hip/hip_runtime.h>

#include "openstc/mech.h"
#include "ostc_select.hpp"
#include "ostc_weno.hpp"

namespace ostc {
namespace fr {

constexpr double kRu = 8314.462618;   // src/Constants.h:19
constexpr double kPatm = 101325;      // src/Constants.h:26

// The mechanism's tables and what the kernels would otherwise derive from
// them at every point: quotients by the molar masses (an IEEE division costs
// 11 instructions), the NASA-7 polynomials scaled and in Horner order, the
// constant factors of the collision integrals.  Filled on the host
// (derive_tables).
struct Tab : ostc_mech_tables {
  double imw[OSTC_MAX_SPEC], r[OSTC_MAX_SPEC];  // 1 / W, R_u / W
  double mid_lo, mid_hi, low_max;               // least and largest t_mid, largest t_low
  double cpp[2][OSTC_MAX_SPEC][5];              // cp = sum cpp[k] t^k; [0] low range, [1] high range
  double h0[2][OSTC_MAX_SPEC];                  // h = h0 + sum cpp[k] t^(k+1) / (k+1)
  double gp[2][OSTC_MAX_SPEC][7];               // g/RT = gp[0] (1 - log t) + sum_1..4 gp[k] t^k + gp[5]/t + gp[6]
  double vis_k[OSTC_MAX_SPEC];                  // lj_potent_inv^-0.145
  double dif_k[OSTC_MAX_SPEC][OSTC_MAX_SPEC];   // kb_over_eps_jk^-0.145
  double inv_bin[OSTC_MAX_SPEC][OSTC_MAX_SPEC]; // 1 / binary_diffusivity_coeff
  double dnu[OSTC_MAX_REAC][OSTC_MAX_SPEC];     // stoi_b - stoi_f
  int use_kc;                                   // some reaction takes kb from equilibrium
};

// Calls f(i, c, tt) for every species with the row index of its range and the
// temperature at which its polynomials are evaluated (not below t_low, beyond
// which h continues linearly).  A wave whose lanes all lie in one range, as
// nearly every wave does, reads the coefficients by scalar loads (range is the
// same for the wave); a mixed wave selects them per lane.  A NaN temperature
// stays one (fmax would make it t_low and every property finite).
template <int NS, class F>
__device__ __forceinline__ void each_species(const Tab* __restrict__ T, double t, F f) {
  if (__all(t >= T->mid_hi)) {
#pragma unroll
    for (int i = 0; i < NS; ++i) f(i, 1, t);
  } else if (__all(t < T->mid_lo)) {
#pragma unroll
    for (int i = 0; i < NS; ++i) f(i, 0, t < T->t_low[i] ? T->t_low[i] : t);
  } else {
#pragma unroll
    for (int i = 0; i < NS; ++i) f(i, t >= T->t_mid[i] ? 1 : 0, t < T->t_low[i] ? T->t_low[i] : t);
  }
}

__device__ __forceinline__ double poly_cp(const double* c, double t) {
  return __builtin_fma(t, __builtin_fma(t, __builtin_fma(t, __builtin_fma(t, c[4], c[3]), c[2]), c[1]), c[0]);
}
__device__ __forceinline__ double poly_h(const double* c, double t) {
  return __builtin_fma(t, poly_cp(c, t), c[5]);
}

// One species' enthalpy and heat capacity in the reference's operation order
// and rounding: what the face decomposition reads has to match it bit by bit
// (see char_face).  The quotients are the shorter sequences of div64 with the
// same result.
__device__ __forceinline__ double species_cp(const double* c, double t) {
  const double t2 = t * t, t3 = t2 * t, t4 = t3 * t;
  return c[0] + c[1] * t + c[2] * t2 + c[3] * t3 + c[4] * t4;
}
__device__ __forceinline__ double species_h(const double* c, double t) {
  const double t2 = t * t, t3 = t2 * t, t4 = t3 * t, t5 = t4 * t;
  return c[0] * t + 0.5 * c[1] * t2 + div64(c[2] * t3, 3.0, 1.0 / 3.0) + 0.25 * c[3] * t4 + 0.2 * c[4] * t5 + c[5];
}
__device__ __forceinline__ const double* coefficients(const Tab* __restrict__ T, int i, int side) {
  return side ? T->high_coeff[i] : T->low_coeff[i];
}

// compute_enthalpy (Combustion2Part), src/Thermo.cu:130-148
template <int NS>
__device__ __forceinline__ void enthalpy(const Tab* __restrict__ T, double t, double* h) {
  each_species<NS>(T, t, [&](int i, int side, double tt) {
    const double* c = coefficients(T, i, side);
    double v = species_h(c, tt);
    if (t < T->t_low[i]) v += species_cp(c, tt) * (t - tt);
    h[i] = v * T->r[i];
  });
}

// compute_enthalpy_and_cp (Combustion2Part), src/Thermo.cu:150-172
template <int NS>
__device__ __forceinline__ void enthalpy_cp(const Tab* __restrict__ T, double t, double* h, double* cp) {
  each_species<NS>(T, t, [&](int i, int side, double tt) {
    const double* c = coefficients(T, i, side);
    const double k = species_cp(c, tt);
    double v = species_h(c, tt);
    if (t < T->t_low[i]) v += k * (t - tt);
    h[i] = v * T->r[i];
    cp[i] = k * T->r[i];
  });
}

// compute_cp (Combustion2Part), src/Thermo.cu:174-188
template <int NS>
__device__ __forceinline__ void heat_capacity(const Tab* __restrict__ T, double t, double* cp) {
  each_species<NS>(T, t, [&](int i, int side, double tt) {
    cp[i] = species_cp(coefficients(T, i, side), tt) * T->r[i];
  });
}

// compute_gibbs_div_rt (Combustion2Part), src/Thermo.cu:190-208
template <int NS>
__device__ __forceinline__ void gibbs_rt(const Tab* __restrict__ T, double t, double log_t, double t_inv, double* g) {
  each_species<NS>(T, t, [&](int i, int side, double tt) {
    const double* c = T->gp[side][i];
    const bool below = tt > t;  // below the table: the functions at t_low
    const double ti = below ? rcp64(tt) : t_inv, lt = below ? log(tt) : log_t;
    const double p = tt * __builtin_fma(tt, __builtin_fma(tt, __builtin_fma(tt, c[4], c[3]), c[2]), c[1]);
    g[i] = __builtin_fma(c[0], 1.0 - lt, p) + __builtin_fma(c[5], ti, c[6]);
  });
}

// compute_transport_property, src/Transport.cu:43-136, with compute_Omega_D
// (:168-170).  Only the off-diagonal binary diffusivities are formed: the
// mixture-averaged rho D_k never reads the diagonal.  (T / scale)^-0.145 of
// every species and pair is T^-0.145 (one logarithm and one exponential a
// point) times a tabulated factor, sqrt(mu_m / mu_n) is a product of 9 roots
// and 9 reciprocals, and a pair's diffusivity enters by its reciprocal.
// 256x128x64 nodes: properties 0.65 -> 0.31 ms a stage.
template <int NS>
__device__ __forceinline__ void transport(const Tab* __restrict__ T, double t, double p, double rho, const double* Y,
                                          double mw_total, const double* cp, double* mu_out, double* lambda_out,
                                          double* rho_d) {
  const double t145 = exp(-0.145 * log(t)), root_t = sqrt64(t);
  double X[NS], vis[NS], s[NS], is[NS];
#pragma unroll
  for (int l = 0; l < NS; ++l) {
    X[l] = Y[l] * mw_total * T->imw[l];
    const double d = __builtin_fma(t, T->lj_potent_inv[l], 0.5);
    vis[l] = T->vis_coeff[l] * root_t * rcp64(__builtin_fma(1.147 * T->vis_k[l], t145, rcp64(d * d)));
    s[l] = sqrt64(vis[l]);
    is[l] = rcp64(s[l]);
  }
  double viscosity = 0, conductivity = 0;
#pragma unroll
  for (int m = 0; m < NS; ++m) {
    double phi = X[m];
#pragma unroll
    for (int n = 0; n < NS; ++n)
      if (m != n) {
        const double q = __builtin_fma(s[m] * is[n], T->wj_div_wi_to_one4th[m][n], 1.0);
        phi = __builtin_fma(q * q * T->sqrt_wi_div_wj_pl1_mul8[m][n], X[n], phi);
      }
    const double vx = vis[m] * X[m];
    viscosity = __builtin_fma(vx, rcp64(phi), viscosity);
    const double lx = vx * __builtin_fma(1.25, T->r[m], cp[m]);
    conductivity = __builtin_fma(lx, rcp64(__builtin_fma(1.065, phi, -0.065 * X[m])), conductivity);
  }
  *mu_out = viscosity;
  *lambda_out = conductivity;
  constexpr double eps{1e-12};
  double num[NS], den[NS];
#pragma unroll
  for (int l = 0; l < NS; ++l) num[l] = den[l] = 0;
#pragma unroll
  for (int m = 0; m < NS; ++m)
#pragma unroll
    for (int n = m + 1; n < NS; ++n) {
      const double d = __builtin_fma(t, T->kb_over_eps_jk[m][n], 0.5);
      const double w = __builtin_fma(T->dif_k[m][n], t145, rcp64(d * d)) * T->inv_bin[m][n];  // t^1.5/p / D_mn
      num[m] = __builtin_fma(X[n] + eps, T->mw[n], num[m]);
      den[m] = __builtin_fma(X[n] + eps, w, den[m]);
      num[n] = __builtin_fma(X[m] + eps, T->mw[m], num[n]);
      den[n] = __builtin_fma(X[m] + eps, w, den[n]);
    }
  const double scale = rho * t * root_t * rcp64(p * mw_total);
#pragma unroll
  for (int l = 0; l < NS; ++l) rho_d[l] = scale * num[l] * rcp64(den[l]);
}

// The point's temperature as arrhenius needs it: 1 / t and log t, each with the
// remainder that its rounding left.
struct Temp { double t, inv, inv_lo, log, log_lo; };
__device__ __forceinline__ Temp temp_of(double t) {
  Temp q;
  q.t = t;
  q.inv = rcp64(t);
  q.inv_lo = __builtin_fma(-t, q.inv, 1.0) * q.inv;
  q.log = log(t);
  q.log_lo = (t - exp(q.log)) * q.inv;
  return q;
}

// arrhenius, src/FiniteRateChem.cu:104-106: A * T^b * exp(-Ea/T) as one
// exponential of b log T - Ea / T.  The exponent reaches 170 (Ea / T at
// 300 K), so its rounding alone would cost 2e-14 of the rate, as the quotient
// in exp(-Ea / T) does: products, sum and the operands' remainders are carried
// to first order.  A reaction without either factor skips it (the tables make
// the test wave-uniform).
__device__ __forceinline__ double arrhenius(const Temp& q, double A, double b, double Ea) {
  if (b == 0 && Ea == 0) return A;
  const double p1 = b * q.log, p2 = Ea * q.inv;
  double lo = __builtin_fma(b, q.log, -p1) - __builtin_fma(Ea, q.inv, -p2);
  lo += __builtin_fma(b, q.log_lo, -(Ea * q.inv_lo));
  const double s = p1 - p2, back = s - p1;
  lo += (p1 - (s - back)) - (p2 + back);
  const double e = A * exp(s);
  return __builtin_fma(e, lo, e);
}

// c^nu for a stoichiometric coefficient: pow(c, 0) = 1 and pow(c, 1) = c
// exactly; c^2 is the correctly rounded square.
__device__ __forceinline__ double stoich_pow(double c, int nu) {
  if (nu == 1) return c;
  if (nu == 2) return c * c;
  return pow(c, (double)nu);
}

// finite_rate_chemistry (explicit), src/FiniteRateChem.cu:7-58 with
// forward_reaction_rate :60-102, backward_reaction_rate :108-150,
// rate_of_progress :152-177, chemical_source :179-195.  The reaction loop
// runs over the runtime reaction count; its tables are wave-uniform.  A
// species takes its net rate times stoi_b - stoi_f, and kb = kf exp(dg) / tp
// needs no division.
template <int NS>
__device__ void chemistry(const Tab* __restrict__ T, double rho, double t, const double* Y, double* omega) {
  const int nr = T->n_reac;
  double c[NS];
#pragma unroll
  for (int l = 0; l < NS; ++l) c[l] = rho * Y[l] * (T->imw[l] * 1e-3);
  const Temp q = temp_of(t);
  double g[NS];
  gibbs_rt<NS>(T, t, q.log, q.inv, g);
  constexpr double temp_p = kPatm / kRu * 1e-3;
  const double temp_t = temp_p * q.inv, inv_temp_t = t * (1.0 / temp_p);
#pragma unroll
  for (int l = 0; l < NS; ++l) omega[l] = 0;
  const bool use_kc = T->use_kc != 0;
  for (int i = 0; i < nr; ++i) {
    const int type = T->label[i];
    double kf = arrhenius(q, T->A[i], T->b[i], T->Ea[i]);
    double cc{0};
    if (type > 3) {
#pragma unroll
      for (int l = 0; l < NS; ++l) cc = __builtin_fma(c[l], T->third_body_coeff[i][l], cc);
    }
    if (type == 3) {
      kf += arrhenius(q, T->A2[i], T->b2[i], T->Ea2[i]);
    } else if (type == 4) {
      kf *= cc;
    } else if (type > 4) {
      const double kf_low = arrhenius(q, T->A2[i], T->b2[i], T->Ea2[i]);
      const double kf_high = kf;
      const double reduced_pressure = kf_low * cc / kf_high;
      double F = 1.0;
      if (type > 5) {
        double f_cent = (1 - T->troe_alpha[i]) * exp(-t / T->troe_t3[i]) + T->troe_alpha[i] * exp(-t / T->troe_t1[i]);
        if (type == 7) f_cent += exp(-T->troe_t2[i] / t);
        const double logFc = log10(f_cent);
        const double cc2 = -0.4 - 0.67 * logFc;
        const double n = 0.75 - 1.27 * logFc;
        const double logPr = log10(reduced_pressure);
        const double tempo = (logPr + cc2) / (n - 0.14 * (logPr + cc2));
        F = exp10(logFc / (1.0 + tempo * tempo));
      }
      kf = kf_high * reduced_pressure / (1.0 + reduced_pressure) * F;
    }
    double kb = 0;
    if (type != 0) {
      if (T->rev_type[i] == 1) {
        kb = arrhenius(q, T->A2[i], T->b2[i], T->Ea2[i]);
        if (type == 4) kb *= cc;
      }
      // then every reversible label takes kb from equilibrium (the
      // reference's test at src/FiniteRateChem.cu:140 only excludes labels 0
      // and 2), REV included
      if (use_kc) {
        double d_gibbs{0};
#pragma unroll
        for (int l = 0; l < NS; ++l) d_gibbs = __builtin_fma(g[l], T->dnu[i][l], d_gibbs);
        const int ord = T->order[i];
        const double tp = ord == 0 ? 1.0 : (ord == 1 ? inv_temp_t : (ord == -1 ? temp_t : pow(temp_t, (double)-ord)));
        kb = kf * (tp * exp(d_gibbs));
      }
    }
    // rate of progress: factors with a zero coefficient are exactly 1
    double q1 = kf, q2 = kb;
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const int nf = T->stoi_f[i][j], nb = T->stoi_b[i][j];
      if (nf != 0) q1 *= stoich_pow(c[j], nf);
      if (type != 0 && nb != 0) q2 *= stoich_pow(c[j], nb);
    }
    const double net = q1 - q2;
#pragma unroll
    for (int l = 0; l < NS; ++l) omega[l] = __builtin_fma(net, T->dnu[i][l], omega[l]);
  }
#pragma unroll
  for (int l = 0; l < NS; ++l) omega[l] *= T->mw[l] * 1e+3;
}

// compute_temperature_and_pressure, src/FieldOperation.cu:3-40.  While every
// lane of the wave stays in one range of the polynomials, the iteration runs
// on the mixture's own polynomial, whose coefficients are summed once.
template <int NS>
__device__ __forceinline__ double temperature(const Tab* __restrict__ T, double e, const double* Y, double gas_const,
                                              double t) {
  const int side = __all(t >= T->mid_hi) ? 1 : (__all(t < T->mid_lo && t >= T->low_max) ? 0 : -1);
  double mc[5] = {0, 0, 0, 0, 0}, mh[6] = {0, 0, 0, 0, 0, 0};
  if (side >= 0) {
#pragma unroll
    for (int i = 0; i < NS; ++i) {
#pragma unroll
      for (int k = 0; k < 5; ++k) mc[k] = __builtin_fma(Y[i], T->cpp[side][i][k], mc[k]);
      mh[5] = __builtin_fma(Y[i], T->h0[side][i], mh[5]);
    }
    constexpr double inv[5]{1.0, 1.0 / 2, 1.0 / 3, 1.0 / 4, 1.0 / 5};
#pragma unroll
    for (int k = 0; k < 5; ++k) mh[k] = mc[k] * inv[k];
  }
  double err{1};
  int iter = 0;
  while (err > 1e-3 && iter++ < 1000) {
    double cp_tot{0}, h{0};
    if ((side == 1 && __all(t >= T->mid_hi)) || (side == 0 && __all(t < T->mid_lo && t >= T->low_max))) {
      cp_tot = poly_cp(mc, t);
      h = poly_h(mh, t);
    } else {
      double h_i[NS], cp_i[NS];
      enthalpy_cp<NS>(T, t, h_i, cp_i);
#pragma unroll
      for (int l = 0; l < NS; ++l) {
        cp_tot = __builtin_fma(cp_i[l], Y[l], cp_tot);
        h = __builtin_fma(h_i[l], Y[l], h);
      }
    }
    const double e_t = h - gas_const * t;
    const double t1 = t - (e_t - e) * rcp64(cp_tot - gas_const);
    err = fabs(1 - t1 / t);
    t = t1;
  }
  return t;
}

// total energy of a mixture point, compute_total_energy<FR>,
// src/FieldOperation.cuh:17-38
template <int NS>
__device__ __forceinline__ double total_energy(const Tab* __restrict__ T, double rho, double u, double v, double w,
                                               double p, double t, const double* Y) {
  double h[NS];
  enthalpy<NS>(T, t, h);
  const double V2 = u * u + v * v + w * w;
  double te = 0.5 * V2;
#pragma unroll
  for (int l = 0; l < NS; ++l) te += h[l] * Y[l];
  te *= rho;
  te -= p;
  return te;
}

}  // namespace fr
}  // namespace ostc

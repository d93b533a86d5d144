// contrib.hip -- the vertical-mixing contributors that are off at the
// reference defaults, on the packed level-major layout (X[k * P + p], k = 0
// the bed, one lane per column):
//
//   k_epbl     energetics-based planetary boundary layer (Reichl & Hallberg
//              2018), epbl_column_kernel (rdb_ocean_epbl.F90:931-1659): MLD
//              root-find around a downward interface sweep with the
//              closed-form energy solve and the embedded forward elimination;
//   k_coeff_tail  the rest of the coefficient build in one top-down pass:
//              PP81 (when EPBL runs), the EPBL merge into kv/kt (:1661-1688),
//              KV_ML_INVZ2 (rdb_ocean_vmix.F90:1716-1748), convective
//              adjustment (:1768-1799), the heat/salt split with double
//              diffusion (ddiff_iface, :1936-2028) and vmix_assemble.
//
// The EPBL sweep needs, per level, the pre-mixing T/S and the pressure-
// weighted PE and column-height sensitivities.  The reference fills six
// column work arrays once and re-reads them in every MLD iteration; here
// each iteration recomputes them on the fly while it walks down (the same
// pressure stack, summed in the same order, so the same bits): every
// iteration streams h, T and S only, and no work array is written.
#include "colphys_kernels.h"
#include "safe_math.h"

namespace colphys {

#define LV(arr, k) (arr)[(size_t)(k) * (size_t)P + (size_t)p]

namespace {

constexpr double H_NEGLECT = H_DIV_EPS;

// eos_specvol_derivs, Wright (1997) branch (rdb_eos.F90:1551-1622).
__device__ __forceinline__ void specvol_derivs(double T, double S, double p, double& dsv_dt, double& dsv_ds) {
  const double T_sq = T * T;
  const double p_0 = 5.790749e8 + 3.516535e6 * T + -4.002714e4 * T_sq + 2.084372e2 * T_sq * T + 5.944068e5 * S +
                     -9.643486e3 * S * T;
  const double lambda = 1.704853e5 + 7.904722e2 * T + -7.984422e0 * T_sq + 5.140652e-2 * T_sq * T +
                        -2.302158e2 * S + -3.079464e0 * S * T;
  const double dp0_dt = 3.516535e6 + 2.0 * -4.002714e4 * T + 3.0 * 2.084372e2 * T_sq + -9.643486e3 * S;
  const double dlam_dt = 7.904722e2 + 2.0 * -7.984422e0 * T + 3.0 * 5.140652e-2 * T_sq + -3.079464e0 * S;
  const double dp0_ds = 5.944068e5 + -9.643486e3 * T;
  const double dlam_ds = -2.302158e2 + -3.079464e0 * T;
  const double big_p = p + p_0;
  const double inv_p = 1.0 / big_p;
  const double inv_p2 = inv_p * inv_p;
  dsv_dt = 3.480336e-7 + dlam_dt * inv_p - lambda * dp0_dt * inv_p2;
  dsv_ds = -1.112733e-7 + dlam_ds * inv_p - lambda * dp0_ds * inv_p2;
}

__device__ __forceinline__ double cube(double x) { return (x * x) * x; }

// epbl_find_mstar (rdb_ocean_epbl.F90:630-688).
template <bool GEN>
__device__ __forceinline__ double find_mstar(const EpblParams& c, double b0, double ustar, double bld, double absf) {
  double mstar;
  const double absf_floor = fmx(absf, 1.0e-20);
  if (c.mstar_scheme == RDB_EPBL_MSTAR_OM4) {
    const double mstar_s = c.mstar_coef1 * sqrt(fmx(0.0, b0) / (ustar * ustar * absf_floor));
    double mstar_n = 0.0;
    if (ustar > absf_floor * bld) mstar_n = c.c_ek * sm::log(ustar / (absf_floor * fmx(bld, 1.0e-10)));
    mstar = fmx(mstar_s, fmn(1.25, mstar_n));
    if (c.mstar_cap > 0.0) mstar = fmn(c.mstar_cap, mstar);
  } else if (GEN && c.mstar_scheme == RDB_EPBL_MSTAR_RH18) {
    const double msn_term = c.cn2 * sm::exp(c.cn3 * bld * absf / ustar);
    const double mstar_n = c.cn1 * msn_term / (1.0 + msn_term);
    const double bp = fmx(0.0, b0);
    const double u5 = cube(ustar) * (ustar * ustar);
    const double mstar_s = c.cs1 * sm::pow(bp * bp * bld / (u5 * absf_floor), c.cs2);
    mstar = mstar_n + mstar_s;
    if (c.mstar_cap > 0.0) mstar = fmn(c.mstar_cap, mstar);
  } else {
    mstar = c.mstar_const;
  }
  if (c.mstar_conv_adj > 0.0) {
    const double t1 = -bld * fmn(0.0, b0);
    const double t2 = 2.0 * mstar * cube(ustar);
    if (t2 > 0.0)
      mstar = mstar * ((1.0 - c.mstar_conv_adj) * t1 + t2) / (t1 + t2);
    else
      mstar = mstar * (1.0 - c.mstar_conv_adj);
  }
  return mstar;
}

// epbl_mixlen_shape (:690-714).
template <bool GEN>
__device__ __forceinline__ double mixlen_shape(const EpblParams& c, double z, double mld_guess) {
  if (!c.mld_iteration || c.translay >= 1.0 || c.translay < 0.0 || mld_guess <= 0.0) return 1.0;
  const double fr = fmx(0.0, (mld_guess - z) / mld_guess);
  if (!GEN || c.mixlen_exponent == 2.0) return c.translay + (1.0 - c.translay) * fr * fr;
  return c.translay + (1.0 - c.translay) * sm::pow(fr, c.mixlen_exponent);
}

constexpr double LT_PI = 3.141592653589793116;

// epbl_lf17_wave_state (:716-765).
__device__ __noinline__ void lf17_wave_state(double ustar_w, double rho_ocn, double& ustokes, double& kphil) {
  const double ustar_air = ustar_w * sqrt(rho_ocn / 1.225);
  const double z0_smooth = 0.11 * 1.0e-6 / ustar_air;
  double u = ustar_air * sqrt(1000.0);
  bool converged = false;
  for (int itt = 1; itt <= 20; ++itt) {
    const double alpha_ch = fmn(0.028, 0.0017 * u + -0.005);
    const double z0w = fmx(z0_smooth + alpha_ch * (ustar_air * ustar_air) / GRAVITY, 1.0e-10);
    const double u_new = ustar_air * sm::log(10.0 / z0w) / 0.40;
    if (fabs(u_new - u) <= 1.0e-3 * u) {
      u = u_new;
      converged = true;
      break;
    }
    u = u_new;
  }
  if (!converged) u = 25.82 * ustar_air;
  ustokes = 0.0162 * u;
  const double hm0 = 0.0246 * u * u;
  const double f_mean = 1.296 * 0.877 * GRAVITY / (2.0 * LT_PI * 1.075 * u);
  const double vstokes = 0.125 * LT_PI * 0.667 * f_mean * hm0 * hm0;
  kphil = 0.176 * ustokes / fmx(vstokes, 1.0e-30);
}

__device__ __forceinline__ double one_m_exp_x(double x) {
  if (x < 1.0e-4) return 1.0 - x * (0.5 - x / 6.0);
  return (1.0 - sm::exp(-x)) / x;
}

// epbl_lf17_la (:767-804).
__device__ __noinline__ double lf17_la(double ustar_w, double zsl, double ustokes, double kphil) {
  const double xkz = kphil * zsl;
  const double root2kz = sqrt(2.0 * xkz);
  const double r1 = (0.302 - 1.68 * xkz) * one_m_exp_x(2.0 * xkz);
  const double r3 = (0.1264 + 0.64 * xkz) * one_m_exp_x(5.12 * xkz);
  double r5;
  if (root2kz > 1.0e-3) {
    const double ec1 = sm::erfc(root2kz);
    const double ec2 = sm::erfc(1.6 * root2kz);
    r5 = sqrt(LT_PI) * (root2kz * (-(0.84 * ec1) + 0.2 * ec2) + 0.1182 * (ec2 - ec1) / root2kz);
  } else {
    r5 = -(0.64 * sqrt(LT_PI) * root2kz) + (-0.14184 + 1.0839648 * root2kz * root2kz);
  }
  const double ustokes_sl = fmx(ustokes * (0.715 + r1 + r3 + r5), 1.0e-10);
  return sqrt(ustar_w / ustokes_sl);
}

// epbl_lt_enhance (:818-858).
__device__ __noinline__ double lt_enhance(const EpblParams& c, double la, double b0, double ustar, double bld,
                                          double absf, double mstar) {
  const double vk = c.von_karman;
  const double mld_ek = bld * absf / ustar;
  const double ek_ob = fabs(b0 * vk) / (fmx(absf, 1.0e-20) * ustar * ustar);
  const double mld_ob = fabs(bld * b0 * vk) / cube(ustar);
  double la_mod;
  if (b0 >= 0.0)
    la_mod = la * ((1.0 + fmx(-0.5, c.lac1 * mld_ek)) + c.lac4 * ek_ob + c.lac2 * mld_ob);
  else
    la_mod = la * ((1.0 + fmx(-0.5, c.lac1 * mld_ek)) + c.lac5 * ek_ob + c.lac3 * mld_ob);
  la_mod = fmx(la_mod, 1.0e-10);
  if (c.lt_scheme == RDB_EPBL_LT_ADDITIVE) return mstar + c.lt_coef * sm::pow(la_mod, c.lt_exp);
  const double enh = fmn(c.lt_max, 1.0 + c.lt_coef * sm::pow(la_mod, c.lt_exp));
  return mstar * enh;
}

template <bool GEN>
__device__ __forceinline__ double vstar_of(const EpblParams& c, double tke_here, double conv_perel, double htot,
                                           double mld_guess, double ustar, double dt, double rho0) {
  if (GEN && c.vstar_scheme == RDB_EPBL_VSTAR_RH18) {
    const double surf_scale = fmx(0.05, 1.0 - htot / mld_guess);
    return c.vstar_scale_fac * surf_scale *
           (c.vstar_surf_fac * ustar + cbrt_kahan(c.wstar_ustar_coef * conv_perel / (dt * rho0)));
  }
  return c.vstar_scale_fac * cbrt_kahan(tke_here / (dt * rho0));
}

__device__ __forceinline__ double kd_of(const EpblParams& c, double vstar, double htot, double hbs, double absf) {
  if (c.mld_iteration) {
    const double mixlen = fmx(c.min_mix_len, (htot * hbs * vstar) / (c.ekman_scale_coef * absf * htot * hbs + vstar));
    return vstar * c.von_karman * mixlen;
  }
  return vstar * c.von_karman * (htot * hbs * vstar) / (c.ekman_scale_coef * absf * htot * hbs + vstar);
}

// Pre-mixing T/S of a layer and its PE / column-height sensitivities at the
// mid-layer pressure of the stack (the prep sweep, :1087-1183).
struct LevelPrep {
  double t0, s0, dpe_t, dpe_s, dch_t, dch_s;
};

__device__ __forceinline__ LevelPrep level_prep(double hk, double T, double S, double rho0, double& pres) {
  LevelPrep q;
  q.t0 = 0.0;
  q.s0 = 0.0;
  if (hk > 0.0) {
    q.t0 = T;
    q.s0 = S;
  }
  const double dmass = rho0 * hk;
  const double dpres = GRAVITY * dmass;
  const double p_mid = pres + 0.5 * dpres;
  double dsv_dt, dsv_ds;
  specvol_derivs(q.t0, q.s0, p_mid, dsv_dt, dsv_ds);
  q.dpe_t = dmass * p_mid * dsv_dt;
  q.dpe_s = dmass * p_mid * dsv_ds;
  q.dch_t = dmass * dsv_dt;
  q.dch_s = dmass * dsv_ds;
  pres = pres + dpres;
  return q;
}

// The state of one downward sweep between two interfaces; A is the layer
// above the next interface.
struct EpblSweep {
  double mech_tke, conv_perel;
  double hA, pres, hp_a, dpe_t_a, dpe_s_a, dch_t_a, dch_s_a, th_a, sh_a, te_lag, se_lag, kddt_prev;
  double htot, z_int, pres_int, mld_output;
  double A_t0, A_s0, A_dch_t, A_dch_s;
  double d_wind, d_conv, d_forcing, d_mixing, d_mdecay, d_cdecay;
  bool sfc_connected;
};

// Values of one column that every sweep uses.
struct EpblColumn {
  double h_sum, absf, idecay, ustar, rho0, dt, mld_guess;
};

// h, T and S of one level, loaded ahead of the sweep.
struct EpblLevel {
  double h, T, S;
};

// The levels of one lane's column that its sweep comes to next, a block of N
// in LDS.  (Loaded a level or two ahead into registers they cost a full
// memory round trip an interface: the compiler waits for every load in
// flight where the slots rotate, and for the stores of kd_int with them.)
template <int N>
struct EpblLevels {
  const StateView& s;
  double* slot;  // this lane's first of 3 N, 64 apart
  int p, base;   // levels base .. base + N - 1 are held
  __device__ __forceinline__ EpblLevels(const StateView& sv, double* lds, int col)
      : s(sv), slot(lds + (threadIdx.x & 63)), p(col), base(-N) {}
  __device__ __forceinline__ EpblLevel at(int k) {
    const int P = s.P;
    if (k < base || k >= base + N) {
      base = max(k - (N - 1), 0);
      double v[3 * N];
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const int kk = min(base + j, s.nz - 1);
        v[3 * j] = LV(s.h, kk);
        v[3 * j + 1] = LV(s.T, kk);
        v[3 * j + 2] = LV(s.S, kk);
      }
#pragma unroll
      for (int j = 0; j < 3 * N; ++j) slot[64 * j] = v[j];
    }
    const double* q = slot + 192 * (k - base);
    return EpblLevel{q[0], q[64], q[128]};
  }
};

// One interface ki of the sweep (between the layer above, in st, and layer
// B = ki - 1): the energy solve and the embedded forward elimination.
// Returns whether the sweep disconnects from the surface here.
//
// The reference evaluates v* and K for the mechanical energy first, then, in
// a convecting interface (pe_max < 0), again with the energy that convection
// releases, and keeps the first only if the second would cost energy.  The
// sign test needs neither, so it comes first and a single evaluation serves
// both branches; the first value is formed only in that rare case.  The
// energy of the accepted K is the same expression in both branches.
template <bool GEN>
__device__ __forceinline__ bool epbl_interface(const EpblParams& c, const EpblColumn& q, bool first, EpblLevel lev,
                                               EpblSweep& st, double& kd_out) {
  const double G = GRAVITY, nstar = c.nstar, rho0 = q.rho0, dt = q.dt;
  const double hB = lev.h;
  const LevelPrep B = level_prep(hB, lev.T, lev.S, rho0, st.pres);
  const double h_ka = st.hA + H_NEGLECT;
  const double h_kb = hB + H_NEGLECT;
  bool sfc_disconnect = false;
  // with no mechanical TKE left the decay changes nothing:
  // (1 - e) * 0 and 0 * e are 0 for the finite e in (0, 1]
  if (st.mech_tke != 0.0) {
    const double exp_kh = sm::exp(-h_ka * q.idecay);
    st.d_mdecay = st.d_mdecay + (1.0 - exp_kh) * st.mech_tke;
    st.mech_tke = st.mech_tke * exp_kh;
  }
  double nstar_fc = nstar;
  if (st.conv_perel > 0.0 && q.absf > 0.0) {
    const double ah = q.absf * st.htot;
    nstar_fc = nstar * st.conv_perel / (st.conv_perel + 0.2 * sqrt(0.5 * dt * rho0 * cube(ah) * st.conv_perel));
  }
  const double tot_tke = st.mech_tke + nstar_fc * st.conv_perel;
  const double dt_h = dt / fmx(0.5 * (h_ka + h_kb), 1.0e-15 * q.h_sum);
  double kd_val;
  if (tot_tke <= 0.0 &&
      0.0 <= (B.dch_t + st.A_dch_t) * (st.A_t0 - B.t0) + (B.dch_s + st.A_dch_s) * (st.A_s0 - B.s0)) {
    kd_val = 0.0;
    sfc_disconnect = true;
  } else {
    const double hp_b = h_kb;
    const double th_b = h_kb * B.t0, sh_b = h_kb * B.s0;
    const double hps = st.hp_a + hp_b;
    const double bdt1 = st.hp_a * hp_b;
    const double dt_c = st.hp_a * th_b - hp_b * st.th_a;
    const double ds_c = st.hp_a * sh_b - hp_b * st.sh_a;
    double pec_core = hp_b * (st.dpe_t_a * dt_c + st.dpe_s_a * ds_c) - st.hp_a * (B.dpe_t * dt_c + B.dpe_s * ds_c);
    const double colht_core =
        hp_b * (st.dch_t_a * dt_c + st.dch_s_a * ds_c) - st.hp_a * (B.dch_t * dt_c + B.dch_s * ds_c);
    if (colht_core < 0.0) pec_core = pec_core - st.pres_int * colht_core;
    const double pe_max = pec_core / (bdt1 * hps);
    const bool conv = pe_max < 0.0;
    const double hb_hs = (q.h_sum - st.z_int) / q.h_sum;
    const double hbs = fmn(hb_hs, mixlen_shape<GEN>(c, st.z_int, q.mld_guess));
    auto kd_for = [&](double tke) -> double {
      if (!(tke > 0.0)) return 0.0;
      const double vstar = vstar_of<GEN>(c, tke, st.conv_perel, st.htot, q.mld_guess, q.ustar, dt, rho0);
      return kd_of(c, vstar, st.htot, hbs, q.absf);
    };
    kd_val = kd_for(st.mech_tke + c.wstar_ustar_coef * (conv ? st.conv_perel - pe_max : st.conv_perel));
    const double dkddt = kd_val * dt_h;
    const double num = pec_core * dkddt, den = bdt1 * (bdt1 + dkddt * hps);
    double energy = num / den;
    if (conv) {
      if (energy > 0.0) {
        kd_val = kd_for(st.mech_tke + c.wstar_ustar_coef * st.conv_perel);
        const double dk0 = kd_val * dt_h;
        energy = pec_core * dk0 / (bdt1 * (bdt1 + dk0 * hps));
      }
      st.conv_perel = st.conv_perel - energy;
      st.d_conv = st.d_conv - nstar * energy;
      if (st.sfc_connected) st.mld_output = st.mld_output + hB;
    } else {
      double frac_bl = 1.0;
      if (!((num <= tot_tke * den) || (pec_core <= 0.0))) {
        kd_val = ((bdt1 * bdt1) * tot_tke) / (dt_h * (pec_core - bdt1 * hps * tot_tke));
        energy = tot_tke;
        frac_bl = tot_tke * den / num;
      }
      if (st.sfc_connected) st.mld_output = st.mld_output + frac_bl * hB;
      if (frac_bl < 1.0) sfc_disconnect = true;
      double r_reduc = 0.0;
      if (tot_tke > 0.0 && tot_tke > energy) r_reduc = (tot_tke - energy) / tot_tke;
      st.d_mixing = st.d_mixing + energy;
      st.d_cdecay = st.d_cdecay + (1.0 - r_reduc) * (nstar - nstar_fc) * st.conv_perel;
      st.mech_tke = r_reduc * st.mech_tke;
      st.conv_perel = r_reduc * st.conv_perel;
    }
  }
  kd_out = kd_val;
  const double kddt_cur = kd_val * dt_h;
  const double b1 = 1.0 / (st.hp_a + kddt_cur);
  const double c1 = kddt_cur * b1;
  if (first) {
    st.te_lag = b1 * (h_ka * st.A_t0);
    st.se_lag = b1 * (h_ka * st.A_s0);
  } else {
    st.te_lag = b1 * (h_ka * st.A_t0 + st.kddt_prev * st.te_lag);
    st.se_lag = b1 * (h_ka * st.A_s0 + st.kddt_prev * st.se_lag);
  }
  st.hp_a = h_kb + (st.hp_a * b1) * kddt_cur;
  st.dpe_t_a = B.dpe_t + c1 * st.dpe_t_a;
  st.dpe_s_a = B.dpe_s + c1 * st.dpe_s_a;
  st.dch_t_a = B.dch_t + c1 * st.dch_t_a;
  st.dch_s_a = B.dch_s + c1 * st.dch_s_a;
  st.th_a = h_kb * B.t0 + kddt_cur * st.te_lag;
  st.sh_a = h_kb * B.s0 + kddt_cur * st.se_lag;
  st.kddt_prev = kddt_cur;
  if (sfc_disconnect) {
    st.htot = hB;
    st.sfc_connected = false;
  } else {
    st.htot = st.htot + hB;
  }
  st.z_int = st.z_int + hB;
  st.pres_int = st.pres_int + G * rho0 * hB;
  st.hA = hB;
  st.A_t0 = B.t0;
  st.A_s0 = B.s0;
  st.A_dch_t = B.dch_t;
  st.A_dch_s = B.dch_s;
  return sfc_disconnect;
}

// What the sweeps of one column start from, and the surface forcing.
struct EpblStart {
  int k_sfc;
  double h_sfc, pres0, b0, ctke_sfc, mech_in, lt_ustokes, lt_kphil;
  LevelPrep top;
};

// The surface layer, column depth and forcing of packed column p
// (:1087-1226).
template <bool GEN>
__device__ __forceinline__ EpblStart epbl_start(const StateView& s, const EpblParams& c, const double* fcor,
                                                double rho0, double cp, double dt, int p, EpblColumn& q) {
  const int P = s.P, nz = s.nz;
  const double G = GRAVITY;
  EpblStart a;
  // the surface layer: the first live layer counting down from the top
  a.k_sfc = nz - 1;
  for (int k = nz - 1; k >= 0; --k)
    if (LV(s.h, k) > H_VANISHED) {
      a.k_sfc = k;
      break;
    }
  // (eight loads a round: the sum is serial, the loads are not)
  double h_sum = 0.0;
  for (int k0 = a.k_sfc; k0 >= 0; k0 -= 8) {
    double hh[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) hh[j] = LV(s.h, max(k0 - j, 0));
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (k0 - j >= 0) h_sum = h_sum + hh[j];
  }
  q.h_sum = h_sum + H_NEGLECT;
  a.h_sfc = LV(s.h, a.k_sfc);
  a.pres0 = 0.0;
  a.top = level_prep(a.h_sfc, LV(s.T, a.k_sfc), LV(s.S, a.k_sfc), rho0, a.pres0);
  const double dmass_s = rho0 * a.h_sfc;
  const double pmid_s = 0.0 + 0.5 * (G * dmass_s);
  double dsv_dt_sfc, dsv_ds_sfc;
  specvol_derivs(a.top.t0, a.top.s0, pmid_s, dsv_dt_sfc, dsv_ds_sfc);
  const double q_t_kin = (1.0 / (rho0 * cp)) * s.Qh[p];
  const double q_s_kin = (1.0 / rho0) * s.Qs[p];
  a.b0 = G * rho0 * (dsv_dt_sfc * q_t_kin + dsv_ds_sfc * q_s_kin);
  a.ctke_sfc = -(0.5 * G * (rho0 * rho0) * a.h_sfc * (q_t_kin * dt * dsv_dt_sfc + q_s_kin * dt * dsv_ds_sfc));
  q.ustar = fmx(sqrt(s.tau_tot[p] / rho0), c.ustar_min);
  const double f = fcor[p];
  q.absf = sqrt((1.0 - c.omega_frac) * (f * f) + c.omega_frac * 4.0 * (c.omega * c.omega));
  q.idecay = c.tke_decay * q.absf / q.ustar;
  q.rho0 = rho0;
  q.dt = dt;
  a.mech_in = dt * rho0 * cube(q.ustar);
  a.lt_ustokes = a.lt_kphil = 0.0;
  if (GEN && c.use_lt) lf17_wave_state(q.ustar, rho0, a.lt_ustokes, a.lt_kphil);
  return a;
}

// The top of a sweep for the guess q.mld_guess (:1290-1350).
template <bool GEN>
__device__ __forceinline__ void epbl_begin(const EpblParams& c, const EpblColumn& q, const EpblStart& a,
                                           EpblSweep& st, double& la_val) {
  double mstar_val = find_mstar<GEN>(c, a.b0, q.ustar, q.mld_guess, q.absf);
  if (GEN && c.use_lt) {
    la_val = lf17_la(q.ustar, c.la_frac_hbl * q.mld_guess, a.lt_ustokes, a.lt_kphil);
    mstar_val = lt_enhance(c, la_val, a.b0, q.ustar, q.mld_guess, q.absf, mstar_val);
  }
  st.mech_tke = mstar_val * a.mech_in;
  st.d_wind = st.mech_tke;
  st.d_conv = st.d_forcing = st.d_mixing = st.d_mdecay = st.d_cdecay = 0.0;
  if (a.ctke_sfc <= 0.0) {
    const double forcing_clip = fmx(a.ctke_sfc, -st.mech_tke);
    st.mech_tke = st.mech_tke + forcing_clip;
    st.conv_perel = 0.0;
    st.d_forcing = forcing_clip;
  } else {
    st.conv_perel = a.ctke_sfc;
    st.d_conv = c.nstar * a.ctke_sfc;
  }
  st.hA = a.h_sfc;
  st.A_t0 = a.top.t0;
  st.A_s0 = a.top.s0;
  st.A_dch_t = a.top.dch_t;
  st.A_dch_s = a.top.dch_s;
  st.pres = a.pres0;
  st.hp_a = a.h_sfc + H_NEGLECT;
  st.dpe_t_a = a.top.dpe_t;
  st.dpe_s_a = a.top.dpe_s;
  st.dch_t_a = a.top.dch_t;
  st.dch_s_a = a.top.dch_s;
  st.th_a = st.hp_a * a.top.t0;
  st.sh_a = st.hp_a * a.top.s0;
  st.te_lag = st.se_lag = st.kddt_prev = 0.0;
  st.htot = a.h_sfc;
  st.z_int = a.h_sfc;
  st.pres_int = GRAVITY * q.rho0 * a.h_sfc;
  st.mld_output = a.h_sfc;
  st.sfc_connected = true;
}

// The MLD root-finder (:1625-1641) between two guesses.
struct EpblRoot {
  double min_mld, max_mld, dmld_min, dmld_max;
  bool have_min, have_max;
  // the guess after iteration it, whose sweep for `guess` found `found`
  __device__ __forceinline__ double next(const EpblParams& c, int it, double guess, double found) {
    if (found > guess) {
      min_mld = guess;
      dmld_min = found - guess;
      have_min = true;
    } else {
      max_mld = guess;
      dmld_max = found - guess;
      have_max = true;
    }
    if (c.mld_bisection) return 0.5 * (min_mld + max_mld);
    if (have_min && have_max && it > 2 && ((it - 1) % 4) > 0)
      return min_mld + dmld_min * (max_mld - min_mld) / (dmld_min - dmld_max);
    if (found > min_mld && found < max_mld) return found;
    return 0.5 * (min_mld + max_mld);
  }
};

// Whether iteration it, with this guess and this result, is the last.
__device__ __forceinline__ bool epbl_last(const EpblParams& c, int it, double guess, double found) {
  return !c.mld_iteration || it == c.mld_max_its || fabs(found - guess) < c.mld_tol;
}

__device__ __forceinline__ void epbl_store(const StateView& s, const EpblParams& c, const EpblView& e, int p,
                                           const EpblSweep& st, double mld, double la, double dt) {
  const int P = s.P;
  e.mld[p] = mld;
  e.la[p] = la;
  if (c.tke_diags) {
    LV(e.tke, 0) = st.d_wind / dt;
    LV(e.tke, 1) = st.d_conv / dt;
    LV(e.tke, 2) = st.d_forcing / dt;
    LV(e.tke, 3) = st.d_mixing / dt;
    LV(e.tke, 4) = st.d_mdecay / dt;
    LV(e.tke, 5) = st.d_cdecay / dt;
  }
}

// A sweep that is still connected where less than the root finder's
// tolerance is left below, in at least this many layers, leaves its column to
// k_epbl_bed.
constexpr int BED_LEVELS = 12;
// Guesses that k_epbl_bed tries at a time, a wavefront each.
constexpr int BED_WAVES = 8;

}  // namespace

// The EPBL solve for the packed columns [p0, p1): kd_int, MLD, B0, La and
// the TKE ledger of each (free surface, no penetrating shortwave).  One lane
// per column: a serial chain of about 550 vector instructions an interface,
// 2 us of it at one or two wavefronts a SIMD, so the longest chain bounds the
// kernel.  On 480 x 360 x 75 (121 000 wet columns) one solve took 1.66 ms,
// eight sweeps of 74 interfaces in the columns over fillers; now 0.22-0.27 ms here
// and 0.49 ms in k_epbl_bed.  What gave it: those columns' sweeps side by
// side; the last guess's sweep carried on where it stopped instead of
// repeated; one evaluation of v* and K an interface; levels through LDS.
// (Branch-free exp and cbrt, to leave the compiler longer blocks, cost
// 0.04 ms; two waves a SIMD need the 256-register cap.)
template <bool GEN>
__global__ void __launch_bounds__(64, 2) k_epbl(StateView s, EpblParams c, EpblView e, const double* __restrict__ fcor,
                                             double rho0, double cp, double dt, int p0, int p1) {
  __shared__ double lds[3 * 8 * 64];
  const int p = p0 + blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= p1) return;
  const int P = s.P, nz = s.nz;
  EpblLevels<8> levels(s, lds, p);
  EpblColumn q;
  const EpblStart a = epbl_start<GEN>(s, c, fcor, rho0, cp, dt, p, q);
  e.b0[p] = a.b0;
  double la_val = 0.0;
  EpblSweep st;
  st.d_wind = st.d_conv = st.d_forcing = st.d_mixing = st.d_mdecay = st.d_cdecay = 0.0;
  double mld_found = 0.0;

  if (s.wet[p] <= 0.0 || q.h_sum <= 2.0 * H_NEGLECT) {
    for (int k = 0; k <= nz; ++k) LV(e.kd, k) = 0.0;
  } else {
    EpblRoot root{0.0, q.h_sum, 0.0, 0.0, false, false};
    q.mld_guess = 0.5 * (root.min_mld + root.max_mld);
    if (c.mld_use_prev_guess && e.mld[p] > 0.0) q.mld_guess = fmn(e.mld[p], root.max_mld);
    for (int k = a.k_sfc + 1; k <= nz; ++k) LV(e.kd, k) = 0.0;
    LV(e.kd, 0) = 0.0;
    // A guess only needs the MLD, which stops growing once its sweep
    // disconnects from the surface: each sweep stops there.  kd_int is
    // written as the sweep goes (a later guess overwrites it), so the sweep
    // of the last guess only has to be carried on from where it stopped,
    // below.
    int ki = a.k_sfc;
    for (int it = 1;; ++it) {
      epbl_begin<GEN>(c, q, a, st, la_val);
      for (ki = a.k_sfc; ki >= 1; --ki) {
        if (it == 1 && c.mld_iteration && ki > BED_LEVELS && q.h_sum - st.z_int < c.mld_tol) {
          // connected to the bottom of the water, fillers below
          e.bed_list[atomicAdd(e.bed_count, 1u)] = p;
          return;
        }
        double kd;
        const bool dis = epbl_interface<GEN>(c, q, ki == a.k_sfc, levels.at(ki - 1), st, kd);
        LV(e.kd, ki) = kd;
        if (dis) {
          --ki;
          break;
        }
      }
      mld_found = st.mld_output;
      if (epbl_last(c, it, q.mld_guess, mld_found)) break;
      q.mld_guess = root.next(c, it, q.mld_guess, mld_found);
    }
    // The last guess's sweep goes on to the bed.  Every lane walks from the
    // wavefront's highest open interface, so that a level stays one
    // coalesced access, and joins at its own.
    int top_open = nz - 1;
    while (top_open >= 1 && !__any(ki >= top_open)) --top_open;
    for (int k = top_open; k >= 1; --k) {
      if (k <= ki) {
        double kd;
        epbl_interface<GEN>(c, q, k == a.k_sfc, levels.at(k - 1), st, kd);
        LV(e.kd, k) = kd;
      }
    }
    st.d_mdecay = st.d_mdecay + st.mech_tke;
    st.d_cdecay = st.d_cdecay + c.nstar * st.conv_perel;
  }
  epbl_store(s, c, e, p, st, mld_found, la_val, dt);
}

// The columns that are mixed to the bottom of the water and hold a stack of
// fillers below it (two or three live layers of 75, above all): the root
// finder halves its way to the column depth, about eight sweeps of the whole
// column one after the other, eight times the length of any other column's
// chain (592 interfaces of 75 layers).  Each of those sweeps finds the whole
// column, so the guesses are known beforehand: a workgroup takes 64 columns
// and each wavefront sweeps one guess of the sequence that results when
// every sweep finds the column's thickness.  Then the first wavefront
// replays the root finder on the results; a guess that is not the foreseen
// one (a sweep found something else) is swept there.  The guesses, their
// sweeps and the order of the decisions are the sequential ones, so the bits
// are.
template <bool GEN>
__global__ void __launch_bounds__(64 * BED_WAVES) k_epbl_bed(StateView s, EpblParams c, EpblView e,
                                                             const double* __restrict__ fcor, double rho0, double cp,
                                                             double dt) {
  __shared__ double lds[BED_WAVES][3 * 4 * 64], sh_guess[BED_WAVES][64], sh_found[BED_WAVES][64];
  __shared__ int sh_owner[64];
  const int P = s.P, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = (int)*e.bed_count;
  for (int i0 = blockIdx.x * 64; i0 < n; i0 += gridDim.x * 64) {
    const bool on = i0 + lane < n;
    const int p = e.bed_list[on ? i0 + lane : i0];
    EpblColumn q;
    const EpblStart a = epbl_start<GEN>(s, c, fcor, rho0, cp, dt, p, q);
    EpblLevels<4> levels(s, lds[wave], p);
    EpblRoot root{0.0, q.h_sum, 0.0, 0.0, false, false};
    double guess = 0.5 * (root.min_mld + root.max_mld);
    if (c.mld_use_prev_guess && e.mld[p] > 0.0) guess = fmn(e.mld[p], root.max_mld);
    int it = 1;
    // this wavefront's guess of the foreseen sequence: iteration 1 + wave,
    // where every sweep adds up the column (h_sum: the same sum in the same
    // order, H_NEGLECT vanishes in it)
    bool foreseen = on;
    double my_guess = guess;
    {
      EpblRoot r = root;
      for (int j = 0; j < wave && foreseen; ++j) {
        if (epbl_last(c, 1 + j, my_guess, q.h_sum))
          foreseen = false;
        else
          my_guess = r.next(c, 1 + j, my_guess, q.h_sum);
      }
    }
    // kd_int of this sweep, until it is known whose guess is the last: a
    // column of the scratch arrays fa and fb, if there are that many
    const long long slot = (long long)i0 * BED_WAVES + 64 * wave + lane;
    foreseen = foreseen && slot < 2LL * P;
    double* const kds = slot < P ? s.fa + slot : s.fb + (slot < 2LL * P ? slot - P : 0);
    // One sweep loop serves every phase (three copies of it spill): first
    // each wavefront's foreseen guess, then the first wavefront's guesses
    // that were not foreseen, then the last guess's sweep on to the bed.
    EpblSweep st;
    double la_val = 0.0;
    int ki = 0, k_kept = 0;
    int phase = 0;
    bool go = foreseen, decided = !on;
    double* kd_to = kds;
    q.mld_guess = my_guess;
    for (;;) {
      if (go) {
        if (phase < 2) {
          epbl_begin<GEN>(c, q, a, st, la_val);
          ki = a.k_sfc;
        }
        for (; ki >= 1; --ki) {
          double kd;
          const bool dis = epbl_interface<GEN>(c, q, ki == a.k_sfc, levels.at(ki - 1), st, kd);
          kd_to[(size_t)ki * (size_t)P] = kd;
          if (dis && phase < 2) {
            --ki;
            break;
          }
        }
      }
      if (phase == 2) break;
      if (phase == 0) {
        sh_guess[wave][lane] = my_guess;
        sh_found[wave][lane] = foreseen ? st.mld_output : -1.0;
        k_kept = ki;  // interfaces k_sfc .. k_kept + 1 are in kds
        kd_to = e.kd + p;
        phase = 1;
        go = false;
        __syncthreads();
      }
      if (wave == 0) {
        // replay the root finder on the results at hand
        while (!decided) {
          const int w = it - 1;
          double f = st.mld_output;
          const bool swept = go;
          if (!swept) {
            if (!(w < BED_WAVES && sh_found[w][lane] >= 0.0 && sh_guess[w][lane] == guess)) {
              q.mld_guess = guess;
              go = true;
              break;
            }
            f = sh_found[w][lane];
          }
          go = false;
          if (epbl_last(c, it, guess, f)) {
            sh_owner[lane] = swept ? BED_WAVES : w;
            decided = true;
          } else {
            guess = root.next(c, it, guess, f);
            ++it;
          }
        }
        if (__any(!decided)) continue;
      }
      __syncthreads();
      const int owner = on ? sh_owner[lane] : -1;
      go = owner == wave || (wave == 0 && owner == BED_WAVES);
      if (owner == wave)
        for (int k0 = a.k_sfc; k0 > k_kept; k0 -= 16) {
          double v[16];
#pragma unroll
          for (int j = 0; j < 16; ++j) v[j] = kds[(size_t)max(k0 - j, 0) * (size_t)P];
#pragma unroll
          for (int j = 0; j < 16; ++j)
            if (k0 - j > k_kept) LV(e.kd, k0 - j) = v[j];
        }
      phase = 2;
    }
    if (go) {
      st.d_mdecay = st.d_mdecay + st.mech_tke;
      st.d_cdecay = st.d_cdecay + c.nstar * st.conv_perel;
      epbl_store(s, c, e, p, st, st.mld_output, la_val, dt);
    }
    __syncthreads();  // the next columns reuse the shared arrays
  }
  // the last workgroup to finish empties the list for the next solve
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence();
    if (atomicAdd(e.bed_done, 1u) == gridDim.x - 1) {
      *e.bed_count = 0u;
      *e.bed_done = 0u;
    }
  }
}
#define INST(GEN)                                                                                                 \
  template __global__ void k_epbl<GEN>(StateView, EpblParams, EpblView, const double*, double, double, double, int, \
                                       int);                                                                      \
  template __global__ void k_epbl_bed<GEN>(StateView, EpblParams, EpblView, const double*, double, double, double);
INST(false)
INST(true)
#undef INST

// The coefficient build after the surface scheme, one pass per column from
// the top: PP81 at each interface (when the surface scheme did not need it
// first, i.e. with EPBL), the EPBL merge, KV_ML_INVZ2, convective
// adjustment, then the heat/salt split with double diffusion, the guard and
// the floors/ceilings of vmix_assemble (rdb_ocean_vmix.F90:2265-2385).  Each
// is a per-interface update applied in the reference's order, so one pass
// gives the bits of the separate sweeps; kv, kt and ks are written once.
// TAIL interfaces' loads are in flight together.  us with 1, 2 and 4 of them:
// 4096 columns x 20 23, 18, 17; 330 x 300 x 75 257, 197, 191; 480 x 360 x 75
// 280, 220, 222; 800 x 640 x 60 481, 474, 486; 1440 x 1080 x 75 1710, 1715, 1749.
constexpr int TAIL = 2;
__global__ void __launch_bounds__(256) k_coeff_tail(StateView s, Params pr, ContribParams c, EpblView e, int do_pp81, int p0, int p1,
                             unsigned int* guard_count) {
  const int p = p0 + blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= p1) return;
  const int P = s.P, nz = s.nz;
  const double bld = c.epbl ? e.mld[p] : s.bl[p];
  const bool invz2 = c.kv_ml_invz2 > 0.0 && c.hmix > 0.0;
  const double hmix_sq = c.hmix * c.hmix;
  const double dz_min_safe = 0.5 * c.hmix / (double)(nz > 1 ? nz : 1);
  bool inv_done = !invz2;
  unsigned int bad = 0;
  auto finish = [&](int k, double kv, double kt, double kd_t, double kd_s) {
    double ks = kt;
    if (pr.ddiff) {
      ks = kt + kd_s;
      kt = kt + kd_t;
    }
    if (pr.guard && (isnan(kv) || isnan(kt) || isnan(ks) || kv < 0.0 || kt < 0.0 || ks < 0.0)) ++bad;
    if (k >= 1 && k < nz) {
      kv = fmn(fmx(kv, pr.kv_bg), pr.kv_max);
      kt = fmn(fmx(kt, pr.kt_bg), pr.kd_max);
      ks = fmn(fmx(ks, pr.ks_bg), pr.kd_max);
    }
    LV(s.kv, k) = kv;
    LV(s.kt, k) = kt;
    LV(s.ks, k) = ks;
  };
  if (do_pp81) {
    finish(nz, 0.0, 0.0, 0.0, 0.0);
  } else {
    finish(nz, LV(s.kv, nz), LV(s.kt, nz), 0.0, 0.0);
  }
  double z = 0.0;
  double h_up = LV(s.h, nz - 1), rho_up = LV(s.rho, nz - 1);
  double ub_up = do_pp81 ? LV(s.ub, nz - 1) : 0.0, vb_up = do_pp81 ? LV(s.vb, nz - 1) : 0.0;
  double T_up = LV(s.T, nz - 1), S_up = LV(s.S, nz - 1);
  // the layers below TAIL interfaces at a time
  for (int k0 = nz - 1; k0 >= 1; k0 -= TAIL) {
    double bh[TAIL], br[TAIL], bT[TAIL], bS[TAIL], bu[TAIL], bv[TAIL], bk[TAIL];
#pragma unroll
    for (int j = 0; j < TAIL; ++j) {
      const int kd = max(k0 - j - 1, 0);
      bh[j] = LV(s.h, kd);
      br[j] = LV(s.rho, kd);
      bT[j] = LV(s.T, kd);
      bS[j] = LV(s.S, kd);
      // centred velocities below the interface, or its kv and kt
      bu[j] = do_pp81 ? LV(s.ub, kd) : LV(s.kv, kd + 1);
      bv[j] = do_pp81 ? LV(s.vb, kd) : LV(s.kt, kd + 1);
      bk[j] = c.epbl ? LV(e.kd, kd + 1) : 0.0;
    }
#pragma unroll
    for (int j = 0; j < TAIL; ++j) {
      const int k = k0 - j;
      if (k < 1) continue;
      const double h_dn = bh[j], rho_dn = br[j];
      const double T_dn = bT[j], S_dn = bS[j];
      double ub_dn = 0.0, vb_dn = 0.0;
      double kv, kt;
      if (do_pp81) {
        ub_dn = bu[j];
        vb_dn = bv[j];
        pp81_iface<double>(pr, ub_dn, vb_dn, ub_up, vb_up, h_dn, h_up, rho_up - rho_dn, kv, kt);
      } else {
        kv = bu[j];
        kt = bv[j];
      }
      if (c.epbl) {
        const double kd = bk[j];
        if (c.combine == RDB_EPBL_COMBINE_MAX) {
          kt = fmx(kt, kd);
          kv = fmx(kv, c.prandtl * kd);
        } else {
          kt = kt + kd;
          kv = kv + c.prandtl * kd;
        }
      }
      z = z + h_up;
      if (!inv_done) {
        if (z >= c.hmix) {
          inv_done = true;
        } else {
          const double m = fmx(z, dz_min_safe);
          kv = kv + c.kv_ml_invz2 * hmix_sq / (m * m);
        }
      }
      if (c.conv) {
        const double dz_face = 0.5 * (h_dn + h_up);
        if (dz_face > H_VANISHED && !(z < bld)) {
          const double n2 = -(GRAVITY * (rho_up - rho_dn) / (c.rho0 * dz_face));
          if (n2 < c.n2_thresh) {
            kt = fmx(kt, c.conv_kd);
            kv = fmx(kv, c.conv_prandtl * c.conv_kd);
          }
        }
      }
      double kd_t = 0.0, kd_s = 0.0;
      if (pr.ddiff) ddiff_iface(pr, h_up, h_dn, T_up, T_dn, S_up, S_dn, kd_t, kd_s);
      finish(k, kv, kt, kd_t, kd_s);
      h_up = h_dn;
      rho_up = rho_dn;
      ub_up = ub_dn;
      vb_up = vb_dn;
      T_up = T_dn;
      S_up = S_dn;
    }
  }
  if (do_pp81)
    finish(0, 0.0, 0.0, 0.0, 0.0);
  else
    finish(0, LV(s.kv, 0), LV(s.kt, 0), 0.0, 0.0);
  if (bad) atomicAdd(guard_count, bad);
}

// The device safe math over n arguments (fn: 0 exp, 1 log, 2 pow, 3 erfc),
// checked against the reference's golden rows.
__global__ void k_safe_math_eval(int fn, const double* x, const double* y, double* out, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double r;
  switch (fn) {
    case 0: r = sm::exp(x[i]); break;
    case 1: r = sm::log(x[i]); break;
    case 2: r = sm::pow(x[i], y[i]); break;
    default: r = sm::erfc(x[i]); break;
  }
  out[i] = r;
}

}  // namespace colphys

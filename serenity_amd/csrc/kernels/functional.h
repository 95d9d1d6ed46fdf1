// Exchange-correlation functionals of the XC Fock build, FP64, evaluated per
// grid point with forward-mode derivatives so the potential terms come from
// the same code as the energy.
//
// The formulas restate the basic functionals Serenity takes from XCFun (or
// LibXC) for the LDA, PBE and BP86 composites (functional_definitions.dat:44,47,48;
// basic_functionals.dat:35,78,99,113,168,226,230): Slater exchange, VWN5 correlation
// (Vosko-Wilk-Nusair 1980 with their spin interpolation), PBE exchange and
// correlation (Perdew-Burke-Ernzerhof 1996 with the Perdew-Wang 1992 LDA
// correlation), Becke 1988 exchange, Perdew 1986 correlation on Perdew-Zunger
// 1981, and Thomas-Fermi kinetic energy.
//
// Restricted inputs: total density rho and sigma = |grad rho|^2 (partials in
// that order); XCFun's XC_N_NX_NY_NZ outputs are then
//   eps (energy per volume), v = d eps/d rho, g = 2 d eps/d sigma * grad rho.
// Unrestricted inputs (XC_A_B_AX_AY_AZ_BX_BY_BZ): rho_a, rho_b and
// sigma_aa, sigma_ab, sigma_bb (partials in that order); outputs
//   v_a = d eps/d rho_a, g_a = 2 d eps/d sigma_aa grad rho_a + d eps/d sigma_ab grad rho_b
// and likewise for b.
#pragma once

#include <cmath>

#if defined(__HIPCC__)
#define SXC_HD __host__ __device__ inline
#else
#define SXC_HD inline
#endif

namespace sxc {

// Value and N first partials.
template <int N>
struct Dual {
  double v;
  double d[N];
};
typedef Dual<2> D2;  // (rho, sigma)
typedef Dual<5> D5;  // (rho_a, rho_b, sigma_aa, sigma_ab, sigma_bb)

template <int N>
SXC_HD Dual<N> mkc(double v) {
  Dual<N> r;
  r.v = v;
  for (int i = 0; i < N; ++i) r.d[i] = 0.0;
  return r;
}
template <int N>
SXC_HD Dual<N> var(double v, int k) {
  Dual<N> r = mkc<N>(v);
  r.d[k] = 1.0;
  return r;
}
SXC_HD D2 mk(double v) { return mkc<2>(v); }

template <int N>
SXC_HD Dual<N> operator+(Dual<N> a, Dual<N> b) {
  a.v += b.v;
  for (int i = 0; i < N; ++i) a.d[i] += b.d[i];
  return a;
}
template <int N>
SXC_HD Dual<N> operator-(Dual<N> a, Dual<N> b) {
  a.v -= b.v;
  for (int i = 0; i < N; ++i) a.d[i] -= b.d[i];
  return a;
}
template <int N>
SXC_HD Dual<N> operator-(Dual<N> a) {
  a.v = -a.v;
  for (int i = 0; i < N; ++i) a.d[i] = -a.d[i];
  return a;
}
template <int N>
SXC_HD Dual<N> operator*(Dual<N> a, Dual<N> b) {
  Dual<N> r;
  r.v = a.v * b.v;
  for (int i = 0; i < N; ++i) r.d[i] = a.d[i] * b.v + a.v * b.d[i];
  return r;
}
template <int N>
SXC_HD Dual<N> operator/(Dual<N> a, Dual<N> b) {
  const double ib = 1.0 / b.v, q = a.v * ib;
  Dual<N> r;
  r.v = q;
  for (int i = 0; i < N; ++i) r.d[i] = (a.d[i] - q * b.d[i]) * ib;
  return r;
}
template <int N>
SXC_HD Dual<N> operator+(Dual<N> a, double b) {
  a.v += b;
  return a;
}
template <int N>
SXC_HD Dual<N> operator+(double b, Dual<N> a) {
  a.v += b;
  return a;
}
template <int N>
SXC_HD Dual<N> operator-(Dual<N> a, double b) {
  a.v -= b;
  return a;
}
template <int N>
SXC_HD Dual<N> operator-(double b, Dual<N> a) {
  a.v = b - a.v;
  for (int i = 0; i < N; ++i) a.d[i] = -a.d[i];
  return a;
}
template <int N>
SXC_HD Dual<N> operator*(Dual<N> a, double b) {
  a.v *= b;
  for (int i = 0; i < N; ++i) a.d[i] *= b;
  return a;
}
template <int N>
SXC_HD Dual<N> operator*(double b, Dual<N> a) {
  return a * b;
}
template <int N>
SXC_HD Dual<N> operator/(Dual<N> a, double b) {
  return a * (1.0 / b);
}
template <int N>
SXC_HD Dual<N> operator/(double b, Dual<N> a) {
  const double ia = 1.0 / a.v, q = b * ia, dq = -q * ia;
  Dual<N> r;
  r.v = q;
  for (int i = 0; i < N; ++i) r.d[i] = dq * a.d[i];
  return r;
}
template <int N>
SXC_HD Dual<N> chain(Dual<N> a, double f, double df) {
  Dual<N> r;
  r.v = f;
  for (int i = 0; i < N; ++i) r.d[i] = df * a.d[i];
  return r;
}
template <int N>
SXC_HD Dual<N> dlog(Dual<N> a) {
  return chain(a, log(a.v), 1.0 / a.v);
}
template <int N>
SXC_HD Dual<N> dexpm1(Dual<N> a) {
  const double e = expm1(a.v);
  return chain(a, e, e + 1.0);
}
template <int N>
SXC_HD Dual<N> dsqrt(Dual<N> a) {
  const double s = sqrt(a.v);
  return chain(a, s, 0.5 / s);
}
template <int N>
SXC_HD Dual<N> datan(Dual<N> a) {
  return chain(a, atan(a.v), 1.0 / (1.0 + a.v * a.v));
}

// A density (or 1 +- zeta) and the cube root of its value, from which every fractional power of the
// functionals is a product: FP64 pow takes some 250 instructions, and PBE asked for four of them (the
// functional stage of PBE at 237 000 points 22 us, of the spin-polarised PBE at 63 392 points 27; 14 and 12 so).
template <class D>
struct Rooted {
  D n;
  double c;
};
template <class D>
SXC_HD Rooted<D> rooted(D n) {
  return {n, cbrt(n.v)};
}
// n^(4/3), n^(5/3), n^(7/3), n^(8/3), n^(2/3) and n^(7/6); the derivatives of the first two are finite at 0
template <class D>
SXC_HD D pow43(const Rooted<D>& r) {
  return chain(r.n, r.n.v * r.c, (4.0 / 3.0) * r.c);
}
template <class D>
SXC_HD D pow53(const Rooted<D>& r) {
  return chain(r.n, r.n.v * r.c * r.c, (5.0 / 3.0) * r.c * r.c);
}
template <class D>
SXC_HD D pow73(const Rooted<D>& r) {
  const double p = r.n.v * r.c;
  return chain(r.n, r.n.v * p, (7.0 / 3.0) * p);
}
template <class D>
SXC_HD D pow83(const Rooted<D>& r) {
  const double p = r.n.v * r.c;
  return chain(r.n, p * p, (8.0 / 3.0) * p * r.c);
}
template <class D>
SXC_HD D pow23(const Rooted<D>& r) {
  return chain(r.n, r.c * r.c, (2.0 / 3.0) / r.c);
}
template <class D>
SXC_HD D pow76(const Rooted<D>& r) {
  const double s = sqrt(r.c);
  return chain(r.n, r.n.v * s, (7.0 / 6.0) * s);
}
// r_s = (3 / (4 pi))^(1/3) n^(-1/3)
template <class D>
SXC_HD D rs_of(const Rooted<D>& r) {
  const double i = 1.0 / r.c, rs = 0.62035049089940001667 * i;
  return chain(r.n, rs, (-1.0 / 3.0) * rs * i * i * i);
}
template <int N>
SXC_HD Dual<N> dexp(Dual<N> a) {
  const double e = exp(a.v);
  return chain(a, e, e);
}
template <int N>
SXC_HD Dual<N> dasinh(Dual<N> a) {
  return chain(a, asinh(a.v), 1.0 / sqrt(1.0 + a.v * a.v));
}

// Constants of the functionals (the published VWN5, PW92 and PBE values).
// The two PBE evaluators Serenity offers differ in the exchange mu: XCFun
// (its default for LDA/PBE) takes mu = 0.066725 pi^2 / 3 from the PBE paper's
// rounded beta, LibXC takes mu = beta pi^2 / 3 with the accurate beta.  Both
// use A = 0.0310907 in PW92 and the accurate beta in the correlation.  The
// full-SCF energies of Serenity's water/STO-3G PBE tests decide these values
// (qcserenity/tests/test_tasks.py:50-76: 2.8e-8 for XCFun, 2.2e-10 for LibXC).
// Spin-polarised parts: VWN5 ferromagnetic and spin-stiffness fits, PW92
// ferromagnetic and spin-stiffness fits (the A of the "modified" PW92 that
// goes with 0.0310907), f''(0) = 4 / (9 (2^(1/3) - 1)).
struct XcConstants {
  double vwn_A = 0.0310907, vwn_b = 3.72744, vwn_c = 12.9352, vwn_x0 = -0.10498;
  double pw_A = 0.0310907, pw_a1 = 0.21370, pw_b1 = 7.5957, pw_b2 = 3.5876, pw_b3 = 1.6382, pw_b4 = 0.49294;
  double pbe_kappa = 0.804, pbe_mu = 0.066725 * M_PI * M_PI / 3.0, pbe_beta = 0.06672455060314922;
  double pbe_mu_libxc = 0.2195149727645171;
  // VWN5: ferromagnetic (A, b, c, x0) and spin stiffness
  double vwnF_A = 0.01554535, vwnF_b = 7.06042, vwnF_c = 18.0578, vwnF_x0 = -0.32500;
  double vwnS_A = -1.0 / (6.0 * M_PI * M_PI), vwnS_b = 1.13107, vwnS_c = 13.0045, vwnS_x0 = -0.0047584;
  // PW92: ferromagnetic and (minus) spin stiffness
  double pwF_A = 0.01554535, pwF_a1 = 0.20548, pwF_b1 = 14.1189, pwF_b2 = 6.1977, pwF_b3 = 3.3662,
         pwF_b4 = 0.62517;
  double pwS_A = 0.0168869, pwS_a1 = 0.11125, pwS_b1 = 10.357, pwS_b2 = 3.6231, pwS_b3 = 0.88026,
         pwS_b4 = 0.49671;
  // BP86: Becke 1988 exchange (beta), Perdew-Zunger 1981 correlation (paramagnetic U and
  // ferromagnetic P fits: gamma, beta1, beta2 for r_s >= 1; A, B, C, D for r_s < 1, the published
  // values) and the Perdew 1986 gradient correction (C(n) = c0 + (c1 + alpha r_s + beta r_s^2) /
  // (1 + gamma r_s + delta r_s^2 + 1e4 beta r_s^3), f~ = 0.11).  The reference's BP86 Fock
  // matrix (FuncPotential_test.cpp:148-232) decides the one choice the paper leaves open: the
  // prefactor of Phi is f~ (9 pi)^(1/6) (1.745 in the paper is its rounding), with the original
  // PZ81 constants; 1.745 f~ misses by 8e-6, the continuity-corrected PZ81 C, D by 2.7e-6.
  double b88_beta = 0.0042;
  double pzU_g = -0.1423, pzU_b1 = 1.0529, pzU_b2 = 0.3334, pzU_A = 0.0311, pzU_B = -0.048, pzU_C = 0.0020,
         pzU_D = -0.0116;
  double pzP_g = -0.0843, pzP_b1 = 1.3981, pzP_b2 = 0.2611, pzP_A = 0.01555, pzP_B = -0.0269, pzP_C = 0.0007,
         pzP_D = -0.0048;
  double p86_alpha = 0.023266, p86_beta = 7.389e-6, p86_gamma = 8.723, p86_delta = 0.472, p86_c0 = 0.001667,
         p86_c1 = 0.002568, p86_ft = 0.11;
};
constexpr XcConstants kXc{};
constexpr double kCbrt2 = 1.25992104989487316477;            // 2^(1/3)
constexpr double kPbeGamma = (1.0 - M_LN2) / (M_PI * M_PI);  // gamma of H

// f''(0) of the spin interpolation f(zeta) = ((1+zeta)^(4/3) + (1-zeta)^(4/3) - 2) / (2^(4/3) - 2)
constexpr double kFpp0 = 1.709920934161365617563962776245;

template <class D>
SXC_HD D slater_x(const Rooted<D>& rho) {
  // -(3/4) (3/pi)^(1/3) rho^(4/3)
  return -0.73855876638202240588 * pow43(rho);
}

// VWN per-particle correlation fit as a function of x = sqrt(r_s)
template <class D>
SXC_HD D vwn_fit(D x, double A, double b, double c, double x0) {
  const double Q = __builtin_sqrt(4.0 * c - b * b);
  const double X0 = x0 * x0 + b * x0 + c;
  D X = x * x + b * x + c;
  D at = datan(Q / (2.0 * x + b));
  D t1 = dlog(x * x / X) + (2.0 * b / Q) * at;
  D t2 = dlog((x - x0) * (x - x0) / X) + (2.0 * (b + 2.0 * x0) / Q) * at;
  return A * (t1 - (b * x0 / X0) * t2);
}

template <class D>
SXC_HD D vwn5_c(const Rooted<D>& rho) {
  return rho.n * vwn_fit(dsqrt(rs_of(rho)), kXc.vwn_A, kXc.vwn_b, kXc.vwn_c, kXc.vwn_x0);
}

// Perdew-Wang 1992 fit G(r_s) (p = 1)
template <class D>
SXC_HD D pw_fit(D rs, D srs, double A, double a1, double b1, double b2, double b3, double b4) {
  D den = 2.0 * A * (b1 * srs + b2 * rs + b3 * rs * srs + b4 * rs * rs);
  return -2.0 * A * (1.0 + a1 * rs) * dlog(1.0 + 1.0 / den);
}

template <class D>
SXC_HD D pw92_eps(D rs) {
  // Perdew-Wang 1992 unpolarised correlation energy per particle
  return pw_fit(rs, dsqrt(rs), kXc.pw_A, kXc.pw_a1, kXc.pw_b1, kXc.pw_b2, kXc.pw_b3, kXc.pw_b4);
}

template <class D>
SXC_HD D pbe_x(const Rooted<D>& rho, D sigma, double mu) {
  // s^2 = sigma / (4 (3 pi^2)^(2/3) rho^(8/3))
  D s2 = sigma / (38.28312000250922421226 * pow83(rho));
  D Fx = (1.0 + kXc.pbe_kappa) - kXc.pbe_kappa / (1.0 + (mu / kXc.pbe_kappa) * s2);
  return slater_x(rho) * Fx;
}

// PBE gradient correction H(eps, t^2, phi) per particle (phi = 1 unpolarised)
template <class D>
SXC_HD D pbe_H(D eps, D t2, D phi3) {
  const double bg = kXc.pbe_beta / kPbeGamma;
  D gp = kPbeGamma * phi3;
  D A = bg / dexpm1(-eps / gp);
  D At2 = A * t2;
  return gp * dlog(1.0 + bg * t2 * (1.0 + At2) / (1.0 + At2 * (1.0 + At2)));
}

// t^2 = sigma pi / (16 (3 pi^2)^(1/3) rho^(7/3)) / phi^2
constexpr double kPbeT2 = 0.06346820609770370420;

template <class D>
SXC_HD D pbe_c(const Rooted<D>& rho, D sigma) {
  const double bg = kXc.pbe_beta / kPbeGamma;
  D eps = pw92_eps(rs_of(rho));
  D t2 = kPbeT2 * sigma / pow73(rho);  // zeta = 0, phi = 1
  D A = bg / dexpm1(eps * (-1.0 / kPbeGamma));
  D At2 = A * t2;
  D H = kPbeGamma * dlog(1.0 + bg * t2 * (1.0 + At2) / (1.0 + At2 * (1.0 + At2)));
  return rho.n * (eps + H);
}

template <class D>
SXC_HD D tf_k(const Rooted<D>& rho) {
  // C_F rho^(5/3), C_F = (3/10)(3 pi^2)^(2/3)
  return 2.87123400018819181594 * pow53(rho);
}

// x asinh(x) as a function of u = x^2: smooth at u = 0, where sqrt is not (series below 1e-12)
template <class D>
SXC_HD D xasinhx(D u) {
  if (u.v < 1e-12) return u - u * u / 6.0;
  D x = dsqrt(u);
  return x * dasinh(x);
}

// Becke 1988 exchange, restricted: two spins with rho_s = rho / 2, sigma_ss = sigma / 4, each
// -C rho_s^(4/3) - beta rho_s^(4/3) x^2 / (1 + 6 beta x asinh x), x^2 = sigma_ss / rho_s^(8/3)
template <class D>
SXC_HD D b88_x(const Rooted<D>& rho, D sigma) {
  D r43 = (0.5 / kCbrt2) * pow43(rho);
  D ss = 0.25 * sigma;
  D u = ss / (r43 * r43);
  return slater_x(rho) - 2.0 * kXc.b88_beta * (ss / r43) / (1.0 + 6.0 * kXc.b88_beta * xasinhx(u));
}

// Perdew-Zunger 1981 correlation energy per particle of one spin state
template <class D>
SXC_HD D pz81_fit(D rs, double g, double b1, double b2, double A, double B, double C, double Dd) {
  if (rs.v >= 1.0) return g / (1.0 + b1 * dsqrt(rs) + b2 * rs);
  D l = dlog(rs);
  return A * l + B + C * rs * l + Dd * rs;
}

// Perdew 1986 gradient correction exp(-Phi) C(n) sigma / (d n^(4/3)), Phi = f~ (9 pi)^(1/6)
// C(inf) / C(n) |grad n| / n^(7/6); dz = d(zeta) (1 for a closed shell)
template <class D>
SXC_HD D p86_corr(const Rooted<D>& rho, D rs, D sigma, D dz) {
  D Cn = kXc.p86_c0 + (kXc.p86_c1 + kXc.p86_alpha * rs + kXc.p86_beta * rs * rs) /
                          (1.0 + kXc.p86_gamma * rs + kXc.p86_delta * rs * rs + 1.0e4 * kXc.p86_beta * rs * rs * rs);
  const double k = kXc.p86_ft * 1.74541510612512397888 * (kXc.p86_c0 + kXc.p86_c1);  // (9 pi)^(1/6)
  // |grad n|: at sigma = 0 the correction is C(n) sigma / n^(4/3) to first order
  D g = sigma.v > 0.0 ? dsqrt(sigma) : 0.0 * sigma;
  D Phi = k * g / (Cn * pow76(rho));
  return dexp(-Phi) * Cn * sigma / (dz * pow43(rho));
}

template <class D>
SXC_HD D bp86(const Rooted<D>& rho, D sigma) {
  D rs = rs_of(rho);
  D eU = pz81_fit(rs, kXc.pzU_g, kXc.pzU_b1, kXc.pzU_b2, kXc.pzU_A, kXc.pzU_B, kXc.pzU_C, kXc.pzU_D);
  return b88_x(rho, sigma) + rho.n * eU + p86_corr(rho, rs, sigma, 1.0 + 0.0 * rho.n);
}

// ---- spin-polarised forms ---------------------------------------------------
// Spin densities below kTinyDensity count as zero: their terms are dropped.

// spin interpolation f(zeta) from 1 + zeta = 2 rho_a / rho and 1 - zeta = 2 rho_b / rho
template <class D>
SXC_HD D spin_f(const Rooted<D>& opz, const Rooted<D>& omz) {
  return (pow43(opz) + pow43(omz) - 2.0) / (2.0 * kCbrt2 - 2.0);
}

template <class D>
SXC_HD D vwn5_c_pol(D ra, D rb) {
  Rooted<D> rho = rooted(ra + rb);
  D x = dsqrt(rs_of(rho));
  D zeta = (ra - rb) / rho.n;
  D f = spin_f(rooted(1.0 + zeta), rooted(1.0 - zeta));
  D z4 = zeta * zeta * zeta * zeta;
  D eP = vwn_fit(x, kXc.vwn_A, kXc.vwn_b, kXc.vwn_c, kXc.vwn_x0);
  D eF = vwn_fit(x, kXc.vwnF_A, kXc.vwnF_b, kXc.vwnF_c, kXc.vwnF_x0);
  D aS = vwn_fit(x, kXc.vwnS_A, kXc.vwnS_b, kXc.vwnS_c, kXc.vwnS_x0);
  return rho.n * (eP + aS * f * (1.0 - z4) / kFpp0 + (eF - eP) * f * z4);
}

template <class D>
SXC_HD D pw92_eps_pol(D rs, D zeta, D f) {
  D z4 = zeta * zeta * zeta * zeta;
  D srs = dsqrt(rs);
  D e0 = pw_fit(rs, srs, kXc.pw_A, kXc.pw_a1, kXc.pw_b1, kXc.pw_b2, kXc.pw_b3, kXc.pw_b4);
  D e1 = pw_fit(rs, srs, kXc.pwF_A, kXc.pwF_a1, kXc.pwF_b1, kXc.pwF_b2, kXc.pwF_b3, kXc.pwF_b4);
  // -alpha_c
  D mac = pw_fit(rs, srs, kXc.pwS_A, kXc.pwS_a1, kXc.pwS_b1, kXc.pwS_b2, kXc.pwS_b3, kXc.pwS_b4);
  return e0 - mac * f * (1.0 - z4) / kFpp0 + (e1 - e0) * f * z4;
}

template <class D>
SXC_HD D pbe_c_pol(D ra, D rb, D sigma) {
  Rooted<D> rho = rooted(ra + rb);
  D zeta = (ra - rb) / rho.n;
  Rooted<D> opz = rooted(1.0 + zeta), omz = rooted(1.0 - zeta);
  D eps = pw92_eps_pol(rs_of(rho), zeta, spin_f(opz, omz));
  // phi = ((1+zeta)^(2/3) + (1-zeta)^(2/3)) / 2, arguments kept away from 0 (its slope diverges there)
  if (opz.n.v < 1e-12) opz.c = 1e-4;
  if (omz.n.v < 1e-12) omz.c = 1e-4;
  D phi = 0.5 * (pow23(opz) + pow23(omz));
  D phi3 = phi * phi * phi;
  D t2 = kPbeT2 * sigma / (phi * phi * pow73(rho));
  return rho.n * (eps + pbe_H(eps, t2, phi3));
}

// BP86 correlation, spin-polarised: PZ81 with the spin interpolation f(zeta) between its
// paramagnetic and ferromagnetic fits, P86 correction of the total density with
// d(zeta) = 2^(1/3) sqrt(((1+zeta)/2)^(5/3) + ((1-zeta)/2)^(5/3))
template <class D>
SXC_HD D bp86_c_pol(D ra, D rb, D sigma) {
  Rooted<D> rho = rooted(ra + rb);
  D rs = rs_of(rho);
  D zeta = (ra - rb) / rho.n;
  Rooted<D> opz = rooted(1.0 + zeta), omz = rooted(1.0 - zeta);
  D f = spin_f(opz, omz);
  D eU = pz81_fit(rs, kXc.pzU_g, kXc.pzU_b1, kXc.pzU_b2, kXc.pzU_A, kXc.pzU_B, kXc.pzU_C, kXc.pzU_D);
  D eP = pz81_fit(rs, kXc.pzP_g, kXc.pzP_b1, kXc.pzP_b2, kXc.pzP_A, kXc.pzP_B, kXc.pzP_C, kXc.pzP_D);
  // 2^(1/3) sqrt(2^(-5/3) (...)) = sqrt((...) / 2)
  D dz = dsqrt(0.5 * (pow53(opz) + pow53(omz)));
  return rho.n * (eU + f * (eP - eU)) + p86_corr(rho, rs, sigma, dz);
}

// Functional ids as in serenity_xc.h.
constexpr int kNumFunctionals = 9;  // LDA, PBE, TF, SLATER, VWN5, PBEX, PBEC, PBE (LibXC constants), BP86
SXC_HD bool functional_is_gga(int f) { return f == 1 || f == 5 || f == 6 || f == 7 || f == 8; }

SXC_HD D2 eval_functional(int f, D2 density, D2 sigma) {
  const Rooted<D2> rho = rooted(density);
  switch (f) {
    case 0:
      return slater_x(rho) + vwn5_c(rho);
    case 1:
      return pbe_x(rho, sigma, kXc.pbe_mu) + pbe_c(rho, sigma);
    case 2:
      return tf_k(rho);
    case 3:
      return slater_x(rho);
    case 4:
      return vwn5_c(rho);
    case 5:
      return pbe_x(rho, sigma, kXc.pbe_mu);
    case 6:
      return pbe_c(rho, sigma);
    case 7:
      return pbe_x(rho, sigma, kXc.pbe_mu_libxc) + pbe_c(rho, sigma);
    case 8:
      return bp86(rho, sigma);
    default:
      return mk(0.0);
  }
}

// Spin-polarised evaluation: v = (rho_a, rho_b, sigma_aa, sigma_ab, sigma_bb) as D5
// variables; a_on / b_on say whether each spin density is above kTinyDensity.
SXC_HD D5 eval_functional_pol(int f, D5 ra, D5 rb, D5 saa, D5 sab, D5 sbb, bool a_on, bool b_on) {
  D5 sigma = saa + 2.0 * sab + sbb;
  D5 e = mkc<5>(0.0);
  // exchange-type parts by spin scaling, E[rho_a, rho_b] = (E[2 rho_a] + E[2 rho_b]) / 2
  // with 4 sigma_ss as the gradient invariant
  // kind: 0 Slater, 1 Thomas-Fermi, 2 PBE exchange (XCFun mu), 3 PBE exchange (LibXC mu), 4 Becke 88
  auto one = [&](int kind, const Rooted<D5>& r2, D5 s4) {
    switch (kind) {
      case 0:
        return slater_x(r2);
      case 1:
        return tf_k(r2);
      case 2:
        return pbe_x(r2, s4, kXc.pbe_mu);
      case 3:
        return pbe_x(r2, s4, kXc.pbe_mu_libxc);
      default:
        return b88_x(r2, s4);
    }
  };
  auto xpart = [&](int kind) {
    D5 out = mkc<5>(0.0);
    if (a_on) {
      D5 r2 = 2.0 * ra, s4 = 4.0 * saa;
      out = out + 0.5 * one(kind, rooted(r2), s4);
    }
    if (b_on) {
      D5 r2 = 2.0 * rb, s4 = 4.0 * sbb;
      out = out + 0.5 * one(kind, rooted(r2), s4);
    }
    return out;
  };
  // a fully polarised point (one spin density zero) keeps the exact zeta = +-1 limits
  D5 ra_c = a_on ? ra : mkc<5>(0.0), rb_c = b_on ? rb : mkc<5>(0.0);
  switch (f) {
    case 0:
      e = xpart(0) + vwn5_c_pol(ra_c, rb_c);
      break;
    case 1:
      e = xpart(2) + pbe_c_pol(ra_c, rb_c, sigma);
      break;
    case 2:
      e = xpart(1);
      break;
    case 3:
      e = xpart(0);
      break;
    case 4:
      e = vwn5_c_pol(ra_c, rb_c);
      break;
    case 5:
      e = xpart(2);
      break;
    case 6:
      e = pbe_c_pol(ra_c, rb_c, sigma);
      break;
    case 7:
      e = xpart(3) + pbe_c_pol(ra_c, rb_c, sigma);
      break;
    case 8:
      e = xpart(4) + bp86_c_pol(ra_c, rb_c, sigma);
      break;
    default:
      break;
  }
  return e;
}

// Densities below this value contribute nothing (energy and potential zero).
constexpr double kTinyDensity = 1e-14;

// One grid point: returns eps and writes v and (for GGA) g = dEps/dGradRho.
SXC_HD double xc_point(int f, double rho, double gx, double gy, double gz, double* v, double* g) {
  g[0] = g[1] = g[2] = 0.0;
  if (!(rho >= kTinyDensity)) {
    *v = 0.0;
    return 0.0;
  }
  const double sigma = gx * gx + gy * gy + gz * gz;
  D2 r = var<2>(rho, 0);
  D2 s = var<2>(sigma, 1);
  D2 e = eval_functional(f, r, s);
  *v = e.d[0];
  if (functional_is_gga(f)) {
    g[0] = 2.0 * e.d[1] * gx;
    g[1] = 2.0 * e.d[1] * gy;
    g[2] = 2.0 * e.d[1] * gz;
  }
  return e.v;
}

// One grid point, spin-polarised: ga / gb are the spin density gradients (3 each);
// writes v[0..1] = d eps/d rho_a, d eps/d rho_b and (GGA) g[0..2] = d eps/d grad rho_a,
// g[3..5] = d eps/d grad rho_b.  Zero when the total density is below kTinyDensity.
SXC_HD double xc_point_pol(int f, double ra, double rb, const double* ga, const double* gb, double* v,
                           double* g) {
  for (int i = 0; i < 6; ++i) g[i] = 0.0;
  v[0] = v[1] = 0.0;
  const bool a_on = ra >= kTinyDensity, b_on = rb >= kTinyDensity;
  if (!(ra + rb >= kTinyDensity) || !(a_on || b_on)) return 0.0;
  const double saa = ga[0] * ga[0] + ga[1] * ga[1] + ga[2] * ga[2];
  const double sbb = gb[0] * gb[0] + gb[1] * gb[1] + gb[2] * gb[2];
  const double sab = ga[0] * gb[0] + ga[1] * gb[1] + ga[2] * gb[2];
  D5 e = eval_functional_pol(f, var<5>(a_on ? ra : 0.0, 0), var<5>(b_on ? rb : 0.0, 1), var<5>(saa, 2),
                             var<5>(sab, 3), var<5>(sbb, 4), a_on, b_on);
  v[0] = e.d[0];
  v[1] = e.d[1];
  if (functional_is_gga(f)) {
    for (int c = 0; c < 3; ++c) {
      g[c] = 2.0 * e.d[2] * ga[c] + e.d[3] * gb[c];
      g[3 + c] = 2.0 * e.d[4] * gb[c] + e.d[3] * ga[c];
    }
  }
  return e.v;
}

}  // namespace sxc

// Device-side physics of the compressible Euler / Navier-Stokes split-form path.
//
// Each function names the reference routine (project-fluxo/fluxo) it computes; the
// arithmetic follows the reference's formulas so that FP64 results agree with the
// reference to rounding.  Three deliberate reformulations, all exact in real
// arithmetic:
//  * the logarithmic mean takes ln(a), ln(b) precomputed once per node, so
//    (b-a)/ln(b/a) becomes (b-a)/(ln b - ln a); the near-equal branch keeps the
//    reference's series and switch (LN_MEAN, navierstokes/flux_average.f90:1945-1965);
//  * surface fluxes are evaluated in the Cartesian frame instead of rotating the
//    momentum into (n,t1,t2) and back (riemann.f90:174-246), which is an
//    orthogonal change of basis;
//  * inside the two-point fluxes, quotients use the hardware reciprocal refined by a
//    Newton step (about 1 ulp) instead of a correctly rounded division.
#pragma once
#include <hip/hip_runtime.h>

namespace fx {

constexpr double LNMEAN_SQEPS = 1.0e-2;  // the reference's switch u = ((b-a)/(a+b))^2 < 1e-4

// Reciprocal from the hardware estimate refined by one Newton step (error ~1 ulp); used
// where a correctly rounded quotient is not needed for FP64 parity at 1e-12.
__device__ __forceinline__ double rcp_nr(double x)
{
  double r = __builtin_amdgcn_rcp(x);
  double e = fma(-x, r, 1.0);
  return fma(r, e, r);
}
__device__ __forceinline__ float rcp_nr(float x) { return __builtin_amdgcn_rcpf(x); }

// Log mean of a, b given la = ln a, lb = ln b, evaluated without branches: the near-equal series
// and the log quotient are formed and one is selected, so divergent lanes cost one quotient instead
// of both paths.  Both share one reciprocal (of a + b for the series, of the quotient's
// denominator otherwise): with q = (b-a)/(a+b) and u = q^2 < 1e-4 the reference's series
// 52.5 (a+b) / (105 + 35 u + 21 u^2 + 15 u^3) is (a+b) times its own expansion in u, whose
// neglected u^4 term is below 4e-18.
template <typename R>
__device__ __forceinline__ R ln_mean(R a, R b, R la, R lb)
{
  const R d = b - a, s = a + b;
  const bool series = fabs(d) < fabs(R(LNMEAN_SQEPS) * s);
  const R q = d * rcp_nr(series ? s : lb - la);
  const R u = q * q;
  const R P = R(0.5) - u * (R(1.0 / 6.0) + u * (R(2.0 / 45.0) + u * R(22.0 / 945.0)));
  return series ? s * P : q;
}

// 1 / ln_mean(a, b)
template <typename R>
__device__ __forceinline__ R inv_ln_mean(R a, R b, R la, R lb)
{
  const R d = b - a, s = a + b;
  const bool series = fabs(d) < fabs(R(LNMEAN_SQEPS) * s);
  const R r = rcp_nr(series ? s : d);
  const R q = d * r, u = q * q;
  const R P = R(2.0) + u * (R(2.0 / 3.0) + u * (R(2.0 / 5.0) + u * R(2.0 / 7.0)));
  return r * (series ? P : lb - la);
}

// FP32 log mean of the split-precision volume integral.  The near-equal branch is kept in
// FP64: with per-node logs rounded to FP32, (b-a)/(ln b - ln a) loses ~|ln a|/|ln b - ln a|
// ulps, so the series of LN_MEAN is used up to u < 4e-2 (|b-a|/(b+a) < 0.2) instead of
// 1e-4; its truncation error u^4/9 stays below 3e-7 there.  u itself is formed in FP32
// (its rounding moves the series value by < 1e-9); the series and its quotient are FP64.
constexpr float LNMEAN_EPS32 = 4.0e-2f;

template <bool INV>
__device__ __forceinline__ float ln_mean32(float a, float b, float la, float lb)
{
  const float d = b - a, s = a + b, d2 = d * d, s2 = s * s;
  const bool series = d2 < LNMEAN_EPS32 * s2;
  const double u = (double)(d2 * rcp_nr(s2));
  const double P = 105.0 + u * (35.0 + u * (21.0 + u * 15.0));
  const double s52 = (double)a * 52.5 + (double)b * 52.5;
  const double ser = INV ? P * rcp_nr(s52) : s52 * rcp_nr(P);
  const float q = INV ? (lb - la) * rcp_nr(d) : d * rcp_nr(lb - la);
  return series ? (float)ser : q;
}
__device__ __forceinline__ float ln_mean(float a, float b, float la, float lb)
{
  return ln_mean32<false>(a, b, la, lb);
}
__device__ __forceinline__ float inv_ln_mean(float a, float b, float la, float lb)
{
  return ln_mean32<true>(a, b, la, lb);
}

// Per-node quantities staged for the two-point fluxes.
//   rho, v1, v2, v3, p, ln(rho), X, ln(X), |v|^2, rhoE
// X = rho/p for Ranocha (RanochaFluxVec), X = beta = rho/(2p) for Chandrashekar
// (EntropyAndEnergyConservingFluxVec); EvalUaux (flux_average.f90:305-332).  For the
// Ismail-Roe flux (VF=10) the slots RHO/LNRHO/X/LNX hold z1 = sqrt(rho/p), ln z1, z5 = z1 p,
// ln z5 (TwoPointEntropyConservingFluxVec flux_average.f90:574-673).
enum { NF_RHO = 0, NF_V1, NF_V2, NF_V3, NF_P, NF_LNRHO, NF_X, NF_LNX, NF_VV, NF_E, NF_COUNT };

// Fields a volume flux reads (the others are never staged).
// NF_E holds rhoE (VF 0, 1, 3), e = rhoE/rho (VF 2), H = (rhoE+p)/rho (VF 8, 9); for VF 9
// NF_RHO holds sqrt(rho); X = beta = rho/(2p) for VF 5, 6, 7.
template <int VF>
__host__ __device__ constexpr bool uses_field(int f)
{
  return (VF == 32 || VF == 10) ? (f <= NF_LNX)
       : VF == 5 ? (f <= NF_VV)
       : VF == 4 ? (f <= NF_P || f == NF_VV)
       : VF == 6 ? (f <= NF_V3 || f == NF_X || f == NF_VV)
       : VF == 7 ? (f <= NF_P || f == NF_X || f == NF_LNX || f == NF_VV)
       : VF == 107 ? (f <= NF_LNX || f == NF_VV)
       : VF == 9 ? (f <= NF_V3 || f == NF_E)
       : (f <= NF_P || f == NF_E);
}
// Volume fluxes with an FP32-split instantiation; the others run in FP64 only.
__host__ __device__ constexpr bool has_fp32(int VF) { return VF == 0 || VF == 5 || VF == 10 || VF == 32; }
template <int VF>
__host__ __device__ constexpr int n_fields()
{
  int c = 0;
  for (int f = 0; f < NF_COUNT; f++) c += uses_field<VF>(f) ? 1 : 0;
  return c;
}
// LDS slot of field f (fields are packed in enum order)
template <int VF>
__host__ __device__ constexpr int field_slot(int f)
{
  int c = 0;
  for (int g = 0; g < f; g++) c += uses_field<VF>(g) ? 1 : 0;
  return c;
}

template <int VF>
__device__ __forceinline__ void node_fields(const double *u, double kappaM1, double *f)
{
  double srho = 1.0 / u[0];
  double v1 = u[1] * srho, v2 = u[2] * srho, v3 = u[3] * srho;
  double vv = v1 * v1 + v2 * v2 + v3 * v3;
  double p = kappaM1 * (u[4] - 0.5 * u[0] * vv);
  f[NF_RHO] = u[0]; f[NF_V1] = v1; f[NF_V2] = v2; f[NF_V3] = v3; f[NF_P] = p; f[NF_VV] = vv;
  f[NF_E] = u[4];
  if (VF == 32) {
    double X = u[0] / p;
    f[NF_LNRHO] = log(u[0]); f[NF_X] = X; f[NF_LNX] = log(X);
  } else if (VF == 5) {
    double X = 0.5 * u[0] / p;
    f[NF_LNRHO] = log(u[0]); f[NF_X] = X; f[NF_LNX] = log(X);
  } else if (VF == 10) {
    double z1 = sqrt(u[0] / p), z5 = z1 * p;
    f[NF_RHO] = z1; f[NF_LNRHO] = log(z1); f[NF_X] = z5; f[NF_LNX] = log(z5);
  } else if (VF == 6 || VF == 7 || VF == 107) {
    double X = 0.5 * u[0] / p;
    f[NF_LNRHO] = VF == 107 ? log(u[0]) : 0.0; f[NF_X] = X; f[NF_LNX] = VF != 6 ? log(X) : 0.0;
  } else if (VF == 2 || VF == 8 || VF == 9) {
    f[NF_E] = VF == 2 ? srho * u[4] : (u[4] + p) * srho;
    if (VF == 9) f[NF_RHO] = sqrt(u[0]);
    f[NF_LNRHO] = 0.0; f[NF_X] = 0.0; f[NF_LNX] = 0.0;
  } else {
    f[NF_LNRHO] = 0.0; f[NF_X] = 0.0; f[NF_LNX] = 0.0;
  }
}

// Metric-dealiased two-point volume flux Fstar(U_L, U_R, {{m}}).
//  VF=32: RanochaFluxVec (flux_average.f90:1876-1929)
//  VF=5 : EntropyAndEnergyConservingFluxVec (flux_average.f90:1277-1356)
//  VF=10: TwoPointEntropyConservingFluxVec, Ismail-Roe (flux_average.f90:574-673)
//  VF=1 : StandardDGFluxDealiasedMetricVec (flux_average.f90:446-494)
//  VF=2 : KennedyAndGruberFluxVec1 (flux_average.f90:731-803)
//  VF=8 : KennedyAndGruberFluxVec2 (flux_average.f90:857-929)
//  VF=3 : DucrosFluxVec (flux_average.f90:986-1059)
//  VF=4 : MorinishiFluxVec (flux_average.f90:1121-1205), kappa/(kappa-1) = 1 + 1/(kappa-1)
//  VF=6 : EntropyAndEnergyConservingFluxVec2 (flux_average.f90:1427-1504)
//  VF=7 : ggFluxVec (flux_average.f90:1580-1653); VF=107 its surface form ggflux
//         (flux_average.f90:1513-1574), whose mass flux takes the log mean of rho
//  VF=9 : GassnerWintersWalchFluxVec (flux_average.f90:1724-1799), (kappa-1)/kappa =
//         1/(1 + 1/(kappa-1))
//  VF=0 : StandardDGFluxVec (flux_average.f90:394-439)
// Momenta rhoU of the reference enter as rho*v (one rounding apart).
template <int VF, typename R>
__device__ __forceinline__ void volume_flux(const R *L, const R *Rt, const R *mL, const R *mR,
                                            R skappaM1, R *F)
{
  if (VF == 32) {
    R m0 = R(0.5) * (mL[0] + mR[0]), m1 = R(0.5) * (mL[1] + mR[1]), m2 = R(0.5) * (mL[2] + mR[2]);
    R rhoLN = ln_mean(L[NF_RHO], Rt[NF_RHO], L[NF_LNRHO], Rt[NF_LNRHO]);
    R va0 = R(0.5) * (L[NF_V1] + Rt[NF_V1]);
    R va1 = R(0.5) * (L[NF_V2] + Rt[NF_V2]);
    R va2 = R(0.5) * (L[NF_V3] + Rt[NF_V3]);
    R v2zip = R(0.5) * (L[NF_V1] * Rt[NF_V1] + L[NF_V2] * Rt[NF_V2] + L[NF_V3] * Rt[NF_V3]);
    R pavg = R(0.5) * (L[NF_P] + Rt[NF_P]);
    R vmL = L[NF_V1] * m0 + L[NF_V2] * m1 + L[NF_V3] * m2;
    R vmR = Rt[NF_V1] * m0 + Rt[NF_V2] * m1 + Rt[NF_V3] * m2;
    R srspM = inv_ln_mean(L[NF_X], Rt[NF_X], L[NF_LNX], Rt[NF_LNX]);
    F[0] = rhoLN * R(0.5) * (vmL + vmR);
    F[1] = F[0] * va0 + m0 * pavg;
    F[2] = F[0] * va1 + m1 * pavg;
    F[3] = F[0] * va2 + m2 * pavg;
    F[4] = F[0] * (v2zip + srspM * skappaM1) + R(0.5) * (L[NF_P] * vmR + Rt[NF_P] * vmL);
  } else if (VF == 5) {
    R m0 = R(0.5) * (mL[0] + mR[0]), m1 = R(0.5) * (mL[1] + mR[1]), m2 = R(0.5) * (mL[2] + mR[2]);
    R rho_mean = R(0.5) * (L[NF_RHO] + Rt[NF_RHO]);
    R rhoHat = ln_mean(L[NF_RHO], Rt[NF_RHO], L[NF_LNRHO], Rt[NF_LNRHO]);
    R beta_mean = R(0.5) * (L[NF_X] + Rt[NF_X]);
    R sbeta_hat = inv_ln_mean(L[NF_X], Rt[NF_X], L[NF_LNX], Rt[NF_LNX]);
    R uH = R(0.5) * (L[NF_V1] + Rt[NF_V1]);
    R vH = R(0.5) * (L[NF_V2] + Rt[NF_V2]);
    R wH = R(0.5) * (L[NF_V3] + Rt[NF_V3]);
    R p1 = R(0.5) * rho_mean / beta_mean;
    R qH = uH * m0 + vH * m1 + wH * m2;
    F[0] = rhoHat * qH;
    F[1] = F[0] * uH + m0 * p1;
    F[2] = F[0] * vH + m1 * p1;
    F[3] = F[0] * wH + m2 * p1;
    F[4] = F[0] * R(0.5) * (skappaM1 * sbeta_hat - R(0.5) * (L[NF_VV] + Rt[NF_VV])) + uH * F[1] +
           vH * F[2] + wH * F[3];
  } else if (VF == 10) {
    R m0 = R(0.5) * (mL[0] + mR[0]), m1 = R(0.5) * (mL[1] + mR[1]), m2 = R(0.5) * (mL[2] + mR[2]);
    const R z1L = L[NF_RHO], z1R = Rt[NF_RHO];
    R z1M = R(0.5) * (z1L + z1R);
    R sz1LN = inv_ln_mean(z1L, z1R, L[NF_LNRHO], Rt[NF_LNRHO]);
    R z5LN = ln_mean(L[NF_X], Rt[NF_X], L[NF_LNX], Rt[NF_LNX]);
    R sz1 = R(1) / z1M;
    R uH = R(0.5) * (z1L * L[NF_V1] + z1R * Rt[NF_V1]) * sz1;
    R vH = R(0.5) * (z1L * L[NF_V2] + z1R * Rt[NF_V2]) * sz1;
    R wH = R(0.5) * (z1L * L[NF_V3] + z1R * Rt[NF_V3]) * sz1;
    R p1 = R(0.5) * (L[NF_X] + Rt[NF_X]) * sz1;
    R qH = uH * m0 + vH * m1 + wH * m2;
    F[0] = z1M * z5LN * qH;
    F[1] = F[0] * uH + m0 * p1;
    F[2] = F[0] * vH + m1 * p1;
    F[3] = F[0] * wH + m2 * p1;
    F[4] = R(0.5) * (qH * (R(1) + R(2) * skappaM1) * (z5LN * sz1LN) + uH * F[1] + vH * F[2] + wH * F[3]);
  } else if (VF == 1) {
    R m0 = R(0.5) * (mL[0] + mR[0]), m1 = R(0.5) * (mL[1] + mR[1]), m2 = R(0.5) * (mL[2] + mR[2]);
    R qL = L[NF_V1] * m0 + L[NF_V2] * m1 + L[NF_V3] * m2;
    R qR = Rt[NF_V1] * m0 + Rt[NF_V2] * m1 + Rt[NF_V3] * m2;
    R rqL = L[NF_RHO] * qL, rqR = Rt[NF_RHO] * qR, ps = L[NF_P] + Rt[NF_P];
    F[0] = R(0.5) * (rqL + rqR);
    F[1] = R(0.5) * (rqL * L[NF_V1] + rqR * Rt[NF_V1] + m0 * ps);
    F[2] = R(0.5) * (rqL * L[NF_V2] + rqR * Rt[NF_V2] + m1 * ps);
    F[3] = R(0.5) * (rqL * L[NF_V3] + rqR * Rt[NF_V3] + m2 * ps);
    F[4] = R(0.5) * ((L[NF_E] + L[NF_P]) * qL + (Rt[NF_E] + Rt[NF_P]) * qR);
  } else if (VF == 2 || VF == 8 || VF == 3) {
    R m0 = R(0.5) * (mL[0] + mR[0]), m1 = R(0.5) * (mL[1] + mR[1]), m2 = R(0.5) * (mL[2] + mR[2]);
    R uH = R(0.5) * (L[NF_V1] + Rt[NF_V1]);
    R vH = R(0.5) * (L[NF_V2] + Rt[NF_V2]);
    R wH = R(0.5) * (L[NF_V3] + Rt[NF_V3]);
    R p1 = R(0.5) * (L[NF_P] + Rt[NF_P]);
    R qH = uH * m0 + vH * m1 + wH * m2;
    F[0] = R(0.5) * (L[NF_RHO] + Rt[NF_RHO]) * qH;
    if (VF == 3) {
      F[1] = R(0.5) * (L[NF_RHO] * L[NF_V1] + Rt[NF_RHO] * Rt[NF_V1]) * qH + m0 * p1;
      F[2] = R(0.5) * (L[NF_RHO] * L[NF_V2] + Rt[NF_RHO] * Rt[NF_V2]) * qH + m1 * p1;
      F[3] = R(0.5) * (L[NF_RHO] * L[NF_V3] + Rt[NF_RHO] * Rt[NF_V3]) * qH + m2 * p1;
      F[4] = (R(0.5) * (L[NF_E] + Rt[NF_E]) + p1) * qH;
    } else {
      F[1] = F[0] * uH + m0 * p1;
      F[2] = F[0] * vH + m1 * p1;
      F[3] = F[0] * wH + m2 * p1;
      F[4] = F[0] * (R(0.5) * (L[NF_E] + Rt[NF_E])) + (VF == 2 ? p1 * qH : R(0));
    }
  } else if (VF == 4) {
    R m0 = R(0.5) * (mL[0] + mR[0]), m1 = R(0.5) * (mL[1] + mR[1]), m2 = R(0.5) * (mL[2] + mR[2]);
    R uH = R(0.5) * (L[NF_V1] + Rt[NF_V1]);
    R vH = R(0.5) * (L[NF_V2] + Rt[NF_V2]);
    R wH = R(0.5) * (L[NF_V3] + Rt[NF_V3]);
    R p1 = R(0.5) * (L[NF_P] + Rt[NF_P]);
    R qL = L[NF_V1] * m0 + L[NF_V2] * m1 + L[NF_V3] * m2;
    R qR = Rt[NF_V1] * m0 + Rt[NF_V2] * m1 + Rt[NF_V3] * m2;
    R rqL = R(0.5) * L[NF_RHO] * qL, rqR = R(0.5) * Rt[NF_RHO] * qR;
    F[0] = rqL + rqR;
    F[1] = F[0] * uH + m0 * p1;
    F[2] = F[0] * vH + m1 * p1;
    F[3] = F[0] * wH + m2 * p1;
    F[4] = R(0.5) * ((R(1) + skappaM1) * (L[NF_P] * qL + Rt[NF_P] * qR) - (rqL * L[NF_VV] + rqR * Rt[NF_VV])) +
           rqL * (L[NF_V1] * uH + L[NF_V2] * vH + L[NF_V3] * wH) +
           rqR * (Rt[NF_V1] * uH + Rt[NF_V2] * vH + Rt[NF_V3] * wH);
  } else if (VF == 6 || VF == 7 || VF == 107) {
    R m0 = R(0.5) * (mL[0] + mR[0]), m1 = R(0.5) * (mL[1] + mR[1]), m2 = R(0.5) * (mL[2] + mR[2]);
    R rho_mean = VF == 107 ? ln_mean(L[NF_RHO], Rt[NF_RHO], L[NF_LNRHO], Rt[NF_LNRHO])
                           : R(0.5) * (L[NF_RHO] + Rt[NF_RHO]);
    R uH = R(0.5) * (L[NF_V1] + Rt[NF_V1]);
    R vH = R(0.5) * (L[NF_V2] + Rt[NF_V2]);
    R wH = R(0.5) * (L[NF_V3] + Rt[NF_V3]);
    R sbeta, p1;
    if (VF == 6) {
      sbeta = R(2) * rcp_nr(L[NF_X] + Rt[NF_X]);
      p1 = R(0.5) * rho_mean * sbeta;
    } else {
      sbeta = inv_ln_mean(L[NF_X], Rt[NF_X], L[NF_LNX], Rt[NF_LNX]);
      p1 = R(0.5) * (L[NF_P] + Rt[NF_P]);
    }
    R qH = uH * m0 + vH * m1 + wH * m2;
    F[0] = rho_mean * qH;
    F[1] = F[0] * uH + m0 * p1;
    F[2] = F[0] * vH + m1 * p1;
    F[3] = F[0] * wH + m2 * p1;
    F[4] = F[0] * R(0.5) * (skappaM1 * sbeta - R(0.5) * (L[NF_VV] + Rt[NF_VV])) + uH * F[1] + vH * F[2] +
           wH * F[3];
  } else if (VF == 9) {
    R m0 = R(0.5) * (mL[0] + mR[0]), m1 = R(0.5) * (mL[1] + mR[1]), m2 = R(0.5) * (mL[2] + mR[2]);
    const R sL = L[NF_RHO], sR = Rt[NF_RHO];
    R rhoH = R(0.5) * (sL + sR);
    R uH = R(0.5) * (sL * L[NF_V1] + sR * Rt[NF_V1]);
    R vH = R(0.5) * (sL * L[NF_V2] + sR * Rt[NF_V2]);
    R wH = R(0.5) * (sL * L[NF_V3] + sR * Rt[NF_V3]);
    R HH = R(0.5) * (sL * L[NF_E] + sR * Rt[NF_E]);
    R p1 = (rhoH * HH - R(0.5) * (uH * uH + vH * vH + wH * wH)) * rcp_nr(R(1) + skappaM1);
    R qH = uH * m0 + vH * m1 + wH * m2;
    F[0] = rhoH * qH;
    F[1] = qH * uH + m0 * p1;
    F[2] = qH * vH + m1 * p1;
    F[3] = qH * wH + m2 * p1;
    F[4] = qH * HH;
  } else {
    R qL = L[NF_V1] * mL[0] + L[NF_V2] * mL[1] + L[NF_V3] * mL[2];
    R qR = Rt[NF_V1] * mR[0] + Rt[NF_V2] * mR[1] + Rt[NF_V3] * mR[2];
    F[0] = R(0.5) * (L[NF_RHO] * qL + Rt[NF_RHO] * qR);
    F[1] = R(0.5) * (L[NF_RHO] * L[NF_V1] * qL + Rt[NF_RHO] * Rt[NF_V1] * qR + mL[0] * L[NF_P] + mR[0] * Rt[NF_P]);
    F[2] = R(0.5) * (L[NF_RHO] * L[NF_V2] * qL + Rt[NF_RHO] * Rt[NF_V2] * qR + mL[1] * L[NF_P] + mR[1] * Rt[NF_P]);
    F[3] = R(0.5) * (L[NF_RHO] * L[NF_V3] * qL + Rt[NF_RHO] * Rt[NF_V3] * qR + mL[2] * L[NF_P] + mR[2] * Rt[NF_P]);
    F[4] = R(0.5) * ((L[NF_E] + L[NF_P]) * qL + (Rt[NF_E] + Rt[NF_P]) * qR);
  }
}

// The two-point fluxes as the node-form volume kernel evaluates them.  For the Ranocha flux the
// factors 1/2 of its means are taken out of the pair loop, which that kernel's vector
// instructions bound: the metrics come halved (hL, hR, so that {{m}} = hL + hR), the result is twice
// the flux and belongs with halved operator entries (two_point_ds).  With the means' single
// reciprocal it takes 64 instead of 87 FP64 instructions (LSERK kernel at N = 5, 13^3 elements: 45 -> 39 us).
// The other fluxes are volume_flux as it stands.
__host__ __device__ constexpr bool two_point_halved(int VF) { return VF == 32; }
template <int VF>
__device__ __forceinline__ void two_point(const double *L, const double *Rt, const double *hL, const double *hR,
                                          double skappaM1, double *F)
{
  if constexpr (two_point_halved(VF)) {
    const double m0 = hL[0] + hR[0], m1 = hL[1] + hR[1], m2 = hL[2] + hR[2];
    const double vmL = L[NF_V1] * m0 + L[NF_V2] * m1 + L[NF_V3] * m2;
    const double vmR = Rt[NF_V1] * m0 + Rt[NF_V2] * m1 + Rt[NF_V3] * m2;
    const double ps = L[NF_P] + Rt[NF_P];
    const double vv = L[NF_V1] * Rt[NF_V1] + L[NF_V2] * Rt[NF_V2] + L[NF_V3] * Rt[NF_V3];
    const double sx = inv_ln_mean(L[NF_X], Rt[NF_X], L[NF_LNX], Rt[NF_LNX]);
    const double f0 = ln_mean(L[NF_RHO], Rt[NF_RHO], L[NF_LNRHO], Rt[NF_LNRHO]) * (vmL + vmR), fh = 0.5 * f0;
    F[0] = f0;
    F[1] = fh * (L[NF_V1] + Rt[NF_V1]) + m0 * ps;
    F[2] = fh * (L[NF_V2] + Rt[NF_V2]) + m1 * ps;
    F[3] = fh * (L[NF_V3] + Rt[NF_V3]) + m2 * ps;
    F[4] = fh * (vv + sx * (2.0 * skappaM1)) + (L[NF_P] * vmR + Rt[NF_P] * vmL);
  } else {
    volume_flux<VF, double>(L, Rt, hL, hR, skappaM1, F);
  }
}

// Numerical surface flux in the normal direction n (unit), unscaled by SurfElem.
//  RS=1 : RiemannSolverByRusanov (riemann.f90:279-313) with EvalEulerFlux1D (flux.f90:298-329)
//  RS=0 : RiemannSolverCentral (riemann.f90:251-272)
//  RS=32: RiemannSolver_VolumeFluxAverage + RanochaFlux (riemann.f90:980-1005,
//         flux_average.f90:1806-1866)
//  RS=9 : RiemannSolver_VolumeFluxAverage + EntropyAndEnergyConservingFlux
//         (flux_average.f90:1214-1270)
// Two-point flux of the volume-flux-average surface fluxes (equation.f90:292-404): Riemann
// 6 / 14 Kennedy-Gruber 1, 7 / 15 Ducros, 8 / 19 Morinishi, 10 EC with arithmetic means,
// 11 / 17 gg (surface form), 12 / 18 Kennedy-Gruber 2, 20 / 21 Gassner-Winters-Walch; -1 for
// the others.  Riemann 5 (Ismail-Roe) runs through riemann_es.
__host__ __device__ constexpr int riemann_volflux(int RS)
{
  return (RS == 6 || RS == 14) ? 2 : (RS == 7 || RS == 15) ? 3 : (RS == 8 || RS == 19) ? 4 : RS == 10 ? 6
       : (RS == 11 || RS == 17) ? 107 : (RS == 12 || RS == 18) ? 8 : (RS == 20 || RS == 21) ? 9 : -1;
}
// Surface fluxes that take the face-wide largest wave speed LambdaMaxMax (riemann.f90:1011-1209).
__host__ __device__ constexpr bool riemann_face_lambda(int RS)
{
  return RS == 13 || RS == 14 || RS == 15 || RS == 16 || RS == 17 || RS == 18 || RS == 19 || RS == 21;
}

// HLL-type and Roe solvers in the Cartesian frame (the reference rotates into (n, t1, t2),
// riemann.f90:174-246; every formula below is the rotated one written with n and the
// tangential projection v - (v.n) n):
//   RS=2  : RiemannSolverByHLLC (riemann.f90:552-615)
//   RS=22 : RiemannSolverByHLL (:320-388), its wave speeds from the Roe-averaged normal
//           velocity alone
//   RS=23 : RiemannSolverByHLLE (:396-462); RS=24 HLLEM (:468-547) with the anti-diffusion
//           of the contact and shear waves
//   RS=3  : RiemannSolverByRoe (:746-869) with the average of the Euler fluxes as central
//           part; 302 / 303 / 308 with the Kennedy-Gruber 1 / Ducros / Kennedy-Gruber 2
//           two-point flux, the reference's choice for VolumeFlux 2 / 3 / 4 (split form),
//           302 and 308 with max(|u-c|,|u+c|) on both acoustic waves.
template <int RS>
__device__ __forceinline__ void riemann_hll_roe(const double *UL, const double *UR, const double *n, double kappa,
                                                double *F)
{
  const double km1 = kappa - 1.0;
  const double sL = 1.0 / UL[0], sR = 1.0 / UR[0];
  const double vL[3] = {UL[1] * sL, UL[2] * sL, UL[3] * sL}, vR[3] = {UR[1] * sR, UR[2] * sR, UR[3] * sR};
  const double pL = km1 * (UL[4] - 0.5 * (UL[1] * vL[0] + UL[2] * vL[1] + UL[3] * vL[2]));
  const double pR = km1 * (UR[4] - 0.5 * (UR[1] * vR[0] + UR[2] * vR[1] + UR[3] * vR[2]));
  const double unL = vL[0] * n[0] + vL[1] * n[1] + vL[2] * n[2], unR = vR[0] * n[0] + vR[1] * n[1] + vR[2] * n[2];
  double FL[5], FR[5];
  FL[0] = UL[1] * n[0] + UL[2] * n[1] + UL[3] * n[2];
  FR[0] = UR[1] * n[0] + UR[2] * n[1] + UR[3] * n[2];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    FL[1 + d] = UL[1 + d] * unL + pL * n[d];
    FR[1 + d] = UR[1 + d] * unR + pR * n[d];
  }
  FL[4] = (UL[4] + pL) * unL;
  FR[4] = (UR[4] + pR) * unR;
  if constexpr (RS == 2) {
    const double Ssl = unL - sqrt(kappa * pL * sL), Ssr = unR + sqrt(kappa * pR * sR);
    if (Ssl >= 0.0) {
#pragma unroll
      for (int v = 0; v < 5; v++) F[v] = FL[v];
      return;
    }
    if (Ssr <= 0.0) {
#pragma unroll
      for (int v = 0; v < 5; v++) F[v] = FR[v];
      return;
    }
    const double sMuL = Ssl - unL, sMuR = Ssr - unR;
    const double SStar = (pR - pL + FL[0] * sMuL - FR[0] * sMuR) / (UL[0] * sMuL - UR[0] * sMuR);
    const bool left = (Ssl <= 0.0) && (SStar >= 0.0);
    const double *u = left ? UL : UR, *Fk = left ? FL : FR, *vk = left ? vL : vR;
    const double sk = left ? sL : sR, sMu = left ? sMuL : sMuR, Ss = left ? Ssl : Ssr, pk = left ? pL : pR;
    const double unk = left ? unL : unR;
    const double c = u[0] * sMu / (Ss - SStar);
    F[0] = Fk[0] + Ss * (c - u[0]);
#pragma unroll
    for (int d = 0; d < 3; d++) F[1 + d] = Fk[1 + d] + Ss * (c * (SStar * n[d] + (vk[d] - unk * n[d])) - u[1 + d]);
    F[4] = Fk[4] + Ss * (c * (u[4] * sk + (SStar - unk) * (SStar + pk * sk / sMu)) - u[4]);
    return;
  }
  const double HL = (UL[4] + pL) * sL, HR = (UR[4] + pR) * sR;
  const double qL = sqrt(UL[0]), qR = sqrt(UR[0]);
  if constexpr (RS == 22) {
    const double Ht = (qL * HL + qR * HR) / (qL + qR), vt = (qL * unL + qR * unR) / (qL + qR);
    const double at = sqrt(km1 * (Ht - 0.5 * vt * vt));
    const double Ssl = vt - at, Ssr = vt + at;
    if (Ssl >= 0.0 && Ssr > 0.0) {
#pragma unroll
      for (int v = 0; v < 5; v++) F[v] = FL[v];
    } else if (Ssr <= 0.0 && Ssl < 0.0) {
#pragma unroll
      for (int v = 0; v < 5; v++) F[v] = FR[v];
    } else {
      const double sd = 1.0 / (Ssr - Ssl);
#pragma unroll
      for (int v = 0; v < 5; v++) F[v] = (Ssr * FL[v] - Ssl * FR[v] + Ssl * Ssr * (UR[v] - UL[v])) * sd;
    }
    return;
  }
  const double sq = 1.0 / (qL + qR);
  double rv[3];
#pragma unroll
  for (int d = 0; d < 3; d++) rv[d] = (qR * vR[d] + qL * vL[d]) * sq;
  const double rH = (qR * HR + qL * HL) * sq, av = rv[0] * rv[0] + rv[1] * rv[1] + rv[2] * rv[2];
  const double rc = sqrt(km1 * (rH - 0.5 * av));
  const double un = rv[0] * n[0] + rv[1] * n[1] + rv[2] * n[2];
  if constexpr (RS == 23 || RS == 24) {
    const double beta = sqrt(0.5 * km1 / kappa);
    const double aL = sqrt(kappa * pL * sL), aR = sqrt(kappa * pR * sR);
    const double Ssl = fmin(fmin(un - rc, unL - beta * aL), 0.0);
    const double Ssr = fmax(fmax(un + rc, unR + beta * aR), 0.0);
    if (Ssl >= 0.0 && Ssr > 0.0) {
#pragma unroll
      for (int v = 0; v < 5; v++) F[v] = FL[v];
      return;
    }
    if (Ssr <= 0.0 && Ssl < 0.0) {
#pragma unroll
      for (int v = 0; v < 5; v++) F[v] = FR[v];
      return;
    }
    double anti[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    if (RS == 24) {
      const double delta = rc / (rc + fabs(0.5 * (Ssl + Ssr)));
      const double rd = sqrt(UL[0] * UR[0]);
      const double A2 = (UR[0] - UL[0]) - (pR - pL) / (rc * rc);
      double dvt[3];
#pragma unroll
      for (int d = 0; d < 3; d++) dvt[d] = rd * ((vR[d] - vL[d]) - ((unR - unL) * n[d]));
      anti[0] = delta * A2;
#pragma unroll
      for (int d = 0; d < 3; d++) anti[1 + d] = delta * (rv[d] * A2 + dvt[d]);
      anti[4] = delta * (0.5 * av * A2 + rv[0] * dvt[0] + rv[1] * dvt[1] + rv[2] * dvt[2]);
    }
    const double sd = 1.0 / (Ssr - Ssl);
#pragma unroll
    for (int v = 0; v < 5; v++) F[v] = (Ssr * FL[v] - Ssl * FR[v] + Ssl * Ssr * (UR[v] - UL[v] - anti[v])) * sd;
    return;
  }
  // Roe: [U], the tangential momentum jump relative to the Roe velocity, the wave strengths
  double dU[5];
#pragma unroll
  for (int v = 0; v < 5; v++) dU[v] = UR[v] - UL[v];
  const double dmn = dU[1] * n[0] + dU[2] * n[1] + dU[3] * n[2];
  double At[3];
#pragma unroll
  for (int d = 0; d < 3; d++) At[d] = (dU[1 + d] - rv[d] * dU[0]) - (dmn - un * dU[0]) * n[d];
  const double dU6 = dU[4] - (At[0] * rv[0] + At[1] * rv[1] + At[2] * rv[2]);
  const double A2 = km1 / (rc * rc) * (dU[0] * (rH - un * un) - dU6 + un * dmn);
  const double A1 = 0.5 / rc * (dU[0] * (un + rc) - dmn - rc * A2);
  const double A5 = dU[0] - A1 - A2;
  double a1 = fabs(un - rc), a5 = fabs(un + rc);
  const double a2 = fabs(un);
  double Fc[5];
  if constexpr (RS == 302 || RS == 303 || RS == 308) {
    constexpr int VFC = RS - 300;
    double fL[NF_COUNT], fR[NF_COUNT];
    node_fields<VFC>(UL, km1, fL);
    node_fields<VFC>(UR, km1, fR);
    volume_flux<VFC, double>(fL, fR, n, n, 1.0 / km1, Fc);
    if (RS != 303) { a1 = fmax(a1, a5); a5 = a1; }
  } else {
#pragma unroll
    for (int v = 0; v < 5; v++) Fc[v] = 0.5 * (FL[v] + FR[v]);
  }
  const double w1 = A1 * a1, w2 = A2 * a2, w5 = A5 * a5;
  F[0] = Fc[0] - 0.5 * (w1 + w2 + w5);
#pragma unroll
  for (int d = 0; d < 3; d++)
    F[1 + d] = Fc[1 + d] - 0.5 * (w1 * (rv[d] - rc * n[d]) + w2 * rv[d] + a2 * At[d] + w5 * (rv[d] + rc * n[d]));
  F[4] = Fc[4] - 0.5 * (w1 * (rH - un * rc) + w2 * 0.5 * av + a2 * (At[0] * rv[0] + At[1] * rv[1] + At[2] * rv[2]) +
                        w5 * (rH + un * rc));
}

template <int RS>
__device__ __forceinline__ void riemann(const double *UL, const double *UR, const double *nv,
                                        double kappa, double *F, double lam_face = 0.0)
{
  const double km1 = kappa - 1.0;
  double sL = 1.0 / UL[0], sR = 1.0 / UR[0];
  double vL[3] = {UL[1] * sL, UL[2] * sL, UL[3] * sL};
  double vR[3] = {UR[1] * sR, UR[2] * sR, UR[3] * sR};
  if (RS == 0 || RS == 1) {
    double mnL = UL[1] * nv[0] + UL[2] * nv[1] + UL[3] * nv[2];   // rotated rho*u_n
    double mnR = UR[1] * nv[0] + UR[2] * nv[1] + UR[3] * nv[2];
    double unL = mnL * sL, unR = mnR * sR;
    double pL = km1 * (UL[4] - 0.5 * (UL[1] * vL[0] + UL[2] * vL[1] + UL[3] * vL[2]));
    double pR = km1 * (UR[4] - 0.5 * (UR[1] * vR[0] + UR[2] * vR[1] + UR[3] * vR[2]));
    double FL[5], FR[5];
    FL[0] = mnL; FR[0] = mnR;
    FL[1] = UL[1] * unL + pL * nv[0]; FR[1] = UR[1] * unR + pR * nv[0];
    FL[2] = UL[2] * unL + pL * nv[1]; FR[2] = UR[2] * unR + pR * nv[1];
    FL[3] = UL[3] * unL + pL * nv[2]; FR[3] = UR[3] * unR + pR * nv[2];
    FL[4] = (UL[4] + pL) * unL;       FR[4] = (UR[4] + pR) * unR;
    if (RS == 0) {
#pragma unroll
      for (int v = 0; v < 5; v++) F[v] = 0.5 * (FL[v] + FR[v]);
    } else {
      double mm2L = mnL * mnL, mm2R = mnR * mnR;
      (void)mm2L; (void)mm2R;
      double c2L = kappa * km1 * (UL[4] * UL[0] - 0.5 * (UL[1] * UL[1] + UL[2] * UL[2] + UL[3] * UL[3])) / (UL[0] * UL[0]);
      double c2R = kappa * km1 * (UR[4] * UR[0] - 0.5 * (UR[1] * UR[1] + UR[2] * UR[2] + UR[3] * UR[3])) / (UR[0] * UR[0]);
      double lam = fmax(fabs(mnL / UL[0]), fabs(mnR / UR[0])) + sqrt(fmax(c2L, c2R));
#pragma unroll
      for (int v = 0; v < 5; v++) F[v] = 0.5 * ((FL[v] + FR[v]) - lam * (UR[v] - UL[v]));
    }
  } else if constexpr (RS == 2 || RS == 22 || RS == 23 || RS == 24 || RS == 3 || RS == 302 || RS == 303 ||
                       RS == 308) {
    riemann_hll_roe<RS>(UL, UR, nv, kappa, F);
  } else if constexpr (riemann_volflux(RS) >= 0) {
    // RiemannSolver_VolumeFluxAverage (riemann.f90:980-1005) and, with the face's
    // LambdaMaxMax, RiemannSolver_VolumeFluxAverage_LLF (:1118-1151)
    constexpr int VFS = riemann_volflux(RS);
    double fL[NF_COUNT], fR[NF_COUNT];
    node_fields<VFS>(UL, km1, fL);
    node_fields<VFS>(UR, km1, fR);
    volume_flux<VFS, double>(fL, fR, nv, nv, 1.0 / km1, F);
    if (riemann_face_lambda(RS)) {
#pragma unroll
      for (int v = 0; v < 5; v++) F[v] = F[v] - 0.5 * lam_face * (UR[v] - UL[v]);
    }
  } else {
    double vv_L = vL[0] * vL[0] + vL[1] * vL[1] + vL[2] * vL[2];
    double vv_R = vR[0] * vR[0] + vR[1] * vR[1] + vR[2] * vR[2];
    double pL = km1 * (UL[4] - 0.5 * UL[0] * vv_L);
    double pR = km1 * (UR[4] - 0.5 * UR[0] * vv_R);
    double fL[NF_COUNT], fR[NF_COUNT];
    fL[NF_RHO] = UL[0]; fL[NF_V1] = vL[0]; fL[NF_V2] = vL[1]; fL[NF_V3] = vL[2]; fL[NF_P] = pL;
    fR[NF_RHO] = UR[0]; fR[NF_V1] = vR[0]; fR[NF_V2] = vR[1]; fR[NF_V3] = vR[2]; fR[NF_P] = pR;
    fL[NF_VV] = vv_L; fR[NF_VV] = vv_R; fL[NF_E] = UL[4]; fR[NF_E] = UR[4];
    fL[NF_LNRHO] = log(UL[0]); fR[NF_LNRHO] = log(UR[0]);
    if (RS == 32) { fL[NF_X] = UL[0] / pL; fR[NF_X] = UR[0] / pR; }
    else { fL[NF_X] = 0.5 * UL[0] / pL; fR[NF_X] = 0.5 * UR[0] / pR; }
    fL[NF_LNX] = log(fL[NF_X]); fR[NF_LNX] = log(fR[NF_X]);
    volume_flux<(RS == 32 ? 32 : 5), double>(fL, fR, nv, nv, 1.0 / km1, F);
  }
}

// Entropy-stable surface fluxes in the Cartesian frame.  The reference rotates the states
// into (n, t1, t2) (riemann.f90:174-246) and applies, at one face point,
//   RS=4, 44, 33: RiemannSolver_EntropyStable (riemann.f90:874-975): the Ismail-Roe
//     (TwoPointEntropyConservingFlux flux_average.f90:500-572), Chandrashekar
//     (EntropyAndEnergyConservingFlux :1214-1269) or Ranocha (RanochaFlux :1806-1866) flux
//     minus 1/2 R D R^T [v] (entropy variables v, right eigenvectors R, D of the averaged
//     state: 1/2|u-a| rho/kappa, |u|(kappa-1)/kappa rho, |u| p1 (twice), 1/2|u+a| rho/kappa);
//   RS=16: RiemannSolver_ECKEP_LLF (riemann.f90:1157-1209): the Chandrashekar flux minus
//     1/2 lam times the entropy-consistent jump, lam the face's largest wave speed.
// Here the averaged velocity stays a Cartesian vector vh (u = vh.n is the normal part), the
// eigenvectors of the two tangential waves enter only through their sum, which is the
// projection onto the face plane; the result equals the rotated-back reference flux in
// exact arithmetic.
__device__ __forceinline__ double ln_mean2(double a, double b) { return ln_mean(a, b, log(a), log(b)); }

template <int RS>
__device__ __forceinline__ void riemann_es(const double *UL, const double *UR, const double *n, double kappa,
                                           double lam_face, double *F)
{
  const double km1 = kappa - 1.0, skm1 = 1.0 / km1;
  const double sL = 1.0 / UL[0], sR = 1.0 / UR[0];
  const double vL[3] = {UL[1] * sL, UL[2] * sL, UL[3] * sL}, vR[3] = {UR[1] * sR, UR[2] * sR, UR[3] * sR};
  const double pL = km1 * (UL[4] - 0.5 * (UL[1] * vL[0] + UL[2] * vL[1] + UL[3] * vL[2]));
  const double pR = km1 * (UR[4] - 0.5 * (UR[1] * vR[0] + UR[2] * vR[1] + UR[3] * vR[2]));
  const double vnL = vL[0] * n[0] + vL[1] * n[1] + vL[2] * n[2];
  const double vnR = vR[0] * n[0] + vR[1] * n[1] + vR[2] * n[2];
  double rhoH, vh[3], p1H, aH, HH, Fc[5];
  if (RS == 4 || RS == 5 || RS == 13) {  // Ismail-Roe
    const double z1L = sqrt(UL[0] / pL), z1R = sqrt(UR[0] / pR);
    const double z1M = 0.5 * (z1L + z1R), z1LN = ln_mean2(z1L, z1R);
    const double z5L = pL * z1L, z5R = pR * z1R;
    const double z5M = 0.5 * (z5L + z5R), z5LN = ln_mean2(z5L, z5R);
    rhoH = z1M * z5LN;
    const double sz1 = 1.0 / z1M;
#pragma unroll
    for (int d = 0; d < 3; d++) vh[d] = (0.5 * (z1L * vL[d] + z1R * vR[d])) * sz1;
    p1H = z5M * sz1;
    const double kp2 = 0.5 * ((kappa + 1.0) * (z5LN / z1LN) + km1 * p1H);
    aH = sqrt(kp2 / rhoH);
    HH = kp2 / (rhoH * km1) + 0.5 * (vh[0] * vh[0] + vh[1] * vh[1] + vh[2] * vh[2]);
    const double un = vh[0] * n[0] + vh[1] * n[1] + vh[2] * n[2];
    Fc[0] = rhoH * un;
#pragma unroll
    for (int d = 0; d < 3; d++) Fc[1 + d] = Fc[0] * vh[d] + p1H * n[d];
    Fc[4] = Fc[0] * HH;
    if (RS == 5) {  // RiemannSolver_VolumeFluxAverage with TwoPointEntropyConservingFlux
#pragma unroll
      for (int v = 0; v < 5; v++) F[v] = Fc[v];
      return;
    }
  } else if (RS == 44 || RS == 16) {  // Chandrashekar
    const double v2s2L = 0.5 * (vL[0] * vL[0] + vL[1] * vL[1] + vL[2] * vL[2]);
    const double v2s2R = 0.5 * (vR[0] * vR[0] + vR[1] * vR[1] + vR[2] * vR[2]);
    const double bL = 0.5 * UL[0] / pL, bR = 0.5 * UR[0] / pR;
    rhoH = ln_mean2(UL[0], UR[0]);
    const double bH = ln_mean2(bL, bR);
#pragma unroll
    for (int d = 0; d < 3; d++) vh[d] = 0.5 * (vL[d] + vR[d]);
    aH = sqrt(kappa * 0.5 * (pL + pR) / rhoH);
    HH = kappa / (2.0 * km1 * bH) + 0.5 * (vL[0] * vR[0] + vL[1] * vR[1] + vL[2] * vR[2]);
    p1H = 0.5 * (0.5 * (UL[0] + UR[0])) / (0.5 * (bL + bR));
    const double un = vh[0] * n[0] + vh[1] * n[1] + vh[2] * n[2];
    Fc[0] = rhoH * un;
#pragma unroll
    for (int d = 0; d < 3; d++) Fc[1 + d] = Fc[0] * vh[d] + p1H * n[d];
    Fc[4] = Fc[0] * 0.5 * (skm1 / bH - (v2s2L + v2s2R)) + (vh[0] * Fc[1] + vh[1] * Fc[2] + vh[2] * Fc[3]);
    if (RS == 16) {
      const double rhoa = 0.5 * (UR[0] + UL[0]);
      const double jump = (0.5 / (km1 * bH) + 0.5 * (vL[0] * vR[0] + vL[1] * vR[1] + vL[2] * vR[2])) * (UR[0] - UL[0]) +
                          rhoa * (vh[0] * (vR[0] - vL[0]) + vh[1] * (vR[1] - vL[1]) + vh[2] * (vR[2] - vL[2]) +
                                  0.5 / km1 * (1.0 / bR - 1.0 / bL));
#pragma unroll
      for (int v = 0; v < 4; v++) F[v] = Fc[v] - 0.5 * lam_face * (UR[v] - UL[v]);
      F[4] = Fc[4] - 0.5 * lam_face * jump;
      return;
    }
  } else {  // Ranocha (33)
    rhoH = ln_mean2(UL[0], UR[0]);
#pragma unroll
    for (int d = 0; d < 3; d++) vh[d] = 0.5 * (vL[d] + vR[d]);
    const double v2zip = 0.5 * (vL[0] * vR[0] + vL[1] * vR[1] + vL[2] * vR[2]);
    p1H = 0.5 * (pL + pR);
    aH = sqrt(kappa * p1H / rhoH);
    HH = kappa * p1H * skm1 / rhoH + 0.5 * (vh[0] * vh[0] + vh[1] * vh[1] + vh[2] * vh[2]);
    const double rspM = ln_mean2(UL[0] / pL, UR[0] / pR);
    const double un = vh[0] * n[0] + vh[1] * n[1] + vh[2] * n[2];
    Fc[0] = rhoH * un;
#pragma unroll
    for (int d = 0; d < 3; d++) Fc[1 + d] = Fc[0] * vh[d] + p1H * n[d];
    Fc[4] = Fc[0] * (v2zip + 1.0 / rspM * skm1) + 0.5 * (pL * vnR + pR * vnL);
  }
  // 1/2 R D R^T [v]
  const double un = vh[0] * n[0] + vh[1] * n[1] + vh[2] * n[2];
  const double D1 = 0.5 * fabs(un - aH) * rhoH / kappa, D2 = fabs(un) * (km1 / kappa) * rhoH;
  const double D3 = fabs(un) * p1H, D5 = 0.5 * fabs(un + aH) * rhoH / kappa;
  const double rpL = UL[0] / pL, rpR = UR[0] / pR;
  const double sEL = log(pL) - kappa * log(UL[0]), sER = log(pR) - kappa * log(UR[0]);
  const double wv2L = vL[0] * vL[0] + vL[1] * vL[1] + vL[2] * vL[2];
  const double wv2R = vR[0] * vR[0] + vR[1] * vR[1] + vR[2] * vR[2];
  const double dv0 = ((kappa - sER) / km1 - 0.5 * rpR * wv2R) - ((kappa - sEL) / km1 - 0.5 * rpL * wv2L);
  double dm[3];
#pragma unroll
  for (int d = 0; d < 3; d++) dm[d] = rpR * vR[d] - rpL * vL[d];
  const double dv4 = rpL - rpR;  // -rho/p
  const double dmn = dm[0] * n[0] + dm[1] * n[1] + dm[2] * n[2];
  const double dmv = dm[0] * vh[0] + dm[1] * vh[1] + dm[2] * vh[2];
  const double vh2 = vh[0] * vh[0] + vh[1] * vh[1] + vh[2] * vh[2];
  if (RS == 13) {
    // RiemannSolver_EC_LLF (riemann.f90:1011-1112): Fc - 1/2 lam H [v] with H = dU/dv at the
    // Ismail-Roe averages (a Cartesian-frame form of the reference's rotated 5x5 matrix)
    const double rhoea = p1H * skm1 + 0.5 * rhoH * vh2;
    const double h0 = rhoH * dv0 + rhoH * dmv + rhoea * dv4;
    F[0] = Fc[0] - 0.5 * lam_face * h0;
#pragma unroll
    for (int d = 0; d < 3; d++)
      F[1 + d] = Fc[1 + d] - 0.5 * lam_face * (rhoH * vh[d] * (dv0 + dmv + HH * dv4) + p1H * dm[d]);
    F[4] = Fc[4] - 0.5 * lam_face * (rhoea * dv0 + rhoH * HH * dmv + (rhoH * HH * HH - aH * aH * p1H * skm1) * dv4);
    return;
  }
  const double c1 = D1 * (dv0 + dmv - aH * dmn + (HH - un * aH) * dv4);
  const double c2 = D2 * (dv0 + dmv + 0.5 * vh2 * dv4);
  const double c5 = D5 * (dv0 + dmv + aH * dmn + (HH + un * aH) * dv4);
  double wt[3], vt[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    vt[d] = vh[d] - un * n[d];
    wt[d] = (dm[d] - dmn * n[d]) + dv4 * vt[d];
  }
  const double vtw = vt[0] * wt[0] + vt[1] * wt[1] + vt[2] * wt[2];
  F[0] = Fc[0] - 0.5 * (c1 + c2 + c5);
#pragma unroll
  for (int d = 0; d < 3; d++)
    F[1 + d] = Fc[1 + d] - 0.5 * (c1 * (vh[d] - aH * n[d]) + c2 * vh[d] + c5 * (vh[d] + aH * n[d]) + D3 * wt[d]);
  F[4] = Fc[4] - 0.5 * (c1 * (HH - un * aH) + c2 * 0.5 * vh2 + c5 * (HH + un * aH) + D3 * vtw);
}

// The largest wave speed of one face point (the LambdaMaxMax term of riemann.f90:1176-1181).
__device__ __forceinline__ double face_lambda(const double *UL, const double *UR, const double *n, double kappa)
{
  const double km1 = kappa - 1.0;
  const double mL = UL[1] * n[0] + UL[2] * n[1] + UL[3] * n[2], mR = UR[1] * n[0] + UR[2] * n[1] + UR[3] * n[2];
  const double c2L = kappa * km1 * (UL[4] * UL[0] - 0.5 * (UL[1] * UL[1] + UL[2] * UL[2] + UL[3] * UL[3])) / (UL[0] * UL[0]);
  const double c2R = kappa * km1 * (UR[4] * UR[0] - 0.5 * (UR[1] * UR[1] + UR[2] * UR[2] + UR[3] * UR[3])) / (UR[0] * UR[0]);
  return fmax(fabs(mL / UL[0]), fabs(mR / UR[0])) + sqrt(fmax(c2L, c2R));
}

// 1/rho, velocity, |v|^2/2 and pressure of a state.  The lifting kernel forms entropy variables,
// primitive gradients and viscous fluxes from one state: as the same expressions they are evaluated
// once per state, with one division each for 1/rho and rho/p.
struct PrimState {
  double srho, v1, v2, v3, v2s2, p;
  __device__ __forceinline__ PrimState(const double *U, double kappa)
  {
    srho = 1.0 / U[0];
    v1 = U[1] * srho; v2 = U[2] * srho; v3 = U[3] * srho;
    v2s2 = 0.5 * (v1 * v1 + v2 * v2 + v3 * v3);
    p = (kappa - 1.0) * (U[4] - U[0] * v2s2);
  }
};

// ConsToEntropy (navierstokes/equation_vars.f90:362-391); s = -ln(rho_sp*rho^(kappa-1)) is
// evaluated as -(ln rho_sp + (kappa-1) ln rho).
__device__ __forceinline__ void cons_to_entropy(const double *U, double kappa, double skappaM1, double *w)
{
  const PrimState q(U, kappa);
  const double rho_sp = U[0] / q.p;
  const double s = -(log(rho_sp) + (kappa - 1.0) * log(U[0]));
  w[0] = (kappa - s) * skappaM1 - rho_sp * q.v2s2;
  w[1] = rho_sp * q.v1;
  w[2] = rho_sp * q.v2;
  w[3] = rho_sp * q.v3;
  w[4] = -rho_sp;
}

// ConvertToGradPrimVec for entropy-variable lifting (equation_vars.f90:571-647).
__device__ __forceinline__ void grad_entropy_to_prim(const double *U, double kappa, double skappaM1, double *g)
{
  const PrimState q(U, kappa);
  const double rho_sp = U[0] / q.p, p_srho = q.p * q.srho;
  const double g1 = g[0], g5 = g[4];
  const double gu = p_srho * (g[1] + q.v1 * g5);
  const double gv = p_srho * (g[2] + q.v2 * g5);
  const double gw = p_srho * (g[3] + q.v3 * g5);
  g[0] = U[0] * g1 - g5 * (U[0] * q.v2s2 - q.p * skappaM1) + rho_sp * (U[1] * gu + U[2] * gv + U[3] * gw);
  g[1] = gu; g[2] = gv; g[3] = gw;
  g[4] = p_srho * (g[0] + q.p * g5);
}

// EvalDiffFlux3D with constant viscosity (flux.f90:407-517): Cartesian viscous fluxes
// f, g, h; component 0 (mass) is identically zero and omitted: out[d*4 + (v-1)].
__device__ __forceinline__ void diff_flux(const double *U, const double *gx, const double *gy,
                                          const double *gz, double kappa, double skm1, double mu0,
                                          double KappasPr, double *out)
{
  const double s23 = 2.0 / 3.0;
  const PrimState q(U, kappa);
  const double srho = q.srho, v1 = q.v1, v2 = q.v2, v3 = q.v3, p = q.p;
  double muS = mu0, lambda = muS * KappasPr;
  double divv = gx[1] + gy[2] + gz[3];
  double cTx = skm1 * srho * (gx[4] - srho * p * gx[0]);
  double cTy = skm1 * srho * (gy[4] - srho * p * gy[0]);
  double cTz = skm1 * srho * (gz[4] - srho * p * gz[0]);
  double f1 = -muS * (2 * gx[1] - s23 * divv);
  double f2 = -muS * (gx[2] + gy[1]);
  double f3 = -muS * (gx[3] + gz[1]);
  double f4 = v1 * f1 + v2 * f2 + v3 * f3 - lambda * cTx;
  double g1 = f2;
  double g2 = -muS * (2 * gy[2] - s23 * divv);
  double g3 = -muS * (gy[3] + gz[2]);
  double g4 = v1 * g1 + v2 * g2 + v3 * g3 - lambda * cTy;
  double h1 = f3, h2 = g3;
  double h3 = -muS * (2 * gz[3] - s23 * divv);
  double h4 = v1 * h1 + v2 * h2 + v3 * h3 - lambda * cTz;
  out[0] = f1; out[1] = f2; out[2] = f3; out[3] = f4;
  out[4] = g1; out[5] = g2; out[6] = g3; out[7] = g4;
  out[8] = h1; out[9] = h2; out[10] = h3; out[11] = h4;
}

}  // namespace fx

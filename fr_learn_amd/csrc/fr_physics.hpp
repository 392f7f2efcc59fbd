// fr_physics.hpp -- pointwise physics shared by the residual kernels:
// Euler / advection fluxes, common (Riemann) fluxes and boundary states.
// Every routine restates one reference function; arithmetic is written in the
// same order so FP64 results agree with the reference to rounding.
#pragma once

#include <type_traits>

#include <hip/hip_runtime.h>

namespace frdev {

struct Phys {
  double gamma, lambda, diffD;
  double advect[3];
  double rhoBound, uBound, vBound, wBound, pBound;
  double TWall, RGas, uWall, vWall, wWall;
  double penFact, tau, mu_inf, prandtl, rt_inf, c_sth;
  int equation, riemannType, fixVis, viscFix;
  // Energy offset of the FP32 states (inviscid Euler): they hold E - eOff,
  // where eOff = pOff / (gamma - 1) for a reference pressure pOff near the
  // flow's mean.  The FP32 flux routines then work with p - pOff, whose
  // rounding is relative to the pressure variation instead of the (low-Mach)
  // background; hOff = gamma * eOff restores the total enthalpy of the energy
  // flux.  The constant pOff dropped from the momentum flux is a
  // divergence-free term of the discretisation (free-stream preservation).
  // Zero in FP64 contexts, whose routines ignore them.
  double eOff, pOff, hOff;
};

// FP32 states carry the energy offset (Phys::eOff); FP64 and dual-number
// states do not.
template <typename T>
constexpr bool hasEnergyOffset() {
  return sizeof(T) == 4;
}

// 1 / x for the flux routines: the hardware reciprocal estimate refined by
// Newton-Raphson steps, e = 1 - x r, r <- r + r e (each step squares the
// relative error), within an ulp of the correctly rounded value for
// densities of ordinary magnitude.  FP64: two steps from the 2^-22-accurate
// estimate, half the instructions of a full IEEE division; FP32: one step
// from the 1-ulp estimate, three instructions instead of ten.
template <typename T>
__device__ __forceinline__ T recip(T x) {
  if constexpr (sizeof(T) == 8) {
    double r = __builtin_amdgcn_rcp(x);
    double e = fma(-x, r, 1.0);
    r = fma(r, e, r);
    e = fma(-x, r, 1.0);
    return fma(r, e, r);
  } else if constexpr (std::is_same<T, float>::value) {
    const float r = __builtin_amdgcn_rcpf(x);
    return fmaf(fmaf(-x, r, 1.0f), r, r);
  } else {
    return (T)1 / x;  // dual numbers (the adjoint's derivatives)
  }
}

// sqrt(x) of a non-negative x of ordinary magnitude (sound speeds, face
// areas); rootAndInv also gives 1 / sqrt(x).  FP64: Goldschmidt's coupled
// iteration for g -> sqrt(x), h -> 1 / (2 sqrt(x)) from the hardware
// reciprocal square root estimate y (relative error below 2^-22): g = x y,
// h = y / 2, then per step r = 1/2 - g h, g <- g + g r, h <- h + h r, which
// squares the relative error; a Newton correction g <- g + (x - g^2) h
// after the step leaves g within an ulp of the correctly rounded root.  An x
// below the smallest normal double is taken as that value (root 1.5e-154
// instead of 0: the estimate of 0 is infinite).  FP32: the hardware root
// and reciprocal (1 ulp each; the IEEE-rounded library root takes about 16
// instructions for its scaling and corrections).
__device__ __forceinline__ void rootSteps(double x, double &g, double &h, int steps) {
  x = fmax(x, 2.2250738585072014e-308);
  const double y = __builtin_amdgcn_rsq(x);
  g = x * y;
  h = 0.5 * y;
  for (int i = 0; i < steps; i++) {
    const double r = fma(-g, h, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
  }
  g = fma(fma(-g, g, x), h, g);
}
template <typename T>
__device__ __forceinline__ T rootPos(T x) {
  if constexpr (sizeof(T) == 8) {
    double g, h;
    rootSteps(x, g, h, 1);
    return g;
  } else if constexpr (std::is_same<T, float>::value) {
    return __builtin_amdgcn_sqrtf(x);
  } else {
    return sqrt(x);  // dual numbers
  }
}
// sqrt(x) as rootPos, of an x that may be negative or NaN, where it is NaN as
// the library's root is (the Roe averages of an unphysical state): the smallest
// normal double is added instead of taken as the least, so that only the root
// of 0 differs (1.5e-154); an infinite x gives NaN, as does the flux of such a
// state with any root (recip(inf) is NaN).  FP32 and dual numbers take the
// library's root: the hardware's is up to an ulp off, which made the Roe flux's
// rounding error up to 4 % larger at strong jumps for 3 % of a triangle stage.
template <typename T>
__device__ __forceinline__ T rootOf(T x) {
  if constexpr (sizeof(T) == 8) {
    x = x + 2.2250738585072014e-308;
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = fma(-g, h, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    return fma(fma(-g, g, x), h, g);
  } else {
    return sqrt(x);
  }
}
template <typename T>
__device__ __forceinline__ void rootAndInv(T x, T &root, T &inv) {
  if constexpr (sizeof(T) == 8) {
    double g, h;
    rootSteps(x, g, h, 2);
    root = g;
    inv = h + h;
  } else if constexpr (std::is_same<T, float>::value) {
    root = __builtin_amdgcn_sqrtf(x);
    inv = __builtin_amdgcn_rcpf(root);
  } else {
    root = sqrt(x);  // dual numbers
    inv = (T)1 / root;
  }
}

// Euler flux F[d][k] (inviscidFlux, reference src/flux.cpp:37-88) or linear
// advection flux.
template <int D, int NF, typename T>
__device__ __forceinline__ void inviscidFlux(const Phys &ph, const T *U, T F[D][NF]) {
  if constexpr (NF == 1) {
#pragma unroll
    for (int d = 0; d < D; d++) F[d][0] = (T)ph.advect[d] * U[0];
  } else if constexpr (D == 2) {
    // velocities use one reciprocal of rho instead of a division each (the
    // reference divides; the difference is at most an ulp per velocity)
    const T g = (T)ph.gamma;
    const T rho = U[0], ri = recip(rho);
    T u = U[1] * ri, v = U[2] * ri, E = U[3];
    T p = (g - (T)1.0) * (E - (T)0.5 * rho * (u * u + v * v));
    // total enthalpy rho*H = E + p (FP32: offset-free E and p plus hOff)
    T Ep = E + p;
    if constexpr (hasEnergyOffset<T>()) Ep = Ep + (T)ph.hOff;
    F[0][0] = rho * u;         F[1][0] = rho * v;
    F[0][1] = rho * u * u + p; F[1][1] = rho * u * v;
    F[0][2] = rho * v * u;     F[1][2] = rho * v * v + p;
    F[0][3] = Ep * u;          F[1][3] = Ep * v;
  } else {
    const T g = (T)ph.gamma;
    const T rho = U[0], ri = recip(rho);
    T u = U[1] * ri, v = U[2] * ri, w = U[3] * ri, E = U[4];
    T p = (g - (T)1.0) * (E - (T)0.5 * rho * (u * u + v * v + w * w));
    T Ep = E + p;
    if constexpr (hasEnergyOffset<T>()) Ep = Ep + (T)ph.hOff;
    F[0][0] = rho * u;         F[1][0] = rho * v;         F[2][0] = rho * w;
    F[0][1] = rho * u * u + p; F[1][1] = rho * u * v;     F[2][1] = rho * u * w;
    F[0][2] = rho * v * u;     F[1][2] = rho * v * v + p; F[2][2] = rho * v * w;
    F[0][3] = rho * w * u;     F[1][3] = rho * w * v;     F[2][3] = rho * w * w + p;
    F[0][4] = Ep * u;          F[1][4] = Ep * v;          F[2][4] = Ep * w;
  }
}

// Normal Euler flux F(U).n of one side plus its normal velocity and squared
// sound speed: the sum over d of n[d] F[d][i] that face::rusanovFlux forms
// from inviscidFlux (flux.cpp:37-88), factored through the normal velocity
// vn = v.n -- mass rho vn, momentum rho vn v_c + p n_c, energy (E + p) vn --
// without holding the D x NF flux table (the same terms, summed in another
// order: an ulp-level difference).  One reciprocal of rho (recip) replaces
// the reference's divisions (also an ulp-level difference).
template <int D, typename T>
__device__ __forceinline__ void normalFlux(const Phys &ph, const T g, const T *U, const T *n, T *Fn, T &vn, T &csq) {
  constexpr int NF = D + 2;
  const T rho = U[0], E = U[D + 1], ri = recip(rho);
  T v[D];
#pragma unroll
  for (int d = 0; d < D; d++) v[d] = U[d + 1] * ri;
  T q = v[0] * v[0] + v[1] * v[1];
  if (D == 3) q = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
  const T p = (g - (T)1.0) * (E - (T)0.5 * rho * q);
  T Ep = E + p, pAbs = p;  // FP32: offset-free E and p (Phys::eOff)
  if constexpr (hasEnergyOffset<T>()) {
    Ep = Ep + (T)ph.hOff;
    pAbs = p + (T)ph.pOff;
  }
  vn = n[0] * v[0];
#pragma unroll
  for (int d = 1; d < D; d++) vn += n[d] * v[d];
  const T mn = rho * vn;
  Fn[0] = mn;
#pragma unroll
  for (int c = 0; c < D; c++) Fn[1 + c] = mn * v[c] + p * n[c];
  Fn[D + 1] = Ep * vn;
  csq = fmax(g * pAbs * ri, (T)0.0);
}

// Rusanov / local Lax-Friedrichs flux for Euler (face::rusanovFlux,
// src/face.cpp:289-356, static mesh).  eigOut (may be null) receives
// max(eigL, eigR), the wave speed the reference stores for the CFL time step
// (face.cpp:354).  swap = true takes UA as the right state and UB as the
// left one: the flux is symmetric in the two sides but for the sign of the
// dissipation term eig (UR - UL), and sums, fmax and a negated product are
// exact under the exchange, so the result is bit for bit the flux of the
// exchanged arguments -- a lane picks its side by a sign, not by selecting
// every field.
template <int D, typename T>
__device__ __forceinline__ void rusanovN(const Phys &ph, const T *UA, const T *UB, const T *n, T *Fn,
                                         T *eigOut = nullptr, bool swap = false) {
  constexpr int NF = D + 2;
  const T g = (T)ph.gamma;
  T FnA[NF], FnB[NF], vnA, vnB, csqA, csqB;
  normalFlux<D, T>(ph, g, UA, n, FnA, vnA, csqA);
  normalFlux<D, T>(ph, g, UB, n, FnB, vnB, csqB);
  const T eig = fmax(fabs(vnA) + rootPos(csqA), fabs(vnB) + rootPos(csqB));
  if (eigOut) *eigOut = eig;
  const T eigS = swap ? -eig : eig;
#pragma unroll
  for (int i = 0; i < NF; i++) Fn[i] = (T)0.5 * (FnA[i] + FnB[i] - eigS * (UB[i] - UA[i]));
}

// Roe flux with Harten-type entropy fix, 2D (face::roeFlux,
// src/face.cpp:358-484).  The reference's divisions by the densities, by eps
// and by the Roe sound speed are multiplications by reciprocals (recip), and
// its FP64 roots rootOf, ulp-level differences (the library's root and its
// scaling are about twenty instructions; quads P4 128^2 20.8 -> 20.2 us a stage).
template <typename T>
__device__ __forceinline__ void roe2d(const Phys &ph, const T *UL, const T *UR, const T *n, T *Fn) {
  const T g = (T)ph.gamma;
  const T riL = recip(UL[0]), riR = recip(UR[0]);
  T vL[2], vR[2], um[2], du[4];
  for (int i = 0; i < 2; i++) {
    vL[i] = UL[i + 1] * riL;
    vR[i] = UR[i + 1] * riR;
  }
  T pL = (g - (T)1.0) * (UL[3] - ((T)0.5 * UL[0] * (vL[0] * vL[0] + vL[1] * vL[1])));
  T pR = (g - (T)1.0) * (UR[3] - ((T)0.5 * UR[0] * (vR[0] * vR[0] + vR[1] * vR[1])));
  // FP32 (Phys::eOff): pL, pR are offset-free; the enthalpies and sound
  // speeds take the absolute values
  T EpL = UL[3] + pL, EpR = UR[3] + pR, pAL = pL, pAR = pR;
  if constexpr (hasEnergyOffset<T>()) {
    EpL = EpL + (T)ph.hOff;
    EpR = EpR + (T)ph.hOff;
    pAL = pL + (T)ph.pOff;
    pAR = pR + (T)ph.pOff;
  }
  T hL = EpL * riL, hR = EpR * riR;
  T sq_rho = rootOf(UR[0] * riL);
  T rrho = recip(sq_rho + (T)1.);
  T usq = 0, unm = 0;
  for (int i = 0; i < 2; i++) {
    um[i] = rrho * (vL[i] + sq_rho * vR[i]);
    usq += (T)0.5 * um[i] * um[i];
    unm += um[i] * n[i];
  }
  T hm = rrho * (hL + sq_rho * hR);
  T am_sq = (g - (T)1.) * (hm - usq);
  T am = rootOf(am_sq);
  T rhoUnL = 0, rhoUnR = 0;
  for (int i = 0; i < 2; i++) {
    rhoUnL += UL[i + 1] * n[i];
    rhoUnR += UR[i + 1] * n[i];
  }
  Fn[0] = rhoUnL + rhoUnR;
  Fn[1] = rhoUnL * vL[0] + rhoUnR * vR[0] + (pL + pR) * n[0];
  Fn[2] = rhoUnL * vL[1] + rhoUnR * vR[1] + (pL + pR) * n[1];
  Fn[3] = rhoUnL * hL + rhoUnR * hR;
  for (int i = 0; i < 4; i++) du[i] = UR[i] - UL[i];
  T lambda0 = fabs(unm), lambdaP = fabs(unm + am), lambdaM = fabs(unm - am);
  T eps = (T)0.5 * (fabs(rhoUnL * riL - rhoUnR * riR) + fabs(rootOf(g * pAL * riL) - rootOf(g * pAR * riR)));
  const T reps = recip(eps);
  if (lambda0 < (T)2. * eps) lambda0 = (T)0.25 * lambda0 * lambda0 * reps + eps;
  if (lambdaP < (T)2. * eps) lambdaP = (T)0.25 * lambdaP * lambdaP * reps + eps;
  if (lambdaM < (T)2. * eps) lambdaM = (T)0.25 * lambdaM * lambdaM * reps + eps;
  T a2 = (T)0.5 * (lambdaP + lambdaM) - lambda0;
  T a3 = (T)0.5 * (lambdaP - lambdaM) * recip(am);
  T a1 = a2 * (g - (T)1.) * recip(am_sq);
  T a4 = a3 * (g - (T)1.);
  T a5 = usq * du[0] - um[0] * du[1] - um[1] * du[2] + du[3];
  T a6 = unm * du[0] - n[0] * du[1] - n[1] * du[2];
  T aL1 = a1 * a5 - a3 * a6, bL1 = a4 * a5 - a2 * a6;
  Fn[0] -= lambda0 * du[0] + aL1;
  Fn[1] -= lambda0 * du[1] + aL1 * um[0] + bL1 * n[0];
  Fn[2] -= lambda0 * du[2] + aL1 * um[1] + bL1 * n[1];
  Fn[3] -= lambda0 * du[3] + aL1 * hm + bL1 * unm;
  for (int i = 0; i < 4; i++) Fn[i] *= (T)0.5;
}

// Lax-Friedrichs flux for linear advection (face::laxFriedrichsFlux,
// src/face.cpp:486-514).
template <int D, typename T>
__device__ __forceinline__ void laxFriedrichs(const Phys &ph, const T *UL, const T *UR, const T *n, T *Fn) {
  T uAvg = (T)0.5 * (UL[0] + UR[0]);
  T uDiff = UL[0] - UR[0];
  T vNorm = (T)ph.advect[0] * n[0] + (T)ph.advect[1] * n[1];
  if constexpr (D == 3) vNorm += (T)ph.advect[2] * n[2];
  Fn[0] = vNorm * uAvg + (T)0.5 * (T)ph.lambda * fabs(vNorm) * uDiff;
}

// Ghost (right) state of a boundary flux point (boundFace::applyBCs,
// src/boundFace.cpp:33-277; static grid, so the grid velocity is zero).
template <int D, int NF, typename T>
__device__ __forceinline__ void boundaryState(const Phys &ph, int bc, const T *UL, const T *n, T *UR) {
  if constexpr (NF == 1) {
    UR[0] = (T)0;  // the reference leaves the advection ghost state at zero
  } else {
    const T g = (T)ph.gamma, gmo = g - (T)1.;
    // FP32 states hold E - eOff (Phys::eOff): pL and the ghost energies below
    // are then offset-free (p - pOff, E - eOff), the absolute pressure pLa is
    // used where the formulas need it.  FP64: pLa = pL, pOff = 0.
    constexpr bool OFF = hasEnergyOffset<T>();
    T rhoR = 0, pR = 0, ER = 0;
    T vL[3] = {0, 0, 0}, vR[3] = {0, 0, 0};
    const T vB[3] = {(T)ph.uBound, (T)ph.vBound, (T)ph.wBound};
    T rhoL = UL[0], eL = UL[D + 1];
    for (int i = 0; i < D; i++) vL[i] = UL[i + 1] / UL[0];
    T vSq = 0;
    for (int i = 0; i < D; i++) vSq += vL[i] * vL[i];
    T pL = (g - (T)1.0) * (eL - (T)0.5 * rhoL * vSq);
    const T pLa = OFF ? pL + (T)ph.pOff : pL;
    // the ghost pressure pR is offset-free like pL
    const T pBnd = OFF ? (T)(ph.pBound - ph.pOff) : (T)ph.pBound;
    auto energy = [&](void) {
      T s = 0;
      for (int i = 0; i < D; i++) s += vR[i] * vR[i];
      return (pR / (g - (T)1.0)) + (T)0.5 * rhoR * s;
    };
    switch (bc) {
      case 4:  // SUB_IN
        rhoR = (T)ph.rhoBound;
        for (int i = 0; i < D; i++) vR[i] = vB[i];
        pR = pL;
        ER = energy();
        break;
      case 5:  // SUB_OUT
        rhoR = rhoL;
        for (int i = 0; i < D; i++) vR[i] = vL[i];
        pR = pBnd;
        ER = energy();
        break;
      case 2:  // SUP_IN
        rhoR = (T)ph.rhoBound;
        vR[0] = vB[0]; vR[1] = vB[1]; vR[2] = vB[2];
        pR = pBnd;
        ER = energy();
        break;
      case 3:  // SUP_OUT
        rhoR = rhoL;
        for (int i = 0; i < D; i++) vR[i] = vL[i];
        ER = eL;
        break;
      case 8:   // SLIP_WALL
      case 12: {  // SYMMETRY
        rhoR = rhoL;
        T vnL = 0;
        for (int i = 0; i < D; i++) vnL += vL[i] * n[i];
        for (int i = 0; i < D; i++) vR[i] = vL[i] - (T)2.0 * vnL * n[i];
        ER = eL;
        break;
      }
      case 13:  // ISOTHERMAL_NOSLIP_MOVING
        pR = pL;
        rhoR = pLa / ((T)ph.RGas * (T)ph.TWall);
        vR[0] = (T)ph.uWall;
        vR[1] = (T)ph.vWall;
        if (D == 3) vR[2] = (T)ph.wWall;
        ER = energy();
        break;
      case 9:  // ISOTHERMAL_NOSLIP
        pR = pL;
        rhoR = pLa / ((T)ph.RGas * (T)ph.TWall);
        ER = energy();
        break;
      case 10:  // ADIABATIC_NOSLIP
        rhoR = rhoL;
        pR = pL;
        ER = energy();
        break;
      case 1: {  // CHAR_INOUT (Riemann invariants)
        T vnL = 0, vnB = 0;
        for (int i = 0; i < D; i++) vnL += vL[i] * n[i];
        for (int i = 0; i < D; i++) vnB += vB[i] * n[i];
        T cL = sqrt(g * pLa / rhoL), cB = sqrt(g * (T)ph.pBound / (T)ph.rhoBound);
        T R_L = (fabs(vnB) >= cB && vnL >= 0) ? vnB + (T)2. / gmo * cB : vnL + (T)2. / gmo * cL;
        T R_B = (fabs(vnB) >= cB && vnL < 0) ? vnL - (T)2. / gmo * cL : vnB - (T)2. / gmo * cB;
        T rhoFac = (T).25 * (g - (T)1.) * (R_L - R_B);
        T rhoBG = rhoFac * rhoFac / g;
        if (vnL < 0) rhoBG *= pow((T)ph.rhoBound, g) / (T)ph.pBound;
        else rhoBG *= pow(rhoL, g) / pLa;
        rhoR = pow(rhoBG, (T)1. / gmo);
        pR = rhoFac * rhoFac * rhoR / g;
        if constexpr (OFF) pR = pR - (T)ph.pOff;
        T VB = (T)0.5 * (R_L + R_B);
        for (int i = 0; i < D; i++) vR[i] = (vnL < 0) ? vB[i] + (VB - vnB) * n[i] : vL[i] + (VB - vnL) * n[i];
        T vM2 = 0;
        for (int i = 0; i < D; i++) vM2 += vR[i] * vR[i];
        ER = pR / gmo + (T).5 * rhoR * vM2;
        break;
      }
      default:
        break;
    }
    UR[0] = rhoR;
    for (int i = 0; i < D; i++) UR[i + 1] = rhoR * vR[i];
    UR[D + 1] = ER;
  }
}

// ---------------------------------------------------------------------------
// viscous terms
// ---------------------------------------------------------------------------
// Navier-Stokes viscous flux Fv[d][k] from U and the physical gradient
// g[d][k] (viscousFlux, reference src/flux.cpp:90-226).  viscFix = 0 keeps the
// reference's index defects: tauxz = mu(du/dz + dv/dx), tauyz = mu(du/dz +
// dv/dy) (flux.cpp:197-198) and Fv[0][3] = -tauzz (flux.cpp:216); viscFix = 1
// uses the physical tauxz = mu(du/dz + dw/dx), tauyz = mu(dv/dz + dw/dy),
// Fv[0][3] = -tauxz.  Advection-diffusion: Fv = -diffD grad u
// (viscousFluxAD, flux.cpp:361-366).
template <int D, int NF, typename T>
__device__ __forceinline__ void viscousFlux(const Phys &ph, const T *U, const T g[D][NF], T Fv[D][NF]) {
  if constexpr (NF == 1) {
#pragma unroll
    for (int d = 0; d < D; d++) Fv[d][0] = -(T)ph.diffD * g[d][0];
  } else {
    // Written for few operations: one reciprocal of rho for the reference's
    // divisions, the velocity gradients (grad m - v grad rho) / rho, and the
    // energy gradient from that of the total energy,
    //   grad e = (grad E - (E / rho) grad rho) / rho - sum_c v_c grad v_c,
    // which is the reference's grad E - grad(rho |v|^2 / 2) - e grad rho
    // regrouped; the ratio gamma / Pr and the third of the divergence are
    // constants.  Ulp-level differences.  FP32 divides by rho and by 3: with
    // the products the rounding error of its momentum flux was 7-15 % larger
    // (random states of order one with density gradients), with the divisions
    // it is below that of the reference's grouping.
    constexpr bool F64 = sizeof(T) == 8;
    const T ri = F64 ? recip(U[0]) : (T)0;
    auto over = [&](const T &x) -> T {
      if constexpr (F64) return x * ri;
      else return x / U[0];
    };
    T v[D];
#pragma unroll
    for (int c = 0; c < D; c++) v[c] = over(U[c + 1]);
    const T H = over(U[D + 1]);
    T mu = (T)ph.mu_inf;
    if (!ph.fixVis) {  // Sutherland's law
      T q = v[0] * v[0];
#pragma unroll
      for (int c = 1; c < D; c++) q += v[c] * v[c];
      const T rt = ((T)ph.gamma - (T)1.0) * (H - (T)0.5 * q) / (T)ph.rt_inf;
      mu *= pow(rt, (T)1.5) * ((T)1. + (T)ph.c_sth) / (rt + (T)ph.c_sth);
    }
    const T mr = over(mu);  // mu / rho: the stresses need mu grad v
    // G[d][c] = mu dv_c/dx_d and h[d] = mu de/dx_d
    T G[D][D], h[D];
#pragma unroll
    for (int d = 0; d < D; d++) {
#pragma unroll
      for (int c = 0; c < D; c++) G[d][c] = mr * (g[d][c + 1] - v[c] * g[d][0]);
      h[d] = mr * (g[d][D + 1] - H * g[d][0]);
#pragma unroll
      for (int c = 0; c < D; c++) h[d] -= v[c] * G[d][c];
    }
    T diag = G[0][0] + G[1][1];
    if constexpr (D == 3) diag += G[2][2];
    diag = F64 ? diag * (T)(1.0 / 3.0) : diag / (T)3.0;
    const T kq = (T)(ph.gamma / ph.prandtl);
    T tau[D][D];  // tau[d][c], symmetric
#pragma unroll
    for (int d = 0; d < D; d++) tau[d][d] = (T)2.0 * (G[d][d] - diag);
    tau[0][1] = tau[1][0] = G[1][0] + G[0][1];
    if constexpr (D == 3) {
      tau[0][2] = tau[2][0] = ph.viscFix ? G[2][0] + G[0][2] : G[2][0] + G[0][1];
      tau[1][2] = tau[2][1] = ph.viscFix ? G[2][1] + G[1][2] : G[2][0] + G[1][1];
    }
#pragma unroll
    for (int d = 0; d < D; d++) {
      T q = kq * h[d];
#pragma unroll
      for (int c = 0; c < D; c++) q += v[c] * tau[d][c];
      Fv[d][0] = (T)0.0;
#pragma unroll
      for (int c = 0; c < D; c++) Fv[d][c + 1] = -tau[d][c];
      Fv[d][D + 1] = -q;
    }
    if constexpr (D == 3)
      if (!ph.viscFix) Fv[0][3] = -tau[2][2];
  }
}

// The physical gradient JGinv^T gr / detJ of a reference-space gradient gr at
// one point, J = JGinv(dimRef, dimPhys).  FP64: one reciprocal (recip) folded
// into the metrics; FP32 divides, after the sum.
template <int D, int NF, typename T>
__device__ __forceinline__ void physicalGradient(const T gr[D][NF], const T *J, T detJ, T g[D][NF]) {
  constexpr bool F64 = sizeof(T) == 8;
  const T invDet = F64 ? recip(detJ) : (T)1 / detJ;
#pragma unroll
  for (int d1 = 0; d1 < D; d1++) {
    T Jd[D];
#pragma unroll
    for (int d = 0; d < D; d++) Jd[d] = F64 ? J[d * D + d1] * invDet : J[d * D + d1];
#pragma unroll
    for (int k = 0; k < NF; k++) {
      T acc = gr[0][k] * Jd[0] + gr[1][k] * Jd[1];
      if constexpr (D == 3) acc = acc + gr[2][k] * Jd[2];
      g[d1][k] = F64 ? acc : invDet * acc;
    }
  }
}

// Adiabatic no-slip wall gradient state (boundFace::applyViscousBCs,
// boundFace.cpp:279-320): gR = gL, then the energy gradient is rebuilt with
// zero temperature gradient.  Other boundaries keep gR = gL.
template <int D, int NF, typename T>
__device__ __forceinline__ void boundaryGradient(const Phys &ph, int bc, const T *UL, const T *UR, const T gL[D][NF],
                                                 T gR[D][NF]) {
#pragma unroll
  for (int d = 0; d < D; d++)
#pragma unroll
    for (int k = 0; k < NF; k++) gR[d][k] = gL[d][k];
  if constexpr (NF > 1) {
    if (bc != 10) return;
    T rhovSq = 0;
    for (int d = 0; d < D; d++) rhovSq += UL[d + 1] * UL[d + 1];
    const T pL = ((T)ph.gamma - (T)1.) * (UL[D + 1] - (T)0.5 * rhovSq / UL[0]);
    const T e = pL / (((T)ph.gamma - (T)1.) * UR[0]);
    T gv[D][D];
    for (int d1 = 0; d1 < D; d1++)
      for (int d2 = 0; d2 < D; d2++) gv[d1][d2] = (gR[d1][d2 + 1] - gR[d1][0] * UR[d2 + 1] / UR[0]) / UR[0];
    T vSq = 0;
    for (int d = 0; d < D; d++) vSq += UR[d + 1] * UR[d + 1] / (UR[0] * UR[0]);
    for (int d1 = 0; d1 < D; d1++) {
      gR[d1][D + 1] = (e + (T)0.5 * vSq) * gR[d1][0];
      for (int d2 = 0; d2 < D; d2++) gR[d1][D + 1] += UR[d2 + 1] * gv[d2][d1];
    }
  }
}

// LDG penalty direction switch (face.cpp:587-597 / 206-215): -penFact when
// n.(1, 1, sqrt 2) < 0 (n.(1,1) in 2D).
template <int D, typename T>
__device__ __forceinline__ T ldgPenalty(const Phys &ph, const T *n) {
  T pen = (T)ph.penFact;
  if (D == 2) {
    if (n[0] + n[1] < 0) pen = -(T)ph.penFact;
  } else if (n[0] + n[1] + (T)1.4142135623730951 * n[2] < 0) {
    pen = -(T)ph.penFact;
  }
  return pen;
}

// Fields with a viscous flux: all but the mass of Navier-Stokes (fields
// NF - viscFields .. NF - 1).
template <int NF>
constexpr int viscFields() {
  return NF == 1 ? 1 : NF - 1;
}

// The weights w of one side's viscous flux F in the LDG common normal flux
// sum_d Fc[d] n[d] (face::calcViscousFlux, face.cpp:177-287), the same for
// every field: with Fc[d] = (FL + FR)[d] / 2 + pen n[d] n.(FL - FR), the left
// side enters with w = n / 2 + pen |n|^2 n and the right one with
// n / 2 - pen |n|^2 n; face.cpp:245 takes F_L,y for F_L,z in n.(FL - FR)
// (viscFix = 0).  Boundaries take one side's flux alone (w = n), and
// advection-diffusion the central flux of -diffD grad u (face.cpp:270-279;
// its boundaries a zero outside gradient).  n is the left element's normal.
template <int D, int NF, typename T>
__device__ __forceinline__ void ldgWeights(const Phys &ph, bool bnd, bool right, const T *n, T *w) {
  if constexpr (NF == 1) {
#pragma unroll
    for (int d = 0; d < D; d++) w[d] = (T)0.5 * n[d];
  } else {
    T nn = n[0] * n[0];
#pragma unroll
    for (int d = 1; d < D; d++) nn += n[d] * n[d];
    const T pn = ldgPenalty<D, T>(ph, n) * nn;
#pragma unroll
    for (int d = 0; d < D; d++) w[d] = bnd ? n[d] : (T)0.5 * n[d] + (right ? -pn * n[d] : pn * n[d]);
    if constexpr (D == 3)
      if (!bnd && !right && !ph.viscFix) {
        w[1] += pn * n[2];
        w[2] -= pn * n[2];
      }
  }
}

// One side's share of the viscous common normal flux, w . F_v(U, g), for the
// fields that have one (viscFields).
template <int D, int NF, typename T>
__device__ __forceinline__ void viscousShare(const Phys &ph, bool bnd, bool right, const T *U, const T g[D][NF],
                                             const T *n, T *C) {
  constexpr int NV = viscFields<NF>();
  T F[D][NF], w[D];
  viscousFlux<D, NF, T>(ph, U, g, F);
  ldgWeights<D, NF, T>(ph, bnd, right, n, w);
#pragma unroll
  for (int k = 0; k < NV; k++) {
    T acc = w[0] * F[0][NF - NV + k];
#pragma unroll
    for (int d = 1; d < D; d++) acc += w[d] * F[d][NF - NV + k];
    C[k] = acc;
  }
}

}  // namespace frdev

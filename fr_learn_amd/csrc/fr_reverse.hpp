// fr_reverse.hpp -- reverse-mode derivatives of the pointwise physics
// (fr_physics.hpp), FP64: given the cotangent of a flux, the cotangents of the
// states and gradients it was formed from.
//
// One reverse pass costs a small multiple of the flux itself, where forward
// (dual-number) passes cost one flux evaluation per direction -- NF states and
// D NF gradient components for a viscous face point -- and hold every value
// of a pass twice or more.  The boundaries' ghost states and the Roe flux keep
// the dual numbers (fr_dual.hpp): many cases, few points.  Each routine
// differentiates the branch the forward routine takes.
#pragma once

#include "fr_dual.hpp"
#include "fr_physics.hpp"

namespace frdev {

// Cotangents of the primitives (rho, v, p), of the momentum and of the energy
// pulled back to the conserved state: p = (gamma - 1)(E - rho v.v / 2),
// v = m / rho.  lU is overwritten.
template <int D>
__device__ __forceinline__ void primitiveVjp(double gmo, double rho, double ri, const double *v, double lrho,
                                             const double *lv, double lp, const double *lm, double lE, double *lU) {
  double q = v[0] * v[0];
#pragma unroll
  for (int c = 1; c < D; c++) q += v[c] * v[c];
  const double s = gmo * lp;
  lU[D + 1] = lE + s;
  lrho -= 0.5 * q * s;
  double vs = 0.0;
#pragma unroll
  for (int c = 0; c < D; c++) {
    const double l = lv[c] - rho * v[c] * s;
    lU[c + 1] = lm[c] + l * ri;
    vs += l * v[c];
  }
  lU[0] = lrho - vs * ri;
}

// Point flux (inviscidFlux): lU = sum lF[d][k] dF[d][k] / dU.
template <int D, int NF>
__device__ __forceinline__ void inviscidFluxVjp(const Phys &ph, const double *U, const double (&lF)[D][NF],
                                                double *lU) {
  if constexpr (NF == 1) {
    lU[0] = 0.0;
#pragma unroll
    for (int d = 0; d < D; d++) lU[0] += ph.advect[d] * lF[d][0];
  } else {
    const double gmo = ph.gamma - 1.0, rho = U[0], ri = recip(rho), E = U[D + 1];
    double v[D], q = 0.0;
#pragma unroll
    for (int c = 0; c < D; c++) {
      v[c] = U[c + 1] * ri;
      q += v[c] * v[c];
    }
    const double p = gmo * (E - 0.5 * rho * q);
    double lp = 0.0, lE = 0.0, lm[D], lv[D];
#pragma unroll
    for (int d = 0; d < D; d++) {
      lp += lF[d][d + 1] + lF[d][D + 1] * v[d];
      lE += lF[d][D + 1] * v[d];
      lm[d] = lF[d][0];
      lv[d] = lF[d][D + 1] * (E + p);
    }
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
      for (int c = 0; c < D; c++) {
        lm[d] += lF[d][c + 1] * v[c];
        lv[c] += lF[d][c + 1] * U[d + 1];
      }
    primitiveVjp<D>(gmo, rho, ri, v, 0.0, lv, lp, lm, lE, lU);
  }
}

// One side of the Rusanov flux: velocity, pressure, normal velocity and sound
// speed of its state.
template <int D>
struct RusanovSide {
  double ri, v[D], p, vn, c, eig;
  __device__ __forceinline__ RusanovSide(const Phys &ph, const double *U, const double *n) {
    ri = recip(U[0]);
    double q = 0.0;
    vn = 0.0;
#pragma unroll
    for (int d = 0; d < D; d++) {
      v[d] = U[d + 1] * ri;
      q += v[d] * v[d];
      vn += v[d] * n[d];
    }
    p = (ph.gamma - 1.0) * (U[D + 1] - 0.5 * U[0] * q);
    const double csq = fmax(ph.gamma * p * ri, 0.0);
    c = csq > 0.0 ? rootPos(csq) : 0.0;
    eig = fabs(vn) + c;
  }
  // lU = (d(F.n / 2) / dU)^T g + we d(eig)/dU
  __device__ __forceinline__ void pullBack(const Phys &ph, const double *U, const double *n, const double *g,
                                           double we, double *lU) const {
    const double mn = U[0] * vn;
    double gv = 0.0, gn = 0.0;
#pragma unroll
    for (int d = 0; d < D; d++) {
      gv += g[d + 1] * v[d];
      gn += g[d + 1] * n[d];
    }
    const double gE = 0.5 * g[D + 1];
    // |v.n| and the sound speed c = sqrt(gamma p / rho)
    const double lvn = gE * (U[D + 1] + p) + (vn < 0.0 ? -we : we);
    double lp = 0.5 * gn + gE * vn, lrho = 0.0;
    if (c > 0.0) {
      lp += 0.5 * we * ph.gamma * ri * recip(c);
      lrho = -0.5 * we * c * ri;
    }
    const double lmn = 0.5 * (g[0] + gv), hm = 0.5 * mn;
    double lm[D], lv[D];
#pragma unroll
    for (int d = 0; d < D; d++) {
      lm[d] = lmn * n[d];
      lv[d] = hm * g[d + 1] + lvn * n[d];
    }
    primitiveVjp<D>(ph.gamma - 1.0, U[0], ri, v, lrho, lv, lp, lm, gE * vn, lU);
  }
};

// Common flux of the own state uo and the neighbour's (or ghost's) un, as
// commonFluxSided forms it, with cotangent g: lO = (dFn / duo)^T g and, where
// lN is not null, lN = (dFn / dun)^T g.  Rusanov and Lax-Friedrichs.
template <int D, int NF>
__device__ __forceinline__ void commonFluxVjp(const Phys &ph, bool right, const double *uo, const double *un,
                                              const double *n, const double *g, double *lO, double *lN) {
  if constexpr (NF == 1) {
    double vN = ph.advect[0] * n[0] + ph.advect[1] * n[1];
    if constexpr (D == 3) vN += ph.advect[2] * n[2];
    const double s = 0.5 * ph.lambda * fabs(vN) * (right ? -1.0 : 1.0);
    lO[0] = (0.5 * vN + s) * g[0];
    if (lN) lN[0] = (0.5 * vN - s) * g[0];
  } else {
    const RusanovSide<D> o(ph, uo, n), m(ph, un, n);
    // Fn = (Fo.n + Fm.n - sgn eig (un - uo)) / 2, eig the larger one (the left
    // element's where both are equal)
    const bool own = right ? o.eig > m.eig : !(m.eig > o.eig);
    const double sgn = right ? -1.0 : 1.0, he = 0.5 * sgn * (own ? o.eig : m.eig);
    double w = 0.0;
#pragma unroll
    for (int k = 0; k < NF; k++) w -= g[k] * (un[k] - uo[k]);
    w *= 0.5 * sgn;
    o.pullBack(ph, uo, n, g, own ? w : 0.0, lO);
#pragma unroll
    for (int k = 0; k < NF; k++) lO[k] += he * g[k];
    if (lN) {
      m.pullBack(ph, un, n, g, own ? 0.0 : w, lN);
#pragma unroll
      for (int k = 0; k < NF; k++) lN[k] -= he * g[k];
    }
  }
}

// The same for the Roe flux (2D, interior points), by dual numbers.
__device__ __forceinline__ void roeFluxVjp(const Phys &ph, bool right, const double *uo, const double *un,
                                           const double *n, const double *g, double *lO) {
  using DN = Dual<4>;
  DN sa[4], sb[4], nd[2], Fn[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const DN o = DN::var(uo[k], k), m = DN(un[k]);
    sa[k] = right ? m : o;
    sb[k] = right ? o : m;
  }
#pragma unroll
  for (int c = 0; c < 2; c++) nd[c] = DN(n[c]);
  roe2d<DN>(ph, sa, sb, nd, Fn);
#pragma unroll
  for (int j = 0; j < 4; j++) {
    double acc = 0.0;
#pragma unroll
    for (int k = 0; k < 4; k++) acc += g[k] * Fn[k].d[j];
    lO[j] = acc;
  }
}

// Viscous flux (viscousFlux) of the state U and gradient g, with cotangent lF:
// lU is added to, lg overwritten.  Names as in viscousFlux: G = mu grad v,
// h = mu grad e, mr = mu / rho.
template <int D, int NF>
__device__ __forceinline__ void viscousFluxVjp(const Phys &ph, const double *U, const double (&g)[D][NF],
                                               const double (&lF)[D][NF], double *lU, double (&lg)[D][NF]) {
  if constexpr (NF == 1) {
#pragma unroll
    for (int d = 0; d < D; d++) lg[d][0] = -ph.diffD * lF[d][0];
  } else {
    const double ri = recip(U[0]), H = U[D + 1] * ri, kq = ph.gamma / ph.prandtl;
    double v[D], q = 0.0;
#pragma unroll
    for (int c = 0; c < D; c++) {
      v[c] = U[c + 1] * ri;
      q += v[c] * v[c];
    }
    double mu = ph.mu_inf, dmu = 0.0;  // mu and its derivative with respect to e
    if (!ph.fixVis) {
      const double ce = (ph.gamma - 1.0) / ph.rt_inf, rt = ce * (H - 0.5 * q);
      mu *= pow(rt, 1.5) * (1.0 + ph.c_sth) / (rt + ph.c_sth);
      dmu = mu * ce * (1.5 / rt - 1.0 / (rt + ph.c_sth));
    }
    const double mr = mu * ri;
    double G[D][D];
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
      for (int c = 0; c < D; c++) G[d][c] = mr * (g[d][c + 1] - v[c] * g[d][0]);
    double diag = G[0][0] + G[1][1];
    if constexpr (D == 3) diag += G[2][2];
    diag *= 1.0 / 3.0;
    double tau[D][D];
#pragma unroll
    for (int d = 0; d < D; d++) tau[d][d] = 2.0 * (G[d][d] - diag);
    tau[0][1] = tau[1][0] = G[1][0] + G[0][1];
    if constexpr (D == 3) {
      tau[0][2] = tau[2][0] = ph.viscFix ? G[2][0] + G[0][2] : G[2][0] + G[0][1];
      tau[1][2] = tau[2][1] = ph.viscFix ? G[2][1] + G[1][2] : G[2][0] + G[1][1];
    }
    // the energy flux -(kq h + v.tau) and the momentum flux -tau
    double T[D][D], lv[D], lG[D][D], lH = 0.0, lmr = 0.0;
#pragma unroll
    for (int c = 0; c < D; c++) lv[c] = 0.0;
#pragma unroll
    for (int d = 0; d < D; d++) {
      const double e = lF[d][D + 1], lh = -kq * e;
#pragma unroll
      for (int c = 0; c < D; c++) {
        T[d][c] = -lF[d][c + 1] - e * v[c];
        lv[c] -= e * tau[d][c] + lh * G[d][c];
        lG[d][c] = -lh * v[c];
      }
      const double Z = g[d][D + 1] - H * g[d][0], lZ = mr * lh;
      lmr += lh * Z;
      lg[d][D + 1] = lZ;
      lg[d][0] = -H * lZ;
      lH -= lZ * g[d][0];
    }
    if constexpr (D == 3)
      if (!ph.viscFix) {  // Fv[0][3] is -tau_zz
        T[2][2] -= lF[0][3];
        T[0][2] += lF[0][3];
      }
    double tr = T[0][0] + T[1][1];
    if constexpr (D == 3) tr += T[2][2];
    tr *= 2.0 / 3.0;
#pragma unroll
    for (int d = 0; d < D; d++) lG[d][d] += 2.0 * T[d][d] - tr;
    const double xy = T[0][1] + T[1][0];
    lG[1][0] += xy;
    lG[0][1] += xy;
    if constexpr (D == 3) {
      const double xz = T[0][2] + T[2][0], yz = T[1][2] + T[2][1];
      lG[2][0] += xz;
      if (ph.viscFix) {
        lG[0][2] += xz;
        lG[2][1] += yz;
        lG[1][2] += yz;
      } else {
        lG[0][1] += xz;
        lG[2][0] += yz;
        lG[1][1] += yz;
      }
    }
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
      for (int c = 0; c < D; c++) {
        const double lY = mr * lG[d][c];
        lmr += lG[d][c] * (g[d][c + 1] - v[c] * g[d][0]);
        lg[d][c + 1] = lY;
        lg[d][0] -= v[c] * lY;
        lv[c] -= lY * g[d][0];
      }
    const double le = lmr * ri * dmu;  // through mu(e), e = H - v.v / 2
    lH += le;
    // v = m / rho, H = E / rho, mr = mu / rho
    double lri = lmr * mu + lH * U[D + 1];
#pragma unroll
    for (int c = 0; c < D; c++) {
      lv[c] -= le * v[c];
      lU[c + 1] += lv[c] * ri;
      lri += lv[c] * U[c + 1];
    }
    lU[D + 1] += lH * ri;
    lU[0] -= ri * ri * lri;
  }
}

// lU += (dghost / duo)^T lN of a boundary's ghost state (boundaryState), one
// direction per dual pass.
template <int D, int NF>
__device__ __forceinline__ void ghostVjp(const Phys &ph, int bc, const double *uo, const double *n,
                                         const double *lN, double *lU) {
  using DM = Dual<1>;
#pragma unroll 1
  for (int j = 0; j < NF; j++) {
    DM u[NF], w[NF], nd[D];
#pragma unroll
    for (int k = 0; k < NF; k++) {
      u[k] = DM(uo[k]);
      u[k].d[0] = k == j ? 1.0 : 0.0;
    }
#pragma unroll
    for (int c = 0; c < D; c++) nd[c] = DM(n[c]);
    boundaryState<D, NF, DM>(ph, bc, u, nd, w);
    double acc = 0.0;
#pragma unroll
    for (int k = 0; k < NF; k++) acc += lN[k] * w[k].d[0];
#pragma unroll
    for (int k = 0; k < NF; k++) lU[k] += k == j ? acc : 0.0;
  }
}

// Viscous common flux at one face point: this side's share (viscousShare) and
// the penalty tau (uL - uR), with the common flux's cotangent gc: lO (own
// state) is added to, lg (own gradient) overwritten; at boundaries lN (ghost
// state un) is added to.
template <int D, int NF>
__device__ __forceinline__ void viscousFaceVjp(const Phys &ph, bool bnd, int bc, bool right, const double *uo,
                                               const double *un, const double (&g)[D][NF], const double *n,
                                               const double *gc, double *lO, double *lN, double (&lg)[D][NF]) {
  double w[D], lF[D][NF];
  ldgWeights<D, NF, double>(ph, bnd, right, n, w);
#pragma unroll
  for (int d = 0; d < D; d++)
#pragma unroll
    for (int k = 0; k < NF; k++) lF[d][k] = w[d] * gc[k];
  if constexpr (NF > 1) {
    const double t = right ? -ph.tau : ph.tau;
#pragma unroll
    for (int k = 0; k < NF; k++) lO[k] += t * gc[k];
    if (bnd)
#pragma unroll
      for (int k = 0; k < NF; k++) lN[k] -= t * gc[k];
    if (bnd && bc == 10) {
      // adiabatic wall: the flux of the ghost state (at rest) with the ghost
      // gradient, whose energy row is e grad rho with
      // e = (E - |m|^2 / (2 rho)) / rho_ghost (boundaryGradient)
      double m2 = 0.0;
#pragma unroll
      for (int c = 0; c < D; c++) m2 += uo[c + 1] * uo[c + 1];
      const double ro = 1.0 / uo[0], rg = 1.0 / un[0], e = (uo[D + 1] - 0.5 * m2 * ro) * rg;
      double gn[D][NF];
#pragma unroll
      for (int d = 0; d < D; d++) {
#pragma unroll
        for (int k = 0; k <= D; k++) gn[d][k] = g[d][k];
        gn[d][D + 1] = e * g[d][0];
      }
      viscousFluxVjp<D, NF>(ph, un, gn, lF, lN, lg);
      double le = 0.0;
#pragma unroll
      for (int d = 0; d < D; d++) {
        le += lg[d][D + 1] * g[d][0];
        lg[d][0] += e * lg[d][D + 1];
        lg[d][D + 1] = 0.0;
      }
      lN[0] -= le * e * rg;
      le *= rg;
      lO[0] += 0.5 * le * m2 * ro * ro;
#pragma unroll
      for (int c = 0; c < D; c++) lO[c + 1] -= le * uo[c + 1] * ro;
      lO[D + 1] += le;
      return;
    }
  }
  viscousFluxVjp<D, NF>(ph, uo, g, lF, lO, lg);
}

}  // namespace frdev

// fr_viscous.hpp -- one RK stage of the viscous (LDG) path: two launches.
//
// The corrected gradient needs the neighbours' state traces and the viscous
// common flux their gradient traces, so a stage exchanges face data twice.
//
// k_visc_flux does all the work on the stage state: the LDG jumps and the
// corrected gradient, the point fluxes (inviscid and viscous) and their
// divergence, and at each flux point this element's share of the common flux.
// The common flux (face::calcInviscidFlux and calcViscousFlux,
// face.cpp:132-287) is
//   F(uL, uR).n + tau (uL - uR) + sum over the two sides of w_side . F_v(u_side, grad u_side)
// with weights w of the normal and the side alone (ldgWeights); both sides
// form the first two terms from the same states, so each side's share is half
// of them plus its own viscous term, and the two shares add up to the flux.
// Boundary points hold the whole flux (boundFace::applyViscousBCs,
// boundFace.cpp:279-320).
//
// k_visc_update adds the shares of the two sides, corrects the divergence,
// updates the state and extrapolates it to the flux points.
//
// What crosses between the launches is one value per field and flux point
// (written once, read by both sides) and the divergence: hex P3 FP64 3.8 and
// 2.6 KB per element.  Exchanging the gradient traces instead (D NF values per
// point) moved 11.5 KB out, 23 KB in and, with the common flux formed by a
// launch of its own, 77 KB per element and stage in all against 35 KB.
// Navier-Stokes 24^3 P3 (13824 elements, FP64): a stage took 61 us (gradient)
// + 61 (common flux) + 88 (stage) and takes 60 (k_visc_flux: LDS and latency at
// two waves per SIMD; three spill 20 registers and ran 83 us) + 41
// (k_visc_update, 57 in the final stage; bound by its bytes, 6.9 TB/s with the
// caches).
#pragma once

#include "fr_kernels.hpp"

namespace frdev {

// OUT: what a launch writes.
constexpr int VISC_SHARES = 1;    // the shares Gv and the divergence divW (a stage)
constexpr int VISC_GRADIENT = 2;  // the gradient traces dUf[ele][dim][field][fpt] and, with dUs
                                  // set, the gradient at the solution points

template <int D, int P, int NF, typename T, bool BND, int OUT = VISC_SHARES>
__global__ __launch_bounds__((ElemGeo<D, P>::NTH), 2) void k_visc_flux(StageArgs<T> a, T *dUf, T *dUs) {
  using G = ElemGeo<D, P>;
  using O = OneD<P>;
  constexpr int NS = G::NS, NFP = G::NFP, NFPF = G::NFPF, P1 = G::P1, TPE = G::TPE, EPB = G::EPB;
  constexpr int NSP = G::NSP, NFACE = G::NFACE, NQ = (NFP + TPE - 1) / TPE, NV = viscFields<NF>();
  // hex P3: the divergence on the matrix cores, and in FP64 the face values
  // and the gradient too (lane t handles flux point mfmaFpt(t, r) in round r);
  // gradients then stay in the lanes' registers
  constexpr bool MF = FR_MFMA && D == 3 && P == 3, MG = MF && sizeof(T) == 8;
  constexpr bool SH = (OUT & VISC_SHARES) != 0, TR = (OUT & VISC_GRADIENT) != 0;
  __shared__ T sU[EPB][NF][NSP];
  __shared__ T sC[EPB][NF][NFP];                         // LDG jumps u^ - u
  __shared__ T sG[MG ? 1 : EPB][D][NF][MG ? 1 : NSP];    // the gradient, later F~_d (not MF)
  __shared__ T s1[O::SIZE];
  const int b = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int slot = threadIdx.x / TPE, t = threadIdx.x - slot * TPE;
  const int tP = padIdx<P>(t);
  const int e = b * EPB + slot;
  const bool act = e < a.nEles;
  const bool hasS = act && t < NS;
  const size_t ec = (size_t)(act ? e : a.nEles - 1);
  const int tc = t < NS ? t : NS - 1;
  auto fq = [&](int r) { return MG ? mfmaFpt(t, r) : t + r * TPE; };
  // loads before the barrier, branch-free (idle lanes read clamped indices):
  // the face records first, which the neighbour traces' addresses need
  int pfi[NQ], pnb[NQ];
#pragma unroll
  for (int r = 0; r < NQ; r++) {
    const int f = min(fq(r), NFP - 1) / NFPF;
    pfi[r] = a.finfo[ec * NFACE + f];
    pnb[r] = a.fnbr[ec * NFACE + f];
  }
  T u[NF];  // the state at this thread's solution point
#pragma unroll
  for (int k = 0; k < NF; k++) u[k] = a.Uin[(ec * NF + k) * NS + tc];
  for (int i = threadIdx.x; i < O::SIZE; i += blockDim.x) s1[i] = a.oned[i];
  const GeoAddr<D, P> ga(a.affine, tc);
  T pn[NQ][D], pu[NQ][NF];
#pragma unroll
  for (int r = 0; r < NQ; r++) {
    const int qc = min(fq(r), NFP - 1);
#pragma unroll
    for (int c = 0; c < D; c++) pn[r][c] = a.fgeo[ga.fg(ec, c, qc)];
    const bool fetch = !(BND && pfi[r] >= FINFO_BOUNDARY);
    const T *Ur = fetch ? a.UfIn + (size_t)pnb[r] * NF * NFP + neighbourFpt<D, P>(qc, pfi[r]) : a.oned;
    const int st = fetch ? NFP : 0;
#pragma unroll
    for (int k = 0; k < NF; k++) pu[r][k] = Ur[k * st];
  }
  T pJ[D * D];
#pragma unroll
  for (int c = 0; c < D * D; c++) pJ[c] = a.JG[ga.jg(ec, c)];
  const T pdet = (T)a.detJ[ga.det(ec)];
  if (hasS)
#pragma unroll
    for (int k = 0; k < NF; k++) sU[slot][k][tP] = u[k];
  __syncthreads();
  // the state at the lane's flux point q of round r (matrix cores: all lanes)
  auto ownTrace = [&](int r, int q, T *uo) {
    if constexpr (MG) {
      T v[NF];
      mfmaFaceRound<NF, NSP, T>(s1, &sU[slot][0][0], t, u, r, v);
#pragma unroll
      for (int k = 0; k < NF; k++) uo[k] = v[k];
    } else {
      int base, stride, side, dn;
      fptLine<D, P>(q, base, stride, side, dn);
      const int lb = padIdx<P>(base), ls = padStride<P>(stride);
      const T *l1 = s1 + (side ? O::LR : O::LL);
#pragma unroll
      for (int k = 0; k < NF; k++) {
        T acc = (T)0;
#pragma unroll
        for (int m = 0; m < P1; m++) acc += l1[m] * sU[slot][k][lb + m * ls];
        uo[k] = acc;
      }
    }
  };
  // (0) at every flux point the LDG jump, and what both sides form alike of
  // the common flux
  T I[SH ? NQ : 1][NF];
  // matrix cores: the state at the lane's flux points, kept for (2) (20 registers
  // below the limit of two waves; formed again there, a stage of Navier-Stokes
  // 24^3 P3 took 116.5 us on average against 114.0, 40^3 547 against 537.
  // Staging the gradient in LDS for (2) as well, instead of lane pulls, gained
  // nothing: 114.5 and 540)
  T uf[MG ? NQ : 1][NF];
#pragma unroll
  for (int r = 0; r < NQ; r++) {
    const int q = fq(r);
    T(&uo)[NF] = uf[MG ? r : 0];
    if (MG && act) ownTrace(r, q, uo);
    if (act && q < NFP) {
      if (!MG) ownTrace(r, q, uo);
      T un[NF], dUc[NF];
      const int fi = pfi[r];
      const bool bnd = BND && fi >= FINFO_BOUNDARY;
      const bool right = !bnd && ((fi >> 5) & 1);
      if (bnd) {
        boundaryState<D, NF, T>(a.ph, fi - FINFO_BOUNDARY, uo, pn[r], un);
      } else {
#pragma unroll
        for (int k = 0; k < NF; k++) un[k] = pu[r][k];
      }
      ldgJump<D, NF, T>(a.ph, bnd, right, uo, un, pn[r], dUc);
#pragma unroll
      for (int k = 0; k < NF; k++) sC[slot][k][q] = dUc[k];
      if constexpr (SH) {
        T ws, Fn[NF];
        const bool hasWs = commonFluxSided<D, NF, T>(a.ph, bnd, right, uo, un, pn[r], Fn, &ws);
        // the CFL wave speed at the face's left points (and boundary points);
        // the right element's points keep theirs (face.cpp:74-80)
        if (a.waveSp && hasWs && !right) a.waveSp[(size_t)e * NFP + q] = (double)ws;
        const T tau = NF == 1 ? (T)0 : right ? -(T)a.ph.tau : (T)a.ph.tau;
#pragma unroll
        for (int k = 0; k < NF; k++) {
          const T f = NF == 1 ? Fn[k] : Fn[k] + tau * (uo[k] - un[k]);
          I[r][k] = bnd ? f : (T)0.5 * f;
        }
      }
    }
  }
  elementSync<TPE>();
  // (1) the corrected physical gradient
  int si, sj, sk;
  if (D == 3) {
    sk = tc / (P1 * P1);
    sj = (tc - P1 * P1 * sk) / P1;
    si = tc - P1 * sj - P1 * P1 * sk;
  } else {
    si = tc % P1;
    sj = tc / P1;
    sk = 0;
  }
  T g[D][NF];
  if (MG ? act : hasS) {
    if constexpr (MG) {
      mfmaGradient<NF, NSP, T>(s1, &sU[slot][0][0], u, &sC[slot][0][0], t, pJ, pdet, g);
    } else {
      correctedGradient<D, P, NF, T>(s1, &sU[slot][0][0], &sC[slot][0][0], t, si, sj, sk, pJ, pdet, g);
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int k = 0; k < NF; k++) sG[slot][d][k][tP] = g[d][k];
    }
    if constexpr (TR)
      if (dUs)
#pragma unroll
        for (int d = 0; d < D; d++)
#pragma unroll
          for (int k = 0; k < NF; k++) dUs[(((size_t)e * D + d) * NF + k) * NS + t] = g[d][k];
  }
  if constexpr (!MG) elementSync<TPE>();
  // (2) the gradient at the flux points, and from it the share's viscous term
#pragma unroll
  for (int r = 0; r < NQ; r++) {
    const int q = fq(r);
    T gf[D][NF];
    T(&uo)[NF] = uf[MG ? r : 0];
    if constexpr (MG) {
      if (act) {
#pragma unroll
        for (int d = 0; d < D; d++) mfmaFaceRoundReg<NF, T>(s1, t, g[d], r, gf[d]);
      }
    }
    if (!act || q >= NFP) continue;
    if constexpr (!MG) {
      int base, stride, side, dn;
      fptLine<D, P>(q, base, stride, side, dn);
      const int lb = padIdx<P>(base), ls = padStride<P>(stride);
      const T *l1 = s1 + (side ? O::LR : O::LL);
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int k = 0; k < NF; k++) {
          T acc = (T)0;
#pragma unroll
          for (int m = 0; m < P1; m++) acc += l1[m] * sG[slot][d][k][lb + m * ls];
          gf[d][k] = acc;
        }
      if (SH) ownTrace(r, q, uo);
    }
    if constexpr (TR) {
      T *Ge = dUf + (size_t)e * D * NF * NFP;
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int k = 0; k < NF; k++) Ge[(d * NF + k) * NFP + q] = gf[d][k];
    }
    if constexpr (SH) {
      const int fi = pfi[r];
      const bool bnd = BND && fi >= FINFO_BOUNDARY;
      T C[NV];
      if (bnd && NF > 1 && fi - FINFO_BOUNDARY == 10) {
        // adiabatic wall: the ghost state's flux with the ghost gradient
        T un[NF], gn[D][NF];
        boundaryState<D, NF, T>(a.ph, 10, uo, pn[r], un);
        boundaryGradient<D, NF, T>(a.ph, 10, uo, un, gf, gn);
        viscousShare<D, NF, T>(a.ph, true, false, un, gn, pn[r], C);
      } else {
        viscousShare<D, NF, T>(a.ph, bnd, !bnd && ((fi >> 5) & 1), uo, gf, pn[r], C);
      }
#pragma unroll
      for (int k = 0; k < NF; k++)
        a.Gv[((size_t)e * NF + k) * NFP + q] = k < NF - NV ? I[r][k] : I[r][k] + C[k < NF - NV ? 0 : k - (NF - NV)];
    }
  }
  if constexpr (!SH) return;
  // (3) the point flux (calcInviscidFlux_spts, solver.cpp:514-539, and
  // calcViscousFlux_spts, solver.cpp:562-596), its contravariant components
  // and their derivatives, with the correction of the extrapolated flux folded
  // in (OneD::DMF)
  T F[D][NF], div[NF];
  if (hasS) {
    T Fv[D][NF];
    if constexpr (!MG) {
      // read back instead of kept in registers through (2)
#pragma unroll
      for (int k = 0; k < NF; k++) {
        u[k] = sU[slot][k][tP];
#pragma unroll
        for (int d = 0; d < D; d++) g[d][k] = sG[slot][d][k][tP];
      }
    }
    inviscidFlux<D, NF, T>(a.ph, u, F);
    viscousFlux<D, NF, T>(a.ph, u, g, Fv);
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
      for (int k = 0; k < NF; k++) F[d][k] = Fv[d][k] + F[d][k];
  }
  if constexpr (MF) {
    if (act) mfmaDivergence<NF, T>(s1, t, pJ, F, div);
  } else {
    elementSync<TPE>();  // the gradient in sG has been read
    if (hasS)
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int k = 0; k < NF; k++) {
          T acc = (T)0;
#pragma unroll
          for (int d2 = 0; d2 < D; d2++) acc += pJ[d * D + d2] * F[d2][k];
          sG[slot][d][k][tP] = acc;
        }
    elementSync<TPE>();
    if (hasS)
#pragma unroll
      for (int d = 0; d < D; d++) {
        const int id = (d == 0) ? si : (d == 1) ? sj : sk;
#pragma unroll
        for (int k = 0; k < NF; k++) {
          T acc = (T)0;
#pragma unroll
          for (int m = 0; m < P1; m++) {
            const int sp = (d == 0)   ? m + P1 * (sj + P1 * sk)
                           : (d == 1) ? si + P1 * (m + P1 * sk)
                                      : si + P1 * (sj + P1 * m);
            acc += s1[O::DMF + id * P1 + m] * sG[slot][d][k][padIdx<P>(sp)];
          }
          div[k] = (d == 0) ? acc : acc + div[k];
        }
      }
  }
  if (hasS)
#pragma unroll
    for (int k = 0; k < NF; k++) a.divW[((size_t)e * NF + k) * NS + t] = div[k];
}

// The end of a viscous stage, as phases (4) and (5) of stageBody: the correction of the
// jumps sJe [NF][NFP] (correctDivFlux, solver.cpp:789-806) added to the
// divergence div, the stage update from the base pb (final stages: with the
// earlier residuals' terms already subtracted), and the face traces of the
// updated state, staged in sSe [NF][NSP].
template <int D, int P, int NF, typename T, bool FIN>
__device__ __forceinline__ void viscUpdate(const StageArgs<T> &a, const T *s1, const T *sJe, T *sSe, const int e,
                                           const int t, const bool act, const T *div, const double *pb,
                                           const double pdet, const double pdt) {
  using G = ElemGeo<D, P>;
  using O = OneD<P>;
  constexpr int NS = G::NS, NSP = G::NSP, NFP = G::NFP, P1 = G::P1, TPE = G::TPE, NFACE = G::NFACE;
  constexpr int NQ = (NFP + TPE - 1) / TPE;
  constexpr bool MF = FR_MFMA && D == 3 && P == 3, MFF = MF && sizeof(T) == 8;
  // the FP64 base of the final stages is absolute; FP32 stage states hold the
  // energy less Phys::eOff
  constexpr bool base64 = FIN;
  T utv[NF];  // the updated state at this thread's point
  if (act && t < NS) {
    int cq[NFACE], cside[NFACE], cax[NFACE];
    corrEntries<D, P>(t, cq, cside, cax);
    T cw[NFACE];  // correction weights, read once for all fields
#pragma unroll
    for (int f = 0; f < NFACE; f++) cw[f] = s1[(cside[f] ? O::GR : O::GL) + cax[f]];
    const size_t eo = (size_t)e * NF * NS;
#pragma unroll
    for (int k = 0; k < NF; k++) {
      T corr = (T)0;
#pragma unroll
      for (int f = 0; f < NFACE; f++) corr += cw[f] * sJe[k * NFP + cq[f]];
      const T dv = corr + div[k];
      const size_t gi = eo + (size_t)k * NS + t;
      if (a.divF) __builtin_nontemporal_store(dv, a.divF + gi);
      if (!FIN && a.mode == 0) continue;
      // stage terms RK * divF / detJ * dt, with dt / detJ formed once per point
      const double dtJ = pdt / pdet;
      double u = pb[k];
      if (FIN && a.mode == 2) {
        // earlier residuals: already subtracted from pb
        const double cl = (a.nprev == 0) ? a.c0 : (a.nprev == 1) ? a.c1 : (a.nprev == 2) ? a.c2 : a.c3;
        u -= cl * (double)dv * dtJ;
      } else {
        u = u - a.rk * (double)dv * dtJ;
      }
      // the updated state in the residual precision, for the traces
      double ut = u;
      if constexpr (hasEnergyOffset<T>())
        if (k == NF - 1 && base64) ut = u - a.ph.eOff;
      if constexpr (!FIN) {
        if (a.Unext) __builtin_nontemporal_store((T)u, a.Unext + gi);
      } else {
        __builtin_nontemporal_store(u, a.Uout + gi);
        if (a.Uout32) __builtin_nontemporal_store((float)ut, a.Uout32 + gi);
      }
      sSe[k * NSP + padIdx<P>(t)] = (T)ut;
      utv[k] = (T)ut;
    }
  }
  if (!FIN && a.mode == 0) return;
  elementSync<TPE>();
  if (!act) return;
  T *Fe = a.UfOut + (size_t)e * NF * NFP;
#pragma unroll
  for (int r = 0; r < NQ; r++) {
    const int q = MF ? mfmaFpt(t, r) : t + r * TPE;
    T tv[NF];
    if constexpr (MFF) mfmaFaceRound<NF, NSP, T>(s1, sSe, t, utv, r, tv);
    if (q >= NFP) continue;
    if constexpr (MFF) {
#pragma unroll
      for (int k = 0; k < NF; k++) __builtin_nontemporal_store(tv[k], Fe + k * NFP + q);
      continue;
    }
    int base, stride, side, dn;
    fptLine<D, P>(q, base, stride, side, dn);
    const int lb = padIdx<P>(base), ls = padStride<P>(stride);
    const T *l1 = s1 + (side ? O::LR : O::LL);
#pragma unroll
    for (int k = 0; k < NF; k++) {
      T acc = (T)0;
#pragma unroll
      for (int m = 0; m < P1; m++) acc += l1[m] * sSe[k * NSP + lb + m * ls];
      __builtin_nontemporal_store(acc, Fe + k * NFP + q);
    }
  }
}

// The second half of a viscous stage: the common flux from the two sides'
// shares, then the end of the stage as in the inviscid kernel (viscUpdate).
// Bound by its bytes (the shares, the divergence, the base and the outputs);
// no element reads another's LDS, so beyond the barrier for the 1D table the
// elements of a workgroup run on their own.
template <int D, int P, int NF, typename T, bool BND, bool FIN>
__global__ __launch_bounds__((ElemGeo<D, P>::NTH)) void k_visc_update(StageArgs<T> a) {
  using G = ElemGeo<D, P>;
  using O = OneD<P>;
  constexpr int NS = G::NS, NFP = G::NFP, NFPF = G::NFPF, TPE = G::TPE, EPB = G::EPB;
  constexpr int NSP = G::NSP, NFACE = G::NFACE, NQ = (NFP + TPE - 1) / TPE;
  __shared__ T sJ[EPB][NF][NFP];
  __shared__ T sS[EPB][NF][NSP];
  __shared__ T s1[O::SIZE];
  const int R = gridDim.x >> 3, j = blockIdx.x >> 3;
  const int b = (blockIdx.x & 7) * R + (a.rev ? R - 1 - j : j);
  const int slot = threadIdx.x / TPE, t = threadIdx.x - slot * TPE;
  const int e = b * EPB + slot;
  const bool act = e < a.nEles;
  const size_t ec = (size_t)(act ? e : a.nEles - 1);
  const int tc = t < NS ? t : NS - 1;
  // coalesced: flux point t + r TPE (the traces below use their own order)
  int pfi[NQ], pnb[NQ];
#pragma unroll
  for (int r = 0; r < NQ; r++) {
    const int f = min(t + r * TPE, NFP - 1) / NFPF;
    pfi[r] = a.finfo[ec * NFACE + f];
    pnb[r] = a.fnbr[ec * NFACE + f];
  }
  const GeoAddr<D, P> ga(a.affine, tc);
  T So[NQ][NF], Sn[NQ][NF], dA[NQ];
#pragma unroll
  for (int r = 0; r < NQ; r++) {
    const int qc = min(t + r * TPE, NFP - 1);
    const bool bnd = BND && pfi[r] >= FINFO_BOUNDARY;
    const T *go = a.Gv + ec * NF * NFP + qc;
    const T *gn = bnd ? go : a.Gv + (size_t)pnb[r] * NF * NFP + neighbourFpt<D, P>(qc, pfi[r]);
    dA[r] = a.fgeo[ga.fg(ec, D, qc)];
#pragma unroll
    for (int k = 0; k < NF; k++) So[r][k] = go[k * NFP];
#pragma unroll
    for (int k = 0; k < NF; k++) Sn[r][k] = gn[k * NFP];
  }
  T div[NF], pd[3][NF];
  double pb[NF];
#pragma unroll
  for (int k = 0; k < NF; k++) {
    const size_t gi = (ec * NF + k) * NS + tc;
    div[k] = a.divW[gi];
    pb[k] = FIN ? a.Ubase[gi] : (double)a.UbaseT[gi];
  }
  const double pdet = a.detJ[ga.det(ec)], pdt = a.dtE[ec * a.dtStride];
  if constexpr (FIN) {
    const T *dp[3] = {a.dprev0, a.dprev1, a.dprev2};
#pragma unroll
    for (int r = 0; r < 3; r++)
      if (a.mode == 2 && r < a.nprev)
#pragma unroll
        for (int k = 0; k < NF; k++) pd[r][k] = __builtin_nontemporal_load(dp[r] + (ec * NF + k) * NS + tc);
  }
  for (int i = threadIdx.x; i < O::SIZE; i += blockDim.x) s1[i] = a.oned[i];
  if (act)
#pragma unroll
    for (int r = 0; r < NQ; r++) {
      const int q = t + r * TPE;
      const bool bnd = BND && pfi[r] >= FINFO_BOUNDARY;
      const T scale = (!bnd && ((pfi[r] >> 5) & 1)) ? -dA[r] : dA[r];
      if (q < NFP)
#pragma unroll
        for (int k = 0; k < NF; k++) sJ[slot][k][q] = (bnd ? So[r][k] : So[r][k] + Sn[r][k]) * scale;
    }
  if constexpr (FIN)
    if (a.mode == 2) subtractEarlier<NF, T>(a, pd, pdt / pdet, pb);
  __syncthreads();
  viscUpdate<D, P, NF, T, FIN>(a, s1, &sJ[slot][0][0], &sS[slot][0][0], e, t, act, div, pb, pdet, pdt);
}

}  // namespace frdev

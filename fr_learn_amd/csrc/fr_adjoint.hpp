// fr_adjoint.hpp -- hand-written adjoint (vector-Jacobian product) of the
// FR residual and of one RK step, FP64.
//
// For a cotangent nu of divF (layout [ele][field][spt]) the kernels form
// w = nu^T d divF / dU in the state's layout.  They transpose the residual
// phase by phase, with the same index maps:
//   correction  divF[t] += sum_f corr(t, q_f) J[q_f]  ->  lamJ[q] = sum over
//               the solution points on q's line of corr * nu  (a g-line
//               contraction, like an extrapolation with g_L / g_R weights);
//   face flux   J[q] = Fn(U_L, U_R, n_L) * scale - disFn[q]: the cotangent of
//               the common flux at a face point is gc = lamJ * scale of this
//               element plus that of the neighbour's paired point (both
//               elements evaluate the same Fn), pulled back to this element's
//               traces (commonFluxVjp, viscousFaceVjp);
//   volume      divF[t] = sum_d Dm F~_d and -disFn = -extrapolation(F~_d):
//               transposed along the lines, then F~ = JGinv F transposed,
//               then the point fluxes (inviscidFluxVjp, viscousFluxVjp);
//   gradient    (viscous) Q = JGinv^T (Dm U + lift(u^ - u)) / detJ transposed:
//               to the state along the lines and to the jumps u^ - u, whose
//               cotangents B the neighbours exchange once more (k_vjp_ldg);
//   traces      u_o[q] = extrapolation of U: transposed with corrEntries.
// Element-parallel and gather-only: the scaled face cotangents A = lamJ * scale
// and B are written by every element in one launch and read by its neighbours
// in the next, so no atomics are needed.
//
// One RK stage of the step's adjoint is one launch (inviscid) or two
// (viscous): the last kernel of a stage has w in registers, so it also adds w
// to the step's cotangent, forms the next stage's nu and its face cotangents
// (vjpTail).  With a launch for each of those and the traces of the stage states
// extrapolated again, a step was 27 launches (viscous 42) and is 9 (16).
#pragma once

#include <hip/hip_runtime.h>

#include "fr_kernels.hpp"
#include "fr_reverse.hpp"

namespace frdev {

struct VjpArgs {
  const double *U, *nu;        // the state and the cotangent of divF [ele][field][spt]
  const double *Uf;            // traces of the state [ele][field][fpt], every face
  const double *A;             // face cotangents of nu [ele][field][fpt]
  const double *JG, *fgeo, *detJ;
  const int32_t *fnbr;
  const int8_t *finfo;
  const double *oned;
  Phys ph;
  int nEles, affine;           // affine: geometry layout (GeoAddr)
  double *out;                 // w (viscous: less the common solution's part until k_vjp_ldg)
  double *B;                   // viscous: cotangents of the jumps u^ - u [ele][field][fpt]
  // the RK step around it (all null for the residual's VJP alone)
  const double *lam1;          // cotangent of the step's result
  double *lam0;                // += w
  double *nuNext, *ANext;      // nu = dt / detJ (alpha lam1 + beta w) and its face cotangents
  double alpha, beta;
  const double *dtE;
  int dtStride;
};

// Block of this workgroup, each XCD walking a contiguous range of elements (as
// k_stage; the grid is a multiple of 8), so that neighbours share its L2.
__device__ __forceinline__ int vjpBlock() { return (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3); }

// sum_m g_side[m] * x[line_q(m)] at flux point q: lamJ of a cotangent x
// ([NF][NSP] in LDS, padded rows)
template <int D, int P, int NF>
__device__ __forceinline__ void lamJAt(const double *s1, const double *x, int q, double *out) {
  using O = OneD<P>;
  constexpr int NSP = ElemGeo<D, P>::NSP, P1 = P + 1;
  int base, stride, side, dn;
  fptLine<D, P>(q, base, stride, side, dn);
  const int lb = padIdx<P>(base), ls = padStride<P>(stride);
  const double *g = s1 + (side ? O::GR : O::GL);
#pragma unroll
  for (int k = 0; k < NF; k++) {
    double acc = 0;
#pragma unroll
    for (int m = 0; m < P1; m++) acc += g[m] * x[k * NSP + lb + m * ls];
    out[k] = acc;
  }
}

// Face cotangents A = lamJ * (+dA left / boundary, -dA right) of element e's
// cotangent x (LDS, [NF][NSP]).
template <int D, int P, int NF>
__device__ __forceinline__ void faceCotangents(const VjpArgs &a, const double *s1, const double *x, const size_t e,
                                               const int t, double *A) {
  using G = ElemGeo<D, P>;
  constexpr int NFP = G::NFP, NFPF = G::NFPF, TPE = G::TPE, NFACE = G::NFACE;
  const GeoAddr<D, P> ga(a.affine, 0);
  for (int q = t; q < NFP; q += TPE) {
    double lj[NF];
    lamJAt<D, P, NF>(s1, x, q, lj);
    const int fi = a.finfo[e * NFACE + q / NFPF];
    const double dA = a.fgeo[ga.fg(e, D, q)];
    const double scale = fi < FINFO_BOUNDARY && ((fi >> 5) & 1) ? -dA : dA;
#pragma unroll
    for (int k = 0; k < NF; k++) A[(e * NF + k) * NFP + q] = lj[k] * scale;
  }
}

// The end of a stage's VJP, with w at this thread's solution point: w to
// out (where there is no step around it), the step's cotangent, and the next
// stage's nu with its face cotangents, staged in sX [NF][NSP].
template <int D, int P, int NF>
__device__ __forceinline__ void vjpTail(const VjpArgs &a, const double *s1, double *sX, const int e, const int t,
                                        const bool act, const double *w) {
  using G = ElemGeo<D, P>;
  constexpr int NS = G::NS, NSP = G::NSP, TPE = G::TPE;
  const bool hasS = act && t < NS;
  const size_t g0 = (size_t)e * NF * NS + t;
  if (!a.lam0) {
    if (hasS)
#pragma unroll
      for (int k = 0; k < NF; k++) a.out[g0 + k * NS] = w[k];
    return;
  }
  if (hasS) {
    double dtJ = 0.0;
    if (a.nuNext) dtJ = a.dtE[(size_t)e * a.dtStride] / a.detJ[GeoAddr<D, P>(a.affine, t).det((size_t)e)];
#pragma unroll
    for (int k = 0; k < NF; k++) {
      const size_t gi = g0 + k * NS;
      a.lam0[gi] += w[k];
      if (a.nuNext) {
        const double v = (a.alpha * a.lam1[gi] + a.beta * w[k]) * dtJ;
        a.nuNext[gi] = v;
        sX[k * NSP + padIdx<P>(t)] = v;
      }
    }
  }
  if (!a.nuNext) return;
  elementSync<TPE>();
  if (act) faceCotangents<D, P, NF>(a, s1, sX, (size_t)e, t, a.ANext);
}

// The first nu of a step, dt / detJ alpha lam1, with its face cotangents, and
// lam0 = lam1; or (lam0 null) the face cotangents of nu alone.
template <int D, int P, int NF>
__global__ __launch_bounds__((ElemGeo<D, P>::NTH)) void k_vjp_seed(VjpArgs a) {
  using G = ElemGeo<D, P>;
  using O = OneD<P>;
  constexpr int NS = G::NS, NSP = G::NSP, TPE = G::TPE, EPB = G::EPB;
  __shared__ double sX[EPB][NF][NSP];
  __shared__ double s1[O::SIZE];
  const int slot = threadIdx.x / TPE, t = threadIdx.x - slot * TPE;
  const int e = blockIdx.x * EPB + slot;
  const bool act = e < a.nEles;
  for (int i = threadIdx.x; i < O::SIZE; i += blockDim.x) s1[i] = a.oned[i];
  if (act && t < NS) {
    double f = 1.0;
    if (a.lam0) f = a.alpha * a.dtE[(size_t)e * a.dtStride] / a.detJ[GeoAddr<D, P>(a.affine, t).det((size_t)e)];
#pragma unroll
    for (int k = 0; k < NF; k++) {
      const size_t gi = ((size_t)e * NF + k) * NS + t;
      const double l = (a.lam0 ? a.lam1 : a.nu)[gi], v = f * l;
      if (a.lam0) {
        a.lam0[gi] = l;
        a.nuNext[gi] = v;
      }
      sX[slot][k][padIdx<P>(t)] = v;
    }
  }
  __syncthreads();
  if (act) faceCotangents<D, P, NF>(a, s1, &sX[slot][0][0], (size_t)e, t, a.ANext);
}

// Cotangents of the contravariant fluxes F~_d at solution point t and from
// them those of the physical point fluxes: along the lines the transposed
// derivative of nu (sL, padded rows), less the jump's part (sJ = lamJ).
template <int D, int P, int NF>
__device__ __forceinline__ void pointFluxCotangent(const double *s1, const double *sL, const double *sJ, const int t,
                                                   const double *pJ, double (&lF)[D][NF]) {
  using G = ElemGeo<D, P>;
  using O = OneD<P>;
  constexpr int NSP = G::NSP, NFP = G::NFP, P1 = G::P1, NFACE = G::NFACE;
  const int sk = D == 3 ? t / (P1 * P1) : 0, sj = (t / P1) % P1, si = t % P1;
  int cq[NFACE], cside[NFACE], cax[NFACE];
  corrEntries<D, P>(t, cq, cside, cax);
  double lw[NFACE];
#pragma unroll
  for (int f = 0; f < NFACE; f++) lw[f] = cside[f] ? -s1[O::LR + cax[f]] : s1[O::LL + cax[f]];
#pragma unroll
  for (int d2 = 0; d2 < D; d2++)
#pragma unroll
    for (int k = 0; k < NF; k++) lF[d2][k] = 0.0;
#pragma unroll
  for (int d = 0; d < D; d++) {
    const int id = (d == 0) ? si : (d == 1) ? sj : sk;
#pragma unroll
    for (int k = 0; k < NF; k++) {
      double acc = 0;
      if constexpr (FR_MFMA && D == 3 && P == 3) {
        const MfmaLane<double> L(s1, t);
        const double b = sL[k * NSP + (d == 2 ? padIdx<P>(t) : d == 0 ? L.px : L.py)];
        const double der = MfmaVec<double>::mma(L.aDT, b, 0.0);
        acc = d < 2 ? lanePull(d == 0 ? L.ix : L.iy, der) : der;
      } else {
#pragma unroll
        for (int m = 0; m < P1; m++) {
          const int sp = (d == 0)   ? m + P1 * (sj + P1 * sk)
                         : (d == 1) ? si + P1 * (m + P1 * sk)
                                    : si + P1 * (sj + P1 * m);
          acc += s1[O::DM + m * P1 + id] * sL[k * NSP + padIdx<P>(sp)];
        }
      }
#pragma unroll
      for (int f = 0; f < NFACE; f++)
        if (faceAxis<D>(f) == d) acc += lw[f] * sJ[k * NFP + cq[f]];
#pragma unroll
      for (int d2 = 0; d2 < D; d2++) lF[d2][k] += pJ[d * D + d2] * acc;
    }
  }
}

// Inviscid VJP, one TPE-thread group per element.  ROE: meshes with the Roe
// flux (2D), whose interior face points take its Jacobian from dual numbers.
template <int D, int P, int NF, bool BND, bool ROE>
__global__ __launch_bounds__((ElemGeo<D, P>::NTH)) void k_vjp_state(VjpArgs a) {
  using G = ElemGeo<D, P>;
  using O = OneD<P>;
  constexpr int NS = G::NS, NSP = G::NSP, NFP = G::NFP, NFPF = G::NFPF, P1 = G::P1, TPE = G::TPE, EPB = G::EPB;
  constexpr int NFACE = G::NFACE, NQ = (NFP + TPE - 1) / TPE;
  __shared__ double sU[EPB][NF][NSP];
  __shared__ double sL[EPB][NF][NSP];
  __shared__ double sJ[EPB][NF][NFP];   // lamJ
  __shared__ double sUo[EPB][NF][NFP];  // cotangent of this element's traces
  __shared__ double s1[O::SIZE];
  const int slot = threadIdx.x / TPE, t = threadIdx.x - slot * TPE;
  const int e = vjpBlock() * EPB + slot;
  const bool act = e < a.nEles;
  const bool hasS = act && t < NS;
  const size_t ec = (size_t)(act ? e : a.nEles - 1);
  const int tc = t < NS ? t : NS - 1, tP = padIdx<P>(t);
  // loads before the barrier (idle lanes read clamped indices), the face
  // records first, which the neighbours' addresses need
  int pfi[NQ], pnb[NQ];
#pragma unroll
  for (int r = 0; r < NQ; r++) {
    const int f = min(t + r * TPE, NFP - 1) / NFPF;
    pfi[r] = a.finfo[ec * NFACE + f];
    pnb[r] = a.fnbr[ec * NFACE + f];
  }
  for (int i = threadIdx.x; i < O::SIZE; i += blockDim.x) s1[i] = a.oned[i];
  double u[NF], l[NF];
#pragma unroll
  for (int k = 0; k < NF; k++) {
    u[k] = a.U[(ec * NF + k) * NS + tc];
    l[k] = a.nu[(ec * NF + k) * NS + tc];
  }
  const GeoAddr<D, P> ga(a.affine, tc);
  double pn[NQ][D + 1], pu[NQ][NF], pA[NQ][NF];
#pragma unroll
  for (int r = 0; r < NQ; r++) {
    const int qc = min(t + r * TPE, NFP - 1);
#pragma unroll
    for (int c = 0; c <= D; c++) pn[r][c] = a.fgeo[ga.fg(ec, c, qc)];
    const bool bnd = BND && pfi[r] >= FINFO_BOUNDARY;
    const size_t o = bnd ? ec * NF * NFP + qc : (size_t)pnb[r] * NF * NFP + neighbourFpt<D, P>(qc, pfi[r]);
#pragma unroll
    for (int k = 0; k < NF; k++) {
      pu[r][k] = a.Uf[o + k * NFP];
      pA[r][k] = a.A[o + k * NFP];
    }
  }
  double pJ[D * D];
#pragma unroll
  for (int c = 0; c < D * D; c++) pJ[c] = a.JG[ga.jg(ec, c)];
  if (hasS)
#pragma unroll
    for (int k = 0; k < NF; k++) {
      sU[slot][k][tP] = u[k];
      sL[slot][k][tP] = l[k];
    }
  __syncthreads();
  // face points: lamJ, the flux cotangent and its pull-back to this trace
  if (act) {
#pragma unroll
    for (int r = 0; r < NQ; r++) {
      const int q = t + r * TPE;
      if (q >= NFP) continue;
      double lj[NF], uo[NF], gc[NF], lO[NF];
      lamJAt<D, P, NF>(s1, &sL[slot][0][0], q, lj);
      int base, stride, side, dn;
      fptLine<D, P>(q, base, stride, side, dn);
      const int lb = padIdx<P>(base), ls = padStride<P>(stride);
      const double *l1 = s1 + (side ? O::LR : O::LL);
#pragma unroll
      for (int k = 0; k < NF; k++) {
        double acc = 0;
#pragma unroll
        for (int m = 0; m < P1; m++) acc += l1[m] * sU[slot][k][lb + m * ls];
        uo[k] = acc;
        sJ[slot][k][q] = lj[k];
      }
      const int fi = pfi[r];
      const bool bnd = BND && fi >= FINFO_BOUNDARY;
      const bool right = !bnd && ((fi >> 5) & 1);
      const double *n = pn[r], dA = pn[r][D];
      if (bnd) {
        double un[NF], lN[NF];
#pragma unroll
        for (int k = 0; k < NF; k++) gc[k] = lj[k] * dA;
        boundaryState<D, NF, double>(a.ph, fi - FINFO_BOUNDARY, uo, n, un);
        commonFluxVjp<D, NF>(a.ph, false, uo, un, n, gc, lO, lN);
        ghostVjp<D, NF>(a.ph, fi - FINFO_BOUNDARY, uo, n, lN, lO);
      } else {
#pragma unroll
        for (int k = 0; k < NF; k++) gc[k] = lj[k] * (right ? -dA : dA) + pA[r][k];
        if constexpr (ROE) {
          roeFluxVjp(a.ph, right, uo, pu[r], n, gc, lO);
        } else {
          commonFluxVjp<D, NF>(a.ph, right, uo, pu[r], n, gc, lO, nullptr);
        }
      }
#pragma unroll
      for (int k = 0; k < NF; k++) sUo[slot][k][q] = lO[k];
    }
  }
  elementSync<TPE>();
  double w[NF];
  if (hasS) {
    double lF[D][NF];
    pointFluxCotangent<D, P, NF>(s1, &sL[slot][0][0], &sJ[slot][0][0], t, pJ, lF);
    inviscidFluxVjp<D, NF>(a.ph, u, lF, w);
    // trace extrapolation, transposed
    int cq[NFACE], cside[NFACE], cax[NFACE];
    corrEntries<D, P>(t, cq, cside, cax);
#pragma unroll
    for (int f = 0; f < NFACE; f++) {
      const double c = s1[(cside[f] ? O::LR : O::LL) + cax[f]];
#pragma unroll
      for (int k = 0; k < NF; k++) w[k] += c * sUo[slot][k][cq[f]];
    }
  }
  vjpTail<D, P, NF>(a, s1, &sU[slot][0][0], e, t, act, w);
}

// Viscous (LDG) VJP, less the common solution's part: everything that hangs on
// one element's state and gradient, in one kernel.  The gradient and its
// traces are formed again from the state (as k_visc_flux does), the fluxes
// pulled back at the flux and solution points, and the gradient's cotangent
// taken back to the state and, as B, to the jumps u^ - u.
//
// A block is one wavefront (or one element where that takes more): the LDS of
// an element -- 26 KB at hex P3, of which the cotangents of the gradient traces
// are half -- decides how many run on a CU.  20^3 P3 (8000 elements): 95 us and
// about 20 KB per element, against 37 + 280 + 136 us and 110 KB with launches of
// their own for the gradient traces, the face points and the state and
// dual-number passes (256 VGPRs and 210 AGPRs in the face kernel).  Six blocks
// fit a CU at P3, so two waves per SIMD are asked for (23 spilled registers);
// elsewhere the LDS leaves little over one wave per SIMD and the kernel takes
// the registers it wants.
template <int D, int P>
struct VjpTile {
  static constexpr int TPE = ElemGeo<D, P>::TPE;
  static constexpr int EPB = TPE < 64 ? 64 / TPE : 1, NTH = TPE * EPB;
};

template <int D, int P, int NF, bool BND>
__global__ __launch_bounds__((VjpTile<D, P>::NTH), (P == 3 && !BND) ? 2 : 1) void k_vjp_visc(VjpArgs a) {
  using G = ElemGeo<D, P>;
  using O = OneD<P>;
  constexpr int NS = G::NS, NSP = G::NSP, NFP = G::NFP, NFPF = G::NFPF, P1 = G::P1, TPE = G::TPE;
  constexpr int EPB = VjpTile<D, P>::EPB, NFACE = G::NFACE, NQ = (NFP + TPE - 1) / TPE;
  // hex P3: line operators on the matrix cores (lane t handles flux point
  // mfmaFpt(t, r) in round r)
  constexpr bool MG = FR_MFMA && D == 3 && P == 3;
  // LDS of an element: state, nu, lamJ, jumps (later the cotangents of the state
  // traces), cotangents of the gradient traces (before that the gradient); the
  // reference gradient's cotangent takes the place of all but the state at
  // the end
  constexpr int oL = NF * NSP, oJ = oL + NF * NSP, oC = oJ + NF * NFP, oQ = oC + NF * NFP;
  constexpr int nQ = D * NF * (MG || NFP > NSP ? NFP : NSP), SIZE = oQ + nQ;
  __shared__ double sm[EPB][SIZE];
  __shared__ double s1[O::SIZE];
  const int slot = threadIdx.x / TPE, t = threadIdx.x - slot * TPE;
  double *sU = sm[slot], *sL = sU + oL, *sJ = sU + oJ, *sC = sU + oC, *sQ = sU + oQ, *sLQ = sU + oL;
  const int e = vjpBlock() * EPB + slot;
  const bool act = e < a.nEles;
  const bool hasS = act && t < NS;
  const size_t ec = (size_t)(act ? e : a.nEles - 1);
  const int tc = t < NS ? t : NS - 1, tP = padIdx<P>(t);
  auto fq = [&](int r) { return MG ? mfmaFpt(t, r) : t + r * TPE; };
  int pfi[NQ], pnb[NQ];
#pragma unroll
  for (int r = 0; r < NQ; r++) {
    const int f = min(fq(r), NFP - 1) / NFPF;
    pfi[r] = a.finfo[ec * NFACE + f];
    pnb[r] = a.fnbr[ec * NFACE + f];
  }
  for (int i = threadIdx.x; i < O::SIZE; i += blockDim.x) s1[i] = a.oned[i];
  double u[NF];
  {
    double l[NF];
#pragma unroll
    for (int k = 0; k < NF; k++) {
      u[k] = a.U[(ec * NF + k) * NS + tc];
      l[k] = a.nu[(ec * NF + k) * NS + tc];
    }
    if (hasS)
#pragma unroll
      for (int k = 0; k < NF; k++) {
        sU[k * NSP + tP] = u[k];
        sL[k * NSP + tP] = l[k];
      }
  }
  const GeoAddr<D, P> ga(a.affine, tc);
  // face records of round r, read where they are used (cached after the first)
  auto normal = [&](int r, double *n) {
    const int qc = min(fq(r), NFP - 1);
#pragma unroll
    for (int c = 0; c < D; c++) n[c] = a.fgeo[ga.fg(ec, c, qc)];
  };
  auto other = [&](int r, const double *x, double *v) {  // the neighbour's face data
    const int qc = min(fq(r), NFP - 1);
    const bool bnd = BND && pfi[r] >= FINFO_BOUNDARY;
    const size_t o = bnd ? ec * NF * NFP + qc : (size_t)pnb[r] * NF * NFP + neighbourFpt<D, P>(qc, pfi[r]);
#pragma unroll
    for (int k = 0; k < NF; k++) v[k] = x[o + k * NFP];
  };
  auto ownTrace = [&](int r, double *uo) {  // (matrix cores: all lanes)
    if constexpr (MG) {
      double v[NF];
      mfmaFaceRound<NF, NSP, double>(s1, sU, t, u, r, v);
#pragma unroll
      for (int k = 0; k < NF; k++) uo[k] = v[k];
    } else {
      int base, stride, side, dn;
      fptLine<D, P>(min(fq(r), NFP - 1), base, stride, side, dn);
      const int lb = padIdx<P>(base), ls = padStride<P>(stride);
      const double *l1 = s1 + (side ? O::LR : O::LL);
#pragma unroll
      for (int k = 0; k < NF; k++) {
        double acc = 0;
#pragma unroll
        for (int m = 0; m < P1; m++) acc += l1[m] * sU[k * NSP + lb + m * ls];
        uo[k] = acc;
      }
    }
  };
  __syncthreads();
  // (0) lamJ, the common flux's cotangent and the LDG jump at every flux point
  double gc[NQ][NF];
#pragma unroll
  for (int r = 0; r < NQ; r++) {
    const int q = fq(r);
    double uo[NF], un[NF], n[D], lj[NF], pA[NF], dUc[NF];
    other(r, a.Uf, un);
    other(r, a.A, pA);
    normal(r, n);
    const double dA = a.fgeo[ga.fg(ec, D, min(q, NFP - 1))];
    if (MG && act) ownTrace(r, uo);
    if (act && q < NFP) {
      if (!MG) ownTrace(r, uo);
      const int fi = pfi[r];
      const bool bnd = BND && fi >= FINFO_BOUNDARY;
      const bool right = !bnd && ((fi >> 5) & 1);
      lamJAt<D, P, NF>(s1, sL, q, lj);
      if (bnd) boundaryState<D, NF, double>(a.ph, fi - FINFO_BOUNDARY, uo, n, un);
      ldgJump<D, NF, double>(a.ph, bnd, right, uo, un, n, dUc);
#pragma unroll
      for (int k = 0; k < NF; k++) {
        gc[r][k] = bnd ? lj[k] * dA : lj[k] * (right ? -dA : dA) + pA[k];
        sJ[k * NFP + q] = lj[k];
        sC[k * NFP + q] = dUc[k];
      }
    }
  }
  elementSync<TPE>();
  // (1) the corrected gradient
  double g[D][NF];
  double pJ[D * D];
#pragma unroll
  for (int c = 0; c < D * D; c++) pJ[c] = a.JG[ga.jg(ec, c)];
  const double pdet = a.detJ[ga.det(ec)];
  const int sk = D == 3 ? tc / (P1 * P1) : 0, sj = (tc / P1) % P1, si = tc % P1;
  if (MG ? act : hasS) {
    if constexpr (MG) {
      mfmaGradient<NF, NSP, double>(s1, sU, u, sC, t, pJ, pdet, g);
    } else {
      correctedGradient<D, P, NF, double>(s1, sU, sC, t, si, sj, sk, pJ, pdet, g);
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int k = 0; k < NF; k++) sQ[(d * NF + k) * NSP + tP] = g[d][k];
    }
  }
  elementSync<TPE>();
  // (2) the common flux pulled back at every flux point: to the state trace
  // (sC) and to the gradient traces, kept until every gradient trace has been
  // read (not the matrix-core variant, which takes them from registers)
  double lgf[MG ? 1 : NQ][D][NF];
#pragma unroll
  for (int r = 0; r < NQ; r++) {
    const int q = fq(r);
    double gf[D][NF], uo[NF], un[NF], n[D], lO[NF];
    other(r, a.Uf, un);
    normal(r, n);
    if constexpr (MG) {
      if (act) {
#pragma unroll
        for (int d = 0; d < D; d++) mfmaFaceRoundReg<NF, double>(s1, t, g[d], r, gf[d]);
        ownTrace(r, uo);
      }
    }
    if (!act || q >= NFP) continue;
    if constexpr (!MG) {
      int base, stride, side, dn;
      fptLine<D, P>(q, base, stride, side, dn);
      const int lb = padIdx<P>(base), ls = padStride<P>(stride);
      const double *l1 = s1 + (side ? O::LR : O::LL);
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int k = 0; k < NF; k++) {
          double acc = 0;
#pragma unroll
          for (int m = 0; m < P1; m++) acc += l1[m] * sQ[(d * NF + k) * NSP + lb + m * ls];
          gf[d][k] = acc;
        }
      ownTrace(r, uo);
    }
    const int fi = pfi[r], bc = fi - FINFO_BOUNDARY;
    const bool bnd = BND && fi >= FINFO_BOUNDARY;
    const bool right = !bnd && ((fi >> 5) & 1);
    double(&lg)[D][NF] = lgf[MG ? 0 : r];
    if (bnd) {
      double lN[NF];
      boundaryState<D, NF, double>(a.ph, bc, uo, n, un);
      commonFluxVjp<D, NF>(a.ph, false, uo, un, n, gc[r], lO, lN);
      viscousFaceVjp<D, NF>(a.ph, true, bc, false, uo, un, gf, n, gc[r], lO, lN, lg);
      ghostVjp<D, NF>(a.ph, bc, uo, n, lN, lO);
    } else {
      bool roe = false;
      if constexpr (D == 2 && NF > 1)
        if (a.ph.riemannType == 1) {
          roe = true;
          roeFluxVjp(a.ph, right, uo, un, n, gc[r], lO);
        }
      if (!roe) commonFluxVjp<D, NF>(a.ph, right, uo, un, n, gc[r], lO, nullptr);
      viscousFaceVjp<D, NF>(a.ph, false, 0, right, uo, un, gf, n, gc[r], lO, nullptr, lg);
    }
#pragma unroll
    for (int k = 0; k < NF; k++) {
      sC[k * NFP + q] = lO[k];
      if constexpr (MG)
#pragma unroll
        for (int d = 0; d < D; d++) sQ[(d * NF + k) * NFP + q] = lg[d][k];
    }
  }
  if constexpr (!MG) {
    if (hasS) {
      // read back instead of kept in registers through (2)
#pragma unroll
      for (int k = 0; k < NF; k++) {
        u[k] = sU[k * NSP + tP];
#pragma unroll
        for (int d = 0; d < D; d++) g[d][k] = sQ[(d * NF + k) * NSP + tP];
      }
    }
    elementSync<TPE>();
#pragma unroll
    for (int r = 0; r < NQ; r++)
      if (act && fq(r) < NFP)
#pragma unroll
        for (int d = 0; d < D; d++)
#pragma unroll
          for (int k = 0; k < NF; k++) sQ[(d * NF + k) * NFP + fq(r)] = lgf[r][d][k];
  }
  elementSync<TPE>();
  // (3) the point fluxes pulled back, the transposed traces, and the
  // reference gradient's cotangent lQ
  double w[NF], lQ[D][NF];
  if (hasS) {
    double lg[D][NF];
    {
      double lF[D][NF];
      pointFluxCotangent<D, P, NF>(s1, sL, sJ, t, pJ, lF);
      inviscidFluxVjp<D, NF>(a.ph, u, lF, w);
      viscousFluxVjp<D, NF>(a.ph, u, g, lF, w, lg);
    }
    int cq[NFACE], cside[NFACE], cax[NFACE];
    corrEntries<D, P>(t, cq, cside, cax);
#pragma unroll
    for (int f = 0; f < NFACE; f++) {
      const double c = s1[(cside[f] ? O::LR : O::LL) + cax[f]];
#pragma unroll
      for (int k = 0; k < NF; k++) {
        w[k] += c * sC[k * NFP + cq[f]];
#pragma unroll
        for (int d = 0; d < D; d++) lg[d][k] += c * sQ[(d * NF + k) * NFP + cq[f]];
      }
    }
    // Q = JGinv^T Qref / detJ, transposed
    const double invDet = recip(pdet);
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
      for (int k = 0; k < NF; k++) {
        double acc = 0;
#pragma unroll
        for (int d1 = 0; d1 < D; d1++) acc += pJ[d * D + d1] * lg[d1][k];
        lQ[d][k] = invDet * acc;
      }
  }
  elementSync<TPE>();
  if (hasS)
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
      for (int k = 0; k < NF; k++) sLQ[(d * NF + k) * NSP + tP] = lQ[d][k];
  elementSync<TPE>();
  // (4) Qref = Dm U + lift(u^ - u): to the state along the lines, and the
  // jumps' cotangents
  if (hasS) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int id = (d == 0) ? si : (d == 1) ? sj : sk;
#pragma unroll
      for (int k = 0; k < NF; k++) {
        double acc = 0;
#pragma unroll
        for (int m = 0; m < P1; m++) {
          const int sp = (d == 0)   ? m + P1 * (sj + P1 * sk)
                         : (d == 1) ? si + P1 * (m + P1 * sk)
                                    : si + P1 * (sj + P1 * m);
          acc += s1[O::DM + m * P1 + id] * sLQ[(d * NF + k) * NSP + padIdx<P>(sp)];
        }
        w[k] += acc;
      }
    }
#pragma unroll
    for (int k = 0; k < NF; k++) a.out[((size_t)e * NF + k) * NS + t] = w[k];
  }
  if (act)
    for (int q = t; q < NFP; q += TPE) {
      int base, stride, side, dn;
      fptLine<D, P>(q, base, stride, side, dn);
      const int lb = padIdx<P>(base), ls = padStride<P>(stride);
      const double *gq = s1 + (side ? O::GR : O::GL);
      const double sg = side ? 1.0 : -1.0;
#pragma unroll
      for (int k = 0; k < NF; k++) {
        double acc = 0;
#pragma unroll
        for (int m = 0; m < P1; m++) acc += gq[m] * sLQ[(dn * NF + k) * NSP + lb + m * ls];
        a.B[((size_t)e * NF + k) * NFP + q] = sg * acc;
      }
    }
}

// The common solution's pull-back: u^ = (uL+uR)/2 - pen (uL-uR) inside
// (either side's jump u^ - u uses it), (u + ghost(u))/2 on boundaries.  Adds
// it to k_vjp_visc's part and ends the stage.
template <int D, int P, int NF, bool BND>
__global__ __launch_bounds__((ElemGeo<D, P>::NTH)) void k_vjp_ldg(VjpArgs a) {
  using G = ElemGeo<D, P>;
  using O = OneD<P>;
  constexpr int NS = G::NS, NSP = G::NSP, NFP = G::NFP, NFPF = G::NFPF, P1 = G::P1, TPE = G::TPE, EPB = G::EPB;
  constexpr int NFACE = G::NFACE;
  __shared__ double sX[EPB][NF][NSP];  // the state (boundary meshes), then the next nu
  __shared__ double sUo[EPB][NF][NFP];
  __shared__ double s1[O::SIZE];
  const int slot = threadIdx.x / TPE, t = threadIdx.x - slot * TPE;
  const int e = vjpBlock() * EPB + slot;
  const bool act = e < a.nEles;
  const bool hasS = act && t < NS;
  const size_t ec = (size_t)(act ? e : a.nEles - 1);
  const GeoAddr<D, P> ga(a.affine, 0);
  for (int i = threadIdx.x; i < O::SIZE; i += blockDim.x) s1[i] = a.oned[i];
  double w[NF];
  if (hasS)
#pragma unroll
    for (int k = 0; k < NF; k++) {
      w[k] = a.out[(ec * NF + k) * NS + t];
      if (BND) sX[slot][k][padIdx<P>(t)] = a.U[(ec * NF + k) * NS + t];
    }
  __syncthreads();
  if (act)
    for (int q = t; q < NFP; q += TPE) {
      const int fi = a.finfo[ec * NFACE + q / NFPF];
      const bool bnd = BND && fi >= FINFO_BOUNDARY;
      double n[D], bo[NF], lO[NF];
#pragma unroll
      for (int c = 0; c < D; c++) n[c] = a.fgeo[ga.fg(ec, c, q)];
#pragma unroll
      for (int k = 0; k < NF; k++) bo[k] = a.B[(ec * NF + k) * NFP + q];
      if (bnd) {
        int base, stride, side, dn;
        fptLine<D, P>(q, base, stride, side, dn);
        const int lb = padIdx<P>(base), ls = padStride<P>(stride);
        const double *l1 = s1 + (side ? O::LR : O::LL);
        double uo[NF], hb[NF];
#pragma unroll
        for (int k = 0; k < NF; k++) {
          double acc = 0;
#pragma unroll
          for (int m = 0; m < P1; m++) acc += l1[m] * sX[slot][k][lb + m * ls];
          uo[k] = acc;
          hb[k] = 0.5 * bo[k];
          lO[k] = -hb[k];
        }
        ghostVjp<D, NF>(a.ph, fi - FINFO_BOUNDARY, uo, n, hb, lO);
      } else {
        const size_t o = (size_t)a.fnbr[ec * NFACE + q / NFPF] * NF * NFP + neighbourFpt<D, P>(q, fi);
        const double pen = ldgPenalty<D, double>(a.ph, n);
        const double coef = ((fi >> 5) & 1) ? 0.5 + pen : 0.5 - pen;
#pragma unroll
        for (int k = 0; k < NF; k++) lO[k] = coef * (bo[k] + a.B[o + k * NFP]) - bo[k];
      }
#pragma unroll
      for (int k = 0; k < NF; k++) sUo[slot][k][q] = lO[k];
    }
  elementSync<TPE>();
  if (hasS) {
    int cq[NFACE], cside[NFACE], cax[NFACE];
    corrEntries<D, P>(t, cq, cside, cax);
#pragma unroll
    for (int f = 0; f < NFACE; f++) {
      const double c = s1[(cside[f] ? O::LR : O::LL) + cax[f]];
#pragma unroll
      for (int k = 0; k < NF; k++) w[k] += c * sUo[slot][k][cq[f]];
    }
  }
  vjpTail<D, P, NF>(a, s1, &sX[slot][0][0], e, t, act, w);
}

// gradient of the kinetic energy sum_e sum_s w_s detJ |m|^2 / (2 rho) with
// respect to U: (-|m|^2 / (2 rho^2), m / rho, 0) * w_s detJ
template <int D>
__global__ void k_ke_grad(const double *__restrict__ U, const double *__restrict__ detJ,
                          const double *__restrict__ wts, int NS, long nPts, double *__restrict__ out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nPts) return;
  const long e = i / NS;
  const int s = (int)(i % NS);
  const double *Ue = U + (size_t)e * (D + 2) * NS;
  double *Oe = out + (size_t)e * (D + 2) * NS;
  const double w = wts[s] * detJ[i];
  const double rho = Ue[s];
  double m2 = 0;
  for (int d = 0; d < D; d++) m2 += Ue[(d + 1) * NS + s] * Ue[(d + 1) * NS + s];
  Oe[s] = -0.5 * m2 / (rho * rho) * w;
  for (int d = 0; d < D; d++) Oe[(d + 1) * NS + s] = Ue[(d + 1) * NS + s] / rho * w;
  Oe[(D + 1) * NS + s] = 0.0;
}

}  // namespace frdev

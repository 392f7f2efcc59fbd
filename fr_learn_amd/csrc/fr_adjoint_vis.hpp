// fr_adjoint_vis.hpp -- launches of the viscous (LDG) adjoint of one RK stage:
// k_vjp_visc and k_vjp_ldg.  Instantiated per (nDims, nFields) in
// fr_adjoint_v2.hip, fr_adjoint_v3.hip and fr_adjoint_v3ad.hip, which compile
// in parallel.
#pragma once

#include "fr_adjoint.hpp"
#include "fr_ctx.hpp"

namespace frimpl {

template <int D, int NF>
hipError_t vjpViscousLaunch(fr_ctx *c, const frdev::VjpArgs &a, bool bnd);

template <int D, int P, int NF>
hipError_t vjpViscousLaunchP(fr_ctx *c, const frdev::VjpArgs &a, bool bnd) {
  using G = frdev::ElemGeo<D, P>;
  using V = frdev::VjpTile<D, P>;
  auto blocks = [&](int epb) { return dim3((unsigned)(((c->nE + epb - 1) / epb + 7) / 8 * 8)); };
  if (bnd) {
    hipLaunchKernelGGL((frdev::k_vjp_visc<D, P, NF, true>), blocks(V::EPB), dim3(V::NTH), 0, c->stream, a);
    hipLaunchKernelGGL((frdev::k_vjp_ldg<D, P, NF, true>), blocks(G::EPB), dim3(G::NTH), 0, c->stream, a);
  } else {
    hipLaunchKernelGGL((frdev::k_vjp_visc<D, P, NF, false>), blocks(V::EPB), dim3(V::NTH), 0, c->stream, a);
    hipLaunchKernelGGL((frdev::k_vjp_ldg<D, P, NF, false>), blocks(G::EPB), dim3(G::NTH), 0, c->stream, a);
  }
  return hipGetLastError();
}

#define FR_VJP_VIS_INSTANCE(DD, NFF)                                                                    \
  template <>                                                                                           \
  hipError_t vjpViscousLaunch<DD, NFF>(fr_ctx * c, const frdev::VjpArgs &a, bool bnd) {                     \
    switch (c->P) {                                                                                     \
      case 1: return vjpViscousLaunchP<DD, 1, NFF>(c, a, bnd);                               \
      case 2: return vjpViscousLaunchP<DD, 2, NFF>(c, a, bnd);                               \
      case 3: return vjpViscousLaunchP<DD, 3, NFF>(c, a, bnd);                               \
      case 4: return vjpViscousLaunchP<DD, 4, NFF>(c, a, bnd);                               \
      case 5: return vjpViscousLaunchP<DD, 5, NFF>(c, a, bnd);                               \
      default: return hipErrorInvalidValue;                                                             \
    }                                                                                                   \
  }

template <>
hipError_t vjpViscousLaunch<2, 4>(fr_ctx *c, const frdev::VjpArgs &a, bool bnd);
template <>
hipError_t vjpViscousLaunch<2, 1>(fr_ctx *c, const frdev::VjpArgs &a, bool bnd);
template <>
hipError_t vjpViscousLaunch<3, 5>(fr_ctx *c, const frdev::VjpArgs &a, bool bnd);
template <>
hipError_t vjpViscousLaunch<3, 1>(fr_ctx *c, const frdev::VjpArgs &a, bool bnd);

}  // namespace frimpl

// fr_stage_impl.hpp -- launches of the stage kernel (on the viscous path, of its
// two kernels); instantiated per precision in
// fr_stage64.hip and fr_stage32.hip so that the two compile in parallel.
#pragma once

#include "fr_ctx.hpp"
#include "fr_viscous.hpp"

namespace frimpl {

// Launch of the stage kernel variant for `mode` with arguments `a`, quads (DD = 2) or hexes
// (DD = 3); the four (precision, DD) instances compile in their own
// translation units (fr_stage{64,32}_{2,3}d.hip).
template <typename T, int DD>
int launchStageArgsD(fr_ctx *c, const frdev::StageArgs<T> &a, int mode) {
  const bool bnd = c->conn.nIntFaces < (int)c->conn.faces.size();
  const bool vis = c->cfg.viscous != 0;
  hipError_t err = hipSuccess;
  bool ok = dispatch(c->D, c->P, c->NF, [&](auto Dc, auto Pc, auto NFc) {
    constexpr int D = decltype(Dc)::value, P = decltype(Pc)::value, NF = decltype(NFc)::value;
    if constexpr (D != DD) {
      err = hipErrorInvalidValue;
      return;
    } else {
    using G = frdev::ElemGeo<D, P>;
    // grids padded to a multiple of the 8 XCDs (the kernels remap block ids)
    if (vis) {
      const unsigned nb = (unsigned)(((c->nE + G::EPB - 1) / G::EPB + 7) / 8 * 8);
      {
        TimeScope ts(c, 3);
        if (bnd) hipLaunchKernelGGL((frdev::k_visc_flux<D, P, NF, T, true>), dim3(nb), dim3(G::NTH), 0, c->stream, a,
                                    (T *)nullptr, (T *)nullptr);
        else hipLaunchKernelGGL((frdev::k_visc_flux<D, P, NF, T, false>), dim3(nb), dim3(G::NTH), 0, c->stream, a,
                                (T *)nullptr, (T *)nullptr);
      }
      if ((err = hipGetLastError()) != hipSuccess) return;
      TimeScope ts(c, 0);
      auto launch = [&](auto Bc, auto Fc) {
        hipLaunchKernelGGL((frdev::k_visc_update<D, P, NF, T, decltype(Bc)::value, decltype(Fc)::value>), dim3(nb),
                           dim3(G::NTH), 0, c->stream, a);
      };
      if (bnd && mode >= 2) launch(std::true_type{}, std::true_type{});
      else if (bnd) launch(std::true_type{}, std::false_type{});
      else if (mode >= 2) launch(std::false_type{}, std::true_type{});
      else launch(std::false_type{}, std::false_type{});
    } else {
      TimeScope ts(c, 0);
      // the inviscid variants: boundary faces or not, final stage or not,
      // geometry from the stored arrays or from the nodal map (GM)
      auto launchL = [&](auto Bc, auto Fc, auto Gc, auto Lc) {
        constexpr int L = decltype(Lc)::value;
        using GL = frdev::ElemGeo<D, P, L>;
        const unsigned n = (unsigned)(((c->nE + GL::EPB - 1) / GL::EPB + 7) / 8 * 8);
        hipLaunchKernelGGL((frdev::k_stage<D, P, NF, T, decltype(Bc)::value, decltype(Fc)::value,
                                           decltype(Gc)::value, L>),
                           dim3(n), dim3(GL::NTH), 0, c->stream, a);
      };
      auto launch = [&](auto Bc, auto Fc, auto Gc) {
        if constexpr (frdev::packedOrder(D, P)) {
          if (frdev::stageTile(D, P, c->nE)) {
            launchL(Bc, Fc, Gc, std::integral_constant<int, 1>{});
            return;
          }
        }
        launchL(Bc, Fc, Gc, std::integral_constant<int, 0>{});
      };
      auto byGeo = [&](auto Bc, auto Fc) {
        if (a.nodal == 1) launch(Bc, Fc, std::integral_constant<int, 1>{});
        else if (a.nodal == 2) launch(Bc, Fc, std::integral_constant<int, 2>{});
        else launch(Bc, Fc, std::integral_constant<int, 0>{});
      };
      auto byFin = [&](auto Bc) {
        if (mode >= 2) byGeo(Bc, std::true_type{});
        else byGeo(Bc, std::false_type{});
      };
      if (bnd) byFin(std::true_type{});
      else byFin(std::false_type{});
    }
    err = hipGetLastError();
    }
  });
  if (!ok) return fail(FR_EINVAL, "no kernel instance for this (nDims, order, nFields)");
  if (err != hipSuccess) return fail(FR_EHIP, std::string("stage launch: ") + hipGetErrorString(err));
  return 0;
}

template <typename T>
int launchStageArgs(fr_ctx *c, const frdev::StageArgs<T> &a, int mode) {
  if (c->tri) return launchTriStage<T>(c, a, mode);
  return c->D == 3 ? launchStageArgsD<T, 3>(c, a, mode) : launchStageArgsD<T, 2>(c, a, mode);
}

}  // namespace frimpl

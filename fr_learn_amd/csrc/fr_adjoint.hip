// fr_adjoint.hip -- launches of the adjoint kernels (fr_adjoint.hpp).
#include "fr_adjoint.hpp"
#include "fr_adjoint_vis.hpp"
#include "fr_ctx.hpp"

namespace frimpl {

frdev::VjpArgs vjpArgs(const fr_ctx *c, const double *Us, const double *tr, const double *nu, const double *A) {
  frdev::VjpArgs a{};
  const bool aff = c->geoActive() == 1;
  a.U = Us;
  a.nu = nu;
  a.Uf = tr;
  a.A = A;
  a.JG = aff ? c->JGc64 : c->JG64;
  a.fgeo = aff ? c->fgeoc64 : c->fgeo64;
  a.detJ = aff ? c->detJc : c->detJ;
  a.fnbr = c->fnbr;
  a.finfo = c->finfo;
  a.oned = c->oned64;
  a.ph = c->ph;
  a.nEles = c->nE;
  a.affine = aff ? 1 : 0;
  a.out = c->adjW;
  a.B = c->adjB;
  a.dtE = dtSource(c).first;
  a.dtStride = dtSource(c).second;
  return a;
}

int vjpSeed(fr_ctx *c, const frdev::VjpArgs &a) {
  hipError_t err = hipSuccess;
  bool ok = dispatch(c->D, c->P, c->NF, [&](auto Dc, auto Pc, auto NFc) {
    constexpr int D = decltype(Dc)::value, P = decltype(Pc)::value, NF = decltype(NFc)::value;
    using G = frdev::ElemGeo<D, P>;
    hipLaunchKernelGGL((frdev::k_vjp_seed<D, P, NF>), dim3((unsigned)((c->nE + G::EPB - 1) / G::EPB)), dim3(G::NTH), 0,
                       c->stream, a);
    err = hipGetLastError();
  });
  if (!ok) return fail(FR_EINVAL, "no kernel instance for this (nDims, order, nFields)");
  if (err != hipSuccess) return fail(FR_EHIP, std::string("adjoint launch: ") + hipGetErrorString(err));
  return 0;
}

int vjpStage(fr_ctx *c, const frdev::VjpArgs &a) {
  const bool bnd = c->conn.nIntFaces < (int)c->conn.faces.size();
  hipError_t err = hipSuccess;
  if (c->cfg.viscous) {
    if (c->D == 2)
      err = (c->NF == 1) ? vjpViscousLaunch<2, 1>(c, a, bnd) : vjpViscousLaunch<2, 4>(c, a, bnd);
    else
      err = (c->NF == 1) ? vjpViscousLaunch<3, 1>(c, a, bnd) : vjpViscousLaunch<3, 5>(c, a, bnd);
    if (err != hipSuccess) return fail(FR_EHIP, std::string("viscous adjoint launch: ") + hipGetErrorString(err));
    return 0;
  }
  bool ok = dispatch(c->D, c->P, c->NF, [&](auto Dc, auto Pc, auto NFc) {
    constexpr int D = decltype(Dc)::value, P = decltype(Pc)::value, NF = decltype(NFc)::value;
    using G = frdev::ElemGeo<D, P>;
    const unsigned nb = (unsigned)(((c->nE + G::EPB - 1) / G::EPB + 7) / 8 * 8);
    auto launch = [&](auto Bc, auto Rc) {
      hipLaunchKernelGGL((frdev::k_vjp_state<D, P, NF, decltype(Bc)::value, decltype(Rc)::value>), dim3(nb),
                         dim3(G::NTH), 0, c->stream, a);
    };
    if constexpr (D == 2 && NF > 1) {
      if (c->cfg.riemannType == 1) {
        if (bnd) launch(std::true_type{}, std::true_type{});
        else launch(std::false_type{}, std::true_type{});
        err = hipGetLastError();
        return;
      }
    }
    if (bnd) launch(std::true_type{}, std::false_type{});
    else launch(std::false_type{}, std::false_type{});
    err = hipGetLastError();
  });
  if (!ok) return fail(FR_EINVAL, "no kernel instance for this (nDims, order, nFields)");
  if (err != hipSuccess) return fail(FR_EHIP, std::string("adjoint launch: ") + hipGetErrorString(err));
  return 0;
}

}  // namespace frimpl

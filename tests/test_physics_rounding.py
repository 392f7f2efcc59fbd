"""Rounding of the pointwise physics (fr_learn_amd/csrc/fr_physics.hpp), the
very header compiled for the CPU.  The hardware's root and reciprocal
estimates are stood in for by functions whose error is set by the test, up to
their bounds: one ulp in single precision, 2^-22 in double.

Single precision: the Roe flux's roots are rounded correctly, the viscous flux
and the physical gradient round no worse than the reference's operations."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fr_learn_amd", "csrc")

# what the header takes from the HIP headers and the compiler
STAND_IN = r"""
#pragma once
#include <cmath>
#define __device__
#define __host__
#define __forceinline__ inline
using std::fabs; using std::fma; using std::fmax; using std::fmin; using std::pow; using std::sqrt;
extern int gOff;  // -1, 0, 1: the estimates' error in units of its bound
inline float estimate(float x) { return gOff ? std::nextafter(x, gOff > 0 ? INFINITY : 0.0f) : x; }
inline float __builtin_amdgcn_sqrtf(float x) { return estimate(std::sqrt(x)); }
inline float __builtin_amdgcn_rcpf(float x) { return estimate(1.0f / x); }
inline double __builtin_amdgcn_rsq(double x) { return 1.0 / std::sqrt(x) * (1.0 + gOff * 0x1p-22); }
inline double __builtin_amdgcn_rcp(double x) { return 1.0 / x * (1.0 + gOff * 0x1p-22); }
"""

MAIN = r"""
#include "fr_physics.hpp"
int gOff = 0;
using namespace frdev;
static Phys phys() {
  Phys ph{};
  ph.gamma = 1.4; ph.mu_inf = 0.05; ph.prandtl = 0.72; ph.viscFix = ph.fixVis = 1;
  return ph;
}
template <int D>
static void viscous(int n, const float *U, const float *g, float *F) {
  constexpr int K = D + 2;
  for (int i = 0; i < n; i++)
    viscousFlux<D, K, float>(phys(), U + i * K, (const float(*)[K])(g + i * D * K), (float(*)[K])(F + i * D * K));
}
extern "C" {
void offset(int o) { gOff = o; }
void roots32(const float *x, float *y, int n) { for (int i = 0; i < n; i++) y[i] = rootOf(x[i]); }
void viscous32(int D, int n, const float *U, const float *g, float *F) {
  if (D == 3) viscous<3>(n, U, g, F);
  else viscous<2>(n, U, g, F);
}
void gradient32(const float *gr, const float *J, float det, float *g) {
  physicalGradient<3, 5, float>((const float(*)[5])gr, J, det, (float(*)[5])g);
}
void roe64(const double *UL, const double *UR, const double *n, double *F) { roe2d<double>(phys(), UL, UR, n, F); }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("physics")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(STAND_IN)
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-w", "-I", str(d), "-I", CSRC,
                    str(d / "main.cpp"), "-o", str(d / "physics.so")], check=True)
    return ctypes.CDLL(str(d / "physics.so"))


def _p(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def test_single_precision_roots_are_rounded_correctly(lib):
    x = np.concatenate([10.0 ** np.random.default_rng(0).uniform(-30, 30, 4000), [0.0, 1.0, np.inf]]).astype(np.float32)
    y = np.empty_like(x)
    for o in (-1, 0, 1):
        lib.offset(o)
        lib.roots32(_p(x), _p(y), len(x))
        assert np.array_equal(y, np.sqrt(x))


def _reference_viscous_flux(U, g, cfg, t):
    """The reference's viscous flux (src/flux.cpp:90-226, with the physical
    stresses) operation by operation in type t: U [n][K], g [n][D][K]."""
    U, g = U.astype(t), g.astype(t)
    D = g.shape[1]
    mu, pr, gam = (t(cfg[k]) for k in ("mu_inf", "prandtl", "gamma"))
    rho = U[:, 0]
    v = [U[:, 1 + c] / rho for c in range(D)]
    q = v[0] * v[0] + v[1] * v[1] + (v[2] * v[2] if D == 3 else t(0))
    e = U[:, D + 1] / rho - t(0.5) * q
    dv = [[(g[:, d, 1 + c] - g[:, d, 0] * v[c]) / rho for c in range(D)] for d in range(D)]
    F = np.zeros(g.shape, t)
    diag = sum(dv[d][d] for d in range(D)) / t(3)
    tau = [[t(2) * mu * (dv[d][d] - diag) if c == d else mu * (dv[d][c] + dv[c][d]) for c in range(D)]
           for d in range(D)]
    for d in range(D):
        dK = t(0.5) * q * g[:, d, 0] + rho * sum(v[c] * dv[d][c] for c in range(D))
        de = (g[:, d, D + 1] - dK - g[:, d, 0] * e) / rho
        for c in range(D):
            F[:, d, 1 + c] = -tau[d][c]
        F[:, d, D + 1] = -(sum(v[c] * tau[d][c] for c in range(D)) + mu / pr * gam * de)
    return F


@pytest.mark.parametrize("jump", [0.0, 0.1, 1.0])
@pytest.mark.parametrize("mach", [0.1, 2.0])
@pytest.mark.parametrize("D", [2, 3])
def test_viscous_flux_rounds_no_worse_than_the_reference(lib, D, mach, jump):
    """Single precision, random states of order one at two Mach numbers, with
    density gradients of relative size jump: the flux's r.m.s. error is at
    most that of the reference's own operations in single precision.  100000
    points each: the ratio of two such errors scatters by some 0.3 %."""
    n, cfg = 100000, dict(gamma=1.4, mu_inf=0.05, prandtl=0.72)
    r = np.random.default_rng(5)
    rho = np.maximum(0.2, 1.0 + 0.3 * jump * r.standard_normal(n))
    v, drho = r.standard_normal((n, D)), jump * r.standard_normal((n, D))
    dv, dp = r.standard_normal((n, D, D)), r.standard_normal((n, D))
    U = np.concatenate([rho[:, None], rho[:, None] * v, (1 / (0.4 * 1.4 * mach ** 2) + 0.5 * rho * (v * v).sum(1))[:, None]], 1)
    g = np.zeros((n, D, D + 2))
    g[:, :, 0] = drho
    g[:, :, 1:-1] = drho[:, :, None] * v[:, None, :] + rho[:, None, None] * dv
    g[:, :, -1] = dp / 0.4 + 0.5 * drho * (v * v).sum(1)[:, None] + rho[:, None] * (dv * v[:, None, :]).sum(2)
    U, g = U.astype(np.float32), g.astype(np.float32)
    exact = _reference_viscous_flux(U, g, cfg, np.float64)
    ref = _reference_viscous_flux(U, g, cfg, np.float32)
    for o in (-1, 0, 1):
        lib.offset(o)
        F = np.zeros(g.shape, np.float32)
        lib.viscous32(D, n, _p(U), _p(g), _p(F))
        for part in (slice(1, D + 1), slice(D + 1, D + 2)):  # momentum, energy
            err = [np.sqrt(((A[..., part] - exact[..., part]) ** 2).mean()) for A in (F, ref)]
            print(f"D={D} M={mach} jump={jump} error {err[0]:.3e}, the reference's {err[1]:.3e}")
            assert err[0] <= 1.01 * err[1]


def test_physical_gradient_divides_after_the_sum(lib):
    """Bit for bit (1 / detJ) times the sum of the metric products."""
    r = np.random.default_rng(1)
    lib.gradient32.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_float, ctypes.c_void_p]
    for _ in range(2000):
        gr, J = r.standard_normal((3, 5)).astype(np.float32), r.standard_normal((3, 3)).astype(np.float32)
        det = np.float32(r.uniform(0.1, 10.0))
        want = np.stack([np.float32(1) / det * (gr[0] * J[0, d] + gr[1] * J[1, d] + gr[2] * J[2, d]) for d in range(3)])
        for o in (-1, 0, 1):
            lib.offset(o)
            g = np.zeros((3, 5), np.float32)
            lib.gradient32(_p(gr), _p(J), float(det), _p(g))
            assert np.array_equal(g, want)


def test_roe_flux_of_an_infinite_state_is_nan(lib):
    """rootOf(inf) is NaN in double precision; so is every component of the
    flux of a state that leads to it, whatever the root."""
    n = np.array([0.6, 0.8])
    fine = np.array([1.0, 0.3, 0.1, 2.5])
    lib.offset(0)
    for bad in ([1.0, 0.3, 0.1, np.inf], [np.inf, 0.3, 0.1, 2.5], [1.0, np.inf, 0.1, 2.5]):
        for UL, UR in ((np.array(bad), fine), (fine, np.array(bad))):
            F = np.zeros(4)
            lib.roe64(_p(UL), _p(UR), _p(n), _p(F))
            assert np.isnan(F).all()

"""Rounding of the pointwise physics (fr_learn_amd/csrc/fr_physics.hpp), the
very header compiled for the CPU.  The hardware's root and reciprocal
estimates are stood in for by functions whose error is set by the test, up to
their bounds: one ulp in single precision, 2^-22 in double.

Single precision: the Roe flux's roots are rounded correctly."""
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
extern "C" {
void offset(int o) { gOff = o; }
void roots32(const float *x, float *y, int n) { for (int i = 0; i < n; i++) y[i] = rootOf(x[i]); }
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

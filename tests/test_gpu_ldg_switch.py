"""The LDG direction switch (the sign of n.(1, 1, sqrt 2), n.(1, 1) in 2D) on
faces where it is zero but for rounding: an affine box turned 45 degrees.  The
two elements of a face weight their viscous fluxes by it, and the weights add
to one only if both take the same sign, whatever it is."""
import numpy as np
import pytest

from fr_learn_amd import Solver, mesh

from helpers import perturbed_state
from test_gpu_viscous import ns_cfg

pytestmark = pytest.mark.gpu

SIDE = 0.1


def _turned_box(D, n):
    m = mesh.box(D, (n,) * D, (0.0,) * D, (n * SIDE,) * D, periodic=[True] * D, rotate=True, shuffle=True, seed=2)
    c, s = np.cos(np.pi / 4), np.sin(np.pi / 4)
    cell = np.floor(m.element_nodes().mean(axis=1)[:, :D] / SIDE).astype(int)
    m.xv[:, :2] = m.xv[:, :2] @ np.array([[c, s], [-s, c]])
    return m, cell


def _smooth(x):
    """Conserved fields of degree 1 in each coordinate, which every order holds
    exactly: traces and gradients agree across faces but for rounding."""
    D = x.shape[-1]
    lin = [1.0 + sum((0.3 + 0.1 * k - 0.17 * d) * x[..., d] for d in range(D)) for k in range(D + 2)]
    return np.stack([lin[0]] + [0.3 * f for f in lin[1:-1]] + [4.0 * lin[-1]], axis=-1)


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-9), ("fp32", 0.05)])
@pytest.mark.parametrize("geometry", [0, 1])
@pytest.mark.parametrize("D,P,n", [(3, 2, 8), (3, 3, 7), (2, 3, 16)])
def test_weights_of_the_sides_add_to_one(D, P, n, geometry, precision, tol):
    """Where state and gradient are continuous the switch drops out of the
    common flux: the residual is that of the central flux (penFact 0).  tol: a
    jump of the gradient's rounding (some hundred ulps of U / SIDE) against
    the residual, which is of the order of the viscosity times the gradient's
    change over an element; a face's flux dropped or doubled is of order
    P^2 gradient / SIDE, above all of them."""
    m, cell = _turned_box(D, n)
    out = []
    for pen in (0.0, 0.5, -0.5):
        g = Solver(ns_cfg(D, P, penFact=pen, viscFix=1, fixVis=1), m, precision=precision)
        g.geometry_mode(geometry)
        g.set_state(_smooth(g.positions()))
        g.calc_residual(0)
        out.append(g.residual(0))
        g.close()
    # the gradients of elements on the periodic boundary see the state's jump there
    inner = ((cell >= 2) & (cell < n - 2)).all(axis=1)
    assert inner.sum() >= 3 ** D
    for R in out[1:]:
        err = np.abs(R - out[0])[:, inner].max() / np.abs(out[0][:, inner]).max()
        print(f"switch D={D} P={P} geometry={geometry} {precision} err {err:.1e}", flush=True)
        assert err <= tol


@pytest.mark.parametrize("geometry", [0, 1])
@pytest.mark.parametrize("D,P,n", [(3, 3, 4), (2, 4, 8)])
def test_vjp_takes_the_same_sign(D, P, n, geometry):
    """<lam, J v> from a central difference (error below 1e-9 |J v|: its step
    is 1e-6 of the state) against <J^T lam, v>."""
    m, _ = _turned_box(D, n)
    g = Solver(ns_cfg(D, P, penFact=0.5, viscFix=1, fixVis=1), m)
    g.geometry_mode(geometry)
    U = perturbed_state(_smooth(g.positions()), seed=P, amp=2e-2)
    rng = np.random.default_rng(17)
    lam, v = rng.standard_normal(U.shape), U * rng.standard_normal(U.shape)
    eps, R = 1e-6, []
    for s in (eps, -eps):
        g.set_state(U + s * v)
        g.calc_residual(0)
        R.append(g.residual(0))
    Jv = (R[0] - R[1]) / (2 * eps)
    g.set_state(U)
    w = g.vjp_residual(lam)
    err = abs(np.sum(lam * Jv) - np.sum(w * v)) / (np.linalg.norm(lam) * np.linalg.norm(Jv))
    print(f"vjp D={D} P={P} geometry={geometry} error {err:.1e}", flush=True)
    assert err <= 1e-7
    g.close()

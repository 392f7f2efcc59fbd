"""The Roe flux's roots (rootOf): parity near the sonic and the vacuum ends of
its range, and an unphysical state stays NaN as the library root makes it."""
import numpy as np
import pytest

from fr_learn_amd import Solver, cases, mesh
from fr_learn_amd._lib import FrError
from oracle import Oracle

from helpers import TOL_FP64, euler_cfg, perturbed_state, rel_err

pytestmark = pytest.mark.gpu


def _state(cfg, m, rho, vel, p):
    o = Oracle(cfg, m)
    U = perturbed_state(o.initialize(lambda x, c: cases.ic_uniform(x, c, rho=rho, vel=vel, p=p)), seed=8, amp=1e-3)
    return o, U


@pytest.mark.parametrize("elem", ["quad", "tri"])
@pytest.mark.parametrize("rho,vel,p", [(1.0, [0.3, 0.2], 1.0 / 1.4), (1e-6, [0.01, 0.02], 1e-8), (1e4, [3.0, 1.0], 1e7),
                                       (1.0, [3.0, 1.5], 0.4)])
def test_roe_over_magnitudes(elem, rho, vel, p):
    cfg = euler_cfg(2, 3, riemannType=1)
    m = mesh.box(2, (5, 4), (0.0, 0.0), (1.0, 1.0), perturb=0.1, seed=2)
    print(f"roe {elem} rho={rho} p={p}", flush=True)
    o, U = _state(cfg, m, rho, vel, p)
    if elem == "tri":
        # no oracle for triangles here: a uniform state has no residual, against
        # the largest flux derivative the state could have
        mt = mesh.tri_box((5, 4), (0.0, 0.0), (1.0, 1.0), perturb=0.1, seed=2)
        g = Solver(cfg, mt)
        g.initialize(lambda x, c: cases.ic_uniform(x, c, rho=rho, vel=vel, p=p))
        g.calc_residual(0)
        E = p / 0.4 + 0.5 * rho * (vel[0] ** 2 + vel[1] ** 2)
        scale = np.array([rho * 4, rho * 16 + p, rho * 16 + p, (E + p) * 4])
        assert (np.abs(g.residual(0)).max(axis=(0, 1)) <= 1e-11 * scale).all()
        return
    g = Solver(cfg, m)
    for s in (o, g):
        s.set_state(U)
        s.calc_residual(0)
    assert rel_err(g.residual(0), o.residual(0)).max() <= TOL_FP64
    o.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("elem", ["quad", "tri"])
def test_roe_unphysical_state_is_nan(elem, precision):
    cfg = euler_cfg(2, 2, riemannType=1)
    m = (mesh.tri_box if elem == "tri" else lambda *a: mesh.box(2, *a))((4, 4), (0.0, 0.0), (1.0, 1.0))
    g = Solver(cfg, m, precision=precision)
    U = g.initialize(lambda x, c: cases.ic_uniform(x, c, vel=[0.3, 0.2], p=1.0 / 1.4))
    U[:, 5, 3] = -U[:, 5, 3]  # negative pressure in one element
    g.set_state(U)
    g.calc_residual(0)
    with pytest.raises(FrError) as ei:
        g.norm_residual(2)
    assert ei.value.code == -5

"""The CFL time step is formed by groups of lanes per element (16, 32 or 64 by
the element's flux points) and reduced over the mesh in two launches: every
lane count, element counts that leave the last workgroup part empty, and meshes
of more workgroups than the final reduction has threads, against the oracle
(quads, hexes) and the closed form of a uniform state (triangles)."""
import numpy as np
import pytest

from fr_learn_amd import Solver, cases, mesh
from oracle import Oracle

from helpers import TOL_FP64, euler_cfg, perturbed_state, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtType", [1, 2])
@pytest.mark.parametrize("P,n", [(1, (3, 3)), (3, (5, 7)), (5, (7, 3)), (2, (70, 61)), (1, (3, 4, 5)), (2, (3, 3, 5)),
                                 (3, (11, 11, 11)), (4, (3, 3, 3))])
def test_cfl_sizes_vs_oracle(P, n, dtType):
    D = len(n)
    cfg = euler_cfg(D, P, timeType=4)
    m = mesh.box(D, n, (0.0,) * D, (1.0,) * D, perturb=0.15, rotate=True, shuffle=True, seed=6)
    print(f"cfl D={D} P={P} n={n} dtType={dtType}", flush=True)
    o, g = Oracle(cfg, m), Solver(cfg, m)
    vel = [0.3, 0.1, -0.05][:D]
    U = perturbed_state(o.initialize(lambda x, c: cases.ic_uniform(x, c, vel=vel, p=1.0 / 1.4)), seed=1, amp=2e-2)
    for s in (o, g):
        s.set_state(U)
        s.calc_dt(dtType, 0.3)
        s.update(2)  # the second step's dt comes from the stored wave speeds
    want = np.array([o.dt(e if dtType == 2 else -1) for e in range(o.nEles)])
    # sums of at most 150 positive terms in another order: a few 1e-15
    assert np.abs(g.dt() - want).max() <= 1e-12 * want.max()
    assert rel_err(g.get_state(), o.get_state()).max() <= TOL_FP64
    o.close()
    g.close()


@pytest.mark.parametrize("P,n", [(1, (3, 3)), (2, (101, 83)), (3, (61, 47)), (4, (7, 5)), (5, (51, 43))])
def test_cfl_triangles_uniform_state(P, n):
    cfg = euler_cfg(2, P)
    m = mesh.tri_box(n, (0.0, 0.0), (1.0, 2.0), perturb=0.1, seed=4)
    print(f"cfl triangles P={P} n={n}", flush=True)
    g = Solver(cfg, m)
    g.initialize(lambda x, c: cases.ic_uniform(x, c, vel=[0.3, 0.2], p=1.0 / 1.4))
    cfl = 0.4
    got = g.calc_dt(2, cfl)
    dt = g.dt()
    lim = [1.393, 0.464, 0.235, 0.1453, 0.100, 0.0736][P]
    X = m.element_nodes()[:, :, :2]
    E = np.roll(X, -1, axis=1) - X  # edge vectors
    a, b = X[:, 1] - X[:, 0], X[:, 2] - X[:, 0]
    area = 0.5 * (a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0])
    L = np.linalg.norm(E, axis=2)
    vn = np.abs(0.3 * E[:, :, 1] - 0.2 * E[:, :, 0]) / L
    want = cfl * lim * 2 * area / ((vn + 1.0) * L).sum(axis=1)  # sound speed sqrt(1.4 p / rho) = 1
    # sums of at most 21 terms with 15-digit quadrature weights
    assert np.abs(dt - want).max() <= 1e-12 * want.max()
    assert abs(got - want.min()) <= 1e-12 * want.min()
    g.close()

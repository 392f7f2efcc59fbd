"""The layout changes at the ABI edge run on the device: arrays of up to 8 MB
into a pinned host buffer, larger ones through a scratch buffer of the stage
state's size, in chunks of points where that is smaller than the array (FP32
contexts, traces).  Sizes at the edges: element counts
that are no multiple of a workgroup's elements, one field, the smallest and
largest elements."""
import numpy as np
import pytest

from fr_learn_amd import Solver, _lib, cases, mesh

pytestmark = pytest.mark.gpu

SHAPES = [("quad", 1, (3, 3)), ("quad", 4, (7, 5)), ("quad", 5, (41, 3)), ("tri", 2, (5, 4)), ("tri", 5, (3, 7)),
          ("quad", 5, (103, 101)), ("hex", 1, (3, 4, 5)), ("hex", 3, (3, 3, 4)), ("hex", 5, (3, 3, 3)), ("hex", 3, (17, 16, 19))]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("equation", [0, 1])
@pytest.mark.parametrize("elem,P,n", SHAPES)
def test_state_layouts(elem, P, n, equation, precision):
    D = len(n)
    cfg = cases.config(nDims=D, order=P, equation=equation, advectVz=1.0)
    box = (mesh.tri_box if elem == "tri" else lambda *a, **k: mesh.box(D, *a, **k))
    m = box(n, (0.0,) * D, (1.0,) * D, shuffle=True, seed=3)
    print(f"layout {elem} P={P} {n} eq={equation} {precision}", flush=True)
    g = Solver(cfg, m, precision=precision)
    rng = np.random.default_rng(5)
    U = 1.0 + 0.1 * rng.standard_normal(g.state_shape())
    if equation == 1:
        U[..., -1] += 5.0
    g.set_state(U)
    dev = np.zeros((g.nEles, g.nFields, g.nSpts))
    _lib.check(g._lib.fr_get_state(g._h, _lib.dptr(dev), _lib.FR_LAYOUT_DEVICE))
    # device element i is mesh element order[i]; copies are exact
    assert np.array_equal(dev, U.transpose(1, 2, 0)[g.element_order()])
    assert np.array_equal(g.get_state(), U)
    # residuals and traces: reference layout against the device's
    g.calc_residual(0)
    R = g.residual(0)
    _lib.check(g._lib.fr_get_residual(g._h, 0, _lib.dptr(dev), _lib.FR_LAYOUT_DEVICE))
    assert np.array_equal(dev, R.transpose(1, 2, 0)[g.element_order()])
    # FP64: the dense extrapolation, sums of at most 21 terms of order 1..10;
    # FP32: 24-bit values of the same sums
    want = np.einsum("qs,sek->qek", g.operator(0), U)
    tol = 1e-13 if precision == "fp64" else 2e-6
    assert np.abs(g.traces() - want).max() <= tol * np.abs(want).max()
    g.close()


def test_scratch_holds_a_point_of_the_normals():
    """The smallest stage state, 3 FP32 values an element, against the 2 FP64
    components of a normal, on a mesh whose normals pass the pinned buffer's
    size: the same array as from an FP64 context, bit for bit."""
    n = (310, 290)
    m = mesh.tri_box(n, (0.0, 0.0), (1.0, 1.0), perturb=0.2, seed=1)
    out = []
    for precision in ("fp32", "fp64"):
        g = Solver(cases.config(nDims=2, order=1, equation=0), m, precision=precision)
        out.append(g.geometry(2))
        g.close()
    assert out[0].nbytes > 8 << 20
    assert np.array_equal(out[0], out[1])


def test_read_backs_from_several_threads():
    """The pinned buffer is one for the process: threads that meet at it get
    their own context's state."""
    import threading
    solvers, states = [], []
    for i in range(4):
        cfg = cases.config(nDims=2, order=3)
        s = Solver(cfg, mesh.box(2, (9 + i, 40), (0.0, 0.0), (1.0, 1.0)))
        U = np.random.default_rng(i).uniform(1.0, 2.0, s.state_shape())
        s.set_state(U)
        solvers.append(s)
        states.append(U)
    wrong = []

    def work(i):
        for _ in range(200):
            if not np.array_equal(solvers[i].get_state(), states[i]):
                wrong.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    for s in solvers:
        s.close()

"""What crosses the ABI keeps every bit: negative zeros, subnormal numbers,
infinities and NaN payloads, through the pinned buffer and (arrays above 8 MB)
the copies."""
import numpy as np
import pytest

from fr_learn_amd import Solver, cases, mesh

pytestmark = pytest.mark.gpu

ODD = np.array([0x8000000000000000, 0x0000000000000001, 0x800fffffffffffff, 0x7ff0000000000000, 0xfff0000000000000,
                0x7ff8000000001234, 0xfff8000000000001], dtype=np.uint64).view(np.float64)


@pytest.mark.parametrize("equation", [0, 1])
@pytest.mark.parametrize("D,P,n", [(2, 3, (5, 7)), (3, 2, (3, 4, 3)), (2, 4, (251, 203))])
def test_state_bits(D, P, n, equation):
    g = Solver(cases.config(nDims=D, order=P, equation=equation), mesh.box(D, n, (0.0,) * D, (1.0,) * D))
    U = np.random.default_rng(1).uniform(1.0, 2.0, g.state_shape())
    # odd entries in every field
    flat = U.reshape(-1, g.nFields)
    for k in range(g.nFields):
        flat[k:k + 3 * len(ODD):3, k] = ODD
    g.set_state(U)
    assert np.array_equal(g.get_state().view(np.uint64), U.view(np.uint64))
    g.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_residual_bits(precision):
    """A residual of a medium at rest holds zeros of both signs; the reference
    layout has the device layout's bits."""
    from fr_learn_amd import _lib
    g = Solver(cases.config(nDims=2, order=3, equation=1), mesh.box(2, (6, 5), (0.0, 0.0), (1.0, 1.0)),
               precision=precision)
    U = np.zeros(g.state_shape())
    U[..., 0], U[..., -1] = 1.0, 2.5
    U[..., 1] = -1e-30 * np.random.default_rng(2).uniform(0.0, 1.0, U.shape[:2])
    g.set_state(U)
    g.calc_residual(0)
    dev = np.zeros((g.nEles, g.nFields, g.nSpts))
    _lib.check(g._lib.fr_get_residual(g._h, 0, _lib.dptr(dev), _lib.FR_LAYOUT_DEVICE))
    want = np.empty(g.state_shape())
    want[:, g.element_order()] = dev.transpose(2, 0, 1)
    assert np.array_equal(g.residual(0).view(np.uint64), want.view(np.uint64))
    g.close()

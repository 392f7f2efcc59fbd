"""A HIP error that another caller of the thread left behind is not the
read-back's: setting and getting arrays go by their own calls' status."""
import numpy as np
import pytest

from fr_learn_amd import Solver, cases, mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(6, 5), (301, 200)])  # through the pinned buffer, and above 8 MB
def test_older_errors_are_not_reported(n):
    g = Solver(cases.config(nDims=2, order=3, equation=0), mesh.box(2, n, (0.0, 0.0), (1.0, 1.0)))
    U = np.random.default_rng(0).uniform(1.0, 2.0, g.state_shape())
    g.set_state(U)
    g.calc_residual(0)
    R = g.residual(0)
    for call, want in ((g.get_state, U), (lambda: g.residual(0), R), (lambda: g.set_state(U), None)):
        assert g._lib.hipSetDevice(1 << 20) != 0  # no such device: an error of the host's check alone
        out = call()
        assert want is None or np.array_equal(out, want)
        g._lib.hipGetLastError()
    g.close()

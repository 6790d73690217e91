"""The Schur smoother with several steps per launch, through V-cycles against
the oracle: levels one short of, exactly and one past the region that a
workgroup holds (14 x 14 x 15 nodes, 30 x 30), cores that end inside a region, thin levels."""
import numpy as np
import pytest

import oracle as O
from aspect_amd import StokesMatrixFreeHandler, make_box

pytestmark = pytest.mark.gpu

SIZES = [((1, 1, 1), 1), ((13, 13, 14), 1), ((14, 2, 15), 1), ((3, 14, 14), 1), ((20, 9, 31), 1), ((8, 5, 7), 2), ((7, 12, 4), 2),
         ((1, 1), 1), ((29, 29), 1), ((30, 3), 1), ((2, 45), 1), ((47, 62), 1), ((15, 24), 2)]


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n,nl", SIZES)
def test_schur_vcycle_matches_oracle(n, nl, prec):
    n3, ext, bc = n + (1,) * (3 - len(n)), (1.0, 0.7, 1.9), (1,) * 6
    p = O.make_problem(len(n), 2, n3, nl, ext, bc)
    h = StokesMatrixFreeHandler(make_box(len(n), 2, n3, nl, ext, bc), prec)
    print("schur", n, nl, prec, flush=True)
    rng = np.random.default_rng(3)
    s = O.sizes(p, nl - 1)
    eta = np.exp(rng.normal(size=(s["cells"], h.n_qp)))
    h.assemble(eta, "arithmetic")
    h.build_preconditioner()
    x = rng.normal(size=s["np"])
    ref = O.vcycle(p, eta.mean(axis=1), 1, x)
    # eigenvalue estimates and 16 steps a sweep: the bar of the V-cycle tests; in single the
    # smoother's intervals are those of the oracle, and mass matrices lose a factor ~ 20
    tol = 1e-10 if prec == "fp64" else 16 * 20 * 2.0 ** -24 * 10
    assert np.linalg.norm(h.vcycle(1, x) - ref) < tol * np.linalg.norm(ref)

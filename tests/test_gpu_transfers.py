"""One-launch transfers of degree-2 levels at the edges of their blocks of
cells, against the oracle: single cells, sides where a block of 128 threads ends
inside or at a row, free, normal-fixed and fixed faces."""
import numpy as np
import pytest

import oracle as O
from aspect_amd import StokesMatrixFreeHandler, make_box

pytestmark = pytest.mark.gpu

# three nested sums of at most 5 products with weights of magnitude <= 1: ~ 20 roundings
TOL = 50 * 2.0 ** -53


@pytest.mark.parametrize("bc", [(1, 2, 0, 1, 1, 2), (2, 1, 1, 0, 0, 1)])
@pytest.mark.parametrize("n", [(1, 1, 1), (3, 1, 2), (1, 5, 1), (11, 10, 3), (15, 7, 2), (1, 1), (7, 15), (126, 2), (2, 127)])
def test_transfers_match_oracle(n, bc):
    ext = (1.0, 0.7, 1.9)
    p = O.make_problem(len(n), 2, n + (1,) * (3 - len(n)), 2, ext, bc)
    h = StokesMatrixFreeHandler(make_box(len(n), 2, n + (1,) * (3 - len(n)), 2, ext, bc), "fp64")
    print("transfers", n, bc, flush=True)
    rng = np.random.default_rng(7)
    h.assemble(np.ones((O.sizes(p, 1)["cells"], h.n_qp)), "arithmetic")
    for kind, key in ((0, "nu"), (1, "np")):
        xc, xf = rng.normal(size=O.sizes(p, 0)[key]), rng.normal(size=O.sizes(p, 1)[key])
        for got, ref in ((h.prolongate(1, kind, xc), O.prolongate(p, 1, kind, xc)),
                         (h.restrict(1, kind, xf), O.restrict(p, 1, kind, xf))):
            assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref)

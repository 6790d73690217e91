"""The Schur smoother with several steps per launch, through V-cycles against
the oracle: levels one short of, exactly and one past the region that a
workgroup holds (14 x 14 x 16 nodes, 30 x 30), cores that end inside a region, thin levels.
The finest of two levels smooths with degree 4, a single level with degree 8: in 3D that is
more than a region's margin holds, so that a single level beyond the region takes one step
per launch."""
import numpy as np
import pytest

import oracle as O
from aspect_amd import StokesMatrixFreeHandler, make_box

pytestmark = pytest.mark.gpu

SIZES = [((1, 1, 1), 1), ((13, 13, 14), 1), ((14, 2, 15), 1), ((3, 14, 14), 1), ((20, 9, 31), 1), ((8, 5, 7), 2), ((7, 12, 4), 2),
         ((13, 13, 15), 1), ((13, 13, 16), 1), ((2, 2, 7), 2), ((7, 2, 7), 2), ((2, 3, 8), 2), ((2, 2, 13), 2), ((7, 12, 13), 2),
         ((12, 8, 20), 2), ((1, 1), 1), ((29, 29), 1), ((30, 3), 1), ((2, 45), 1), ((47, 62), 1), ((15, 24), 2)]


def blocks(n, nl):
    """Blocks per direction on the finest level; None: one step per launch."""
    dim, degree = len(n), 4 if nl > 1 else 8
    nodes, width = [(c << (nl - 1)) + 1 for c in n], (14, 14, 16) if dim == 3 else (30, 30)
    if all(m <= w for m, w in zip(nodes, width)):
        return (1,) * dim
    if dim == 3 and degree > 4:
        return None
    margin = 3 if dim == 3 else 7  # one sweep of 4, two of 4 or one of 8
    return tuple(1 if m <= w else 2 + max(0, -(-(m - 2 * (w - margin)) // (w - 2 * margin))) for m, w in zip(nodes, width))


def test_every_number_of_blocks_is_reached():
    got = [blocks(n, nl) for n, nl in SIZES if len(n) == 3]
    for d, most in ((0, 3), (1, 3), (2, 4)):
        assert {b[d] for b in got if b and max(b) > 1} >= set(range(1, most + 1))
    assert (2, 3, 3) in got and (1, 1, 1) in got and None in got
    assert {1, 2, 3} <= {b[1] for n, nl in SIZES if len(n) == 2 for b in [blocks(n, nl)]}


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

"""Assembly of general-mesh applies where a master carries many constrained
DoFs (across components, with lines without masters between them) and where a
node belongs to 4 or 8 cells, against the oracle at its bar."""
import numpy as np
import pytest

from aspect_amd import TriaOperators
from aspect_amd import tria as T
from oracle import tria as OT

pytestmark = pytest.mark.gpu


def lines(n, n_slaves, rng):
    """n_slaves DoFs constrained to the same two masters, and three fixed ones."""
    pick = rng.permutation(n)
    masters, slaves, fixed = pick[:2], pick[2:2 + n_slaves], pick[2 + n_slaves:5 + n_slaves]
    dofs = np.sort(np.concatenate([slaves, fixed]))
    offs, mas, w = [0], [], []
    for d in dofs:
        if d in slaves:
            mas += list(masters)
            w += list(rng.uniform(0.2, 0.8, 2))
        offs.append(len(mas))
    return dofs, np.array(offs), np.array(mas, dtype=np.int64), np.array(w)


@pytest.mark.parametrize("n_slaves", [0, 1, 3, 4, 5, 9, 40])
@pytest.mark.parametrize("mesh", ["box2d", "box3d", "shell2d"])
def test_many_lines_on_one_master(mesh, n_slaves):
    t = T.Tria(T.ShellCoarse(2), 1) if mesh == "shell2d" else \
        T.Tria(T.BoxCoarse(int(mesh[3]), (4, 3, 2)[:int(mesh[3])], (1.5, 1.0, 1.2)[:int(mesh[3])]), 1)
    m = t.build({})
    rng = np.random.default_rng(n_slaves)
    m.con_u, m.con_p = lines(m.n_dofs_u, n_slaves, rng), lines(m.n_dofs_p, min(n_slaves, 9), rng)
    print("lines", mesh, n_slaves, m.n_cells, flush=True)
    eta = np.exp(rng.normal(size=(m.n_cells, 3 ** m.dim)))
    ref, gpu = OT.Operators(m, eta), TriaOperators(m)
    gpu.set_viscosity(eta)
    u, p = rng.normal(size=m.n_dofs_u), rng.normal(size=m.n_dofs_p)
    for got, want in ((gpu.vmult("ablock", u), ref.ablock(u)), (gpu.vmult("mass", p), ref.mass(p)),
                      (gpu.vmult("bt", p), ref.bt(p))):
        assert np.max(np.abs(got - want)) <= 1e-12 * np.max(np.abs(want))


@pytest.mark.parametrize("n_u,n_p", [(0, 0), (1, 0), (0, 1), (63, 2), (64, 9), (65, 1)])
def test_stokes_with_lines_in_either_block(n_u, n_p):
    # both blocks' line sums in one launch, split at a whole block of 64 threads
    m = T.Tria(T.BoxCoarse(3, (4, 3, 2), (1.5, 1.0, 1.2)), 1).build({})
    rng = np.random.default_rng(n_u)
    m.con_u, m.con_p = lines(m.n_dofs_u, n_u, rng), lines(m.n_dofs_p, n_p, rng)
    print("stokes lines", n_u, n_p, flush=True)
    eta = np.exp(rng.normal(size=(m.n_cells, 27)))
    ref, gpu = OT.Operators(m, eta), TriaOperators(m)
    gpu.set_viscosity(eta)
    x = rng.normal(size=m.n_dofs_u + m.n_dofs_p)
    got, want = gpu.vmult("stokes", x), ref.stokes(x)
    assert np.max(np.abs(got - want)) <= 1e-12 * np.max(np.abs(want))

"""Applies from the cell matrices (levels with one viscosity per cell) at the
edges of their boxes of columns and marches, against the quadrature form: an
in-place call cannot take the one-launch kernel (a workgroup would overwrite
what its neighbours read) and runs the split quadrature kernels."""
import numpy as np
import pytest
import torch

import oracle as O
from aspect_amd import StokesMatrixFreeHandler, make_box

pytestmark = pytest.mark.gpu

MIXED = (1, 2, 0, 1, 1, 2)
# a box owns 7 x 7 columns of cells or a longer strip, small levels march one layer:
# one cell, one short of / exactly / one past a box, strips
SIZES = [(1, 1, 1), (6, 7, 8), (7, 8, 2), (8, 6, 13), (21, 2, 3), (2, 30, 5), (15, 14, 12), (40, 33, 24)]
# larger levels march up to 11 layers in double and 6 in single, with and without a rest
LONG = [(56, 100, 3), (56, 100, 6), (64, 72, 12), (56, 100, 14), (56, 64, 33), (100, 120, 10), (72, 72, 33), (56, 64, 45),
        (64, 64, 41)]
# a row sums at most 8 cells x 36 products after 6 sums: ~ sqrt(8 * 42) rounding errors of the largest
# terms, which the smooth part of a random field leaves ~ 10 times larger than the row
TOL = {"fp64": 200 * 2.0 ** -53 * 10, "fp32": 200 * 2.0 ** -24 * 10}


def _box(n, bc, compressible, prec):
    h = StokesMatrixFreeHandler(make_box(len(n), 2, n, 1, (1.0, 0.7, 1.9), bc, compressible, 1.3), prec)
    s = h.sizes(0)
    rng = np.random.default_rng(sum(n))
    h.assemble(np.exp(rng.normal(scale=2.0, size=(s["cells"], h.n_qp))), "harmonic")
    return h, s, rng


def _against_in_place(apply, x):
    y, z = torch.full_like(x, float("nan")), x.clone()
    torch.cuda.synchronize()
    apply(x.data_ptr(), y.data_ptr())
    apply(z.data_ptr(), z.data_ptr())
    torch.cuda.synchronize()
    return float((y - z).norm() / z.norm())


def march_layers(n, size):
    """Layers per march of the launch rule (values of size bytes)."""
    boxes = min(-(-(n[0] + 1) // (tx - 1)) * -(-(n[1] + 1) // (64 // tx - 1)) for tx in range(3, 22))
    best, cost = 1, None
    for layers in (1, 2, 3, 4, 6, 8, 11)[:7 if size == 8 else 5]:
        r = boxes * ((n[2] + layers) // layers) / (512 if size == 8 else 1024)
        c = (np.ceil(r) if r < 3 else r + 0.5) * (layers + 1.5)
        if cost is None or c < cost:
            best, cost = layers, c
    return best


def test_long_marches_are_reached():
    for size, layers in ((8, {2, 3, 4, 6, 8, 11}), (4, {1, 2, 3, 4, 6})):
        got = [(march_layers(n, size), (n[2] + 1) % march_layers(n, size) == 0) for n in LONG]
        assert {g[0] for g in got} == layers and {g[1] for g in got if g[0] > 1} == {True, False}
    assert all(march_layers(n, 4) == 1 for n in SIZES)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n", LONG)
def test_long_march_chebyshev_matches_quadrature(n, prec):
    # the step fused into the march, eight times, against the recurrence with in-place applies in double
    h, s, rng = _box(n, MIXED, True, prec)
    q = h if prec == "fp64" else _box(n, MIXED, True, "fp64")[0]
    print("chebyshev", n, prec, flush=True)
    h.build_preconditioner()
    theta, delta = h.smoother_info()[0, 0, 2:4]
    b = rng.normal(size=s["nu"])
    b = b if prec == "fp64" else b.astype(np.float32).astype(float)
    bd, dinv = torch.tensor(b, device="cuda:0"), 1.0 / torch.tensor(q.ablock_diagonal(0), device="cuda:0")

    def apply(x):
        y = x.clone()
        torch.cuda.synchronize()
        q.ablock_vmult_device(0, y.data_ptr(), y.data_ptr())
        q.synchronize()
        return y

    x = d = dinv * bd / theta
    rho = delta / theta
    for _ in range(1, 8):
        new = 1.0 / (2.0 * theta / delta - rho)
        d = new * rho * d + 2.0 * new / delta * dinv * (bd - apply(x))
        x, rho = x + d, new
    got = torch.tensor(h.chebyshev(0, 0, b), device="cuda:0")
    assert float((got - x).norm() / x.norm()) < 8 * TOL[prec]  # an apply's error each step


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("compressible", [False, True])
@pytest.mark.parametrize("n", LONG + SIZES + [(1, 1), (7, 7), (8, 6), (50, 3), (33, 40)])
def test_ablock_apply_matches_quadrature(n, compressible, prec):
    h, s, rng = _box(n, MIXED, compressible, prec)
    print("ablock", n, prec, compressible, flush=True)
    x = torch.tensor(rng.normal(size=s["nu"]), dtype=torch.float64 if prec == "fp64" else torch.float32, device="cuda:0")
    assert _against_in_place(lambda a, b: h.ablock_vmult_device(0, a, b), x) < TOL[prec]


@pytest.mark.parametrize("n", SIZES + LONG)
def test_stokes_apply_matches_quadrature(n):
    for bc in (MIXED, (2,) * 6, (0,) * 6):
        h, s, rng = _box(n, bc, False, "fp64")
        print("stokes", n, bc, flush=True)
        x = torch.tensor(rng.normal(size=s["nu"] + s["np"]), device="cuda:0")
        assert _against_in_place(h.stokes_vmult_device, x) < TOL["fp64"]


@pytest.mark.parametrize("n", [(1, 1), (7, 7), (8, 6), (50, 3)])
def test_stokes_2d_matches_oracle(n):
    # the 2D quadrature form runs in tile colours and takes no in-place call
    bc = MIXED[:4]
    h, s, rng = _box(n, bc, True, "fp64")
    eta = np.exp(np.random.default_rng(sum(n)).normal(scale=2.0, size=(s["cells"], 9)))
    p = O.make_problem(2, 2, n, 1, (1.0, 0.7), bc, pressure_scaling=1.3, compressible=True)
    x = rng.normal(size=s["nu"] + s["np"])
    ref = O.stokes_vmult(p, 0, 1.0 / np.mean(1.0 / eta, axis=1), x)
    assert np.linalg.norm(h.stokes_vmult(x) - ref) < TOL["fp64"] * np.linalg.norm(ref)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("coarse", [(2, 1, 3), (3, 5)])
def test_tables_of_every_level(coarse, prec):
    # made once for all levels, when the first viscosity of one value per cell comes,
    # here after a table per quadrature point and kept over the next viscosity
    dim, ext, bc = len(coarse), (1.0, 0.7, 1.9), (0, 2, 1, 0, 0, 1)
    p = O.make_problem(dim, 2, coarse + (1,) * (3 - dim), 3, ext, bc[:2 * dim], pressure_scaling=1.3, compressible=True)
    h = StokesMatrixFreeHandler(make_box(dim, 2, coarse, 3, ext[:dim], bc[:2 * dim], True, 1.3), prec)
    rng = np.random.default_rng(5)
    cells = O.sizes(p, 2)["cells"]
    h.assemble(np.exp(rng.normal(size=(cells, h.n_qp))), "project to Q1 only viscosity")
    h.build_preconditioner()
    for _ in range(2):
        eta = np.exp(rng.normal(scale=2.0, size=(cells, h.n_qp)))
        h.assemble(eta, "harmonic")
        h.build_preconditioner()
        levels = O.level_viscosity(p, 1.0 / np.mean(1.0 / eta, axis=1))
        for l in range(3):
            x = rng.normal(size=O.sizes(p, l)["nu"])
            x = x if prec == "fp64" else x.astype(np.float32).astype(float)
            ref = O.ablock_vmult(p, l, levels[l], x)
            assert np.linalg.norm(h.ablock_vmult(l, x) - ref) < TOL[prec] * np.linalg.norm(ref), l
        x = rng.normal(size=O.sizes(p, 2)["nu"] + O.sizes(p, 2)["np"])
        ref = O.stokes_vmult(p, 2, levels[2], x)
        assert np.linalg.norm(h.stokes_vmult(x) - ref) < TOL["fp64"] * np.linalg.norm(ref)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("compressible", [False, True])
@pytest.mark.parametrize("n", [(9, 8, 10), (40, 33, 24), (1, 1, 1), (17, 9), (50, 3)])
def test_constant_velocity_has_no_strain(n, compressible, prec):
    # exactly zero, without a remainder of rounded entries: it would be the same in every
    # cell of a level, like a small mass term
    h, s, rng = _box(n, (0,) * (2 * len(n)), compressible, prec)
    print("constant", n, prec, compressible, flush=True)
    value = torch.tensor(rng.normal(size=(len(n), 1)), dtype=torch.float64 if prec == "fp64" else torch.float32, device="cuda:0")
    x = value.expand(len(n), s["nu"] // len(n)).reshape(-1).contiguous()
    y = torch.full_like(x, float("nan"))
    torch.cuda.synchronize()
    h.ablock_vmult_device(0, x.data_ptr(), y.data_ptr())
    torch.cuda.synchronize()
    assert bool((y == 0).all())


def test_set_up_of_cellwise_levels_keeps_no_work_array():
    # the estimate of level 0 runs the split form: its work array has that
    # level's size, not the finest one's (72 MB here)
    for n in (8, 64):  # the first handle pays what the process pays once
        h = StokesMatrixFreeHandler(make_box(3, 2, (1, 1, 1), n.bit_length(), (1.0,) * 3, (1,) * 6), "fp64")
        h.assemble(np.ones((n ** 3, h.n_qp)), "harmonic")
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        h.build_preconditioner()
        used = before - torch.cuda.mem_get_info()[0]
    assert used < 16 << 20  # the inverse cell viscosities: 2.4 MB over the levels


def test_source_outside_the_mesh_is_not_read_into_rows():
    # columns beyond the mesh read the nearest cells and discard the values:
    # an infinity at one node reaches only the rows of the cells that hold it
    h, s, rng = _box((9, 8, 10), (0,) * 6, False, "fp64")
    x = torch.tensor(rng.normal(size=s["nu"]), device="cuda:0")
    x[0] = float("inf")
    y = torch.zeros_like(x)
    torch.cuda.synchronize()
    h.ablock_vmult_device(0, x.data_ptr(), y.data_ptr())
    torch.cuda.synchronize()
    bad = ~torch.isfinite(y.cpu().reshape(3, 21, 17, 19))
    assert bad[:, :3, :3, :3].any() and not bad[:, 3:].any() and not bad[:, :, 3:].any() and not bad[..., 3:].any()

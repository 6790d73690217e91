"""The allocation-free A-block apply (mfs_ablock_vmult_device_noalloc) against
mfs_ablock_vmult_device through the C-ABI: bit-identical results (same
kernels, only the work array differs), on two calls in a row with the second
on a smaller level, in both GMG precisions, and the size limit of the scratch
array reported as an error before any launch.  The work array is read with
viscosities at the quadrature points (project to Q1) and in place; with one
viscosity per cell (harmonic) both calls run the kernel that needs none."""
import numpy as np
import pytest
import torch

from aspect_amd import StokesMatrixFreeHandler, make_box
from aspect_amd.mfs import SolverError

pytestmark = pytest.mark.gpu

AVERAGING = {"q1": "project to Q1 only viscosity", "cell": "harmonic"}


def _handler(prec, coarse, n_levels, seed, averaging):
    box = make_box(3, 2, coarse, n_levels, (1.0, 1.0, 1.0), (1, 2, 0, 1, 1, 2), pressure_scaling=1.3)
    h = StokesMatrixFreeHandler(box, prec)
    s = h.sizes(h.top)
    rng = np.random.default_rng(seed)
    h.assemble(np.exp(rng.normal(size=(s["cells"], h.n_qp))), AVERAGING[averaging])
    return h, rng


def _pair(h, rng, level, dtype, in_place=False):
    n = h.sizes(level)["nu"]
    src = torch.tensor(rng.normal(size=n), dtype=dtype, device="cuda:0")
    ref = src.clone() if in_place else torch.full((n,), float("nan"), dtype=dtype, device="cuda:0")
    out = src.clone() if in_place else torch.full((n,), float("nan"), dtype=dtype, device="cuda:0")
    torch.cuda.synchronize()
    h.ablock_vmult_device(level, ref.data_ptr() if in_place else src.data_ptr(), ref.data_ptr())
    h.lib.mfs_synchronize(h._h)
    h.ablock_vmult_device_noalloc(level, out.data_ptr() if in_place else src.data_ptr(), out.data_ptr())
    h.lib.mfs_synchronize(h._h)
    return ref.cpu().numpy(), out.cpu().numpy()


@pytest.mark.parametrize("averaging,in_place", [("q1", False), ("cell", False), ("cell", True)])
@pytest.mark.parametrize("prec,dtype", [("fp32", torch.float32), ("fp64", torch.float64)])
def test_noalloc_matches_allocating_apply(prec, dtype, averaging, in_place):
    # 24x16x8 cells on the finest level (partial tiles), then a smaller level
    h, rng = _handler(prec, (3, 2, 1), 4, 7, averaging)
    for level in (h.top, h.top - 2):
        print(f"noalloc {prec} {averaging} level {level}", flush=True)
        ref, out = _pair(h, rng, level, dtype, in_place)
        assert np.all(np.isfinite(ref)) and np.array_equal(ref, out), level


@pytest.mark.parametrize("averaging,in_place", [("q1", False), ("cell", False), ("cell", True)])
@pytest.mark.parametrize("prec,dtype", [("fp32", torch.float32), ("fp64", torch.float64)])
def test_noalloc_2d_split_apply(prec, dtype, averaging, in_place):
    # 2D degree 2: the split A-block apply's work array (2 x 17^2 per 8x8-cell
    # tile) also comes from the scratch array; 40x24 cells (partial tiles),
    # then a smaller level
    box = make_box(2, 2, (5, 3), 4, (2.0, 1.0), (1, 2, 0, 1), pressure_scaling=1.1)
    h = StokesMatrixFreeHandler(box, prec)
    s = h.sizes(h.top)
    rng = np.random.default_rng(11)
    h.assemble(np.exp(rng.normal(size=(s["cells"], h.n_qp))), AVERAGING[averaging])
    for level in (h.top, h.top - 2):
        print(f"noalloc 2D {prec} {averaging} level {level}", flush=True)
        ref, out = _pair(h, rng, level, dtype, in_place)
        assert np.all(np.isfinite(ref)) and np.array_equal(ref, out), level


@pytest.mark.parametrize("averaging", ["q1", "cell"])
def test_noalloc_size_limit(averaging):
    # 96x96x64 cells = 9216 tiles: 9216 x 3 x 386 FP64 values (85 MB) exceed
    # the 72 MiB array (rejected before any launch, also where the call would need
    # no work array); the FP32 work array fits
    h64, rng = _handler("fp64", (3, 3, 2), 6, 3, averaging)
    n = h64.sizes(h64.top)["nu"]
    src = torch.zeros(n, dtype=torch.float64, device="cuda:0")
    dst = torch.zeros(n, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    with pytest.raises(SolverError, match="scratch array"):
        h64.ablock_vmult_device_noalloc(h64.top, src.data_ptr(), dst.data_ptr())
    del h64, src, dst
    h32, rng = _handler("fp32", (3, 3, 2), 6, 3, averaging)
    print("noalloc fp32 96x96x64", flush=True)
    ref, out = _pair(h32, rng, h32.top, torch.float32)
    assert np.array_equal(ref, out)

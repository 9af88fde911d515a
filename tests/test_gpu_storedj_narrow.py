"""Stored-J products of few right-hand sides against the full-width product.

A product of at most 32 (FP32) or 16 (FP64) right-hand sides runs on one narrow matrix-core
tile instead of the 64-wide one.  Every right-hand side's sums keep their order, so each
column equals the same column of a 64-wide product bit for bit; both are also compared with
a NumPy float64 product of the FP64 J (bound: n eps of the sum of magnitudes, n the sums'
length)."""
import numpy as np
import pytest

from jif3d_amd import _native as nat
from jif3d_amd.model import ThreeDGravityModel, TensorGravityData

pytestmark = pytest.mark.gpu


def context(nx, ny, nz, nsites, fp64, host_block_cells=None):
    rng = np.random.default_rng(nx * ny + nsites)
    m = ThreeDGravityModel()
    m.SetMeshSize(nx, ny, nz)
    m.SetXCellSizes(np.full(nx, 20.0))
    m.SetYCellSizes(np.full(ny, 30.0))
    m.SetZCellSizes(10.0 * 1.1 ** np.arange(nz))
    m.SetDensities(rng.normal(size=nx * ny * nz))
    d = TensorGravityData()
    d.SetMeasurementPoints(rng.uniform(0, 20.0 * nx, nsites), rng.uniform(0, 30.0 * ny, nsites),
                           -rng.uniform(5, 50, nsites))
    ctx = nat.Context()
    ctx.configure(m, d)
    ctx.storedj_build(nat.KIND_SCALAR_TENSOR, nat.FP64, host_block_cells, fp64=fp64)
    return ctx


def product(ctx, fp64, transpose, X):
    n = ctx.storedj_cols() if transpose else ctx.storedj_rows()
    dt = np.float64 if fp64 else np.float32
    x, y = ctx.to_device(np.ascontiguousarray(X, dtype=dt)), ctx.alloc((X.shape[0], n), dt)
    if fp64:
        (ctx.storedj_apply_t_f64 if transpose else ctx.storedj_apply_f64)(x, y)
    else:
        (ctx.storedj_apply_t if transpose else ctx.storedj_apply)(nat.GEMM_FP32, x, y)
    out = y.to_host()
    x.free()
    y.free()
    return out


@pytest.mark.parametrize("fp64", [False, True])
@pytest.mark.parametrize("mesh", [(1, 1, 1, 1), (7, 5, 3, 9), (16, 16, 1, 64), (13, 11, 17, 75)])
def test_narrow_equals_wide(mesh, fp64):
    ctx = context(*mesh, fp64)
    rng = np.random.default_rng(3)
    ref = context(*mesh, True)
    J = product(ref, True, False, np.eye(ref.storedj_cols())).T
    eps = np.finfo(np.float64 if fp64 else np.float32).eps
    for transpose in (False, True):
        k = ctx.storedj_rows() if transpose else ctx.storedj_cols()
        X = rng.normal(size=(64, k)).astype(np.float64 if fp64 else np.float32)
        wide = product(ctx, fp64, transpose, X)
        Jx = J if transpose else J.T
        bound = (k + 4) * eps * (np.abs(X).astype(np.float64) @ np.abs(Jx))
        assert np.all(np.abs(wide - X.astype(np.float64) @ Jx) <= bound)
        for n in (1, 2, 15, 16, 17, 31, 32, 33, 63):
            assert np.array_equal(product(ctx, fp64, transpose, X[:n]), wide[:n]), (transpose, n)


def test_narrow_streamed_from_host():
    """J in host memory, streamed in blocks: the narrow products equal the wide ones."""
    ctx = context(13, 11, 17, 75, False, host_block_cells=512)
    rng = np.random.default_rng(4)
    for transpose in (False, True):
        k = ctx.storedj_rows() if transpose else ctx.storedj_cols()
        X = rng.normal(size=(64, k)).astype(np.float32)
        wide = product(ctx, False, transpose, X)
        for n in (1, 32, 33):
            assert np.array_equal(product(ctx, False, transpose, X[:n]), wide[:n]), (transpose, n)

"""Calls whose natural launch would pass the 2^32 threads that a launch dimension can have: they
take the kernels whose grids stay below it."""
import ctypes
import types

import numpy as np
import pytest

from jif3d_amd import _native as nat

pytestmark = pytest.mark.gpu
G = 6.67428e-11


def mesh(dims, cell=20.0):
    return types.SimpleNamespace(
        nx=dims[0], ny=dims[1], nz=dims[2], sizes=[np.full(n, cell) for n in dims],
        coords=[cell * np.arange(n + 1.0) for n in dims], bg_thicknesses=np.zeros(0))


def entry(ctx, rows, at):
    out = np.empty(1)
    nat.check(ctx.lib.jgm_copy_to_host(ctx.handle, out.ctypes.data_as(ctypes.c_void_p),
                                       ctypes.c_void_p(rows.ptr + 8 * at), 8))
    return out[0]


def test_rows_of_a_mesh_with_two_to_the_23_bricks(orc):
    """8192 x 1025 bricks of 7 columns are 2^32 threads of 512 each and more; three rows of three
    values a cell take 17 GB."""
    dims = (8192, 7175, 4)
    ctx = nat.Context()
    ctx.set_mesh(mesh(dims))
    site = np.array([20.0 * dims[0] - 33.0, 20.0 * dims[1] - 47.0, -30.0])
    ctx.set_sites(*site[:, None])
    n = dims[0] * dims[1] * dims[2]
    rows = ctx.alloc((3, 3 * n))
    ctx.sensitivity_rows(nat.KIND_MAGNETIZATION, 0, 1, rows)
    ctx.synchronize()
    largest = 0.0
    errors = []
    for i, j, k in [(dims[0] - 1, dims[1] - 1, 3), (dims[0] - 2, dims[1] - 3, 0),
                    (dims[0] - 9, dims[1] - 8, 1)]:
        c = (i * dims[1] + j) * dims[2] + k
        t = 100.0 / G * orc.tensor_box_term(*site, 20.0 * i, 20.0 * j, 20.0 * k, 20.0, 20.0, 20.0,
                                            long_double=True)
        largest = max(largest, np.max(np.abs(t)))
        errors += [abs(entry(ctx, rows, (r * 3 + p) * n + c) - t[r, p])
                   for r in range(3) for p in range(3)]
    rows.free()
    # offsets of whole metres are exact; eight logarithms and arctangents each
    assert max(errors) <= 1e-11 * largest


def test_data_of_two_to_the_24_sites():
    """A workgroup of 256 threads per site would be 2^32 threads."""
    rng = np.random.default_rng(1)
    dims, n = (100, 100, 6), 1 << 24
    rho = 2670 + 200 * rng.normal(size=dims[0] * dims[1] * dims[2])
    p = [rng.uniform(0, 2000, n), rng.uniform(0, 2000, n), -rng.uniform(3, 60, n)]
    at = [0, 12345678, n - 1]
    few, many = nat.Context(), nat.Context()
    for ctx, sites in ((few, [v[at] for v in p]), (many, p)):
        ctx.set_mesh(mesh(dims))
        ctx.set_sites(*sites)
    ref = few.forward(nat.KIND_SCALAR, nat.FP64, rho)
    many.profile_enable(True)
    out = many.forward(nat.KIND_SCALAR, nat.FP64, rho)
    assert "forward_corners_fp64_gz" in many.profile()
    assert np.max(np.abs(out[at] - ref)) <= 1e-12 * np.max(np.abs(ref))

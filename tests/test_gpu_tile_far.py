"""FP64 data and gradients of large meshes through the tile expansions (gz, gz + FTG), against
the closed form: data against the allocation-free forward, gradients of a few stations'
residuals against their sensitivity rows.  Bounds of the FP64 path: gz 1e-12, each tensor
component 1e-11 of its largest magnitude, gradients 1e-10 of the largest entry.  The closed form's
logarithms lose more where a station looks along a row of corners: an ulp of r moves log(u + r) by
eps r / (u + r); stations beyond the plain bound are held to six standard deviations of the sum of
these roundings (two ulp each) over the mesh's corners.  Mesh sizes leave remainders against the
tiles of 8 on every axis."""
import ctypes

import numpy as np
import pytest

from jif3d_amd import _native as nat
from jif3d_amd.model import ThreeDGravityModel, TensorGravityData

pytestmark = pytest.mark.gpu
KIND = {"gz": nat.KIND_SCALAR, "joint": nat.KIND_SCALAR_TENSOR}
CASES = [("gz", (100, 99, 61), 1.0, 333), ("gz", (64, 61, 31), 1.0, 1000), ("gz", (127, 101, 63), 1.03, 700),
         ("joint", (125, 119, 61), 1.0, 260), ("joint", (128, 128, 64), 1.0, 130)]


def setup(kind, dims, growth, nsites, uniform=False, on_line=False):
    rng = np.random.default_rng(dims[0] + nsites)
    m = ThreeDGravityModel()
    m.SetMeshSize(*dims)
    m.SetXCellSizes(np.full(dims[0], 20.0))
    m.SetYCellSizes(20.0 + (np.arange(dims[1]) % 3 if growth > 1 else np.zeros(dims[1])))
    m.SetZCellSizes(15.0 * growth ** np.arange(dims[2]))
    m.SetBackgroundThicknesses([400.0, 1e4])
    m.SetBackgroundDensities([2500.0, 2700.0])
    d = TensorGravityData()
    x = rng.uniform(-100, 20.0 * dims[0] + 100, nsites)
    y = rng.uniform(-100, 20.0 * dims[1] + 100, nsites)
    z = -rng.uniform(3, 60, nsites)
    z[:2] = 200.0, 30.5  # inside the mesh
    if on_line:
        x[5], y[5] = 40.0, m.coords[1][3]
    d.SetMeasurementPoints(x, y, z)
    ctx = nat.Context()
    ctx.configure(m, d)
    ctx.mesh, ctx.data = m, d
    m.shape = dims
    n = dims[0] * dims[1] * dims[2]
    rho = np.full(n, 2670.0) if uniform else 2670 + 200 * rng.normal(size=n)
    return ctx, np.concatenate([rho, [2500.0, 2700.0]]), rng


def kernels(ctx, call):
    ctx.profile_enable(True)
    ctx.profile_reset()
    call()
    names = set(ctx.profile())
    ctx.profile_enable(False)
    return names


def closed_form(ctx, kind, mv, n):
    dm, out = ctx.to_device(mv), ctx.alloc(n)
    nat.check(ctx.lib.jgm_forward_noalloc(ctx.handle, kind, nat.FP64, ctypes.c_void_p(dm.ptr),
                                          ctypes.c_void_p(out.ptr)))
    ctx.synchronize()
    return out.to_host()


def rounding(m, d, rho, s, axis):
    """Six standard deviations of the closed form's roundings in the component whose logarithm
    has u along `axis`, at station s."""
    w = np.zeros(tuple(n + 1 for n in m.shape))
    rho = rho.reshape(m.shape)
    for a in (0, 1):
        for b in (0, 1):
            for c in (0, 1):
                w[a:a + m.shape[0], b:b + m.shape[1], c:c + m.shape[2]] += (
                    rho if (a + b + c) % 2 else -rho)
    off = np.meshgrid(*(p[s] - c for p, c in zip(d.positions, m.coords)), indexing="ij")
    r = np.sqrt(sum(v * v for v in off))
    eps = np.finfo(float).eps
    term = 2 * eps * w * (1 + r / np.maximum(off[axis] + r, eps))
    return 6 * 6.67428e-11 * np.sqrt(np.sum(term ** 2))


LOG_AXIS = {2: 2, 4: 2, 3: 1, 7: 1, 6: 0, 8: 0}  # gz, then Uxx .. Uzz: xy, xz, yz


def check_data(ctx, mv, got, ref, kind):
    k = 1 if kind == "gz" else 10
    got, ref = got.reshape(-1, k), ref.reshape(-1, k)
    for c in range(k):
        tol = (1e-12 if c == 0 else 1e-11) * np.max(np.abs(ref[:, c]))
        diff = np.abs(got[:, c] - ref[:, c])
        beyond = np.nonzero(diff > tol)[0]
        assert len(beyond) == 0 or c in LOG_AXIS, c
        for s in beyond[np.argsort(diff[beyond])][-3:]:  # the largest
            extra = rounding(ctx.mesh, ctx.data, mv[:-2], s, LOG_AXIS[c])
            assert diff[s] <= tol + extra, (c, s, diff[s], extra)


@pytest.mark.parametrize("kind,dims,growth,nsites", CASES)
def test_data_and_gradient(orc, kind, dims, growth, nsites):
    ctx, mv, rng = setup(kind, dims, growth, nsites)
    K, k = KIND[kind], 1 if kind == "gz" else 10
    assert "tile_far_forward_fp64" in kernels(ctx, lambda: ctx.forward(K, nat.FP64, mv))
    check_data(ctx, mv, ctx.forward(K, nat.FP64, mv), closed_form(ctx, K, mv, nsites * k), kind)
    # three stations, one of them inside the mesh, in extended precision
    at = [0, 7, nsites - 1]
    out = ctx.forward(K, nat.FP64, mv).reshape(-1, k)
    p = [np.asarray(v)[at] for v in ctx.data.positions]
    exact = [orc.calculate_ld(orc.SCALAR, ctx.mesh, mv, p).reshape(-1, 1)]
    if k == 10:
        exact.append(orc.calculate_ld(orc.TENSOR, ctx.mesh, mv, p).reshape(-1, 9))
    error = np.abs(out[at] - np.hstack(exact))
    assert np.all(error <= 1e-12 * np.max(np.abs(out), axis=0)), error
    # residuals at five stations only: one inside the mesh, the others anywhere
    r = np.zeros((nsites, k))
    at = [0, 1, nsites // 2, nsites - 2, nsites - 1]
    r[at] = rng.normal(size=(5, k)) * ([1.0] if k == 1 else [1.0] + [500.0] * 9)
    g = ctx.adjoint(K, nat.FP64, None, r.ravel())
    ref = np.zeros(mv.size)
    for s in at:
        rows = ctx.alloc((k, mv.size))
        ctx.sensitivity_rows(K, s, 1, rows)
        ctx.synchronize()
        ref += 2.0 * rows.to_host().T @ r[s]
        rows.free()
    n = mv.size - 2
    assert np.max(np.abs(g[:n] - ref[:n])) <= 1e-10 * np.max(np.abs(ref[:n]))
    assert np.max(np.abs(g[n:] - ref[n:])) <= 1e-10 * np.max(np.abs(ref[n:]))


def test_uniform_mesh_is_one_box():
    """A uniform model's tensor is a small remainder of its cells' fields; the expansions carry
    only what differs from a reference density, so it agrees as the closed form does."""
    ctx, mv, _ = setup("joint", (125, 119, 61), 1.0, 260, uniform=True)
    got = ctx.forward(KIND["joint"], nat.FP64, mv)
    check_data(ctx, mv, got, closed_form(ctx, KIND["joint"], mv, got.size), "joint")


def test_gz_of_a_station_on_a_mesh_line():
    """The guarded logarithms of the closed form carry a factor of zero in gz."""
    ctx, mv, rng = setup("gz", (100, 99, 61), 1.0, 333, on_line=True)
    assert "tile_far_forward_fp64" in kernels(ctx, lambda: ctx.forward(KIND["gz"], nat.FP64, mv))
    check_data(ctx, mv, ctx.forward(KIND["gz"], nat.FP64, mv),
               closed_form(ctx, KIND["gz"], mv, 333), "gz")
    r = np.zeros(333)
    r[5] = 1.0
    g, rows = ctx.adjoint(KIND["gz"], nat.FP64, None, r), ctx.alloc((1, mv.size))
    ctx.sensitivity_rows(KIND["gz"], 5, 1, rows)
    ctx.synchronize()
    ref = 2.0 * rows.to_host()[0]
    rows.free()
    assert np.max(np.abs(g - ref)[:-2]) <= 1e-10 * np.max(np.abs(ref[:-2]))


@pytest.mark.parametrize("count", [3, 8, 15])  # launches of 2 + 1, 8 and 8 + 4 + 2 + 1
@pytest.mark.parametrize("kind", ["gz", "joint"])
def test_batches_equal_single_calls(kind, count):
    dims, nsites = ((100, 99, 61), 333) if kind == "gz" else ((125, 119, 61), 260)
    ctx, mv, rng = setup(kind, dims, 1.0, nsites)
    K, k = KIND[kind], 1 if kind == "gz" else 10
    M = mv[None, :] * (1 + 0.01 * rng.normal(size=(count, 1)))
    R = rng.normal(size=(count, nsites * k))
    F, G = ctx.forward_batch(K, nat.FP64, M), ctx.adjoint_batch(K, nat.FP64, None, R)
    for b in range(count):
        assert np.array_equal(F[b], ctx.forward(K, nat.FP64, M[b]))
        assert np.array_equal(G[b], ctx.adjoint(K, nat.FP64, None, R[b]))


def test_where_the_closed_form_stays():
    """A tensor station on a mesh line, a small mesh, and the tensor kind keep the closed form."""
    ctx, mv, _ = setup("joint", (125, 119, 61), 1.0, 260, on_line=True)
    names = kernels(ctx, lambda: ctx.forward(KIND["joint"], nat.FP64, mv))
    assert "forward_corners_fp64_gz_ftg" in names and "tile_far_forward_fp64" not in names
    ctx, mv, _ = setup("gz", (30, 30, 20), 1.0, 100)
    assert "forward_corners_fp64_gz" in kernels(ctx, lambda: ctx.forward(KIND["gz"], nat.FP64, mv))
    ctx, mv, _ = setup("gz", (100, 99, 61), 1.0, 333)
    names = kernels(ctx, lambda: ctx.forward(nat.KIND_TENSOR, nat.FP64, mv))
    assert "forward_corners_fp64_ftg" in names and "tile_far_forward_fp64" not in names

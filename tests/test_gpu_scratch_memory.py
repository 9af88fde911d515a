"""Device memory that a context keeps between calls: a batch's buffers stay within the stated 2 GiB
however large the mesh, and the operands of host calls within 512 MB whichever calls came before."""
import ctypes

import numpy as np
import pytest

from jif3d_amd import _native as nat
from test_gpu_launch_limits import mesh

pytestmark = pytest.mark.gpu
SLACK = 64 << 20  # allocation granularity, site-sized and small buffers


def free_bytes(ctx):
    ctx.synchronize()
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    hip = ctypes.CDLL("libamdhip64.so")
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_batch_on_a_large_mesh():
    """8.4 million cells, 16384 tiles: the near gradient of eight models at once would hold 3 GB."""
    dims, nsites, models = (256, 256, 128), 1024, 8
    rng = np.random.default_rng(0)
    ctx = nat.Context()
    ctx.set_mesh(mesh(dims))
    ctx.set_sites(rng.uniform(0, 5120, nsites), rng.uniform(0, 5120, nsites),
                  -rng.uniform(3, 60, nsites))
    n = dims[0] * dims[1] * dims[2]
    r, grad = ctx.to_device(rng.normal(size=(models, nsites))), ctx.alloc((models, n))
    before = free_bytes(ctx)
    ctx.profile_enable(True)
    ctx.adjoint_batch(nat.KIND_SCALAR, nat.FP64, None, r, grad, nmodels=models)
    used = before - free_bytes(ctx)
    assert "tile_near_adjoint_fp64" in ctx.profile()
    assert used <= (2 << 30) + SLACK
    last = grad.to_host()[models - 1]
    one = ctx.alloc((n,))
    ctx.adjoint(nat.KIND_SCALAR, nat.FP64, None, ctx.to_device(r.to_host()[models - 1]), one)
    assert np.array_equal(one.to_host(), last)


def test_operands_of_host_calls():
    """A model of 480 MB in the one call, a gradient of 480 MB in the next."""
    dims = (400, 400, 375)
    n = dims[0] * dims[1] * dims[2]
    ctx = nat.Context()
    ctx.set_mesh(mesh(dims))
    ctx.set_sites([3993.0], [4007.0], [-30.0])
    model, grad = ctx.to_device(np.full(n, 2670.0)), ctx.alloc((n,))
    data = ctx.alloc((1,))
    ctx.forward(nat.KIND_SCALAR, nat.FP64, model, data)  # the kernels' own buffers
    ctx.adjoint(nat.KIND_SCALAR, nat.FP64, None, data, grad)
    before = free_bytes(ctx)
    out = ctx.forward(nat.KIND_SCALAR, nat.FP64, np.full(n, 2670.0))
    assert np.array_equal(out, data.to_host())
    g = ctx.adjoint(nat.KIND_SCALAR, nat.FP64, None, out)
    assert np.array_equal(g, grad.to_host())
    assert before - free_bytes(ctx) <= (512 << 20) + SLACK

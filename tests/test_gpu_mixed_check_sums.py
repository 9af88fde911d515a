"""The check of a mixed gradient against FP64 sums each site's difference over a cell's corners, so
that its rounding stays a site's rounding however many sites there are.  With every cell in the near
box the mixed gradient is FP64 itself, summed the same way: the reported error is the rounding of
the two, six standard deviations of one half ulp of each corner term over the sites (corner sums
over all sites, differenced at the end, reported four times as much)."""
import numpy as np
import pytest

from jif3d_amd import _native as nat
from jif3d_amd.model import ThreeDGravityModel, TensorGravityData

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsites", [4099, 262144])
def test_check_of_a_gradient_over_many_sites(nsites):
    rng = np.random.default_rng(0)
    m = ThreeDGravityModel()
    m.SetMeshSize(6, 6, 6)
    for f in (m.SetXCellSizes, m.SetYCellSizes, m.SetZCellSizes):
        f(np.full(6, 10.0))
    d = TensorGravityData()
    d.SetMeasurementPoints(rng.uniform(0, 60, nsites), rng.uniform(0, 60, nsites),
                           -rng.uniform(150, 200, nsites))
    ctx = nat.Context()
    ctx.configure(m, d)
    ctx.set_mixed_threshold(1000.0)
    ctx.set_mixed_check(4, 216, 5e-7)
    g = ctx.adjoint(nat.KIND_SCALAR, nat.MIXED, None, np.ones(nsites))
    _, error, fallbacks = ctx.mixed_check_report()
    term = 2 * 60 * np.log(60 + 270.0) + 260 * np.pi  # x log + y log + z arctangent, at most
    site = np.sqrt(8) * 0.5 * np.finfo(float).eps * term
    bound = 6 * np.sqrt(2) * site * np.sqrt(nsites) * 2 * 6.67428e-11 / np.max(np.abs(g))
    assert fallbacks == 0
    assert error <= bound, (error, bound)

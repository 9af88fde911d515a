"""FP64 corner terms at offsets where their evaluation changes form: coordinates that are
exactly zero (stations on corner planes, mesh lines and corners), arguments of the logarithms
at or below the guard, stations inside the mesh, and far stations; every kind against the
oracle (data within 1e-12 of gz, 1e-11 of a component's largest magnitude, gradients within
1e-10, the bounds of the FP64 path's other parity tests)."""
import numpy as np
import pytest

from jif3d_amd import _native as nat
from jif3d_amd.imp import (ScalarHipGravityImp, TensorHipGravityImp, ScalarTensorHipGravityImp)
from jif3d_amd.model import ThreeDGravityModel, TensorGravityData

pytestmark = pytest.mark.gpu


def survey(which, rng):
    m = ThreeDGravityModel()
    m.SetMeshSize(5, 4, 3)
    m.SetXCellSizes([10.0, 20.0, 10.0, 15.0, 10.0])
    m.SetYCellSizes([10.0, 10.0, 30.0, 10.0])
    m.SetZCellSizes([8.0, 16.0, 32.0])
    m.SetDensities(rng.normal(size=60) * 100 + 2000)
    d = TensorGravityData()
    pts = {
        "x_plane": [(10.0, 7.3, -4.0), (30.0, 21.0, -1.0), (0.0, 33.0, -9.0)],
        "y_plane": [(7.0, 10.0, -4.0), (21.0, 20.0, -1.0)],
        "z_plane": [(7.0, 13.0, 0.0), (21.0, 23.0, 8.0), (-400.0, 23.0, 56.0)],
        "inside": [(7.0, 13.0, 3.0), (21.5, 23.5, 30.0)],
        "lines": [(10.0, 20.0, -4.0), (-50.0, 20.0, 8.0), (200.0, 20.0, 8.0), (10.0, 300.0, 8.0),
                  (10.0, -300.0, 24.0), (30.0, 20.0, 90.0)],
        "far": [(-3.0e4, 12.0, -3.0), (5.0e4, 2.0e4, -1.0e3), (12.0, 4.1e4, 7.0)],
    }[which]
    for p in pts:
        d.AddMeasurementPoint(*p)
    return m, d


@pytest.mark.parametrize("which", ["x_plane", "y_plane", "z_plane", "inside", "lines", "far"])
def test_edge_offsets_match_the_oracle(orc, which):
    rng = np.random.default_rng(11)
    m, d = survey(which, rng)
    mv = m.GetModelParameters()
    ref_g = orc.calculate(orc.SCALAR, m, mv, d.positions)
    ref_t = orc.calculate(orc.TENSOR, m, mv, d.positions)
    _, Jg = orc.calculate(orc.SCALAR, m, mv, d.positions, want_sens=True)
    _, Jt = orc.calculate(orc.TENSOR, m, mv, d.positions, want_sens=True)
    # where the reference's own terms cancel (far stations) the data are compared on the scale
    # of the corner sums that both evaluate: |sum| <= G max(rho) times the terms' magnitude
    reach = max(np.max(np.abs(p)) for p in d.positions) + 100.0
    scale_t = 6.67428e-11 * 2500.0 * 60 * 8 * np.log(2 * reach) * 2.0 ** -52
    scale_g = scale_t * 2 * reach
    gz = ScalarHipGravityImp().Calculate(m, d)
    t = TensorHipGravityImp().Calculate(m, d)
    both = ScalarTensorHipGravityImp().Calculate(m, d).reshape(-1, 10)
    ok = np.isfinite(ref_g)
    assert np.all(np.abs(gz - ref_g)[ok] <= 1e-12 * np.max(np.abs(ref_g[ok])) + scale_g)
    assert np.array_equal(np.isnan(gz), np.isnan(ref_g))
    assert np.all(np.abs(t - ref_t) <= 1e-11 * np.max(np.abs(ref_t)) + scale_t)
    assert np.all(np.abs(both[:, 1:].ravel() - ref_t) <= 1e-11 * np.max(np.abs(ref_t)) + scale_t)
    rows = TensorHipGravityImp().SensitivityRows(m, d)
    entry = 6.67428e-11 * 8 * np.log(2 * reach) * 2.0 ** -52
    assert np.all(np.abs(rows - Jt) <= 1e-12 * np.max(np.abs(Jt)) + entry)
    r = rng.normal(size=t.size)
    g = TensorHipGravityImp().LQDerivative(m, d, r)
    gref = 2.0 * Jt.T @ r
    bound = 1e-10 * np.max(np.abs(gref)) + 2 * entry * np.sum(np.abs(r)) * len(ref_g)
    assert np.all(np.abs(g - gref) <= bound)
    if np.all(np.isfinite(Jg)):
        rg = rng.normal(size=gz.size)
        gg = ScalarHipGravityImp().LQDerivative(m, d, rg)
        gref = 2.0 * Jg.T @ rg
        bound = 1e-10 * np.max(np.abs(gref)) + 4 * entry * reach * np.sum(np.abs(rg))
        assert np.all(np.abs(gg - gref) <= bound)

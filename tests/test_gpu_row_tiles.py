"""Sensitivity rows evaluated corner by corner in bricks of the mesh, at mesh sizes around the
bricks' edges (4 x 5 or 1 x 7 columns of at most 33 cells), for every kind against the oracle's rows, and
on a mesh whose cells do not share their corners (a gap beside a layer of cells), where every
cell takes its own eight corners and the other cells' entries stay the same.  Bounds of the FP64 path: 1e-12 of the largest entry for gz, 1e-11
for the tensor and magnetic kinds, plus, entry by entry, the rounding of the closed form itself:
an ulp of r changes the logarithm of u + r by eps r / (u + r), which is large for corners far
along a line that passes near the station.  The joint kind's rows are the gz rows and the tensor
rows."""
import numpy as np
import pytest

from jif3d_amd import _native as nat
from jif3d_amd.imp import (ScalarHipGravityImp, TensorHipGravityImp, ScalarTensorHipGravityImp,
                           HipMagneticSusceptibilityImp, HipMagneticGradImp, HipMagnetizationImp)
from jif3d_amd.model import (ThreeDGravityModel, ThreeDSusceptibilityModel,
                             ThreeDMagnetizationModel, TensorGravityData)

pytestmark = pytest.mark.gpu
FIELD = (0.9, 0.2, 48000.0)
MESHES = [(1, 1, 1), (4, 5, 33), (5, 6, 34), (9, 11, 1), (3, 2, 67), (8, 5, 66), (2, 7, 33), (3, 15, 35)]


def geometry(kind, dims, nsites=3):
    rng = np.random.default_rng(sum(dims))
    cls = {"mag": ThreeDSusceptibilityModel, "grad": ThreeDSusceptibilityModel,
           "magnetization": ThreeDMagnetizationModel}.get(kind, ThreeDGravityModel)
    m = cls()
    m.SetMeshSize(*dims)
    m.SetXCellSizes(np.full(dims[0], 20.0))
    m.SetYCellSizes(rng.integers(10, 30, dims[1]).astype(float))
    m.SetZCellSizes(10.0 + np.arange(dims[2]) / 4)
    if cls is ThreeDGravityModel:
        m.SetBackgroundThicknesses([30.0, 400.0])
        m.SetBackgroundDensities([1.0, 2.0])
    d = TensorGravityData()
    d.SetMeasurementPoints(rng.uniform(0, 20.0 * dims[0], nsites), rng.uniform(0, 60.0, nsites),
                           -rng.uniform(3, 20, nsites))
    return m, d


def implementation(kind):
    return {"gz": ScalarHipGravityImp, "ftg": TensorHipGravityImp,
            "joint": ScalarTensorHipGravityImp, "mag": lambda: HipMagneticSusceptibilityImp(*FIELD),
            "grad": lambda: HipMagneticGradImp(*FIELD),
            "magnetization": HipMagnetizationImp}[kind]()


def rounding(m, d, first):
    """Per station (from `first`) and cell: G sum over the corners of 4 ulp of each logarithm's
    argument through the rounding of r, in tensor units."""
    eps = np.finfo(float).eps
    x, y, z = (p[first:, None, None, None] for p in d.positions)
    X, Y, Z = np.meshgrid(*m.coords, indexing="ij")
    u = [x - X, y - Y, z - Z]
    r = np.sqrt(sum(v * v for v in u))
    f = sum(4 * eps * (1.0 + r / np.maximum(v + r, eps)) for v in u)
    for axis in (1, 2, 3):
        f = np.take(f, range(1, f.shape[axis]), axis) + np.take(f, range(f.shape[axis] - 1), axis)
    return 6.67428e-11 * f.reshape(len(f), -1)


def unit(kind):
    """Data units of a kind per tensor unit (gz terms are covered by their relative bound)."""
    g = 6.67428e-11
    return {"gz": 0.0, "ftg": 1.0, "joint": 1.0, "mag": FIELD[2] / (4 * np.pi * g),
            "grad": 2 * FIELD[2] * 1e-7 / g, "magnetization": 1e9 * 1e-7 / g}[kind]


def padded(noise, k, columns):
    """The cells' bounds repeated over the k rows of a station and over model blocks; zero for
    background columns."""
    n = noise.shape[1]
    if columns % n == 0:
        noise = np.tile(noise, (1, columns // n))
    else:
        noise = np.pad(noise, ((0, 0), (0, columns - n)))
    return np.repeat(noise, k, 0)


def check(orc, kind, m, d):
    rows = implementation(kind).SensitivityRows(m, d, 1, 2)
    okind = {"gz": orc.SCALAR, "ftg": orc.TENSOR, "mag": orc.MAGNETIC, "grad": orc.MAGGRAD,
             "magnetization": orc.MAGNETIZATION}[kind]
    _, J = orc.calculate(okind, m, m.GetModelParameters(), d.positions,
                         field=FIELD if kind in ("mag", "grad") else None, want_sens=True)
    J = J[len(J) // 3:]
    assert rows.shape == J.shape
    tol = 1e-12 if kind == "gz" else 1e-11
    noise = padded(unit(kind) * rounding(m, d, 1), len(J) // 2, J.shape[1])
    assert np.all(np.abs(rows - J) <= tol * np.max(np.abs(J)) + noise)


@pytest.mark.parametrize("dims", MESHES)
@pytest.mark.parametrize("kind", ["gz", "ftg", "mag", "grad", "magnetization"])
def test_bricks_match_the_oracle(orc, kind, dims):
    check(orc, kind, *geometry(kind, dims))


@pytest.mark.parametrize("kind", ["gz", "ftg", "mag", "grad", "magnetization"])
def test_cells_with_a_gap(kind):
    m, d = geometry(kind, (5, 6, 7))
    m.sizes[0][2] = 15.0  # the third cell ends 5 m before the fourth begins
    rows = implementation(kind).SensitivityRows(m, d)
    whole, _ = geometry(kind, (5, 6, 7))
    ref = implementation(kind).SensitivityRows(whole, d)
    cell = np.arange(5 * 6 * 7).reshape(5, 6, 7)
    other = np.delete(cell, 2, 0).ravel()
    scale = np.max(np.abs(ref))
    tol = 1e-12 if kind == "gz" else 1e-11
    assert np.max(np.abs(rows[:, other] - ref[:, other])) <= tol * scale
    short = cell[2].ravel()  # a quarter of these cells is missing
    assert np.max(np.abs(rows[:, short] - ref[:, short])) > 0.1 * np.max(np.abs(ref[:, short]))


@pytest.mark.parametrize("dims", MESHES)
def test_joint_rows_are_gz_and_tensor_rows(dims):
    m, d = geometry("joint", dims)
    both = implementation("joint").SensitivityRows(m, d).reshape(d.nsites, 10, -1)
    gz = implementation("gz").SensitivityRows(m, d)
    t = implementation("ftg").SensitivityRows(m, d).reshape(d.nsites, 9, -1)
    assert np.max(np.abs(both[:, 0] - gz)) <= 1e-12 * np.max(np.abs(gz))
    noise = padded(rounding(m, d, 0), 9, t.shape[2]).reshape(t.shape)
    assert np.all(np.abs(both[:, 1:] - t) <= 1e-11 * np.max(np.abs(t)) + noise)

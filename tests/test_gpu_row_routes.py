"""Which kernel evaluates sensitivity rows: bricks of cells that share their corners on deep
meshes, every cell by itself on flat and thin ones (where a brick's workgroup has too little to do),
whatever the number of sites; and either side of the line against the oracle's rows."""
import numpy as np
import pytest

from jif3d_amd import _native as nat
from test_gpu_row_tiles import check, geometry, implementation

pytestmark = pytest.mark.gpu
KINDS = {"gz": nat.KIND_SCALAR, "ftg": nat.KIND_TENSOR, "joint": nat.KIND_SCALAR_TENSOR,
         "mag": nat.KIND_MAGNETIC, "grad": nat.KIND_MAGNETIC_GRADIENT,
         "magnetization": nat.KIND_MAGNETIZATION}
# layers of a 64 x 63 mesh: the last that cells take by themselves (and a little), the first of bricks
LINE = {"gz": (8, 16), "ftg": (10, 20), "joint": (3, 8), "mag": (10, 20), "grad": (10, 20),
        "magnetization": (1, 5)}


def route(kind, dims, nsites):
    m, d = geometry(kind, dims, max(nsites, 3))
    ctx = nat.Context()
    ctx.configure(m, d, (0.9, 0.2, 48000.0) if kind in ("mag", "grad") else None)
    K = KINDS[kind]
    rows = ctx.alloc((nsites * nat.RAW_PER_SITE[K], ctx.model_size(K)))
    ctx.profile_enable(True)
    ctx.sensitivity_rows(K, 0, nsites, rows)
    names = set(ctx.profile())
    out = rows.to_host()
    rows.free()
    return names, out


@pytest.mark.parametrize("kind", sorted(KINDS))
def test_flat_and_thin_meshes_take_cells(kind):
    flat, deep = LINE[kind]
    cells, bricks = {"sensitivity_rows_cells_fp64"}, {"sensitivity_rows_bricks_fp64"}
    assert route(kind, (64, 63, 1), 3)[0] == cells
    assert route(kind, (64, 63, flat), 3)[0] == cells
    names, three = route(kind, (64, 63, deep), 3)
    assert names == bricks
    one = route(kind, (64, 63, deep), 1)[1]
    assert np.array_equal(one, three[:len(one)])
    if kind != "magnetization":
        assert route(kind, (1, 1, 4000), 1)[0] == cells


@pytest.mark.parametrize("kind", sorted(set(KINDS) - {"joint"}))
@pytest.mark.parametrize("side", [0, 1])
def test_either_side_matches_the_oracle(orc, kind, side):
    dims = (64, 63, LINE[kind][side])
    check(orc, kind, *geometry(kind, dims))


@pytest.mark.parametrize("side", [0, 1])
def test_joint_rows_are_gz_and_tensor_rows(side):
    m, d = geometry("joint", (64, 63, LINE["joint"][side]))
    both = implementation("joint").SensitivityRows(m, d).reshape(d.nsites, 10, -1)
    gz = implementation("gz").SensitivityRows(m, d)
    assert np.max(np.abs(both[:, 0] - gz)) <= 1e-12 * np.max(np.abs(gz))

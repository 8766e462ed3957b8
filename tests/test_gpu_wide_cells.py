"""Cells far wider than the cut-off: the FP32 records' resolution grows with
the cell, and a shell that it mistakes is found again in FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def boundary(tmp_path_factory):
    import screen_cases

    return screen_cases.boundary_system(tmp_path_factory.mktemp("boundary"))


# the pairs on the screen's decision boundaries, `spacing` A from each other,
# in cells of 11, 55, 275, 1 500 and 6 000 A
@pytest.mark.parametrize("spacing,cells", [(22, 20), (110, 20), (110, 4), (600, 4), (2400, 4)])
def test_bulk_prediction_matches_oracle(require_gpu, boundary, spacing, cells):
    import screen_cases
    from conftest import fast_bulk_vs_oracle
    from sdmd_amd.engine import System

    system, exps, _ = boundary
    arr = system.arrays.copy()
    a, sc = arr.arr, arr.scalars
    g = int(np.ceil(len(exps) ** (1 / 3)))
    e = np.repeat(np.arange(len(exps)), system.natom // len(exps))
    for k, (f, at) in enumerate(zip(("x", "y", "z"), (e % g, (e // g) % g, e // (g * g)))):
        a[f][1:] += (spacing - screen_cases.SPACING) * at
        sc["box"][k] = g * spacing
        sc["cellnum"][k] = cells
        sc["cellsize"][k] = sc["box"][k] / cells
    a["celllist"] = np.zeros(sc["natom"] + cells ** 3 + 1, np.int32)
    sc["ncelllist"] = len(a["celllist"])
    screen_cases.relink(arr)
    fast_bulk_vs_oracle(System(None, arr))

"""Validation mode compares a screened prediction with a scan that shares
nothing with it but the cell arrays: a candidate that the screened path does
not look at (its cell taken to be out of reach) shows as a disagreement."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COLI = 0


def _relist(arr, j, cell):
    """Atom j out of its cell's list and into that of `cell` (x, y, z)."""
    a, sc = arr.arr, arr.scalars
    N, n = sc["natom"], list(sc["cellnum"])
    number = lambda c: (c[2] * n[1] + c[1]) * n[0] + c[0] + 1
    cl = a["celllist"]
    k = N + number([a[f][j] for f in ("cellx", "celly", "cellz")])
    while cl[k] != j:
        k = cl[k]
    cl[k] = cl[j]
    k = N + number(cell)
    cl[j], cl[k] = cl[k], j
    a["cellx"][j], a["celly"][j], a["cellz"][j] = cell


@pytest.fixture(scope="module")
def wide_cells(tmp_path_factory):
    """The dense chain in 4 x 4 x 4 cells of 18 A, cut-off 12 A (scan radius 10.8 A)."""
    import screen_cases
    from sdmd_amd import builder
    from sdmd_amd.engine import System

    d = tmp_path_factory.mktemp("widecells")
    builder.write_input_dir(builder.single_chain(["TRP", "ARG", "LYS", "PHE", "TYR"] * 6, 8, 72.0), str(d), cutoff=12.0,
                            thermostat="no")
    s = System.load(str(d))
    arr = s.arrays
    sc, a = arr.scalars, arr.arr
    for k in range(3):
        sc["cellnum"][k] = 4
        sc["cellsize"][k] = sc["box"][k] / 4
    a["celllist"] = np.zeros(sc["natom"] + 65, np.int32)
    sc["ncelllist"] = len(a["celllist"])
    screen_cases.relink(arr)
    return s


def _predicted(system, **kw):
    from sdmd_amd.engine import GpuEngine

    eng = GpuEngine([system], mode="fast", validate=True, **kw)
    eng.prepare()
    st, fs = eng.state(0).arr, eng.fast_stats(0)
    eng.close()
    return st, fs


@pytest.mark.parametrize("block", [64, 256, 512])
def test_validation_sees_a_candidate_out_of_the_screens_reach(require_gpu, wide_cells, block):
    from sdmd_amd.engine import System

    st, fs = _predicted(wide_cells, block=block)
    n = wide_cells.natom
    assert fs["validated"] == fs["agree"] == n
    # atoms whose event is a collision with an atom of their own cell, in the
    # half of the cell from which the next cell (along x) is out of reach
    sc, lost = wide_cells.arrays.scalars, 0
    L = sc["cellsize"][0]
    for i in range(1, n + 1):
        j = int(st["ev_partner"][i])
        c = [int(st[f][i]) for f in ("cellx", "celly", "cellz")]
        if st["ev_type"][i] != COLI or st["x"][i] - c[0] * L > L - 11.0 or not 1 <= c[0] <= 2:
            continue
        if c != [int(st[f][j]) for f in ("cellx", "celly", "cellz")]:
            continue
        arr = wide_cells.arrays.copy()
        _relist(arr, j, [c[0] + 1, c[1], c[2]])
        bad, fs = _predicted(System(None, arr), block=block)
        assert fs["validated"] == n
        if bad["ev_partner"][i] != j or bad["ev_type"][i] != COLI:       # the screened path lost it
            assert fs["agree"] < n
            lost += 1
        if lost == 3:
            break
    assert lost == 3

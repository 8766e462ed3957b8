"""The plain engine's postponed position steps and its cell arrays: a run cut
into pieces (every piece ends with all atoms at its time) and a run mixed
with single operations (which work on that state) reach the state of one
run, bit for bit."""
import numpy as np
import pytest

from conftest import golden_system

pytestmark = pytest.mark.gpu

FIELDS = ("x", "y", "z", "vx", "vy", "vz", "ev_time", "ev_pot", "ev_partner", "ev_type", "ev_sub", "ev_counter",
          "ev_pcounter", "celllist", "cellx", "celly", "cellz", "hb_bond", "type")


def engine(name, pops, block):
    from sdmd_amd.engine import GpuEngine

    eng = GpuEngine([golden_system(name)[0]], block=block, max_pops=pops)
    eng.prepare()
    return eng


def assert_same(a, b):
    for f in FIELDS:
        assert np.array_equal(a.state(0).arr[f], b.state(0).arr[f]), f
    for x, y in zip(a.tree(0), b.tree(0)):
        assert np.array_equal(x, y)
    assert a.stats(0)["pops"] == b.stats(0)["pops"] and a.stats(0)["error"] == b.stats(0)["error"] == 0


# 59 atoms (a sweep every 8 pops), 1 695 (every 26), 431 with cells above and
# below the 64 atoms a cell array holds
@pytest.mark.parametrize("name,block", [("ala10helix", 64), ("cyl8x20", 256), ("dense30", 128), ("mix4x20", 512)])
def test_pieces_equal_one_run(require_gpu, name, block):
    pieces = [1, 2, 7, 8, 9, 25, 26, 27, 31, 32, 33, 64, 500, 1235]
    whole, cut = engine(name, sum(pieces), block), engine(name, sum(pieces), block)
    whole.run(sum(pieces))
    for n in pieces:
        cut.run(n)
    assert_same(whole, cut)
    whole.close()
    cut.close()


@pytest.mark.parametrize("name", ["dense30", "ala10cyl"])
def test_single_operations_between_runs(require_gpu, name):
    whole, mixed = engine(name, 1300, 256), engine(name, 1300, 256)
    whole.run(1300)
    done = 0
    while done < 1300:
        mixed.run(min(60, 1300 - done))
        done += min(60, 1300 - done)
        for _ in range(min(5, 1300 - done)):
            ev = mixed.pop(0)
            partner = max(ev["partner"], 0)
            mixed.advance(0, ev["time"])
            renew = [ev["target"]]
            if not ev["stale"]:
                mixed.do_event(0, ev["target"], partner)
                renew += [partner] if partner else []
            mixed.predict(0, renew)
            mixed.update_tree(0, renew)
            done += 1
    for f in FIELDS:
        assert np.array_equal(whole.state(0).arr[f], mixed.state(0).arr[f]), f
    whole.close()
    mixed.close()


# helix: H bonds formed (records that depend on H-bond slots); window 5: every
# atom predicted in windows; 0.9 of the box edge from a wall; an odd and an
# even number of atoms
@pytest.mark.parametrize("name,pops,window", [("ala10helix", 0, 0), ("ala10helix", 3000, 0), ("mix4x20", 2000, 0),
                                              ("cyl8x20", 3001, 0), ("dense30", 500, 0), ("dense30", 500, 100),
                                              ("ala10cyl", 1000, 5)])
def test_bulk_prediction_of_evolved_states(require_gpu, name, pops, window):
    """The bulk prediction of a state reached by a run, atom for atom and
    the tree, as the oracle predicts it in order."""
    import oracle_lib
    from sdmd_amd.engine import GpuEngine, System

    eng = engine(name, pops + 10, 256)
    eng.run(pops)
    arr = eng.state(0)
    eng.close()
    sysm = System(None, arr)
    again = GpuEngine([sysm, sysm], window=window, max_pops=10)     # two systems share the launch
    again.prepare()
    o = oracle_lib.Oracle(arr)
    assert o.bulk() == 0
    ref = o.state()
    for k in range(2):
        got = again.state(k)
        for f in ("ev_partner", "ev_type", "ev_sub", "ev_time", "ev_pot", "ev_pcounter", "nb_partnernum", "hb_itype"):
            assert np.array_equal(got.arr[f][1:], ref.arr[f][1:]), (k, f)
        assert again.stats(k)["error"] == 0
    again.close()

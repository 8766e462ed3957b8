"""A plain run that ends in an error stops at the pop that made it: the
context holds the state of that pop, and nothing of the next one."""
import numpy as np
import pytest

from conftest import golden_system
from sdmd_amd._lib import SdmdError

pytestmark = pytest.mark.gpu

STATE = ("x", "y", "z", "vx", "vy", "vz", "cellx", "celly", "cellz", "celllist", "hb_bond", "type", "ev_counter")
RECORD = ("ev_partner", "ev_type", "ev_sub", "ev_time", "ev_pot", "ev_pcounter")
THER, INVD = 4, 15
SUBTYPE, NORMALS = 3, 12      # device error codes
POPS = 1500


def run(draws, pops, block=256):
    from sdmd_amd.engine import GpuEngine

    s, _ = golden_system("ala10ext")
    eng = GpuEngine([s], block=block, trace=True, trace_capacity=POPS)
    eng.feed_normals(draws)
    eng.prepare()
    if pops:
        eng.run(pops)
        return eng
    with pytest.raises(SdmdError):
        eng.run(POPS)
    return eng


# the stream ends in a prediction: 1 to 6 draws more end it in other pops, at
# the first or the second atom of two
@pytest.mark.parametrize("block", [64, 256])
@pytest.mark.parametrize("more", range(1, 7))
def test_normals_used_up_in_a_prediction(require_gpu, more, block):
    short = run(59 + 300 + more, 0, block)
    st = short.stats(0)
    whole = run(20000, st["pops"], block)
    want, last = whole.stats(0), whole.trace(0)[-1]
    assert st["error"] == NORMALS and 0 < st["pops"] < POPS
    assert want["normals_used"] > 59 + 300 + more         # that pop's predictions lacked a draw
    assert st["frame"] + st["recal"] == st["pops"]
    for f in ("pops", "frame", "recal", "currenttime", "last_exec"):
        assert st[f] == want[f], f
    assert np.array_equal(st["per_type"], want["per_type"])
    assert len(short.trace(0)) == st["pops"]
    got, ref = short.state(0).arr, whole.state(0).arr
    for f in STATE:
        assert np.array_equal(got[f], ref[f]), f
    # every record but those of that pop
    others = np.setdiff1d(np.arange(1, 60), [last["r"][k]["atom"] for k in range(last["nrenew"])])
    for f in RECORD:
        assert np.array_equal(got[f][others], ref[f][others]), f
    assert np.all(got["ev_type"][1:] != INVD)
    short.close()
    whole.close()


# ... in a thermostat event: the clock and the positions are at the event, the
# records as before it
@pytest.mark.parametrize("have", [0, 1, 2])
def test_normals_used_up_in_an_event(require_gpu, have):
    whole = run(20000, POPS)
    tr = whole.trace(0)
    whole.close()
    pop = int(np.flatnonzero((tr["type"] == THER) & (tr["exec"] == 1) & (np.arange(len(tr)) > 100))[0])
    before = run(20000, pop)
    used, ref = before.stats(0)["normals_used"], before.state(0).arr
    before.close()
    short = run(used + have, 0)
    st, got = short.stats(0), short.state(0).arr
    assert st["error"] == NORMALS and st["pops"] == pop and st["frame"] + st["recal"] == pop + 1
    assert len(short.trace(0)) == pop
    short.close()
    for f in RECORD:
        if f != "ev_time":
            assert np.array_equal(got[f][1:], ref[f][1:]), f
    assert np.array_equal(got["ev_time"][1:], ref["ev_time"][1:] - tr["dt"][pop])


# a context in error still predicts: the records and the tree of its state,
# while the call reports the error
def test_prepare_of_a_context_in_error(require_gpu):
    import oracle_lib

    eng = run(59 + 300, 0)
    o = oracle_lib.Oracle(eng.state(0))
    assert o.bulk() == 0
    ref = o.state().arr
    eng.feed_normals(1000)
    with pytest.raises(SdmdError):
        eng.prepare()
    got = eng.state(0).arr
    for f in RECORD:
        assert np.array_equal(got[f][1:], ref[f][1:]), f
    node, leaf = eng.tree(0)
    eng.close()
    want, wleaf = o.tree()
    assert np.array_equal(node[1:], want[1:]) and np.array_equal(leaf[1:], wleaf[1:])


# a record that no event can be made of: the clock moves on, the records stay
@pytest.mark.parametrize("ty", [0, 1])
def test_bad_record(require_gpu, ty):
    from sdmd_amd.engine import GpuEngine, System

    s, _ = golden_system("ala10ext")
    eng = GpuEngine([s], max_pops=100)
    eng.prepare()
    node, _ = eng.tree(0)
    arr = eng.state(0)
    eng.close()
    a = arr.arr
    t = int(node[1])
    assert a["ev_partner"][t] > 0
    a["ev_type"][t], a["ev_sub"][t] = ty, 8
    eng = GpuEngine([System(None, arr)], max_pops=100)
    eng.create_tree(0)
    with pytest.raises(SdmdError):
        eng.run(10)
    st, got = eng.stats(0), eng.state(0).arr
    eng.close()
    assert st["error"] == SUBTYPE and st["pops"] == 0
    for f in RECORD:
        if f != "ev_time":
            assert np.array_equal(got[f][1:], a[f][1:]), f
    assert np.array_equal(got["ev_time"][1:], a["ev_time"][1:] - a["ev_time"][t])

"""The plain bulk prediction of states whose records depend on what an atom
carries besides its position: H bonds and their neighbour slots, and the flag
that a skipped H-bond event leaves (the next prediction leaves HBTime out
once, TimePrediction.c:309-330)."""
import numpy as np
import pytest

import oracle_lib
from conftest import golden_system

pytestmark = pytest.mark.gpu

HB, HBSKIP = 2, 3             # SDMD_HB, SDMD_HBSKIP
FIELDS = ("ev_partner", "ev_type", "ev_sub", "ev_time", "ev_pot", "ev_pcounter", "nb_partnernum", "hb_itype")


@pytest.fixture(scope="module")
def helix():
    """States of the helix run just before H-bond events of atoms 35 and 55
    (pop numbers found with the oracle): pop -> state."""
    s, _ = golden_system("ala10helix")
    o = oracle_lib.Oracle(s.arrays)
    o.bulk()
    out, done = {}, 0
    for pop in (9270, 24009, 35568):
        o.run(pop - done, trace=False)
        out[pop], done = o.state(), pop
    return out


@pytest.mark.parametrize("skip", ["none", "higher", "lower", "all"])
@pytest.mark.parametrize("pop", [9270, 24009, 35568])
def test_bulk_prediction_with_hbonds_and_skips(require_gpu, helix, pop, skip):
    from sdmd_amd.engine import GpuEngine, System

    arr = helix[pop].copy()
    N = arr.scalars["natom"]
    assert (arr.arr["hb_bond"][1:] > 0).sum() >= 2 and (arr.arr["nb_status"][1:] > 0).sum() >= 4
    arr.arr["hb_itype"][{"none": [], "higher": [55], "lower": [35], "all": np.arange(1, N + 1)}[skip]] = HBSKIP
    o = oracle_lib.Oracle(arr)
    assert o.bulk() == 0
    ref = o.state().arr
    # the earliest event is theirs; flagged, an atom leaves it out, while the
    # lower one's record names the higher one
    assert (ref["ev_type"][55] == HB) == (skip in ("none", "lower"))
    assert (ref["ev_type"][35] == HB) == (skip in ("none", "higher"))
    eng = GpuEngine([System(None, arr)], max_pops=10)
    eng.prepare()
    got = eng.state(0).arr
    assert eng.stats(0)["error"] == 0
    eng.close()
    for f in FIELDS:
        assert np.array_equal(got[f][1:], ref[f][1:]), (f, np.flatnonzero(got[f] != ref[f]))

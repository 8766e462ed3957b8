"""The plain engine's prediction in windows of candidates: a run through H
bonds formed, broken and skipped reaches the state of the unwindowed run, bit
for bit, whatever the window (from a few candidates to just below and above a
neighbourhood's 59)."""
import numpy as np
import pytest

import oracle_lib
from conftest import golden_system

pytestmark = pytest.mark.gpu

HB = 2


@pytest.fixture(scope="module")
def helix():
    from sdmd_amd.engine import GpuEngine, System

    s, _ = golden_system("ala10helix")
    o = oracle_lib.Oracle(s.arrays)
    o.bulk()
    o.run(54000, trace=False)
    system = System(None, o.state())

    def run(**kw):
        eng = GpuEngine([system], trace=True, trace_capacity=8000, max_pops=8000, **kw)
        eng.prepare()
        eng.run(8000)
        out = eng.state(0).arr, eng.stats(0), eng.trace(0)
        eng.close()
        return out

    return run, run()


@pytest.mark.parametrize("window,block", [(5, 64), (17, 256), (58, 64), (58, 512), (59, 256)])
def test_windows_keep_the_trajectory(require_gpu, helix, window, block):
    run, (ref, sref, tref) = helix
    assert (tref["type"] == HB).sum() >= 10
    got, st, tr = run(window=window, block=block)
    assert st["error"] == 0
    for f in ("pops", "frame", "recal", "pair_evals", "candidates"):
        assert st[f] == sref[f], f
    assert np.array_equal(tr, tref)
    for f in ("x", "vx", "ev_time", "ev_partner", "ev_type", "ev_sub", "ev_pcounter", "hb_bond", "hb_itype", "nb_status"):
        assert np.array_equal(got[f], ref[f]), f


# every atom a neighbour of every other one (3 cells of 55 A per edge, up to
# some 300 atoms in a cell): fewer and more than the 6 144 candidates whose
# lists are walked once
@pytest.mark.parametrize("chains", [16, 21])
def test_wide_neighbourhoods_match_oracle(require_gpu, tmp_path, chains):
    import copy

    from sdmd_amd import builder
    from sdmd_amd.engine import GpuEngine, System

    unique = builder.build_chains(builder.random_sequences(2, 30, 4), 4, workers=1)
    placed = builder.place_chains([copy.deepcopy(unique[k % 2]) for k in range(chains)], (165.0,) * 3,
                                  np.random.default_rng([4, 0]))
    builder.write_input_dir(builder.System(placed, (165.0,) * 3, "peptides"), str(tmp_path), cutoff=54.0)
    s = System.load(str(tmp_path))
    assert (s.natom > 6144) == (chains == 21) and list(s.arrays.scalars["cellnum"]) == [3, 3, 3]
    o = oracle_lib.Oracle(s.arrays)
    assert o.bulk() == 0
    ref, _ = o.run(150)
    eng = GpuEngine([s], trace=True, trace_capacity=150, max_pops=150)
    eng.prepare()
    eng.run(150)
    tr, st = eng.trace(0), eng.stats(0)
    eng.close()
    assert st["error"] == 0
    for f in ("target", "partner", "type", "sub", "exec", "dt", "pot"):
        assert np.array_equal(tr[f], ref[f]), f

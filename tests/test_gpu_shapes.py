"""Workgroup shapes of the fast engine: with a number of helper workgroups
asked for, every block size runs as asked (the automatic number goes with the
automatic shape); all reach the same state, screened as the FP64 scan."""
import numpy as np
import pytest

from conftest import STATE_FIELDS

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def runs(tmp_path_factory):
    from sdmd_amd import builder
    from sdmd_amd.engine import GpuEngine, System

    d = tmp_path_factory.mktemp("shapes")
    builder.write_input_dir(builder.random_peptides(12, 30, seed=11, mM=5.0), str(d), cutoff=7.25)
    s = System.load(str(d))

    def run(block, helpers, validate=False, t=1.0):
        eng = GpuEngine([s], block=block, mode="fast", helpers=helpers, validate=validate)
        eng.prepare()
        eng.run_until(t)
        out = eng.state(0).arr, eng.stats(0), eng.fast_stats(0)
        eng.close()
        return out

    return run, run(256, -1)


@pytest.mark.parametrize("helpers", [-1, 1, 5])
@pytest.mark.parametrize("block", [64, 256, 512, 1024])
def test_shapes_keep_the_trajectory(require_gpu, runs, block, helpers):
    run, (ref, sref, fref) = runs
    st, s, fs = run(block, helpers)
    assert s["error"] == 0 and fs["causal"] == 0 and fs["helpers"] == max(helpers, 0)
    assert s["frame"] == sref["frame"] > 10000 and s["pair_evals"] == sref["pair_evals"]
    for f in STATE_FIELDS:
        assert np.array_equal(st[f], ref[f]), f


@pytest.mark.parametrize("block", [64, 256, 512, 1024])
def test_shapes_agree_with_fp64(require_gpu, runs, block):
    run, _ = runs
    st, s, fs = run(block, 3, validate=True, t=0.3)
    assert s["error"] == 0 and fs["causal"] == 0
    assert fs["agree"] == fs["validated"] > 3000, fs

"""The fast engine's list of candidates inside the scan radius: shorter than
a wavefront, several wavefronts long, and longer than the list holds (the
unlisted path), on every workgroup shape that has its own list length."""
import copy

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dense(tmp_path_factory):
    from sdmd_amd import builder
    from sdmd_amd.engine import System

    geometry = builder.single_chain(["TRP", "ARG", "LYS", "PHE", "TYR"] * 6, 8, 72.0)
    out = {}
    for cutoff in (8.0, 12.0, 18.0):
        d = tmp_path_factory.mktemp("dense%d" % cutoff)
        builder.write_input_dir(geometry, str(d), cutoff=cutoff, thermostat="no")
        out[cutoff] = System.load(str(d))
    return out


# cut-off 8, 12, 18 A: up to about 60, 170, 350 atoms inside the scan radius
@pytest.mark.parametrize("cutoff", [8.0, 12.0, 18.0])
def test_bulk_prediction_matches_oracle(require_gpu, dense, cutoff):
    from conftest import fast_bulk_vs_oracle

    fast_bulk_vs_oracle(dense[cutoff])


@pytest.mark.parametrize("cutoff,block,helpers", [(12.0, 64, -1), (12.0, 512, -1), (12.0, 1024, -1), (18.0, 256, 0),
                                                  (18.0, 512, -1), (18.0, 1024, -1)])
def test_screens_agree_with_fp64(require_gpu, dense, cutoff, block, helpers):
    from sdmd_amd.engine import GpuEngine

    eng = GpuEngine([dense[cutoff]], block=block, mode="fast", validate=True, helpers=helpers)
    eng.prepare()
    eng.run_events(1500)
    st, fs = eng.stats(0), eng.fast_stats(0)
    assert st["error"] == 0 and fs["causal"] == 0
    assert fs["validated"] > 1500 and fs["agree"] == fs["validated"], fs
    eng.close()


# one cut-off wider than 2 048 candidates (two windows of first-candidate
# marks) in cells of up to a few hundred atoms: 5 014 atoms in 27 cells
def test_many_candidates_match_oracle(require_gpu, tmp_path):
    from conftest import fast_bulk_vs_oracle
    from sdmd_amd import builder
    from sdmd_amd.engine import System

    chains = builder.build_chains(builder.random_sequences(2, 30, 4), 4, workers=1)
    unit = [copy.deepcopy(chains[k % 2]) for k in range(16)]
    edge = 165.0
    placed = builder.place_chains(unit, (edge,) * 3, np.random.default_rng([4, 0]))
    d = tmp_path / "wide"
    builder.write_input_dir(builder.System(placed, (edge,) * 3, "peptides"), str(d), cutoff=54.0, thermostat="no")
    s = System.load(str(d))
    assert s.natom > 4000 and min(s.arrays.scalars["cellnum"][:]) == 3
    fast_bulk_vs_oracle(s)

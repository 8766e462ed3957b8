"""The fast engine's list of candidates inside the scan radius: shorter than
a wavefront, several wavefronts long, and longer than the list holds (the
unlisted path), on every workgroup shape that has its own list length."""
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

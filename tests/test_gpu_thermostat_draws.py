"""The fast engine's thermostat times: a draw is worked out in full only where
its lower bound can be the atom's earliest event, and the events are those of
the draws all the same."""
import numpy as np
import pytest

from conftest import golden_system

pytestmark = pytest.mark.gpu

THER = 4


def philox_normals(seed, system, atoms, draw):
    """Philox4x32-10 (key: seed and system; counter: atom, draw) and Box-Muller in FP64."""
    M = np.uint64(0xffffffff)
    key1 = (seed >> 32) ^ ((0x9E3779B9 * (system + 1)) & 0xffffffff)
    k = [np.uint64(seed & 0xffffffff), np.uint64(key1)]
    c = [atoms.astype(np.uint64), np.full(len(atoms), draw, np.uint64), np.full(len(atoms), 0x5344, np.uint64),
         np.full(len(atoms), 0x4d44, np.uint64)]
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ k[0], p1 & M, (p0 >> np.uint64(32)) ^ c[3] ^ k[1], p0 & M]
        k = [(k[0] + np.uint64(0x9E3779B9)) & M, (k[1] + np.uint64(0xBB67AE85)) & M]
    u = [(((a << np.uint64(32)) | b) >> np.uint64(11)).astype(np.float64) for a, b in ((c[0], c[1]), (c[2], c[3]))]
    u1, u2 = (u[0] + 0.5) * 2.0 ** -53, (u[1] + 0.5) * 2.0 ** -53
    return np.sqrt(-2 * np.log(u1)) * np.cos(2 * np.pi * u2)


# thermo_freq from far above the other events' times (few thermostat events)
# to far below (nearly all): every side of the bound decides somewhere
@pytest.mark.parametrize("freq", [3.0, 0.3, 0.03, 3e-3, 1e-4])
def test_thermostat_times_are_the_draws(require_gpu, freq):
    from sdmd_amd.engine import GpuEngine, System

    s, _ = golden_system("cyl8x20")
    seeds = range(101, 121)                 # 20 systems of 1 695 atoms

    def predicted(thermostat):
        systems = []
        for _ in seeds:
            arr = s.arrays.copy()
            arr.scalars.update(thermostat=thermostat, thermo_freq=freq, currenttime=0.0)
            systems.append(System(None, arr))
        eng = GpuEngine(systems, mode="fast", seed=(7 << 32) + 12345)
        eng.prepare()
        out = [eng.state(k) for k in range(len(systems))]
        eng.close()
        return [(st.arr["ev_type"][1:], st.arr["ev_time"][1:] + st.scalars["currenttime"]) for st in out]

    seen = 0
    for k, ((ty, t), (ty0, t0)) in enumerate(zip(predicted(1), predicted(0))):
        tt = freq * np.abs(philox_normals((7 << 32) + 12345, k, np.arange(1, len(t) + 1), 0))
        first = tt < t0
        assert np.array_equal(ty == THER, first), k
        assert np.array_equal(ty[~first], ty0[~first])
        # the snapshot time is taken off and added again: 2^-52 of it twice
        np.testing.assert_allclose(t, np.where(first, tt, t0), rtol=1e-12, atol=1e-15)
        seen += int(first.sum())
    assert seen > 0

"""The bulk prediction of more atoms than a grid of 32-atom pieces holds
(65 536 in its second dimension): 33 x 33 x 33 copies of the alanine 10-mer,
each predicted as one alone."""
import numpy as np
import pytest

import oracle_lib
from conftest import golden_system

pytestmark = pytest.mark.gpu


def copies(arr, k):
    """k^3 copies of a system side by side, in order of their atoms."""
    out = arr.copy()
    a, sc = out.arr, out.scalars
    n, m = sc["natom"], k ** 3
    box, num = np.array(sc["box"][:]), np.array(sc["cellnum"][:])
    at = np.stack(np.unravel_index(np.arange(m), (k, k, k)))               # copy -> its box
    first = n * np.arange(m)

    def tile(f, per=1, add=None):
        v = np.tile(a[f][per:].reshape(1, -1), (m, 1))
        if add is not None:
            v = np.where(v > 0, v + add[:, None], v)
        a[f] = np.concatenate([a[f][:per], v.ravel().astype(a[f].dtype)])

    for d, (x, c) in enumerate(zip(("x", "y", "z"), ("cellx", "celly", "cellz"))):
        v = a[x][1:][None] + (box[d] * at[d])[:, None]
        w = a[c][1:][None] + (num[d] * at[d])[:, None]
        a[x], a[c] = np.concatenate([a[x][:1], v.ravel()]), np.concatenate([a[c][:1], w.ravel().astype(np.int32)])
    old, N = a["celllist"], n * m
    for f in ("vx", "vy", "vz", "mass", "type", "aatype", "aanum", "hb_role", "hb_itype", "nb_partnernum", "nb_status",
              "ev_counter", "ev_pcounter", "ev_time", "ev_pot", "ev_type", "ev_sub"):
        tile(f)
    for f in ("hb_neighbor", "hb_bond", "ev_partner"):
        tile(f, add=first)
    tile("protein", add=np.arange(m) * sc["nprotein"])
    tile("nb_partner", 5, first)
    tile("dyn_j", 8, first)
    tile("dyn_bits", 8)
    for f, js, more in (("bond_off", "bond_j", ("bond_dmin", "bond_dmax")), ("con_off", "con_j", ("con",)),
                        ("cmap_off", "cmap_j", ("cmap_bits",))):
        off, e = a[f], len(a[js])
        a[f] = np.concatenate([off[:1], (off[1:n + 1][None] + e * np.arange(m)[:, None]).ravel(), [e * m]]).astype(np.int32)
        a[js] = (a[js][None] + first[:, None]).ravel().astype(np.int32)
        for g in more:
            a[g] = np.tile(a[g], m)
    cells = np.stack(np.unravel_index(np.arange(num.prod()), num[::-1]))[::-1]        # x fastest
    here = [cells[d][None] + (num[d] * at[d])[:, None] for d in range(3)]
    number = (here[2] * (k * num[1]) + here[1]) * (k * num[0]) + here[0] + 1
    shifted = lambda v: np.where(v > 0, v[None] + first[:, None], 0).ravel()
    a["celllist"] = np.zeros(N + m * num.prod() + 1, np.int32)
    a["celllist"][1:N + 1] = shifted(old[1:n + 1])
    a["celllist"][N + number.ravel()] = shifted(old[n + 1:])
    sc.update(natom=N, nprotein=sc["nprotein"] * m, ncelllist=len(a["celllist"]))
    for d in range(3):
        sc["box"][d], sc["cellnum"][d] = box[d] * k, int(num[d] * k)
    return out


@pytest.mark.parametrize("k", [2, 33])
def test_every_copy_is_predicted_as_one_alone(require_gpu, k):
    from sdmd_amd.engine import GpuEngine, System

    s, _ = golden_system("ala10nve")
    o = oracle_lib.Oracle(s.arrays)
    assert o.bulk() == 0
    ref = o.state().arr
    arr = copies(s.arrays, k)
    N = arr.scalars["natom"]
    assert (N > 32 * 65535) == (k == 33)
    eng = GpuEngine([System(None, arr)])
    eng.prepare()
    got, node = eng.state(0).arr, eng.tree(0)[0]
    assert eng.stats(0)["error"] == 0
    eng.close()
    of = lambda f: got[f][1:].reshape(-1, s.natom)
    partner = of("ev_partner")
    partner = np.where(partner > 0, partner - s.natom * np.arange(k ** 3)[:, None], partner)
    assert np.array_equal(partner, np.tile(ref["ev_partner"][1:], (k ** 3, 1)))
    for f in ("ev_type", "ev_sub"):
        assert np.array_equal(of(f), np.tile(ref[f][1:], (k ** 3, 1))), f
    assert np.array_equal(of("ev_time")[0], ref["ev_time"][1:])
    # 1 650 A away positions are rounded to 2^-43 A, which a time just before contact feels
    assert np.abs(of("ev_time") / ref["ev_time"][1:] - 1).max() < 1e-6
    assert got["ev_time"][node[1]] == got["ev_time"][1:].min()

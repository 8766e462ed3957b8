"""What the event engine is timed on: seeded peptide systems run through the
package's public entry points (GpuEngine, Remd).

A case is a dict of plain values:

  path      "abi"   pops driven one call at a time through the fine-grained
                    entry points (pop, advance, do_event, predict,
                    update_tree): the drop-in use from a host event loop
            "pops"  the event loop on the device for a number of pops
            "until" the event loop on the device up to a time, then the state
                    (a run to its next output frame)
            "remd"  one exchange cycle: an event window per replica, the
                    energies, the exchange pass, the new temperatures
            "bulk"  the bulk prediction of every atom (and the event tree),
                    the energies and the state: the start of a run
  engine    "plain" (FP64, the reference's event order) or "fast" (local
            time, FP32 screen, FP64 confirmation)
  systems   systems in the context
  chains, length   chains per system and residues per chain; with
            mixed = True the systems are uneven, drawn with up to these
            numbers of chains and residues
  cutoff    cell size at least this (A)
  thermostat, wall, validate   options of the run
  amount    pops ("abi", "pops"), time units ("until"), events per replica
            ("remd"); 1 for "bulk"

Sizes come from the package's own workloads: the 59-atom alanine 10-mer, the
dense single chain, 8 x 20 residues in a cylinder (replicas), 12 x 30 and
64 x 40 residues at 5 mM, and the uneven batch.  A geometry is built once and
shared by the seeds; the seed draws every velocity (Maxwell-Boltzmann at the
system's temperature) and the thermostat's random stream, which is what two
independent runs of one input differ in.
"""
import copy
import functools
import os
import tempfile
from concurrent.futures import ThreadPoolExecutor

import numpy as np

from sdmd_amd import builder
from sdmd_amd._ctypes_types import NTYPE
from sdmd_amd.engine import GpuEngine, System
from sdmd_amd.remd import Remd, ladder

TEMPERATURE = 0.5962          # 300 K in reduced units
EVENTS_PER_ATOM = 13.2        # executed events per atom and time unit at 300 K
BOND, CONSTRAINT = 1, 2       # connection bits (SDMD_BOND_CONNECT, SDMD_CONSTRAINT_CONNECT)
# what a run changes: returned whole (one array per field, systems in order)
STATE = ("x", "y", "z", "vx", "vy", "vz", "type", "cellx", "celly", "cellz", "hb_bond", "hb_itype", "nb_partner",
         "nb_partnernum", "nb_status", "dyn_j", "dyn_bits", "ev_partner", "ev_counter", "ev_pcounter", "ev_time",
         "ev_pot", "ev_type", "ev_sub", "celllist")


def _case(name, path, engine, systems, chains, length, amount, cutoff=7.25, mixed=False, thermostat=True, wall=False,
          validate=False):
    c = dict(path=path, engine=engine, systems=systems, chains=chains, length=length, mixed=mixed, cutoff=cutoff,
             thermostat=thermostat, wall=wall, validate=validate, amount=amount)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a host event loop that calls the engine pop by pop (the reference's
        # calls replaced one by one): the smallest calls
        _case("abi_ala10", "abi", "plain", 1, 1, 10, 24, cutoff=9.0),
        # the plain engine on the smallest system, the thermostat on
        _case("plain_ala10", "pops", "plain", 1, 1, 10, 4000, cutoff=9.0),
        # ... in a smooth cylinder wall (one REMD replica's system)
        _case("plain_cylinder", "pops", "plain", 1, 8, 20, 2000, wall=True),
        # ... on the largest system
        _case("plain_64x40", "pops", "plain", 1, 64, 40, 1000, thermostat=False),
        # ... on an uneven batch
        _case("plain_batch", "pops", "plain", 12, 16, 60, 1000, mixed=True, thermostat=False),
        # the start of a plain run
        _case("plain_bulk", "bulk", "plain", 1, 12, 30, 1, thermostat=False),
        # the smallest system on the fast engine: few events are independent
        _case("fast_ala10", "until", "fast", 1, 1, 10, 10.0, cutoff=9.0),
        # bulky residues, wide cells (over 64 atoms in a cell), every screen
        # validated in FP64: the precision form, without a thermostat
        _case("fast_dense_check", "until", "fast", 1, 1, 30, 1.0, cutoff=12.0, thermostat=False, validate=True),
        # one large system up to its next frame
        _case("fast_64x40", "until", "fast", 1, 64, 40, 0.2),
        # the uneven batch up to its next frame
        _case("fast_batch", "until", "fast", 24, 32, 80, 0.2, mixed=True),
        # replica exchange: 64 replicas, exchange every 10^4 events
        _case("remd64", "remd", "fast", 64, 8, 20, 10000, wall=True),
        # the start of a fast run of one large system
        _case("fast_bulk", "bulk", "fast", 1, 64, 40, 1),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    path, engine = rng.choice([("abi", "plain"), ("pops", "plain"), ("bulk", "plain"), ("until", "fast"),
                               ("until", "fast"), ("until", "fast"), ("remd", "fast"), ("bulk", "fast")])
    thermo = rng.random() < 0.5
    if path == "abi":
        return _case("", "abi", "plain", 1, _log(rng, 1, 16), rng.randint(10, 30), rng.randint(5, 24),
                     thermostat=thermo)
    if path == "remd":
        return _case("", "remd", "fast", _log(rng, 3, 64), rng.randint(3, 8), rng.randint(10, 20),
                     _log(rng, 1000, 9000), wall=True)
    chains, length = _log(rng, 1, 64), rng.randint(10, 40)
    atoms = 10.45 * chains * length
    if path == "bulk":
        chains = min(chains, 12) if engine == "plain" else chains
        return _case("", "bulk", engine, 1, chains, length, 1, thermostat=False if engine == "plain" else thermo)
    if engine == "plain":
        if rng.random() < 0.4:
            return _case("", "pops", "plain", rng.randint(2, 11), _log(rng, 4, 16), rng.randint(30, 60),
                         rng.randint(300, 900), mixed=True, thermostat=False)
        return _case("", "pops", "plain", 1, chains, length, rng.randint(300, 1000), thermostat=thermo,
                     wall=chains <= 8 and length <= 20)
    if rng.random() < 0.4:
        return _case("", "until", "fast", rng.randint(2, 23), _log(rng, 6, 32), rng.randint(30, 80),
                     round(rng.uniform(0.02, 0.15), 3), mixed=True)
    events = _log(rng, 10000, 40000)
    return _case("", "until", "fast", 1, chains, length, float("%.3g" % (events / (EVENTS_PER_ATOM * atoms))),
                 thermostat=thermo, wall=chains <= 8 and length <= 20, validate=rng.random() < 0.25,
                 cutoff=rng.choice([7.25, 7.25, 9.0]))


# ---------------------------------------------------------------- geometries
@functools.lru_cache(maxsize=None)
def _chains(length):
    """Seeded chains of random sequence; a system is made of copies, each
    with its own place and orientation."""
    return builder.build_chains(builder.random_sequences(2 if length <= 40 else 1, length, 4), 4, workers=1)


def _copies(length, n):
    unique = _chains(length)
    return [copy.deepcopy(unique[k % len(unique)]) for k in range(n)]


def _specs(case):
    if not case["mixed"]:
        return [(case["chains"], case["length"])] * case["systems"]
    specs = builder.batch_specs(case["systems"], 4, length=(10, case["length"]), chains=(1, case["chains"]),
                                min_atoms=min(2000, 4 * case["chains"] * case["length"]))
    return [(_tiles(nc) * _unit(nc), 10 * max(1, (L + 5) // 10)) for nc, L in specs]


def _tiles(chains):
    """More than 8 chains: a cube of 2 x 2 x 2 boxes of one eighth of them
    each (placing is quadratic in the chains placed)."""
    return 8 if chains > 8 else 1


def _unit(chains):
    return max(1, round(chains / _tiles(chains)))


def _geometry(case, k, chains, length):
    if case["wall"]:
        box = (160.0, 80.0, 80.0)
        placed = builder.place_chains(_copies(length, chains), box, np.random.default_rng([5, k]), cylinder=34.0)
        return builder.System(placed, box, "peptides in a cylinder")
    if chains == 1 and length == 10:
        return builder.ala10_extended()
    if case["cutoff"] > 9.0:
        return builder.single_chain((["TRP", "ARG", "LYS", "PHE", "TYR"] * 16)[:length], 8, 2.4 * length)
    mine = _copies(length, _unit(chains))
    extent = max(np.max(np.linalg.norm(c.xyz, axis=1)) for c in mine)
    edge = max(builder.box_for_concentration(len(mine), 5.0), 2 * extent + 8.0)
    placed = builder.place_chains(mine, (edge,) * 3, np.random.default_rng([4, k]))
    if _tiles(chains) == 8:
        placed = [copy.deepcopy(c) for _ in range(8) for c in placed]
        for q, c in enumerate(placed):
            c.xyz = c.xyz + edge * np.array(np.unravel_index(q // len(mine), (2, 2, 2)))
        edge = 2 * edge
    return builder.System(placed, (edge,) * 3, "peptides")


def _temperatures(case):
    return ladder(case["systems"]) if case["path"] == "remd" else [TEMPERATURE] * case["systems"]


@functools.lru_cache(maxsize=None)
def _loaded(key):
    """The host-prepared systems (positions, tables, cell lists): one for
    each uneven system, else one for all."""
    case = dict(key)
    kw = dict(wall="smooth", wall_type="cylinder") if case["wall"] else {}
    with tempfile.TemporaryDirectory(prefix="sdmd_cases_") as tmp:
        dirs = [builder.write_input_dir(_geometry(case, k, *spec), os.path.join(tmp, "s%02d" % k),
                                        temperature=TEMPERATURE, cutoff=case["cutoff"], **kw)
                for k, spec in enumerate(_specs(case) if case["mixed"] else _specs(case)[:1])]
        with ThreadPoolExecutor(max_workers=8) as ex:
            return list(ex.map(System.load, dirs))


def _systems(case, seed):
    """The case's systems with the seed's velocities and random streams."""
    key = tuple((k, case[k]) for k in ("systems", "chains", "length", "mixed", "cutoff", "wall"))
    loaded, out = _loaded(key), []
    for k, T in enumerate(_temperatures(case)):
        arr = loaded[k if case["mixed"] else 0].arrays.copy()
        rng = np.random.default_rng([seed, k])
        sigma = np.sqrt(T / arr.arr["mass"][1:])
        for f in ("vx", "vy", "vz"):
            arr.arr[f][1:] = sigma * rng.standard_normal(len(sigma))
        arr.scalars.update(seed=(seed * 64 + k) % (1 << 31) + 1, temperature=T, thermostat=int(case["thermostat"]))
        out.append(System(None, arr))
    return out


# ---------------------------------------------------------------- passes
def prepare(case, seed):
    systems = _systems(case, seed)
    if case["path"] == "remd":
        r = Remd(systems, _temperatures(case), seed=seed % 1000 + 1, interval=case["amount"])
        r.prepare()
        return {"case": case, "remd": r}
    fast = case["engine"] == "fast"
    natom = max(s.natom for s in systems)
    kw = dict(block=512 if fast or natom > 2000 else 256)
    if fast:
        kw["validate"] = case["validate"]
    eng = GpuEngine(systems, mode=case["engine"], **kw)
    if not fast and case["thermostat"]:
        eng.feed_normals(4000000)
    if case["path"] != "bulk":
        eng.prepare()
    return {"case": case, "eng": eng, "t": 0.0}


def _state(eng):
    got = [eng.state(k).arr for k in range(len(eng.systems))]
    return {f: got[0][f] if len(got) == 1 else np.concatenate([a[f] for a in got]) for f in STATE}


def _abi(eng, pops):
    events = []
    for _ in range(pops):
        ev = eng.pop(0)
        target, partner = ev["target"], max(ev["partner"], 0)
        eng.advance(0, ev["time"])
        if ev["stale"]:
            renew = [target]
        else:
            eng.do_event(0, target, partner)
            renew = [target, partner] if partner else [target]
        eng.predict(0, renew)
        eng.update_tree(0, renew)
        events.append((ev["target"], ev["partner"], ev["type"], ev["sub"], ev["time"], ev["potential"]))
    return events


def run(state):
    case = state["case"]
    if case["path"] == "remd":
        r = state["remd"]
        epot = r.run(1)
        kinetic, potential = r.eng.energy()
        temperature, number = r.temperatures()
        return {"epot": epot, "kinetic": kinetic, "potential": potential, "temperature": temperature,
                "number": number, "counts": r.counts.copy()}
    eng = state["eng"]
    if case["path"] == "abi":
        ev = _abi(eng, case["amount"])
        out = _state(eng)
        out["events"] = np.array([e[:4] for e in ev], np.int64)
        out["event_values"] = np.array([e[4:] for e in ev])
        return out
    if case["path"] == "bulk":
        eng.prepare()
        kinetic, potential = eng.energy()
        return dict(_state(eng), kinetic=kinetic, potential=potential)
    if case["path"] == "pops":
        eng.run(case["amount"])
    else:
        state["t"] += case["amount"]
        eng.run_until(state["t"])
    return _state(eng)


# ---------------------------------------------------------------- work and exact values
ATOMS_PER_RESIDUE = 10.45
STATE_BYTES = 250             # per atom: the fields of STATE


def _natoms(case):
    return [59 if (nc, L) == (1, 10) and not case["wall"] else ATOMS_PER_RESIDUE * _tiles(nc) * _unit(nc) * L for nc, L in _specs(case)]


def work(case):
    """Bytes: per prediction, position, velocity, type and exclusion word (56 B)
    of the atom and of each neighbour; per event a 40 B record and the tree
    path; the state once where it is returned; the plain engine's sweep of
    positions and times per pop (its state advances all atoms by definition).
    Flops: about 60 per neighbour pair."""
    N = _natoms(case)
    neighbours = 60 if max(N) < 100 else 105 * (case["cutoff"] / 7.25) ** 1.5
    if case["path"] == "bulk":
        predictions, events, sweeps = sum(N), 0, 0
    elif case["path"] in ("abi", "pops"):
        pops = case["amount"] * len(N)
        predictions, events, sweeps = 1.6 * pops, 0.63 * pops, case["amount"] * sum(N) * 88
    else:
        per = [case["amount"] if case["path"] == "remd" else EVENTS_PER_ATOM * n * case["amount"] for n in N]
        events, sweeps = sum(per), 0
        predictions = 2.6 * events
    tree = events * 24 * np.ceil(np.log2(max(N)))
    returned = 0 if case["path"] == "remd" else sum(N) * STATE_BYTES
    return {"bytes": float(predictions * (neighbours + 1) * 56 + events * 40 + tree + sweeps + returned),
            "flops": float(predictions * neighbours * 60 + sweeps / 88 * 8)}


def exact(case, seed):
    """The energies at the start of a run, by definition: m v^2 / 2 summed, and
    over every pair inside the cut-off the accumulated energy of the shell it
    is in (constraint pairs from their own shells; bonded pairs add nothing).
    No pair has crossed a shell before the first event, so the energies hold
    at the snapshot time too.  A trajectory has no such closed form."""
    if case["path"] != "bulk":
        return None
    out = dict.fromkeys(STATE)
    ke, pe = zip(*(_energies(s) for s in _systems(case, seed)))
    return dict(out, kinetic=np.array(ke), potential=np.array(pe))


def _energies(system):
    a, sc = system.arrays.arr, system.arrays.scalars
    n = sc["natom"]
    v2 = sum(a[f][1:] ** 2 for f in ("vx", "vy", "vz"))
    kinetic = float(np.sum(0.5 * a["mass"][1:] * v2))
    box = np.array(sc["box"][:])
    pos = np.stack([a["x"], a["y"], a["z"]], 1)
    cell = np.stack([a["cellx"], a["celly"], a["cellz"]], 1).astype(np.int64)
    num = np.array(sc["cellnum"][:], np.int64)
    cid = (cell[:, 2] * num[1] + cell[:, 1]) * num[0] + cell[:, 0]
    order = np.argsort(cid[1:], kind="stable") + 1
    start = np.searchsorted(cid[order], np.arange(num.prod() + 1))
    left, right = [], []
    for off in np.ndindex(3, 3, 3):
        nc = cell[1:] + np.array(off) - 1
        shift = np.where(nc < 0, -box, np.where(nc >= num, box, 0.0))
        nc = np.where(nc < 0, num - 1, np.where(nc >= num, 0, nc))
        c = (nc[:, 2] * num[1] + nc[:, 1]) * num[0] + nc[:, 0]
        for q in range(int((start[c + 1] - start[c]).max())):
            i = np.flatnonzero(start[c] + q < start[c + 1]) + 1
            j = order[start[c[i - 1]] + q]
            r = pos[i] - (pos[j] + shift[i - 1])
            keep = (j > i) & (np.sum(r * r, 1) <= sc["cutoffr"] ** 2)
            left.append(i[keep])
            right.append(np.stack([j[keep], np.sum(r * r, 1)[keep]], 1))
    i = np.concatenate(left)
    j, rr = np.concatenate(right).T
    j = j.astype(np.int64)
    # each pair's connection bits (rows are sorted) and constraint entry
    def entry(off, cols):
        rows = np.repeat(np.arange(n + 1), np.diff(off[:n + 2]))
        keys = rows * (n + 1) + cols
        o = np.argsort(keys, kind="stable")
        at = np.minimum(np.searchsorted(keys[o], i * (n + 1) + j), len(keys) - 1)
        return np.where(keys[o[at]] == i * (n + 1) + j, o[at], -1)

    m = entry(a["cmap_off"], a["cmap_j"])
    bits = np.where(m >= 0, a["cmap_bits"][m], 0)
    con = (bits & CONSTRAINT) != 0
    if con.any():
        at = np.where(con, entry(a["con_off"], a["con_j"]), 0)
    else:
        at = np.zeros(len(i), np.int64)
    # collision pairs: the table's entry, else that of the types without
    # their hydrogen-bond state
    back = np.arange(NTYPE)
    back[[3, 4, 27]] = [1, 2, 26]
    t1, t2 = a["type"][i], a["type"][j]
    pick = np.full(len(i), -1)
    for u, w in ((t1, t2), (back[t1], t2), (t1, back[t2]), (back[t1], back[t2])):
        pick = np.where((pick < 0) & (a["pair"]["dmin"][u * NTYPE + w] > 0), u * NTYPE + w, pick)

    def shell(field):
        of_con = a["con"][field][at] if con.any() else 0
        return np.where(con, of_con, a["pair"][field][pick])

    # the shell a pair is in: the number of radii it has passed; past the
    # last one, and inside the core, it adds nothing
    step0, nstep = shell("step0"), shell("nstep")
    passed = np.zeros(len(i), np.int64)
    for k in range(int(nstep.max())):
        inside = k < nstep
        passed += inside & (rr >= a["step_d"][np.where(inside, step0 + k, 0)])
    adds = ((bits & BOND) == 0) & (rr >= shell("dmin")) & (passed < nstep)
    return kinetic, float(np.sum(a["step_acc"][np.where(adds, step0 + passed, 0)][adds]))

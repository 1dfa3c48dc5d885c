"""Performance cases of the MI355X PRIME20 DMD engine.

Each case is one call pattern of a program that uses the engine through
pdmd.py: advance resident systems and read their states (trajectory frames),
upload and start a system, force a list update and read the observables, or
serve a burst of trajectory requests.  Sizes follow the repository's own
configurations: chains of 8 to 32 residues, 128 to 23 424 beads, reduced
densities 0.005 to 0.1 (dilute solutions mostly, as in the benchmark), T*
0.15 to 0.50, 1 to 8 wavefronts per system, batches of 1 to 320 systems.

A case names the sizes; the sequences, coils, velocities and thermostat
streams come from the seed.
"""
import math
import os
import random
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "parallel-dmd-for-biomolecules_amd"))

import pdmd  # noqa: E402

LENGTHS = (8, 12, 16, 24, 32)


def advance(name, nsys, chains, length, entries, waves, density=0.01, canon=True, species=1, observe=False, mix=0,
            chains_hi=0, length_hi=0):
    """nsys resident systems, `entries` calendar entries each in one launch,
    then their states.  mix > 0: uneven systems, chain counts log-uniform in
    [chains, chains_hi] and lengths among LENGTHS in [length, length_hi], the
    sizes drawn from the number mix; else all of chains x length residues.
    species 2: the last third of the chains is a second, longer species."""
    return dict(kind="advance", name=name, nsys=nsys, chains=chains, length=length, entries=entries, waves=waves,
                density=density, canon=canon, species=species, observe=observe, mix=mix, chains_hi=chains_hi,
                length_hi=length_hi)


def start(name, chains, length, density=0.01):
    """One system uploaded and started (lists, calendar), its state read,
    then removed: what every new trajectory pays."""
    return dict(kind="start", name=name, nsys=1, chains=chains, length=length, density=density, waves=4, canon=True,
                species=1, mix=0)


def rebuild(name, nsys, chains, length, mix, chains_hi, length_hi, density=0.01):
    """Lists and calendars of resident systems rebuilt at the current time
    in one call, then the calendars and the observables read."""
    return dict(kind="rebuild", name=name, nsys=nsys, chains=chains, length=length, density=density, waves=4,
                canon=True, species=1, mix=mix, chains_hi=chains_hi, length_hi=length_hi)


def serve(name, nreq, chains, length, mix, chains_hi, length_hi, lo, hi, density=0.01):
    """A burst of trajectory requests through the server: uneven systems,
    lo to hi entries each (log-uniform), until the last one is done."""
    return dict(kind="serve", name=name, nsys=nreq, chains=chains, length=length, density=density, waves=4, canon=True,
                species=1, mix=mix, chains_hi=chains_hi, length_hi=length_hi, lo=lo, hi=hi)


def listed():
    return [
        # the smallest call: a monitored run that reads observables every
        # 100 entries; launch, event and host latency count
        advance("monitor_128", 1, 4, 8, 100, 4, observe=True),
        # the smallest system of the benchmark's distribution on its own
        advance("one_128", 1, 4, 8, 5000, 4),
        # the 512-bead system at the engine's default of one wavefront
        advance("one_512_default", 1, 8, 16, 2500, 1),
        # ... and at the four wavefronts that the README's example sets
        advance("one_512", 1, 8, 16, 5000, 4),
        # the 6144-bead system, as many wavefronts as may be asked for
        advance("one_6144", 1, 96, 16, 8000, 8, density=0.0101),
        # two species, denser, thermostat off: long lists, many wells, NVE
        advance("dense_1920_nve", 1, 30, 16, 5000, 4, density=0.1, canon=False, species=2),
        # the largest system of the benchmark's distribution
        advance("one_23424", 1, 183, 32, 8000, 4, density=0.012),
        # the benchmark's batch: 64 uneven systems, 20 000 entries each
        advance("uneven64", 64, 4, 8, 20000, 4, mix=2024, chains_hi=192, length_hi=32),
        # more systems than compute units: a screening run of small systems
        advance("many_320", 320, 4, 8, 2000, 4, mix=11, chains_hi=24, length_hi=16),
        # admission of a large trajectory
        start("start_23424", 183, 32, density=0.012),
        # list update and observables of a batch, as at an output point
        rebuild("rebuild_16", 16, 4, 8, 7, 192, 32),
        # continuous batching: 24 requests of 2 000 to 20 000 entries
        serve("serve_24", 24, 4, 8, 5, 96, 24, 2000, 20000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("one", "batch", "many", "start", "rebuild", "serve"), (8, 3, 1, 1, 1, 1))[0]
    density = math.exp(rng.uniform(math.log(0.005), math.log(0.02)))
    waves = rng.choices((1, 2, 4, 8), (2, 1, 6, 3))[0]
    mix = rng.randrange(1, 1 << 20)
    if kind == "one":
        chains, length = _log_int(rng, 4, 180), rng.choice(LENGTHS)
        if 4 * chains * length >= 960 and rng.random() < 0.3:
            density = math.exp(rng.uniform(math.log(0.02), math.log(0.1)))
        top = 8000 if waves >= 4 else 4000
        c = advance("", 1, chains, length, _log_int(rng, 50, top), waves, density, canon=rng.random() < 0.8,
                    species=rng.choice((1, 1, 2)), observe=rng.random() < 0.3)
    elif kind == "batch":
        # a temperature ladder of one system, or uneven systems
        nsys = _log_int(rng, 2, 64)
        if rng.random() < 0.4:
            c = advance("", min(nsys, 16), _log_int(rng, 4, 96), rng.choice(LENGTHS), _log_int(rng, 500, 5000), waves,
                        density)
        else:
            c = advance("", nsys, 4, 8, _log_int(rng, 500, 5000), waves, density, mix=mix, chains_hi=_log_int(rng, 8, 192),
                        length_hi=rng.choice(LENGTHS[1:]))
    elif kind == "many":
        c = advance("", _log_int(rng, 65, 320), 4, 8, _log_int(rng, 200, 2000), waves, density, mix=mix, chains_hi=24,
                    length_hi=16)
    elif kind == "start":
        c = start("", _log_int(rng, 4, 183), rng.choice(LENGTHS), density)
    elif kind == "rebuild":
        c = rebuild("", _log_int(rng, 1, 16), 4, 8, mix, _log_int(rng, 8, 192), rng.choice(LENGTHS[1:]), density)
    else:
        c = serve("", _log_int(rng, 4, 32), 4, 8, mix, _log_int(rng, 8, 96), 24, 1000, _log_int(rng, 2000, 10000),
                  density)
    del c["name"]
    return c


def _sizes(case):
    """Chain lengths of every system of the case."""
    if not case["mix"]:
        lens = [case["length"]] * case["chains"]
        if case["species"] == 2:
            n2 = max(1, len(lens) // 3)
            lens[-n2:] = [case["length"] + 4] * n2
        return [lens] * case["nsys"]
    rng = random.Random(case["mix"])
    pick = [L for L in LENGTHS if case["length"] <= L <= case["length_hi"]]
    return [[rng.choice(pick)] * _log_int(rng, case["chains"], case["chains_hi"]) for _ in range(case["nsys"])]


def _beads(case):
    return [4 * sum(lens) for lens in _sizes(case)]


def _entries(case):
    """Calendar entries of each system or request."""
    if case["kind"] == "advance":
        return [case["entries"]] * case["nsys"]
    if case["kind"] == "serve":
        rng = random.Random(case["mix"] + 1)
        return [_log_int(rng, case["lo"], case["hi"]) for _ in range(case["nsys"])]
    return [0] * case["nsys"]


def _inputs(case, seed):
    """Generated systems with their thermostat seeds and species blocks."""
    rng = random.Random(seed)
    out = []
    for lens in _sizes(case):
        s = pdmd.generate(lens, density=case["density"], tstar=rng.uniform(0.15, 0.50), seed=rng.randrange(1 << 40))
        sp = None
        if case["species"] == 2:
            sp = [0 if L == lens[0] else 1 for L in lens]
        out.append((s, rng.randrange(1 << 40), sp))
    return out


def prepare(case, seed):
    eng = pdmd.Engine(waves=case["waves"])
    inputs = _inputs(case, seed)
    st = dict(case=case, eng=eng, inputs=inputs, entries=np.array(_entries(case), np.int64))
    if case["kind"] in ("advance", "rebuild"):
        st["ids"] = [eng.add_system(s, seed=sd, canon=case["canon"], species=sp) for s, sd, sp in inputs]
    return st


OBS = ("ered", "tred", "sumvel", "ehh_ii", "ehh_ij", "rg_avg", "e2e_avg", "hb_alpha", "hb_ii", "hb_ij")


def _frames(eng, ids):
    """The states of the listed systems, concatenated array by array."""
    got = [eng.download(i) for i in ids]
    if len(got) == 1:
        return got[0]
    return {k: np.concatenate([g[k] for g in got]) for k in got[0]}


def _observables(eng, ids):
    obs = [eng.observables(i) for i in ids]
    return {k: np.array([getattr(o, k) for o in obs]) for k in OBS}


def run(st):
    case, eng = st["case"], st["eng"]
    kind = case["kind"]
    if kind == "advance":
        eng.advance(st["ids"], st["entries"])
        out = _frames(eng, st["ids"])
        if case["observe"]:
            out["observables"] = _observables(eng, st["ids"])
        return out
    if kind == "start":
        s, sd, sp = st["inputs"][0]
        sid = eng.add_system(s, seed=sd, canon=case["canon"], species=sp)
        out = eng.download(sid)
        eng.remove_system(sid)
        return out
    if kind == "rebuild":
        eng.rebuild(st["ids"])
        out = _frames(eng, st["ids"])
        out["observables"] = _observables(eng, st["ids"])
        return out
    srv = pdmd.Server(eng, mem_budget_bytes=64 << 30, quantum=200000, slice_ms=25.0)
    rids = [srv.submit(s, int(n), seed=sd, canon=case["canon"], species=sp)
            for (s, sd, sp), n in zip(st["inputs"], st["entries"])]
    while True:
        srv.step()
        queued, resident, _ = srv.pending()
        if queued == 0 and resident == 0:
            break
    res = [srv.result(r, with_state=True) for r in rids]
    out = {"state": np.array([i.state for i, _ in res]), "done": np.array([i.done for i, _ in res]),
           "nevents": np.array([list(i.stats.nevents) for i, _ in res]),
           "sv": np.concatenate([sv for _, sv in res])}
    srv.close()
    return out


# mean list lengths of the dilute systems, both directions
K_LIST = 10.44
# one prediction: the partner's state, its list entry and code; free flight,
# minimum image, dot products, discriminant and root
PRED_BYTES, PRED_FLOPS = 53, 37
# a state read to the host: sv, identity, partner, shoulders and calendar
FRAME_BYTES = 48 + 4 + 4 + 16 + 16


def work(case):
    """A committed entry predicts every listed partner of its two beads once
    (lists in both directions), updates six calendar links and writes two
    states; a start or a list update reads every bead, writes its lists and
    predicts each listed pair once."""
    n, entries = sum(_beads(case)), sum(_entries(case))
    b = entries * (2 * K_LIST * PRED_BYTES + 6 * 4 + 2 * 48)
    f = entries * 2 * K_LIST * PRED_FLOPS
    if case["kind"] != "advance":
        b += n * (64 + 4 * K_LIST + 0.5 * K_LIST * PRED_BYTES + 16)
        f += n * 0.5 * K_LIST * PRED_FLOPS
    b += n * FRAME_BYTES
    return {"bytes": float(b), "flops": float(f)}


def _masses():
    """Bead mass by identity (parameters/mass.data: name, identity, mass)."""
    with open(os.path.join(pdmd.PARAM_DIR, "mass.data")) as f:
        rows = [line.split() for line in f if line.strip()]
    return {int(r[1]): float(r[2]) for r in rows}


def _bead_masses(system):
    m, out, r = _masses(), [], 0
    for L in (int(v) for v in system["chain_len"]):
        ident = [2] * L + [1] * L + [4] * L + [int(v) for v in system["restype"][r:r + L]]
        out += [m[k] for k in ident]
        r += L
    return np.array(out)


def _exact_observables(system):
    """tred, sumvel, radius of gyration and end-to-end distance of a start
    state, from the input arrays (chains of one length)."""
    sv = system["sv"].reshape(-1, 6).astype(np.float64)
    pos, vel = sv[:, :3] - np.round(sv[:, :3]), sv[:, 3:]
    lens = [int(v) for v in system["chain_len"]]
    mass = _bead_masses(system)
    sumvel = float((mass * (vel * vel).sum(1)).sum())
    rg, nbb, e2e, s = 0.0, 0, 0.0, 0
    for L in lens:
        q = pos[s:s + 3 * L].copy()
        # backbone unwrapped along the C-alphas, then N and C beads to their C-alpha
        for k in range(1, L):
            q[k] -= np.where(q[k] - q[k - 1] > 0.5, 1.0, np.where(q[k] - q[k - 1] < -0.5, -1.0, 0.0))
        for k in range(L, 3 * L):
            d = q[k] - q[k % L]
            q[k] -= np.where(d > 0.5, 1.0, np.where(d < -0.5, -1.0, 0.0))
        rg += float(((q - q.mean(0)) ** 2).sum())
        nbb += 3 * L
        d = pos[s + L] - pos[s + 3 * L - 1]
        e2e += float(np.sqrt(((d - np.round(d)) ** 2).sum()))
        s += 4 * L
    n = len(sv)
    return dict(tred=sumvel / 3.0 / n, sumvel=sumvel, rg_avg=math.sqrt(rg / nbb) * system["boxl"],
                e2e_avg=e2e / len(lens) * system["boxl"])


def exact(case, seed):
    """The observables of start states, in 64 bits from the inputs.  States
    after committed events have no closed form: an event-driven trajectory
    is chaotic, and replaying it takes the whole event loop."""
    if case["kind"] != "rebuild":
        return None
    obs = [_exact_observables(s) for s, _, _ in _inputs(case, seed)]
    got = {k: np.array([o[k] for o in obs]) if k in obs[0] else None for k in OBS}
    return {k: None for k in ("sv", "identity", "bptnr", "extra", "tim", "nptnr", "coltype")} | {"observables": got}

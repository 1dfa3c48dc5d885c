"""Dispatch branches of the engine at the sizes where they can go wrong."""
import numpy as np
import pytest

import pdmd
from oracle import Oracle

pytestmark = pytest.mark.gpu


def _bits(a):
    return {k: v.view(np.int64) if v.dtype == np.float64 else v for k, v in a.items()}


@pytest.mark.parametrize("waves", [1, 7])
def test_more_systems_than_compute_units(waves):
    """A launch of more systems than the GPU has compute units, whose
    workgroups share them: every system ends where it ends in a launch of a
    few, bit for bit."""
    s = pdmd.generate([8] * 4, density=0.01, tstar=0.3, seed=3)
    print(f"300 systems, {waves} wavefronts", flush=True)
    e = pdmd.Engine(waves=waves)
    few = pdmd.Engine(waves=waves)
    try:
        n, kinds = 300, 4
        ids = [e.add_system(s, seed=k % kinds) for k in range(n)]
        e.advance(ids, [300] * n)
        ref_ids = [few.add_system(s, seed=k) for k in range(kinds)]
        few.advance(ref_ids, [300] * kinds)
        ref = [_bits(few.download(i)) for i in ref_ids]
        for k, i in enumerate(ids):
            got = _bits(e.download(i))
            for f, v in ref[k % kinds].items():
                assert np.array_equal(got[f], v), (k, f)
    finally:
        e.close()
        few.close()


@pytest.mark.parametrize("chains,length,second", [(1, 4, 0), (5, 8, 0), (3, 65, 0), (2, 128, 0), (40, 16, 14)])
def test_observables_at_the_edges(chains, length, second):
    """Observables against NumPy sums: one short chain, bead counts around a
    workgroup's 64, chains longer than a wavefront, two species.  The sums
    hold n terms of 64-bit rounding each, in any order: the tolerance is
    n * 2^-52 of the sum of their magnitudes."""
    lens = [length] * chains
    if second:
        lens[-second:] = [length + 4] * second
    s = pdmd.generate(lens, density=0.01, tstar=0.3, seed=chains + length)
    species = [0 if k < chains - second else 1 for k in range(chains)]
    print(f"observables of {chains} chains of {length}", flush=True)
    e = pdmd.Engine(waves=2)
    try:
        sid = e.add_system(s, seed=1, species=species)
        e.advance([sid], [200])
        o, st = e.observables(sid), e.download(sid)
        tf = e.stats(sid).tfalse
    finally:
        e.close()
    sv = st["sv"].reshape(-1, 6)
    pos = sv[:, :3] + sv[:, 3:] * tf
    n = len(sv)

    def near(a, b):
        d = a - b
        return np.where(d > 0.5, a - 1.0, np.where(d < -0.5, a + 1.0, a))

    q = pos.copy()
    start = np.concatenate([[0], np.cumsum([4 * L for L in lens])])
    for c, L in enumerate(lens):
        b = start[c]
        for k in range(b + 1, b + L):
            q[k] = near(q[k], q[k - 1])
        for k in range(b, b + L):
            q[L + k] = near(q[L + k], q[k])
            q[2 * L + k] = near(q[2 * L + k], q[k])
    rg = e2e = 0.0
    nfirst = chains - second
    for c, L in enumerate(lens):
        b = start[c]
        rb = c * 4 * L if second and c >= nfirst and c * 4 * L + 3 * L <= b + 4 * L else b
        x = q[rb:rb + 3 * L]
        rg += ((x - x.mean(0)) ** 2).sum()
        d = pos[b + L] - pos[b + 3 * L - 1]
        e2e += np.sqrt(((d - np.round(d)) ** 2).sum())
    tol = 4 * n * 2.0 ** -52
    assert abs(o.rg_avg - np.sqrt(rg / (3 * n // 4)) * s["boxl"]) <= tol * o.rg_avg
    assert abs(o.e2e_avg - e2e / chains * s["boxl"]) <= tol * o.e2e_avg
    bond = st["bptnr"]
    chain_of = np.repeat(np.arange(chains), [4 * L for L in lens])
    pairs = [(i, j - 1) for i, j in enumerate(bond) if j - 1 > i]
    assert o.hb_ii == sum(chain_of[i] == chain_of[j] for i, j in pairs)
    assert o.hb_ij == sum(chain_of[i] != chain_of[j] for i, j in pairs)
    assert o.tred > 0.0 and abs(o.sumvel - 3.0 * n * o.tred) <= tol * o.sumvel


def _same_log_and_state(eng, sid, orc, n):
    g, o = eng.log_read(sid, n), orc.run(n, log_cap=n)
    assert eng.stats(sid).status == 0 and len(g) == n
    for f in ("i", "j", "type"):
        bad = np.nonzero(g[f] != o[f])[0]
        assert bad.size == 0, f"{f} differs first at event {bad[0] + 1}: gpu {g[bad[0]]} oracle {o[bad[0]]}"
    assert np.array_equal(g["t"].view(np.int64), o["t"].view(np.int64))
    gs, os_ = _bits(eng.download(sid)), _bits(orc.state())
    for f in ("sv", "identity", "bptnr", "extra", "tim", "nptnr", "coltype"):
        assert np.array_equal(gs[f], os_[f]), f


@pytest.mark.parametrize("waves", [1, 7])
def test_events_near_a_pass_of_64(param_dir, waves):
    """Rows of up to 51 entries for a colliding pair, with the candidates of
    the beads recomputed on top: events on both sides of the 62 entries that
    one pass takes."""
    n = 4000
    sysd = pdmd.generate([16] * 20, density=0.4, tstar=0.3, seed=77)
    print(f"1280 dense beads, {waves} wavefronts", flush=True)
    eng = pdmd.Engine(waves=waves)
    try:
        sid = eng.add_system(sysd, seed=9)
        eng.log_enable(sid, n)
        eng.advance([sid], [n])
        _same_log_and_state(eng, sid, Oracle(sysd, seed=9, param_dir=param_dir), n)
    finally:
        eng.close()


def _copies(length, per_axis, density, seed):
    """One chain copied onto a cubic lattice: every event happens per_axis**3
    times at (nearly) one time."""
    s = pdmd.generate([length], density=density, tstar=0.3, seed=seed)
    x = s["sv"].reshape(-1, 6).copy()
    p = x[:, :3]
    for k in range(1, length):
        p[k] = p[k] - np.round(p[k] - p[k - 1])
    for k in range(length, 4 * length):
        p[k] = p[k] - np.round(p[k] - p[k % length])
    out = []
    for cell in np.ndindex(per_axis, per_axis, per_axis):
        y = x / per_axis
        y[:, :3] += (np.array(cell) - (per_axis - 1) / 2) / per_axis
        out.append(y)
    sv = np.concatenate(out)
    sv[:, :3] -= np.round(sv[:, :3])
    m = per_axis ** 3
    return dict(s, chain_len=np.full(m, length, np.int32), restype=np.tile(s["restype"], m), hp=np.tile(s["hp"], m),
                sv=np.ascontiguousarray(sv.ravel()), boxl=per_axis * s["boxl"])


@pytest.mark.parametrize("waves", [1, 4, 7])
@pytest.mark.parametrize("per_axis", [2, 3, 4])
def test_many_entries_of_one_time(param_dir, waves, per_axis):
    """8, 27 and 64 copies of one chain: more entries of one time than the
    selection's pool of 24 holds, whose order is that of their insertion."""
    n = 2500
    sysd = _copies(8, per_axis, 0.002, 5)
    print(f"{per_axis ** 3} copies, {waves} wavefronts", flush=True)
    eng = pdmd.Engine(waves=waves)
    try:
        sid = eng.add_system(sysd, seed=3, canon=False)
        eng.log_enable(sid, n)
        eng.advance([sid], [n])
        orc = Oracle(sysd, seed=3, param_dir=param_dir, canon=False)
        _same_log_and_state(eng, sid, orc, n)
        t = eng.log_read(sid, n)["t"][:per_axis ** 3]
        assert t.max() - t.min() < 1e-14, "the copies' first events are not of one time"
    finally:
        eng.close()


def test_footprint_marks_shared_between_beads():
    """33 600 beads: more than the LDS holds marks for, so beads share them.
    A round may then be cut short, never wrong: seven wavefronts end where
    one (whose rounds need no marks) ends."""
    sysd = pdmd.generate([120] * 70, density=0.01, tstar=0.3, seed=12)
    out = []
    for waves in (7, 1):
        print(f"33600 beads, {waves} wavefronts", flush=True)
        eng = pdmd.Engine(waves=waves)
        try:
            sid = eng.add_system(sysd, seed=4)
            eng.advance([sid], [3000])
            out.append(_bits(eng.download(sid)))
        finally:
            eng.close()
    for f in out[0]:
        assert np.array_equal(out[0][f], out[1][f]), f


@pytest.mark.parametrize("chains", [[4], [4] * 4, [5] * 12, [7, 9] * 4, [4] * 17, [16] * 16, [13] * 20])
def test_forced_update_at_the_edges(param_dir, chains):
    """A forced list update, whose steps are launches of 256 items each over
    the whole GPU, at bead counts around 64, 256 and 1024: rows, calendar
    and the events that follow are the oracle's."""
    n = 4 * sum(chains)
    sysd = pdmd.generate(chains, density=0.02, tstar=0.3, seed=n)
    print(f"forced update of {n} beads", flush=True)
    eng = pdmd.Engine(waves=4)
    try:
        sid = eng.add_system(sysd, seed=8)
        eng.advance([sid], [500])
        eng.rebuild([sid])
        orc = Oracle(sysd, seed=8, param_dir=param_dir)
        orc.run(500)
        orc.rebuild()
        up, dn = eng.lists(sid)
        for i in range(1, n + 1):
            assert np.array_equal(up[i - 1], orc.nb_up(i)), f"up row of bead {i}"
            assert np.array_equal(dn[i - 1], orc.nb_dn(i)), f"down row of bead {i}"
        eng.log_enable(sid, 1000)
        eng.advance([sid], [1000])
        _same_log_and_state(eng, sid, orc, 1000)
    finally:
        eng.close()


def test_counters_of_a_batch():
    """The counters and row lengths that one launch sums for a system are
    those of the lists it returns, at bead counts around a workgroup's 1024."""
    eng = pdmd.Engine(waves=2)
    try:
        ids = [eng.add_system(pdmd.generate(c, density=0.02, tstar=0.3, seed=5), seed=6)
               for c in ([4], [16] * 15, [16] * 16, [17] * 16)]
        eng.advance(ids, [100, 200, 300, 400])
        for sid, want in zip(ids, (100, 200, 300, 400)):
            st = eng.stats(sid)
            up, dn = eng.lists(sid)
            n = st.nbeads
            assert st.coll == want and st.status == 0
            assert st.avg_up == sum(r.size for r in up) / n and st.avg_dn == sum(r.size for r in dn) / n
    finally:
        eng.close()

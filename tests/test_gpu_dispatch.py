"""Dispatch branches of the engine at the sizes where they can go wrong."""
import numpy as np
import pytest

import pdmd

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

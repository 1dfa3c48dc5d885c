"""pdmd_observables_noalloc against sums over the downloaded state, at the most
chains a system may have (its chain tables are the largest that the
page-locked memory of a new context has to hold), before and after a state
read.  The sums hold n terms of 64-bit rounding each, in any order: the
tolerance is 4 n 2^-52 of the sum of their magnitudes."""
import numpy as np
import pytest

import pdmd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chains,length", [(1, 4), (2047, 4), (2047, 8)])
def test_noalloc_observables_are_the_states_sums(chains, length):
    s = pdmd.generate([length] * chains, density=0.01, tstar=0.3, seed=7)
    print(f"noalloc observables of {chains} chains of {length}", flush=True)
    eng = pdmd.Engine(waves=4)
    try:
        sid = eng.add_system(s, seed=2)
        eng.advance([sid], [300])
        first = eng.observables_noalloc(sid)
        st, tf = eng.download(sid), eng.stats(sid).tfalse
        again = eng.observables_noalloc(sid)
    finally:
        eng.close()
    sv = st["sv"].reshape(chains, 4, length, 6)
    pos = sv[..., :3] + sv[..., 3:] * tf

    def near(a, b):
        d = a - b
        return np.where(d > 0.5, a - 1.0, np.where(d < -0.5, a + 1.0, a))

    q = pos[:, :3].copy()  # Calpha, N, C
    for k in range(1, length):
        q[:, 0, k] = near(q[:, 0, k], q[:, 0, k - 1])
    q[:, 1] = near(q[:, 1], q[:, 0])
    q[:, 2] = near(q[:, 2], q[:, 0])
    q = q.reshape(chains, 3 * length, 3)
    rg = np.sqrt(((q - q.mean(1, keepdims=True)) ** 2).sum() / (3 * length * chains)) * s["boxl"]
    d = pos[:, 1, 0] - pos[:, 2, -1]
    e2e = np.sqrt(((d - np.round(d)) ** 2).sum(1)).sum() / chains * s["boxl"]
    n = 4 * length * chains
    tol = 4 * n * 2.0 ** -52
    for o in (first, again):
        assert abs(o.rg_avg - rg) <= tol * rg and abs(o.e2e_avg - e2e) <= tol * e2e
        assert o.sumvel > 0.0 and abs(o.sumvel - 3.0 * n * o.tred) <= tol * o.sumvel
        bond = st["bptnr"]
        assert o.hb_ii + o.hb_ij == np.count_nonzero(bond > np.arange(1, n + 1))

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

"""The context's autotuner (pdmd_autotune_waves) and the trials that a launch
can tell apart: alone on a compute unit a system runs up to seven event
wavefronts, so the widest setting is tried; in a launch of more systems than
compute units three at most, so it is not.  The trials are ordinary committed
entries: the state is that of an engine that was never tuned."""
import numpy as np
import pytest

import pdmd

pytestmark = pytest.mark.gpu

PROBE = 1000


def _bits(a):
    return {k: v.view(np.int64) if v.dtype == np.float64 else v for k, v in a.items()}


def test_the_widest_setting_is_tried():
    s = pdmd.generate([16] * 8, density=0.01, tstar=0.3, seed=3)
    tuned, plain = pdmd.Engine(), pdmd.Engine()
    try:
        a, b = tuned.add_system(s, seed=1), plain.add_system(s, seed=1)
        w, rates = tuned.autotune_waves([a], PROBE)
        print("autotune_waves:", w, rates, flush=True)
        assert set(rates) == {1, 2, 4, 8} and w == max(rates, key=rates.get)
        assert tuned.stats(a).coll == 4 * PROBE
        plain.advance([b], [4 * PROBE])
        x, y = _bits(tuned.download(a)), _bits(plain.download(b))
        for f in x:
            assert np.array_equal(x[f], y[f]), f
    finally:
        tuned.close()
        plain.close()


def test_only_settings_that_a_shared_compute_unit_runs():
    s = pdmd.generate([8] * 4, density=0.01, tstar=0.3, seed=3)
    eng = pdmd.Engine()
    try:
        ids = [eng.add_system(s, seed=k) for k in range(300)]
        w, rates = eng.autotune_waves(ids, 100)
        print("300 systems, autotune_waves:", w, rates, flush=True)
        assert set(rates) == {1, 2, 4} and w in rates
        ws, _, per = eng.autotune_systems(ids, 100)
        assert set(ws) <= {1, 2, 4}
        assert (per[:, :3] > 0.0).all() and (per[:, 3] == 0.0).all()
        assert all(eng.stats(i).coll == 600 for i in ids[::50])
    finally:
        eng.close()

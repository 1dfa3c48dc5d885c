"""A step on an empty server: pdmd_server_step returns at once, so a caller
with other servers or work of its own in the same loop loses nothing to it;
the Python server spaces steps that find nothing to do by idle_pause, and only
steps that follow each other closer than that."""
import ctypes
import time

import pytest

import pdmd

pytestmark = pytest.mark.gpu


def _least(f, n):
    best = 1e9
    for _ in range(n):
        t = time.perf_counter()
        f()
        best = min(best, time.perf_counter() - t)
    return best


def test_an_empty_step_returns_at_once():
    eng = pdmd.Engine()
    srv = pdmd.Server(eng, mem_budget_bytes=1 << 30, quantum=1000)
    srv.idle_pause = 0.0
    n = ctypes.c_int32(0)
    try:
        c = _least(lambda: pdmd.lib().pdmd_server_step(srv._h, ctypes.byref(n)), 200)
        p = _least(srv.step, 200)
        print(f"empty step: {c * 1e6:.1f} us, from Python {p * 1e6:.1f} us", flush=True)
        assert c < 20e-6 and p < 20e-6
    finally:
        srv.close()
        eng.close()


def test_idle_pause_spaces_polls_only():
    pause = 10e-3
    eng = pdmd.Engine()
    srv = pdmd.Server(eng, mem_budget_bytes=1 << 30, quantum=1000, idle_pause=pause)

    def work_and_step():
        time.sleep(1.5 * pause)
        t = time.perf_counter()
        srv.step()
        return time.perf_counter() - t

    try:
        srv.step()
        t = time.perf_counter()
        for _ in range(5):
            srv.step()
        assert time.perf_counter() - t >= 5 * pause
        assert min(work_and_step() for _ in range(5)) < pause / 2
        # a request is taken without a pause and runs as ever
        rid = srv.submit(pdmd.generate([8] * 4, density=0.01, tstar=0.3, seed=3), 500, seed=1)
        while srv.pending()[:2] != (0, 0):
            srv.step()
        assert srv.result(rid)[0].done == 500
    finally:
        srv.close()
        eng.close()

"""The first state read of a program costs what later ones cost: the
page-locked memory that it goes through is there, and in use, once the system
is added.  (Where the read allocated it, the first one of 65 408 beads took
eight times a later one's time.)  In a process of its own: page-locked memory
that an earlier context gave back comes back without that cost."""
import os
import subprocess
import sys

import pytest

import pdmd

pytestmark = pytest.mark.gpu

PROGRAM = """
import time
import numpy as np
import pdmd
eng = pdmd.Engine()
sid = eng.add_system(pdmd.generate([32] * 511, density=0.01, tstar=0.3, seed=5), seed=1)
t = []
for _ in range(8):
    t0 = time.perf_counter()
    eng.download(sid)
    t.append(time.perf_counter() - t0)
eng.close()
print(t[0] / np.median(t[1:]))
"""


def test_first_read_of_a_large_state():
    env = dict(os.environ, PYTHONPATH=pdmd.PKG_DIR)
    print("first read of 65408 beads", flush=True)
    run = subprocess.run([sys.executable, "-c", PROGRAM], env=env, capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, run.stderr
    print("first read over later ones:", run.stdout.strip(), flush=True)
    assert float(run.stdout) < 4.0

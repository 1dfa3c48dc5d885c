"""H-bonds that form and break beside events of their own shoulder beads, at
the most event wavefronts: a speculative event may read the H-bond partner and
the identities that the round's first event is writing.  Whatever it reads, it
only looks at beads of the system, and the round's check discards it: every
event and the final state are the oracle's."""
import numpy as np
import pytest

import pdmd
from oracle import Oracle
from test_gpu_dispatch import _same_log_and_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chains,length,density,tstar", [(24, 8, 0.2, 0.14), (30, 6, 0.3, 0.12)])
def test_shoulder_events_beside_bond_events(param_dir, chains, length, density, tstar):
    n = 400000
    sysd = pdmd.generate([length] * chains, density=density, tstar=tstar, seed=11)
    print(f"{chains} chains of {length}, T* {tstar}, 7 wavefronts", flush=True)
    eng = pdmd.Engine(waves=7)
    try:
        sid = eng.add_system(sysd, seed=3)
        eng.log_enable(sid, n)
        eng.advance([sid], [n])
        types = eng.log_read(sid, n)["type"]
        assert np.isin(types, (20, 21)).sum() > 100 and np.isin(types, (24, 25, 26, 27)).sum() > 10
        _same_log_and_state(eng, sid, Oracle(sysd, seed=3, param_dir=param_dir), n)
    finally:
        eng.close()

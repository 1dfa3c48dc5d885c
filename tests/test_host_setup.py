"""Host half of a system's start-up without a GPU: the cell grid follows from
the largest pair cutoff, which is looked for over classes of bead pairs; it is
the oracle's, which looks at every pair."""
import pytest

import pdmd
from oracle import Oracle


def _grid_bytes(mq):
    return sum((b + 4095) // 4096 * 4096 for b in (4 * (mq ** 3 + 1), 4 * mq ** 3))


@pytest.mark.parametrize("flags", [{}, {"no_hbs": True}, {"no_h": True}, {"chaptype2": True}],
                         ids=lambda f: next(iter(f), "plain"))
@pytest.mark.parametrize("first,second", [([4], []), ([5], []), ([9] * 3, []), ([16] * 2, [7] * 2), ([4] * 3, [12]),
                                          ([32], [4, 4])])
def test_cell_grid_of_every_pair(param_dir, first, second, flags):
    if second and "chaptype2" in flags:
        pytest.skip("the oracle refuses generated coils as unbonded second-species chains (their beads overlap)")
    species = [0] * len(first) + [1] * len(second)
    got, want = [], []
    for density in (5e-5, 2e-3):
        for seed in (1, 2):
            sysd = pdmd.generate(first + second, density=density, tstar=0.2, seed=seed)
            d, keep = pdmd.Engine.make_desc(sysd, seed=1, species=species, **flags)
            b = pdmd.lib().pdmd_system_bytes(d)
            assert b > 0, pdmd.lib().pdmd_last_error()
            got.append(b)
            m = Oracle(sysd, seed=1, param_dir=param_dir, species=species, **flags).stats().num_cell - 4
            want.append(_grid_bytes(m // 2))
    assert [b - got[0] for b in got] == [g - want[0] for g in want]

"""The force launch whose blocks share a tile where tiles differ: a drop (long
lists, so that launch is taken) among scattered atoms (tiles of empty and
short lists, parts without a row group).  The forces are those of the launch
with statistics, bit for bit, also after moves, and where the longest list is
just below the line (the unsplit launch)."""
import numpy as np
import pytest

from sre import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("drop", [2, 5, 9])      # longest lists of 7, some 75 and some 300
@pytest.mark.parametrize("n", [730, 1900])
def test_forces_equal_unsplit(torch_cuda, lanes, drop, n):
    rng = np.random.default_rng(drop)
    m, a = 13, 6.0
    edge = np.full(3, a * m, np.float32)
    xyz = np.zeros((n, 4), np.float32)
    k = drop ** 3
    xyz[:k, :3] = np.stack(np.unravel_index(np.arange(k), (drop,) * 3), 1) * 1.05 + 1.0
    far = np.stack(np.unravel_index(rng.permutation(m ** 3), (m,) * 3), 1)
    far = far[(far > (1.05 * drop + 4.0) / a).any(1)][:n - k]       # clear of the drop
    xyz[k:, :3] = (far[:n - k] + 0.5) * a + rng.uniform(-2.4, 2.4, (n - k, 3))
    xyz = xyz[rng.permutation(n)]
    rc = 4.0 if drop == 9 else 2.5
    e = Engine(skin=0.3)
    e.set_tuning(force_lanes=lanes)
    e.set_system([n], [edge])
    e.set_types(np.zeros(n, np.int32))
    one = np.ones((1, 1), np.float32)
    e.set_pair_params(one, one)
    e.set_rc_table(np.full((1, 1, 1), rc, np.float32))
    e.upload_positions(xyz)
    e.rebuild()
    for step in range(2):
        e.compute(stats=True)
        want = e.forces_fixed()
        e.compute(stats=False)
        assert np.array_equal(e.forces_fixed(), want)
        assert np.abs(want).max() > 0
        e.perturb(0.01, 3, step)
        e.update_positions()
    e.close()

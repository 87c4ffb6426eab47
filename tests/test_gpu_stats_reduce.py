"""The statistics reduction at the sizes where its chunks (1 024 atoms, longer
ones above 524 288) and its count of finished blocks can go wrong: against the
exact sums of the per-atom values, read several times."""
import math

import numpy as np
import pytest

from sre import Engine

pytestmark = pytest.mark.gpu

# a value passes at most 4 + 10 + 512 / 16 + 4 additions (per thread, block,
# chunks per lane, lanes), 2 more per doubling of the chunk: below 64, each
# within 2^-53 of a partial sum that is at most the sum of magnitudes
TOL = 64 * 2.0 ** -53


@pytest.mark.parametrize("ns", [[1], [63], [1023], [1024], [1025], [2049], [64, 3000, 1024, 65],
                                [64] * 40, [524289], [600000, 64]])
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_totals_equal_sums_of_atoms(torch_cuda, ns, precision):
    rng = np.random.default_rng(sum(ns))
    xyz, boxes = [], []
    for n in ns:
        m = max(6, math.ceil(n ** (1.0 / 3.0)))     # a jittered cubic lattice
        g = np.stack(np.unravel_index(np.arange(n), (m, m, m)), 1) + 0.5
        x = np.zeros((n, 4), np.float32)
        x[:, :3] = 1.1 * (g + rng.uniform(-0.05, 0.05, g.shape))
        xyz.append(x)
        boxes.append(np.full(3, 1.1 * m, np.float32))
    e = Engine(skin=0.3, precision=precision)
    e.set_system(ns, boxes)
    e.set_types(np.zeros(sum(ns), np.int32))
    one = np.ones((1, 1), np.float32)
    e.set_pair_params(one, one)
    for r in range(len(ns)):
        e.set_rc_table(np.full((1, 1, 1), 2.5, np.float32), replica=r)
    e.upload_positions(np.concatenate(xyz))
    e.rebuild()
    off = np.concatenate([[0], np.cumsum(ns)])
    seen = []
    for _ in range(3):
        e.compute(stats=True)
        total, a = e.stats(), e.atom_stats()
        for r in range(len(ns)):
            part = a[off[r]:off[r + 1]]
            for c in range(4):
                want = math.fsum(part[:, c])
                assert abs(total[r, c] - want) <= TOL * math.fsum(np.abs(part[:, c]))
        assert np.array_equal(total, e.stats())
        seen.append(total)
    e.close()
    assert np.array_equal(seen[0], seen[1]) and np.array_equal(seen[0], seen[2])

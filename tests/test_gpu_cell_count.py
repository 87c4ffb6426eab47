"""The cell histogram made in LDS (16 atoms or more per cell, at most 4 096
cells) and one by one, at the edges of that rule and of a block's 1 024 atoms:
the order of the counting sort is the radix sort's, seen in the last bits of
FP64 forces and in the pair lists."""
import numpy as np
import pytest

from sre import Engine

pytestmark = pytest.mark.gpu

# atoms, cell_xy and cell_z (in units of rc + skin): 3 x 3 columns of 4 to 240 cells
CASES = [(1023, 1.0, 1.0), (1024, 1.0, 0.3), (1025, 1.0, 0.1), (5000, 1.0, 0.35),
         (5000, 0.5, 0.1), (20000, 1.0, 0.1), (65537, 0.35, 0.1)]


@pytest.mark.parametrize("n,cell_xy,cell_z", CASES)
def test_order_equals_radix_sort(torch_cuda, n, cell_xy, cell_z):
    rng = np.random.default_rng(n)
    m = int(np.ceil((n / 3.0) ** (1.0 / 3.0)))
    x = np.stack(np.unravel_index(rng.permutation(3 * m ** 3)[:n], (m, m, 3 * m)), 1)
    a = 9.0 / m if m > 8 else 1.1
    xyz = np.zeros((n, 4), np.float32)
    xyz[:, :3] = a * (x + 0.5 + rng.uniform(-0.05, 0.05, x.shape))
    box = np.array([a * m, a * m, 3 * a * m], np.float32)
    out = []
    for mode in (2, 1):
        e = Engine(skin=0.2, precision="fp64")
        e.set_tuning(sort_mode=mode, cell_xy=cell_xy, cell_z=cell_z)
        e.set_system([n], [box])
        e.set_types(np.zeros(n, np.int32))
        e.set_pair_params(np.ones((1, 1), np.float32), np.full((1, 1), 0.9 * a, np.float32))
        e.set_rc_table(np.full((1, 1, 1), min(2.5 * a, 2.5), np.float32))
        e.upload_positions(xyz)
        for _ in range(2):          # the counts are zero again
            e.rebuild()
        e.compute(stats=True)
        out.append((e.forces(), *e.export_pairs()))
        e.close()
    for u, v in zip(*out):
        assert np.array_equal(u, v)

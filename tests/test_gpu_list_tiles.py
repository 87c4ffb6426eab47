"""The list build's tiles at the sizes where they can go wrong: fewer atoms
than a wavefront takes, remainders, tiles across cell columns, windows that
take in whole directions of a small box, second images of cells that are a
large part of the box, and both tile sizes.  Pair sets equal the oracle's,
for several list layouts."""
import numpy as np
import pytest

from oracle import oracle as O
from sre import Engine

pytestmark = pytest.mark.gpu

# atoms, box, (rc_min, rc_max), rc bins
CASES = [
    (1, (8.0, 8.0, 8.0), (2.5, 2.5), 1),
    (5, (5.7, 5.8, 5.9), (2.5, 2.5), 1),          # every window is the whole box
    (13, (30.0, 30.0, 30.0), (3.0, 3.0), 1),      # a column per atom
    (130, (6.0, 6.5, 40.0), (2.5, 2.5), 1),
    (2000, (12.0, 50.0, 9.0), (2.5, 4.1), 7),     # whole columns along z
    (3001, (21.0, 21.0, 60.0), (7.5, 7.5), 1),    # second images along x and y
    (1501, (21.0, 40.0, 33.0), (5.0, 9.0), 16),   # along x alone
    (4097, (16.0, 16.0, 16.0), (2.5, 2.5), 1),
    (79999, (33.0, 33.0, 110.0), (2.5, 4.0), 64),
    (80007, (33.0, 33.0, 110.0), (2.5, 4.0), 64),
]


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("lanes", [1, 4, 16])
def test_pair_set_equals_oracle(torch_cuda, case, lanes):
    n, box, (lo, hi), nz = CASES[case]
    rng = np.random.default_rng(100 + case)
    box = np.asarray(box, np.float32)
    xyz = np.zeros((n, 4), np.float32)
    xyz[:, :3] = rng.random((n, 3)) * box
    table = np.linspace(lo, hi, nz).astype(np.float32).reshape(1, 1, nz)
    e = Engine(skin=0.3)
    e.set_tuning(force_lanes=lanes)
    e.set_system([n], [box])
    e.set_types(np.zeros(n, np.int32))
    one = np.ones((1, 1), np.float32)
    e.set_pair_params(one, one)
    e.set_rc_table(table)
    e.upload_positions(xyz)
    e.rebuild()
    rc, _ = O.assign_rc(xyz, box, table)
    off, j = O.build_pairs(xyz, box, rc, 0.3)
    goff, gj = e.export_pairs()
    assert np.array_equal(goff, off)
    assert np.array_equal(gj, j)
    assert e.neighbor_count(in_rc=False) == (int(off[-1]), -1, int(np.diff(off).max()))
    e.close()

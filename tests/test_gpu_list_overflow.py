"""Lists that outgrow their capacity while many pairs lie within rounding of
the list radius (a lattice with a neighbour shell at rc + skin, exactly and
slightly disturbed): entries past the capacity are dropped, so steps that run
on the cut lists before the overflow is known meet no pair that is not one,
and the next evaluation is exact.  Both tile sizes of the list build, several
list layouts."""
import numpy as np
import pytest

from oracle import oracle as O
from sre import Engine
from sre.engine import ShortNeighborList

pytestmark = pytest.mark.gpu

RC, SKIN, A = 3.7, 0.3, 0.8       # rc + skin = 4.0 in float32: the shell (3, 4, 0) A
EPS = 0.01


def lattice(m, spacing, box, jitter=0.0):
    g = (np.arange(m) - 0.5 * (m - 1)) * spacing + 0.5 * box
    x = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    x = x + np.random.default_rng(3).uniform(-jitter, jitter, x.shape)
    return np.concatenate([x, np.zeros((len(x), 1))], 1).astype(np.float32)


@pytest.mark.parametrize("m,box", [(20, 40.0), (44, 80.0)])     # below, above 80 000 atoms
@pytest.mark.parametrize("jitter", [0.0, 1e-4])
@pytest.mark.parametrize("lanes", [4, 16])
def test_cut_lists_hold_no_other_pairs(torch_cuda, m, box, jitter, lanes):
    torch = torch_cuda
    x, y = lattice(m, box / m, box), lattice(m, A, box, jitter)
    n, edges = len(x), np.full(3, box, np.float32)
    one = np.ones((1, 1), np.float32)
    table = np.full((1, 1, 1), RC, np.float32)
    e = Engine(skin=SKIN)
    e.set_tuning(force_lanes=lanes)
    e.set_system([n], [edges])
    e.set_types(np.zeros(n, np.int32))
    e.set_pair_params(EPS * one, one)
    e.set_rc_table(table)
    pos = torch.from_numpy(x).cuda()
    torch.cuda.synchronize()
    e.bind_positions(pos)
    e.rebuild()
    pos.copy_(torch.from_numpy(y))
    torch.cuda.synchronize()
    with pytest.raises(ShortNeighborList):      # segments 1 and 2 run on cut lists
        e.run_segments(3, 2, stats=True)
    rc, _ = O.assign_rc(y, edges, table)
    off, j = O.build_pairs(y, edges, rc, SKIN)
    goff, gj = e.export_pairs()
    assert np.array_equal(goff, off) and np.array_equal(gj, j)
    e.compute(stats=True)
    E = e.stats()[0][0]           # a pair at distance 0 would have raised the range flag
    F, Eo, _, _ = O.forces(y, edges, np.zeros(n, np.int32), EPS * one, one, rc, off, j)
    rms = np.sqrt((F ** 2).sum(1).mean())
    assert np.sqrt(((e.forces() - F) ** 2).sum(1)).max() / rms <= 1e-5
    assert abs(E - Eo.sum()) / np.abs(Eo).sum() <= 1e-6
    e.close()

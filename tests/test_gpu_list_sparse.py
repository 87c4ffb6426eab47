"""The list build of large dilute systems and of batches of small boxes (a
window per atom) against the oracle's pair sets and, entry for entry, against
the build by tiles, which the same engine takes once it has met long lists, or a
smaller batch: FP64 forces are summed in list order.  Both sides of the rule,
remainders of a wavefront's atoms, whole-box windows, lists that outgrow their
capacity, replicas."""
import numpy as np
import pytest

from oracle import oracle as O
from sre import Engine
from sre.engine import forces_static

pytestmark = pytest.mark.gpu

ONE = np.ones((1, 1), np.float32)


def gas(n, box, seed):
    """n atoms on a jittered lattice, all sites at least 0.8 apart."""
    rng = np.random.default_rng(seed)
    c = np.maximum(1, np.floor(box / (np.prod(box.astype(float)) / n) ** (1 / 3))).astype(int)
    while np.prod(c) < n:
        c[np.argmax(box / c)] += 1
    site = np.stack(np.unravel_index(rng.permutation(np.prod(c))[:n], c), 1)
    d = box / c
    x = (site + 0.5) * d + rng.uniform(-0.5, 0.5, (n, 3)) * np.maximum(d - 0.8, 0.0)
    xyz = np.zeros((n, 4), np.float32)
    xyz[:, :3] = np.mod(x, box)
    return xyz


def with_drop(xyz, box, rc):
    """The same with 1 000 atoms in a drop: lists of a liquid."""
    y = xyz.copy()
    g = np.stack(np.unravel_index(np.arange(1000), (10, 10, 10)), 1) * 1.1
    y[:1000, :3] = np.mod(0.5 * box + g - 5.0, box)
    return y


def engine(ns, boxes, table, prec, lanes):
    e = Engine(skin=0.3, precision=prec)
    e.set_tuning(force_lanes=lanes)
    e.set_system(ns, boxes)
    e.set_types(np.zeros(sum(ns), np.int32))
    e.set_pair_params(0.1 * ONE, ONE)
    for r in range(len(ns)):
        e.set_rc_table(table, replica=r)
    return e


# atoms, box, (rc_min, rc_max), rc bins
CASES = [
    (40000, (100.0, 100.0, 200.0), (2.5, 2.5), 1),
    (40017, (110.0, 90.0, 170.0), (2.5, 5.0), 16),
    (100001, (240.0, 240.0, 240.0), (2.5, 3.4), 64),
    (40961, (7.1, 7.4, 40000.0), (3.0, 3.0), 1),     # whole box along x and y
    (39999, (100.0, 100.0, 200.0), (2.5, 2.5), 1),   # below the rule: tiles
]


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("lanes", [1, 4, 16])
def test_lists_equal_oracle_and_tiles(torch_cuda, case, lanes):
    n, box, (lo, hi), nz = CASES[case]
    box = np.asarray(box, np.float32)
    table = np.linspace(lo, hi, nz).astype(np.float32).reshape(1, 1, nz)
    xyz = gas(n, box, case)
    rc, _ = O.assign_rc(xyz, box, table)
    off, j = O.build_pairs(xyz, box, rc, 0.3)
    out = []
    for long_lists_first in (False, True):
        e = engine([n], [box], table, "fp64", lanes)
        if long_lists_first:
            e.upload_positions(with_drop(xyz, box, hi))
            e.rebuild()
            assert e.neighbor_count(in_rc=False)[2] > 48
        e.upload_positions(xyz)
        e.rebuild()
        goff, gj = e.export_pairs()
        assert np.array_equal(goff, off) and np.array_equal(gj, j)
        assert e.neighbor_count(in_rc=False) == (int(off[-1]), -1, int(np.diff(off).max()))
        e.compute(stats=True)
        out.append((e.forces(), e.stats()))
        e.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("prec", ["mixed", "fp64"])
def test_first_lists_outgrow_the_capacity(torch_cuda, prec):
    """A drop in a large box: a low mean density, so the first build has a
    window per atom and little room; the next build is by tiles."""
    n, box = 50001, np.array([150.0, 150.0, 150.0], np.float32)
    xyz = with_drop(gas(n, box, 7), box, 3.0)
    table = np.full((1, 1, 1), 3.0, np.float32)
    rc, _ = O.assign_rc(xyz, box, table)
    off, j = O.build_pairs(xyz, box, rc, 0.3)
    assert np.diff(off).max() > 2 * 4.19 * 3.3 ** 3 * n / np.prod(box.astype(float)) + 32
    e = engine([n], [box], table, prec, 4)
    e.upload_positions(xyz)       # (the drop lies over gas atoms: lists alone)
    for _ in range(2):
        e.rebuild()
        goff, gj = e.export_pairs()
        assert np.array_equal(goff, off) and np.array_equal(gj, j)
    e.close()


def test_replicas(torch_cuda):
    ns = [30001, 500, 15007]
    boxes = np.array([[120, 120, 120], [40, 30, 20], [90, 95, 100]], np.float32)
    table = np.linspace(2.5, 3.5, 8).astype(np.float32).reshape(1, 1, 8)
    xs = [gas(n, b, 11 + r) for r, (n, b) in enumerate(zip(ns, boxes))]
    e = engine(ns, boxes, table, "mixed", 4)
    e.upload_positions(np.concatenate(xs))
    e.rebuild()
    goff, gj = e.export_pairs()
    e.close()
    first = 0
    for x, b in zip(xs, boxes):
        rc, _ = O.assign_rc(x, b, table)
        off, j = O.build_pairs(x, b, rc, 0.3)
        o = goff[first:first + len(x) + 1]
        assert np.array_equal(o - o[0], off)
        assert np.array_equal(gj[o[0]:o[-1]] - first, j)
        first += len(x)


# box, cutoff, replicas: columns that a tile's window fills, second images along
# both or one of x and y, plates, replicas of which most atoms want it or do not
BATCHES = [
    [((8.1, 8.1, 8.1), 2.5, 46)],
    [((6.1, 6.3, 5.9), 2.5, 360)],
    [((7.3, 22.0, 22.0), 2.5, 18)],
    [((16.8, 16.8, 5.75), 2.5, 38)],
    [((11.0, 11.1, 11.05), 3.5, 21)],
    [((15.45, 15.45, 15.45), 5.0, 6)],
    [((16.55, 16.6, 16.55), 5.0, 25)],          # above 80 000 atoms
    [((8.1, 8.1, 8.1), 2.5, 40), ((14.0, 14.0, 14.0), 2.5, 3)],
    [((8.1, 8.1, 8.1), 2.5, 20), ((14.0, 14.0, 14.0), 2.5, 6)],
    [((8.1, 8.1, 8.1), 2.5, 91), ((14.0, 14.0, 14.0), 2.5, 32)],   # a third, 80 000
]


@pytest.mark.parametrize("batch", range(len(BATCHES)))
@pytest.mark.parametrize("lanes", [4, 16])
def test_batches_of_small_boxes(torch_cuda, batch, lanes):
    rng = np.random.default_rng(batch)
    ns, boxes, xs, rc = [], [], [], 0.0
    for box, rc, copies in BATCHES[batch]:
        box = np.asarray(box, np.float32)
        c = np.maximum(1, np.floor(box / 1.1)).astype(int)
        for _ in range(copies):
            n = int(np.prod(c)) - rng.integers(0, 9)
            s = np.stack(np.unravel_index(rng.permutation(np.prod(c))[:n], c), 1)
            x = np.zeros((n, 4), np.float32)
            x[:, :3] = np.mod((s + 0.5 + rng.uniform(-0.07, 0.07, (n, 3))) * (box / c), box)
            ns.append(n)
            boxes.append(box)
            xs.append(x)
    table = np.full((1, 1, 1), rc, np.float32)

    def run(which):
        e = engine([ns[r] for r in which], np.array([boxes[r] for r in which]), table, "fp64", lanes)
        e.upload_positions(np.concatenate([xs[r] for r in which]))
        e.rebuild()
        off, j = e.export_pairs()
        e.compute(stats=True)
        f, a = e.forces(), e.atom_stats()
        e.close()
        return off, j, f, a

    R = len(ns)
    off, j, f, a = run(range(R))
    start = np.concatenate([[0], np.cumsum(ns)])
    few = sorted({0, 1, R - 1})            # a small batch: by tiles in all but one of the cases
    assert sum(ns[r] for r in few) < 15000 < sum(ns)
    off1, j1, f1, a1 = run(few)
    first = 0
    for r in few:
        s, n = start[r], ns[r]
        o = off[s:s + n + 1]
        rcs, _ = O.assign_rc(xs[r], boxes[r], table)
        want, wj = O.build_pairs(xs[r], boxes[r], rcs, 0.3)
        assert np.array_equal(o - o[0], want) and np.array_equal(j[o[0]:o[-1]] - s, wj)
        assert np.array_equal(f[s:s + n], f1[first:first + n])
        assert np.array_equal(a[s:s + n], a1[first:first + n])
        first += n


@pytest.mark.parametrize("n", [6003, 5997])     # both sides of the rule
def test_allocation_free_call(torch_cuda, n):
    torch = torch_cuda
    box = np.array([12.47, 51.6, 12.47], np.float32)
    c = np.array([11, 50, 11])
    rng = np.random.default_rng(n)
    s = np.stack(np.unravel_index(rng.permutation(np.prod(c))[:n], c), 1)
    xyz = np.zeros((n, 4), np.float32)
    xyz[:, :3] = np.mod((s + 0.5 + rng.uniform(-0.07, 0.07, (n, 3))) * (box / c), box)
    table = np.array([4.0], np.float32)
    x = torch.from_numpy(xyz).cuda()
    torch.cuda.synchronize()
    e = engine([n], [box], table.reshape(1, 1, 1), "mixed", 4)
    e.upload_positions(xyz)
    e.rebuild()
    off, j = e.export_pairs()
    rc, _ = O.assign_rc(xyz, box, table.reshape(1, 1, 1))
    want, wj = O.build_pairs(xyz, box, rc, 0.3)
    assert np.array_equal(off, want) and np.array_equal(j, wj)
    e.compute(stats=True)
    f, stats = e.forces(), e.stats()[0]
    e.close()
    F, st = forces_static(x, box, table, skin=0.3, eps=0.1 * ONE, sigma=ONE)
    torch.cuda.synchronize()
    assert np.array_equal(F.cpu().numpy(), f) and np.array_equal(np.asarray(st), stats)

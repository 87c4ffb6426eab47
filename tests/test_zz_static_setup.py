"""The allocation-free call's one copy of parameters, its check of the types on
the device and its two sorts (counting sort up to 30 720 cells, radix sort
above): the engine's forces bit for bit, and a bad type refused by its atom."""
import numpy as np
import pytest

from sre import Engine
from sre.engine import InvalidArgument, forces_static

pytestmark = pytest.mark.gpu


def system(n, rc, edge, species):
    rng = np.random.default_rng(n)
    m = int(edge / 1.05)
    x = np.stack(np.unravel_index(rng.permutation(m ** 3)[:n], (m, m, m)), 1)
    xyz = np.zeros((n, 4), np.float32)
    xyz[:, :3] = edge / m * (x + 0.5 + rng.uniform(-0.05, 0.05, x.shape))
    eps = np.full((species, species), 0.5, np.float32) + 0.5 * np.eye(species, dtype=np.float32)
    return (xyz, np.full(3, edge, np.float32), np.linspace(0.7 * rc, rc, 9).astype(np.float32),
            rng.integers(0, species, n).astype(np.int32), eps,
            np.ones((species, species), np.float32))


@pytest.mark.parametrize("n,rc,edge,species", [
    (1, 2.5, 20.0, 1), (257, 2.5, 20.0, 2), (1024, 2.5, 20.0, 3), (5001, 2.5, 22.0, 1),
    (16384, 2.5, 27.5, 2),
    (5001, 0.6, 40.0, 2), (16384, 0.6, 60.0, 1)])          # above 30 720 cells
def test_static_equals_engine(torch_cuda, n, rc, edge, species):
    torch = torch_cuda
    xyz, box, table, types, eps, sig = system(n, rc, edge, species)
    x, t = torch.from_numpy(xyz).cuda(), torch.from_numpy(types).cuda()
    torch.cuda.synchronize()
    e = Engine(n_types=species, skin=0.3)
    e.set_system([n], [box])
    e.set_types(types)
    e.set_pair_params(eps, sig)
    e.set_rc_table(table.reshape(1, 1, -1))
    e.bind_positions(x)
    e.rebuild()
    e.compute(stats=True)
    want, stats = e.forces(), e.stats()[0]
    e.close()
    for _ in range(2):
        F, st = forces_static(x, box, table, skin=0.3, types=t, eps=eps, sigma=sig,
                              n_types=species)
        torch.cuda.synchronize()
        assert np.array_equal(F.cpu().numpy(), want)
        assert np.array_equal(np.asarray(st), stats)
    if species == 1:
        F, _ = forces_static(x, box, table, skin=0.3, eps=eps, sigma=sig)
        assert np.array_equal(F.cpu().numpy(), want)


@pytest.mark.parametrize("bad", [-1, 2, 255, 256, 2 ** 30, -2 ** 31])
def test_bad_type_is_named(torch_cuda, bad):
    torch = torch_cuda
    xyz, box, table, types, eps, sig = system(3000, 2.5, 20.0, 2)
    types[[1234, 2100]] = bad
    x, t = torch.from_numpy(xyz).cuda(), torch.from_numpy(types).cuda()
    F = torch.full((3000, 3), 7.0, dtype=torch.float64, device="cuda")
    with pytest.raises(InvalidArgument, match=f"type of atom 1234 is {bad}"):
        forces_static(x, box, table, skin=0.3, types=t, eps=eps, sigma=sig, n_types=2, forces=F)
    with pytest.raises(InvalidArgument, match="type of atom 1234"):     # before a small box
        forces_static(x, box, table * 9, skin=0.3, types=t, eps=eps, sigma=sig, n_types=2,
                      forces=F)
    assert bool((F == 7.0).all())

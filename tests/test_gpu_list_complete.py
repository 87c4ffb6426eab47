"""Lists that nothing is missing from: after adaptive MD that outgrew its
capacity behind queued stretches, and in a box whose cells are a large part of
it, with both tile sizes of the list build."""
import numpy as np
import pytest

from oracle import oracle as O
from sre import Engine

pytestmark = pytest.mark.gpu

ONE = np.ones((1, 1), np.float32)


def engine(n, box, rc, eps=1.0):
    e = Engine(skin=0.3)
    e.set_system([n], [np.asarray(box, np.float32)])
    e.set_types(np.zeros(n, np.int32))
    e.set_pair_params(eps * ONE, ONE)
    e.set_rc_table(np.full((1, 1, 1), rc, np.float32))
    return e


@pytest.mark.parametrize("n,lz", [(20001, 500.0), (80007, 2000.0)])
@pytest.mark.parametrize("lanes", [4, 16])
def test_second_images_at_both_tile_sizes(torch_cuda, n, lz, lanes):
    box = np.array([21.0, 21.0, lz], np.float32)
    xyz = np.zeros((n, 4), np.float32)
    xyz[:, :3] = np.random.default_rng(n).random((n, 3)) * box
    e = engine(n, box, 7.5)
    e.set_tuning(force_lanes=lanes)
    e.upload_positions(xyz)
    e.rebuild()
    rc, _ = O.assign_rc(xyz, box, np.full((1, 1, 1), 7.5, np.float32))
    off, j = O.build_pairs(xyz, box, rc, 0.3)
    goff, gj = e.export_pairs()
    e.close()
    assert np.array_equal(goff, off) and np.array_equal(gj, j)


def test_md_keeps_no_list_that_was_cut(torch_cuda):
    """A lattice squeezed along z to three times its density, in runs of many
    lengths: the exported lists (what the build stored) hold every entry that
    it counted, at the end of each run."""
    torch = torch_cuda
    dt, rc, nx, nz, ax, az, squeeze, steps = 0.004, 4.0, 12, 24, 1.1, 3.0, 0.36, 300
    x = np.stack(np.meshgrid(np.arange(nx), np.arange(nx), np.arange(nz), indexing="ij"), -1)
    x = (x.reshape(-1, 3) + 0.5) * np.array([ax, ax, az])
    n = len(x)
    box = np.array([nx * ax, nx * ax, nz * az], np.float32)
    xyz = np.zeros((n, 4), np.float32)
    xyz[:, :3] = x
    v = np.zeros((n, 3), np.float32)
    v[:, 2] = (x[:, 2] - 0.5 * nz * az) * (squeeze - 1.0) / (dt * steps)
    e = engine(n, box, rc, 0.01)
    pos = torch.from_numpy(xyz).cuda()
    torch.cuda.synchronize()
    e.bind_positions(pos)
    e.set_masses([1.0])
    e.set_velocities(v)
    e.set_integrator(dt, None, 1.0, 0.5, remove_com=False)
    longest = []
    for c in [7, 1, 20, 33, 2, 60, 41, 56, 80]:
        e.md_run(c, rebuild_every="adaptive", stats=True)
        off, _ = e.export_pairs()
        total, _, mx = e.neighbor_count(in_rc=False)
        assert off[-1] == total and np.diff(off).max() == mx
        longest.append(mx)
    # the capacity of the first lists, twice the mean density's, was outgrown
    assert longest[-1] > 2 * 4.19 * (rc + 0.3) ** 3 / (ax * ax * az) + 32 > longest[0]
    e.close()

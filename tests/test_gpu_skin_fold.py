"""The displacement test whose largest value the refresh itself reduces (up to
65 536 atoms) or a launch of its own: one atom moved to either side of half the
skin, in the first, a middle and the last wavefront, at the edges of a block
and of that rule; the largest since the rebuild is kept until the next one."""
import numpy as np
import pytest

from sre import Engine

pytestmark = pytest.mark.gpu

SKIN = 0.4


@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 5000, 65535, 65536, 65537])
def test_one_atom_over_half_the_skin(torch_cuda, n):
    torch = torch_cuda
    m = max(5, int(np.ceil(n ** (1.0 / 3.0))))
    xyz = np.zeros((n, 4), np.float32)
    xyz[:, :3] = 1.2 * (np.stack(np.unravel_index(np.arange(n), (m, m, m)), 1) + 0.5)
    e = Engine(skin=SKIN)
    e.set_system([n], [np.full(3, 1.2 * m, np.float32)])
    e.set_types(np.zeros(n, np.int32))
    one = np.ones((1, 1), np.float32)
    e.set_pair_params(one, one)
    e.set_rc_table(np.full((1, 1, 1), 2.0, np.float32))
    pos = torch.from_numpy(xyz.copy()).cuda()
    torch.cuda.synchronize()
    e.bind_positions(pos)

    def move(i, dx):
        p = xyz.copy()
        p[i, 0] += np.float32(dx)
        pos.copy_(torch.from_numpy(p))
        torch.cuda.synchronize()

    for i in sorted({0, n // 2, n - 1}):
        move(0, 0.0)
        e.rebuild()
        assert e.update_positions() is False
        move(i, 0.49 * SKIN)
        assert e.update_positions() is False
        move(i, 0.51 * SKIN)
        assert e.update_positions() is True
        move(i, 0.0)
        assert e.update_positions() is True      # since the rebuild
        e.rebuild()
        assert e.update_positions() is False
    e.close()

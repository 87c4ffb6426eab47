"""The velocity factors worked out by the drift's own blocks (up to 131 072
atoms) or by a launch of their own (above), at the edges of a block's 256
atoms and of that rule: a lattice too wide for any force, thermostat and
centre-of-mass removal, against the FP64 oracle's steps."""
import numpy as np
import pytest

from oracle import md as M
from sre import Engine

pytestmark = pytest.mark.gpu

DT, STEPS, A = 0.004, 3, 1.5
# three steps of some six FP32 roundings (6e-8) each move a velocity by at most
# 1.1e-6 of the largest one
TOL_V = 2e-6


@pytest.mark.parametrize("policy", ["adaptive", 2, 0])
@pytest.mark.parametrize("n", [64, 255, 256, 257, 4099, 131072, 131073])
def test_free_flight_matches_oracle(torch_cuda, n, policy):
    m = max(4, int(np.ceil(n ** (1.0 / 3.0))))
    rng = np.random.default_rng(n)
    xyz = np.zeros((n, 4), np.float32)
    xyz[:, :3] = A * (np.stack(np.unravel_index(np.arange(n), (m, m, m)), 1) + 0.5)
    box = np.full(3, A * m, np.float32)
    v0 = (rng.normal(size=(n, 3)) + 0.3).astype(np.float32)
    e = Engine(skin=0.4)
    e.set_system([n], [box])
    e.set_types(np.zeros(n, np.int32))
    one = np.ones((1, 1), np.float32)
    e.set_pair_params(one, one)
    e.set_rc_table(np.full((1, 1, 1), 1.0, np.float32))
    pos = torch_cuda.from_numpy(xyz.copy()).cuda()
    torch_cuda.cuda.synchronize()
    e.bind_positions(pos)
    e.set_masses([1.0])
    e.set_velocities(v0)
    e.set_integrator(DT, "nhc2", 1.5, 0.2, remove_com=True)
    e.md_run(1, rebuild_every=policy)
    e.md_run(STEPS - 1, rebuild_every=policy)
    x1, v1, st = pos.cpu().numpy()[:, :3], e.velocities(), e.md_state()
    e.close()
    nhc = M.NHC2(n, 1.5, 0.2)
    zero = np.zeros((n, 3))
    xo, vo, _, rec = M.md_run(xyz[:, :3], v0, np.ones(n), lambda x: zero, DT, STEPS, nhc=nhc,
                              com=True, box=box)
    top = np.abs(v0).max()
    assert np.abs(v1 - vo).max() <= TOL_V * top
    d = x1 - xo
    d -= box * np.round(d / box)
    # the drift of those velocities and three roundings of a coordinate
    assert np.abs(d).max() <= STEPS * DT * TOL_V * top + 2 * STEPS * 6e-8 * box[0]
    assert abs(st["kinetic"] - rec[-1][0]) <= 2 * TOL_V * rec[-1][0]
    for k in ("xi1", "xi2"):
        assert abs(st[k] - getattr(nhc, k)) < 1e-6 * max(abs(getattr(nhc, k)), 1.0)
    for k in ("vxi1", "vxi2"):
        assert abs(st[k] - getattr(nhc, k)) < 1e-5 * max(abs(getattr(nhc, k)), 1e-3)

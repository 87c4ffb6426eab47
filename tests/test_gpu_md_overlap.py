"""Adaptive MD stretches queued while the list before them is still being
built: lists that outgrow their capacity (a lattice squeezed along z to three
times its density) are found a stretch later, and the stretch is run again.
The trajectory, the list and the statistics are those of the per-step check."""
import numpy as np
import pytest

from sre import Engine

pytestmark = pytest.mark.gpu

DT, STEPS, RC, SKIN = 0.004, 300, 4.0, 0.3
NX, NZ, AX, AZ = 12, 24, 1.1, 3.0
SQUEEZE = 0.36            # final over initial spacing along z


def run(torch, policy, chunks, sort_mode, thermostat=None):
    x = np.stack(np.meshgrid(np.arange(NX), np.arange(NX), np.arange(NZ), indexing="ij"), -1)
    x = (x.reshape(-1, 3) + 0.5) * np.array([AX, AX, AZ])
    n = len(x)
    xyz = np.zeros((n, 4), np.float32)
    xyz[:, :3] = x
    v = np.zeros((n, 3), np.float32)
    v[:, 2] = (x[:, 2] - 0.5 * NZ * AZ) * (SQUEEZE - 1.0) / (DT * STEPS)
    box = np.array([NX * AX, NX * AX, NZ * AZ], np.float32)
    e = Engine(skin=SKIN)
    e.set_tuning(sort_mode=sort_mode)
    e.set_system([n], [box])
    e.set_types(np.zeros(n, np.int32))
    one = np.ones((1, 1), np.float32)
    e.set_pair_params(0.01 * one, one)
    e.set_rc_table(np.full((1, 1, 1), RC, np.float32))
    pos = torch.from_numpy(xyz).cuda()
    torch.cuda.synchronize()
    e.bind_positions(pos)
    e.set_masses([1.0])
    e.set_velocities(v)
    e.set_integrator(DT, thermostat, 1.0, 0.5, remove_com=False)
    counts = []
    for c in chunks:
        e.md_run(c, rebuild_every=policy, stats=True)
        counts.append(e.neighbor_count(in_rc=False))
    out = pos.cpu().numpy().copy(), e.velocities(), e.forces_fixed()
    e.rebuild()
    last = e.neighbor_count(in_rc=False)
    e.close()
    return out, counts, last


@pytest.mark.parametrize("sort_mode", [0, 1])
def test_outgrown_lists_are_rebuilt(torch_cuda, sort_mode):
    guess = 2 * 4.19 * (RC + SKIN) ** 3 / (AX * AX * AZ) + 32   # the first capacity, or more
    (x0, v0, f0), _, last0 = run(torch_cuda, 0, [STEPS], sort_mode)
    assert last0[2] > guess                      # at least one overflow on the way
    for chunks in ([STEPS], [1, 140, 59, STEPS - 200]):
        (x1, v1, f1), counts, last1 = run(torch_cuda, "adaptive", chunks, sort_mode)
        assert np.array_equal(x0, x1) and np.array_equal(v0, v1) and np.array_equal(f0, f1)
        assert last0 == last1
        for total, _, longest in counts:         # never a list that was cut short
            assert longest >= total / len(x0)
        assert counts[-1][2] >= 0.8 * last1[2]

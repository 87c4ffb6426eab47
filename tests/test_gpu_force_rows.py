"""The force launch whose blocks share a tile (no statistics, at most one tile
per SIMD): the forces of the launch with statistics, bit for bit, for every
lane map, at remainders of a tile, with empty and short lists, two species, a
tail; and the same refusal of overlapping atoms."""
import numpy as np
import pytest

from sre import Engine
from sre.engine import ForceRange

pytestmark = pytest.mark.gpu


def engine(n, lanes, species, rc, tail, spacing=1.05, seed=0):
    rng = np.random.default_rng(seed + n)
    m = max(int(np.ceil(n ** (1.0 / 3.0))), int(np.ceil(2.0 * (rc + 0.3) / spacing)) + 1)
    site = rng.permutation(m ** 3)[:n] if spacing > 2 else np.arange(n)
    xyz = np.zeros((n, 4), np.float32)
    xyz[:, :3] = spacing * (np.stack(np.unravel_index(site, (m, m, m)), 1) + 0.5
                            + rng.uniform(-0.06, 0.06, (n, 3)))
    box = np.full(3, spacing * m, np.float32)
    e = Engine(n_types=species, skin=0.3)
    e.set_tuning(force_lanes=lanes)
    e.set_system([n], [box])
    e.set_types((np.arange(n) % 3 % species).astype(np.int32))
    eps = np.ones((species, species), np.float32) * np.float32(0.9)
    e.set_pair_params(eps, np.ones((species, species), np.float32))
    e.set_rc_table(np.linspace(0.8 * rc, rc, 8).astype(np.float32).reshape(1, 1, 8))
    if tail:
        e.set_density_profile(np.full((species, 16), n / float(np.prod(box)) / species))
    e.upload_positions(xyz)
    e.rebuild()
    return e, xyz


@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("n,species,rc,tail,spacing", [
    (1, 1, 2.5, False, 1.05), (17, 1, 2.5, True, 1.05), (200, 1, 2.5, False, 2.9),
    (1000, 2, 3.1, True, 1.05), (4097, 1, 2.5, False, 1.05), (3001, 2, 5.0, False, 1.05),
    (16385, 1, 2.5, True, 1.05)])
def test_forces_equal_unsplit(torch_cuda, lanes, n, species, rc, tail, spacing):
    e, _ = engine(n, lanes, species, rc, tail, spacing)
    e.compute(stats=True, tail=tail)
    want = e.forces_fixed()
    e.compute(stats=False, tail=tail)
    got = e.forces_fixed()
    e.close()
    assert np.array_equal(got, want)


@pytest.mark.parametrize("stats", [False, True])
def test_overlap_is_refused(torch_cuda, stats):
    e, xyz = engine(500, 4, 1, 2.5, False)
    xyz[3, :3] = xyz[4, :3]
    xyz[3, 0] += 0.02
    e.upload_positions(xyz)
    e.rebuild()
    e.compute(stats=stats)
    with pytest.raises(ForceRange):
        e.forces()
    e.close()

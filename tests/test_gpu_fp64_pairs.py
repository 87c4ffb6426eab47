"""The FP64 pair evaluation (reciprocal by refinement, fused multiply-adds)
over the distances it meets, one dimer at a time, for each lane map, one and
two species, and remainders of a wavefront's atoms."""
import numpy as np
import pytest

from sre import Engine

pytestmark = pytest.mark.gpu

RC, BOX = 4.0, 96.0
# |dF| against the sum of the magnitudes of the two terms: 14 relative errors
# of a distance >= 0.7, whose components carry the residual's rounding (2^-25
# of a lattice step of 2.3e-8) and two of the displacement's (<= 4e-16 each),
# below 3e-14, and some 20 roundings of 1.1e-16
TOL = 1e-13


def dimers(n_pairs, seed):
    """Dimers on a grid of 12: distances 0.7 to 3.9, no pair between dimers."""
    rng = np.random.default_rng(seed)
    r = np.linspace(0.7, 3.9, n_pairs) if n_pairs > 1 else np.array([0.9])
    u = rng.normal(size=(n_pairs, 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    g = np.stack(np.unravel_index(np.arange(n_pairs), (8, 8, 8)), 1) * 12.0 + 4.0
    xyz = np.zeros((2 * n_pairs, 4), np.float32)
    xyz[0::2, :3] = g
    xyz[1::2, :3] = g + r[:, None] * u
    return xyz


def engine(xyz, lanes, types, sig, eps):
    e = Engine(skin=0.3, n_types=len(eps), precision="fp64")
    e.set_tuning(force_lanes=lanes)
    e.set_system([len(xyz)], [np.full(3, BOX, np.float32)])
    e.set_types(types)
    e.set_pair_params(eps, sig)
    e.set_rc_table(np.full((1, 1, 1), RC, np.float32))
    e.upload_positions(xyz)
    e.rebuild()
    return e


@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("n_pairs,species", [(1, 1), (37, 1), (512, 1), (509, 2)])
def test_dimers_match_float64(torch_cuda, lanes, n_pairs, species):
    xyz = dimers(n_pairs, 5 + n_pairs)
    types = (np.arange(2 * n_pairs) % 3 % species).astype(np.int32)
    eps = np.ones((species, species), np.float32)
    sig = np.ones((species, species), np.float32)
    if species == 2:
        eps[1, 1], sig[1, 1] = 0.5, 0.75
        eps[0, 1] = eps[1, 0] = 0.75
        sig[0, 1] = sig[1, 0] = 0.875
    e = engine(xyz, lanes, types, sig, eps)
    out = []
    for stats in (False, True):
        e.compute(stats=stats)
        out.append(e.forces())
    E = e.atom_stats()[:, 0]
    e.close()
    d = xyz[0::2, :3].astype(np.float64) - xyz[1::2, :3].astype(np.float64)
    r2 = (d * d).sum(1)
    ep = eps[types[0::2], types[1::2]].astype(np.float64)
    s6 = (sig[types[0::2], types[1::2]].astype(np.float64) ** 2 / r2) ** 3
    f = (ep * (48 * s6 * s6 - 24 * s6) / r2)[:, None] * d
    scale = ep * (48 * s6 * s6 + 24 * s6) / np.sqrt(r2)
    for F in out:
        assert np.all(np.abs(F[0::2] - f).max(1) <= TOL * scale)
        assert np.all(np.abs(F[1::2] + f).max(1) <= TOL * scale)
    pe = 0.5 * ep * 4 * (s6 * s6 - s6)
    assert np.all(np.abs(E[0::2] - pe) <= TOL * ep * 2 * (s6 * s6 + s6))
    assert np.array_equal(E[0::2], E[1::2])


@pytest.mark.parametrize("lanes", [4, 16])
def test_coincident_atoms_have_infinite_energy(torch_cuda, lanes):
    xyz = dimers(3, 1)
    xyz[3] = xyz[2]
    one = np.ones((1, 1), np.float32)
    e = engine(xyz, lanes, np.zeros(6, np.int32), one, one)
    e.compute(stats=True)
    E = e.atom_stats()[:, 0]
    e.close()
    assert np.all(np.isposinf(E[2:4]))
    assert np.all(np.isfinite(E[[0, 1, 4, 5]]))

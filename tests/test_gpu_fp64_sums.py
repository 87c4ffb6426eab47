"""The FP64 form's sums over whole lists (the pipelined loop: odd and even
numbers of row groups, masked rows, partial tiles; and the loop of short lists,
with empty ones) against a float64 evaluation of the same pairs on
the host, and a coordinate that is no number."""
import numpy as np
import pytest

from sre import Engine

pytestmark = pytest.mark.gpu

RC = 2.5
# per pair, of the sum of the magnitudes of the force's (or energy's) two
# terms: the displacement's error (lattice step 7e-9 times 2^-25 for each
# residual, one rounding of a component below 2.8: 7e-16 of a distance >= 0.9,
# 14 times over in r^-14) 1.1e-14; some 20 roundings in either evaluation,
# 4.4e-15; at most 120 additions of a list, 1.4e-14
TOL = 5e-14


def engine(xyz, box, lanes, eps, sig, types, rc=RC):
    e = Engine(n_types=len(eps), skin=0.3, precision="fp64")
    e.set_tuning(force_lanes=lanes)
    e.set_system([len(xyz)], [box])
    e.set_types(types)
    e.set_pair_params(eps, sig)
    e.set_rc_table(np.full((1, 1, 1), rc, np.float32))
    e.upload_positions(xyz)
    e.rebuild()
    return e


@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("n,species,spacing", [
    (343, 1, 1.05), (1327, 2, 1.05), (4095, 1, 1.05),
    (1327, 2, 1.9), (2001, 1, 2.4)])      # short lists: from 8 lanes on, for all lanes
def test_list_sums_match_float64(torch_cuda, lanes, n, species, spacing):
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    xyz = np.zeros((n, 4), np.float32)
    site = np.stack(np.unravel_index(rng.permutation(m ** 3)[:n], (m, m, m)), 1)
    xyz[:, :3] = spacing * (site + 0.5 + rng.uniform(-0.06, 0.06, (n, 3)))
    box = np.full(3, spacing * m, np.float32)
    types = (np.arange(n) % 3 % species).astype(np.int32)
    eps = np.array([[1.0, 0.75], [0.75, 0.5]], np.float32)[:species, :species]
    sig = np.array([[1.0, 0.875], [0.875, 0.75]], np.float32)[:species, :species]
    e = engine(xyz, box, lanes, eps, sig, types)
    off, j = e.export_pairs()
    e.compute(stats=False)
    plain = e.forces()
    e.compute(stats=True)
    F, A = e.forces(), e.atom_stats()
    e.close()
    i = np.repeat(np.arange(n), np.diff(off))
    x = xyz[:, :3].astype(np.float64)
    L = box.astype(np.float64)
    d = x[j] - x[i]
    d -= L * np.rint(d / L)
    r2 = (d * d).sum(1)
    assert np.abs(r2 - RC * RC).min() > 1e-6     # no pair that rounding decides
    k = r2 < RC * RC
    i, j, d, r2 = i[k], j[k], d[k], r2[k]
    ep = eps[types[i], types[j]].astype(np.float64)
    s6 = (sig[types[i], types[j]].astype(np.float64) ** 2 / r2) ** 3
    fs = ep * (24 * s6 - 48 * s6 * s6) / r2
    mag = ep * (24 * s6 + 48 * s6 * s6) / np.sqrt(r2)
    scale = np.bincount(i, mag, n)
    want = np.stack([np.bincount(i, fs * d[:, c], n) for c in range(3)], 1)
    assert np.all(np.abs(F - want).max(1) <= TOL * scale)
    assert np.array_equal(F, plain)
    pe = 0.5 * np.bincount(i, 4 * ep * (s6 * s6 - s6), n)
    assert np.all(np.abs(A[:, 0] - pe)
                  <= TOL * 0.5 * np.bincount(i, 4 * ep * (s6 * s6 + s6), n))
    vir = np.stack([0.5 * np.bincount(i, fs * d[:, c] ** 2, n) for c in range(3)], 1)
    assert np.all(np.abs(A[:, 1:] - vir).max(1)
                  <= TOL * 0.5 * np.bincount(i, mag * np.sqrt(r2), n))


@pytest.mark.parametrize("lanes", [4, 16])
def test_undefined_position_has_undefined_energy(torch_cuda, lanes):
    """Such an atom's lattice coordinate is 0 (cells, lists and tables stay in
    range); its residual keeps what the coordinate was, and so do the sums."""
    xyz = np.zeros((5, 4), np.float32)
    xyz[:, :3] = 10.0
    xyz[:, 0] = [np.nan, 1.1, 8.0, 9.2, 14.0]
    one = np.ones((1, 1), np.float32)
    e = engine(xyz, np.full(3, 20.0, np.float32), lanes, one, one, np.zeros(5, np.int32))
    off, j = e.export_pairs()
    e.compute(stats=True)
    E = e.atom_stats()[:, 0]
    e.close()
    assert list(np.diff(off)) == [1, 1, 1, 1, 0]
    assert np.all(np.isnan(E[:2])) and np.all(np.isfinite(E[2:]))

"""The tail's adjoint where most bins of the cutoff profile hold no atoms (they
are left out) and where one species is absent from some: the gradients are the
oracle's, and zero in the empty bins.  Tolerances as for the full slab: FP64
pair terms to round-off, the oracle's rc derivatives are central differences."""
import numpy as np
import pytest

from oracle import oracle as O
from sre import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("species", [1, 2, 3])
@pytest.mark.parametrize("bins", [40, 130])
def test_gradients_equal_oracle(torch_cuda, species, bins):
    torch = torch_cuda
    rng = np.random.default_rng(10 * bins + species)
    n, box = 600, np.array([9.0, 9.0, 36.0], np.float32)
    site = np.stack(np.unravel_index(rng.permutation(8 * 8 * 10)[:n], (8, 8, 10)), 1)
    xyz = np.zeros((n, 4), np.float32)
    xyz[:, :3] = 1.125 * (site + 0.5 + rng.uniform(-0.05, 0.05, (n, 3))) + [0.0, 0.0, 9.0]
    types = np.minimum((xyz[:, 2] - 9.0) // 4.0, species - 1).astype(np.int32)   # in layers
    eps = (0.5 + rng.random((species, species))).astype(np.float32)
    sig = (0.8 + 0.1 * rng.random((species, species))).astype(np.float32)
    eps, sig = (eps + eps.T) / 2, (sig + sig.T) / 2
    table = np.linspace(2.5, 3.5, bins).astype(np.float32).reshape(1, 1, bins)
    rho = 0.2 + 0.5 * rng.random((species, bins))
    e = Engine(n_types=species, skin=0.3, precision="fp64")
    e.set_system([n], [box])
    e.set_types(types)
    e.set_pair_params(eps, sig)
    e.set_rc_table(table)
    e.set_density_profile(rho)
    e.upload_positions(xyz)
    e.rebuild()
    e.compute(stats=True, tail=True)
    g = rng.normal(size=(n, 3))
    gpu = torch.from_numpy(g).cuda()
    torch.cuda.synchronize()
    ge, gs, grc = e.adjoint(dLdE=[0.7], dLdF=gpu, tail=True, n_rc=bins)
    pge, pgs, _ = e.adjoint(dLdE=[0.7], dLdF=gpu, tail=False)
    e.close()
    rc, _ = O.assign_rc(xyz, box, table)
    off, j = O.build_pairs(xyz, box, rc, 0.3)
    pe, ps = O.grad_pairs(xyz, box, types, eps, sig, rc, off, j, 0.7, g)
    te, ts, trc = O.grad_tail(xyz, box, types, eps, sig, table.ravel(), rho, 0.7, g, h=1e-4)
    # the tail's part (the pairs' exact totals, of terms rounded to 2^-32, cancel)
    assert np.abs(ge - pge - te).max() <= 1e-8 * np.abs(pe + te).max()
    assert np.abs(gs - pgs - ts).max() <= 1e-8 * np.abs(ps + ts).max()
    np.testing.assert_allclose(grc, trc, rtol=1e-6, atol=1e-6 * np.abs(trc).max())
    used = np.unique((xyz[:, 2] * np.float32(bins) / box[2]).astype(int))
    empty = np.setdiff1d(np.arange(bins), used)
    assert len(empty) > bins // 2 and np.all(grc[empty] == 0.0) and np.any(grc[used] != 0.0)

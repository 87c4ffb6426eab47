"""The error estimate's transforms on grids at the edges of their kernel's
tiles: one cell, one tile of outputs and one more, both line counts per block,
the largest edge of the matrix-core form and the first one beyond it.  The
device's own kernel tables go through numpy's FFT; a transform of n terms per
axis may differ from it by the rounding of its sums, n 2^-52 per axis times
the sum of the terms' magnitudes (twice, for the two of them)."""
import numpy as np
import pytest

from oracle import arc as A
from sre import Arc

pytestmark = pytest.mark.gpu

BOXES = [(1.2, 1.4, 1.9), (3.5, 17.2, 1.1), (31.4, 33.3, 5.2), (61.3, 3.3, 59.4),
         (5.5, 63.2, 9.1), (9.3, 7.3, 121.6), (227.3, 1.5, 3.3), (3.3, 3.1, 227.9),
         (3.2, 229.4, 5.3)]


@pytest.mark.parametrize("box", BOXES)
def test_errors_equal_numpy_fft(torch_cuda, box):
    arc = Arc(box, 1.0)
    arc.set_candidates(2.5, 3.5, 0.5)
    rng = np.random.default_rng(int(10 * sum(box)))
    rho = 0.1 + 0.7 * rng.random(arc.dims)
    arc.set_density(rho)
    arc.cal_error(keep_parts=True)
    err, parts = arc.errors(parts=True)
    S1, G = arc.kernels()
    kv = A.k_grid(box, arc.dims)
    want, e1, e2 = A.cal_error(rho, box, S1, G, kv, parts=True)
    V = float(np.prod(np.asarray(box, np.float32).astype(np.float64)))
    rhok = np.abs(np.fft.fftn(rho)) * (V / rho.size)
    n = sum(arc.dims)
    for c in range(len(arc.rcs)):
        for a in range(4):
            k = S1[c] if a == 0 else kv[a - 1] * G[c]
            # rho_k carries the forward transform's own rounding
            mag = (np.abs(k) * rhok).sum() / V
            fwd = np.abs(k).sum() * rho.sum() / rho.size
            tol = 2 * n * 2.0 ** -52 * (mag + fwd) + 1e-300
            ref = e1[c] if a == 0 else e2[c][a - 1]
            assert np.abs(parts[c][..., a] - ref).max() <= tol
    total = parts[..., 0] + (parts[..., 1:] ** 2).sum(-1)
    assert np.allclose(err ** 2, total, rtol=1e-13, atol=0)
    assert want.shape == err.shape
    arc.cal_rcut(0.02)
    _, _, idx = arc.result()
    assert np.array_equal(idx, A.cal_rcut(err, 0.02))
    arc.close()

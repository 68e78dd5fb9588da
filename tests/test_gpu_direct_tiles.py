"""GPU: direct summation at the edges of its source tiles and chunks, where the
tiles with and without a target of the wave meet."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n", (1, 2, 255, 256, 257, 4096, 66049))
@pytest.mark.parametrize("eps", (0.0, 1e-2))
def test_direct_sum_tile_edges(n, eps, require_gpu):
    from jaccpot_amd import direct_sum_gravitational_acceleration

    rng = np.random.default_rng(n)
    x, m = rng.uniform(-1, 1, (n, 3)), rng.uniform(0.5, 1.5, n)
    if n > 2:
        x[n // 2] = x[1]  # a coincident pair
    tgt = np.unique(np.clip([0, 1, n // 2, 63, 64, 255, 256, 257, n - 1], 0, n - 1))
    a, p = (np.asarray(torch.as_tensor(v).cpu()) for v in
            direct_sum_gravitational_acceleration(x, m, softening=eps, target_indices=tgt, return_potential=True))
    xl, ml = x.astype(np.longdouble), m.astype(np.longdouble)
    for i, t in enumerate(tgt):
        d = xl - xl[t]
        r2 = (d * d).sum(1) + np.longdouble(eps) ** 2
        keep = (np.arange(n) != t) & (r2 > 0)
        w = np.where(keep, ml / np.sqrt(np.where(keep, r2, 1)), 0)
        f = (w / np.where(keep, r2, 1))[:, None] * d
        # per term: 4 roundings in d and r2, 2 in 1/r, 3 products (1/r enters three
        # times); per sum of n terms at most n roundings of the sum of the moduli
        # (differences of coordinates of modulus <= 1 are as exact as their terms)
        bound = (n + 24) * 2.0 ** -53
        assert abs(float(p[i] + w.sum())) <= bound * float(w.sum())
        assert (np.abs((a[i] - f.sum(0)).astype(float)) <= bound * np.abs(f).sum(0).astype(float)).all()


def test_infinite_mass_acts_on_others_only(require_gpu):
    from jaccpot_amd import direct_sum_gravitational_acceleration

    rng = np.random.default_rng(5)
    x, m = rng.uniform(-1, 1, (700, 3)), rng.uniform(0.5, 1.5, 700)
    m[300] = np.inf
    a, p = (np.asarray(torch.as_tensor(v).cpu()) for v in
            direct_sum_gravitational_acceleration(x, m, softening=1e-2, target_indices=[300, 301, 699],
                                                  return_potential=True))
    assert np.isfinite(a[0]).all() and np.isfinite(p[0])
    assert np.isinf(p[1:]).all() and np.isinf(a[1:]).all()

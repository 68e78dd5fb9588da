"""Direct (rotation-free) translations against the oracle over the separations
they have to hold at, through the host instantiation of the kernels' templates.

M2L leaves its plain form where r^-(p+1) would leave the type's range: float32
cases lie on both sides of that line and on it, and the two forms have to agree
with the oracle alike.  Tolerances: a coefficient is a sum of at most (p+1)^2
products of three rounded factors, so 2e-5 (float32) and 1e-12 (float64) of the
largest coefficient of its degree, as for the operators in test_abi.py, times
16 for float32 sums whose terms cancel."""

from __future__ import annotations

import numpy as np
import pytest

from jaccpot_amd import _native as nat
from oracle import harmonics as H

OPS = {"m2m": 0, "m2l": 1, "l2l": 2, "m2l_cascade": 5}


def _apply(op, p, dtype, v, d):
    lib = nat.load()
    out = np.zeros((p + 1) ** 2)
    v = np.ascontiguousarray(v, np.float64)
    d = np.ascontiguousarray(d, np.float64)
    assert lib.jfm_host_operator(OPS[op], p, dtype, v.ctypes.data, d.ctypes.data, out.ctypes.data) == 0
    return out


def _by_degree(a, p):
    return [a[n * n:(n + 1) ** 2] for n in range(p + 1)]


@pytest.mark.parametrize("p", range(1, 9))
@pytest.mark.parametrize("scale", (1.0, 2.0 ** -20, 2.0 ** 18))
def test_translations_hold_at_every_separation(p, scale):
    """The sources of a cell of size 0.3 r; in float32 their masses keep the
    largest coefficient (p! r^-(p+1)) and the smallest inside the type's range."""
    rng = np.random.default_rng(100 * p)
    for dtype, tol in ((nat.JFM_F64, 1e-12), (nat.JFM_F32, 16 * 2e-5)):
        if dtype == nat.JFM_F32 and p > 4 and scale != 1.0:
            scale = scale ** (4.0 / p)  # the same powers of r as at order 4
        for d in (np.array([0.6, -0.5, 0.7]), np.array([0.0, 0.0, 1.0]), np.array([1.0, 0.0, 0.0]), -np.ones(3)):
            d = d * scale
            M = H.p2m(rng.uniform(-0.3, 0.3, size=(4, 3)) * scale, rng.uniform(0.5, 1.5, 4), p)
            if dtype == nat.JFM_F32:
                d, M = d.astype(np.float32).astype(np.float64), M.astype(np.float32).astype(np.float64)
            r = np.linalg.norm(d)
            L = H.m2l(M, d, p)
            if dtype == nat.JFM_F32:
                L = L.astype(np.float32).astype(np.float64)
            for op, v, ref in (("m2m", M, H.m2m(M, d, p)), ("m2l", M, H.m2l(M, d, p)), ("l2l", L, H.l2l(L, d, p))):
                for got in [_apply(op, p, dtype, v, d)] + ([_apply("m2l_cascade", p, dtype, v, d)] if op == "m2l" else []):
                    v_deg = [np.abs(x).max() for x in _by_degree(v, p)]
                    for n, (g, w) in enumerate(zip(_by_degree(got, p), _by_degree(ref, p))):
                        terms = np.abs(w).max()  # the largest term that enters the degree
                        if op == "l2l":
                            terms = max(v_deg[k] * r ** (k - n) for k in range(n, p + 1))
                        if op == "m2m":
                            terms = max(v_deg[k] * r ** (n - k) for k in range(n + 1))
                        assert np.abs(g - w).max() <= tol * terms, (op, dtype, n)


@pytest.mark.gpu
@pytest.mark.parametrize("p,leaf,exponent", ((4, 4, -18), (4, 16, -18), (3, 8, -23), (5, 8, -14), (4, 8, 18)))
def test_m2l_outside_the_plain_range(p, leaf, exponent):
    """Some pairs of a wave, all or none leave the range of the plain form (lists of
    at least 56 pairs a target and shorter ones).  Scaling all lengths by a power of
    two scales every float32 result exactly in the plain form; the scaled form may
    differ by its rounding: the float32 parity tolerance of 1e-5."""
    import torch

    from jaccpot_amd import FastMultipoleMethod
    from oracle import ics

    x, m = ics.plummer(3000, 5)
    x = x.astype(np.float32)
    f = 2.0 ** exponent
    out = []
    for scale in (1.0, f):
        fmm = FastMultipoleMethod(precision="fp32", theta=0.7, softening=2.0 ** -7 * scale)
        acc = fmm.compute_accelerations(torch.as_tensor(x * np.float32(scale)).cuda(),
                                        torch.as_tensor(m.astype(np.float32)).cuda(), leaf_size=leaf, max_order=p)
        out.append(acc.double().cpu().numpy() * scale ** 2)
    rel = np.linalg.norm(out[1] - out[0]) / np.linalg.norm(out[0])
    print(f"p {p} leaf {leaf} 2^{exponent}: rel-L2 {rel:.2e}", flush=True)
    assert rel < 1e-5

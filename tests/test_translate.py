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


@pytest.mark.parametrize("p", range(2, 6))
def test_direct_m2l_rounds_no_worse_than_the_cascade(p):
    """float32 rounding of one M2L against float64, over cells of eight masses at
    separations of 2.5 to 8 cell sizes: the potential at the target's centre and, with
    the gradient there, of the direct form and of the rotation cascade.  400 pairs
    leave the two root mean squares uncertain by 4% each, so 1.15 for the ratio."""
    rng = np.random.default_rng(p)
    err = {"m2l": np.zeros(2), "m2l_cascade": np.zeros(2)}
    for _ in range(400):
        u = rng.normal(size=3)
        d = (u / np.linalg.norm(u) * rng.uniform(2.5, 8)).astype(np.float32)
        M = H.p2m(rng.uniform(-0.5, 0.5, size=(8, 3)), rng.uniform(0.5, 1.5, 8), p).astype(np.float32)
        ref = _apply("m2l_cascade", p, nat.JFM_F64, M, d)
        for op, e in err.items():
            diff = _apply(op, p, nat.JFM_F32, M, d) - ref
            e += (diff[0] / ref[0]) ** 2, np.sum(diff[1:4] ** 2) / np.sum(ref[1:4] ** 2)
    ratio = np.sqrt(err["m2l"] / err["m2l_cascade"])
    print(p, np.sqrt(err["m2l_cascade"] / 400), ratio)
    assert np.all(ratio <= 1.15), ratio


@pytest.mark.gpu
@pytest.mark.parametrize("p", (2, 4, 5))
def test_m2l_sums_round_no_worse_than_the_cascades(p):
    """The same over whole far lists (long ones, flat and by target) on the GPU: the
    local potentials and gradients of the direct engine and of the matrix-core one,
    which is the cascade, against float64 locals of the same multipoles."""
    import torch

    from jaccpot_amd import FastMultipoleMethod
    from jaccpot_amd.flatlist import build_flat_list, pair_targets
    from oracle import ics

    x, m = ics.plummer(20000, 8)
    fmm = FastMultipoleMethod(precision="fp32", theta=0.5)
    st = fmm.prepare_state(torch.as_tensor(x).cuda(), torch.as_tensor(m).cuda(), leaf_size=16, max_order=p)
    C, topo, s = (p + 1) ** 2, st.topology, nat.current_stream()
    wide = [torch.zeros((topo.num_nodes, nat.coeff_stride(p, torch.float64)), dtype=torch.float64, device="cuda")
            for _ in range(2)]
    wide[0][:, :C] = st.multipoles[:, :C].double()
    c64 = st.centers4.double()
    nat.call("jfm_m2l", s, nat.JFM_F64, p, st.m2l_targets.data_ptr(), topo.num_m2l_targets, st.far_off.data_ptr(),
             st.far_src.data_ptr(), wide[0].data_ptr(), c64.data_ptr(), wide[1].data_ptr())
    ref = wide[1][:, :C][st.m2l_targets.long()]
    flat = build_flat_list(pair_targets(st), st.far_src[:topo.num_far_pairs], p, st.dtype, "cuda")
    for name, lists in (("target", None), ("flat", flat)):
        st.extra["flat"] = lists
        err = {}
        for engine in ("valu", "mfma"):
            fmm.m2l_engine = engine
            st.locals.zero_()
            fmm._m2l(st, s, nat.JFM_F32)
            diff = st.locals[:, :C][st.m2l_targets.long()].double() - ref
            err[engine] = np.array([float(torch.sqrt((diff[:, a:b] ** 2).sum() / (ref[:, a:b] ** 2).sum()))
                                    for a, b in ((0, 1), (1, 4))])
        print(f"p {p} {name}: cascade {err['mfma']}, ratio {err['valu'] / err['mfma']}", flush=True)
        assert np.all(err["valu"] <= 1.15 * err["mfma"]), name
    nat.call("jfm_set_m2l_engine", nat.M2L_VALU)


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

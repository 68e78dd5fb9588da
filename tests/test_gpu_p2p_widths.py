"""GPU: the near field at leaf widths around every edge of its thread mapping,
softened and not, compensated and not, whole leaves and work items, against the
float64 direct sum.  With an opening angle of 1e-6 every pair is a near pair.
Tolerances: float64 1e-12 (sums of 700 terms of a few roundings each); float32
1e-5, the parity tolerance (a term carries about eight roundings of 6e-8, and
the terms of a sum cancel by at most a factor of ten on these inputs)."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import direct, ics

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

WIDTHS = (2, 3, 5, 7, 8, 12, 16, 24, 31, 33, 64, 65, 85, 86, 127, 128, 129, 200, 256)


@pytest.mark.parametrize("leaf", WIDTHS)
def test_near_field_at_every_width(leaf, require_gpu):
    from jaccpot_amd import FastMultipoleMethod, nearsplit

    n = 701  # a ragged last leaf at every width above 1
    x, m = ics.plummer(n, leaf)
    for eps in (0.0, 1e-2):
        ref_a, ref_p = direct.direct_sum(x, m, eps=eps, return_potential=True)
        for precision, tol in (("fp64", 1e-12), ("fp32", 1e-5)):
            for comp in (True, False):
                fmm = FastMultipoleMethod(precision=precision, theta=1e-6, softening=eps, compensated=comp)
                st = fmm.prepare_state(x, m, leaf_size=leaf, max_order=1)
                for items in (False, True):
                    if items:
                        st.extra["p2p_items"] = nearsplit.build_p2p_items(st.topology.near_off, leaf, st.dtype, "cuda",
                                                                          chunk_slots=max(leaf, 300))
                    a, p = fmm.evaluate_prepared_state(st, return_potential=True)
                    b = fmm.evaluate_prepared_state(st)
                    ea = np.linalg.norm(a - ref_a) / np.linalg.norm(ref_a)
                    ep = np.linalg.norm(p - ref_p) / np.linalg.norm(ref_p)
                    eb = np.linalg.norm(b - ref_a) / np.linalg.norm(ref_a)
                    print(f"leaf {leaf} eps {eps} {precision} comp {comp} items {items}: {ea:.1e} {ep:.1e}", flush=True)
                    assert max(ea, ep, eb) < tol


def test_near_field_of_single_particle_leaves(require_gpu):
    """Leaves of one particle have no extent, so the walk makes none of their pairs
    near: a near list of all other leaves by hand."""
    from jaccpot_amd import FastMultipoleMethod
    from jaccpot_amd import _native as nat

    n = 300
    x, m = ics.plummer(n, 1)
    for eps in (0.0, 1e-2):
        ref = direct.direct_sum(x, m, eps=eps)
        for precision, tol in (("fp64", 1e-12), ("fp32", 1e-5)):
            fmm = FastMultipoleMethod(precision=precision, theta=0.6, softening=eps)
            st = fmm.prepare_state(x, m, leaf_size=1, max_order=1)
            others = np.arange(n)[None, :].repeat(n, 0)[~np.eye(n, dtype=bool)]
            st.near_off = torch.arange(0, n * n, n - 1, dtype=torch.int32, device="cuda")[: n + 1]
            st.near_src = torch.as_tensor(others.astype(np.int32), device="cuda")
            st.extra["p2p_items"] = None
            acc = torch.empty((n, 3), dtype=st.dtype, device="cuda")
            fmm._p2p_device(st, acc, None, nat.EVAL_COMPENSATED, accumulate=False)
            err = np.linalg.norm(acc.double().cpu().numpy() - ref) / np.linalg.norm(ref)
            print(f"eps {eps} {precision}: {err:.1e}", flush=True)
            assert st.near_off.numel() == n + 1 and err < tol

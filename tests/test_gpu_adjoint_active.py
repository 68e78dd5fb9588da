"""GPU: the adjoint near field with the flags of leaves that hold cotangents
against the same call without flags (every pair evaluated): the skipped pairs
contribute exact zeros, so only the order of the sums differs (float64 1e-12,
float32 1e-5 of the largest entry)."""

from __future__ import annotations

import pytest

from oracle import ics

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("share", (0.0, 0.002, 0.05, 1.0))
@pytest.mark.parametrize("leaf,precision,eps", ((5, "fp64", 0.0), (8, "fp64", 1e-2), (16, "fp32", 1e-2),
                                                (33, "fp32", 0.0), (100, "fp64", 1e-2)))
def test_flags_skip_only_zeros(leaf, precision, eps, share, require_gpu):
    from jaccpot_amd import FastMultipoleMethod, nearsplit
    from jaccpot_amd import _native as nat
    from jaccpot_amd.autodiff import active_leaves

    n = 4003
    x, m = ics.plummer(n, leaf)
    fmm = FastMultipoleMethod(precision=precision, theta=0.6, softening=eps)
    st = fmm.prepare_state(x, m, leaf_size=leaf, max_order=2)
    topo, s, code = st.topology, nat.current_stream(), nat.dtype_code(st.dtype)
    g = torch.Generator(device="cuda").manual_seed(leaf)
    cot = torch.randn((n, 4), generator=g, device="cuda", dtype=st.dtype)
    cot[torch.rand(n, generator=g, device="cuda") >= share] = 0
    flags = active_leaves(topo, code, s, cot)
    want = torch.zeros(topo.num_leaves * leaf, dtype=torch.bool, device="cuda")
    want[:n] = (cot != 0).any(1)
    assert torch.equal(flags.bool(), want.view(-1, leaf).any(1))
    rung = torch.randint(0, 3, (n,), generator=g, device="cuda", dtype=torch.int32)
    lw = torch.rand(3, generator=g, device="cuda", dtype=st.dtype)
    items = nearsplit.build_p2p_items(topo.near_off, leaf, st.dtype, "cuda", chunk_slots=4 * leaf)
    head = (s, code, st.pos4.data_ptr(), cot.data_ptr(), n, topo.num_leaves, leaf)
    lists = (st.near_off.data_ptr(), st.near_src.data_ptr())
    cut = (items.num_items, items.leaf.data_ptr(), items.s0.data_ptr(), items.s1.data_ptr(), items.part.data_ptr(),
           items.num_part, items.partials.data_ptr())
    level = (rung.data_ptr(), lw.data_ptr(), 3)
    for name, pre, post in (("jfm_p2p_adjoint", (), ()), ("jfm_p2p_adjoint_items", cut, ()),
                            ("jfm_p2p_adjoint_weighted", (), level), ("jfm_p2p_adjoint_weighted_items", cut, level)):
        out = []
        for active in (None, flags.data_ptr()):
            grad = torch.full((n, 4), float("nan"), dtype=st.dtype, device="cuda")
            nat.call(name, *head, *pre, *lists, active, *post, eps ** 2, 1.0, grad.data_ptr())
            if pre:
                nat.call("jfm_p2p_adjoint_reduce", s, code, cot.data_ptr(), n, leaf, items.num_split,
                         items.split_leaf.data_ptr(), items.split_p0.data_ptr(), items.split_p1.data_ptr(),
                         items.partials.data_ptr(), eps ** 2, 1.0, grad.data_ptr())
            out.append(grad)
        off = float((out[0] - out[1]).abs().max())
        top = float(out[0].abs().max())
        print(f"{name} leaf {leaf} {precision} share {share}: off {off:.1e} of {top:.1e}", flush=True)
        assert bool(torch.isfinite(out[1]).all())
        assert off <= (1e-12 if precision == "fp64" else 1e-5) * top

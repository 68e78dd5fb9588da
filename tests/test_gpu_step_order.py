"""GPU: a step on one stream (few near pairs) and with the P2P forked give the
same bits, and compute_accelerations, which steps on a new state, gives those of
refresh + evaluation."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import ics

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("precision,leaf,mixed", (("fp32", 16, False), ("fp32", 7, True), ("fp64", 8, False)))
def test_forked_step_matches_one_stream(precision, leaf, mixed, require_gpu):
    from jaccpot_amd import FastMultipoleMethod

    x, m = ics.plummer(3001, 2)
    fmm = FastMultipoleMethod(precision=precision, theta=0.6, softening=1e-2, mixed_precision=mixed)
    dtype = torch.float64 if precision == "fp64" else torch.float32
    xd, md = (torch.as_tensor(v, device="cuda").to(dtype) for v in (x, m))
    st = fmm.prepare_state(xd, md, leaf_size=leaf, max_order=4)
    rows = []
    for pairs in (0, 1 << 62):  # always forked, never forked
        fmm._fork_pairs = pairs
        acc = torch.empty((3001, 3), dtype=st.dtype, device="cuda")
        pot = torch.empty(3001, dtype=st.dtype, device="cuda")
        fmm.step_device(st, xd, md, acc, pot)
        rows.append((acc, pot))
    assert ("far_rows" in st.extra) and torch.equal(rows[0][0], rows[1][0]) and torch.equal(rows[0][1], rows[1][1])
    for pairs in (0, 1 << 62):
        fmm._fork_pairs = pairs
        a, p = fmm.compute_accelerations(xd, md, leaf_size=leaf, max_order=4, return_potential=True)
        new = fmm._last_state
        assert torch.equal(a, rows[0][0]) and torch.equal(p, rows[0][1])
        assert torch.equal(new.locals, st.locals) and torch.equal(new.multipoles, st.multipoles)
    some = fmm.compute_accelerations(xd, md, leaf_size=leaf, max_order=4, target_indices=[5, 0, 3000])
    assert np.array_equal(some.cpu().numpy(), rows[0][0][[5, 0, 3000]].cpu().numpy())


@pytest.mark.parametrize("precision,split", (("fp32", False), ("fp32", True), ("fp64", False)))
def test_every_path_adds_in_one_order(precision, split, require_gpu):
    """A gravitational constant that is no power of two: near and far field added in
    another order round differently.  New call, reused state, prepare + evaluate and
    step, with near lists cut into work items or not."""
    from jaccpot_amd import FastMultipoleMethod

    x, m = ics.plummer(20003, 7)
    fmm = FastMultipoleMethod(precision=precision, theta=0.6, softening=1e-2, G=4.3e-3, split_near=split)
    dtype = torch.float64 if precision == "fp64" else torch.float32
    xd, md = (torch.as_tensor(v, device="cuda").to(dtype) for v in (x, m))
    kw = {"leaf_size": 16, "max_order": 4, "return_potential": True}
    new = fmm.compute_accelerations(xd, md, **kw)
    again = fmm.compute_accelerations(xd, md, reuse_prepared_state=True, **kw)
    st = fmm.prepare_state(xd, md, leaf_size=16, max_order=4)
    assert (st.extra.get("p2p_items") is not None) == split
    prepared = fmm.evaluate_prepared_state(st, return_potential=True)
    step = torch.empty_like(new[0]), torch.empty_like(new[1])
    fmm.step_device(st, xd, md, *step)
    for name, got in (("reused", again), ("prepared", prepared), ("step", step)):
        assert torch.equal(got[0], new[0]) and torch.equal(got[1], new[1]), name

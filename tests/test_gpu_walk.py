"""GPU: the device walk where its first buffers are too small and where it takes
several launches of steps (the same lists as the host builder's, bit for bit),
and what is built on those lists on the device."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import ics

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("first,group,n,leaf", (
    (((1, 1), (1, 1), (1, 1)), 12, 20000, 8),  # every list and the frontier outgrow 1024 entries
    (((1, 1), (960, 320), (96, 32)), 12, 5000, 4),  # the far list only
    (((448, 128), (960, 320), (96, 32)), 1, 70000, 2),  # 35,000 leaves: 64-bit far keys; one step a group
))
def test_walk_grows_its_buffers(monkeypatch, require_gpu, first, group, n, leaf):
    from jaccpot_amd import dtopology
    from jaccpot_amd.topology import build_topology

    monkeypatch.setattr(dtopology, "WALK_FIRST", first)
    monkeypatch.setattr(dtopology, "WALK_GROUP", group)
    x, m = ics.plummer(n, 11)
    host = build_topology(x, m, leaf_size=leaf, theta=0.7)
    dev = dtopology.build_topology_device(torch.as_tensor(x, device="cuda"), torch.as_tensor(m, device="cuda"),
                                          leaf_size=leaf, theta=0.7)
    print(f"n {n} leaf {leaf}: {host.num_far_pairs} far, {host.num_near_entries} near", flush=True)
    for f in ("far_off", "far_src", "near_off", "near_src", "radius"):
        assert np.array_equal(getattr(dev, f), getattr(host, f)), f


@pytest.mark.parametrize("n,leaf,theta", ((20000, 8, 0.3), (50001, 16, 0.3), (100000, 16, 0.4)))
def test_walk_at_small_angles(monkeypatch, require_gpu, n, leaf, theta):
    """Opening angles whose frontier outgrows 96 items a leaf, the first buffer: every
    workgroup leaves the steps after it as a whole and the walk is repeated."""
    from jaccpot_amd import dtopology
    from jaccpot_amd.topology import build_topology

    monkeypatch.setattr(dtopology, "WALK_FIRST", ((448, 128), (960, 320), (96, 32)))
    x, m = ics.plummer(n, 13)
    host = build_topology(x, m, leaf_size=leaf, theta=theta)
    dev = dtopology.build_topology_device(torch.as_tensor(x, device="cuda"), torch.as_tensor(m, device="cuda"),
                                          leaf_size=leaf, theta=theta)
    print(f"n {n} leaf {leaf} theta {theta}: {host.num_far_pairs} far, {host.num_near_entries} near", flush=True)
    for f in ("far_off", "far_src", "near_off", "near_src"):
        assert np.array_equal(getattr(dev, f), getattr(host, f)), f


@pytest.mark.parametrize("n,leaf,theta", (
    (1100, 1, 0.7),  # frontiers of a few items a workgroup
    (160001, 3, 0.7),  # tiles of some rounds, the last one partly filled
    (700001, 8, 0.6),  # frontiers of more than 256 full tiles
))
def test_walk_tiles(require_gpu, n, leaf, theta):
    from jaccpot_amd import dtopology
    from jaccpot_amd.topology import build_topology

    x, m = ics.plummer(n, 12)
    host = build_topology(x, m, leaf_size=leaf, theta=theta)
    dev = dtopology.build_topology_device(torch.as_tensor(x, device="cuda"), torch.as_tensor(m, device="cuda"),
                                          leaf_size=leaf, theta=theta)
    print(f"n {n} leaf {leaf}: {host.num_far_pairs} far, {host.num_near_entries} near", flush=True)
    for f in ("far_off", "far_src", "near_off", "near_src"):
        assert np.array_equal(getattr(dev, f), getattr(host, f)), f


@pytest.mark.parametrize("n,leaf,chunk", ((3000, 8, 64), (3000, 7, 96), (3000, 8, 8192), (200, 16, 16), (5, 8, 8)))
def test_device_items_match_host(require_gpu, n, leaf, chunk):
    """Work items cut on the device: every list equal to the host's (None where no leaf is cut)."""
    from jaccpot_amd import nearsplit
    from jaccpot_amd.dtopology import build_topology_device

    x, m = ics.plummer(n, 4)
    topo = build_topology_device(torch.as_tensor(x, device="cuda"), torch.as_tensor(m, device="cuda"), leaf_size=leaf,
                                 theta=0.6)
    host = nearsplit.build_p2p_items(topo.near_off, leaf, torch.float32, "cuda", chunk_slots=chunk)
    dev = nearsplit.build_p2p_items_device(topo.extra["device"]["near_off"], topo.num_near_entries, leaf,
                                           torch.float32, chunk_slots=chunk)
    assert (host is None) == (dev is None)
    if host is None:
        return
    assert (host.num_items, host.num_part, host.num_split) == (dev.num_items, dev.num_part, dev.num_split)
    for f in ("leaf", "s0", "s1", "part", "split_leaf", "split_p0", "split_p1"):
        assert torch.equal(getattr(host, f), getattr(dev, f)), f
    assert host.partials.shape == dev.partials.shape


@pytest.mark.parametrize("split", (True, False))
def test_judged_rows_are_the_full_near_field(require_gpu, split):
    """The judge's near field: at its targets the same bits as the P2P over every leaf."""
    from jaccpot_amd import FastMultipoleMethod
    from jaccpot_amd import _native as nat
    from jaccpot_amd.judge import _near_rows

    x, m = ics.plummer(20011, 6)
    fmm = FastMultipoleMethod(precision="fp32", theta=0.6, split_near=split)
    st = fmm.prepare_state(x, m, leaf_size=16, max_order=2)
    assert (st.extra.get("p2p_items") is not None) == split
    tgt = torch.as_tensor(np.random.default_rng(1).choice(20011, 300, replace=False), device="cuda")
    full = torch.empty((20011, 3), dtype=st.dtype, device="cuda")
    fmm._p2p_device(st, full, None, nat.EVAL_COMPENSATED, accumulate=False)
    assert torch.equal(_near_rows(fmm, st, tgt)[tgt], full[tgt])


def test_topology_host_arrays_are_read_late(require_gpu):
    """Host arrays of a device topology appear on first read and stay."""
    from jaccpot_amd import FastMultipoleMethod

    x, m = ics.uniform(2000, 2)
    fmm = FastMultipoleMethod(precision="fp64", theta=0.6)
    st = fmm.prepare_state(torch.as_tensor(x, device="cuda"), torch.as_tensor(m, device="cuda"), leaf_size=8)
    a = st.topology.parent
    assert isinstance(a, np.ndarray) and st.topology.parent is a
    for bad in (np.nan, np.inf):
        y, w = x.copy(), m.copy()
        w[7] = bad
        with pytest.raises(ValueError, match="finite"):
            fmm.prepare_state(x, w, leaf_size=8)
        y[3, 1] = bad
        with pytest.raises(ValueError, match="finite"):
            fmm.prepare_state(y, m, leaf_size=8)

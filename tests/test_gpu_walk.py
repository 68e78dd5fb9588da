"""GPU: the device walk where its first buffers are too small and where it takes
several launches of steps: the same lists as the host builder's, bit for bit."""

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

"""GPU: whole passes over the levels (runs of narrow levels in one launch) against
one call per level.

M2M and L2L: level widths on both sides of what a run's workgroup takes at once, of
its limit and of what it cuts in four parts (orders 6 and up, where a part is computed
directly and a level's launch by rotations: equal to rounding only).  Tolerance: the
operators' of the host parity tests, 2e-5 (float32) and 1e-12 (float64) of the largest
coefficient of a degree, for each of the six levels that a row may have passed."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import harmonics as H
from oracle import ics

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# each in a run of its own kind: wide, run, wide, run to the end
WIDTHS = ([300, 33, 32, 1, 2, 65, 64, 129, 128, 257], [513, 600], [256, 31, 5, 127], [192, 48, 193, 49, 512, 47])


def _levels(rng, widths, leaves):
    """Internal nodes 0.. of levels of the given widths; children anywhere in the six
    levels before (or among the leaves), so that a row passes few levels."""
    count = sum(widths)
    off = np.concatenate([[0], np.cumsum(widths)]).astype(np.int32)
    kids = np.zeros((2, count), np.int32)
    depth = np.zeros(count + leaves, np.int32)
    for lev, w in enumerate(widths):
        a, b = off[lev], off[lev + 1]
        old = np.nonzero((np.arange(count + leaves) < a) & (depth < 6) | (np.arange(count + leaves) >= count))[0]
        kids[:, a:b] = rng.choice(old, size=(2, w))
        depth[a:b] = 1 + depth[kids[:, a:b]].max(0)
    return off, kids[0], kids[1], count


def _by_degree(a, p):
    return torch.stack([a[:, n * n:(n + 1) ** 2].abs().amax(1) for n in range(p + 1)], 1)


@pytest.mark.parametrize("dtype", (torch.float32, torch.float64))
@pytest.mark.parametrize("p", (4, 5, 6, 8))
@pytest.mark.parametrize("widths", WIDTHS)
def test_translation_passes_match_levels(require_gpu, p, dtype, widths):
    from jaccpot_amd import _native as nat

    rng = np.random.default_rng(p)
    leaves = 50
    off, left, right, count = _levels(rng, widths, leaves)
    nodes, C, cs = count + leaves, (p + 1) ** 2, nat.coeff_stride(p, dtype)
    code, s = nat.dtype_code(dtype), nat.current_stream()
    tol = 6 * (2e-5 if dtype == torch.float32 else 1e-12)

    def dev(a, t):
        return torch.as_tensor(np.ascontiguousarray(a), device="cuda").to(t)

    centers = np.concatenate([rng.uniform(-1, 1, size=(nodes, 3)), rng.uniform(0.5, 1.5, size=(nodes, 1))], 1)
    mult = np.zeros((nodes, cs))
    local = np.zeros((nodes, cs))
    for k in range(count, nodes):
        mult[k, :C] = H.p2m(rng.uniform(-0.3, 0.3, size=(4, 3)), rng.uniform(0.5, 1.5, 4), p)
    for k in range(nodes):
        local[k, :C] = H.m2l(mult[count + k % leaves, :C], np.array([2.0, -1.5, 1.0]) + rng.uniform(-0.5, 0.5, 3), p)
    order = dev(np.arange(count), torch.int32)
    lc, rc, par = dev(left, torch.int32), dev(right, torch.int32), dev(np.append(left, np.zeros(leaves)), torch.int32)
    rng2 = dev(np.zeros((nodes, 2)), torch.int32)
    rows = []
    for whole in (True, False):
        m, c, loc = dev(mult, dtype), dev(centers, dtype), dev(local, dtype)
        # upward; then downward over the same levels (a node's parent: its left child)
        head = (s, code, p, order.data_ptr())
        if whole:
            nat.call("jfm_m2m_pass", *head, nat.ptr(off), len(widths), lc.data_ptr(), rc.data_ptr(), rng2.data_ptr(),
                     m.data_ptr(), c.data_ptr())
            nat.call("jfm_l2l_pass", *head, nat.ptr(off), len(widths), par.data_ptr(), c.data_ptr(), loc.data_ptr())
        else:
            for a, w in zip(off, widths):
                nat.call("jfm_m2m_level", s, code, p, order.data_ptr() + 4 * int(a), w, lc.data_ptr(), rc.data_ptr(),
                         rng2.data_ptr(), m.data_ptr(), c.data_ptr())
            for a, w in zip(off, widths):
                nat.call("jfm_l2l_level", s, code, p, order.data_ptr() + 4 * int(a), w, par.data_ptr(), c.data_ptr(),
                         loc.data_ptr())
        rows.append((m, c, loc))
    (m1, c1, l1), (m2, c2, l2) = rows
    assert torch.equal(c1, c2)
    assert torch.equal(m1[:, C:], m2[:, C:]) and torch.equal(l1[:, C:], l2[:, C:])
    for name, a, b in (("m2m", m1, m2), ("l2l", l1, l2)):
        err = float((_by_degree(a[:, :C] - b[:, :C], p) / _by_degree(b[:, :C], p).clamp_min(1e-300)).max())
        print(f"{name} p {p} {dtype} {widths}: {err:.1e}", flush=True)
        assert err <= tol, name


@pytest.mark.parametrize("n,leaf", ((3, 2), (900, 4), (9000, 4), (70000, 8)))
def test_geometry_and_rung_passes_match_levels(require_gpu, n, leaf):
    """Centres (with massless nodes) and rungs of a real tree: equal bits."""
    from jaccpot_amd import _native as nat
    from jaccpot_amd.topology import build_topology

    x, m = ics.plummer(n, 5)
    m = np.where(np.arange(n) % 5 < 3, 0.0, m)
    t = build_topology(x, m, leaf_size=leaf, theta=0.7)
    s, I, L = nat.current_stream(), t.num_internal, t.num_leaves
    xd, md = torch.as_tensor(x, device="cuda"), torch.as_tensor(m, device="cuda")
    perm, left, right, span, order = (torch.as_tensor(np.ascontiguousarray(a, np.int32), device="cuda")
                                      for a in (t.perm, t.left, t.right, t.node_range, t.m2m_nodes))
    rung = torch.as_tensor(np.random.default_rng(2).integers(-1, 9, t.num_nodes).astype(np.int32), device="cuda")
    off = nat.host_i32(t.m2m_off)
    rows = []
    for whole in (True, False):
        mass = torch.zeros(t.num_nodes, dtype=torch.float64, device="cuda")
        center = torch.zeros((t.num_nodes, 3), dtype=torch.float64, device="cuda")
        r = rung.clone()
        nat.call("jfm_tree_leaf_geometry", s, L, I, xd.data_ptr(), md.data_ptr(), perm.data_ptr(), span.data_ptr(),
                 mass.data_ptr(), center.data_ptr())
        geo = (xd.data_ptr(), md.data_ptr(), perm.data_ptr(), left.data_ptr(), right.data_ptr(), span.data_ptr(),
               mass.data_ptr(), center.data_ptr())
        kin = (left.data_ptr(), right.data_ptr(), r.data_ptr())
        if whole:
            nat.call("jfm_tree_geometry_pass", s, nat.ptr(off), len(off) - 1, order.data_ptr(), *geo)
            nat.call("jfm_mutual_rungs_pass", s, order.data_ptr(), nat.ptr(off), len(off) - 1, *kin)
        else:
            for a, b in zip(off[:-1], off[1:]):
                nat.call("jfm_tree_level_geometry", s, int(b - a), order.data_ptr() + 4 * int(a), *geo)
                nat.call("jfm_mutual_rungs_level", s, order.data_ptr() + 4 * int(a), int(b - a), *kin)
        rows.append((mass, center, r))
    for a, b in zip(*rows):
        assert torch.equal(a, b)

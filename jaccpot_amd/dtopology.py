"""Topology built on the GPU: the host builder's spec, bit-identical output.

Same role as ``topology.build_topology`` (yggdrax's tree and interaction-list
builders for the reference, jaccpot/runtime/fmm_state.py:630-800,
runtime/_interaction_cache.py:523,564), run as libjfm device kernels
(``csrc/treebuild.hip``): bounds, Morton codes, stable radix sort, radix tree,
levels, centres of mass and radii, breadth-first dual-tree walk, CSR lists.
Returns a ``Topology`` (its host arrays are copied from the device when first
read, so every host consumer works unchanged) with the device arrays in
``extra["device"]`` so that ``prepare_state`` does not upload them again.
"""

from __future__ import annotations

import ctypes
import time

import numpy as np
import torch

from . import _native as nat
from .topology import Topology

MAX_TREE_HEIGHT = 128  # depths of a radix tree over 63-bit codes with index tie-breaks stay below it


class _Lazy:
    """A device array whose host copy is made on first access (from whatever
    stream that happens on, so after a device-wide wait)."""

    __slots__ = ("t",)

    def __init__(self, t: torch.Tensor):
        self.t = t

    def host(self) -> np.ndarray:
        torch.cuda.synchronize(self.t.device)
        return self.t.cpu().numpy()


class LazyExtra(dict):
    """A dict whose ``_Lazy`` values become host arrays when first read by key."""

    def __getitem__(self, key):
        v = dict.__getitem__(self, key)
        if type(v) is _Lazy:
            v = v.host()
            self[key] = v
        return v

    def get(self, key, default=None):
        return self[key] if key in self else default


class DeviceTopology(Topology):
    """``Topology`` whose host arrays are copied from the device only when first
    read; the device build and the evaluation never need them."""

    def __getattribute__(self, name):
        v = object.__getattribute__(self, name)
        if type(v) is _Lazy:
            v = v.host()
            object.__setattr__(self, name, v)
        return v

    @property
    def num_m2l_targets(self) -> int:
        return int(self.extra["num_m2l_targets"])

    @property
    def num_far_pairs(self) -> int:
        return int(self.extra["num_far_pairs"])

    @property
    def num_near_entries(self) -> int:
        return int(self.extra["num_near_entries"])


def _sort_u64(keys: torch.Tensor, end_bit: int, vals: torch.Tensor | None = None):
    n = int(keys.numel())
    out_k = torch.empty_like(keys)
    out_v = torch.empty_like(vals) if vals is not None else None
    if n == 0:
        return out_k, out_v
    nb = ctypes.c_int64(0)
    nat.call("jfm_sort_scratch_bytes", n, 1 if vals is not None else 0, ctypes.byref(nb))
    scratch = torch.empty(max(int(nb.value), 1), dtype=torch.uint8, device=keys.device)
    nat.call("jfm_sort_u64", nat.current_stream(), n, int(end_bit), keys.data_ptr(), out_k.data_ptr(),
             nat.ptr(vals), nat.ptr(out_v), scratch.data_ptr(), int(nb.value))
    return out_k, out_v


def _csr(sorted_keys: torch.Tensor, rows: int):
    dev = sorted_keys.device
    off = torch.empty(rows + 1, dtype=torch.int32, device=dev)
    col = torch.empty(max(int(sorted_keys.numel()), 1), dtype=torch.int32, device=dev)
    nat.call("jfm_keys_to_csr", nat.current_stream(), nat.ptr(sorted_keys) if sorted_keys.numel() else None,
             int(sorted_keys.numel()), int(rows), off.data_ptr(), col.data_ptr())
    return off, col[: int(sorted_keys.numel())]


def _key_bits(max_key: int) -> int:
    return max(1, int(nat.call("jfm_key_bits", ctypes.c_uint64(int(max_key)))))


# Steps of the walk launched before the host looks at its state: groups of
# WALK_GROUP whole-GPU steps, each behind a workgroup that runs small frontiers
# by itself.  A step whose frontier is empty costs about 2.5 us, a look 20 to 30.
WALK_GROUP = 12
# First buffer sizes per leaf (far entries, near entries, frontier items): the
# longest lists seen on clustered inputs at opening angles from 0.55 are 410, 885
# and 83.  Where they would pass WALK_LIMIT_BYTES, that or the second figures (4.9
# GB in all at 524,288 leaves).  Smaller angles find them too small and walk two or
# three times; a whole build of Plummer bodies takes 0.97 / 1.05 / 1.8 / 1.9 ms at
# angles 0.6 / 0.5 / 0.4 / 0.3 (65,536 bodies, leaf 16) and 2.1 / 4.1 / 6.7 / 11.7
# (524,288), where lists grown between the steps took 4.3 to 4.8 and 6.8 to 19.5.
WALK_FIRST = ((448, 128), (960, 320), (96, 32))
WALK_LIMIT_BYTES = 1 << 31


def _walk(I: int, nodes: int, L: int, node4: torch.Tensor, left: torch.Tensor, right: torch.Tensor, theta: float):
    """Far and near packed keys of the dual-tree walk: ((keys, n, shift, wide), ...).
    A buffer that proves too small is allocated again and the walk repeated."""
    dev = node4.device
    s = nat.current_stream()
    shifts = (_key_bits(max(nodes - 1, 1)), _key_bits(max(L - 1, 1)))
    wide = tuple(0 if 2 * b <= 32 else 1 for b in shifts)
    width = tuple(8 if w else 4 for w in wide)
    far_cap, near_cap, fcap = (max(1024, min(per * L, max(WALK_LIMIT_BYTES // b, least * L)))
                               for (per, least), b in zip(WALK_FIRST, width + (16,)))
    caps = [far_cap, near_cap]
    # more groups in the first call spare looks at deep trees and cost shallow ones empty
    # steps: a build with 1 / 2 / 4 groups takes 642 / 664 / 716 us at 256 leaves, 919 /
    # 881 / 872 at 1024, 1338 / 1309 / 1208 at 8192, 1641 / 1605 / 1532 at 16,384
    groups = 1 if L <= 1024 else 2 if L <= 8192 else 4
    while True:
        frontier = torch.empty((2, fcap, 2), dtype=torch.int32, device=dev)
        lists = [torch.empty(c, dtype=torch.int64 if w else torch.int32, device=dev) for c, w in zip(caps, wide)]
        frontier[0, 0].zero_()
        state = None
        while True:
            # a further call goes on by single groups: what is left is mostly a few
            # steps (a 256k galaxy: 39 of 104 step launches fewer, of 4 us each)
            call_groups = groups if state is None else 1
            last = None if state is None else 48 + 2 * steps
            steps = call_groups * (1 + WALK_GROUP) + 1
            nxt = torch.zeros(int(nat.call("jfm_tree_walk_state_words", steps)), dtype=torch.int64, device=dev)
            if state is None:
                nxt[48].fill_(1)
            else:  # go on from the counters and the frontier of the last call
                nxt[:48].copy_(state[:48])
                nxt[48:50].copy_(state[last:])
            state = nxt
            nat.call("jfm_tree_walk", s, I, node4.data_ptr(), left.data_ptr(), right.data_ptr(), float(theta),
                     frontier[0].data_ptr(), frontier[1].data_ptr(), fcap, lists[0].data_ptr(), caps[0], shifts[0],
                     wide[0], lists[1].data_ptr(), caps[1], shifts[1], wide[1], state.data_ptr(), 0, call_groups,
                     WALK_GROUP)
            h = state.cpu().numpy()
            full = int(h[32])
            if int(h[48 + 2 * steps]) == 0 or full & 1:
                break
        counts = (int(h[0]), int(h[16]))
        if not full:
            return tuple((k[:n], n, b, w) for k, n, b, w in zip(lists, counts, shifts, wide))
        # larger buffers for another walk: the lists were counted to the end unless the frontier was full
        if full & 1:
            fcap = max(2 * fcap, int(1.25 * int(h[33])))
        for i, n in enumerate(counts):
            if n > caps[i]:
                caps[i] = int(1.25 * n) if full & 1 else n
        del frontier, lists


def _packed_csr(keys: torch.Tensor, n: int, shift: int, wide: int, rows: int):
    dev = keys.device
    off = torch.empty(rows + 1, dtype=torch.int32, device=dev)
    col = torch.empty(max(n, 1), dtype=torch.int32, device=dev)
    nb = ctypes.c_int64(0)
    nat.call("jfm_sort_packed_scratch_bytes", n, wide, ctypes.byref(nb))
    scratch = torch.empty(max(int(nb.value), 1), dtype=torch.uint8, device=dev)
    out = torch.empty_like(keys)
    nat.call("jfm_packed_to_csr", nat.current_stream(), n, wide, shift, nat.ptr(keys), nat.ptr(out),
             scratch.data_ptr(), int(scratch.numel()), rows, off.data_ptr(), col.data_ptr())
    return off, col[:n]


def build_topology_device(x: torch.Tensor, m: torch.Tensor, *, leaf_size: int, theta: float,
                          bounds=None, check_masses: bool = False) -> Topology:
    """Build the topology for input-order float64 device tensors x [N,3], m [N].
    ``check_masses``: masses that are not finite raise as positions do.  The last
    kernels (the near list's sort) may still run when this returns."""
    if x.dtype != torch.float64 or m.dtype != torch.float64 or x.device.type != "cuda":
        raise ValueError("build_topology_device needs float64 CUDA tensors")
    if x.ndim != 2 or x.shape[1] != 3 or m.shape != (x.shape[0],):
        raise ValueError("positions must be [N,3] and masses [N]")
    n = int(x.shape[0])
    if n < 1 or n > (1 << 30):
        raise ValueError("need 1 <= N <= 2^30 particles")
    if leaf_size < 1 or leaf_size > 256:
        raise ValueError("leaf_size must be in [1, 256]")
    if not (theta > 0.0) or not np.isfinite(theta):
        raise ValueError("theta must be > 0")
    x = x.contiguous()
    m = m.contiguous()
    dev = x.device
    s = nat.current_stream()
    t0 = time.perf_counter()
    L = (n + leaf_size - 1) // leaf_size
    I = L - 1
    nodes = 2 * L - 1

    # ---- bounds, Morton codes, sort ------------------------------------------------------
    flags = torch.zeros(1, dtype=torch.int32, device=dev)
    bscratch = torch.empty(int(nat.call("jfm_tree_bounds_scratch_doubles")), dtype=torch.float64, device=dev)
    if bounds is not None:
        lo, hi = bounds
        b6 = torch.as_tensor(np.concatenate([np.asarray(lo, np.float64), np.asarray(hi, np.float64)]), device=dev)
    else:
        b6 = torch.empty(6, dtype=torch.float64, device=dev)
    nat.call("jfm_tree_bounds", s, x.data_ptr(), n, 1 if bounds is not None else 0, bscratch.data_ptr(),
             b6.data_ptr(), flags.data_ptr())
    if check_masses:
        flags |= (~torch.isfinite(m)).any().to(torch.int32) * 4
    codes = torch.empty(n, dtype=torch.int64, device=dev)
    index = torch.empty(n, dtype=torch.int32, device=dev)
    nat.call("jfm_tree_morton", s, x.data_ptr(), n, b6.data_ptr(), codes.data_ptr(), index.data_ptr())
    sorted_codes, perm = _sort_u64(codes, 63, index)
    del codes, index
    bounds_used = b6

    # ---- radix tree, levels ---------------------------------------------------------------
    parent = torch.empty(nodes, dtype=torch.int32, device=dev)
    left = torch.empty(max(I, 1), dtype=torch.int32, device=dev)
    right = torch.empty(max(I, 1), dtype=torch.int32, device=dev)
    node_range = torch.empty((nodes, 2), dtype=torch.int32, device=dev)
    nat.call("jfm_tree_radix", s, n, int(leaf_size), sorted_codes.data_ptr(), parent.data_ptr(), left.data_ptr(),
             right.data_ptr(), node_range.data_ptr())
    depth = torch.empty(nodes, dtype=torch.int32, device=dev)
    maxd = torch.zeros(1, dtype=torch.int32, device=dev)
    m2m_keys = torch.empty(max(I, 1), dtype=torch.int64, device=dev)
    l2l_keys = torch.empty(max(nodes - 1, 1), dtype=torch.int64, device=dev)
    nat.call("jfm_tree_levels", s, nodes, I, parent.data_ptr(), depth.data_ptr(), maxd.data_ptr(), flags.data_ptr(),
             m2m_keys.data_ptr(), l2l_keys.data_ptr())
    # level tables over every depth a radix tree can have (unused rows are
    # empty), read back together with the flags
    if I > 0:
        sk, _ = _sort_u64(m2m_keys[:I], 32 + _key_bits(MAX_TREE_HEIGHT))
        m2m_off_d, m2m_nodes = _csr(sk, MAX_TREE_HEIGHT + 1)
        sk, _ = _sort_u64(l2l_keys[: nodes - 1], 32 + _key_bits(MAX_TREE_HEIGHT))
        l2l_off_d, l2l_nodes = _csr(sk, MAX_TREE_HEIGHT)
        shallow = torch.zeros(14, dtype=torch.int32, device=dev)  # nodes of depths 1 to 3, at most
        shallow[: min(14, nodes - 1)] = l2l_nodes[:14]
        hdr = torch.cat([flags, maxd, m2m_off_d, l2l_off_d, shallow]).cpu().numpy()
    else:
        m2m_nodes = torch.empty(0, dtype=torch.int32, device=dev)
        l2l_nodes = torch.empty(0, dtype=torch.int32, device=dev)
        hdr = torch.cat([flags, maxd]).cpu().numpy()
    if hdr[0] & 5:
        raise ValueError("positions and masses must be finite" if check_masses else "positions must be finite")
    if hdr[0] & 2:
        raise RuntimeError("device topology build: parent chain exceeds the maximum tree height")
    D = int(hdr[1])
    if I > 0:
        m2m_off = nat.host_i32(hdr[2:2 + D + 2])
        l2l_off = nat.host_i32(hdr[2 + MAX_TREE_HEIGHT + 2:][:D + 1])
    else:
        m2m_off = np.zeros(1, np.int32)
        l2l_off = np.zeros(1, np.int32)
    del m2m_keys, l2l_keys

    # ---- geometry ------------------------------------------------------------------------
    mass = torch.empty(nodes, dtype=torch.float64, device=dev)
    center = torch.empty((nodes, 3), dtype=torch.float64, device=dev)
    radius = torch.empty(nodes, dtype=torch.float64, device=dev)
    nat.call("jfm_tree_leaf_geometry", s, L, I, x.data_ptr(), m.data_ptr(), perm.data_ptr(), node_range.data_ptr(),
             mass.data_ptr(), center.data_ptr())
    nat.call("jfm_tree_geometry_pass", s, nat.ptr(m2m_off), len(m2m_off) - 1, m2m_nodes.data_ptr(), x.data_ptr(),
             m.data_ptr(), perm.data_ptr(), left.data_ptr(), right.data_ptr(), node_range.data_ptr(), mass.data_ptr(),
             center.data_ptr())
    xs = torch.empty((n, 3), dtype=torch.float64, device=dev)
    cap = int(nat.call("jfm_tree_radius_work", nodes, n, D))
    work = torch.empty(2 + 2 * cap, dtype=torch.int32, device=dev)
    nat.call("jfm_tree_radius", s, nodes, n, x.data_ptr(), perm.data_ptr(), node_range.data_ptr(), center.data_ptr(),
             xs.data_ptr(), work.data_ptr(), cap, radius.data_ptr())
    del xs, work

    # ---- dual-tree walk, lists ------------------------------------------------------------
    node4 = torch.empty((nodes, 4), dtype=torch.float64, device=dev)
    nat.call("jfm_tree_pack_nodes", s, nodes, center.data_ptr(), radius.data_ptr(), node4.data_ptr())
    (fk, n_far, fb, fw), (nk, n_near, nb, nw) = _walk(I, nodes, L, node4, left, right, theta)
    del node4
    far_off, far_src = _packed_csr(fk, n_far, fb, fw, nodes)
    del fk
    m2l_targets = torch.nonzero(far_off[1:] > far_off[:-1]).reshape(-1).to(torch.int32)
    near_off, near_src = _packed_csr(nk, n_near, nb, nw, L)
    del nk
    device = dict(perm=perm, parent=parent, left=left, right=right, node_range=node_range, depth=depth,
                  center=center, radius=radius, mass=mass, far_off=far_off, far_src=far_src, near_off=near_off,
                  near_src=near_src, m2m_nodes=m2m_nodes, l2l_nodes=l2l_nodes, m2l_targets=m2l_targets,
                  sorted_codes=sorted_codes, bounds=bounds_used)
    topo = DeviceTopology(
        num_particles=n, leaf_size=int(leaf_size), num_leaves=L, num_internal=I, num_nodes=nodes, max_depth=D,
        theta=float(theta), perm=_Lazy(perm), parent=_Lazy(parent), left=_Lazy(left[:I]), right=_Lazy(right[:I]),
        node_range=_Lazy(node_range), depth=_Lazy(depth), center=_Lazy(center), radius=_Lazy(radius),
        mass=_Lazy(mass), far_off=_Lazy(far_off), far_src=_Lazy(far_src), near_off=_Lazy(near_off),
        near_src=_Lazy(near_src), m2m_nodes=_Lazy(m2m_nodes), m2m_off=m2m_off, l2l_nodes=_Lazy(l2l_nodes),
        l2l_off=l2l_off, m2l_targets=_Lazy(m2l_targets), build_seconds=0.0,
    )
    topo.extra["num_far_pairs"] = n_far
    topo.extra["num_near_entries"] = n_near
    topo.extra["num_m2l_targets"] = int(m2l_targets.numel())
    if I > 0:
        topo.extra["shallow_nodes"] = nat.host_i32(hdr[2 + 2 * MAX_TREE_HEIGHT + 3:])
    topo.build_seconds = time.perf_counter() - t0
    topo.extra["device"] = device
    topo.extra["device_build_seconds"] = topo.build_seconds
    return topo


def sorted_morton(x: torch.Tensor, bounds=None):
    """(sorted Morton codes, perm) of float64 device positions x [N,3]: the first
    steps of ``build_topology_device`` (the topology reuse check)."""
    n = int(x.shape[0])
    dev = x.device
    s = nat.current_stream()
    x = x.contiguous()
    flags = torch.zeros(1, dtype=torch.int32, device=dev)
    bscratch = torch.empty(int(nat.call("jfm_tree_bounds_scratch_doubles")), dtype=torch.float64, device=dev)
    if bounds is not None:
        lo, hi = bounds
        b6 = torch.as_tensor(np.concatenate([np.asarray(lo, np.float64), np.asarray(hi, np.float64)]), device=dev)
    else:
        b6 = torch.empty(6, dtype=torch.float64, device=dev)
    nat.call("jfm_tree_bounds", s, x.data_ptr(), n, 1 if bounds is not None else 0, bscratch.data_ptr(),
             b6.data_ptr(), flags.data_ptr())
    codes = torch.empty(n, dtype=torch.int64, device=dev)
    index = torch.empty(n, dtype=torch.int32, device=dev)
    nat.call("jfm_tree_morton", s, x.data_ptr(), n, b6.data_ptr(), codes.data_ptr(), index.data_ptr())
    sc, perm = _sort_u64(codes, 63, index)
    if int(flags.item()) & 1:
        raise ValueError("positions must be finite")
    return sc, perm

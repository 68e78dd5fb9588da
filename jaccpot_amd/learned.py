"""Learned per-pair M2L order (p_gears) on the GPU.

The reference tags each accepted far pair with a gear -- the smallest order
that passes its error model -- inside the traversal
(runtime/_adaptive_policy.py:2216-2385) and hands ``far_pairs_by_gear`` to the
downward sweep (runtime/fmm_prepare.py:2412-2482), whose real-basis M2L then
ignores it (runtime/kernels/_l2l.py:491-493).  Here the tag comes from a small
MLP that predicts each pair's truncation error at every gear, and the M2L
really runs each pair at its gear (``jfm_m2l_gear``).

Training data are generated by the FMM itself: pair features from the order-p
multipoles and labels from order-8 translations (``jfm_pair_labels``).  The
network's forward, backward and Adam kernels are libjfm's.
"""

from __future__ import annotations

from dataclasses import dataclass
from typing import Optional, Sequence

import numpy as np
import torch

from . import _native as nat
from .flatlist import build_flat_list, pair_targets, prefers_flat

NUM_FEATURES = 8
NUM_OUTPUTS = 3


def _dev():
    return torch.device("cuda", torch.cuda.current_device())


class OrderModel:
    """8 -> 64 -> 64 -> 3 MLP predicting log10 truncation error at gears (2, 4, 6)."""

    def __init__(self, gears: Sequence[int] = (2, 4, 6), seed: int = 0, device=None):
        if len(tuple(gears)) != 3:
            raise ValueError("exactly three gears are supported")
        self.gears = tuple(int(g) for g in gears)
        self.device = device or _dev()
        n = int(nat.load().jfm_mlp_num_params())
        self.num_params = n
        rng = np.random.default_rng(seed)
        theta = np.zeros(n, np.float32)
        o = 0
        for fan_in, fan_out in ((8, 64), (64, 64), (64, 3)):
            w = rng.normal(0.0, np.sqrt(2.0 / fan_in), size=(fan_out, fan_in)).astype(np.float32)
            theta[o : o + w.size] = w.ravel()
            o += w.size + fan_out  # bias stays zero
        self.master = torch.as_tensor(theta, device=self.device)
        self.m1 = torch.zeros_like(self.master)
        self.m2 = torch.zeros_like(self.master)
        self.wbf16 = torch.empty(n, dtype=torch.int16, device=self.device)
        self.step = 0
        self._set_stats(np.zeros(NUM_FEATURES), np.ones(NUM_FEATURES))
        self._refresh_bf16()

    def _refresh_bf16(self):
        nat.call("jfm_mlp_to_bf16", nat.current_stream(), self.master.data_ptr(), self.wbf16.data_ptr())

    def _set_stats(self, mean, std) -> None:
        """Feature normalisation (host float32, uploaded once)."""
        mean = np.asarray(mean, np.float32)
        std = np.asarray(std, np.float32)
        self.feature_mean = torch.as_tensor(mean, device=self.device)
        self.feature_std = torch.as_tensor(std, device=self.device)
        self.feature_inv_std = torch.as_tensor((1.0 / std).astype(np.float32), device=self.device)

    def normalise(self, X: torch.Tensor) -> torch.Tensor:
        return ((X - self.feature_mean) / self.feature_std).contiguous()

    def predict(self, X: torch.Tensor, normalised: bool = False, exact: bool = False) -> torch.Tensor:
        """[K, 3] predicted log10 errors; raw features are normalised inside the kernel.

        Inference runs on the matrix cores (bf16 MFMA, activations rounded to
        bf16 between layers); ``exact=True`` uses the VALU forward with float32
        activations (the one the training kernels differentiate)."""
        X = X.contiguous()
        K = int(X.shape[0])
        Y = torch.empty((K, NUM_OUTPUTS), dtype=torch.float32, device=self.device)
        if K:
            mean = None if normalised else self.feature_mean.data_ptr()
            inv = None if normalised else self.feature_inv_std.data_ptr()
            fn = "jfm_mlp_forward" if exact else "jfm_mlp_forward_mfma"
            nat.call(fn, nat.current_stream(), K, X.data_ptr(), mean, inv, self.wbf16.data_ptr(), Y.data_ptr())
        return Y

    def loss_and_grad(self, Xn: torch.Tensor, T: torch.Tensor, per_block: int = 256):
        K = int(Xn.shape[0])
        scratch = torch.empty(int(nat.load().jfm_mlp_backward_scratch_floats(K, per_block)), dtype=torch.float32,
                              device=self.device)
        out = torch.empty(self.num_params + 1, dtype=torch.float32, device=self.device)
        nat.call("jfm_mlp_backward", nat.current_stream(), K, per_block, Xn.data_ptr(), T.contiguous().data_ptr(),
                 self.wbf16.data_ptr(), scratch.data_ptr(), out.data_ptr())
        return out[self.num_params], out[: self.num_params]

    def adam(self, grad: torch.Tensor, lr: float = 1e-3, beta1: float = 0.9, beta2: float = 0.999, eps: float = 1e-8):
        self.step += 1
        nat.call("jfm_mlp_adam", nat.current_stream(), self.step, lr, beta1, beta2, eps, self.master.data_ptr(),
                 grad.data_ptr(), self.m1.data_ptr(), self.m2.data_ptr(), self.wbf16.data_ptr())

    def fit(self, X: torch.Tensor, T: torch.Tensor, *, steps: int = 400, batch: int = 32768, lr: float = 2e-3,
            seed: int = 0, log_every: int = 0):
        """Adam on minibatches of (features, log10-error labels); returns the loss history."""
        self._set_stats(X.mean(0).cpu().numpy(), X.std(0).clamp_min(1e-3).cpu().numpy())
        Xn = self.normalise(X)
        K = int(Xn.shape[0])
        g = torch.Generator(device="cpu").manual_seed(seed)
        hist = []
        for it in range(steps):
            idx = torch.randint(0, K, (min(batch, K),), generator=g).to(self.device)
            cur_lr = lr * (0.5 * (1 + np.cos(np.pi * it / steps)))
            loss, grad = self.loss_and_grad(Xn[idx].contiguous(), T[idx].contiguous())
            self.adam(grad, lr=cur_lr)
            if log_every and (it % log_every == 0 or it == steps - 1):
                hist.append((it, float(loss)))
        return hist

    def select_gears(self, X: torch.Tensor, tol_log10: float, state, budget: str = "node") -> torch.Tensor:
        """Per-pair gears for the far CSR of ``state`` (``X`` in CSR pair order).

        A pair takes the smallest gear whose predicted force-error proxy
        (relative error times m_s / d^2) is within ``10**tol_log10`` of the
        budget of its target: ``budget="node"``, the largest top-gear proxy
        among the target's own pairs; ``"leaf"``, the smallest, over the
        leaves under the target, of the largest top-gear proxy on the path
        from the root to that leaf (the dominant truncation term its
        particles receive from any level)."""
        if budget not in ("node", "leaf"):
            raise ValueError(f"budget must be 'node' or 'leaf', got {budget!r}")
        Y = self.predict(X)
        K = int(Y.shape[0])
        out = torch.empty(K, dtype=torch.int8, device=self.device)
        g3 = np.asarray(self.gears, np.int32)
        if not K:
            return out
        topo = state.topology
        s = nat.current_stream()
        if budget == "node":
            nat.call("jfm_select_gears", s, topo.num_nodes, state.far_off.data_ptr(), state.far_src.data_ptr(),
                     Y.data_ptr(), state.centers4.data_ptr(), float(tol_log10), nat.ptr(g3), out.data_ptr())
            return out
        b = torch.empty(topo.num_nodes, dtype=torch.float32, device=self.device)
        nat.call("jfm_gear_node_max", s, topo.num_nodes, state.far_off.data_ptr(), state.far_src.data_ptr(),
                 Y.data_ptr(), state.centers4.data_ptr(), nat.ptr(g3), b.data_ptr())
        off = topo.l2l_off  # children by depth, root side first
        for lev in range(len(off) - 1):
            a, e = int(off[lev]), int(off[lev + 1])
            if e > a:
                nat.call("jfm_level_path_max", s, state.l2l_nodes.data_ptr() + 4 * a, e - a,
                         state.parent.data_ptr(), b.data_ptr())
        off = topo.m2m_off  # internal nodes by depth, deepest first
        for lev in range(len(off) - 1):
            a, e = int(off[lev]), int(off[lev + 1])
            if e > a:
                nat.call("jfm_level_subtree_min", s, state.m2m_nodes.data_ptr() + 4 * a, e - a,
                         state.left.data_ptr(), state.right.data_ptr(), b.data_ptr())
        nat.call("jfm_select_gears_budget", s, topo.num_nodes, state.far_off.data_ptr(), state.far_src.data_ptr(),
                 Y.data_ptr(), state.centers4.data_ptr(), float(tol_log10), nat.ptr(g3), b.data_ptr(),
                 out.data_ptr())
        return out

    def state_dict(self) -> dict:
        return {"master": self.master.cpu().numpy(), "gears": np.asarray(self.gears),
                "feature_mean": self.feature_mean.cpu().numpy(), "feature_std": self.feature_std.cpu().numpy()}

    def load_state_dict(self, d: dict) -> None:
        self.master = torch.as_tensor(np.asarray(d["master"], np.float32), device=self.device)
        self.gears = tuple(int(g) for g in d["gears"])
        self._set_stats(d["feature_mean"], d["feature_std"])
        self._refresh_bf16()


def pair_arrays(state):
    """Device (tgt_of, far_src) of the state's far list and float32 node radii."""
    topo = state.topology
    K = topo.num_far_pairs
    dev = state.device
    rad = topo.extra.get("device", {}).get("radius")
    rad = rad.float() if rad is not None else torch.as_tensor(topo.radius.astype(np.float32), device=dev)
    return pair_targets(state), state.far_src[:K], rad


def pair_features(state) -> torch.Tensor:
    """[K, 8] float32 features of every far pair of a float32 prepared state."""
    if state.dtype != torch.float32:
        raise ValueError("pair features are computed from float32 expansions")
    topo = state.topology
    K = topo.num_far_pairs
    tgt, src, rad = pair_arrays(state)
    X = torch.empty((K, NUM_FEATURES), dtype=torch.float32, device=state.device)
    mass = topo.extra.get("device", {}).get("mass")
    total = float(topo.mass[0] if mass is None else mass[0])
    nat.call("jfm_pair_features", nat.current_stream(), state.order, K, tgt.data_ptr(), src.data_ptr(),
             state.multipoles.data_ptr(), state.centers4.data_ptr(), rad.data_ptr(), total, X.data_ptr())
    return X


def pair_labels(state, gears: Sequence[int] = (2, 4, 6)) -> torch.Tensor:
    """[K, 3] log10 force-error labels of three increasing gears (1..8)
    against the order-8 translation (gear 8 is exact: the floor)."""
    topo = state.topology
    K = topo.num_far_pairs
    dev = state.device
    cs8 = nat.coeff_stride(8, torch.float32)
    mult8 = torch.zeros((topo.num_nodes, cs8), dtype=torch.float32, device=dev)
    centers = torch.zeros_like(state.centers4)
    s = nat.current_stream()
    code = nat.JFM_F32
    nat.call("jfm_p2m", s, code, 8, state.pos4.data_ptr(), topo.num_particles, topo.num_leaves, topo.leaf_size,
             topo.num_internal, mult8.data_ptr(), centers.data_ptr())
    off = nat.host_i32(topo.m2m_off)
    nat.call("jfm_m2m_pass", s, code, 8, state.m2m_nodes.data_ptr(), nat.ptr(off), len(off) - 1,
             state.left.data_ptr(), state.right.data_ptr(), state.node_range.data_ptr(), mult8.data_ptr(),
             centers.data_ptr())
    tgt, src, rad = pair_arrays(state)
    T = torch.empty((K, NUM_OUTPUTS), dtype=torch.float32, device=dev)
    g3 = np.asarray(tuple(int(g) for g in gears), np.int32)
    nat.call("jfm_pair_labels", s, K, tgt.data_ptr(), src.data_ptr(), mult8.data_ptr(), centers.data_ptr(),
             rad.data_ptr(), nat.ptr(g3), T.data_ptr())
    return T


@dataclass
class GearSchedule:
    """Per-gear CSR far lists (device) built from per-pair gears."""

    gears: tuple
    targets: list
    num_targets: list
    offsets: list
    sources: list
    counts: dict
    m2l_flops: float
    flat: list = None  # per gear: FlatList (lane-per-pair launch) or None (wave per target)


def build_gear_schedule(state, gear_of_pair, gears: Sequence[int]) -> GearSchedule:
    """Split the far CSR by gear on the device, keeping each target's source order.

    One radix sort of (gear slot << 32 | pair) keys groups the pairs by gear in
    CSR order; each gear's pairs then give its CSR (offsets over all nodes,
    sources), its targets and, when its targets are sparse, its lane-per-pair
    list (``flatlist``)."""
    from .dtopology import _csr, _sort_u64
    from .perf import m2l_flops

    topo = state.topology
    dev = state.device
    s = nat.current_stream()
    nodes = topo.num_nodes
    K = topo.num_far_pairs
    g = torch.as_tensor(gear_of_pair)
    g = g.to(device=dev, dtype=torch.int8).contiguous() if K else torch.zeros(1, dtype=torch.int8, device=dev)
    g3 = np.asarray(tuple(int(x) for x in gears), np.int32)
    row_of = pair_targets(state)
    keys = torch.empty(max(K, 1), dtype=torch.int64, device=dev)
    flags = torch.zeros(1, dtype=torch.int32, device=dev)
    nat.call("jfm_gear_keys", s, K, g.data_ptr(), nat.ptr(g3), keys.data_ptr(), flags.data_ptr())
    sk, _ = _sort_u64(keys[:K], 34)
    off3_d, index = _csr(sk, 3)
    off3 = off3_d.cpu().numpy()
    if int(flags.item()) or int(off3[3]) != K:
        raise ValueError(f"every pair's gear must be one of {tuple(g3.tolist())}")
    del keys, sk
    targets, num_targets, offsets, sources, counts, flat = [], [], [], [], {}, []
    flops = 0.0
    one = torch.zeros(1, dtype=torch.int32, device=dev)
    for gi, gear in enumerate(gears):
        a, b = int(off3[gi]), int(off3[gi + 1])
        n = b - a
        pt = torch.empty(max(n, 1), dtype=torch.int32, device=dev)
        ps = torch.empty(max(n, 1), dtype=torch.int32, device=dev)
        nat.call("jfm_gather_pairs", s, n, index[a:].data_ptr() if n else None, row_of.data_ptr() if n else None,
                 state.far_src.data_ptr(), pt.data_ptr(), ps.data_ptr())
        pt, ps = pt[:n], ps[:n]
        pk = torch.empty(max(n, 1), dtype=torch.int64, device=dev)
        nat.call("jfm_pair_keys", s, n, pt.data_ptr(), ps.data_ptr(), pk.data_ptr())
        off, src = _csr(pk[:n], nodes)  # the gear's pairs are already in (target, source) order
        rows = torch.empty(max(nodes, 1), dtype=torch.int64, device=dev)
        cnt = torch.zeros(1, dtype=torch.int64, device=dev)
        nat.call("jfm_nonempty_rows", s, nodes, off.data_ptr(), rows.data_ptr(), cnt.data_ptr())
        nt = int(cnt.item())
        tl, _ = _sort_u64(rows[:nt], 32)
        counts[int(gear)] = n
        flops += m2l_flops(int(gear)) * float(n)
        targets.append(tl.to(torch.int32) if nt else one)
        offsets.append(off)
        sources.append(src if n else one)
        num_targets.append(nt)
        flat.append(build_flat_list(pt, ps, int(gear), state.dtype, dev, grouped=True) if prefers_flat(n, nt) else None)
    return GearSchedule(tuple(int(x) for x in gears), targets, num_targets, offsets, sources, counts, flops, flat)

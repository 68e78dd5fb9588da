"""Run-time judge of the learned per-pair M2L orders, with the plain
fixed-order FMM as fallback.

The reference accepts a far pair at the highest gear (its safety check) and
then tags it with the smallest passing gear (README.md:290-299,
runtime/_adaptive_policy.py:2216-2384).  Here a learned model picks the gear,
so nothing in the model itself guarantees the result: after the gears are
chosen in ``prepare_state``, the judge evaluates, on a seeded sample of
targets,

* the FMM with the learned per-pair gears, and
* the plain FMM with every far pair at the top gear (same topology, same
  near field, same precision policy),

both against the float64 direct sum at those targets.  When the learned
median relative force error exceeds ``factor`` times the plain one (plus a
float32 noise floor), the state falls back to the plain fixed-order far field:
the gear schedule is dropped and the downward pass runs every pair at the top
gear.  The decision and both error figures are recorded in
``state.extra["order_judge"]``.
"""

from __future__ import annotations

import dataclasses

import numpy as np
import torch

from . import _native as nat
from .direct import direct_sum_gravitational_acceleration
from .nearsplit import P2PItems

# relative force errors below this are float32 rounding, not truncation
NOISE_FLOOR = 2e-6


def _errors(acc: torch.Tensor, ref: torch.Tensor) -> np.ndarray:
    a = acc.to(torch.float64)
    return (torch.linalg.norm(a - ref, dim=1) / torch.linalg.norm(ref, dim=1).clamp_min(1e-300)).cpu().numpy()


def _near_rows(fmm, state, targets: torch.Tensor) -> torch.Tensor:
    """Near-field accelerations [N, 3] (input order) of the leaves that hold ``targets``."""
    topo = state.topology
    dev = state.device
    n, leaf = topo.num_particles, topo.leaf_size
    wanted = torch.zeros(n, dtype=torch.bool, device=dev)
    wanted[targets] = True
    of_leaf = torch.zeros(topo.num_leaves * leaf, dtype=torch.bool, device=dev)
    of_leaf[:n] = wanted[state.perm.long()]
    of_leaf = of_leaf.view(topo.num_leaves, leaf).any(1)
    items = state.extra.get("p2p_items")
    if items is None:
        rows = torch.nonzero(of_leaf).reshape(-1)
        slots = ((state.near_off[1:] - state.near_off[:-1] + 1) * leaf)[rows]
        none = torch.zeros(1, dtype=torch.int32, device=dev)
        some = P2PItems(num_items=int(rows.numel()), leaf=rows.to(torch.int32), s0=torch.zeros_like(slots), s1=slots,
                        part=torch.full_like(slots, -1), num_part=0,
                        partials=torch.zeros((1, leaf, 4), dtype=state.dtype, device=dev), num_split=0,
                        split_leaf=none, split_p0=none, split_p1=none)
    else:
        k = torch.nonzero(of_leaf[items.leaf.long()]).reshape(-1)
        c = torch.nonzero(of_leaf[items.split_leaf.long()]).reshape(-1)
        some = dataclasses.replace(items, num_items=int(k.numel()), leaf=items.leaf[k], s0=items.s0[k], s1=items.s1[k],
                                   part=items.part[k], num_split=int(c.numel()), split_leaf=items.split_leaf[c],
                                   split_p0=items.split_p0[c], split_p1=items.split_p1[c])
    acc = torch.zeros((n, 3), dtype=state.dtype, device=dev)
    fmm._p2p_items(state, some, acc, None, nat.EVAL_COMPENSATED if state.compensated else 0, accumulate=False)
    return acc


def _with_far_field(state, acc: torch.Tensor) -> torch.Tensor:
    """``acc`` (near field, input order) with the far field of the state's locals added."""
    topo = state.topology
    nat.call("jfm_l2p", nat.current_stream(), nat.dtype_code(state.dtype), state.order, state.pos4.data_ptr(),
             topo.num_particles, topo.leaf_size, topo.num_internal, state.locals.data_ptr(),
             state.centers4.data_ptr(), state.G, state.perm.data_ptr(), acc.data_ptr(), None, 1)
    return acc


def judge_learned_orders(fmm, state, positions: torch.Tensor, masses: torch.Tensor, *, num_targets: int,
                         factor: float, seed: int) -> dict:
    """Judge the learned gears of ``state`` (prepared, gears set, expansions of
    the learned downward pass in place) on ``num_targets`` seeded targets and
    fall back to the top gear for every pair when they lose.  ``positions`` /
    ``masses`` are the device inputs in input order."""
    sched = state.extra.get("gears")
    if sched is None:
        raise ValueError("the state has no learned gears to judge")
    n = state.num_particles
    k = int(min(max(num_targets, 1), n))
    tgt = np.sort(np.random.default_rng(seed).choice(n, size=k, replace=False)).astype(np.int64)
    tgt_d = torch.as_tensor(tgt, device=state.device)
    ref = direct_sum_gravitational_acceleration(positions, masses, G=state.G, softening=state.softening,
                                                target_indices=tgt)

    # the near field does not depend on the orders: once, and only for the
    # leaves that hold targets (rows of other leaves stay unwritten)
    near = _near_rows(fmm, state, tgt_d)
    acc = _with_far_field(state, near.clone())
    err_learned = _errors(acc[tgt_d], ref)
    locals_learned = state.locals.clone()

    # the judge: every far pair at the top gear on the same expansions
    state.extra["gears"] = None
    s = nat.current_stream()
    fmm._downward(state, s, nat.dtype_code(state.dtype))
    err_plain = _errors(_with_far_field(state, near)[tgt_d], ref)

    med_l, med_p = float(np.median(err_learned)), float(np.median(err_plain))
    accepted = med_l <= factor * med_p + NOISE_FLOOR
    from .perf import m2l_flops

    verdict = {
        "accepted": bool(accepted), "targets": k, "seed": int(seed), "factor": float(factor),
        "median_learned": med_l, "median_plain": med_p,
        "p99_learned": float(np.percentile(err_learned, 99)), "p99_plain": float(np.percentile(err_plain, 99)),
        "m2l_gflop_learned": sched.m2l_flops / 1e9,
        "m2l_gflop_plain": m2l_flops(state.order) * state.topology.num_far_pairs / 1e9,
    }
    if accepted:
        state.extra["gears"] = sched
        state.locals.copy_(locals_learned)
    else:
        # fallback: the plain fixed-order far field just computed stays
        state.extra.pop("gear_of_pair", None)
        state.extra.pop("gears", None)
    state.extra["order_judge"] = verdict
    return verdict

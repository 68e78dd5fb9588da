"""Which steps run their near field on a stream of its own (on the CPU)."""

from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

from jaccpot_amd.solver import FastMultipoleMethod

# pairs measured on either side: float64 ones take 2.5 times as long
CASES = ((8.6e6, torch.float64, False), (1.7e7, torch.float64, True), (2.1e7, torch.float64, True),
         (1.4e7, torch.float32, False), (2.1e7, torch.float32, False), (1.1e8, torch.float32, True))


@pytest.mark.parametrize("pairs,dtype,forks", CASES)
def test_fork_counts_pairs_by_their_cost(pairs, dtype, forks):
    fmm = object.__new__(FastMultipoleMethod)  # the rule reads sizes only
    topo = SimpleNamespace(leaf_size=16, num_leaves=256, num_near_entries=int(pairs / 256) - 256)
    assert fmm._forks(topo, dtype) == forks

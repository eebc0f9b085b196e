"""Edges of the wave-level top-k (selections and experts past one per lane,
masked and tied logits) and of the one-block permute (slot counts around its
waves and its limit, empty and single experts)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _helpers import banner
from oracle import oracle
from reframework_amd.moe import torch_fused_topk
from test_gpu_experts import test_permute_bit_exact as check_permute

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,K", [(1, 1), (63, 63), (64, 64), (65, 65), (130, 129), (256, 65),
                                 (256, 256)])
def test_topk_past_one_per_lane(E, K, dev):
    banner(f"topk E={E} K={K}")
    rng = np.random.default_rng(E + K)
    logits = (rng.normal(size=(37, E)) * 2).astype(np.float32)
    logits[::3] = np.round(logits[::3])      # exact ties
    logits[1::5, (E + 1) // 2:] = -np.inf    # masked experts, selected last in id order
    for renorm in (True, False):
        w, ids = torch_fused_topk(torch.from_numpy(logits).to(dev), K, renorm)
        ow, oids = oracle.topk(logits, K, renorm)
        assert np.array_equal(ids.cpu().numpy(), oids)
        assert np.max(np.abs(w.cpu().numpy() - ow)) <= 1e-6


@pytest.mark.parametrize("T,K,E", [(65, 1, 1), (33, 2, 2), (64, 1, 65), (129, 1, 256), (127, 8, 200),
                                   (511, 2, 8), (1023, 1, 64), (1024, 1, 256), (1025, 1, 256),
                                   (128, 8, 256)])
@pytest.mark.parametrize("drop", [False, True])
def test_one_block_permute_sizes(T, K, E, drop, dev):
    check_permute(T, K, E, False, drop, dev)

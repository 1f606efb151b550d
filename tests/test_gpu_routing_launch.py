"""GPU: the one-launch routing kernel at the edges of its 512-route chunks, of
its largest size (16384 routes, above which the counting launches take over)
and of its id-load batches, equal to the host loop of vllm:119-146."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import mxfp4_amd as mx
from oracle import c_oracle

from _helpers import cuda

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("routes,num_experts,block_m",
                         [(1, 1, 16), (63, 1024, 16), (64, 9, 64), (300, 17, 32),
                          (511, 128, 64), (512, 128, 64), (513, 129, 32), (8191, 3, 48), (8193, 1024, 16), (16383, 64, 128),
                          (16384, 257, 64), (16385, 128, 64)])
@pytest.mark.parametrize("skew", [False, True])
def test_one_launch_routing_matches_host_loop(routes, num_experts, block_m, skew):
    g = torch.Generator().manual_seed(routes * 3 + skew)
    ids = torch.randint(-1, num_experts + 1, (routes, 1), generator=g)
    if skew:  # most routes on the last expert, some dropped
        ids = torch.where(torch.rand((routes, 1), generator=g) < 0.9,
                          torch.full_like(ids, num_experts - 1), ids)
    ref_ids, ref_experts, ref_npp = c_oracle.make_routing(ids.numpy(), num_experts, block_m)
    for dtype in (torch.int64, torch.int32):
        srt, exp_, npp = mx.make_routing(cuda(ids.to(dtype)), block_m=block_m,
                                         num_experts=num_experts)
        used = int(npp[0])
        assert used == int(ref_npp[0])
        assert np.array_equal(srt[:used].cpu().numpy(), ref_ids)
        assert np.array_equal(exp_[:used // block_m].cpu().numpy(), ref_experts)


def test_one_launch_routing_all_dropped():
    ids = torch.full((70, 8), -1)
    _, _, npp = mx.make_routing(cuda(ids), block_m=64, num_experts=16)
    assert int(npp[0]) == 0


# every route on one expert: the largest counts before and after a chunk, on
# one word of each of the kernel's count copies
@pytest.mark.parametrize("num_experts", [1, 2, 129, 1024])
@pytest.mark.parametrize("routes", [512, 16384])
def test_one_launch_routing_single_expert(routes, num_experts):
    for expert in {0, num_experts - 1}:
        ids = torch.full((routes, 1), expert)
        srt, exp_, npp = mx.make_routing(cuda(ids), block_m=64, num_experts=num_experts)
        assert int(npp[0]) == routes
        assert np.array_equal(srt[:routes].cpu().numpy(), np.arange(routes))
        assert (exp_[:routes // 64] == expert).all()

"""GPU: the routed GEMM that loads its weights straight into registers, against
the FP64 oracle and, bit for bit, against the prefill tiles (which the same
call takes when the scale bytes are not 16-byte aligned): expert blocks of
every live row count around the 16-row groups and the 64-row blocks, column
counts that are no whole tile, one, odd and many 128-deep units of K, blocks of
32 / 64 / 128 rows, expert -1 blocks, all three C types, and the MoE layer on
both weight layouts."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import mxfp4_amd as mx
from oracle import mxfp4_oracle as O

from _helpers import assert_parity, cuda, rand_act, rand_mxfp4

pytestmark = pytest.mark.gpu

COUNTS = (0, 1, 15, 16, 17, 32, 33, 48, 49, 64, 65, 130)


def _shifted(t):
    """The same bytes at an address 4 past a 16-byte boundary."""
    buf = torch.empty(t.numel() + 16, dtype=t.dtype, device=t.device)
    s = buf[4:4 + t.numel()].view(t.shape)
    s.copy_(t)
    assert s.data_ptr() % 16 == 4 and s.is_contiguous()
    return s


def _routes(seed):
    ids = np.repeat(np.arange(len(COUNTS)), COUNTS)
    np.random.default_rng(seed).shuffle(ids)
    return ids.reshape(-1, 1)


@pytest.mark.parametrize("n,k", [(48, 128), (200, 384), (1000, 256), (520, 2048)])
@pytest.mark.parametrize("block_m", [32, 64, 128])
@pytest.mark.parametrize("a_dtype,c_dtype", [(torch.bfloat16, torch.bfloat16),
                                             (torch.float16, torch.float16),
                                             (torch.bfloat16, torch.float32)])
def test_routed_blocks(n, k, block_m, a_dtype, c_dtype):
    e = len(COUNTS)
    ids = _routes(n + k)
    m = ids.shape[0]
    rng = np.random.default_rng(n * 7 + k)
    wp, ws = rand_mxfp4(rng, (e, n), k)
    a = rand_act(k, (m, k), a_dtype)
    w = torch.rand((m, 1), generator=torch.Generator().manual_seed(n))
    srt, exp_, npp = (cuda(t) for t in O.make_routing(ids, block_m=block_m, num_experts=e))
    b_scale = torch.linspace(1, 2, e)
    s = cuda(ws)
    outs = []
    for scales, experts in ((s, exp_), (_shifted(s), exp_),
                            (s, torch.where(exp_ == 8, torch.full_like(exp_, -1), exp_))):
        C = torch.full((m, 1, n), 3.0, dtype=c_dtype, device="cuda")
        mx.fused_moe_mxfp4(cuda(a), cuda(wp), C, torch.tensor([0.5], device="cuda"),
                           cuda(b_scale), None, scales, cuda(w), cuda(ids), srt, experts, npp,
                           True, 1, False, False, {"BLOCK_SIZE_M": block_m}, c_dtype)
        outs.append(C)
    direct, tiles, masked = outs
    assert torch.equal(direct, tiles)
    oracle = O.fused_moe_fp64(a.float().numpy(), wp, ws, 0.5, b_scale.numpy(), w.numpy(), ids,
                              True)
    assert_parity(direct.float().cpu().numpy(), oracle)
    keep = cuda(ids[:, 0]) != 8
    assert torch.equal(masked[keep], direct[keep]) and not masked[~keep].any()


# scale byte 255 (NaN) in every other row, an odd number of 128-deep units: the
# rows beside it stay finite (no scale byte past a row's own is applied)
@pytest.mark.parametrize("k", [128, 384, 640])
@pytest.mark.parametrize("n", [64, 200])
def test_nan_scales_stay_in_their_row(n, k):
    e = len(COUNTS)
    ids = _routes(n + k)
    m = ids.shape[0]
    wp, ws = rand_mxfp4(np.random.default_rng(k), (e, n), k)
    ws[:, 1::2, 0] = 255
    a = cuda(rand_act(k, (m, k)))
    srt, exp_, npp = (cuda(t) for t in O.make_routing(ids, block_m=64, num_experts=e))
    one, ones = torch.ones(1, device="cuda"), torch.ones(e, device="cuda")
    outs = []
    for scales in (cuda(ws), _shifted(cuda(ws))):
        C = torch.full((m, 1, n), 3.0, dtype=torch.bfloat16, device="cuda")
        mx.fused_moe_mxfp4(a, cuda(wp), C, one, ones, None, scales,
                           torch.ones((m, 1), device="cuda"), cuda(ids), srt, exp_, npp, False, 1,
                           False, False, {"BLOCK_SIZE_M": 64}, C.dtype)
        outs.append(C)
    assert torch.isnan(outs[0][..., 1::2]).all() and torch.isfinite(outs[0][..., ::2]).all()
    assert torch.equal(outs[0].nan_to_num(7.0), outs[1].nan_to_num(7.0))


# soft op: the safe call's own routing, with dropped ids (zero rows)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,e,top_k,n,k", [(40, 16, 4, 136, 640), (300, 8, 2, 1024, 1408),
                                           (260, 128, 8, 512, 256)])
def test_soft_op(m, e, top_k, n, k, dtype):
    rng = np.random.default_rng(m)
    wp, ws = (cuda(t) for t in rand_mxfp4(rng, (e, n), k))
    a = cuda(rand_act(m, (m, k), dtype))
    g = torch.Generator().manual_seed(m)
    ids = cuda(torch.randint(-1, e + 1, (m, top_k), generator=g))
    w = cuda(torch.rand((m, top_k), generator=g))
    one, ones, none = (torch.ones(1, device="cuda"), torch.ones(e, device="cuda"),
                       torch.empty(0, device="cuda"))
    outs = []
    for scales in (ws, _shifted(ws)):
        C = torch.full((m, top_k, n), 3.0, dtype=dtype, device="cuda")
        mx.fused_moe_mxfp4_soft(a, wp, C, one, ones, None, scales, w, ids, none, none, none, True,
                                top_k, False, False)
        outs.append(C)
    assert torch.equal(outs[0], outs[1])
    assert not outs[0][(ids < 0) | (ids >= e)].any()


# the layer: full and small grids, both layouts, against the prefill tiles
@pytest.mark.parametrize("prepacked", [False, True])
@pytest.mark.parametrize("m,e,top_k,hidden,inter", [(20, 128, 8, 256, 128),
                                                    (100, 16, 4, 512, 384),
                                                    (250, 8, 2, 640, 1408),
                                                    (385, 128, 8, 1024, 256)])
def test_layer(m, e, top_k, hidden, inter, prepacked):
    rng = np.random.default_rng(m + e)
    w13, s13 = (cuda(t) for t in rand_mxfp4(rng, (e, 2 * inter), hidden))
    w2, s2 = (cuda(t) for t in rand_mxfp4(rng, (e, hidden), inter))
    x = cuda(rand_act(m, (m, hidden)))
    g = torch.Generator().manual_seed(m)
    ids = cuda(torch.randint(-1, e, (m, top_k), generator=g))
    w = cuda(torch.rand((m, top_k), generator=g))
    outs = []
    for a13, a2 in ((s13, s2), (_shifted(s13), _shifted(s2))):
        pre = (mx.prepack_w4a16(w13, a13), mx.prepack_w4a16(w2, a2)) if prepacked else (None, None)
        outs.append(mx.moe_layer(x, w13, a13, w2, a2, w, ids, prepacked13=pre[0],
                                 prepacked2=pre[1]))
    assert torch.equal(outs[0], outs[1])

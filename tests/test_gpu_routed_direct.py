"""GPU: the routed GEMM that loads its weights straight into registers, against
the FP64 oracle and, bit for bit, against the prefill tiles (which the same
call takes when the scale bytes are not 16-byte aligned): expert blocks of
every live row count around the 16-row groups and the 64-row blocks, column
counts that are no whole tile, one, odd and many 128-deep units of K up to the
LDS limits, blocks of 32 / 64 / 128 rows, tiles of 128 and 256 columns, expert
-1 blocks, all three C types, the workspace of another plan, and the MoE layer
on both weight layouts.  Which kernel and tile a case is aimed at is asked of
the dispatch rule."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import mxfp4_amd as mx
from mxfp4_amd import _lib
from oracle import mxfp4_oracle as O

from _helpers import assert_parity, cuda, dr_columns, rand_act, rand_mxfp4, shifted

pytestmark = pytest.mark.gpu

COUNTS = (0, 1, 15, 16, 17, 32, 33, 48, 49, 64, 65, 130)


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
    assert dr_columns(m, e, n, k, block_m=block_m, rows=min(block_m, 64)) == 128
    rng = np.random.default_rng(n * 7 + k)
    wp, ws = rand_mxfp4(rng, (e, n), k)
    a = rand_act(k, (m, k), a_dtype)
    w = torch.rand((m, 1), generator=torch.Generator().manual_seed(n))
    srt, exp_, npp = (cuda(t) for t in O.make_routing(ids, block_m=block_m, num_experts=e))
    b_scale = torch.linspace(1, 2, e)
    s = cuda(ws)
    outs = []
    for scales, experts in ((s, exp_), (shifted(s), exp_),
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
    assert dr_columns(m, e, n, k, block_m=64) == 128
    wp, ws = rand_mxfp4(np.random.default_rng(k), (e, n), k)
    ws[:, 1::2, 0] = 255
    a = cuda(rand_act(k, (m, k)))
    srt, exp_, npp = (cuda(t) for t in O.make_routing(ids, block_m=64, num_experts=e))
    one, ones = torch.ones(1, device="cuda"), torch.ones(e, device="cuda")
    outs = []
    for scales in (cuda(ws), shifted(cuda(ws))):
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
    assert dr_columns(m * top_k, e, n, k, block_m=32 if m < 300 else 64)
    rng = np.random.default_rng(m)
    wp, ws = (cuda(t) for t in rand_mxfp4(rng, (e, n), k))
    a = cuda(rand_act(m, (m, k), dtype))
    g = torch.Generator().manual_seed(m)
    ids = cuda(torch.randint(-1, e + 1, (m, top_k), generator=g))
    w = cuda(torch.rand((m, top_k), generator=g))
    one, ones, none = (torch.ones(1, device="cuda"), torch.ones(e, device="cuda"),
                       torch.empty(0, device="cuda"))
    outs = []
    for scales in (ws, shifted(ws)):
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
    for a13, a2 in ((s13, s2), (shifted(s13), shifted(s2))):
        pre = (mx.prepack_w4a16(w13, a13), mx.prepack_w4a16(w2, a2)) if prepacked else (None, None)
        outs.append(mx.moe_layer(x, w13, a13, w2, a2, w, ids, prepacked13=pre[0],
                                 prepacked2=pre[1]))
    assert torch.equal(outs[0], outs[1])


# ------------------------------------------------------- 256-column tiles
# 128 experts whose blocks have 0 to 4 live groups of 16 rows, a ragged last
# column tile (N = 1000, 1032), an odd number of 128-deep units of K
WIDE_COUNTS = (0, 1, 15, 16, 17, 20, 32, 33, 48, 49, 64, 65)


def _wide_routes(seed, e=128):
    ids = np.repeat(np.arange(e), [WIDE_COUNTS[i % len(WIDE_COUNTS)] for i in range(e)])
    np.random.default_rng(seed).shuffle(ids)
    return ids.reshape(-1, 1)


def _aiter(a, wp, scales, C, b_scale, w, ids, block_m, experts=None):
    srt, exp_, npp = mx.make_routing_device(ids, wp.shape[0], block_m)
    mx.fused_moe_mxfp4(a, wp, C, torch.tensor([0.5], device="cuda"), b_scale, None, scales, w, ids,
                       srt, exp_ if experts is None else experts(exp_), npp, True, 1, False, False,
                       {"BLOCK_SIZE_M": block_m}, C.dtype)
    return C


@pytest.mark.parametrize("n,k", [(1000, 384), (1032, 640)])
@pytest.mark.parametrize("block_m", [32, 64])
@pytest.mark.parametrize("a_dtype,c_dtype", [(torch.bfloat16, torch.bfloat16),
                                             (torch.float16, torch.float16),
                                             (torch.bfloat16, torch.float32)])
def test_wide_tiles(n, k, block_m, a_dtype, c_dtype):
    e = 128
    ids = _wide_routes(n + k)
    m = ids.shape[0]
    assert dr_columns(m, e, n, k, block_m=block_m, rows=block_m) == 256
    wp, ws = rand_mxfp4(np.random.default_rng(n * 5 + k), (e, n), k)
    a = rand_act(k + 3, (m, k), a_dtype)
    w = torch.rand((m, 1), generator=torch.Generator().manual_seed(n))
    b_scale = torch.linspace(1, 2, e)
    args = (cuda(b_scale), cuda(w), cuda(ids))
    ad, wd, s = cuda(a), cuda(wp), cuda(ws)

    def run(scales, experts=None):
        C = torch.full((m, 1, n), 3.0, dtype=c_dtype, device="cuda")
        return _aiter(ad, wd, scales, C, *args, block_m, experts)

    direct = run(s)
    assert torch.equal(direct, run(shifted(s)))
    masked = run(s, lambda x: torch.where(x == 8, torch.full_like(x, -1), x))
    keep = cuda(ids[:, 0]) != 8
    assert torch.equal(masked[keep], direct[keep]) and not masked[~keep].any()
    rows = np.arange(0, m, 37)
    oracle = O.fused_moe_fp64(a.float().numpy()[rows], wp, ws, 0.5, b_scale.numpy(),
                              w.numpy()[rows], ids[rows], True)
    assert_parity(direct.float().cpu().numpy()[rows], oracle)
    # NaN scales in every other weight row: the rows beside them stay finite
    s[:, 1::2, 0] = 255
    nan = run(s)
    assert torch.isnan(nan[..., 1::2]).all() and torch.isfinite(nan[..., ::2]).all()
    assert torch.equal(nan.nan_to_num(7.0), run(shifted(s)).nan_to_num(7.0))


# tiles above 64 KB of LDS, at and past the limits of 256 and 128 columns
@pytest.mark.parametrize("n,k,columns", [(1000, 4096, 256), (1000, 6016, 256), (1000, 6144, 128),
                                         (200, 12032, 128), (200, 12160, 0)])
def test_lds_limits(n, k, columns):
    e = 128 if n == 1000 else 12
    ids = cuda(_wide_routes(k, e))
    m = ids.shape[0]
    assert dr_columns(m, e, n, k, block_m=64) == columns
    g = torch.Generator(device="cuda").manual_seed(k)
    wp = torch.randint(0, 256, (e, n, k // 2), dtype=torch.uint8, device="cuda", generator=g)
    ws = torch.randint(120, 129, (e, n, k // 32), dtype=torch.uint8, device="cuda", generator=g)
    a = cuda(rand_act(k + 5, (m, k)))
    w = torch.rand((m, 1), device="cuda", generator=g)
    ones = torch.ones(e, device="cuda")
    C, T = (_aiter(a, wp, s, torch.full((m, 1, n), 3.0, dtype=torch.bfloat16, device="cuda"), ones,
                   w, ids, 64) for s in (ws, shifted(ws)))
    assert torch.equal(C, T)
    rows = np.arange(0, m, max(1, m // 6))
    used = np.unique(ids.cpu().numpy()[rows])
    local = np.searchsorted(used, ids.cpu().numpy()[rows])
    oracle = O.fused_moe_fp64(a.float().cpu().numpy()[rows], wp[used].cpu().numpy(),
                              ws[used].cpu().numpy(), 0.5, np.ones(len(used)),
                              w.cpu().numpy()[rows], local, True)
    assert_parity(C.float().cpu().numpy()[rows], oracle)


# the SiLU epilogue and the down GEMM on 256-column tiles, both layouts
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("prepacked", [False, True])
def test_wide_layer(prepacked, dtype):
    m, e, top_k, hidden, inter = 384, 128, 8, 1152, 640  # 9 and 5 units of K
    assert dr_columns(m * top_k, e, inter, hidden, block_m=32, silu=True,
                      prepacked=prepacked) == 256
    rng = np.random.default_rng(m + e)
    # scales of 2^-11 .. 2^-5: gate * up stays finite in fp16
    w13, s13 = (cuda(t) for t in rand_mxfp4(rng, (e, 2 * inter), hidden, 116, 122))
    w2, s2 = (cuda(t) for t in rand_mxfp4(rng, (e, hidden), inter, 116, 122))
    x = cuda(rand_act(m, (m, hidden), dtype))
    g = torch.Generator().manual_seed(m)
    # skewed, so that blocks of 1 to 4 live groups and experts of several occur
    p = 1.0 / torch.arange(2, e + 2)
    ids = cuda(torch.multinomial(p.expand(m, e), top_k, generator=g))
    w = cuda(torch.rand((m, top_k), generator=g))
    outs = []
    for a13, a2 in ((s13, s2), (shifted(s13), shifted(s2))):
        pre = (mx.prepack_w4a16(w13, a13), mx.prepack_w4a16(w2, a2)) if prepacked else (None, None)
        outs.append(mx.moe_layer(x, w13, a13, w2, a2, w, ids, prepacked13=pre[0],
                                 prepacked2=pre[1]))
    assert torch.isfinite(outs[0]).all() and torch.equal(outs[0], outs[1])


# The C entries on less workspace than the 64-row plan of this kernel needs:
# the least they accept is the other plan's, and the result is bitwise the same
def _least(call, enough):
    """Smallest accepted workspace (refused before anything is enqueued)."""
    low, high = 0, enough
    while low < high:
        mid = (low + high) // 2
        if call(mid) == _lib.OK:
            high = mid
        else:
            low = mid + 1
    return low


def test_soft_op_on_the_other_plans_workspace():
    m, e, top_k, n, k = 300, 16, 4, 200, 640
    assert dr_columns(m * top_k, e, n, k, block_m=64)
    rng = np.random.default_rng(3)
    wp, ws = (cuda(t) for t in rand_mxfp4(rng, (e, n), k))
    a = cuda(rand_act(3, (m, k)))
    g = torch.Generator().manual_seed(3)
    ids = cuda(torch.randint(-1, e + 1, (m, top_k), generator=g).int())
    w = cuda(torch.rand((m, top_k), generator=g))
    C = torch.empty((m, top_k, n), dtype=torch.bfloat16, device="cuda")
    lib, size = _lib.load(), ctypes.c_int64()
    _lib.check(lib.mxfp4_fused_moe_workspace_size(m, top_k, e, _lib.DT_BF16, _lib.DT_BF16,
                                                  ctypes.byref(size)))
    buf = torch.empty(size.value, dtype=torch.uint8, device="cuda")

    def call(nbytes):
        return lib.mxfp4_fused_moe(
            _lib.ptr(a), _lib.DT_BF16, m, k, None, _lib.ptr(wp), _lib.ptr(ws), e, n, k,
            _lib.ptr(C), _lib.DT_BF16, None, None, _lib.ptr(w), 1, _lib.ptr(ids), _lib.DT_I32, m,
            top_k, _lib.ptr(buf), nbytes, _lib.stream_of(a.device))

    outs = []
    for nbytes in (size.value, _least(call, size.value)):
        C.fill_(3.0)
        assert call(nbytes) == _lib.OK
        outs.append(C.clone())
    assert nbytes < size.value and torch.equal(*outs)


@pytest.mark.parametrize("prepacked", [False, True])
def test_layer_on_the_other_plans_workspace(prepacked):
    m, e, top_k, hidden, inter = 100, 16, 4, 512, 384
    assert dr_columns(m * top_k, e, inter, hidden, block_m=32, silu=True, prepacked=prepacked)
    rng = np.random.default_rng(5)
    w13, s13 = (cuda(t) for t in rand_mxfp4(rng, (e, 2 * inter), hidden))
    w2, s2 = (cuda(t) for t in rand_mxfp4(rng, (e, hidden), inter))
    pre = (mx.prepack_w4a16(w13, s13), mx.prepack_w4a16(w2, s2)) if prepacked else ()
    copies = [_lib.ptr(t) for p in pre for t in (p.nibbles, p.scales)] or [None] * 4
    x = cuda(rand_act(5, (m, hidden)))
    g = torch.Generator().manual_seed(5)
    ids = cuda(torch.randint(-1, e, (m, top_k), generator=g).int())
    w = cuda(torch.rand((m, top_k), generator=g))
    out = torch.empty((m, hidden), dtype=torch.bfloat16, device="cuda")
    lib, size = _lib.load(), ctypes.c_int64()
    _lib.check(lib.mxfp4_moe_layer_workspace_size(m, top_k, e, hidden, inter, ctypes.byref(size)))
    buf = torch.empty(size.value, dtype=torch.uint8, device="cuda")

    def call(nbytes):
        return lib.mxfp4_moe_layer_pre(
            _lib.ptr(x), _lib.DT_BF16, m, hidden, _lib.ptr(w13), _lib.ptr(s13), *copies[:2],
            _lib.ptr(w2), _lib.ptr(s2), *copies[2:], e, inter, _lib.ptr(w), _lib.ptr(ids),
            _lib.DT_I32, top_k, _lib.ptr(out), _lib.ptr(buf), nbytes, _lib.stream_of(x.device))

    outs = []
    for nbytes in (size.value, _least(call, size.value)):
        out.fill_(3.0)
        assert call(nbytes) == _lib.OK
        outs.append(out.clone())
    assert nbytes < size.value and torch.equal(*outs)

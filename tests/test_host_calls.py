"""The operators' native call paths: a plain call gives bit for bit what the
general Python path gives, and everything else is handed to that path (None):
CPU tensors, subclasses, modes, functorch wrappers, layouts, types and
shapes the native code does not take."""

from __future__ import annotations

import sys
import warnings
from types import ModuleType, SimpleNamespace

import numpy as np
import pytest
import torch
from torch.overrides import BaseTorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

import mxfp4_amd as mx
from mxfp4_amd import _lib

from _helpers import cuda, rand_act, rand_mxfp4


def _weights(rng, rows, k, dev=lambda a: torch.from_numpy(a)):
    return tuple(dev(t) for t in rand_mxfp4(rng, rows, k))


def test_cpu_tensors_and_wrong_counts_are_not_taken():
    host = _lib.host()
    rng = np.random.default_rng(0)
    w, s = _weights(rng, (32,), 128)
    x = rand_act(0, (2, 128))
    assert host.linear(x, w, s, None, None) is None
    assert host.linear(None, 1, "s", object(), x) is None
    assert host.align(torch.zeros((2, 2), dtype=torch.int64), 4, 16) is None
    assert host.route_topk(torch.zeros(4, 8), 10 ** 30, True, False) is None
    assert host.quant(x, 0) is None and host.w4a4(w, s, w, s, 0) is None
    with pytest.raises(TypeError):
        host.linear(x, w, s)
    with pytest.raises(TypeError):
        host.bind(_lib.check)


@pytest.mark.parametrize("fault", ["another torch", "no module", "no version"])
def test_module_that_does_not_fit_leaves_the_general_path(fault, monkeypatch):
    assert _lib.host().TORCH == _lib.torch_build()
    monkeypatch.setattr(_lib, "_host", None)
    if fault == "another torch":
        monkeypatch.setattr(_lib, "torch_build", lambda: "2.0.0 0123abcd")
    else:
        monkeypatch.setitem(sys.modules, "mxfp4_amd._host",
                            None if fault == "no module" else ModuleType("mxfp4_amd._host"))
    with pytest.warns(RuntimeWarning, match="_host.so"):
        assert _lib.host() is None
    with warnings.catch_warnings():  # said once
        warnings.simplefilter("error")
        assert _lib.host() is None
        # the operators go on to their own checks
        with pytest.raises(RuntimeError, match="ROCm devices only"):
            mx.linear_mxfp4_soft(torch.zeros((2, 128), dtype=torch.bfloat16),
                                 torch.zeros((32, 64), dtype=torch.uint8),
                                 torch.zeros((32, 4), dtype=torch.uint8))


# ------------------------------------------------------------------- GPU

def _cases():
    rng = np.random.default_rng(7)
    w, s = _weights(rng, (200,), 256, cuda)
    x = cuda(rand_act(1, (3, 5, 256)))
    bias = cuda(rand_act(2, (200,)))
    w13, s13 = _weights(rng, (8, 256), 256, cuda)
    w2, s2 = _weights(rng, (8, 256), 128, cuda)
    xm = cuda(rand_act(3, (9, 256)))
    logits = cuda(torch.randn((9, 8), generator=torch.Generator().manual_seed(4)))
    tw, ids = mx.route_topk(logits, 2)
    pre, pre13, pre2 = (mx.prepack_w4a16(*p) for p in ((w, s), (w13, s13), (w2, s2)))
    a8 = xm.to(torch.float8_e4m3fn)
    pk, ps = mx.dynamic_mxfp4_quant(xm, "rne")
    one, ones = torch.full((1,), 0.5, device="cuda"), torch.linspace(1, 2, 8, device="cuda")
    none = torch.empty(0, device="cuda")
    srt, exp_, npp = mx.make_routing_device(ids, 8, 16)

    def soft(a, a_mx, dt):
        C = torch.full((9, 2, 256), 3.0, dtype=dt, device="cuda")
        mx.fused_moe_mxfp4_soft(a, w13, C, one, ones, a_mx, s13, tw, ids, none, none, none, True,
                                2, False, False)
        return C

    def aiter(a, a_mx):
        C = torch.full((9, 2, 256), 3.0, dtype=torch.bfloat16, device="cuda")
        mx.fused_moe_mxfp4(a, w13, C, one, ones, a_mx, s13, tw, ids, srt, exp_, npp, True, 2,
                           False, False, {"BLOCK_SIZE_M": 16}, C.dtype)
        return C

    return {
        "linear": lambda: mx.linear_mxfp4_soft(x, w, s),
        "linear_bias": lambda: mx.linear_mxfp4_soft(x, w, s, bias, prepacked=pre),
        "linear_fp16": lambda: mx.linear_mxfp4_soft(x.half(), w, s),
        "layer": lambda: mx.moe_layer(xm, w13, s13, w2, s2, tw, ids),
        "layer_pre": lambda: mx.moe_layer(xm, w13, s13, w2, s2, tw, ids.int(), prepacked13=pre13,
                                          prepacked2=pre2),
        "soft": lambda: soft(xm, None, torch.bfloat16),
        "soft_f32": lambda: soft(xm, None, torch.float32),
        "soft_packed": lambda: soft(pk, ps, torch.bfloat16),
        "aiter": lambda: aiter(xm, None),
        "aiter_fp8": lambda: aiter(a8, None),
        "aiter_packed": lambda: aiter(pk, ps),
        "align": lambda: mx.make_routing_device(ids, 8, 32)[2],
        "route": lambda: mx.route_topk(logits, 3, False, torch.int32),
        "quant": lambda: mx.dynamic_mxfp4_quant(x, "ties_away"),
        "w4a4": lambda: mx.linear_mxfp4_w4a4(pk, ps, w, s, torch.float16),
    }


def _flat(v):
    return list(v) if isinstance(v, tuple) else [v]


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["linear", "linear_bias", "linear_fp16", "layer", "layer_pre",
                                  "soft", "soft_f32", "soft_packed", "aiter", "aiter_fp8",
                                  "aiter_packed", "align", "route", "quant", "w4a4"])
def test_native_call_equals_general_path(name, monkeypatch):
    call = _cases()[name]
    taken = []
    host = _lib.host()

    class Spy:
        def __getattr__(self, fn):
            def run(*a):
                r = getattr(host, fn)(*a)
                taken.append(r is not None)
                return r
            return run

    monkeypatch.setattr(_lib, "host", Spy)
    native = _flat(call())
    assert taken and taken[-1]
    monkeypatch.setattr(_lib, "host", lambda: None)
    general = _flat(call())
    for a, b in zip(native, general):
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)
    # modes: the general path runs, with the same result
    monkeypatch.setattr(_lib, "host", Spy)

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    for mode in (BaseTorchFunctionMode(), Dispatch()):
        del taken[:]
        with mode:
            under = _flat(call())
        assert taken and not any(taken)
        for a, b in zip(under, general):
            assert torch.equal(a, b)


@pytest.mark.gpu
def test_calls_that_are_not_plain(monkeypatch):
    host = _lib.host()
    rng = np.random.default_rng(9)
    w, s = _weights(rng, (64,), 256, cuda)
    x = cuda(rand_act(5, (4, 256)))

    class Sub(torch.Tensor):
        pass

    assert host.linear(x, w, s, None, None) is not None
    assert host.linear(torch.nn.Parameter(x), w, s, None, None) is not None
    wide = torch.cat([x, x], 1)
    off = torch.empty(4 * 256 + 8, dtype=x.dtype, device="cuda")[1:1 + 4 * 256].view(4, 256)
    for args in ((x.as_subclass(Sub), w, s, None, None), (wide[:, :256], w, s, None, None),
                 (off, w, s, None, None), (x.float(), w, s, None, None),
                 (x[:, :128].contiguous(), w, s, None, None), (x[:0], w, s, None, None),
                 (x, w, s[:, :4], None, None), (x, w, s, torch.zeros(64, device="cuda"), None),
                 (x, w, s, None, object()), (x, w, s.cpu(), None, None)):
        assert host.linear(*args) is None
    # a stale copy and one of other tensors: refused by the general path
    pre = mx.prepack_w4a16(w, s)
    assert host.linear(x, w, s, None, pre) is not None
    assert host.linear(x, w.clone(), s, None, pre) is None
    w.add_(0)
    assert host.linear(x, w, s, None, pre) is None
    with pytest.raises(ValueError):
        mx.linear_mxfp4_soft(x, w, s, prepacked=pre)
    # the other switches
    monkeypatch.setenv("MXFP4_GFX936_BACKEND", "triton")
    assert host.linear(x, w, s, None, None) is None
    monkeypatch.delenv("MXFP4_GFX936_BACKEND")
    assert host.linear(x, w, s, None, None) is not None
    # functorch: a batched wrapper is not a plain tensor
    seen = []
    torch.vmap(lambda t: seen.append(host.linear(t, w, s, None, None)) or t)(x.unsqueeze(0))
    assert seen == [None]
    # another registered copy turns the lookup on
    w2, s2 = w.clone(), s.clone()
    mx.register_prepacked(w2, s2)
    assert torch.equal(mx.linear_mxfp4_soft(x, w2, s2), mx.linear_mxfp4_soft(x, w, s))
    mx.unregister_prepacked(w2)


@pytest.mark.gpu
def test_asserted_strides_of_size_one_dimensions():
    # contiguous tensors all the same, as a dimension of size 1 has any stride
    w13, s13 = _weights(np.random.default_rng(11), (4, 64), 128, cuda)
    a = cuda(rand_act(6, (16, 128)))
    ids = cuda(torch.arange(16).remainder(4).view(16, 1))
    tw = torch.ones((16, 1), device="cuda").as_strided((16, 1), (1, 5))
    assert tw.is_contiguous() and tw.stride(1) == 5
    srt, exp_, npp = mx.make_routing_device(ids, 4, 16)
    C = torch.zeros((16, 1, 64), dtype=torch.bfloat16, device="cuda")
    one, ones = torch.ones(1, device="cuda"), torch.ones(4, device="cuda")
    with pytest.raises(AssertionError):
        mx.fused_moe_mxfp4(a, w13, C, one, ones, None, s13, tw, ids, srt, exp_, npp, True, 1,
                           False, False, {"BLOCK_SIZE_M": 16}, C.dtype)


@pytest.mark.gpu
def test_failing_pointer_read_is_an_ordinary_exception():
    # the read throws after the call has been found plain (as a copy-on-write
    # storage does that cannot be copied): an exception as in the general path,
    # with the interpreter lock held, and the next call runs
    rng = np.random.default_rng(13)
    w, s = _weights(rng, (64,), 256, cuda)
    x = cuda(rand_act(8, (4, 256)))
    bad = x.clone()
    torch._C._set_throw_on_mutable_data_ptr(bad)
    logits = torch.randn((4, 8), device="cuda")
    bad_logits = logits.clone()
    torch._C._set_throw_on_mutable_data_ptr(bad_logits)
    for _ in range(2):
        with pytest.raises(RuntimeError):
            _lib.host().linear(bad, w, s, None, None)
        with pytest.raises(RuntimeError):
            _lib.host().quant(bad, 0)
        with pytest.raises(RuntimeError):
            _lib.host().route_topk(bad_logits, 2, True, False)
    with pytest.raises(RuntimeError):
        mx.linear_mxfp4_soft(bad, w, s)
    assert torch.isfinite(mx.linear_mxfp4_soft(x, w, s)).all()


@pytest.mark.gpu
def test_only_prepacked_weights_pass_as_a_copy():
    # an object with the same attributes is refused, as by the general path
    rng = np.random.default_rng(17)
    w13, s13 = _weights(rng, (4, 256), 128, cuda)
    w2, s2 = _weights(rng, (4, 128), 128, cuda)
    x = cuda(rand_act(9, (20, 128)))
    tw, ids = mx.route_topk(torch.randn((20, 4), device="cuda"), 2)

    def like(pre):
        return SimpleNamespace(**{f: getattr(pre, f) for f in pre.__dataclass_fields__})

    pre, pre13, pre2 = (mx.prepack_w4a16(*p) for p in ((w13[0], s13[0]), (w13, s13), (w2, s2)))
    assert _lib.host().linear(x, w13[0], s13[0], None, pre) is not None
    assert _lib.host().linear(x, w13[0], s13[0], None, like(pre)) is None
    with pytest.raises(TypeError):
        mx.linear_mxfp4_soft(x, w13[0], s13[0], prepacked=like(pre))
    mx.moe_layer(x, w13, s13, w2, s2, tw, ids, prepacked13=pre13, prepacked2=pre2)
    for a, b in ((like(pre13), pre2), (pre13, like(pre2))):
        with pytest.raises(TypeError):
            mx.moe_layer(x, w13, s13, w2, s2, tw, ids, prepacked13=a, prepacked2=b)

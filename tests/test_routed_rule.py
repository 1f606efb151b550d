"""The rule that sends a routed GEMM to the register-weight kernel, on a chip
of 256 CUs: calls that are slower there stay on the decode kernels and the
prefill tiles, those that are faster go, and the tile width and the LDS limits
are where the kernel file says."""

from __future__ import annotations

import pytest

from _helpers import dr_columns


def _columns(op, e, k, n, avg):
    """op: soft / layer / pre (layer on prepacked weights) / a caller's blocks."""
    routes = round(avg * e)
    if op == "soft":
        block_m = (16 if avg <= 1.5 or (k >= 2048 and avg <= 4) else
                   32 if avg <= (30 if k >= 2048 else 32) else
                   64 if avg <= 56 or k < 2048 else 128)
    elif op == "layer":
        block_m = 16 if avg <= 6 else 32 if avg <= 28 else 64 if avg <= 56 else 128
    elif op == "pre":
        block_m = 16 if avg <= 1.5 else 32 if avg <= 32 else 64
    else:
        block_m = op
    return dr_columns(routes, e, n, k, block_m=block_m, silu=op in ("layer", "pre"),
                      prepacked=op == "pre", rows=32 if block_m == 32 and op == 32 else 64)


# (op, experts, K, N, routes per expert): 4 to 20% slower in the register
# kernel with uniform routing (with skewed routing up to 1.8 times)
@pytest.mark.parametrize("op,e,k,n,avg", [
    ("soft", 32, 2048, 1536, 3), ("soft", 32, 2048, 1536, 4), ("soft", 32, 4096, 1024, 3),
    ("soft", 64, 4096, 1024, 2), ("soft", 8, 768, 2048, 128), ("soft", 8, 768, 2048, 192),
    ("layer", 32, 2048, 768, 3), ("layer", 32, 2048, 768, 6), ("layer", 16, 2048, 768, 6),
    ("layer", 16, 1024, 512, 6), ("layer", 128, 1024, 512, 96),
    ("pre", 32, 2048, 1408, 64), ("pre", 32, 2048, 1408, 96), ("pre", 64, 2048, 768, 64),
    ("pre", 64, 2048, 768, 96), ("pre", 32, 2048, 768, 16), ("pre", 64, 2048, 768, 16),
    ("pre", 128, 2048, 768, 40), (32, 64, 768, 2048, 64), (32, 16, 768, 2048, 128),
    (32, 8, 1024, 4096, 128), (64, 8, 768, 2048, 128), (64, 16, 2048, 1536, 256),
    (64, 8, 1024, 4096, 128), (128, 64, 768, 2048, 64), (128, 64, 768, 2048, 96),
    (128, 32, 1024, 4096, 96), (128, 64, 1024, 4096, 96), (128, 128, 2048, 1536, 80),
])
def test_slower_calls_stay(op, e, k, n, avg):
    assert _columns(op, e, k, n, avg) == 0


@pytest.mark.parametrize("op,e,k,n,avg,columns", [
    ("soft", 128, 2048, 1536, 32, 256), ("soft", 32, 4096, 1024, 6, 128),
    ("soft", 8, 4096, 1024, 64, 128), ("soft", 64, 2048, 1536, 3, 128),
    ("layer", 128, 2048, 768, 3, 256), ("layer", 64, 2048, 768, 3, 128),
    ("layer", 16, 2048, 768, 8, 128), ("pre", 128, 2048, 768, 32, 256),
    ("pre", 16, 2048, 768, 64, 128), ("pre", 32, 4096, 1024, 4, 128),
    (32, 128, 2048, 1536, 32, 256), (32, 8, 768, 2048, 64, 128), (64, 8, 4096, 1024, 192, 128),
    (64, 128, 2048, 1536, 8, 256), (128, 32, 2048, 1536, 96, 128),
    (128, 16, 2048, 1536, 192, 128), (128, 128, 4096, 1024, 80, 256),
    # tile width: 384, 384, 417, 480 and 497 tiles of 256 columns
    (64, 64, 2048, 1536, 48, 128), (64, 32, 2048, 1536, 96, 128), (32, 64, 2048, 1536, 24, 256),
    (64, 32, 2048, 1536, 128, 256), (64, 64, 4096, 1024, 80, 256),
])
def test_faster_calls_go(op, e, k, n, avg, columns):
    assert _columns(op, e, k, n, avg) == columns


def test_lds_limits():
    # 80 KB: two activation stages and the tile's scale rows
    for k, columns in ((6016, 256), (6144, 128), (12032, 128), (12160, 0)):
        assert dr_columns(128 * 30, 128, 1000, k, block_m=64) == columns

"""Attention at sizes on both sides of the choices between its kernels: at
d = 128 the 64-query and the 32-query kernels (whole key tiles, one workgroup
per query tile or per pair of them, odd tile counts, a part-filled last tile,
few key tiles, strided heads, causal offsets), and the few-query kernel.

Bounds and reference as in ``test_attn_few_queries_gpu``.
"""

from __future__ import annotations

import pytest
import torch
from test_attn_few_queries_gpu import _case, _check

from catopt_amd import _lib as L

pytestmark = pytest.mark.gpu
Q32, Q64, Q64_PAIRED, FEW = range(4)  # catopt_attn_route


def _route(q, k, mode=L.MASK_NONE):
    B, H, Tq, d = q.shape
    return L.load().catopt_hip_attn_route(B, H, Tq, k.shape[2], d, mode)


SHAPES = [
    (1, 12, 1024, 1024, Q32),          # 48 query tiles of 256
    (1, 75, 700, 768, Q64),            # 225: one tile to a workgroup
    (2, 32, 1000, 1024, Q64),          # 256
    (1, 105, 1024, 1024, Q64_PAIRED),  # 420: in pairs
    (1, 100, 1200, 640, Q64),          # 500, an odd number per head
    (1, 160, 512, 512, Q32),           # two tiles per head
    # fewer key tiles than the loop's three stages, and barely more; the last
    # tile (of a pair, where they go in pairs) with few valid queries
    (1, 80, 520, 64, Q64), (1, 80, 700, 128, Q64), (5, 16, 515, 192, Q64), (1, 150, 600, 320, Q64),
    (1, 95, 1000, 64, Q64_PAIRED), (1, 96, 770, 128, Q64_PAIRED), (3, 32, 800, 192, Q64_PAIRED),
    (1, 90, 769, 320, Q64_PAIRED),
]


@pytest.mark.parametrize("B,H,Tq,Tk,route", SHAPES)
def test_routes(B, H, Tq, Tk, route):
    q, k, v = _case(B, H, Tq, Tk, 128, seed=Tq)
    assert _route(q, k) == route and _route(q, k, L.MASK_CAUSAL) == route
    _check(q, k, v, 128 ** -0.5)
    _check(q, k, v, 128 ** -0.5, causal=True, causal_off=Tk - Tq)
    _check(q, k, v, 128 ** -0.5, causal=True, causal_off=-70)


@pytest.mark.parametrize("B,H,Tq,Tk,route", [(5, 17, 700, 192, Q64), (3, 31, 1000, 320, Q64_PAIRED)])
def test_64_queries_of_strided_heads(B, H, Tq, Tk, route):
    """(B, T, H, d) storage viewed as (B, H, T, d): row stride H d."""
    q, k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in _case(B, H, Tq, Tk, 128, seed=Tk))
    assert _route(q, k) == route
    _check(q, k, v, 0.09)
    _check(q, k, v, 0.09, causal=True, causal_off=-40)


# both sides of the few-query kernel's rule: many heads over short keys, two
# ranges of keys, planes
@pytest.mark.parametrize("H,Tq,Tk,d,route", [
    (2100, 17, 64, 64, Q32), (2048, 17, 64, 64, FEW), (2100, 3, 65, 64, FEW), (256, 17, 300, 128, Q32),
    (256, 16, 300, 128, FEW), (1100, 20, 100, 128, Q32), (1000, 20, 100, 128, FEW)])
def test_few_queries_routes(H, Tq, Tk, d, route):
    q, k, v = _case(1, H, Tq, Tk, d, seed=H + Tq)
    assert _route(q, k) == route
    _check(q, k, v, d ** -0.5)
    _check(q, k, v, d ** -0.5, causal=True, causal_off=Tk - Tq)


@pytest.mark.parametrize("H,Tq,d,route", [(600, 9, 128, Q32), (600, 8, 128, FEW), (700, 17, 64, Q32), (700, 16, 64, FEW)])
def test_few_queries_routes_with_planes(H, Tq, d, route):
    q, k, v = _case(1, H, Tq, 130, d, seed=Tq)
    assert _route(q, k, L.MASK_BOOL) == route and _route(q, k, L.MASK_BIAS) == route
    g = torch.Generator(device="cuda:0").manual_seed(2)
    _check(q, k, v, 0.1, mask=torch.rand((Tq, 130), generator=g, device="cuda:0") < 0.5)
    _check(q, k, v, 0.1, bias=torch.randn((Tq, 130), generator=g, device="cuda:0"))

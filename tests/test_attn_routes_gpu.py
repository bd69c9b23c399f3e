"""d = 128 attention at sizes on both sides of the choice between the 64-query
and the 32-query kernels: whole key tiles, one workgroup per query tile or
per pair of them, odd tile counts, a part-filled last tile, causal offsets.

Bounds and reference as in ``test_attn_few_queries_gpu``.
"""

from __future__ import annotations

import pytest
from test_attn_few_queries_gpu import _case, _check

pytestmark = pytest.mark.gpu

SHAPES = [
    (1, 12, 1024, 1024),   # 48 query tiles of 256: the 32-query kernel
    (1, 75, 700, 768),     # 225: the 64-query kernel, one tile to a workgroup
    (2, 32, 1000, 1024),   # 256
    (1, 105, 1024, 1024),  # 420: in pairs
    (1, 100, 1200, 640),   # 500, an odd number per head
    (1, 160, 512, 512),    # two tiles per head: the 32-query kernel
]


@pytest.mark.parametrize("B,H,Tq,Tk", SHAPES)
def test_routes(B, H, Tq, Tk):
    q, k, v = _case(B, H, Tq, Tk, 128, seed=Tq)
    _check(q, k, v, 128 ** -0.5)
    _check(q, k, v, 128 ** -0.5, causal=True, causal_off=Tk - Tq)
    _check(q, k, v, 128 ** -0.5, causal=True, causal_off=-70)

"""The SSM scan's automatic schedule at the edges of its T-segments.

One pass or several segments by the number of workgroups, every state width,
both forms of ``a``: whole and part stages, fewer steps than a stage, a last
segment with steps past its last stage, channels that do not fill the last
workgroup.  Against the oracle's serial recurrence in float64 at the fp32
gate (1e-5 of the largest output).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from catopt_amd import _lib as L
from catopt_amd import kernels as K

pytestmark = pytest.mark.gpu
TOL_F32 = 1e-5

CASES = [  # B, T, D
    (1, 5, 64), (1, 16, 130), (2, 31, 70), (1, 32, 64), (1, 257, 64),
    (3, 300, 100), (1, 1000, 1), (2, 259, 513), (90, 40, 16), (1, 40, 5700),
    # every remainder of the stages over the three register sets: 3, 7 (and 5
    # above) in one pass, 3, 4 and 5 in each of four segments
    (90, 24, 16), (90, 56, 16), (60, 96, 16), (60, 128, 16), (60, 163, 16),
]


@pytest.mark.parametrize("aps", [True, False])
@pytest.mark.parametrize("N", [4, 8, 16, 32, 64])
@pytest.mark.parametrize("B,T,D", CASES)
def test_ssm_auto(B, T, D, N, aps):
    rng = np.random.default_rng(B + T + D + N)
    a = (1 / (1 + np.exp(rng.standard_normal((B, T, D, N) if aps else (B, T, D))))).astype(np.float32)
    bx, c = (rng.standard_normal((B, T, N)).astype(np.float32) for _ in range(2))
    x = rng.standard_normal((B, T, D)).astype(np.float32)
    h0 = rng.standard_normal((B, D, N)).astype(np.float32) if T % 2 else None
    table = oracle.prefix_chunk_table(T)
    wsb = L.load().catopt_hip_ssm_scan_workspace_bytes(B, T, D, N, len(table) - 1, L.SCAN_AUTO)
    wgs = -(-D // (1024 // N)) * B
    assert (wsb > 0) == (wgs < 84 and T >= 32)  # at least two segments of two stages
    t = lambda z: None if z is None else torch.from_numpy(z).cuda()  # noqa: E731
    y, h = K.ssm_scan(t(a), t(bx), t(c), t(x), t(h0), table, return_state=True)
    f = lambda z: None if z is None else z.astype(np.float64)  # noqa: E731
    a64 = f(a) if aps else np.repeat(f(a)[..., None], N, axis=-1)
    ry, rh = oracle.ssm_serial(a64, f(bx), f(c), f(x), f(h0))
    for ref, out in ((ry, y), (rh, h)):
        rep = oracle.verify_equiv(ref, out.cpu().double().numpy(), rtol=TOL_F32)
        assert rep["passed"], rep


@pytest.mark.parametrize("N,B,T,D", [(16, 60, 163, 16), (8, 1, 257, 64), (4, 3, 300, 100), (16, 90, 56, 16)])
def test_ssm_state_updated_in_place(N, B, T, D):
    """h_final in h0's own buffer: the same values as in a buffer of its own."""
    g = torch.Generator(device="cuda:0").manual_seed(N + T)
    r = lambda *s: torch.randn(s, generator=g, device="cuda:0")  # noqa: E731
    a, bx, c, x, h0 = r(B, T, D, N).sigmoid_(), r(B, T, N), r(B, T, N), r(B, T, D), r(B, D, N)
    lib, cs = L.load(), torch.from_numpy(oracle.prefix_chunk_table(T).astype(np.int64)).cuda()
    wsb = lib.catopt_hip_ssm_scan_workspace_bytes(B, T, D, N, len(cs) - 1, L.SCAN_AUTO)
    outs = []
    for in_place in (False, True):
        ws = torch.full((max(wsb, 16) // 4,), float("nan"), device="cuda:0")
        h, y = h0.clone(), torch.empty_like(x)
        hf = h if in_place else torch.empty_like(h0)
        st = lib.catopt_hip_ssm_scan(B, T, D, N, a.data_ptr(), 1, bx.data_ptr(), c.data_ptr(), x.data_ptr(), h.data_ptr(),
                                     cs.data_ptr(), len(cs) - 1, L.SCAN_AUTO, y.data_ptr(), hf.data_ptr(), ws.data_ptr(),
                                     wsb, torch.cuda.current_stream().cuda_stream)
        assert st == L.OK
        outs.append((y, hf))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    ry, rh = oracle.ssm_serial(*(t.cpu().double().numpy() for t in (a, bx, c, x, h0)))
    for ref, out in zip((ry, rh), outs[1]):
        assert oracle.verify_equiv(ref, out.cpu().double().numpy(), rtol=TOL_F32)["passed"]

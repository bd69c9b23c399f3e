"""bf16 retention with more than eight segments per head (few heads, long T):
segment counts on both sides of eight and at the most, ragged T, small head
dims, decays of 0, 1 and negative, and a workspace that only eight segments fit.

Against the quadratic form in float64 at the repository's bf16 gate, and
against the same call held to eight segments: the two differ in the fp32
rounding of the start states, which can move a state or an output across one
bf16 rounding (2^-8 of its size each, so 2^-7 of the largest output).
"""

from __future__ import annotations

import pytest
import torch

from catopt_amd import _lib as L
from catopt_amd import kernels as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
PIECE = 2 * 128 * 128 * 4  # bytes of a range's two state pieces


def _case(B, H, T, d, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return [(torch.randn((B, H, T, d), generator=g, device=DEV) * d ** -0.25).to(torch.bfloat16) for _ in range(3)]


def _eight(q, k, v, gam, scale):
    """The same call with the workspace of eight segments."""
    B, H, T, d = q.shape
    lib = L.load()
    o = torch.empty_like(v)
    ws = torch.empty(B * H * 8 * PIECE, dtype=torch.uint8, device=DEV)
    st = lib.catopt_hip_retention_fwd(L.BF16, B, H, T, d, 64, q.data_ptr(), k.data_ptr(), v.data_ptr(), gam.data_ptr(),
                                      scale, o.data_ptr(), ws.data_ptr(), ws.numel(),
                                      torch.cuda.current_stream().cuda_stream)
    L.check("catopt_hip_retention_fwd", st)
    return o


def _check(q, k, v, gam, scale):
    out = K.retention(q, k, v, gam, scale).double()
    T = q.shape[2]
    i = torch.arange(T, device=DEV)
    gap = i[:, None] - i[None, :]
    ref = torch.empty_like(out)
    for h in range(q.shape[1]):
        dec = torch.where(gap >= 0, torch.pow(gam[h].double(), gap.clamp(min=0).double()), 0.0)
        s = torch.matmul(q[:, h].double(), k[:, h].double().transpose(-1, -2).contiguous()) * dec
        ref[:, h] = scale * torch.matmul(s, v[:, h].double())
    top = ref.abs().max() + 1e-8
    assert torch.isfinite(out).all()
    assert (out - ref).abs().max() / top <= 2e-2
    assert (out - _eight(q, k, v, gam, scale).double()).abs().max() / top <= 2.0 ** -7


@pytest.mark.parametrize("B,H,T,d", [(1, 1, 2049, 128), (1, 1, 3009, 128), (1, 1, 8192, 128), (2, 2, 4033, 64),
                                     (3, 7, 3073, 128), (1, 14, 4095, 8), (2, 8, 3136, 96), (2, 17, 700, 128)])
def test_shapes(B, H, T, d):
    q, k, v = _case(B, H, T, d, B + H + T + d)
    gam = torch.tensor([1 - 2.0 ** (-4 - h) for h in range(H)], device=DEV)
    nseg = L.load().catopt_hip_retention_workspace_bytes(B, H, T, d, 64) // (B * H * PIECE)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    if cus >= 256:
        assert (nseg > 8) == (T > 3008 and B * H <= cus // 12)
    _check(q, k, v, gam, 0.7)


@pytest.mark.parametrize("gamma", [0.0, 1.0, -0.9, -1.0])
def test_decays(gamma):
    q, k, v = _case(1, 2, 4000, 128, 3)
    _check(q, k, v, torch.tensor([gamma, 0.999], device=DEV), 1.0)

"""fp32 retention at the edges of its chunks and segments: one step, part
chunks, one and many segments per head, head dims on both sides of 64, decays
of 0, 1 and negative, and the call without a workspace.

Against the quadratic form in float64.  Each output is a sum of at most T
terms of d products with an fp32 decay factor: gated at 1e-5 of the largest
output (the repository's fp32 gate).
"""

from __future__ import annotations

import pytest
import torch

from catopt_amd import _lib as L
from catopt_amd import kernels as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(B, H, T, d, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    q, k, v = (torch.randn((B, H, T, d), generator=g, device=DEV) * d ** -0.5 for _ in range(3))
    gam = torch.tensor([1 - 2.0 ** (-1 - h) for h in range(H)], device=DEV)
    return q, k, v, gam


def _reference(q, k, v, gam, scale):
    T = q.shape[2]
    i = torch.arange(T, device=DEV)
    gap = (i[:, None] - i[None, :])
    dec = torch.where(gap >= 0, torch.pow(gam.double()[:, None, None], gap.clamp(min=0).double()), 0.0)
    s = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) * dec
    return scale * torch.matmul(s, v.double())


def _gate(out, ref):
    err = (out.double() - ref).abs().max() / (ref.abs().max() + 1e-8)
    assert err <= 1e-5 and torch.isfinite(out).all(), float(err)


@pytest.mark.parametrize("d", [4, 64, 68, 128])
@pytest.mark.parametrize("B,H,T", [(1, 1, 1), (1, 2, 31), (2, 3, 33), (1, 5, 64), (2, 2, 127), (1, 4, 1000), (3, 7, 515),
                                   (20, 15, 70)])
def test_shapes(B, H, T, d):
    q, k, v, gam = _case(B, H, T, d, B + H + T + d)
    _gate(K.retention(q, k, v, gam, 0.7), _reference(q, k, v, gam, 0.7))


@pytest.mark.parametrize("gamma", [0.0, 1.0, -0.9, -1.0])
def test_decays(gamma):
    q, k, v, _ = _case(1, 2, 400, 96, 1)
    gam = torch.tensor([gamma, 0.97], device=DEV)
    _gate(K.retention(q, k, v, gam), _reference(q, k, v, gam, 1.0))


def test_without_workspace():
    q, k, v, gam = _case(1, 2, 700, 128, 2)
    lib = L.load()
    assert lib.catopt_hip_retention_f32_workspace_bytes(1, 2, 700, 128) > 0
    o = torch.empty_like(v)
    st = lib.catopt_hip_retention_fwd(L.F32, 1, 2, 700, 128, 64, q.data_ptr(), k.data_ptr(), v.data_ptr(),
                                      gam.data_ptr(), 1.0, o.data_ptr(), None, 0,
                                      torch.cuda.current_stream().cuda_stream)
    assert st == L.OK
    _gate(o, _reference(q, k, v, gam, 1.0))

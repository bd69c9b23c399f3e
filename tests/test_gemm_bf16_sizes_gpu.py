"""bf16 GEMMs off the large-tile sizes, against float64: few rows, every
epilogue, tile and K remainders, strided rows with poisoned padding, batches.

Bound per element: the bf16 rounding of the result (2^-8 of its magnitude
covers the half ulp and the fp32 value's own distance), plus the fp32
summation error of K products, at most (K + 16) 2^-24 of the sum of their
magnitudes in any order.  Paired epilogues carry both projections' sums
through silu / sigmoid (slope at most 1.1), whose exp and reciprocal add a
few fp32 ulps.
"""

from __future__ import annotations

import pytest
import torch

from catopt_amd import _lib as L
from catopt_amd import kernels as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16


def _rows(g, r, k, pad):
    """(r, k) bf16 rows of stride k + pad, the padding full of Inf and NaN."""
    t = torch.full((r, k + pad), float("inf"), dtype=BF, device=DEV)
    t[:, k + pad // 2:] = float("nan")
    t[:, :k] = torch.randn((r, k), generator=g, device=DEV).to(BF)
    return t[:, :k]


def _reference(x, w, epi, bias, bias2):
    x64, w64 = x.double(), w.double()
    s, mag = x64 @ w64.T, x64.abs() @ w64.abs().T
    e = (x.shape[1] + 16) * 2.0 ** -24 * mag
    if epi in (L.EPI_SILU_MUL, L.EPI_GLU):
        n = w.shape[0] // 2
        a, b, ea, eb = s[:, :n], s[:, n:], e[:, :n], e[:, n:]
        if epi == L.EPI_SILU_MUL:
            r, e = a * torch.sigmoid(a) * b, 1.1 * ea * b.abs() + eb * a.abs()
        else:
            r, e = a * torch.sigmoid(b), ea + 0.25 * eb * a.abs()
        return r, e + 2.0 ** -20 * r.abs()
    for t in (bias, bias2):
        if t is not None:
            s = s + t.double()
    return s, e + 2.0 ** -22 * (s.abs())


def _check(y, ref, err):
    bound = err + 2.0 ** -8 * ref.abs() + 1e-30
    bad = ((y.double() - ref).abs() > bound) | ~torch.isfinite(y.double())
    assert not bad.any(), (int(bad.sum()), float(((y.double() - ref).abs() / bound).nan_to_num(9e9).max()))


SIZES = [(1, 16, 8), (1, 5, 64), (3, 40, 72), (15, 33, 520), (16, 256, 1024), (17, 1003, 1032), (32, 64, 2048),
         (33, 48, 1096), (48, 17, 64), (49, 130, 4104), (64, 512, 992)]


@pytest.mark.parametrize("epi", [L.EPI_NONE, L.EPI_BIAS, L.EPI_BIAS_ADD2, L.EPI_SILU_MUL, L.EPI_GLU])
@pytest.mark.parametrize("M,N,Kd", SIZES)
@pytest.mark.parametrize("pad", [0, 16])
def test_linear_sizes(M, N, Kd, epi, pad):
    g = torch.Generator(device=DEV).manual_seed(M * 7 + N + Kd + epi)
    paired = epi in (L.EPI_SILU_MUL, L.EPI_GLU)
    x, w = _rows(g, M, Kd, pad), _rows(g, N * (2 if paired else 1), Kd, pad)
    bias = torch.randn(N, generator=g, device=DEV).to(BF) if epi in (L.EPI_BIAS, L.EPI_BIAS_ADD2) else None
    bias2 = torch.randn(N, generator=g, device=DEV).to(BF) if epi == L.EPI_BIAS_ADD2 else None
    y = K.linear(x, w, bias, bias2, epilogue=epi)
    assert y.shape == (M, N)
    _check(y, *_reference(x, w, epi, bias, bias2))


@pytest.mark.parametrize("nb,M,N,Kd", [(3, 1, 40, 64), (5, 20, 96, 136), (2, 64, 33, 256)])
def test_batched_few_rows(nb, M, N, Kd):
    g = torch.Generator(device=DEV).manual_seed(nb + M)
    a = torch.randn((nb, M, Kd), generator=g, device=DEV).to(BF)
    b = torch.randn((nb, N, Kd), generator=g, device=DEV).to(BF)
    y = K.matmul(a, b.transpose(-1, -2))
    for i in range(nb):
        _check(y[i], *_reference(a[i], b[i], L.EPI_NONE, None, None))

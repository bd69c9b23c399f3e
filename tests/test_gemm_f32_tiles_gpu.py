"""fp32 products on the tile kernel, against float64: tile and stage
remainders, every operand layout, biases, batches with a shared operand, and
rows whose padding holds Inf and NaN.

Bound per element: K products summed in fp32 in any order, at most
(K + 16) 2^-24 of the sum of their magnitudes.
"""

from __future__ import annotations

import pytest
import torch

from catopt_amd import kernels as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _padded(g, *shape, pad):
    t = torch.full((*shape[:-1], shape[-1] + pad), float("inf"), device=DEV)
    t[..., shape[-1] + pad // 2:] = float("nan")
    t[..., :shape[-1]] = torch.randn(shape, generator=g, device=DEV)
    return t[..., :shape[-1]]


def _check(y, a, b, extra=None):
    ref = torch.matmul(a.double(), b.double())
    bound = (a.shape[-1] + 16) * 2.0 ** -24 * torch.matmul(a.double().abs(), b.double().abs())
    if extra is not None:
        ref = ref + extra.double()
        bound = bound + 2.0 ** -22 * (ref.abs() + extra.double().abs())
    bad = ((y.double() - ref).abs() > bound + 1e-35) | ~torch.isfinite(y)
    assert not bad.any(), int(bad.sum())


@pytest.mark.parametrize("M,N,Kd", [(1025, 64, 4), (1100, 65, 36), (4096, 512, 512), (2049, 130, 100), (1024, 1027, 68),
                                    (5000, 1, 32)])
@pytest.mark.parametrize("nbias", [0, 1, 2])
def test_linear(M, N, Kd, nbias):
    g = torch.Generator(device=DEV).manual_seed(M + N + Kd)
    x, w = _padded(g, M, Kd, pad=8), _padded(g, N, Kd, pad=4)
    bs = [torch.randn(N, generator=g, device=DEV) for _ in range(nbias)]
    y = K.linear(x, w, *bs)
    _check(y, x, w.T, sum(bs) if bs else None)


@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("nb,M,N,Kd", [(1, 64, 64, 32), (1, 4, 4, 1), (3, 68, 132, 31), (2, 63, 64, 33), (1, 200, 100, 257),
                                       (5, 8, 300, 96), (1, 65, 130, 64), (2, 1, 7, 40)])
def test_matmul_layouts(nb, M, N, Kd, ta, tb):
    g = torch.Generator(device=DEV).manual_seed(nb + M + N + Kd)
    a = _padded(g, nb, Kd, M, pad=4).transpose(1, 2) if ta else _padded(g, nb, M, Kd, pad=4)
    b = _padded(g, nb, N, Kd, pad=8).transpose(1, 2) if tb else _padded(g, nb, Kd, N, pad=8)
    _check(K.matmul(a, b), a, b)


def test_matmul_shared_operand():
    g = torch.Generator(device=DEV).manual_seed(0)
    a, b = torch.randn((6, 96, 128), generator=g, device=DEV), torch.randn((128, 72), generator=g, device=DEV)
    _check(K.matmul(a, b), a, b.expand(6, 128, 72))

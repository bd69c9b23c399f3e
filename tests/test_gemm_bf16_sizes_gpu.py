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


ROWS, M128, M64, LARGE = 1, 2, 3, 4  # catopt_gemm_route


def _route(M, N, Kd, epi, batch=1):
    """(route, tiles done whole, tiles split, K ranges) on this device, with a workspace."""
    plan = L.i64_array([0, 0, 0])
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    return (L.load().catopt_hip_gemm_route(L.BF16, batch, M, N, Kd, epi, cus, 1 << 40, plan), *plan)


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


# the middle tiles: one row past the few-row kernels, tile edges either side,
# whole tiles only, every tile's K in ranges (with a K tail), odd N
MID = [(65, 256, 4096), (64, 1024, 4104), (128, 4096, 1032), (129, 130, 2056), (200, 1003, 2048), (333, 640, 5000),
       (257, 4096, 520), (400, 11008, 72), (1000, 2752, 264), (300, 11010, 1024)]


@pytest.mark.parametrize("epi", [L.EPI_NONE, L.EPI_BIAS, L.EPI_BIAS_ADD2, L.EPI_SILU_MUL, L.EPI_GLU])
@pytest.mark.parametrize("M,N,Kd", MID)
def test_linear_middle_sizes(M, N, Kd, epi):
    test_linear_sizes(M, N, Kd, epi, 16 if M % 2 else 0)


# Whole rounds of tiles and K ranges for those left over, ragged M and N and K
# tails: one and two whole rounds, 2 to 83 tiles split into 2 to 32 ranges.
MIXED = [(333, 11008, 4096, L.EPI_SILU_MUL), (300, 11008, 2056, L.EPI_GLU), (395, 8456, 4104, L.EPI_SILU_MUL),
         (700, 11008, 4104, L.EPI_NONE), (700, 11003, 2056, L.EPI_BIAS_ADD2), (1000, 8456, 4104, L.EPI_GLU),
         (1500, 11008, 2056, L.EPI_BIAS), (2050, 4355, 4104, L.EPI_SILU_MUL)]


@pytest.mark.parametrize("M,N,Kd,epi", MIXED)
def test_linear_whole_rounds_and_split_tiles(M, N, Kd, epi):
    route, whole, split, ranges = _route(M, N, Kd, epi)
    assert route in (M128, M64) and whole > 0 and split > 0 and ranges > 1
    test_linear_sizes(M, N, Kd, epi, 0)


# The persistent 256 x 256 tiles: one row of tiles and ten (a whole group of
# eight and a part of one), one to three rounds, ragged M, N and K, stores of
# whole rows (N a multiple of 8) and column by column.
LARGE_SIZES = [(250, 65541, 264), (1003, 33000, 72), (2310, 8201, 72), (2310, 16400, 136), (4160, 8200, 1032)]


@pytest.mark.parametrize("epi", [L.EPI_NONE, L.EPI_BIAS, L.EPI_BIAS_ADD2, L.EPI_SILU_MUL, L.EPI_GLU])
@pytest.mark.parametrize("M,N,Kd", LARGE_SIZES)
def test_linear_large_tiles(M, N, Kd, epi):
    if epi in (L.EPI_SILU_MUL, L.EPI_GLU):
        N = N // 2
    assert _route(M, N, Kd, epi)[0] == LARGE
    test_linear_sizes(M, N, Kd, epi, 16 if M % 2 else 0)


@pytest.mark.parametrize("epi", [L.EPI_BIAS, L.EPI_GLU])
def test_linear_without_workspace_and_with_too_little(epi):
    """The same product from every workspace the entry point may be given."""
    M, N, Kd = 100, 512, 4096
    g = torch.Generator(device=DEV).manual_seed(3)
    x = torch.randn((M, Kd), generator=g, device=DEV).to(BF)
    w = torch.randn((2 * N if epi == L.EPI_GLU else N, Kd), generator=g, device=DEV).to(BF)
    bias = torch.randn(N, generator=g, device=DEV).to(BF) if epi == L.EPI_BIAS else None
    lib = L.load()
    need = lib.catopt_hip_linear_workspace_bytes(L.BF16, M, N, Kd, epi)
    assert need > 0
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    ref = _reference(x, w, epi, bias, None)
    for p, n in ((None, 0), (ws.data_ptr(), need - 1), (ws.data_ptr(), need)):
        y = torch.empty((M, N), dtype=BF, device=DEV)
        st = lib.catopt_hip_linear_ws(L.BF16, M, N, Kd, x.data_ptr(), Kd, w.data_ptr(), Kd,
                                      None if bias is None else bias.data_ptr(), None, epi, y.data_ptr(), N, p, n,
                                      torch.cuda.current_stream().cuda_stream)
        assert st == L.OK
        _check(y, *ref)


def test_no_workspace_for_the_general_kernel():
    q = L.load().catopt_hip_linear_workspace_bytes
    assert q(L.BF16, 100, 512, 4096, L.EPI_NONE) > 0 and q(L.BF16, 100, 512, 4097, L.EPI_NONE) == 0


@pytest.mark.parametrize("nb,M,N,Kd", [(3, 1, 40, 64), (5, 20, 96, 136), (2, 64, 33, 256)])
def test_batched_few_rows(nb, M, N, Kd, route=ROWS):
    assert _route(M, N, Kd, L.EPI_NONE, nb)[0] == route
    g = torch.Generator(device=DEV).manual_seed(nb + M)
    a = torch.randn((nb, M, Kd), generator=g, device=DEV).to(BF)
    b = torch.randn((nb, N, Kd), generator=g, device=DEV).to(BF)
    y = K.matmul(a, b.transpose(-1, -2))
    for i in range(nb):
        _check(y[i], *_reference(a[i], b[i], L.EPI_NONE, None, None))


# batches that the large tiles run: few rows over many workgroups, rows past the
# few-row kernel (ragged, a K tail, C rows not 16-byte aligned)
@pytest.mark.parametrize("nb,M,N,Kd", [(200, 33, 1030, 136), (40, 64, 4096, 72), (3, 70, 300, 264), (2, 513, 259, 72)])
def test_batched_large_tiles(nb, M, N, Kd):
    test_batched_few_rows(nb, M, N, Kd, LARGE)


def test_linear_more_weight_rows_than_the_few_row_grid_takes():
    # 2^32 work-items at one workgroup of 1024 per 16 rows: other tiles run it
    N, Kd = 67_108_880, 8
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn((1, Kd), generator=g, device=DEV).to(BF)
    w = torch.empty((N, Kd), dtype=BF, device=DEV)
    w.normal_(generator=g)
    y = K.linear(x, w)
    _check(y, *_reference(x, w, L.EPI_NONE, None, None))

"""Which GEMM kernel a product runs on (CPU only: the route query launches nothing)."""

from __future__ import annotations

import pytest

from catopt_amd import _lib as L

BF16, F32 = L.BF16, L.F32
CUS = 256
GENERAL, ROWS, M128, M64, LARGE, F32_ROWS, F32_TILE = range(7)


def route(dt, M, N, K, epi=L.EPI_NONE, batch=1, ws=1 << 40, n_cu=CUS):
    plan = L.i64_array([-1, -1, -1])
    r = L.load().catopt_hip_gemm_route(dt, batch, M, N, K, epi, n_cu, ws, plan)
    return r, tuple(plan)


# One workgroup per 16 weight rows (1024 or 512 work-items) or per tile (512,
# 256): from 2^32 work-items in a grid dimension on the launch is an error, and
# wider tiles or the persistent kernel, whose grid is the CU count, take over.
@pytest.mark.parametrize("M,N,epi,batch", [
    (1, 67_108_880, L.EPI_NONE, 1), (16, 67_108_880, L.EPI_SILU_MUL, 1), (40, 134_217_760, L.EPI_NONE, 3),
    (1, 80_000_000, L.EPI_NONE, 4), (100, (1 << 30) - 1, L.EPI_GLU, 1), (200, 420_000_000, L.EPI_GLU, 1),
    (65, 1_000_000_000, L.EPI_NONE, 1)])
def test_bf16_grids_stay_within_a_launch(M, N, epi, batch):
    r, (whole, split, ranges) = route(BF16, M, N, 8, epi, batch)
    threads = {ROWS: 1024 if M <= 32 else 512, M128: 512, M64: 256, LARGE: 0}[r]
    groups = -(-N // 16) if r == ROWS else whole + split * ranges
    assert groups * threads < 1 << 32


def test_f32_grids_stay_within_a_launch():
    # 2 x 2^23 tiles of 256 work-items: the general kernel, with a grid of two dimensions
    assert route(F32, 65, 1 << 29, 4)[0] == GENERAL
    assert route(F32, 65, (1 << 29) - 64, 4)[0] == F32_TILE


def test_bad_arguments():
    lib = L.load()
    for a in ((BF16, 0, 1, 1, 8, 0), (BF16, 1, 0, 1, 8, 0), (BF16, 1, 1, 1, 8, 9), (7, 1, 1, 1, 8, 0)):
        assert lib.catopt_hip_gemm_route(*a, CUS, 0, None) == -1

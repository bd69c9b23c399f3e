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


# Products that some other kernel runs at least 1.4 times as fast as the
# few-rows kernel or (the last three) the middle tiles do.
@pytest.mark.parametrize("M,N,K,epi,batch,routes", [
    (64, 131072, 4096, L.EPI_NONE, 1, {M128, M64, LARGE}), (33, 131072, 512, L.EPI_NONE, 1, {M128, M64, LARGE}),
    (16, 131072, 512, L.EPI_NONE, 1, {M128, M64, LARGE}), (64, 65536, 4096, L.EPI_SILU_MUL, 1, {M128, M64, LARGE}),
    (64, 2048, 128, L.EPI_NONE, 512, {LARGE}), (17, 1024, 1024, L.EPI_NONE, 256, {LARGE}),
    (64, 4096, 4096, L.EPI_NONE, 32, {LARGE}), (256, 131072, 64, L.EPI_NONE, 1, {LARGE}),
    (200, 131072, 512, L.EPI_NONE, 1, {LARGE}), (1000, 65536, 64, L.EPI_NONE, 1, {LARGE})])
def test_bf16_few_rows_and_short_k(M, N, K, epi, batch, routes):
    for ws in (0, 1 << 40):
        assert route(BF16, M, N, K, epi, batch, ws)[0] in routes


@pytest.mark.parametrize("M", [1, 8, 16, 17, 40, 64, 65, 200, 333, 1000, 3000])
@pytest.mark.parametrize("N,K", [(256, 4096), (1024, 1024), (4096, 11008), (131072, 64), (65536, 4096)])
@pytest.mark.parametrize("epi", [L.EPI_NONE, L.EPI_SILU_MUL])
def test_no_workspace_is_the_plan_of_a_call_that_asks_for_none(M, N, K, epi):
    """A plan that splits no tile asks for no workspace: the launch that follows has none and must plan the same."""
    r, plan = route(BF16, M, N, K, epi)
    if plan[1] == 0:
        assert route(BF16, M, N, K, epi, ws=0) == (r, plan)


def test_f32_grids_stay_within_a_launch():
    # 2 x 2^23 tiles of 256 work-items: the general kernel, with a grid of two dimensions
    assert route(F32, 65, 1 << 29, 4)[0] == GENERAL
    assert route(F32, 65, (1 << 29) - 64, 4)[0] == F32_TILE


def test_bad_arguments():
    lib = L.load()
    for a in ((BF16, 0, 1, 1, 8, 0), (BF16, 1, 0, 1, 8, 0), (BF16, 1, 1, 1, 8, 9), (7, 1, 1, 1, 8, 0)):
        assert lib.catopt_hip_gemm_route(*a, CUS, 0, None) == -1

"""Which attention kernel a call runs on (CPU only: the route query launches nothing)."""

from __future__ import annotations

import pytest

from catopt_amd import _lib as L

Q32, Q64, Q64_PAIRED, FEW = range(4)


def route(heads, Tq, Tk, d, mode=L.MASK_NONE):
    return L.load().catopt_hip_attn_route(1, heads, Tq, Tk, d, mode)


# the 32-query kernel is 1.05 to 1.5 times as fast at the first of each pair
@pytest.mark.parametrize("slow,fast", [
    ((4096, 1, 64, 64), (2048, 1, 64, 64)), ((4096, 32, 128, 64), (4096, 16, 128, 64)),
    ((8192, 5, 1, 64), (8192, 5, 65, 64)), ((256, 32, 1000, 128), (256, 16, 1000, 128)),
    ((2048, 32, 100, 128), (2048, 32, 200, 128)), ((4096, 17, 30, 128), (1000, 17, 30, 128)),
    ((2048, 12, 250, 128, L.MASK_BOOL), (2048, 8, 250, 128, L.MASK_BOOL)),
    ((512, 32, 500, 128, L.MASK_BIAS), (512, 32, 500, 128, L.MASK_CAUSAL))])
def test_few_queries_on_the_faster_kernel(slow, fast):
    assert route(*slow) == Q32 and route(*fast) == FEW


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("mode", [L.MASK_NONE, L.MASK_CAUSAL, L.MASK_BOOL, L.MASK_BIAS])
def test_a_call_with_a_workspace_runs_the_kernel_that_reads_it(d, mode):
    lib = L.load()
    for heads in (1, 8, 100, 171, 256, 257, 512, 4096):
        for Tq in (1, 8, 9, 16, 17, 32):
            for Tk in (1, 64, 200, 1000, 16384):
                if lib.catopt_hip_attn_workspace_bytes(1, heads, Tq, Tk, d) > 0:
                    assert route(heads, Tq, Tk, d, mode) == FEW


def test_bad_arguments():
    lib = L.load()
    for a in ((0, 1, 1, 1, 64, 0), (1, 1, 1, 1, 96, 0), (1, 1, 0, 1, 64, 0), (1, 1, 1, 1, 64, 9)):
        assert lib.catopt_hip_attn_route(*a) == -1

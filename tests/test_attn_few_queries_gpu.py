"""Attention with few queries (at most 32) over split keys: the edges of key
stages and ranges, every mask mode, strided and padded heads, empty rows and
leaves without keys, and the same call without a workspace.

Against float64 softmax of the same bf16 operands.  A score is a dot product
of d terms in fp32: within (d + 8) 2^-24 of the sum of their magnitudes, and
m with it; l's terms are exponentials of differences of two such scores.  The
numerator's weights and the result are rounded to bf16 (2^-9 of the sum of
magnitudes each; 2^-7 of it is gated).
"""

from __future__ import annotations

import pytest
import torch

from catopt_amd import _lib as L
from catopt_amd import kernels as K

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(B, H, Tq, Tk, d, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    r = lambda *s: torch.randn(s, generator=g, device=DEV).to(torch.bfloat16)  # noqa: E731
    return r(B, H, Tq, d), r(B, H, Tk, d), r(B, H, Tk, d)


def _scores(q, k, scale, causal=False, off=0, mask=None, bias=None):
    s = scale * torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous())
    Tq, Tk = s.shape[-2:]
    if causal:
        i, j = torch.arange(Tq, device=DEV)[:, None], torch.arange(Tk, device=DEV)[None, :]
        s = s.masked_fill(j > i + off, float("-inf"))
    if mask is not None:
        s = s.masked_fill(~mask, float("-inf"))
    return s if bias is None else s + bias.double()


def _check(q, k, v, scale, **kw):
    s = _scores(q, k, scale, kw.get("causal", False), kw.get("causal_off", 0), kw.get("mask"), kw.get("bias"))
    a, m, lv = K.attention(q, k, v, scale, normalize=False, return_ml=True, **kw)
    o = K.attention(q, k, v, scale, **kw)
    o0 = K.attention(q, k, v, scale, empty_rows="zero", **kw)
    rm = s.amax(-1, keepdim=True)
    empty = ~torch.isfinite(rm)
    e = torch.where(empty, 0.0, torch.exp(s - torch.where(empty, 0.0, rm)))
    rl, ra, mag = e.sum(-1, keepdim=True), torch.matmul(e, v.double()), torch.matmul(e, v.double().abs())
    assert torch.equal(torch.isneginf(m), empty)
    ok = ~empty
    mags = scale * torch.matmul(q.double().abs(), k.double().abs().transpose(-1, -2).contiguous())
    es = (q.shape[-1] + 8) * 2.0 ** -24 * mags.amax(-1, keepdim=True) + 2.0 ** -22 * torch.where(empty, 0.0, rm.abs())
    assert ((m.double() - rm).abs() <= es)[ok].all()
    assert ((lv.double() - rl).abs() <= (2 * es.clamp(max=1.0) + 2.0 ** -18) * rl + 1e-30).all()
    assert ((a.double() - ra).abs() <= 2.0 ** -7 * mag + 1e-30).all()
    full = ok.expand_as(o)
    assert ((o.double() - ra / rl)[full].abs() <= (2.0 ** -7 * mag / rl)[full] + 1e-30).all()
    assert torch.isnan(o[~full]).all() and (o0[~full] == 0).all() and torch.equal(o0[full], o[full])


SHAPES = [(1, 1, 1, 1), (1, 2, 1, 33), (2, 3, 5, 64), (1, 5, 32, 127), (1, 4, 7, 128), (2, 12, 1, 1000), (1, 1, 2, 4096),
          (3, 40, 1, 700), (1, 600, 3, 130), (1, 8, 31, 2049),
          (1, 4, 33, 700)]  # one query past the kernel


@pytest.mark.parametrize("d", [64, 128, 40])
@pytest.mark.parametrize("B,H,Tq,Tk", SHAPES)
def test_unmasked_and_causal(B, H, Tq, Tk, d):
    q, k, v = _case(B, H, Tq, Tk, d, seed=Tq + Tk + d)
    _check(q, k, v, d ** -0.5)
    for off in (Tk - Tq, 0, Tk // 2, -2):
        _check(q, k, v, d ** -0.5, causal=True, causal_off=off)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("Tq,Tk", [(1, 63), (6, 513), (32, 3000), (33, 513)])
def test_planes(Tq, Tk, d):
    q, k, v = _case(2, 3, Tq, Tk, d, seed=Tk)
    g = torch.Generator(device=DEV).manual_seed(1)
    mask = torch.rand((Tq, Tk), generator=g, device=DEV) < 0.3
    mask[0] = False  # a row with no key
    _check(q, k, v, 0.1, mask=mask)
    bias = torch.randn((Tq, Tk), generator=g, device=DEV)
    bias[:, ::3] = float("-inf")
    bias[-1, 1::3] = torch.finfo(torch.float32).min
    _check(q, k, v, 0.1, bias=bias)


def test_strided_heads_and_large_scores():
    q, k, v = _case(2, 4, 3, 900, 128, seed=5)
    kt, vt = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (k, v))  # (B, T, H, d) storage
    _check(q, kt, vt, 3.0)


def test_no_keys():
    q, k, v = _case(1, 2, 3, 0, 64)
    a, m, lv = K.attention(q, k, v, 1.0, normalize=False, return_ml=True)
    assert (a == 0).all() and (lv == 0).all() and torch.isneginf(m).all()


def test_without_workspace():
    q, k, v = _case(1, 2, 4, 3000, 128, seed=9)
    lib = L.load()
    assert lib.catopt_hip_attn_workspace_bytes(1, 2, 4, 3000, 128) > 0
    o = torch.empty_like(q)
    st3 = lambda t: L.i64_array(t.stride()[:3])  # noqa: E731
    st = lib.catopt_hip_attn_fwd(L.BF16, 1, 2, 4, 3000, 128, 128, q.data_ptr(), st3(q), k.data_ptr(), st3(k),
                                 v.data_ptr(), st3(v), 0.1, L.MASK_NONE, 0, None, 0, 1, o.data_ptr(), st3(o), None, None,
                                 torch.cuda.current_stream().cuda_stream)
    assert st == L.OK
    ref = torch.matmul(torch.softmax(_scores(q, k, 0.1), -1), v.double())
    assert ((o.double() - ref).abs() <= 2.0 ** -7 * (ref.abs() + 1)).all()

"""The framework's main path as measurable cases, each through a public entry point.

A case is a plain dict; ``kind`` names the path it runs:

* ``chain``     -- a folded weight chain (8 stacked fp32 linears with bias) delivered by the sink: one
                   GEMM with bias per call (``x (rows, d)``);
* ``swiglu``    -- the RMSNorm + SwiGLU MLP block delivered by the sink (bf16): norm, gate/up GEMM with the
                   gate fused, down GEMM, over ``rows`` tokens of width ``D`` and hidden width ``F``;
* ``attention`` -- an online-softmax attention layer delivered by the sink (bf16, causal or not);
* ``decode``    -- one step of streaming attention: a new key block folded into a running carrier with
                   ``om_step_qk`` and read out with ``om_apply_state`` (bf16 operands, fp32 carrier);
* ``retention`` -- decayed linear attention over a whole sequence (``kernels.retention``), bf16 or fp32;
* ``ssm``       -- the selective diagonal SSM scan with read-out (``kernels.ssm_scan``), fp32.
"""

from __future__ import annotations

import functools
import math

import torch

DEV = "cuda:0"
BF16 = torch.bfloat16


def listed() -> list[dict]:
    return [
        # the folded 8-layer chain on a small batch: one launch of about a microsecond of work
        {"name": "chain_r64", "kind": "chain", "rows": 64, "d": 512},
        # the same chain over a training-sized batch of rows (8 sequences of 512)
        {"name": "chain_r4096", "kind": "chain", "rows": 4096, "d": 512},
        # generation: eight sequences, one new token each, through the full-width MLP block
        {"name": "swiglu_r8", "kind": "swiglu", "rows": 8, "D": 4096, "F": 11008},
        # a short prompt of an odd length through the same block
        {"name": "swiglu_r333", "kind": "swiglu", "rows": 333, "D": 4096, "F": 11008},
        # prefill of 8 sequences of 2048 tokens (the MLP configuration's own shape)
        {"name": "swiglu_r16384", "kind": "swiglu", "rows": 16384, "D": 4096, "F": 11008},
        # a small encoder-like layer: head dim 64, every key visible, a ragged length
        {"name": "attention_d64_t999", "kind": "attention", "B": 2, "H": 12, "T": 999, "d": 64, "causal": False},
        # causal prefill at the attention configuration's shape
        {"name": "attention_t4096", "kind": "attention", "B": 4, "H": 32, "T": 4096, "d": 128, "causal": True},
        # decode: one query per head against an 8192-key cache block, four sequences
        {"name": "decode_k8192", "kind": "decode", "B": 4, "H": 32, "Tq": 1, "Tk": 8192, "d": 128},
        # retention at the configuration's shape
        {"name": "retention_t8192", "kind": "retention", "B": 4, "H": 16, "T": 8192, "d": 128, "dtype": "bf16"},
        # fp32 retention of one shorter sequence batch
        {"name": "retention_f32_t2048", "kind": "retention", "B": 2, "H": 16, "T": 2048, "d": 128, "dtype": "f32"},
        # one sequence through an SSM layer: few lanes, so the steps are cut into chunks
        {"name": "ssm_b1_t2048", "kind": "ssm", "B": 1, "T": 2048, "D": 1024, "N": 16},
        # a batch of long sequences: the scan streams a from memory
        {"name": "ssm_b8_t8192", "kind": "ssm", "B": 8, "T": 8192, "D": 2048, "N": 16},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["chain", "swiglu", "swiglu", "attention", "decode", "retention", "ssm"])
    if kind == "chain":
        return {"kind": kind, "rows": _log(rng, 1, 8192), "d": 4 * _log(rng, 32, 256)}
    if kind == "swiglu":
        D, F = rng.choice([(1024, 2752), (2048, 5504), (2048, 8192), (4096, 11008)])
        return {"kind": kind, "rows": _log(rng, 1, 16384), "D": D, "F": F}
    if kind == "attention":
        return {"kind": kind, "B": rng.randint(1, 4), "H": rng.choice([8, 12, 16, 32]), "T": _log(rng, 64, 4096),
                "d": rng.choice([64, 128]), "causal": rng.random() < 0.6}
    if kind == "decode":
        return {"kind": kind, "B": _log(rng, 1, 16), "H": rng.choice([8, 12, 16, 32]),
                "Tq": rng.choice([1, 1, 1, 2, 5]), "Tk": _log(rng, 64, 16384), "d": rng.choice([64, 128])}
    if kind == "retention":
        return {"kind": kind, "B": rng.randint(1, 4), "H": rng.choice([4, 8, 16]), "T": _log(rng, 64, 8192),
                "d": rng.choice([64, 128]), "dtype": rng.choice(["bf16", "bf16", "f32"])}
    return {"kind": kind, "B": rng.randint(1, 8), "T": _log(rng, 64, 8192), "D": rng.choice([256, 512, 1000, 1024, 2048]),
            "N": rng.choice([8, 16])}


# ------------------------------------------------------------------ inputs


def _gen(case: dict, seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed) * 2654435761 % (1 << 31))


def _randn(g, *shape, scale: float = 1.0, dtype=torch.float32) -> torch.Tensor:
    t = torch.randn(shape, device=DEV, generator=g)
    if scale != 1.0:
        t *= scale
    return t.to(dtype)


def _inputs(case: dict, seed: int) -> dict:
    """The tensors of a case, from its seed alone."""
    g, kind = _gen(case, seed), case["kind"]
    if kind == "chain":
        r, d = case["rows"], case["d"]
        lim = 1.0 / math.sqrt(d)
        u = lambda *s: (torch.rand(s, device=DEV, generator=g) * 2 - 1) * lim  # noqa: E731
        t = {"x": _randn(g, r, d)}
        for i in range(1, 9):
            t[f"W{i}"], t[f"b{i}"] = u(d, d), u(d)
        return t
    if kind == "swiglu":
        r, D, F = case["rows"], case["D"], case["F"]
        return {"x": _randn(g, 1, r, D, dtype=BF16), "gamma": (1 + 0.02 * _randn(g, D)).to(BF16),
                "W_gate": _randn(g, F, D, scale=0.02, dtype=BF16), "W_up": _randn(g, F, D, scale=0.02, dtype=BF16),
                "W_down": _randn(g, D, F, scale=0.02, dtype=BF16)}
    if kind == "attention":
        s = (case["B"], case["H"], case["T"], case["d"])
        return {n: _randn(g, *s, dtype=BF16) for n in "qkv"}
    if kind == "decode":
        B, H, Tq, Tk, d = (case[n] for n in ("B", "H", "Tq", "Tk", "d"))
        # the query already carries the score scale, as om_step_qk takes it
        t = {"q": _randn(g, B, H, Tq, d, scale=d ** -0.5, dtype=BF16), "k": _randn(g, B, H, Tk, d, dtype=BF16),
             "v": _randn(g, B, H, Tk, d, dtype=BF16)}
        # a running carrier as 64 earlier keys leave it
        s = _randn(g, B, H, Tq, 64)
        t["m"] = s.amax(-1, keepdim=True)
        e = torch.exp(s - t["m"])
        t["l"] = e.sum(-1, keepdim=True)
        t["a"] = torch.matmul(e, _randn(g, B, H, 64, d))
        return t
    if kind == "retention":
        s = (case["B"], case["H"], case["T"], case["d"])
        dt = BF16 if case["dtype"] == "bf16" else torch.float32
        t = {n: _randn(g, *s, scale=case["d"] ** -0.5, dtype=dt) for n in "qkv"}
        t["gamma"] = torch.tensor([1 - 2.0 ** (-5 - h / 2) for h in range(case["H"])], device=DEV)
        return t
    B, T, D, N = (case[n] for n in ("B", "T", "D", "N"))
    a = torch.randn((B, T, D, N), device=DEV, generator=g)
    a.sigmoid_()  # exp(-softplus(z)) = sigmoid(-z), symmetric in z
    return {"a": a, "bx": _randn(g, B, T, N), "c": _randn(g, B, T, N), "x": _randn(g, B, T, D),
            "h0": _randn(g, B, D, N)}


@functools.lru_cache(maxsize=1)
def _sink():
    from catopt_amd.sink import HipSink

    return HipSink(device=DEV)


def _deliver(form, params: dict):
    from catopt_amd.sink import deliver

    return deliver(form[0], params, _sink()).module


def prepare(case: dict, seed: int) -> dict:
    t, kind = _inputs(case, seed), case["kind"]
    from catopt_amd import forms

    if kind == "chain":
        x = t.pop("x")
        return {"kind": kind, "args": (x,), "mod": _deliver(forms.weight_chain_form(8, case["d"], case["rows"]), t)}
    if kind == "swiglu":
        x = t.pop("x")
        return {"kind": kind, "args": (x,),
                "mod": _deliver(forms.swiglu_block_form((1, case["rows"]), case["D"], case["F"]), t)}
    if kind == "attention":
        B, H, T, d = (case[n] for n in ("B", "H", "T", "d"))
        if case["causal"]:
            form = forms.causal_attention_form(B, H, T, d, mask="cmask")
        else:
            from catopt_amd.ir import IR, Const, Op, TensorType, Var

            q, k, v = (Var(n, TensorType((B, H, T, d))) for n in "qkv")
            s = Op.make("div", Op.make("matmul", q, Op.make("transpose", k, dim0=-2, dim1=-1)), Const(math.sqrt(d)))
            form = (IR(Op.make("om_apply", Op.make("om_elem", s, v)), [q, k, v]), {})
        return {"kind": kind, "args": (t["q"], t["k"], t["v"]), "mod": _deliver(form, {})}
    if kind == "ssm":
        from catopt_amd import kernels as K
        from catopt_amd.executors import prefix_chunk_table

        t["table"] = K.ChunkTable(prefix_chunk_table(case["T"]), case["T"])  # kept, as a planned executor keeps its own
    return {"kind": kind, **t}


# -------------------------------------------------------------------- calls


def run(state: dict):
    kind = state["kind"]
    if kind in ("chain", "swiglu", "attention"):
        return state["mod"](*state["args"])
    if kind == "decode":
        from catopt_amd.executors import om_apply_state, om_step_qk

        m, lv, a = om_step_qk((state["m"], state["l"], state["a"]), state["q"], state["k"], state["v"])
        return {"m": m, "l": lv, "a": a, "out": om_apply_state((m, lv, a))}
    from catopt_amd import kernels as K

    if kind == "retention":
        return K.retention(state["q"], state["k"], state["v"], state["gamma"])
    y, h = K.ssm_scan(state["a"], state["bx"], state["c"], state["x"], state["h0"], state["table"], return_state=True)
    return {"y": y, "h": h}


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "chain":
        r, d = case["rows"], case["d"]
        return {"bytes": 4 * (2 * r * d + d * d + 8 * d), "flops": 2 * r * d * d}
    if kind == "swiglu":
        r, D, F = case["rows"], case["D"], case["F"]
        return {"bytes": 2 * (2 * r * D + D + 3 * D * F), "flops": 6 * r * D * F}
    if kind == "attention":
        B, H, T, d = (case[n] for n in ("B", "H", "T", "d"))
        pairs = T * (T + 1) // 2 if case["causal"] else T * T
        return {"bytes": 8 * B * H * T * d, "flops": 4 * B * H * pairs * d}
    if kind == "decode":
        B, H, Tq, Tk, d = (case[n] for n in ("B", "H", "Tq", "Tk", "d"))
        # q, k, v in bf16; the fp32 carrier in and out, the fp32 read-out
        return {"bytes": B * H * (2 * (Tq + 2 * Tk) * d + 4 * Tq * (3 * d + 4)), "flops": 4 * B * H * Tq * Tk * d}
    if kind == "retention":
        B, H, T, d = (case[n] for n in ("B", "H", "T", "d"))
        C = min(64, T)
        # the chunked form: causal products within a chunk, the state between chunks
        return {"bytes": 4 * B * H * T * d * (2 if case["dtype"] == "bf16" else 4),
                "flops": B * H * T * (4 * (C // 2) * d + 4 * d * d)}
    B, T, D, N = (case[n] for n in ("B", "T", "D", "N"))
    return {"bytes": 4 * B * (T * D * N + 2 * T * N + 2 * T * D + 2 * D * N), "flops": 5 * B * T * D * N}


def tolerance(case: dict) -> dict:
    """About four times the error against ``exact`` that the path shows over the declared ranges."""
    kind = case["kind"]
    if kind == "chain":
        return {"rel": 2e-6, "max": 1.2e-5}
    if kind == "swiglu":
        # two bf16 intermediates (the norm's output and the gated activation) and a bf16 result
        return {"rel": 1.3e-2, "max": 8e-2}
    if kind == "attention":
        # bf16 weights in the value product and a bf16 result; late causal rows are small against the first ones
        return {"rel": 9e-3, "max": 1.7e-1}
    if kind == "decode":
        return {"rel": 9e-3, "max": 5e-2}
    if kind == "retention":
        return {"rel": 1.2e-2, "max": 1.2e-1} if case["dtype"] == "bf16" else {"rel": 2.5e-6, "max": 4e-5}
    return {"rel": 1e-6, "max": 5e-6}


# ---------------------------------------------------------- 64-bit references


def exact(case: dict, seed: int):
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "chain":
        y = t["x"].double()
        for i in range(1, 9):
            y = y @ t[f"W{i}"].double().T + t[f"b{i}"].double()
        return y
    if kind == "swiglu":
        x, gam, wd = t["x"].double(), t["gamma"].double(), t["W_down"].double()
        h = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * gam
        del x
        act = torch.nn.functional.silu(h @ t["W_gate"].double().T)
        act *= h @ t["W_up"].double().T
        return act @ wd.T
    if kind == "attention":
        B, H, T, d = (case[n] for n in ("B", "H", "T", "d"))
        out = torch.empty((B, H, T, d), dtype=torch.float64, device=DEV)
        keep = torch.ones((T, T), dtype=torch.bool, device=DEV).tril() if case["causal"] else None
        for b in range(B):
            for h in range(H):
                s = (t["q"][b, h].double() @ t["k"][b, h].double().T) / math.sqrt(d)
                if keep is not None:
                    s.masked_fill_(~keep, -math.inf)
                out[b, h] = torch.softmax(s, -1) @ t["v"][b, h].double()
        return out
    if kind == "decode":
        s = torch.matmul(t["q"].double(), t["k"].double().transpose(-1, -2).contiguous())
        m2 = s.amax(-1, keepdim=True)
        m = torch.maximum(m2, t["m"].double())
        e = torch.exp(s - m)
        c = torch.exp(t["m"].double() - m)
        lv = t["l"].double() * c + e.sum(-1, keepdim=True)
        a = t["a"].double() * c + torch.matmul(e, t["v"].double())
        return {"m": m, "l": lv, "a": a, "out": a / lv}
    if kind == "retention":
        B, H, T, d = (case[n] for n in ("B", "H", "T", "d"))
        out = torch.empty((B, H, T, d), dtype=torch.float64, device=DEV)
        i = torch.arange(T, device=DEV)
        gap = (i[:, None] - i[None, :]).double()
        for h in range(H):
            dec = torch.where(gap >= 0, torch.pow(t["gamma"][h].double(), gap.clamp(min=0)), 0.0)
            for b in range(B):
                q, k, v = (t[n][b, h].double() for n in "qkv")
                out[b, h] = ((q @ k.T) * dec) @ v
        return out
    a, bx, c, x = (t[n] for n in ("a", "bx", "c", "x"))
    h = t["h0"].double()
    y = torch.empty(x.shape, dtype=torch.float64, device=DEV)
    for s in range(x.shape[1]):
        h = a[:, s].double() * h + x[:, s].double()[..., None] * bx[:, s].double()[:, None, :]
        y[:, s] = (h * c[:, s].double()[:, None, :]).sum(-1)
    return {"y": y, "h": h}

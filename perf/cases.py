"""The calls this framework's speed is judged by: attention forward, training
step and decode, the MLP block and a rendered grammar program, each through
the entry point a program calls, over the sizes those calls take in use.

listed() gives the fixed cases, draw() more of the same ranges. prepare()
makes what a program holds before the call, run() makes the call, exact() is
the same result in 64 bits from plain torch."""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "cs348k-fast-attention-grammar_amd"))

from grammar.attention import bind_flash_attention, flash_attention, flash_attention_decode, flash_attention_fwd  # noqa: E402
from grammar.gemm import mlp_fwd  # noqa: E402
from grammar.hip_module import load_module  # noqa: E402
from grammar.kernel_ast import emit_module  # noqa: E402

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
ELEM = {"fp32": 4, "fp16": 2, "bf16": 2}


def listed() -> list:
    return [
        # one short causal sequence on few heads: the smallest call, where latency counts
        {"name": "attn_short", "kind": "attn", "B": 1, "H": 4, "N": 320, "D": 64, "dtype": "bf16", "causal": True,
         "kt": False, "q_scale": 1.0},
        # the benchmark's attention size: an encoder layer of 16 heads
        {"name": "attn_encoder", "kind": "attn", "B": 4, "H": 16, "N": 1024, "D": 64, "dtype": "fp16",
         "causal": False, "kt": False, "q_scale": 1.0},
        # the prefill of a decoder layer: 32 heads of 128, 4,096 tokens, causal
        {"name": "attn_prefill", "kind": "attn", "B": 2, "H": 32, "N": 4096, "D": 128, "dtype": "bf16",
         "causal": True, "kt": False, "q_scale": 0.5},
        # a sequence length that only the smallest tile divides, K stored transposed as the grammar's programs hold it
        {"name": "attn_ragged_kt", "kind": "attn", "B": 1, "H": 12, "N": 1344, "D": 128, "dtype": "bf16",
         "causal": False, "kt": True, "q_scale": 1.0},
        # the reference's own workload: one fp32 head, called in a loop on bound buffers
        {"name": "attn_fp32_loop", "kind": "attn_fp32", "B": 1, "H": 1, "N": 512, "D": 64, "dtype": "fp32",
         "kt": True},
        # a training step of a small causal model, N a multiple of 128 only
        {"name": "train_small", "kind": "train", "B": 4, "H": 12, "N": 1152, "D": 64, "dtype": "fp16",
         "causal": True},
        # a training step at the prefill case's size
        {"name": "train_long", "kind": "train", "B": 2, "H": 32, "N": 4096, "D": 128, "dtype": "bf16",
         "causal": True},
        # one decode step: one new token against a key/value cache that has room for more
        {"name": "decode_step", "kind": "decode", "B": 8, "H": 16, "Nq": 1, "N": 4128, "D": 128, "dtype": "bf16"},
        # a chunk of queries (speculative tokens, a chunked prompt) against a cached context
        {"name": "decode_chunk", "kind": "decode", "B": 2, "H": 8, "Nq": 40, "N": 3104, "D": 64, "dtype": "fp16"},
        # the benchmark's MLP block: a prefill's 8,192 tokens
        {"name": "mlp_prefill", "kind": "mlp", "M": 8192, "D": 4096, "F": 11008, "dtype": "fp16"},
        # the same block in a decode step: a few tokens, every weight read once
        {"name": "mlp_few_rows", "kind": "mlp", "M": 24, "D": 4096, "F": 11008, "dtype": "bf16"},
        # the reference's MLP block with LayerNorm as a rendered program, at its search's size
        {"name": "program_mlp_ln", "kind": "program_ln", "M": 256, "D": 512, "F": 1024, "tile": 64, "dtype": "fp32"},
    ]


def _log(rng, lo: int, hi: int, step: int = 1) -> int:
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    x = math.exp(rng.uniform(math.log(lo), math.log(hi + step - 1)))
    return max(lo, min(hi, int(x) // step * step))


def draw(rng) -> dict:
    kind = rng.choice(("attn", "attn", "attn_fp32", "train", "train", "decode", "decode", "mlp", "mlp", "program_ln"))
    half = rng.choice(("fp16", "bf16"))
    d = rng.choice((64, 128))
    if kind == "attn":
        return {"kind": kind, "B": _log(rng, 1, 4), "H": _log(rng, 1, 32), "N": _log(rng, 64, 4096, 64), "D": d,
                "dtype": half, "causal": rng.random() < 0.5, "kt": rng.random() < 0.4, "q_scale": 1.0}
    if kind == "attn_fp32":
        return {"kind": kind, "B": _log(rng, 1, 2), "H": _log(rng, 1, 8), "N": _log(rng, 32, 2048, 32), "D": d,
                "dtype": "fp32", "kt": rng.random() < 0.5}
    if kind == "train":
        c = {"kind": kind, "B": _log(rng, 1, 4), "H": _log(rng, 1, 32), "N": _log(rng, 128, 4096, 128), "D": d,
             "dtype": half, "causal": rng.random() < 0.6}
        while work(c)["flops"] > 0.8e12:
            c["N"] = max(128, c["N"] // 256 * 128)
        return c
    if kind == "decode":
        u = rng.random()
        nq = 1 if u < 0.5 else _log(rng, 2, 4) if u < 0.65 else _log(rng, 5, 128)
        c = {"kind": kind, "B": _log(rng, 1, 16), "H": _log(rng, 1, 32), "Nq": nq, "N": _log(rng, 128, 16384, 32),
             "D": d, "dtype": half}
        while work(c)["bytes"] > 5e8:
            c["N"] = max(128, c["N"] // 64 * 32)
        return c
    if kind == "mlp":
        return {"kind": kind, "M": _log(rng, 1, 8192), "D": _log(rng, 512, 4096, 32), "F": _log(rng, 1024, 11008, 32),
                "dtype": half}
    return {"kind": kind, "M": _log(rng, 64, 1024, 64), "D": _log(rng, 128, 1024, 64), "F": _log(rng, 256, 2048, 64),
            "tile": rng.choice((32, 64)), "dtype": "fp32"}


def _inputs(case: dict, seed: int) -> dict:
    """The case's tensors, from the seed alone: activations N(0, 1) in the
    storage type, weights N(0, 1 / fan-in) as initialised layers hold them."""
    g = torch.Generator("cuda").manual_seed(seed)
    dt = DTYPES[case["dtype"]]

    def randn(*shape, scale=1.0):
        return (torch.randn(shape, generator=g, device="cuda") * scale).to(dt)

    kind = case["kind"]
    if kind in ("mlp", "program_ln"):
        M, D, F = case["M"], case["D"], case["F"]
        return {"x": randn(M, D), "w1": randn(D, F, scale=1 / math.sqrt(D)), "w2": randn(F, D, scale=1 / math.sqrt(F))}
    B, H, N, D = case["B"], case["H"], case["N"], case["D"]
    if kind == "decode":
        # the cache has room for 256 more tokens: its live part is a strided view
        cache_k, cache_v = randn(B, H, N + 256, D), randn(B, H, N + 256, D)
        return {"q": randn(B, H, case["Nq"], D), "k": cache_k[:, :, :N], "v": cache_v[:, :, :N]}
    t = {n: randn(B, H, N, D, scale=case.get("q_scale", 1.0)) for n in ("q", "k", "v")}
    if case.get("kt"):
        t["k"] = t["k"].transpose(2, 3).contiguous()
    if kind == "train":
        t["do"] = randn(B, H, N, D)
    return t


def prepare(case: dict, seed: int) -> dict:
    s = _inputs(case, seed)
    s["case"] = case
    kind = case["kind"]
    if kind == "train":
        for n in ("q", "k", "v"):
            s[n].requires_grad_()
    elif kind == "attn_fp32":
        s["launch"], _ = bind_flash_attention(s["q"], s["k"], s["v"], k_transposed=case["kt"])
    elif kind == "program_ln":
        from run_mlp_search import build_mlp_ln
        s["module"] = load_module(emit_module(build_mlp_ln(case["M"], case["D"], case["F"], tile=case["tile"],
                                                           dtype=case["dtype"])))
        named = {"X": s["x"], "W1": s["w1"], "W2": s["w2"]}
        s["args"] = [named[n] for n in s["module"].inputs]
    return s


def run(s: dict):
    case = s["case"]
    kind = case["kind"]
    if kind == "attn":
        return flash_attention_fwd(s["q"], s["k"], s["v"], causal=case["causal"], k_transposed=case["kt"])
    if kind == "attn_fp32":
        return s["launch"]()
    if kind == "train":
        o = flash_attention(s["q"], s["k"], s["v"], causal=case["causal"])
        dq, dk, dv = torch.autograd.grad(o, (s["q"], s["k"], s["v"]), s["do"])
        return {"o": o.detach(), "dq": dq, "dk": dk, "dv": dv}
    if kind == "decode":
        return flash_attention_decode(s["q"], s["k"], s["v"])
    if kind == "mlp":
        return mlp_fwd(s["x"], s["w1"], s["w2"])
    return s["module"].fn(*s["args"])


def work(case: dict) -> dict:
    kind, e = case["kind"], ELEM[case["dtype"]]
    if kind in ("mlp", "program_ln"):
        M, D, F = case["M"], case["D"], case["F"]
        return {"bytes": e * (2 * M * D + 2 * D * F), "flops": 4 * M * D * F}
    B, H, N, D = case["B"], case["H"], case["N"], case["D"]
    nq = case.get("Nq", N)
    fwd = 4 * B * H * nq * N * D // (2 if case.get("causal") else 1)
    if kind == "train":
        # Q, K, V, dO in and O, dQ, dK, dV out; two products forward, five back
        return {"bytes": e * 8 * B * H * N * D, "flops": fwd * 7 // 2}
    return {"bytes": e * 2 * B * H * (nq + N) * D, "flops": fwd}


def tolerance(case: dict) -> dict:
    """About four times the distance to exact() measured on an MI355X: at
    most 5.1e-7 in fp32, 3.7e-4 (gradients and the MLP's output: 3.9e-4 and
    3.0e-4) in fp16, 2.6e-3 in bf16."""
    if case["dtype"] == "fp32":
        return {"rel": 2e-6}
    if case["dtype"] == "bf16":
        return {"rel": 1e-2}
    return {"rel": 1.2e-3 if case["kind"] == "mlp" else 1.5e-3}


def exact(case: dict, seed: int):
    s = {n: t.double() for n, t in _inputs(case, seed).items()}
    kind = case["kind"]
    if kind == "mlp":
        h = s["x"] @ s["w1"]
        return (h * torch.sigmoid(h)) @ s["w2"]
    if kind == "program_ln":
        r = torch.relu(s["x"] @ s["w1"]) @ s["w2"] + s["x"]
        return (r - r.mean(1, keepdim=True)) / torch.sqrt(r.var(1, unbiased=False, keepdim=True) + 1e-5)
    q, k, v = s["q"], s["k"], s["v"]
    if case.get("kt"):
        k = k.transpose(2, 3)
    k, v = k.contiguous(), v.contiguous()
    B, H, N, D = k.shape
    nq, scale = q.shape[2], 1.0 / math.sqrt(D)
    mask = torch.ones(nq, N, dtype=torch.bool, device=q.device).triu(1) if case.get("causal") else None
    out = torch.empty_like(q)
    grads = {n: torch.empty_like(q) for n in ("dq", "dk", "dv")} if kind == "train" else None
    for b in range(B):
        for h in range(H):                 # one head at a time: the scores of all would not fit
            sc = (q[b, h] @ k[b, h].t().contiguous()) * scale
            if mask is not None:
                sc.masked_fill_(mask, float("-inf"))
            p = torch.softmax(sc, dim=1)
            out[b, h] = p @ v[b, h]
            if grads is not None:
                do = s["do"][b, h]
                grads["dv"][b, h] = p.t() @ do
                ds = p * (do @ v[b, h].t() - (do * out[b, h]).sum(1, keepdim=True)) * scale
                grads["dq"][b, h] = ds @ k[b, h]
                grads["dk"][b, h] = ds.t() @ q[b, h]
    return out if grads is None else {"o": out, **grads}

"""Performance cases of the gdn2 token mixer: what its users run, from one decode step to a training step.

Every case goes through a public entry point: the ops ``chunk_gdn2`` (prefill, training),
``fused_recurrent_gdn2`` / ``fused_recurrent_gdn2_fwd`` (short prompts, decode), the module
``GatedDeltaNet2`` (prefill, decode, training) and the hybrid decoder's ``GreedyDecoder``.
``exact`` restates each of them in float64 with plain torch, token by token.
"""

from __future__ import annotations

import math
from typing import Any

import torch
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint

from qwendopamine_amd import GatedDeltaNet2, chunk_gdn2, fused_recurrent_gdn2, fused_recurrent_gdn2_fwd
from qwendopamine_amd.hybrid import GreedyDecoder, HybridConfig, HybridDecoder

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
EPS = 1e-5  # the norms' default


def listed() -> list[dict]:
    return [
        # One generated token of a small served batch through one mixer layer, its caches updated
        # in place: the smallest call, bound by launches and latency.
        dict(name="layer-decode-b4", kind="layer_decode", hidden=1024, H=16, D=64, B=4),
        # One generated token of a large served batch: 67 MB of float32 state read and written.
        dict(name="decode-n64-d128", kind="decode", N=64, H=16, D=128, dtype="bf16", pool=False),
        # A short prompt, below the chunkwise path's length.
        dict(name="prompt-b2-t48-d128", kind="prompt", B=2, T=48, H=16, D=128, dtype="bf16"),
        # A small float32 prefill: few chunks and few heads.
        dict(name="prefill-fp32-t512-d64", kind="prefill", B=1, T=512, H=4, D=64, dtype="fp32", gate="scalar", state=False),
        # The headline prefill: a full batch of 4096-token prompts.
        dict(name="prefill-b8-t4096-d128", kind="prefill", B=8, T=4096, H=16, D=128, dtype="bf16", gate="scalar", state=False),
        # One long document that continues from a state, raw gate inputs.
        dict(name="prefill-b1-t16384-d128", kind="prefill", B=1, T=16384, H=16, D=128, dtype="bf16", gate="logits", state=True),
        # Prompts of unequal lengths packed into one row.
        dict(name="prefill-packed-n9-d128", kind="packed", seqs=9, total=7013, H=16, D=128, dtype="bf16"),
        # One mixer layer of the 1.3B preset's width on a ragged prompt batch.
        dict(name="layer-prefill-b2-t1537", kind="layer_prefill", hidden=2304, H=18, D=128, B=2, T=1537),
        # One mixer layer's training step: every parameter's gradient and the input's.
        dict(name="layer-train-b4-t2048", kind="layer_train", hidden=1024, H=16, D=64, B=4, T=2048),
        # The op's training step at full size.
        dict(name="train-b4-t8192-d128", kind="train", B=4, T=8192, H=16, D=128, dtype="bf16", gate="scalar"),
        # A float32 training step with a ragged length, as in numerics work and fine-tuning of small models.
        dict(name="train-fp32-b2-t777-d64", kind="train", B=2, T=777, H=8, D=64, dtype="fp32", gate="module"),
        # One decode step of a whole hybrid model (three mixer layers and an attention layer) as
        # its captured graph runs it, logits kept.
        dict(name="model-decode-b4-t512", kind="model_decode", B=4, T=512, layers=4, vocab=32000),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["layer_decode", "decode", "prompt", "prefill", "prefill", "packed", "layer_prefill",
                       "layer_train", "train", "train", "model_decode"])
    wide = rng.choice([dict(hidden=1024, H=16, D=64), dict(hidden=2304, H=18, D=128), dict(hidden=512, H=8, D=64)])
    if kind == "layer_decode":
        return dict(kind=kind, **wide, B=_log_int(rng, 1, 64))
    if kind == "decode":
        return dict(kind=kind, N=_log_int(rng, 1, 200), H=rng.choice([4, 8, 16]), D=rng.choice([64, 128]),
                    dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]), pool=rng.choice([False, True]))
    if kind == "prompt":
        return dict(kind=kind, B=_log_int(rng, 1, 12), T=rng.randint(2, 64), H=rng.choice([4, 8, 16]),
                    D=rng.choice([64, 128]), dtype=rng.choice(["bf16", "bf16", "fp32"]))
    if kind in ("prefill", "train"):
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        D, H, T = rng.choice([64, 128]), rng.choice([4, 8, 16]), _log_int(rng, 65, 8192 if kind == "train" else 16384)
        most = (40000 if dtype == "fp32" else 300000) // (H * T)
        case = dict(kind=kind, B=_log_int(rng, 1, max(1, min(8, most))), T=T, H=H, D=D, dtype=dtype)
        if dtype == "fp32":
            case["T"] = min(T, 40000 // H)
        case["gate"] = rng.choice(["scalar", "module"] if kind == "train" else ["scalar", "module", "logits"])
        return case if kind == "train" else dict(case, state=rng.choice([False, True]))
    if kind == "packed":
        return dict(kind=kind, seqs=rng.randint(2, 24), total=_log_int(rng, 300, 16000), H=rng.choice([8, 16]),
                    D=rng.choice([64, 128]), dtype="bf16")
    if kind in ("layer_prefill", "layer_train"):
        most = (3000 if kind == "layer_prefill" else 1400) * (1 if wide["hidden"] > 1024 else 4)
        T = _log_int(rng, 65, min(most, 2500))
        return dict(kind=kind, **wide, B=rng.randint(1, min(4, most // T)), T=T)
    return dict(kind=kind, B=rng.randint(1, 8), T=_log_int(rng, 65, 1500), layers=4, vocab=32000)


# ------------------------------------------------------------------------------- inputs
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _gate_params(gen, H: int, K: int) -> tuple[torch.Tensor, torch.Tensor]:
    """A_log and dt_bias as the module draws them: A ~ U(1, 16), dt log-uniform in [1e-3, 1e-1]."""
    A_log = (torch.rand(H, generator=gen, device="cuda") * 15 + 1).log()
    dt = torch.exp(torch.rand(H * K, generator=gen, device="cuda") * math.log(100.0) + math.log(1e-3))
    return A_log, dt + torch.log(-torch.expm1(-dt))


def _op_inputs(gen, B: int, T: int, H: int, D: int, dtype: torch.dtype, gate: str) -> dict[str, Any]:
    """q, k, v ~ N(0, 1) and the gates: "scalar" one decay and one write / erase strength per
    head (the benchmark's recipe), "module" channel-wise ones as the module forms them, "logits"
    the same before their activations (the ops apply them)."""

    def randn(*s):
        return torch.randn(*s, generator=gen, device="cuda")

    x: dict[str, Any] = {n: randn(B, T, H, D).to(dtype) for n in "qkv"}
    if gate == "scalar":
        beta = torch.sigmoid(randn(B, T, H, 1)).expand(B, T, H, D)
        x["g"] = (-F.softplus(randn(B, T, H, 1) + 2.0)).expand(B, T, H, D).contiguous()
        x["b"], x["w"] = beta.to(dtype).contiguous(), beta.to(dtype).contiguous()
        return x
    A_log, dt_bias = _gate_params(gen, H, D)
    f, b, w = randn(B, T, H, D) * 0.5, randn(B, T, H, D), randn(B, T, H, D)
    if gate == "logits":
        x.update(g=f.to(dtype), b=b.to(dtype), w=w.to(dtype), A_log=A_log, dt_bias=dt_bias)
    else:
        x["g"] = -A_log.exp()[:, None] * F.softplus(f + dt_bias.view(H, D))
        x["b"], x["w"] = b.sigmoid().to(dtype), w.sigmoid().to(dtype)
    return x


def _state(gen, N: int, H: int, D: int) -> torch.Tensor:
    return torch.randn(N, H, D, D, generator=gen, device="cuda") * 0.1


def _layer(case: dict, seed: int) -> GatedDeltaNet2:
    torch.manual_seed(seed)
    with torch.device("cuda"):
        m = GatedDeltaNet2(hidden_size=case["hidden"], num_heads=case["H"], head_dim=case["D"])
    return m.to(torch.bfloat16)


def _model(case: dict, seed: int) -> tuple[HybridDecoder, torch.Tensor]:
    torch.manual_seed(seed)
    n = case["layers"]
    config = HybridConfig.c3(n_layer=n, gdn2_layers=[i for i in range(n) if i % 4 != 3], vocab_size=case["vocab"])
    with torch.device("cuda"):
        model = HybridDecoder(config).to(torch.bfloat16).eval()
    return model, torch.randint(0, case["vocab"], (case["B"], case["T"] + 2), generator=_gen(seed), device="cuda")


def prepare(case: dict, seed: int) -> dict[str, Any]:
    kind, gen = case["kind"], _gen(seed)
    if kind in ("prefill", "train"):
        x = _op_inputs(gen, case["B"], case["T"], case["H"], case["D"], DTYPES[case["dtype"]], case["gate"])
        s = {"kind": kind, "x": x, "kw": {}}
        if kind == "train":
            for t in x.values():
                t.requires_grad_(True)
            s["do"] = torch.randn(x["v"].shape, generator=gen, device="cuda").to(x["v"].dtype)
            return s
        if case["gate"] == "logits":
            s["kw"] = dict(use_gate_in_kernel=True, bw_logits=True)
        if case["state"]:
            s["kw"]["initial_state"] = _state(gen, case["B"], case["H"], case["D"])
        return s
    if kind == "packed":
        x = _op_inputs(gen, 1, case["total"], case["H"], case["D"], DTYPES[case["dtype"]], "module")
        cuts = torch.randperm(case["total"] - 1, generator=gen, device="cuda")[:case["seqs"] - 1] + 1
        ends = torch.tensor([0, case["total"]], device="cuda")
        return {"kind": kind, "x": x, "kw": {"cu_seqlens": torch.cat([ends, cuts]).sort().values}}
    if kind == "prompt":
        x = _op_inputs(gen, case["B"], case["T"], case["H"], case["D"], DTYPES[case["dtype"]], "module")
        return {"kind": kind, "x": x}
    if kind == "decode":
        x = _op_inputs(gen, case["N"], 1, case["H"], case["D"], DTYPES[case["dtype"]], "module")
        rows = case["N"] + case["N"] // 2 if case["pool"] else case["N"]
        s = {"kind": kind, "x": x, "state": _state(gen, rows, case["H"], case["D"]), "kw": {}}
        if case["pool"]:
            s["kw"] = {"ssm_state_indices": torch.randperm(rows, generator=gen, device="cuda")[:case["N"]].contiguous()}
        return s
    if kind == "model_decode":
        model, tokens = _model(case, seed)
        dec = GreedyDecoder(model, keep_logits=True)
        dec.prefill(tokens[:, :case["T"]], 256)
        dec.tok.copy_(tokens[:, case["T"]:case["T"] + 1])
        dec.step()  # runs this token and captures the step
        return {"kind": kind, "dec": dec, "tok": tokens[:, case["T"] + 1:].contiguous(), "pos": case["T"] + 1}
    T = 1 if kind == "layer_decode" else case["T"]
    layer = _layer(case, seed)
    s = {"kind": kind, "layer": layer, "x": torch.randn(case["B"], T, case["hidden"], generator=gen, device="cuda").to(torch.bfloat16)}
    if kind == "layer_decode":
        layer.eval()
        s["cache"] = {"recurrent_state": _state(gen, case["B"], case["H"], case["D"]),
                      "conv_state": tuple(torch.randn(case["B"], case["H"] * case["D"], 3, generator=gen,
                                                      device="cuda").to(torch.bfloat16) for _ in range(3))}
    elif kind == "layer_prefill":
        layer.eval()
    else:
        layer.train()
        s["x"].requires_grad_(True)
        s["do"] = torch.randn(s["x"].shape, generator=gen, device="cuda").to(torch.bfloat16)
    return s


# ------------------------------------------------------------------------------- one pass
def run(s: dict[str, Any]) -> Any:
    kind = s["kind"]
    if kind == "train":
        o, _ = chunk_gdn2(**s["x"], use_qk_l2norm_in_kernel=True)
        grads = torch.autograd.grad(o, list(s["x"].values()), s["do"])
        return {"o": o.detach(), **{"d" + n: t for n, t in zip(s["x"], grads)}}
    if kind == "layer_train":
        out, _, _ = s["layer"](s["x"])
        names, params = zip(*s["layer"].named_parameters())
        grads = torch.autograd.grad(out, [s["x"], *params], s["do"])
        return {"out": out.detach(), "dx": grads[0], **dict(zip(names, grads[1:]))}
    with torch.no_grad():
        if kind in ("prefill", "packed"):
            o, state = chunk_gdn2(**s["x"], use_qk_l2norm_in_kernel=True, output_final_state=True, **s["kw"])
            return {"o": o, "state": state}
        if kind == "prompt":
            o, state = fused_recurrent_gdn2(**s["x"], use_qk_l2norm_in_kernel=True, output_final_state=True)
            return {"o": o, "state": state}
        if kind == "decode":
            o, state = fused_recurrent_gdn2_fwd(**s["x"], initial_state=s["state"], inplace_final_state=True,
                                                use_qk_l2norm_in_kernel=True, **s["kw"])
            return {"o": o, "state": state}
        if kind == "layer_decode":
            out, _, c = s["layer"](s["x"], past_key_values=s["cache"], use_cache=True, update_cache_in_place=True)
            return {"out": out, "state": c["recurrent_state"], "conv": list(c["conv_state"])}
        if kind == "layer_prefill":
            out, _, c = s["layer"](s["x"], past_key_values={}, use_cache=True)
            return {"out": out, "state": c["recurrent_state"], "conv": list(c["conv_state"])}
        # A known token scored at its position (the same one again on a repeated pass).
        s["dec"].tok.copy_(s["tok"])
        s["dec"].pos.fill_(s["pos"])
        s["dec"].step()
        return {"logits": s["dec"].logits,
                "states": [blk.gdn2_cache["recurrent_state"] for blk in s["dec"].model.h if blk.use_gdn2]}


# ------------------------------------------------------------------------------- work
def work(case: dict) -> dict[str, float]:
    """Bytes: every input once, every output once. Operations: the chunkwise form's products over
    64-token chunks (the recurrence's own for single tokens and short prompts), a layer's
    projections, a model's layers and head."""
    kind, H, D = case["kind"], case.get("H", 16), case.get("D", 64)
    e = 4 if case.get("dtype") == "fp32" else 2
    fwd_ops = 6 * D * D + 2 * 64 * 5 * D + 64 * 64 / 3
    bwd_ops = 16 * D * D + 24 * 64 * D + 4 * 64 * 64
    if kind in ("prefill", "packed", "train"):
        n = case.get("B", 1) * case.get("T", case.get("total", 0)) * H
        states = case.get("seqs", case.get("B", 1)) * H * D * D * 4
        eg = e if case.get("gate") == "logits" else 4
        fwd = n * (5 * D * e + D * eg + D * e)
        if kind == "train":
            # The backward reads the inputs and do and writes six gradients.
            return {"bytes": 2.0 * fwd + n * (5 * D * e + 4 * D), "flops": float(n * (fwd_ops + bwd_ops))}
        return {"bytes": float(fwd + states * (2 if case.get("state") else 1)), "flops": float(n * fwd_ops)}
    if kind in ("prompt", "decode"):
        seqs = case["B"] if kind == "prompt" else case["N"]
        n = seqs * case.get("T", 1) * H
        return {"bytes": float(n * (6 * D * e + 4 * D) + seqs * H * D * D * 4 * (1 if kind == "prompt" else 2)),
                "flops": float(n * 7 * D * D)}
    if kind == "model_decode":
        B, T, C, inner = case["B"], case["T"], 1024, 3072
        n_attn = case["layers"] // 4
        n_mix = case["layers"] - n_attn
        params = (n_mix * _layer_params(C, 16, 64) + n_attn * 4 * C * C + case["layers"] * 3 * C * inner
                  + case["vocab"] * C)
        cache = n_mix * B * 16 * 64 * 64 * 4 * 2 + n_attn * B * T * C * 2 * 2
        return {"bytes": float(2 * params + cache + 4 * B * case["vocab"]),
                "flops": float(2 * B * params + n_mix * B * 16 * 7 * 64 * 64 + n_attn * 4 * B * T * C)}
    B, T, C = case["B"], case.get("T", 1), case["hidden"]
    params, tokens = _layer_params(C, H, D), B * T
    x = tokens * C * 2
    if kind == "layer_decode":
        return {"bytes": float(2 * params + 2 * x + B * H * D * D * 8 + 2 * 3 * B * H * D * 3 * 2),
                "flops": float(tokens * (2 * params + H * 7 * D * D))}
    if kind == "layer_prefill":
        return {"bytes": float(2 * params + 2 * x + B * H * D * D * 4), "flops": float(tokens * (2 * params + H * fwd_ops))}
    return {"bytes": float(3 * 2 * params + 4 * x), "flops": float(tokens * (6 * params + H * (fwd_ops + bwd_ops)))}


def _layer_params(C: int, H: int, D: int) -> int:
    """The mixer's matrices: q, k, v, b, w and output projections and two low-rank pairs."""
    return 6 * C * H * D + 2 * (C * D + D * H * D)


def tolerance(case: dict) -> dict[str, float]:
    """About four times the error measured against ``exact``: rounding of 16-bit inputs, products and
    results, or float32 sums in another order."""
    if case["kind"] in ("prefill", "packed", "prompt", "decode", "train"):
        return {"rel": 1e-5} if case["dtype"] == "fp32" else {"rel": 2e-2}
    # Through a whole model the layers' bf16 roundings add up.
    return {"rel": 6e-2} if case["kind"] == "model_decode" else {"rel": 4e-2}


# ------------------------------------------------------------------------------- float64
def _tokens64(q, k, v, g, b, w, S):
    """The recurrence over one run of tokens: returns its outputs and the state after it."""
    out = []
    for t in range(q.shape[1]):
        kt = k[:, t]
        S = S * g[:, t].exp().unsqueeze(-1)
        u = w[:, t] * v[:, t] - ((b[:, t] * kt).unsqueeze(-1) * S).sum(-2)
        S = S + kt.unsqueeze(-1) * u.unsqueeze(-2)
        out.append((q[:, t].unsqueeze(-1) * S).sum(-2))
    return torch.stack(out, 1), S


def _recurrence64(q, k, v, g, b, w, S=None):
    """S <- Diag(e^g) S;  S <- S + k (w v - S^T (b k))^T;  o = S^T q, with q and k normalised."""
    K = q.shape[-1]
    q = q / q.norm(dim=-1, keepdim=True).clamp_min(1e-6) * K ** -0.5
    k = k / k.norm(dim=-1, keepdim=True).clamp_min(1e-6)
    if S is None:
        S = q.new_zeros(q.shape[0], q.shape[2], K, v.shape[-1])
    grad = torch.is_grad_enabled() and any(t.requires_grad for t in (q, k, v, g, b, w))
    outs = []
    for t in range(0, q.shape[1], 64):
        part = [x[:, t:t + 64] for x in (q, k, v, g, b, w)]
        o, S = checkpoint(_tokens64, *part, S, use_reentrant=False) if grad else _tokens64(*part, S)
        outs.append(o)
    return torch.cat(outs, 1), S


def _op64(x: dict, S=None):
    x = {n: t.double() for n, t in x.items()}
    g, b, w = x["g"], x["b"], x["w"]
    if "A_log" in x:
        g = -x["A_log"].exp()[:, None] * F.softplus(g + x["dt_bias"].view(g.shape[-2:]))
        b, w = b.sigmoid(), w.sigmoid()
    return _recurrence64(x["q"], x["k"], x["v"], g, b, w, S)


def _layer64(P: dict, x, H: int, D: int, state=None, conv=None):
    """The mixer layer from its parameters: returns output, state and the last three conv inputs."""
    B, T, _ = x.shape

    def heads(t):
        return t.reshape(B, T, H, D)

    raw = [x @ P[n + "_proj.weight"].T for n in "qkv"]
    pad = [torch.cat([r.new_zeros(B, 3, H * D) if conv is None else c.transpose(1, 2), r], 1)
           for r, c in zip(raw, conv or [None] * 3)]
    q, k, v = (heads(F.silu(sum(p[:, j:j + T] * P[n + "_conv1d.conv1d.weight"][:, 0, j] for j in range(4))))
               for n, p in zip("qkv", pad))
    f = x @ P["f_proj.0.weight"].T @ P["f_proj.1.weight"].T
    g = -P["A_log"].exp()[:, None] * F.softplus(heads(f + P["dt_bias"]))
    b, w = (heads((x @ P[n + "_proj.weight"].T).sigmoid()) for n in "bw")
    o, state = _recurrence64(q, k, v, g, b, w, state)
    z = heads(x @ P["g_proj.0.weight"].T @ P["g_proj.1.weight"].T + P["g_proj.1.bias"])
    o = o * torch.rsqrt(o.square().mean(-1, keepdim=True) + EPS) * P["o_norm.weight"] * F.silu(z)
    return o.reshape(B, T, H * D) @ P["o_proj.weight"].T, state, [p[:, T:].transpose(1, 2) for p in pad]


def _norm64(x, weight):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * weight


def _attention64(P: dict, x, heads: int, D: int):
    B, T, _ = x.shape
    q, k, v = (x @ P["attn.weight"].T).reshape(B, T, heads, 3, D).unbind(3)
    theta = 10000.0 ** (-torch.arange(0, D, 2, device=x.device, dtype=x.dtype) / D)
    ang = torch.outer(torch.arange(T, device=x.device, dtype=x.dtype), theta)[:, None]
    c, s = ang.cos(), ang.sin()
    q, k = (torch.stack((t[..., ::2] * c - t[..., 1::2] * s, t[..., ::2] * s + t[..., 1::2] * c), -1).flatten(-2)
            for t in (q, k))
    q, k, v = (t.transpose(1, 2) for t in (q, k, v))
    a = (q @ k.transpose(-1, -2).contiguous()) / math.sqrt(D)
    a = a.masked_fill(torch.ones(T, T, device=x.device, dtype=torch.bool).triu(1), float("-inf")).softmax(-1)
    return (a @ v.contiguous()).transpose(1, 2).reshape(B, T, heads * D) @ P["proj.weight"].T


def _model64(P: dict, tokens, layers: int):
    def sub(prefix):
        return {n[len(prefix):]: t for n, t in P.items() if n.startswith(prefix)}

    x, states = P["wte.weight"][tokens], []
    for i in range(layers):
        L = sub("h.%d." % i)
        n1, A = _norm64(x, L["norm_1.weight"]), sub("h.%d.attn." % i)
        if i % 4 == 3:
            x = x + _attention64(A, n1, 16, 64)
        else:
            h, S, _ = _layer64(A, n1, 16, 64)
            x = x + h
            states.append(S)
        n2 = _norm64(x, L["norm_2.weight"])
        a = F.silu(n2 @ L["mlp.swiglu.w1.weight"].T) * (n2 @ L["mlp.swiglu.w2.weight"].T)
        x = x + a @ L["mlp.swiglu.w3.weight"].T
    return _norm64(x[:, -1], P["ln_f.weight"]) @ P["lm_head.weight"].T, states


def exact(case: dict, seed: int) -> Any:
    kind = case["kind"]
    if kind == "model_decode":
        model, tokens = _model(case, seed)
        with torch.no_grad():
            logits, states = _model64({n: p.double() for n, p in model.named_parameters()}, tokens, case["layers"])
            return {"logits": logits, "states": states}
    s = prepare(case, seed)
    if kind == "train":
        x = {n: t.detach().double().requires_grad_(True) for n, t in s["x"].items()}
        o, _ = _op64(x)
        grads = torch.autograd.grad(o, list(x.values()), s["do"].double())
        return {"o": o.detach(), **{"d" + n: t for n, t in zip(x, grads)}}
    if kind == "layer_train":
        P = {n: p.detach().double().requires_grad_(True) for n, p in s["layer"].named_parameters()}
        x = s["x"].detach().double().requires_grad_(True)
        out, _, _ = _layer64(P, x, case["H"], case["D"])
        grads = torch.autograd.grad(out, [x, *P.values()], s["do"].double())
        return {"out": out.detach(), "dx": grads[0], **dict(zip(P, grads[1:]))}
    with torch.no_grad():
        if kind == "packed":
            cu = s["kw"]["cu_seqlens"].tolist()
            parts = [_op64({n: t[:, a:z] for n, t in s["x"].items()}) for a, z in zip(cu, cu[1:])]
            return {"o": torch.cat([o for o, _ in parts], 1), "state": torch.cat([S for _, S in parts])}
        if kind in ("prefill", "prompt"):
            S = s.get("kw", {}).get("initial_state")
            o, S = _op64(s["x"], None if S is None else S.double())
            return {"o": o, "state": S}
        if kind == "decode":
            rows = s["kw"].get("ssm_state_indices")
            S = s["state"].double()
            o, new = _op64(s["x"], S if rows is None else S[rows])
            return {"o": o, "state": new if rows is None else S.index_copy(0, rows, new)}
        P = {n: p.double() for n, p in s["layer"].named_parameters()}
        cache = s.get("cache")
        state, conv = (None, None) if cache is None else (cache["recurrent_state"].double(), [c.double() for c in cache["conv_state"]])
        out, state, conv = _layer64(P, s["x"].double(), case["H"], case["D"], state, conv)
        return {"out": out, "state": state, "conv": conv}

"""A 16-bit ``GatedDeltaNet2`` training step, whose decay runs on the gate kernels, against the same layer
composed in float64 from torch operations: the output, the input's gradient and every parameter's."""

import pytest
import torch
import torch.nn.functional as F

from tests._helpers import rel_l2

pytestmark = pytest.mark.gpu


def _recurrence(q, k, v, g, b, w):
    q = q / q.norm(dim=-1, keepdim=True) * q.shape[-1] ** -0.5
    k = k / k.norm(dim=-1, keepdim=True)
    S, out = q.new_zeros(*q.shape[1:], v.shape[-1]), []
    for t in range(q.shape[0]):
        S = S * g[t].exp()[..., None]
        u = w[t] * v[t] - ((b[t] * k[t])[..., None] * S).sum(-2)
        S = S + k[t][..., None] * u[..., None, :]
        out.append((q[t][..., None] * S).sum(-2))
    return torch.stack(out)


def _layer64(P, x, lens, D, rep, g_dtype):
    """Sequences of the given lengths, packed [sum, C], through the layer's formula (whose convolutions run
    over the packed row: a sequence's first tokens see the end of the one before)."""
    def heads(t):
        return t.view(x.shape[0], -1, D)

    def conv(n):
        raw = F.pad((x @ P[n + "_proj.weight"].T).T, (3, 0))
        return heads(F.silu(F.conv1d(raw, P[n + "_conv1d.conv1d.weight"], groups=raw.shape[0])).T)

    q, k, v = (conv(n) for n in "qkv")
    f = x @ P["f_proj.0.weight"].T @ P["f_proj.1.weight"].T
    g = -P["A_log"].exp()[:, None] * heads(F.softplus(f + P["dt_bias"]))
    if g_dtype is not None:
        g = g + (g.to(g_dtype).double() - g).detach()  # the layer rounds its decay
    b, w = (heads((x @ P[n + "_proj.weight"].T).sigmoid()) for n in "bw")
    q, k, g, b = (t.repeat_interleave(rep, dim=1) for t in (q, k, g, b))
    o = torch.cat([_recurrence(*part) for part in zip(*(t.split(lens) for t in (q, k, v, g, b, w)))])
    z = heads(x @ P["g_proj.0.weight"].T @ P["g_proj.1.weight"].T + P["g_proj.1.bias"])
    o = o * torch.rsqrt(o.square().mean(-1, keepdim=True) + 1e-5) * P["o_norm.weight"] * F.silu(z)
    return o.flatten(1) @ P["o_proj.weight"].T


@pytest.mark.parametrize("H,HV,D,T,dtype,fp32_decay,masked", [
    (4, 4, 64, 130, torch.bfloat16, True, False),
    (2, 4, 32, 77, torch.bfloat16, True, False),
    (2, 2, 50, 65, torch.float16, True, False),
    (3, 3, 64, 100, torch.bfloat16, True, True),
    (2, 2, 128, 90, torch.float16, True, False),
    (2, 2, 64, 70, torch.bfloat16, False, False),
])
def test_module_gradients_match_float64(gpu_device, H, HV, D, T, dtype, fp32_decay, masked):
    from qwendopamine_amd import GatedDeltaNet2

    print(f"[case] module training H={H} HV={HV} D={D} T={T} {dtype} fp32_decay={fp32_decay} masked={masked}", flush=True)
    torch.manual_seed(T)
    layer = GatedDeltaNet2(hidden_size=128, num_heads=H, num_v_heads=HV, head_dim=D, fp32_decay=fp32_decay)
    layer = layer.to(gpu_device, dtype).train()
    x = torch.randn(2, T, 128).to(gpu_device, dtype).requires_grad_(True)
    do = torch.randn(2, T, 128).to(gpu_device, dtype)
    mask, starts = None, [0, 0]
    if masked:
        starts = [0, T // 3]  # left padding
        mask = torch.ones(2, T, dtype=torch.long, device=gpu_device)
        mask[1, :starts[1]] = 0
    out, _, _ = layer(x, attention_mask=mask)
    out.backward(do)

    P = {n: p.detach().cpu().double().requires_grad_(True) for n, p in layer.named_parameters()}
    x64 = x.detach().cpu().double().requires_grad_(True)
    rows = [x64[i, s:] for i, s in enumerate(starts)]
    args = D, HV // H, None if fp32_decay else dtype
    if masked:
        parts = _layer64(P, torch.cat(rows), [len(r) for r in rows], *args).split([len(r) for r in rows])
    else:
        parts = [_layer64(P, r, [len(r)], *args) for r in rows]
    ref = torch.stack([F.pad(o, (0, 0, s, 0)) for o, s in zip(parts, starts)])
    ref.backward(do.cpu().double())
    errs = {"out": rel_l2(out, ref), "x": rel_l2(x.grad, x64.grad)}
    errs.update((n, rel_l2(p.grad, P[n].grad)) for n, p in layer.named_parameters())
    print("  rel_l2 " + " ".join(f"{n}={e:.1e}" for n, e in errs.items()), flush=True)
    # A dozen roundings to bf16 (half an ulp: 2^-9; the chunk kernels' products take fp16 inputs in bf16 too)
    # on the way to a gradient, and sums of terms that partly cancel: 20 half ulps.
    assert not {n: e for n, e in errs.items() if not e <= 20 * 2.0 ** -9}

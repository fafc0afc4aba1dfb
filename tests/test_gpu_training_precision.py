"""Float32 intermediates of 16-bit training are as exact as torch's own float32 chain: a kernel's values equal
that chain's, or its error against float64 stays within the chain's on the same inputs."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _rms(x, ref):
    return ((x.double() - ref) / ref).square().mean().sqrt().item()


@pytest.mark.parametrize("H,HV,D,dtype", [(4, 4, 64, torch.bfloat16), (2, 4, 32, torch.float16), (2, 2, 100, torch.bfloat16)])
def test_module_decay_equals_torch(gpu_device, monkeypatch, H, HV, D, dtype):
    from qwendopamine_amd import GatedDeltaNet2, ops

    print(f"[case] module decay H={H} HV={HV} D={D} {dtype}", flush=True)
    torch.manual_seed(D)
    layer = GatedDeltaNet2(hidden_size=128, num_heads=H, num_v_heads=HV, head_dim=D).to(gpu_device, dtype).train()
    x = torch.randn(2, 130, 128).to(gpu_device, dtype)
    seen, real = {}, ops.chunk_gdn2

    def spy(q, k, v, g, *rest, **kw):
        seen["g"] = g.detach()
        return real(q, k, v, g, *rest, **kw)

    monkeypatch.setattr(ops, "chunk_gdn2", spy)
    layer(x)
    with torch.no_grad():
        A = layer.A_log.float().exp().repeat_interleave(D)
        g = (-A * F.softplus(layer.f_proj(x).float() + layer.dt_bias)).view(2, 130, H, D)
    assert seen["g"].dtype == torch.float32
    assert torch.equal(seen["g"], g.repeat_interleave(HV // H, dim=-2))


@pytest.mark.parametrize("K,spread", [(64, 2.0), (100, 8.0)])
def test_gate_vjp_is_as_exact_as_torch(gpu_device, K, spread):
    from qwendopamine_amd.ops import GateFunction

    print(f"[case] gate precision K={K} spread={spread}", flush=True)
    gen = torch.Generator().manual_seed(K)
    f = (torch.randn(2000, 8, K, generator=gen) * spread).to(gpu_device)
    A, db = (torch.rand(8, generator=gen) * 15 + 1).log().to(gpu_device), torch.randn(8 * K, generator=gen).to(gpu_device)
    dy = torch.randn(2000, 8, K, generator=gen).to(gpu_device)

    def torch_gate(f, A, db):
        return -A.exp()[:, None] * F.softplus(f + db.view(8, K))

    runs = []
    for gate, up in ((lambda *x: GateFunction.apply(*x, None, True), torch.float32), (torch_gate, torch.float32),
                     (torch_gate, torch.float64)):
        leaves = [t.detach().clone().to(up).requires_grad_(True) for t in (f, A, db)]
        y = gate(*leaves)
        y.backward(dy.to(up))
        runs.append([y.detach(), *(t.grad for t in leaves)])
    hip, ref, exact = runs
    # 1.1: both are the same float32 operations per value up to a contracted product; the sums
    # over tokens differ in order, whose error a few dozen values sample loosely (factor 2).
    for name, a, b, e, room in zip(("y", "dg", "dA_log", "ddt_bias"), hip, ref, exact, (1.1, 1.1, 2.0, 2.0)):
        got, want = _rms(a, e), _rms(b, e)
        print(f"  {name}: rms {got:.3g}, torch {want:.3g}", flush=True)
        assert got <= room * want, name


def _misrounded(x, exact):
    return (x != exact.to(x.dtype)).sum().item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_conv_silu_backward_is_as_exact_as_torch(gpu_device, dtype):
    from qwendopamine_amd.ops import short_conv_autograd

    print(f"[case] conv backward precision {dtype}", flush=True)
    gen = torch.Generator().manual_seed(1)
    x = (torch.randn(4, 2048, 1024, generator=gen) * 3).to(dtype).to(gpu_device)
    dy = torch.randn(x.shape, generator=gen).to(dtype).to(gpu_device)
    w = torch.zeros(1024, 1, 4, dtype=dtype, device=gpu_device)
    w[:, 0, 3] = 1  # the convolution passes x on: dx = round(dy silu'(x))
    hip, ref = x.clone().requires_grad_(True), x.clone().requires_grad_(True)
    short_conv_autograd(hip, w.requires_grad_(True), None, "silu").backward(dy)
    F.silu(ref).backward(dy)
    s = x.double().sigmoid()
    exact = dy.double() * s * (1 + x.double() * (1 - s))
    got, want = _misrounded(hip.grad, exact), _misrounded(ref.grad, exact)
    print(f"  misrounded {got}, torch {want}", flush=True)
    # How often a value rounds to the wrong neighbour is in proportion to its float32 error; products
    # contracted in one and not in the other move that error by up to a fifth.
    assert got <= 1.2 * want + 10


@pytest.mark.parametrize("N,dtype", [(64, torch.float16), (128, torch.float16), (256, torch.float16), (64, torch.bfloat16)])
def test_gated_norm_silu_backward_is_as_exact_as_torch(gpu_device, N, dtype):
    from qwendopamine_amd.ops import gated_rmsnorm_autograd

    print(f"[case] gated norm backward precision N={N} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(N)
    rows = 131072 * 64 // N
    # Rows of +-1 (norm exactly 1), unit weights and gradients: dz = round(x silu'(z)).
    x = (torch.randint(0, 2, (rows, N), generator=gen) * 2 - 1).to(dtype).to(gpu_device)
    z = (torch.randn(rows, N, generator=gen) * 3).to(dtype).to(gpu_device).requires_grad_(True)
    w = torch.ones(N, dtype=dtype, device=gpu_device)
    gated_rmsnorm_autograd(x.clone().requires_grad_(True), z, w.requires_grad_(True), 0.0).backward(torch.ones_like(x))
    s, zd = z.detach().double().sigmoid(), z.detach().double()
    exact = x.double() * s * (1 + zd * (1 - s))
    zf = z.detach().float()
    s = 1 / (1 + torch.exp(-zf))
    got, want = _misrounded(z.grad, exact), _misrounded((x.float() * (s * (1 + zf * (1 - s)))).to(dtype), exact)
    print(f"  misrounded {got}, torch {want}", flush=True)
    assert got <= 1.2 * want + 10  # as above

"""Edges of the training passes' kernels against float64: the gate's backward over rows that do and do not
fill a wave's lanes and token blocks, the gated norm's backward on whole 16-byte pieces and beside them, and
the float32 chunk scans, whose one LDS buffer is refilled from registers between two barriers."""

import pytest
import torch

from oracle import gdn2_oracle as orc
from tests._helpers import REL_TOL, rand_inputs, rel_l2, to_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,tokens,H,dtype", [(64, 257, 3, torch.bfloat16), (128, 64, 2, torch.bfloat16),
                                              (4, 700, 70, torch.float16), (252, 66, 1, torch.float32),
                                              (63, 130, 2, torch.bfloat16)])
def test_gate_backward_lane_splits(gpu_device, K, tokens, H, dtype):
    from qwendopamine_amd.ops import gate_activation

    print(f"[case] gate backward K={K} tokens={tokens} H={H} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(K)
    g = torch.randn(tokens, H, K, generator=gen).to(dtype)
    A, db = torch.randn(H, generator=gen), torch.randn(H * K, generator=gen)
    dy = torch.randn(tokens, H, K, generator=gen)
    dev = [t.to(gpu_device).requires_grad_(True) for t in (g, A, db)]
    gate_activation(*dev, None).backward(dy.to(gpu_device))
    ref = [t.double().requires_grad_(True) for t in (g, A, db)]
    y = -ref[1].exp()[:, None] * torch.nn.functional.softplus(ref[0] + ref[2].view(H, K))
    y.backward(dy.double())
    # dg leaves in g's type (half an ulp of bf16: 2^-9); the sums stay float32.
    for got, want, tol in zip(dev, ref, (1e-5 if dtype == torch.float32 else 4e-3, 1e-5, 1e-5)):
        assert rel_l2(got.grad, want.grad) <= tol


@pytest.mark.parametrize("rows", [1, 17, 5000])
@pytest.mark.parametrize("N,dtype", [(64, torch.bfloat16), (128, torch.float16), (256, torch.bfloat16),
                                     (256, torch.float32), (32, torch.float32), (96, torch.bfloat16)])
def test_gated_norm_backward_row_splits(gpu_device, rows, N, dtype):
    from qwendopamine_amd.ops import gated_rmsnorm_autograd

    print(f"[case] gated norm backward rows={rows} N={N} {dtype}", flush=True)
    gen = torch.Generator().manual_seed(rows + N)
    x, z, dy = (torch.randn(rows, N, generator=gen).to(dtype) for _ in range(3))
    w = (torch.randn(N, generator=gen) * 0.2 + 1).to(dtype)
    dev = [t.to(gpu_device).requires_grad_(True) for t in (x, z, w)]
    gated_rmsnorm_autograd(*dev, 1e-5).backward(dy.to(gpu_device))
    xd, zd, wd = ref = [t.double().requires_grad_(True) for t in (x, z, w)]
    y = xd * torch.rsqrt(xd.square().mean(-1, keepdim=True) + 1e-5) * wd * torch.nn.functional.silu(zd)
    y.backward(dy.double())
    # Every value is formed in float32 and rounded once to the tensors' type.
    for got, want in zip(dev, ref):
        assert rel_l2(got.grad, want.grad) <= (1e-5 if dtype == torch.float32 else 4e-3)


@pytest.mark.parametrize("T", [1, 64, 129, 300])
@pytest.mark.parametrize("K,V", [(64, 64), (128, 40)])
def test_float32_scans_over_chunk_counts(gpu_device, T, K, V):
    from qwendopamine_amd.ops import chunk_gdn2

    print(f"[case] float32 scans T={T} K={K} V={V}", flush=True)
    t, r = to_device(rand_inputs(2, T, 3, K, V, seed=T + K), gpu_device, torch.float32)
    names = ("q", "k", "v", "g", "b", "w")
    leaves = [t[n].detach().requires_grad_(True) for n in names]
    o, _ = chunk_gdn2(*leaves, use_qk_l2norm_in_kernel=True)
    do = torch.randn(o.shape, generator=torch.Generator().manual_seed(T))
    o.backward(do.to(gpu_device))
    tol = REL_TOL[torch.float32]
    vals = [r[n] for n in names]
    assert rel_l2(o, orc.recurrent_fwd(*vals)[0]) <= tol
    for x, ref in zip(leaves, orc.recurrent_vjp(*vals, do.double().numpy())):
        assert rel_l2(x.grad, ref) <= tol


@pytest.mark.parametrize("K,V,T,dtype", [(256, 40, 129, torch.float16), (132, 64, 77, torch.float16),
                                         (192, 48, 200, torch.bfloat16)])
def test_wide_key_backward_over_token_blocks(gpu_device, K, V, T, dtype):
    from qwendopamine_amd.ops import chunk_gdn2

    print(f"[case] wide key backward K={K} V={V} T={T} {dtype}", flush=True)
    t, r = to_device(rand_inputs(2, T, 2, K, V, seed=T + K), gpu_device, dtype)
    names = ("q", "k", "v", "g", "b", "w")
    leaves = [t[n].detach().requires_grad_(True) for n in names]
    o, _ = chunk_gdn2(*leaves, use_qk_l2norm_in_kernel=True)
    # Scaled as a training loop scales its loss in fp16: gradients of about 1e-5 would be subnormal.
    # dg sums pair terms that cancel in exact arithmetic.  Beyond d_k = 128 their factors are one
    # 16-bit plane (two, worth float32, up to 128), so each term keeps its rounding of 2^-9 while
    # the sum loses most of its size: 6e-2 to 7e-2 of it is left, in every build so far.
    do = (torch.randn(o.shape, generator=torch.Generator().manual_seed(T)) * 1024).to(dtype)
    o.backward(do.to(gpu_device))
    for n, x, ref in zip(names, leaves, orc.recurrent_vjp(*(r[n] for n in names), do.double().numpy())):
        assert rel_l2(x.grad, ref) <= (1e-1 if n == "g" else REL_TOL[dtype]), n


def _off_by_one(x):
    """An uninitialised tensor like ``x`` that starts one element past an aligned address."""
    return torch.empty(x.numel() + 8, dtype=x.dtype, device=x.device)[1:1 + x.numel()].view(x.shape)


@pytest.mark.parametrize("K,V,dtype", [(128, 128, torch.bfloat16), (64, 64, torch.float16), (64, 40, torch.float32)])
def test_chunk_backward_into_unaligned_gradients(gpu_device, monkeypatch, K, V, dtype):
    from qwendopamine_amd.backward import chunk_gdn2_bwd
    from qwendopamine_amd.ops import chunk_gdn2_fwd

    print(f"[case] unaligned gradients K={K} V={V} {dtype}", flush=True)
    t, _ = to_device(rand_inputs(2, 130, 2, K, V, seed=K, h0_std=0), gpu_device, dtype)
    args = [t[n] for n in ("q", "k", "v", "g", "b", "w")]
    do = torch.randn(2, 130, 2, V, generator=torch.Generator().manual_seed(V)).to(gpu_device, dtype)
    saved = chunk_gdn2_fwd(*args, K ** -0.5, None, False, use_qk_l2norm_in_kernel=True, save_for_bwd=True)[-1]
    aligned = chunk_gdn2_bwd(saved, do, None, False)
    monkeypatch.setattr(torch, "empty_like", _off_by_one)
    shifted = chunk_gdn2_bwd(saved, do, None, False)
    assert all(x.data_ptr() % 16 for x in shifted[:6])
    assert all(torch.equal(x, y) for x, y in zip(aligned[:6], shifted[:6]))


@pytest.mark.parametrize("library_math", [False, True])
@pytest.mark.parametrize("K,dtype", [(64, torch.bfloat16), (252, torch.float32)])
def test_gate_backward_into_unaligned_gradient(gpu_device, monkeypatch, K, dtype, library_math):
    from qwendopamine_amd.ops import GateFunction

    print(f"[case] unaligned gate gradient K={K} {dtype} library_math={library_math}", flush=True)
    gen = torch.Generator().manual_seed(K)
    leaves = [torch.randn(*s, generator=gen).to(d).to(gpu_device).requires_grad_(True)
              for s, d in (((130, 3, K), dtype), ((3,), torch.float32), ((3 * K,), torch.float32))]
    y = GateFunction.apply(*leaves, None, library_math)
    dy = torch.randn(130, 3, K, generator=gen).to(gpu_device)
    aligned = torch.autograd.grad(y, leaves, dy, retain_graph=True)
    monkeypatch.setattr(torch, "empty_like", _off_by_one)
    shifted = torch.autograd.grad(y, leaves, dy)
    assert shifted[0].data_ptr() % 16
    assert all(torch.equal(a, b) for a, b in zip(aligned, shifted))

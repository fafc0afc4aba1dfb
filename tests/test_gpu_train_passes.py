"""Edges of the training passes' kernels against float64: the gate's backward over rows that do and do not
fill a wave's lanes and token blocks, the gated norm's backward on whole 16-byte pieces and beside them, and
the float32 chunk scans, whose one LDS buffer is refilled from registers between two barriers."""

import pytest
import torch

from oracle import gdn2_oracle as orc
from tests._helpers import REL_TOL, rand_inputs, rel_l2, to_device

pytestmark = pytest.mark.gpu


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

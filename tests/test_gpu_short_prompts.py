"""Token-serial kernel for sequences of several tokens (``recurrent_seq_kernel``) against the oracle:
tile edges of the token loop (16 tokens, 8 beyond d_k = 128), ragged key and value widths, and the
three column splits (few, some and many sequence-heads)."""

import numpy as np
import pytest
import torch

from oracle import gdn2_oracle as orc
from tests._helpers import REL_TOL, rand_inputs, rel_l2, to_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,H,HV,K,V,dtype,decay", [
    (1, 2, 2, 2, 128, 128, torch.bfloat16, "paper"),
    (2, 16, 3, 3, 64, 64, torch.float32, "paper"),
    (1, 17, 2, 4, 128, 128, torch.float32, "unit"),
    (2, 33, 1, 1, 65, 20, torch.float32, "paper"),
    (1, 9, 2, 2, 200, 36, torch.float32, "unit"),
    (1, 64, 2, 2, 256, 128, torch.bfloat16, "paper"),
    (8, 31, 8, 8, 16, 48, torch.float16, "paper"),      # 64 heads of 48 columns: 32-column workgroups
    (16, 18, 16, 16, 128, 132, torch.bfloat16, "unit"),  # 256 heads: 64-column workgroups
    (2, 40, 2, 2, 128, 64, torch.float32, "sheer"),
])
def test_prompt_matches_oracle(gpu_device, B, T, H, HV, K, V, dtype, decay):
    from qwendopamine_amd.ops import fused_recurrent_gdn2

    print(f"[case] prompt B={B} T={T} H={H} HV={HV} K={K} V={V} {dtype} {decay}", flush=True)
    t, r = to_device(rand_inputs(B, T, H, K, V, HV=HV, seed=T + K, decay=decay), gpu_device, dtype)
    o, ht = fused_recurrent_gdn2(*(t[n] for n in ("q", "k", "v", "g", "b", "w")), initial_state=t["h0"],
                                 output_final_state=True, use_qk_l2norm_in_kernel=True)
    o_ref, s_ref = orc.recurrent_fwd(r["q"], r["k"], r["v"], r["g"], r["b"], r["w"], r["h0"])
    assert rel_l2(o, o_ref) <= REL_TOL[dtype]
    # The state stays in float32 whatever the inputs' type.
    assert rel_l2(ht, s_ref) <= 1e-5


@pytest.mark.parametrize("lens", [[2, 2, 2], [1, 0, 40, 16, 3], [33, 1, 1, 1]])
def test_packed_prompts_match_oracle(gpu_device, lens):
    from qwendopamine_amd.ops import fused_recurrent_gdn2

    print(f"[case] packed prompts {lens}", flush=True)
    cu = np.concatenate([[0], np.cumsum(lens)])
    inp = rand_inputs(1, int(cu[-1]), 2, 64, 32, seed=len(lens))
    inp["h0"] = np.random.default_rng(7).standard_normal((len(lens), 2, 64, 32)) * 0.1
    t, r = to_device(inp, gpu_device, torch.float32)
    o, ht = fused_recurrent_gdn2(*(t[n] for n in ("q", "k", "v", "g", "b", "w")), initial_state=t["h0"],
                                 output_final_state=True, use_qk_l2norm_in_kernel=True,
                                 cu_seqlens=torch.from_numpy(cu).to(gpu_device))
    o_ref, s_ref = orc.recurrent_fwd(r["q"], r["k"], r["v"], r["g"], r["b"], r["w"], r["h0"], cu_seqlens=cu)
    assert rel_l2(o, o_ref) <= 1e-5 and rel_l2(ht, s_ref) <= 1e-5

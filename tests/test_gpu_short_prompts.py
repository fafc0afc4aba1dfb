"""Token-serial kernel for sequences of several tokens (``recurrent_seq_kernel``) against the oracle:
tile edges of the token loop (16 tokens, 8 beyond d_k = 128), ragged key and value widths, and the
three column splits (few, some and many sequence-heads).  Few tokens of many heads, which the launch divides
between that kernel and the whole-row one (``recurrent_fwd_kernel``), on both sides of its rule."""

import numpy as np
import pytest
import torch

from oracle import gdn2_oracle as orc
from tests._helpers import REL_TOL, rand_inputs, rel_l2, to_device

pytestmark = pytest.mark.gpu


def _columns(heads, K, V):
    """16-column groups of a workgroup, as the launch picks them: the most that leave 256 workgroups."""
    for nc in (4, 2):
        if heads * -(-V // (16 * nc)) >= 256:
            return nc
    return 2 if K > 128 else 1


@pytest.mark.parametrize("B,T,H,HV,K,V,dtype,decay,nc", [
    (1, 2, 2, 2, 128, 128, torch.bfloat16, "paper", 1),
    (2, 16, 3, 3, 64, 64, torch.float32, "paper", 1),
    (1, 17, 2, 4, 128, 128, torch.float32, "unit", 1),
    (2, 33, 1, 1, 65, 20, torch.float32, "paper", 1),
    (1, 9, 2, 2, 200, 36, torch.float32, "unit", 2),
    (1, 64, 2, 2, 256, 128, torch.bfloat16, "paper", 2),
    (8, 31, 8, 8, 16, 48, torch.float16, "paper", 1),
    (4, 19, 16, 16, 128, 128, torch.float32, "paper", 2),
    (4, 17, 16, 16, 128, 100, torch.bfloat16, "unit", 2),
    (8, 16, 16, 16, 64, 64, torch.float32, "paper", 2),
    (8, 18, 8, 16, 40, 52, torch.bfloat16, "paper", 2),
    (16, 18, 16, 16, 128, 132, torch.bfloat16, "unit", 4),
    (16, 17, 16, 16, 64, 64, torch.float32, "paper", 4),
    (16, 9, 16, 16, 200, 36, torch.float32, "paper", 4),
    (2, 40, 2, 2, 128, 64, torch.float32, "sheer", 1),
])
def test_prompt_matches_oracle(gpu_device, B, T, H, HV, K, V, dtype, decay, nc):
    from qwendopamine_amd.ops import fused_recurrent_gdn2

    assert _columns(B * HV, K, V) == nc
    print(f"[case] prompt B={B} T={T} H={H} HV={HV} K={K} V={V} {dtype} {decay}", flush=True)
    t, r = to_device(rand_inputs(B, T, H, K, V, HV=HV, seed=T + K, decay=decay), gpu_device, dtype)
    o, ht = fused_recurrent_gdn2(*(t[n] for n in ("q", "k", "v", "g", "b", "w")), initial_state=t["h0"],
                                 output_final_state=True, use_qk_l2norm_in_kernel=True)
    o_ref, s_ref = orc.recurrent_fwd(r["q"], r["k"], r["v"], r["g"], r["b"], r["w"], r["h0"])
    assert rel_l2(o, o_ref) <= REL_TOL[dtype]
    # The state stays in float32 whatever the inputs' type.
    assert rel_l2(ht, s_ref) <= 1e-5


FEW = [  # N, lens, K, V of 16 heads
    (20, (2,), 128, 128),  # 320 sequence-heads: whole rows (one round of workgroups against two)
    (40, (2,), 128, 128),  # 640: whole rows (two against three)
    (40, (3,), 128, 128),  # 640 x 3: columns again
    (40, (2, 3), 128, 64), (32, (3, 1, 3), 96, 96), (64, (1, 3, 2), 64, 64),
    (20, (1, 2, 1, 3), 128, 128),  # fewer than two tokens on average
    (19, (2,) * 18 + (40,), 128, 128),  # one long sequence among short ones
]


@pytest.mark.parametrize("N,lens,K,V,packed", [(*c, p) for c in FEW for p in (False, True) if p or len(c[1]) == 1])
def test_few_tokens_of_many_heads(gpu_device, N, lens, K, V, packed):
    """Two or three tokens a sequence of many heads: which kernel runs depends on the rounds its workgroups take."""
    from qwendopamine_amd.ops import fused_recurrent_gdn2

    lens = (lens * N)[:N]
    print(f"[case] few tokens N={N} lens={lens[:4]}.. K={K} V={V} packed={packed}", flush=True)
    cu = np.concatenate([[0], np.cumsum(lens)])
    H, T = 16, int(cu[-1]) if packed else lens[0]
    inp = rand_inputs(1 if packed else N, T, H, K, V, seed=N + K)
    inp["h0"] = np.random.default_rng(N).standard_normal((N, H, K, V)) * 0.1
    t, r = to_device(inp, gpu_device, torch.float32)
    o, ht = fused_recurrent_gdn2(*(t[n] for n in ("q", "k", "v", "g", "b", "w")), initial_state=t["h0"],
                                 output_final_state=True, use_qk_l2norm_in_kernel=True,
                                 cu_seqlens=torch.from_numpy(cu).to(gpu_device) if packed else None)
    o_ref, s_ref = orc.recurrent_fwd(r["q"], r["k"], r["v"], r["g"], r["b"], r["w"], r["h0"],
                                     cu_seqlens=cu if packed else None)
    assert rel_l2(o, o_ref) <= 1e-5 and rel_l2(ht, s_ref) <= 1e-5


@pytest.mark.parametrize("N,width,lens,K,V", [
    (24, 4, (4, 2, 3), 128, 128),   # whole rows from the slot table's width
    (56, 3, (3,), 128, 128),        # whole rows: more than three rounds
    (20, 12, (2, 12, 5), 128, 128),  # columns
])
def test_few_pooled_tokens_of_many_heads(gpu_device, N, width, lens, K, V):
    from qwendopamine_amd.ops import fused_recurrent_gdn2_fwd

    lens = (lens * N)[:N]
    print(f"[case] pooled tokens N={N} width={width} K={K} V={V}", flush=True)
    rng = np.random.default_rng(N)
    cu = np.concatenate([[0], np.cumsum(lens)])
    slots = rng.permutation(N * width).reshape(N, width)
    pool = (rng.standard_normal((N * width, 16, K, V)) * 0.1).astype(np.float32)
    names = ("q", "k", "v", "g", "b", "w")
    t, r = to_device({n: x for n, x in rand_inputs(1, int(cu[-1]), 16, K, V, seed=N, h0_std=0).items() if x is not None},
                     gpu_device, torch.float32)
    dev = torch.from_numpy(pool).to(gpu_device)
    o, ht = fused_recurrent_gdn2_fwd(*(t[n] for n in names), initial_state=dev, inplace_final_state=True,
                                     cu_seqlens=torch.from_numpy(cu).to(gpu_device),
                                     ssm_state_indices=torch.from_numpy(slots).to(gpu_device),
                                     use_qk_l2norm_in_kernel=True)
    # Sequence by sequence: the oracle's states after every token.
    got = ht.cpu().numpy()
    touched = np.zeros(N * width, bool)
    for n in range(0, N, 7):
        S = pool[slots[n, 0]][None].astype(np.float64)
        for i in range(lens[n]):
            tok = slice(int(cu[n]) + i, int(cu[n]) + i + 1)
            o_ref, S = orc.recurrent_fwd(*(r[m][:, tok] for m in names), S)
            assert rel_l2(o[:, tok], o_ref) <= 1e-5
            assert rel_l2(got[slots[n, i]], S[0]) <= 1e-5
    for n in range(N):
        touched[slots[n, :lens[n]]] = True
    assert np.array_equal(got[~touched], pool[~touched])


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

"""The dispatch order of causal grids with at most 32 (batch, head) pairs and at least 256 workgroups, whose
blocks are dealt out longest first over all pairs: every causal kernel family, pairs that are and are not a
multiple of the XCDs, shared walks with and without the sorted order of their blocks. A block that is
missed or done twice in another's place shows in the whole outputs, against the CPU oracle."""
import pytest

import example_matmul_metal4_amd as mtk
import oracle

from test_attention_bwd_gpu import _check_pairs, _run_and_check
from test_attention_gpu import check

# H, H_kv, S_q, S_kv, D, q_rows, dtype, kernel
FORWARD = [(32, 32, 900, 900, 64, 0, "f16", "mtk_attn_fwd_d64_f16_causal"), (29, 29, 1100, 1000, 72, 0, "bf16", "mtk_attn_fwd_bf16_causal"),
           (32, 8, 1800, 1800, 64, 256, "f16", "mtk_attn_fwd_pp_d64_f16_causal"), (32, 32, 900, 500, 100, 0, "f16", "mtk_attn_fwd_g128_f16_causal"),
           (32, 32, 900, 1000, 136, 0, "f16", "mtk_attn_fwd_d256_f16_causal"), (16, 4, 1030, 900, 264, 0, "f16", "mtk_attn_fwd_d512_f16_causal")]
# H, H_kv, S_q, S_kv, D, dtype, dK/dV kernel, dQ kernel: the order is taken where the grid is that large
BACKWARD = [(16, 4, 1300, 1300, 64, "f16", "mtk_attn_bwd_dkdv_d64_f16_causal_shared", "mtk_attn_bwd_dq_d64_f16_causal_shared"),
            (20, 20, 1700, 1650, 64, "bf16", "mtk_attn_bwd_dkdv_d64_bf16_causal", "mtk_attn_bwd_dq_d64_bf16_causal"),
            (8, 8, 1900, 1900, 72, "f16", "mtk_attn_bwd_dkdv_f16_causal", "mtk_attn_bwd_dq_f16_causal_shared"),
            (16, 16, 1300, 1100, 136, "f16", "mtk_attn_bwd256_dkdv_f16_causal", "mtk_attn_bwd256_dq_f16_causal"),
            # more than 64 key or query blocks: shared walks whose blocks are not sorted by share
            (4, 1, 600, 8300, 64, "f16", "mtk_attn_bwd_dkdv_d64_f16_causal_shared", "mtk_attn_bwd_dq_d64_f16_causal_shared"),
            (2, 2, 16500, 1000, 40, "f16", "mtk_attn_bwd_dkdv_d64_f16_causal", "mtk_attn_bwd_dq_d64_f16_causal_shared")]


def _grids(text):
    return [int(x) for x in text.split("grids=")[1].split()[0].split("/")]


def test_cases_reach_the_order():
    # CPU: the planner alone
    for H, Hkv, Sq, Skv, D, q_rows, dtype, kern in FORWARD:
        text = mtk.AttentionPlan(None, 1, H, Sq, Skv, D, causal=True, dtype=dtype, q_rows=q_rows, H_kv=Hkv).describe()
        assert text.endswith("kernels: " + kern) and H <= 32 and int(text.split(" grid=")[1].split()[0]) >= 256, text
    kv = q = 0
    for H, Hkv, Sq, Skv, D, dtype, kern_kv, kern_q in BACKWARD:
        text = mtk.AttentionBwdPlan(None, 1, H, Sq, Skv, D, causal=True, dtype=dtype, H_kv=Hkv).describe()
        names, (_, g_kv, g_q) = text.split("kernels: ")[1].split(), _grids(text)
        assert names[1] == kern_kv and names[2] == kern_q and H <= 32 and max(g_kv, g_q) >= 256, text
        # 1: whole walks, 4: shared ones, 8: shared and not sorted
        kv |= (g_kv >= 256) << (2 * kern_kv.endswith("_shared") + ((Skv + 127) // 128 > 64))
        q |= (g_q >= 256) << (2 * kern_q.endswith("_shared") + ((Sq + 255) // 256 > 64))
    assert kv == 13 and q == 13, (kv, q)


@pytest.mark.gpu
@pytest.mark.parametrize("case", FORWARD, ids=str)
def test_forward(dev, case):
    H, Hkv, Sq, Skv, D, q_rows, dtype, _ = case
    Q = oracle.normal(60, (1, Sq, H, D), 0, 1, dtype)
    K, V = (oracle.normal(s, (1, Skv, Hkv, D), 0, 1, dtype) for s in (61, 62))
    check(dev, Q, K, V, True, dtype, label=str(case), q_rows=q_rows)


@pytest.mark.gpu
@pytest.mark.parametrize("case", BACKWARD, ids=str)
def test_backward(dev, case):
    H, Hkv, Sq, Skv, D, dtype = case[:6]
    group = H // Hkv
    if group == 1:
        _run_and_check(dev, 1, H, Sq, Skv, True, dtype, D=D, pairs=[(i, min(i + 4, H)) for i in range(0, H, 4)])
        return
    Q, G = (oracle.normal(s, (1, Sq, H, D), dtype=dtype) for s in (90, 93))
    K, V = (oracle.normal(s, (1, Skv, Hkv, D), dtype=dtype) for s in (91, 92))
    O, lse = mtk.attention(dev, Q, K, V, causal=True, dtype=dtype, return_lse=True)
    got = mtk.attention_bwd(dev, Q, K, V, O, G, lse, causal=True, dtype=dtype)
    exp = oracle.attention_bwd(Q, K, V, G, causal=True, dtype=dtype)[:3]
    _check_pairs(Q, K, V, G, *got, *exp, True, dtype, group, None, H)

"""Attention backward plans whose long walks are shared by several workgroups (grouped K/V heads, few
key or query blocks): the shares' partial sums, against the CPU oracle of the reference's gradients
(Network.swift:205-281, 313-402) with the acceptance of test_attention_bwd_gpu."""
import numpy as np
import pytest

import example_matmul_metal4_amd as mtk
import oracle

from test_attention_bwd_gpu import _check_pairs

# (B, H, H_kv, S_q, S_kv, D, causal, dtype, dK/dV shared, dQ shared)
CASES = [
    (1, 8, 1, 333, 300, 128, False, "f16", True, False), (1, 16, 2, 400, 417, 64, True, "bf16", True, False),
    (2, 12, 1, 257, 200, 72, True, "f16", True, False), (1, 2, 1, 1100, 1090, 128, True, "f16", True, True),
    (1, 1, 1, 300, 1500, 96, False, "bf16", False, True), (1, 1, 1, 1601, 1400, 64, True, "f16", False, True),
    (1, 1, 1, 2200, 130, 128, False, "f16", True, False), (1, 6, 2, 1030, 1025, 40, False, "f16", True, True),
    (1, 4, 1, 1200, 640, 128, True, "f16", True, False),  # queries that see no key
]


def _plan(dev, case):
    B, H, Hkv, Sq, Skv, D, causal, dtype = case[:8]
    return mtk.AttentionBwdPlan(dev, B, H, Sq, Skv, D, causal=causal, dtype=dtype, H_kv=Hkv)


def _grids(plan):
    return [int(x) for x in plan.describe().split("grids=")[1].split()[0].split("/")]


def test_which_plans_are_shared():
    # CPU: the planner alone
    for c in CASES:
        B, H, Hkv, Sq, Skv = c[:5]
        _, kv, q = _grids(_plan(None, c))
        assert (kv > (Skv + 127) // 128 * B * Hkv) == c[8], (c, kv)
        assert (q > (Sq + 255) // 256 * B * H) == c[9], (c, q)
    # grids that fill the device with equal or short walks are not
    for a in ((2, 32, 4096, 4096, 128), (2, 32, 512, 512, 64)):
        assert "bwd_sum" not in mtk.AttentionBwdPlan(None, *a).describe()


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_shared_walks(dev, case):
    B, H, Hkv, Sq, Skv, D, causal, dtype = case[:8]
    print(f"[attn bwd shared] {_plan(dev, case).describe()}", flush=True)
    Q, G = (oracle.normal(s, (B, Sq, H, D), dtype=dtype) for s in (70, 73))
    K, V = (oracle.normal(s, (B, Skv, Hkv, D), dtype=dtype) for s in (71, 72))
    O, lse = mtk.attention(dev, Q, K, V, causal=causal, dtype=dtype, return_lse=True)
    got = mtk.attention_bwd(dev, Q, K, V, O, G, lse, causal=causal, dtype=dtype)
    again = mtk.attention_bwd(dev, Q, K, V, O, G, lse, causal=causal, dtype=dtype)
    assert all(np.array_equal(x.view(np.uint16), y.view(np.uint16)) for x, y in zip(got, again))
    exp = oracle.attention_bwd(Q, K, V, G, causal=causal, dtype=dtype)[:3]
    _check_pairs(Q, K, V, G, *got, *exp, causal, dtype, H // Hkv, None, H)

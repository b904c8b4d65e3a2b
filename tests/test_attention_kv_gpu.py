"""Attention calls whose keys are split over wavefronts (and, behind a long cache, over workgroups):
few queries, or one short sequence. Whole outputs against the CPU oracle (Network.swift:134-179,
286-311) with the acceptance of test_attention_gpu.check; the row log-sum-exp against float64."""
import ctypes

import numpy as np
import pytest

import example_matmul_metal4_amd as mtk
import oracle

from test_attention_gpu import check

# (B, H, H_kv, S_q, S_kv, D, causal, dtype): rows and keys at, below and past the 32-row and 32-key
# blocks, fewer key tiles than wavefronts, queries that see no key, every output-block width, partial
# d blocks
CASES = [
    (1, 1, 1, 1, 97, 128, False, "f16"), (2, 4, 4, 1, 129, 64, False, "f16"), (1, 8, 2, 1, 255, 128, True, "bf16"),
    (3, 8, 2, 7, 257, 96, True, "f16"), (1, 16, 2, 4, 700, 80, False, "bf16"), (2, 6, 6, 31, 640, 40, True, "f16"),
    (1, 4, 4, 1500, 1030, 64, True, "f16"), (2, 8, 4, 16, 100, 256, True, "f16"), (1, 4, 1, 9, 900, 200, False, "bf16"),
    (16, 16, 16, 1, 300, 128, False, "f16"), (1, 8, 8, 800, 800, 128, True, "f16"), (1, 16, 8, 513, 1030, 64, False, "bf16"),
    # keys split over workgroups: an uneven last split, splits past the causal end, 33 rows
    (1, 8, 2, 1, 4097, 128, False, "f16"), (2, 4, 1, 3, 2500, 64, True, "bf16"), (1, 11, 1, 3, 6000, 128, True, "f16"),
    (1, 8, 8, 1, 3333, 256, False, "bf16"), (1, 2, 1, 40, 1600, 72, True, "f16"),
]
SPLIT = CASES[12:]


def _plan(dev, case):
    B, H, Hkv, Sq, Skv, D, causal, dtype = case
    return mtk.AttentionPlan(dev, B, H, Sq, Skv, D, causal=causal, dtype=dtype, H_kv=Hkv)


def _inputs(case, seed=40):
    B, H, Hkv, Sq, Skv, D, causal, dtype = case
    return (oracle.normal(seed, (B, Sq, H, D), 0, 1, dtype), oracle.normal(seed + 1, (B, Skv, Hkv, D), 0, 1, dtype),
            oracle.normal(seed + 2, (B, Skv, Hkv, D), 0, 1, dtype))


def test_cases_take_the_key_split_kernels():
    # CPU: the planner alone
    for c in CASES:
        assert "mtk_attn_kv_d" in _plan(None, c).describe(), c
        assert ("mtk_attn_kv_combine_" in _plan(None, c).describe()) == (c in SPLIT), (c, _plan(None, c).describe())
    # an explicit block of query rows, rows that are not 16-byte aligned, fewer than four key tiles, a
    # last round of few workgroups and grids of 128-query blocks keep their kernels
    assert "mtk_attn_kv" not in mtk.AttentionPlan(None, 8, 32, 1, 96, 128, H_kv=8).describe()
    assert "mtk_attn_kv" not in mtk.AttentionPlan(None, 19, 16, 1, 1938, 128).describe()
    assert "mtk_attn_kv" not in mtk.AttentionPlan(None, 8, 32, 1, 4096, 128, H_kv=8, q_rows=128).describe()
    assert "mtk_attn_fwd_g128" in mtk.AttentionPlan(None, 8, 32, 1, 4096, 100).describe()
    assert "mtk_attn_kv" not in mtk.AttentionPlan(None, 4, 32, 1024, 1024, 128).describe()


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_key_split_parity(dev, case):
    B, H, Hkv, Sq, Skv, D, causal, dtype = case
    Q, K, V = _inputs(case)
    got, _ = check(dev, Q, K, V, causal, dtype, label=str(case))
    again, lse = mtk.attention(dev, Q, K, V, causal=causal, dtype=dtype, return_lse=True)
    assert np.array_equal(np.ascontiguousarray(got).view(np.uint16), np.ascontiguousarray(again).view(np.uint16))
    q = oracle.to_f32(Q, dtype).astype(np.float64).transpose(0, 2, 1, 3)
    k = np.repeat(oracle.to_f32(K, dtype).astype(np.float64), H // Hkv, 2).transpose(0, 2, 3, 1)
    s = (q @ k) / np.sqrt(D)
    if causal:
        s = np.where(np.arange(Skv)[None, :] > np.arange(Sq)[:, None] + Skv - Sq, -np.inf, s)
    with np.errstate(divide="ignore", invalid="ignore"):
        m = np.maximum(s.max(-1, keepdims=True), -1e300)
        exp = np.log(np.exp(s - m).sum(-1)) + m[..., 0]
    dead = ~np.isfinite(s).any(-1)
    assert np.array_equal(np.isneginf(lse), dead)
    # fp32 scores (D products) and a sum of at most S_kv weights
    assert np.all(np.abs(lse[~dead] - exp[~dead]) <= 2e-5 * (1 + np.abs(exp[~dead])))


@pytest.mark.gpu
@pytest.mark.parametrize("case", SPLIT, ids=str)
def test_split_keys_in_graphs_and_on_other_streams(dev, case):
    # the same bits from an eager call, from a graph (which has partial sums of its own), on a stream that is
    # not the context's own and in a caller's capture of one (where one workgroup walks the splits)
    B, H, Hkv, Sq, Skv, D, causal, dtype = case
    plan = _plan(dev, case)
    Q, K, V = _inputs(case)
    bufs = [dev.upload(x) for x in (Q, K, V)]
    outs = [dev.empty(Q.nbytes) for _ in range(3)]
    lses = [dev.empty(4 * B * H * Sq) for _ in range(2)]
    read = lambda o: dev.download(o, Q.shape, np.uint16)
    plan.run(*bufs, outs[0], lses[0])
    dev.sync()
    ref, ref_lse = read(outs[0]), dev.download(lses[0], (B, H, Sq), np.uint32)
    g = plan.graph([plan.args(*bufs, outs[1])], steps=3)
    try:
        for _ in range(3):
            dev.upload_into(outs[1], np.full(Q.shape, 0x7E00, np.uint16))
            g.launch()
            plan.run(*bufs, outs[0])
            dev.sync()
            assert np.array_equal(read(outs[1]), ref) and np.array_equal(read(outs[0]), ref)
    finally:
        g.close()
    hip = ctypes.CDLL("libamdhip64.so.7")  # the runtime that the library has loaded
    stream = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0  # non-blocking
    graph, graph_exec = ctypes.c_void_p(), ctypes.c_void_p()
    poison = lambda: (dev.upload_into(outs[2], np.full(Q.shape, 0x7E00, np.uint16)),
                      dev.upload_into(lses[1], np.zeros((B, H, Sq), np.uint32)))
    same = lambda: (np.array_equal(read(outs[2]), ref) and
                    np.array_equal(dev.download(lses[1], (B, H, Sq), np.uint32), ref_lse))
    mtk._check(mtk.lib().mtk_set_stream(dev.handle, stream))
    try:
        poison()
        plan.run(*bufs, outs[2], lses[1])
        dev.sync()
        assert same(), "another stream"
        assert hip.hipStreamBeginCapture(stream, 2) == 0  # relaxed
        plan.run(*bufs, outs[2], lses[1])
        assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        assert hip.hipGraphInstantiate(ctypes.byref(graph_exec), graph, None, None, ctypes.c_size_t(0)) == 0
        for _ in range(3):
            poison()
            assert hip.hipGraphLaunch(graph_exec, stream) == 0
            dev.sync()
            assert same(), "a captured call"
    finally:
        mtk._check(mtk.lib().mtk_set_stream(dev.handle, None))
        for destroy, x in (("hipGraphExecDestroy", graph_exec), ("hipGraphDestroy", graph), ("hipStreamDestroy", stream)):
            if x:
                getattr(hip, destroy)(x)
    for x in bufs + outs + lses:
        x.free()

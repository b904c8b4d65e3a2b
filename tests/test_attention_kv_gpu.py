"""Attention calls whose keys are split over wavefronts (and, behind a long cache, over workgroups):
few queries, or one short sequence. Whole outputs against the CPU oracle (Network.swift:134-179,
286-311) with the acceptance of test_attention_gpu.check; the row log-sum-exp against float64."""
import ctypes
import threading

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
    # not the context's own and in a caller's capture of one
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


def _hip():
    return ctypes.CDLL("libamdhip64.so.7")  # the runtime that the library has loaded


class _Stream:
    """A non-blocking stream of the caller's, current in the context while entered."""

    def __init__(self, dev):
        self.dev, self.handle = dev, ctypes.c_void_p()
        assert _hip().hipStreamCreateWithFlags(ctypes.byref(self.handle), 1) == 0

    def __enter__(self):
        mtk._check(mtk.lib().mtk_set_stream(self.dev.handle, self.handle))
        return self

    def __exit__(self, *exc):
        mtk._check(mtk.lib().mtk_set_stream(self.dev.handle, None))

    def close(self):
        assert _hip().hipStreamSynchronize(self.handle) == 0 and _hip().hipStreamDestroy(self.handle) == 0


class _Case:
    """A plan on inputs of its own, an output buffer and the eager result on the context's own stream."""

    def __init__(self, dev, case, seed):
        self.dev, self.plan = dev, _plan(dev, case)
        Q, K, V = _inputs(case, seed)
        self.shape, self.bufs = Q.shape, [dev.upload(x) for x in (Q, K, V)] + [dev.empty(Q.nbytes)]
        self.run()
        dev.sync()
        self.ref = self.read()

    def run(self):
        self.plan.run(*self.bufs)

    def poison(self):
        self.dev.upload_into(self.bufs[3], np.full(self.shape, 0x7E00, np.uint16))

    def read(self):
        return self.dev.download(self.bufs[3], self.shape, np.uint16).copy()

    def close(self):
        for b in self.bufs:
            b.free()


@pytest.mark.gpu
def test_streams_and_captures_have_regions_of_their_own():
    # more streams and captures than there are regions, all at work at once: every result is that of the
    # context's own stream, also once the streams have gone and others take their regions
    dev = mtk.Device(0)  # the captures' regions stay taken in a context
    cases = [_Case(dev, SPLIT[i % len(SPLIT)], 300 + 10 * i) for i in range(20)]
    hip = _hip()
    for _ in range(2):
        streams = [_Stream(dev) for _ in cases]
        for c in cases:
            c.poison()
        for _ in range(3):
            for c, st in zip(cases, streams):
                with st:
                    c.run()
        for st in streams:
            st.close()
        assert all(np.array_equal(c.read(), c.ref) for c in cases)
    st = _Stream(dev)
    with st:
        names = cases[0].plan.profile([cases[0].plan.args(*cases[0].bufs)], warmup=1, iters=2)["kernels"]
    assert any("combine" in n for n in names), names  # the splits are shared out on an external stream too
    graphs = []
    try:
        for c in cases:
            g, e = ctypes.c_void_p(), ctypes.c_void_p()
            with st:
                assert hip.hipStreamBeginCapture(st.handle, 2) == 0  # relaxed
                c.run()
                c.run()
                assert hip.hipStreamEndCapture(st.handle, ctypes.byref(g)) == 0
            assert hip.hipGraphInstantiate(ctypes.byref(e), g, None, None, ctypes.c_size_t(0)) == 0
            graphs.append((g, e))
        others = [_Stream(dev) for _ in range(4)]
        for _ in range(3):
            for c in cases:
                c.poison()
            for i, (_, e) in enumerate(graphs):
                assert hip.hipGraphLaunch(e, others[i % 4].handle) == 0
            for o in others:
                assert hip.hipStreamSynchronize(o.handle) == 0
            assert all(np.array_equal(c.read(), c.ref) for c in cases)
            for c in cases:  # eager calls between the replays
                c.run()
            dev.sync()
        for o in others:
            o.close()
    finally:
        for g, e in graphs:
            hip.hipGraphExecDestroy(e)
            hip.hipGraphDestroy(g)
        st.close()
        for c in cases:
            c.close()
        dev.close()


@pytest.mark.gpu
def test_two_threads_on_one_context(dev):
    # kernels of two threads' calls on the context's own stream do not interleave on its partial sums
    cases = [_Case(dev, SPLIT[i], 500 + 10 * i) for i in (0, 3)]
    errors = []

    def work(c):
        try:
            for _ in range(200):
                c.run()
        except Exception as e:  # noqa: BLE001 - reported below
            errors.append(e)

    for c in cases:
        c.poison()
    threads = [threading.Thread(target=work, args=(c,)) for c in cases]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    dev.sync()
    assert not errors, errors
    for c in cases:
        assert np.array_equal(c.read(), c.ref)
        c.close()


@pytest.mark.gpu
def test_launches_do_not_allocate(dev):
    # what a plan needs is there when it has been created: the first call of a new context takes no memory
    hip = _hip()

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    own = mtk.Device(0)
    try:
        Q, K, V = _inputs(SPLIT[0])
        bufs = [own.upload(x) for x in (Q, K, V)] + [own.empty(Q.nbytes)]
        small = mtk.AttentionPlan(own, 1, 8, 1, 255, 128, H_kv=2)  # another kernel of the same code object first
        small.run(*bufs)
        plan = _plan(own, SPLIT[0])
        own.sync()
        before = free()
        plan.run(*bufs)
        own.sync()
        assert free() == before
        for b in bufs:
            b.free()
    finally:
        own.close()


@pytest.mark.gpu
@pytest.mark.parametrize("case", [CASES[3], CASES[10], SPLIT[0], SPLIT[1], SPLIT[3]], ids=str)
def test_values_that_are_not_finite(dev, case):
    # what is not finite reaches the rows and dims that read it and no others, and rows whose scores all lie
    # far below any weight's range are still averaged
    B, H, Hkv, Sq, Skv, D, causal, dtype = case
    G = H // Hkv
    Q, K, V = (oracle.to_f32(x, dtype) for x in _inputs(case, 640))
    run = lambda q, k, v: mtk.attention(dev, *(oracle.from_f32(x, dtype) for x in (q, k, v)), causal=causal, dtype=dtype,
                                        return_lse=True)
    f = lambda x: oracle.to_f32(x, dtype)
    O, lse = run(Q, K, V)
    # a NaN and an infinity in one query row each: those rows only
    q, rows = Q.copy(), [(0, Sq - 1, 0), (B - 1, Sq - 1, H - 1)]
    q[rows[0]][D // 2], q[rows[1]][0] = np.nan, np.inf
    o, l = run(q, K, V)
    bad = np.zeros((B, Sq, H), bool)
    for r in rows:
        bad[r] = True
    assert np.all(np.isnan(f(o))[bad]) and np.array_equal(o.view(np.uint16)[~bad], O.view(np.uint16)[~bad])
    assert np.array_equal(l.transpose(0, 2, 1)[~bad], lse.transpose(0, 2, 1)[~bad])
    # an infinity and a NaN in V at the last key: one dim each, of the rows that see it (the last queries) and of
    # no row of another K/V head
    v = V.copy()
    v[0, Skv - 1, 0, 1], v[0, Skv - 1, 0, 3] = np.inf, np.nan
    o = f(run(Q, K, v)[0])
    assert not np.isfinite(o[0, Sq - 1, :G, 1]).any() and np.isnan(o[0, Sq - 1, :G, 3]).all()
    other = np.ones(O.shape, bool)
    other[0, :, :G, [1, 3]] = False
    assert np.array_equal(o[other], f(O)[other])
    # equal scores of about -2e7: every weight of a row is the same
    q, k = np.zeros_like(Q), np.zeros_like(K)
    q[..., 0], k[..., 0] = 6e4, -3750
    o, _ = run(q, k, V)
    exp = oracle.attention(*(oracle.from_f32(x, dtype) for x in (np.zeros_like(Q), k, V)), causal=causal, dtype=dtype)
    # equal weights up to a rounding each (16 bits), and the output's
    bound = oracle.ulp(exp, dtype) + 2 * (2.0 ** -11 if dtype == "f16" else 2.0 ** -8) * oracle.attention(
        *(oracle.from_f32(x, dtype) for x in (np.zeros_like(Q), k, np.abs(V))), causal=causal, dtype=dtype)
    assert np.all(np.abs(f(o) - exp) <= bound), np.abs(f(o) - exp).max()


def test_second_rounds_take_the_faster_kernel():
    # CPU: the planner alone. One key-split workgroup fits a CU: calls with a second round of them need long walks,
    # and most calls with more rounds, or short second ones, keep the 128-query kernel
    name = lambda *a, **kw: mtk.AttentionPlan(None, *a, **kw).describe().split("kernels: ")[1].split()[0]
    causal, uncausal = dict(causal=True), {}
    for a, kw, split in (
            # above D 128
            ((6, 4, 557, 557, 256), uncausal, False), ((3, 2, 3700, 3700, 256), uncausal, False),
            ((1, 8, 1024, 735, 256), uncausal, False), ((1, 8, 1024, 740, 256), uncausal, True),
            ((1, 8, 1000, 1000, 256), causal, True), ((1, 8, 1024, 490, 256), causal, True),
            ((1, 8, 1500, 1500, 256), causal, True), ((1, 8, 1500, 1500, 256), uncausal, False),
            ((1, 8, 1500, 1500, 256), dict(causal=True, H_kv=2), False), ((1, 8, 1200, 1800, 256), causal, False),
            ((1, 8, 1800, 1800, 256), causal, False), ((1, 8, 1712, 2622, 256), dict(causal=True, H_kv=1), False),
            # D 128
            ((4, 8, 490, 490, 128), causal, False), ((4, 8, 512, 740, 128), causal, True),
            ((3, 8, 480, 490, 128), causal, True), ((3, 16, 238, 238, 128), dict(H_kv=4), False),
            ((12, 32, 1, 370, 96), uncausal, False), ((12, 32, 1, 420, 96), uncausal, True),
            ((12, 32, 1, 370, 96), dict(H_kv=8), True), ((12, 32, 1, 370, 128), uncausal, True),
            ((12, 32, 1, 370, 128), causal, False)):
        assert name(*a, **kw).startswith("mtk_attn_kv_") == split, (a, kw, name(*a, **kw))

"""The work that a user of this library has it do, as cases that can be timed and checked.

Every case goes through the public Python entry points (plans, `args`, `launch`) on device buffers
that the caller holds. Sizes are this repository's benchmark configurations, the sizes of its tests
(the reference's own sweeps) and generic layer sizes in between; `draw` spreads over the same ranges.
"""
import math

import torch

import example_matmul_metal4_amd as mtk

_TORCH = {"f16": torch.float16, "bf16": torch.bfloat16}
_DEVICE = None


def _device():
    global _DEVICE
    if _DEVICE is None:
        _DEVICE = mtk.Device(0)
    return _DEVICE


# ------------------------------------------------------------------ the cases


def _gemm(name, M, N, K, dtype="f16", layout="nt", bias=True, split_k=0):
    c = {"op": "gemm", "M": M, "N": N, "K": K, "dtype": dtype, "layout": layout, "bias": bias, "split_k": split_k}
    return {"name": name, **c} if name else c


def _conv(name, rank, N, D, H, W, C, O, kd, k, stride=1, pad=0, bias=True, weights="DHWIO"):
    c = {"op": "conv", "rank": rank, "N": N, "D": D, "H": H, "W": W, "C": C, "O": O, "kd": kd, "k": k,
         "stride": stride, "pad": pad, "bias": bias, "weights": weights}
    return {"name": name, **c} if name else c


def _attn(name, B, H, H_kv, S_q, S_kv, D, causal, dtype="f16", backward=False):
    c = {"op": "attn_train" if backward else "attn", "B": B, "H": H, "H_kv": H_kv, "S_q": S_q, "S_kv": S_kv, "D": D,
         "causal": causal, "dtype": dtype}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest product of the benchmark configurations (256 cubed, both operands row-major):
        # a single small layer or head, where a call's latency is what is felt
        _gemm("gemm_256_nn", 256, 256, 256, layout="nn", bias=False, split_k=1),
        # one decode step's up projection for 16 sequences: weights streamed once
        _gemm("gemm_decode_16", 16, 14336, 4096, dtype="bf16", split_k=8),
        # the down projection of a 77-token prompt: between decode and prefill, ragged M, the plan's
        # own choice of split
        _gemm("gemm_prompt_77", 77, 4096, 14336, dtype="bf16"),
        # the headline configuration: square, K with a tail, split-K 4 with bias
        _gemm("gemm_4096_k4100", 4096, 4096, 4100, split_k=4),
        # the reference's correctness sweep runs M = N = K over every size: odd rows, where no row but
        # the first is aligned to more than an element
        _gemm("gemm_odd_1023", 1023, 1023, 1023, split_k=1),
        # a 3x3 layer of a large vision model, batch 8 (benchmark configuration 4a)
        _conv("conv2d_256ch", 2, 8, 1, 128, 128, 256, 256, 1, 3, pad=1),
        # the reference's published small conv2d (128x128, 32 channels in and out): early layers
        _conv("conv2d_32ch", 2, 1, 1, 128, 128, 32, 32, 1, 3, pad=1),
        # a video layer (benchmark configuration 4b) with weights as PyTorch stores them, re-laid out
        # in each run as the reference's permute-then-convolve session does
        _conv("conv3d_oidhw", 3, 1, 16, 64, 64, 128, 128, 3, 3, pad=1, weights="OIDHW"),
        # causal prefill at the benchmark's attention shape with 8 grouped K/V heads
        _attn("attn_prefill_causal", 2, 32, 8, 4096, 4096, 128, True),
        # one decode step over a 4096-token cache: one query per sequence, grouped K/V heads
        _attn("attn_decode_8x4096", 8, 32, 8, 1, 4096, 128, False, dtype="bf16"),
        # one short ragged sequence with 8 heads (the reference's own sweep ends at 1023 keys)
        _attn("attn_short_1023", 1, 8, 8, 1023, 1023, 128, False),
        # an attention layer's training step: forward with the row log-sum-exp, then the gradients
        _attn("attn_train_causal", 2, 32, 8, 2048, 2048, 128, True, backward=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """A size between lo and hi, spread over the logarithm: mostly multiples of 64, some of 8, some odd."""
    n = _log(rng, lo, hi)
    step = rng.choice([64, 64, 64, 8, 2, 1])
    return max(lo, min(hi, n // step * step))


def _draw(rng):
    op = rng.choice(["gemm", "gemm", "gemm", "conv", "conv", "attn", "attn", "train"])
    if op == "gemm":
        layout = rng.choice(["nt", "nt", "nt", "nn", "tt", "tn"])
        M = _log(rng, 1, 4096)
        if layout[0] == "t":
            M = (M + 1) // 2 * 2  # transposed A takes even rows
        N, K = _size(rng, 64, 16384), _size(rng, 64, 16384)
        return _gemm(None, M, N, K, rng.choice(["f16", "bf16"]), layout, rng.random() < 0.7, rng.choice([0, 0, 1, 4]))
    if op == "conv":
        rank = rng.choice([2, 2, 3])
        C = rng.choice([3, 16, 32, 40, 64, 96, 128, 256, 512])
        O = rng.choice([16, 32, 64, 72, 128, 200, 256, 512])
        k = rng.choice([1, 3, 3, 3, 5] if rank == 2 else [1, 3, 3])
        return _conv(None, rank, _log(rng, 1, 8), 1 if rank == 2 else _log(rng, 3, 16), _log(rng, 14, 256),
                     _log(rng, 14, 256), C, O, 1 if rank == 2 else k, k, rng.choice([1, 1, 1, 2]),
                     rng.choice([0, k // 2, k // 2]), rng.random() < 0.7, rng.choice(["DHWIO", "DHWIO", "DHWIO", "OIDHW"]))
    H_kv = rng.choice([1, 2, 4, 8])
    H = H_kv * rng.choice([1, 1, 4, 8])
    B, D = _log(rng, 1, 16), rng.choice([64, 64, 80, 96, 128, 128, 128, 256])
    dtype = rng.choice(["f16", "f16", "bf16"])
    S_kv = _log(rng, 64, 16384)
    if op == "attn":
        # prefill, a few new tokens behind a cache, or one
        S_q = rng.choice([S_kv, S_kv, _log(rng, 1, 64), 1])
        return _attn(None, B, H, H_kv, min(S_q, S_kv), S_kv, D, rng.random() < 0.5, dtype)
    S = min(S_kv, 4096)
    return _attn(None, B, H, H_kv, S, S, D, rng.random() < 0.7, dtype, backward=True)


def draw(rng):
    """One more case of these ranges, no larger than the largest listed one."""
    while True:
        c = _draw(rng)
        w = work(c)
        most = 8e10
        if c["op"] == "gemm" and (c["K"] % 2 or c["N"] % 2) or c["op"] == "conv" and c["C"] % 64:
            most = 1e10  # rows that are not aligned
        if w["flops"] <= most and w["bytes"] <= 4e8:
            return c


# ------------------------------------------------------------------ inputs and passes


def _normal(g, shape, std, dtype):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std).to(_TORCH[dtype])


def _uniform(g, shape, lo, hi, dtype):
    return (torch.rand(shape, generator=g, device="cuda", dtype=torch.float32) * (hi - lo) + lo).to(_TORCH[dtype])


def _conv_dims(c):
    """(depth, height, width) of the output; only rank 3 pads the depth."""
    pd = c["pad"] if c["rank"] == 3 else 0
    sd = c["stride"] if c["rank"] == 3 else 1
    return ((c["D"] + 2 * pd - c["kd"]) // sd + 1, (c["H"] + 2 * c["pad"] - c["k"]) // c["stride"] + 1,
            (c["W"] + 2 * c["pad"] - c["k"]) // c["stride"] + 1)


def _inputs(c, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    if c["op"] == "gemm":
        M, N, K, dt = c["M"], c["N"], c["K"], c["dtype"]
        std = 1 / math.sqrt(K)
        return {"A": _normal(g, (M, K) if c["layout"][0] == "n" else (K, M), 1.0, dt),
                "B": _normal(g, (N, K) if c["layout"][1] == "t" else (K, N), std, dt),
                "bias": _uniform(g, (N,), -0.5, 0.5, dt) if c["bias"] else None}
    if c["op"] == "conv":
        taps = c["kd"] * c["k"] * c["k"]
        w = (c["kd"], c["k"], c["k"], c["C"], c["O"]) if c["weights"] == "DHWIO" else (c["O"], c["C"], c["kd"], c["k"], c["k"])
        return {"x": _uniform(g, (c["N"], c["D"], c["H"], c["W"], c["C"]), -1, 1, "f16"),
                "w": _normal(g, w, 1 / math.sqrt(taps * c["C"]), "f16"),
                "bias": _uniform(g, (c["O"],), -0.5, 0.5, "f16") if c["bias"] else None}
    q, kv, dt = (c["B"], c["S_q"], c["H"], c["D"]), (c["B"], c["S_kv"], c["H_kv"], c["D"]), c["dtype"]
    t = {"Q": _normal(g, q, 1.0, dt), "K": _normal(g, kv, 1.0, dt), "V": _normal(g, kv, 1.0, dt)}
    if c["op"] == "attn_train":
        t["dO"] = _normal(g, q, 1.0, dt)
    return t


def _p(t):
    return None if t is None else t.data_ptr()


def _workspace(plan):
    return torch.empty(plan.workspace_bytes, dtype=torch.uint8, device="cuda") if plan.workspace_bytes else None


def prepare(case, seed):
    """What a program holds before the call: inputs, output buffers, the plan and its workspace."""
    dev, c, t = _device(), case, _inputs(case, seed)
    new = lambda *shape: torch.empty(shape, dtype=_TORCH[c.get("dtype", "f16")], device="cuda")
    if c["op"] == "gemm":
        plan = mtk.GemmPlan(dev, c["M"], c["N"], c["K"], trans_a=c["layout"][0] == "t", trans_b=c["layout"][1] == "t",
                            dtype=c["dtype"], has_bias=c["bias"], split_k=c["split_k"])
        ws, out = _workspace(plan), {"C": new(c["M"], c["N"])}
        steps = [(plan, plan.args(_p(t["A"]), _p(t["B"]), _p(t["bias"]), _p(out["C"]), _p(ws)))]
    elif c["op"] == "conv":
        r3 = c["rank"] == 3
        pd, sd = (c["pad"], c["stride"]) if r3 else (0, 1)
        desc = mtk.ConvDesc(rank=c["rank"], N=c["N"], D=c["D"], H=c["H"], W=c["W"], C=c["C"], O=c["O"], KD=c["kd"],
                            KH=c["k"], KW=c["k"], stride_d=sd, stride_h=c["stride"], stride_w=c["stride"], dil_d=1,
                            dil_h=1, dil_w=1, pad_front=pd, pad_back=pd, pad_top=c["pad"], pad_bottom=c["pad"],
                            pad_left=c["pad"], pad_right=c["pad"], has_bias=int(c["bias"]), dtype=mtk.F16,
                            weight_layout=mtk.WEIGHTS_OIDHW if c["weights"] == "OIDHW" else mtk.WEIGHTS_DHWIO)
        plan = mtk.ConvPlan(dev, desc)
        ws, out = _workspace(plan), {"y": new(c["N"], *_conv_dims(c), c["O"])}
        steps = [(plan, plan.args(_p(t["x"]), _p(t["w"]), _p(t["bias"]), _p(out["y"]), _p(ws)))]
    else:
        shape = (dev, c["B"], c["H"], c["S_q"], c["S_kv"], c["D"])
        opts = {"causal": c["causal"], "dtype": c["dtype"], "H_kv": c["H_kv"]}
        plan = mtk.AttentionPlan(*shape, **opts)
        ws, out = _workspace(plan), {"O": new(*t["Q"].shape)}
        if c["op"] == "attn_train":
            out["lse"] = torch.empty((c["B"], c["H"], c["S_q"]), dtype=torch.float32, device="cuda")
            out.update(dQ=new(*t["Q"].shape), dK=new(*t["K"].shape), dV=new(*t["V"].shape))
        steps = [(plan, plan.args(_p(t["Q"]), _p(t["K"]), _p(t["V"]), _p(out["O"]), _p(out.get("lse"))))]
        if c["op"] == "attn_train":
            bwd = mtk.AttentionBwdPlan(*shape, **opts)
            ws = _workspace(bwd)
            steps.append((bwd, bwd.args(_p(t["Q"]), _p(t["K"]), _p(t["V"]), _p(out["O"]), _p(t["dO"]), _p(out["lse"]),
                                        _p(out["dQ"]), _p(out["dK"]), _p(out["dV"]), _p(ws))))
    torch.cuda.synchronize()  # the inputs were made on torch's stream, the plans run on the library's
    return {"steps": steps, "out": out, "inputs": t, "workspace": ws}


def run(state):
    for plan, args in state["steps"]:
        plan.launch(args)
    return state["out"]


# ------------------------------------------------------------------ work, tolerance, 64-bit results


def _pairs(c):
    """Query-key pairs that the mask keeps (bottom-right aligned)."""
    if not c["causal"]:
        return c["S_q"] * c["S_kv"]
    return sum(max(0, min(i + c["S_kv"] - c["S_q"] + 1, c["S_kv"])) for i in range(c["S_q"]))


def work(case):
    c = case
    if c["op"] == "gemm":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": 2 * (M * K + N * K + M * N + (N if c["bias"] else 0)), "flops": 2 * M * N * K}
    if c["op"] == "conv":
        od, oh, ow = _conv_dims(c)
        m, k = c["N"] * od * oh * ow, c["kd"] * c["k"] * c["k"] * c["C"]
        x = c["N"] * c["D"] * c["H"] * c["W"] * c["C"]
        return {"bytes": 2 * (x + k * c["O"] + m * c["O"] + (c["O"] if c["bias"] else 0)), "flops": 2 * m * c["O"] * k}
    q, kv = c["B"] * c["S_q"] * c["H"] * c["D"], c["B"] * c["S_kv"] * c["H_kv"] * c["D"]
    per, rows = c["B"] * c["H"] * c["D"] * _pairs(c), 4 * c["B"] * c["H"] * c["S_q"]
    if c["op"] == "attn":
        return {"bytes": 2 * (2 * q + 2 * kv), "flops": 4 * per}
    return {"bytes": 2 * (4 * q + 4 * kv) + rows, "flops": 14 * per}


#: About four times what the outputs are off the 64-bit result over these ranges, relative (2-norm)
#: and at the worst element: one rounding to the output's 16 bits after 32-bit sums (2.1e-4 and 4.9e-4
#: in f16, 1.7e-3 and 3.9e-3 in bf16); attention rounds P, and its gradients dS, to 16 bits too.
_TOLERANCE = {("gemm", "f16"): (8e-4, 2e-3), ("gemm", "bf16"): (7e-3, 1.6e-2), ("conv", "f16"): (8e-4, 2e-3),
              ("attn", "f16"): (1.2e-3, 2e-2), ("attn", "bf16"): (9.5e-3, 4.5e-2),
              ("attn_train", "f16"): (1.3e-3, 5e-2), ("attn_train", "bf16"): (1.05e-2, 4e-1)}


def tolerance(case):
    rel, most = _TOLERANCE[case["op"], case.get("dtype", "f16")]
    return {"rel": rel, "max": most}


def _conv_exact(c, t):
    x, w = t["x"].double(), t["w"].double()
    if c["weights"] == "OIDHW":
        w = w.permute(2, 3, 4, 1, 0)
    pd, sd = (c["pad"], c["stride"]) if c["rank"] == 3 else (0, 1)
    p, s = c["pad"], c["stride"]
    x = torch.nn.functional.pad(x, (0, 0, p, p, p, p, pd, pd))
    od, oh, ow = _conv_dims(c)
    y = torch.zeros((c["N"] * od * oh * ow, c["O"]), dtype=torch.float64, device="cuda")
    for kd in range(c["kd"]):
        for kh in range(c["k"]):
            for kw in range(c["k"]):
                v = x[:, kd:kd + (od - 1) * sd + 1:sd, kh:kh + (oh - 1) * s + 1:s, kw:kw + (ow - 1) * s + 1:s]
                y += v.reshape(-1, c["C"]) @ w[kd, kh, kw].contiguous()
    if t["bias"] is not None:
        y += t["bias"].double()
    return y.reshape(c["N"], od, oh, ow, c["O"])


def _attn_exact(c, t):
    B, H, G = c["B"], c["H"], c["H"] // c["H_kv"]
    scale = 1 / math.sqrt(c["D"])
    train = c["op"] == "attn_train"
    out = {"O": torch.empty(t["Q"].shape, dtype=torch.float64, device="cuda")}
    if train:
        out["lse"] = torch.empty((B, H, c["S_q"]), dtype=torch.float64, device="cuda")
        out.update({"d" + n: torch.zeros(t[n].shape, dtype=torch.float64, device="cuda") for n in "QKV"})
    hide = None
    if c["causal"]:
        i = torch.arange(c["S_q"], device="cuda")[:, None] + (c["S_kv"] - c["S_q"])
        hide = torch.arange(c["S_kv"], device="cuda")[None, :] > i
    rows = max(1, (1 << 27) // c["S_kv"])  # query rows whose scores are held at once
    for b in range(B):
        for h in range(H):
            k, v = t["K"][b, :, h // G].double(), t["V"][b, :, h // G].double()
            kt, vt = k.t().contiguous(), v.t().contiguous()
            for r in range(0, c["S_q"], rows):
                q = t["Q"][b, r:r + rows, h].double()
                s = (q @ kt) * scale
                if hide is not None:
                    s = s.masked_fill(hide[r:r + rows], -math.inf)
                lse = torch.logsumexp(s, -1, keepdim=True)
                pr = torch.exp(s - lse)
                o = pr @ v
                out["O"][b, r:r + rows, h] = o
                if not train:
                    continue
                do = t["dO"][b, r:r + rows, h].double()
                out["lse"][b, h, r:r + rows] = lse[:, 0]
                ds = pr * (do @ vt - (do * o).sum(-1, keepdim=True)) * scale
                out["dQ"][b, r:r + rows, h] = ds @ k
                out["dK"][b, :, h // G] += ds.t().contiguous() @ q
                out["dV"][b, :, h // G] += pr.t().contiguous() @ do
    return out


def exact(case, seed):
    c, t = case, _inputs(case, seed)
    if c["op"] == "gemm":
        a = t["A"].double() if c["layout"][0] == "n" else t["A"].double().t().contiguous()
        b = t["B"].double() if c["layout"][1] == "n" else t["B"].double().t().contiguous()
        r = a @ b
        return {"C": r if t["bias"] is None else r + t["bias"].double()}
    if c["op"] == "conv":
        return {"y": _conv_exact(c, t)}
    return _attn_exact(c, t)

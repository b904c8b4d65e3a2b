"""GEMMs on quarter tiles (64x64 workgroups whose 8 or 4 wavefronts share the K-tiles): every operand layout,
edges of the 64x64 tile, K-tiles that do and do not divide over the wavefronts, K tails, padded and
odd rows (NaN in the padding), and the plan's own K partitions. Against the CPU oracle."""
import numpy as np
import pytest

import example_matmul_metal4_amd as mtk
import oracle

from test_gemm_odd_rows_gpu import _padded

# M, N, K, trans_a, trans_b, padding of A's and B's rows, split_k, dtype
CASES = [(m, n, k, ta, tb, pa, pb, 1, dt)
         for (ta, tb) in ((False, True), (False, False), (True, True), (True, False))
         for (m, n, k, pa, pb, dt) in ((64, 64, 256, 0, 0, "f16"), (66, 63, 193, 0, 1, "bf16"), (2, 130, 700, 2, 4, "f16"),
                                       (190, 1, 577, 4, 1, "f16"), (1000, 900, 330, 0, 0, "bf16"))]
CASES += [(60, 128, 9000, False, True, 0, 0, 0, "f16"), (130, 514, 2801, True, False, 0, 0, 0, "bf16"),
          (9, 1001, 5003, False, True, 0, 0, 0, "f16"), (40, 70, 4097, False, False, 1, 1, 0, "f16")]
# more than one quarter per CU, or a layout that no other kernel reads: 4 wavefronts per workgroup
FOUR = [(4, 40, 70, True, True, 0, 1, 1, "f16"), (500, 100, 1025, True, True, 0, 0, 3, "f16"), (1100, 1030, 1300, False, True, 0, 0, 1, "f16"),
        (1030, 1101, 517, False, False, 1, 0, 0, "bf16"), (1100, 1034, 1290, True, False, 0, 0, 1, "bf16")]
CASES += FOUR


def _plan(dev, case):
    M, N, K, ta, tb, pa, pb, split_k, dtype = case
    return mtk.GemmPlan(dev, M, N, K, trans_a=ta, trans_b=tb, dtype=dtype, has_bias=True, split_k=split_k,
                        lda=(M if ta else K) + pa, ldb=(K if tb else N) + pb)


def _tile_and_grid(text, M, N, rows, cols):
    """The description's tile and grid are the workgroups that run."""
    word = lambda key: text.split(f" {key}=")[1].split()[0]
    assert word("tile") == f"{rows}x{cols}", text
    assert int(word("grid")) == -(-M // rows) * -(-N // cols) * int(word("split_k") if " split_k=" in text else 1), text


def test_which_plans_are_quartered():
    # CPU: the planner alone
    for c in CASES:
        kern = _plan(None, c).describe().split("kernels: ")[1].split()[0]
        assert kern.endswith("q4" if c in FOUR else "q"), (c, kern)
        _tile_and_grid(_plan(None, c).describe(), c[0], c[1], 64, 64)
    assert "splitk_reduce" in _plan(None, CASES[20]).describe() and "splitk_reduce" in _plan(None, CASES[22]).describe()
    # larger grids, requested tiles, partitions or schedules, and K of fewer than four K-tiles are not
    for kw in (dict(M=2048, N=2048, K=512), dict(M=1024, N=1024, K=1024, tile=128), dict(M=512, N=512, K=4096, split_k=4),
               dict(M=512, N=512, K=4096, split_k=0, split_mode="two_pass"), dict(M=100, N=100, K=192)):
        M, N, K = kw.pop("M"), kw.pop("N"), kw.pop("K")
        assert "quarters" not in mtk.GemmPlan(None, M, N, K, **kw).describe(), (M, N, K, kw)


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_quarter_tiles(dev, case):
    M, N, K, ta, tb, pa, pb, split_k, dtype = case
    A = oracle.normal(95, (M, K), 0, 1, dtype)
    B = oracle.normal(96, (N, K) if tb else (K, N), 0, 1 / np.sqrt(K), dtype)
    bias = oracle.uniform(97, (N,), -0.5, 0.5, dtype)
    plan = _plan(dev, case)
    print(f"[gemm quarter] {case} {plan.describe()}", flush=True)
    stored = np.ascontiguousarray(A.T) if ta else A
    dA = dev.upload(_padded(stored, stored.shape[1] + pa, 0, dtype))
    dB, dbias, dC = dev.upload(_padded(B, B.shape[1] + pb, 0, dtype)), dev.upload(bias), dev.empty((M * N + 2) * 2)
    ws = dev.empty(plan.workspace_bytes) if plan.workspace_bytes else None
    dev.fill_u16(dC, 0x1234, M * N + 2)
    plan.run(dA, dB, dbias, dC, ws)
    dev.sync()
    raw = dev.download(dC, (M * N + 2,), np.uint16)
    for b in (dA, dB, dbias, dC, ws):
        if b is not None:
            b.free()
    assert np.all(raw[M * N:] == 0x1234)  # nothing past the last row
    got = oracle.to_f32(raw[:M * N].view(A.dtype).reshape(M, N), dtype).astype(np.float64)
    exp = oracle.gemm(A, B, bias, trans_b=tb, dtype=dtype)
    a, b = (np.abs(oracle.to_f32(x, dtype).astype(np.float64)) for x in (A, B))
    # one rounding to the output type, fp32 sums of K products in any order on either side
    bound = oracle.ulp(exp, dtype) + 2 * K * 2.0 ** -24 * (a @ (b.T if tb else b) + np.abs(oracle.to_f32(bias, dtype)))
    assert np.all(np.isfinite(got)) and np.all(np.abs(got - exp) <= bound), np.abs(got - exp).max()


def _odd_t(split_k=1, **kw):
    return mtk.GemmPlan(None, 300, 64, 71, trans_a=True, split_k=split_k, **kw)  # B [64][71]: odd rows


def test_transposed_a_with_odd_rows_is_planned_or_refused():
    # CPU: only the quarter kernels read A [K][M] beside odd rows of B, so every accepted plan names one of
    # them (a kernel that is compiled); a tile or an in-workgroup schedule that they cannot honour is refused
    for plan in (_odd_t(), _odd_t(0), _odd_t(2), _odd_t(split_mode="two_pass"), _odd_t(split_mode="serial"),
                 _odd_t(3, split_mode="two_pass", k_stagger=2),
                 mtk.GemmPlan(None, 300, 63, 60, trans_a=True, trans_b=False, split_k=4, split_mode="serial"),  # one K-tile
                 mtk.GemmPlan(None, 4096, 4095, 8192, trans_a=True, trans_b=False, split_k=0)):
        assert "_128x128_v1q" in plan.describe(), plan.describe()
    for kw in (dict(tile=256), dict(tile=128), dict(tile=256, split_mode="serial"), dict(split_k=2, split_mode="serial"),
               dict(split_k=0, split_mode="serial")):
        with pytest.raises(mtk.MtkError) as e:
            _odd_t(**kw)
        assert e.value.status == mtk.MTK_ERR_UNSUPPORTED, kw

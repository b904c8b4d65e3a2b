"""GEMM operands whose rows start at any 2-byte address: odd leading dimensions, operands that begin in
the middle of a dword, and every remainder of K and N against the 8-element chunks, with padding that
must not reach the result (NaN). Against the CPU oracle with its per-element bound."""
import numpy as np
import pytest

import example_matmul_metal4_amd as mtk
import oracle

# M, N, K, lda, ldb, trans_b, elements before A and B, split_k, dtype
CASES = [(130, 72, 64 + r, 65 + r + (r % 2 == 1), 67 + r + (r % 2 == 1), True, r % 2, (r // 2) % 2, 1, "f16") for r in range(8)]
CASES += [(97, 129 + r, 200 + r, 201 + 2 * r, 131 + 2 * r, False, r % 2, (r + 1) % 2, 1, "bf16") for r in range(4)]
CASES += [(1, 1, 1, 1, 1, True, 1, 1, 1, "f16"), (3, 5, 7, 7, 7, True, 1, 0, 1, "bf16"), (300, 257, 517, 517, 518, True, 1, 1, 4, "f16"),
          (300, 257, 517, 518, 257, False, 0, 1, 3, "f16"), (257, 300, 1023, 1023, 1023, True, 1, 1, 0, "bf16"),
          (1100, 1030, 333, 333, 333, True, 0, 1, 1, "f16")]


def _padded(x, ld, before, dtype):
    """x's rows at leading dimension ld behind `before` elements, NaN everywhere else."""
    nan = np.uint16(0x7E00 if dtype == "f16" else 0x7FC0)
    buf = np.full(before + x.shape[0] * ld + 8, nan, np.uint16)
    rows = buf[before:before + x.shape[0] * ld].reshape(x.shape[0], ld)
    rows[:, :x.shape[1]] = x.view(np.uint16)
    return buf


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_odd_rows(dev, case):
    M, N, K, lda, ldb, trans_b, oa, ob, split_k, dtype = case
    A = oracle.normal(90, (M, K), 0, 1, dtype)
    B = oracle.normal(91, (N, K) if trans_b else (K, N), 0, 1 / np.sqrt(K), dtype)
    bias = oracle.uniform(92, (N,), -0.5, 0.5, dtype)
    plan = mtk.GemmPlan(dev, M, N, K, trans_b=trans_b, dtype=dtype, has_bias=True, split_k=split_k, lda=lda, ldb=ldb)
    print(f"[gemm odd] {case} {plan.describe()}", flush=True)
    dA, dB, dbias = dev.upload(_padded(A, lda, oa, dtype)), dev.upload(_padded(B, ldb, ob, dtype)), dev.upload(bias)
    dC = dev.empty(M * N * 2)
    ws = dev.empty(plan.workspace_bytes) if plan.workspace_bytes else None
    if lda % 2 == 0 and ldb % 2 == 0 and (oa or ob):  # dword-aligned rows: a start inside a dword stays refused
        with pytest.raises(mtk.MtkError):
            plan.run(dA.ptr + 2 * oa, dB.ptr + 2 * ob, dbias, dC, ws)
        return
    plan.run(dA.ptr + 2 * oa, dB.ptr + 2 * ob, dbias, dC, ws)
    dev.sync()
    got = oracle.to_f32(dev.download(dC, (M, N), A.dtype), dtype).astype(np.float64)
    for b in (dA, dB, dbias, dC, ws):
        if b is not None:
            b.free()
    exp = oracle.gemm(A, B, bias, trans_b=trans_b, dtype=dtype)
    absprod = np.abs(oracle.to_f32(A, dtype).astype(np.float64)) @ np.abs(
        (oracle.to_f32(B, dtype).T if trans_b else oracle.to_f32(B, dtype)).astype(np.float64))
    # one rounding to the output type, fp32 sums of K products in any order on either side
    bound = oracle.ulp(exp, dtype) + 2 * K * 2.0 ** -24 * (absprod + np.abs(oracle.to_f32(bias, dtype)))
    assert np.all(np.isfinite(got)) and np.all(np.abs(got - exp) <= bound), np.abs(got - exp).max()

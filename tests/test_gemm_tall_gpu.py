"""GEMMs of 65 to 96 and 129 to 192 rows on 96x64 workgroups: edges of the 96-row tile, ragged columns, K
tails and K-tiles that do not divide over 8 wavefronts, padded rows (NaN in the padding), both B layouts,
with and without K partitions. Against the CPU oracle."""
import pytest

import example_matmul_metal4_amd as mtk

from test_gemm_quarter_gpu import _plan, _tile_and_grid, test_quarter_tiles as _check

# M, N, K, trans_a, trans_b, padding of A's and B's rows, split_k, dtype
CASES = [(65, 16383, 1026, False, True, 0, 0, 1, "f16"), (96, 10946, 1032, False, False, 2, 4, 1, "bf16"),
         (96, 4096, 4096, False, True, 0, 0, 0, "f16"), (77, 3970, 4162, False, False, 0, 0, 0, "f16"),
         (70, 1601, 9986, False, True, 4, 2, 0, "bf16"), (129, 6002, 1090, False, True, 0, 0, 1, "bf16"),
         (192, 8192, 1024, False, False, 0, 0, 0, "f16"), (191, 4033, 6218, False, True, 2, 0, 0, "f16")]


def test_which_plans_are_tall():
    # CPU: the planner alone
    for c in CASES:
        assert "q96" in _plan(None, c).describe(), (c, _plan(None, c).describe())
        _tile_and_grid(_plan(None, c).describe(), c[0], c[1], 96, 64)
    assert "splitk_reduce" in _plan(None, CASES[2]).describe() and "splitk_reduce" in _plan(None, CASES[7]).describe()
    # other row counts, odd rows, transposed A, requested tiles or partitions, short K, few columns are not
    for kw in (dict(M=64), dict(M=97), dict(M=193), dict(K=2049), dict(trans_a=True), dict(tile=128), dict(split_k=4),
               dict(K=960), dict(N=8192, K=2048), dict(N=29184)):
        kw = {**dict(M=96, N=16384, K=2048), **kw}
        M, N, K = kw.pop("M"), kw.pop("N"), kw.pop("K")
        assert "q96" not in mtk.GemmPlan(None, M, N, K, **kw).describe(), (M, N, K, kw)


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=str)
def test_tall_tiles(dev, case):
    _check(dev, case)

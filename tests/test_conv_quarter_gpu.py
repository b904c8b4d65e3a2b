"""Convolutions on quarter tiles (64x64 workgroups whose wavefronts share the K-tiles, gathering 8-channel
chunks): bit exact on the reference's integer generators (ConvolutionShared.swift:4874-4992), on which
every fp32 partial sum is exact in any order."""
import numpy as np
import pytest

import example_matmul_metal4_amd as mtk
import oracle
from oracle import generators as gen

from test_conv_gpu import _bit_exact, _run
from test_gemm_quarter_gpu import _tile_and_grid

C2, C3 = oracle.ConvDims.conv2d, oracle.ConvDims.conv3d
# rank, dims, kernel: edges of the 64-pixel and 64-channel tiles, channels whose chunks share a K-tile with
# other taps, partial last K-tiles, strides, dilations, one-sided padding, 10 taps, output channels of
# every alignment, and both workgroup sizes
CASES = [
    (2, C2(N=1, H=8, W=8, C=32, O=64, PT=1, PB=1, PL=1, PR=1), "q8"), (2, C2(N=1, H=9, W=8, C=40, O=72, PT=1, PB=0, PL=0, PR=2), "q8"),
    (2, C2(N=3, H=21, W=17, C=8, O=66, KH=5, KW=5, SY=2, SX=1, DY=1, DX=2, PT=2, PB=0, PL=3, PR=1), "v1q8"),
    (2, C2(N=1, H=30, W=13, C=24, O=5, PT=1, PB=1, PL=1, PR=1), "v1q8"), (2, C2(N=2, H=11, W=40, C=16, O=1, KH=10, KW=10, PT=4, PB=5, PL=9, PR=0), "v1q8"),
    (2, C2(N=1, H=20, W=20, C=128, O=130, KH=1, KW=7, PL=3, PR=3), "q8"), (2, C2(N=2, H=96, W=90, C=96, O=72, PT=1, PB=1, PL=1, PR=1), "q4"),
    (2, C2(N=2, H=80, W=121, C=64, O=16, KH=5, KW=5, PT=2, PB=2, PL=2, PR=2), "q4"), (2, C2(N=1, H=200, W=190, C=72, O=33, PT=1, PB=1, PL=1, PR=1), "v1q4"),
    (3, C3(N=2, D=7, H=9, W=10, C=56, O=40, SZ=2, SY=1, SX=2, DZ=1, DY=2, DX=1, PF=1, PBk=2, PT=1, PB=1, PL=0, PR=2), "q8"),
    (3, C3(N=1, D=12, H=40, W=41, C=128, O=64, PF=1, PBk=1, PT=1, PB=1, PL=1, PR=1), "q4"),
]


def _plan(dev, rank, dims, **kw):
    return mtk.ConvPlan(dev, mtk.conv_desc(dims, has_bias=True, rank=rank, **kw))


def test_which_plans_are_quartered():
    # CPU: the planner alone
    for rank, dims, kern in CASES:
        text = _plan(None, rank, dims).describe()
        assert text.endswith("_" + kern) and "-quarter grid=" in text, (dims.as_dict(), text)
        _tile_and_grid(text, dims.N * dims.OD * dims.OH * dims.OW, dims.O, 64, 64)
    for dims in (C2(N=1, H=40, W=40, C=12, O=16), C2(N=1, H=40, W=40, C=16, O=16, KH=11, KW=3), C2(N=1, H=40, W=40, C=64, O=64, KH=1, KW=1),
                 C2(N=8, H=128, W=128, C=256, O=256), C2(N=4, H=100, W=100, C=96, O=256)):
        assert not _plan(None, 2, dims).describe().rsplit("_", 1)[1].lstrip("v1").startswith("q"), _plan(None, 2, dims).describe()


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(CASES)))
def test_quarter_conv(dev, case):
    rank, dims, _ = CASES[case]
    x, w, b = gen.conv3d_activation(dims), gen.conv3d_weights(dims), gen.conv3d_bias(dims)
    assert _bit_exact(dims, _run(dev, dims, x, w, b, rank=rank), x, w, b)


@pytest.mark.gpu
def test_quarter_conv_in_the_middle_of_a_dword(dev):
    # output channels of odd count need no more than 2-byte alignment of any operand
    rank, dims, _ = CASES[3]
    x, w, b = gen.conv3d_activation(dims), gen.conv3d_weights(dims), gen.conv3d_bias(dims)
    shifted = [dev.upload(np.concatenate([np.full(1, 0x7E00, np.uint16), a.view(np.uint16).ravel(), np.full(8, 0x7E00, np.uint16)])) for a in (x, w, b)]
    plan, n = _plan(dev, rank, dims), int(np.prod(dims.y_shape()))
    y = dev.empty(2 * n + 4)
    dev.fill_u16(y, 0x1234, n + 2)
    plan.run(shifted[0].ptr + 2, shifted[1].ptr + 2, shifted[2].ptr + 2, y.ptr + 2)
    dev.sync()
    got = dev.download(y, (n + 2,), np.uint16)
    for buf in (*shifted, y):
        buf.free()
    assert got[0] == 0x1234 and got[-1] == 0x1234
    assert _bit_exact(dims, got[1:-1].view(np.float16).reshape(dims.y_shape()), x, w, b)


def test_long_walks_between_two_and_four_quarters_per_cu():
    # CPU: the planner alone. There the 128x128 tiles still run at once: quarters only for walks that are longer
    def quarter(N, H, W, C, O, k):
        dims = C2(N=N, H=H, W=W, C=C, O=O, KH=k, KW=k, PT=k // 2, PB=k // 2, PL=k // 2, PR=k // 2)
        return _plan(None, 2, dims).describe().rsplit("_", 1)[1].endswith("q4")
    for n, c, k, want in ((6, 64, 5, False), (6, 128, 5, True), (7, 64, 5, False), (7, 128, 5, True), (11, 64, 5, True),  # K-tiles
                          (6, 16, 5, False), (6, 32, 5, True), (7, 72, 3, False), (7, 96, 3, True), (11, 56, 3, True)):
        assert quarter(n, 80, 90, c, 64, k) == want, (n, c, k)
    assert quarter(7, 80, 90, 72, 33, 3)  # output channels of odd count: the 128x128 kernel loads single elements


# channels in multiples of 64 and too many quarters: the direct-to-LDS gather on 128x128 tiles, with filters of 36 and
# 49 taps, strides, dilations, one-sided padding, three dimensions and remainders of both tile edges
FAST = [(2, C2(N=2, H=100, W=101, C=64, O=96, KH=6, KW=6, PT=3, PB=2, PL=3, PR=2)),
        (2, C2(N=2, H=100, W=101, C=64, O=70, KH=7, KW=7, PT=3, PB=3, PL=3, PR=3)),
        (2, C2(N=8, H=131, W=133, C=128, O=40, SY=2, SX=2, DY=1, DX=2, PT=0, PB=1, PL=2, PR=1)),
        (2, C2(N=3, H=61, W=97, C=192, O=202, KH=1, KW=5, SY=1, SX=1, PL=1, PR=3)),
        (3, C3(N=1, D=12, H=41, W=43, C=64, O=130, KD=3, KH=2, KW=3, SZ=1, SY=1, SX=1, DZ=2, DY=1, DX=1, PF=2, PBk=1, PT=1, PB=0, PL=0, PR=2)),
        (3, C3(N=2, D=15, H=60, W=62, C=64, O=66, SZ=2, SY=1, SX=2, DZ=1, DY=2, DX=1, PF=1, PBk=2, PT=1, PB=2, PL=1, PR=0))]


def test_which_plans_keep_the_128x128_gather():
    # CPU: the planner alone
    for rank, dims in FAST:
        assert _plan(None, rank, dims).describe().endswith("mtk_conv_f16_fast_128x128_d"), _plan(None, rank, dims).describe()


@pytest.mark.gpu
@pytest.mark.parametrize("case", range(len(FAST)))
def test_128x128_gather(dev, case):
    rank, dims = FAST[case]
    x, w, b = gen.conv3d_activation(dims), gen.conv3d_weights(dims), gen.conv3d_bias(dims)
    assert _bit_exact(dims, _run(dev, dims, x, w, b, rank=rank), x, w, b)

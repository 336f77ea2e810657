"""The stride-2 row kernel (one input block, one channel tile; tiles of 4 rows of 32 output voxels, staged whole): exact operands equal the oracle byte for byte
in every output type at the edges of its tiles and of odd volumes, and random operands give the bytes of the two kernels it
runs in the place of, in the inputs' format as well: the one that reads every tap's rows from memory and the general one, whose pairs are others."""
import numpy as np
import pytest

from ufsm_amd import lib
import orc
from test_gpu_conv import exact_case, rand_case, gpu_conv

pytestmark = pytest.mark.gpu

# (bits, N, Ci, Co, D, H, W): one voxel; odd dims; rows that end one voxel into a second tile; the last row tile of one row; more tiles than workgroups (a walk);
# fewer channels than a block's 32
SHAPES = [(8, 1, 32, 32, 1, 1, 1), (8, 1, 32, 32, 5, 7, 65), (8, 2, 32, 32, 6, 10, 66), (8, 1, 32, 24, 4, 16, 64), (8, 3, 20, 32, 3, 18, 35), (8, 2, 32, 32, 40, 44, 130),
          (4, 1, 32, 32, 2, 2, 2), (4, 1, 32, 32, 8, 10, 66), (4, 2, 32, 32, 4, 18, 128), (4, 2, 32, 32, 40, 44, 130)]


@pytest.mark.parametrize("bits,N,Ci,Co,D,H,W", SHAPES)
def test_stride_2_row_kernel(gpu, bits, N, Ci, Co, D, H, W):
    rng = np.random.default_rng(Ci + Co + D * 5 + W)
    S, xdt = D * H * W, 3 if bits == 8 else 4
    x, w, b = exact_case(rng, N, Ci, Co, S)
    xq = orc.f32_to_mx(bits, x, N, Ci, S)

    def run(mode, xq, w, b, ydt):
        lib.mi_conv_s2_direct(mode)
        try:
            got, _ = gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, ydt, cbits=bits, stride=2)
        finally:
            lib.mi_conv_s2_direct(-1)
        assert ("conv3s2_row_k" in lib.mi_last_kernel().decode()) == (mode == 2), lib.mi_last_kernel().decode()
        return got
    for ydt in (0, 2, xdt):
        want, _ = orc.conv3(xq, xdt, N, Ci, D, H, W, w, b, Co, ydt, cbits=bits, stride=2, acc64=1)
        assert np.array_equal(run(2, xq, w, b, ydt), want), ydt
    x, w, b = rand_case(rng, N, Ci, Co, S)
    xq = orc.f32_to_mx(bits, x, N, Ci, S)
    # (the direct kernel: the same pairs in the same order. The general kernel adds tap by tap; on values of ordinary spread a block's 27 x 32 products are
    # added without a rounding that depends on the order: these bytes are the network's, which must not move with a window's size)
    for ydt in (0, xdt):
        got = run(2, xq, w, b, ydt)
        assert np.array_equal(got, run(1, xq, w, b, ydt)) and np.array_equal(got, run(0, xq, w, b, ydt)), ydt


def test_taps_outside_read_zeros(gpu):
    """NaN on the last voxel of the first sample reaches the outputs whose taps meet it only (and not through the weights' empty last unit)"""
    rng = np.random.default_rng(3)
    N, C, D, H, W = 2, 32, 4, 8, 70
    x, w, b = rand_case(rng, N, C, C, D * H * W)
    x[0, 3, D * H * W - 1] = np.nan
    lib.mi_conv_s2_direct(2)
    try:
        got, _ = gpu_conv(orc.f32_to_mx(8, x, N, C, D * H * W), 3, N, C, D, H, W, w, b, C, 0, stride=2)
    finally:
        lib.mi_conv_s2_direct(-1)
    exp = np.zeros((N, C, 2, 4, 35), bool); exp[0, :, 1, 3, 34] = True
    assert np.array_equal(~np.isfinite(got.reshape(exp.shape)), exp)

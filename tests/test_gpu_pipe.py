"""conv3_pipe_k, the general kernel's one-tile, two-plane launches pipelined: equal to the oracle on exact operands in every form it takes, and not taken outside its range."""
import numpy as np
import pytest

from ufsm_amd import lib
import orc
from test_gpu_conv import exact_case, rand_case, gpu_conv

pytestmark = pytest.mark.gpu

# (bits, N, Ci, Co, D, H, W, pairs of a weight stage, chunk): one block and many; borders cut in every direction; chunks of one to four blocks, one chunk and several; one round of CUs and, with
# stages of three pairs, two workgroups per CU; chunks of three and four past one round; per-channel
# statistics records and rows of 16 output channels
CASES = [(8, 1, 32, 128, 6, 13, 21, 7, 1), (8, 2, 160, 128, 9, 13, 18, 7, 1), (8, 2, 256, 256, 16, 16, 16, 7, 1), (8, 1, 128, 128, 22, 26, 26, 3, 1), (8, 1, 96, 128, 17, 21, 35, 3, 1),
         (4, 2, 32, 128, 9, 14, 18, 7, 1), (4, 1, 64, 128, 14, 15, 20, 7, 2), (4, 2, 192, 192, 10, 16, 16, 7, 3), (4, 1, 96, 192, 9, 11, 33, 7, 3), (4, 2, 128, 256, 12, 12, 12, 7, 4), (4, 1, 384, 128, 15, 16, 19, 7, 4),
         (4, 1, 64, 128, 22, 26, 26, 3, 2), (4, 1, 32, 128, 22, 26, 26, 3, 1), (4, 3, 192, 192, 16, 16, 16, 7, 3), (4, 1, 256, 128, 22, 26, 26, 7, 4),
         (8, 2, 64, 40, 3, 20, 24, 7, 1), (8, 1, 96, 16, 3, 40, 40, 7, 1), (4, 1, 64, 16, 2, 17, 50, 7, 2)]


def _run(case, ydt, stats, x, w, b):
    bits, N, Ci, Co, D, H, W = case[:7]
    xdt = 3 if bits == 8 else 4
    xq = orc.f32_to_mx(bits, x, N, Ci, D * H * W)
    was = lib.mi_conv_keep_records(1)
    try:
        got = gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, ydt, cbits=bits, Go=8 if stats else 0, stats=stats)
    finally:
        lib.mi_conv_keep_records(was)
    return got, orc.conv3(xq, xdt, N, Ci, D, H, W, w, b, Co, ydt, cbits=bits, acc64=1, Go=8 if stats else 0, want_stats=stats), lib.mi_last_kernel().decode()


@pytest.mark.parametrize("case", CASES)
def test_exact_operands(gpu, case):
    rng = np.random.default_rng(sum(case))
    x, w, b = exact_case(rng, case[1], case[2], case[3], case[4] * case[5] * case[6])
    for ydt in (3, 4, 0):
        (got, gs), (want, ws), name = _run(case, ydt, True, x, w, b)
        assert "conv3_pipe_k" in name and "stage %d CB %d " % case[7:9] in name, name
        assert np.array_equal(got, want), ydt
        assert np.allclose(gs, ws, rtol=1e-6)


@pytest.mark.parametrize("case", [CASES[1], CASES[4], CASES[7], CASES[10]])
def test_random_operands(gpu, case):
    """fp32 sums of up to 27 x 384 products against fp64 ones: the tolerance of the conv tests."""
    rng = np.random.default_rng(7 + sum(case))
    x, w, b = rand_case(rng, case[1], case[2], case[3], case[4] * case[5] * case[6])
    (got, gs), (want, ws), name = _run(case, 0, True, x, w, b)
    assert "conv3_pipe_k" in name
    assert np.abs(got - want).max() / np.abs(want).max() < 2e-4
    assert np.abs(gs - ws).max() / np.abs(ws).max() < 1e-5


def test_not_taken(gpu):
    """A last chunk of fewer blocks than the others keeps the general kernel; so does one chunk of four past one round of CUs."""
    for case in [(4, 1, 160, 128, 14, 16, 20), (4, 1, 128, 128, 22, 26, 26)]:
        rng = np.random.default_rng(sum(case))
        x, w, b = exact_case(rng, case[1], case[2], case[3], case[4] * case[5] * case[6])
        (got, gs), (want, ws), name = _run(case, 4, True, x, w, b)
        assert name.startswith("conv3_mx_k<fmt 4, stride 1, MT 1, NT 2"), name
        assert np.array_equal(got, want)

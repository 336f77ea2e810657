"""conv3_pipe_k, the general kernel's one-tile, two-plane launches pipelined: equal to the oracle on exact operands in every form it takes, and not taken outside its range."""
import numpy as np
import pytest

from ufsm_amd import lib
import orc
import test_gpu_dispatch as dispatch
from test_gpu_conv import exact_case, rand_case, gpu_conv
from test_gpu_thin import conv_in_slabs

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


@pytest.fixture
def as_in_networks():
    """The kernels a network's statistics were added on (no flat tiles), for the test's convs."""
    was = lib.mi_conv_keep_records(1)
    yield
    lib.mi_conv_keep_records(was)


def spread_case(rng, N, Ci, Co, S):
    """Operands of several magnitudes, whose fp32 sums depend on their order."""
    x, w, b = rand_case(rng, N, Ci, Co, S)
    return x * np.exp(2 * rng.standard_normal(x.shape)).astype(np.float32), w, b


# (bits, Ci, pairs of a stage at 2 and at 20 samples): chunks of one to four blocks, one chunk and several. Groups of two channels: one channel tile per workgroup at any size, three planes: two per tile, so that
# 32, 320 and 576 workgroups are the same conv on the pipelined kernel's two forms and on the general one
@pytest.mark.parametrize("bits,Ci,pps", [(8, 32, (7, 3)), (8, 96, (7, 3)), (8, 256, (7, 3)), (4, 32, (7, 3)), (4, 64, (7, 3)), (4, 192, (7, 7)), (4, 256, (7, 7)), (4, 384, (7, 7))])
@pytest.mark.parametrize("Co", [64, 40])
def test_the_general_kernels_bits(gpu, as_in_networks, bits, Ci, Co, pps):
    """A sample's fp32 outputs, codes and statistics are the same bits whichever of the two kernels runs, on operands whose sums show their order."""
    rng = np.random.default_rng(Ci + Co + bits)
    N, D, H, W, G, xdt = 36, 3, 16, 32, Co // 2, 3 if bits == 8 else 4
    S = D * H * W
    x, w, b = spread_case(rng, N, Ci, Co, S)
    for ydt in (0, xdt):
        yw, gw = gpu_conv(orc.f32_to_mx(bits, x, N, Ci, S), xdt, N, Ci, D, H, W, w, b, Co, ydt, cbits=bits, Go=G, stats=True)
        assert lib.mi_last_kernel().decode().startswith("conv3_mx_k<fmt %d, stride 1, MT 1, NT 2" % bits), lib.mi_last_kernel().decode()
        dec = (lambda y, n: y) if ydt == 0 else (lambda y, n: orc.mx_to_f32(bits, y, n, Co, S).reshape(n, Co, S))
        yw = dec(yw, N)
        for n, p in ((2, pps[0]), (20, pps[1])):
            y, g = gpu_conv(orc.f32_to_mx(bits, x[:n], n, Ci, S), xdt, n, Ci, D, H, W, w, b, Co, ydt, cbits=bits, Go=G, stats=True)
            assert lib.mi_last_kernel().decode().startswith("conv3_pipe_k ") and "stage %d " % p in lib.mi_last_kernel().decode(), lib.mi_last_kernel().decode()
            assert np.array_equal(dec(y, n).view(np.uint32), yw[:n].view(np.uint32)) and np.array_equal(g, gw[:n])
        if ydt == 0 and bits == 8 and Ci <= 96:                                  # (the operands do what they are for: a tenth and more of the sums are rounded otherwise than in one step)
            assert (yw[:1] != orc.conv3(orc.f32_to_mx(bits, x[:1], 1, Ci, S), xdt, 1, Ci, D, H, W, w, b, Co, 0, cbits=bits, acc64=1)[0]).mean() > 0.1


# whole tensors and slabs on the pipelined kernel, [2x upsampled | skip] too; whole tensors whose slices of three channel tiles stay together and whose slabs divide them
@pytest.mark.parametrize("bits,N,Ci,Co,D,H,W,slab,up,whole", [(8, 2, 256, 256, 16, 16, 16, 4, 0, "conv3_pipe_k"), (8, 1, 192, 128, 18, 26, 26, 4, 1, "conv3_pipe_k"), (4, 2, 384, 128, 16, 16, 18, 8, 1, "conv3_pipe_k"),
                                                              (4, 1, 192, 192, 24, 32, 48, 8, 0, "conv3_mx_k"), (4, 1, 192, 96, 32, 32, 48, 8, 0, "conv3_mx_k"), (4, 2, 192, 192, 12, 16, 20, 4, 0, "conv3_pipe_k")])
def test_slabs_give_the_whole_tensors_bytes(gpu, as_in_networks, bits, N, Ci, Co, D, H, W, slab, up, whole):
    (y, s, k), (yz, sz, kz) = conv_in_slabs(bits, N, Ci, Co, D, H, W, slab, up)
    assert k.split("<")[0].split(" ")[0] == whole and kz.startswith("conv3_pipe_k "), (k, kz)
    assert np.array_equal(y, yz)
    assert np.allclose(s, sz, rtol=1e-12, atol=1e-9)


@pytest.mark.parametrize("bits,N,Ci,Co,D,H,W", [(8, 2, 256, 256, 16, 16, 16), (8, 1, 96, 128, 17, 21, 35), (4, 2, 192, 192, 10, 16, 16), (4, 1, 384, 128, 15, 16, 19)])
def test_statistics_of_a_range_of_planes(gpu, as_in_networks, bits, N, Ci, Co, D, H, W):
    dispatch.test_statistics_of_a_range_of_planes(gpu, bits, N, Ci, Co, D, H, W, "conv3_pipe_k")


@pytest.mark.parametrize("bits,Ci,Co,D,H,W", [(8, 256, 256, 17, 16, 16), (8, 64, 128, 19, 26, 26), (4, 256, 128, 22, 20, 26), (4, 192, 192, 18, 16, 20)])
def test_overlapping_slabs_that_count_their_own_planes(gpu, as_in_networks, bits, Ci, Co, D, H, W):
    dispatch.test_overlapping_slabs_that_count_their_own_planes(gpu, bits, Ci, Co, D, H, W, "conv3_pipe_k")


@pytest.mark.parametrize("bits,N,Cu,Cs,Co,D,H,W", [(8, 2, 64, 96, 128, 9, 13, 18), (8, 1, 32, 64, 128, 17, 21, 35), (4, 2, 96, 96, 192, 10, 16, 16), (4, 1, 256, 128, 128, 15, 16, 19), (4, 1, 64, 320, 128, 15, 16, 19)])
def test_two_input_segments(gpu, as_in_networks, bits, N, Cu, Cs, Co, D, H, W):
    """[x | x2] as stored: chunks inside a segment and across the two, the oracle's bytes on exact operands."""
    rng = np.random.default_rng(Cu + Cs + D)
    S, xdt = D * H * W, 3 if bits == 8 else 4
    x, w, b = exact_case(rng, N, Cu + Cs, Co, S)
    qu, qs = orc.f32_to_mx(bits, np.ascontiguousarray(x[:, :Cu]), N, Cu, S), orc.f32_to_mx(bits, np.ascontiguousarray(x[:, Cu:]), N, Cs, S)
    want, ws = orc.conv3(qu, xdt, N, Cu + Cs, D, H, W, w, b, Co, xdt, cbits=bits, x2=qs, c_split=Cu, acc64=1, Go=8, want_stats=True)
    got, gs = gpu_conv(qu, xdt, N, Cu + Cs, D, H, W, w, b, Co, xdt, cbits=bits, x2=qs, c_split=Cu, Go=8, stats=True)
    assert lib.mi_last_kernel().decode().startswith("conv3_pipe_k "), lib.mi_last_kernel().decode()
    assert np.array_equal(got, want) and np.allclose(gs, ws, rtol=1e-6)


@pytest.mark.parametrize("case", [CASES[1], CASES[4], CASES[7], CASES[10]])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_rows_that_are_not_finite(gpu, as_in_networks, case, bad):
    """A row that is not finite reaches the voxels whose taps meet it and no other: at the volume's corner, inside a tile and across two."""
    bits, N, Ci, Co, D, H, W = case[:7]
    rng = np.random.default_rng(3 + sum(case))
    x, w, b = rand_case(rng, N, Ci, Co, D * H * W)
    conv = lambda: gpu_conv(orc.f32_to_mx(bits, x, N, Ci, D * H * W), 3 if bits == 8 else 4, N, Ci, D, H, W, w, b, Co, 0, cbits=bits, Go=8, stats=True)[0]
    clean = conv()
    assert lib.mi_last_kernel().decode().startswith("conv3_pipe_k ")
    at = [(0, 0, 0, 0, 0), (N - 1, Ci - 1, D - 1, H - 1, W - 1), (0, Ci // 2, D // 2, 8, min(16, W - 1))]
    x5, exp = x.reshape(N, Ci, D, H, W), np.zeros((N, D, H, W), bool)
    for n, c, z, y, v in at:
        x5[n, c, z, y, v] = bad
        exp[n, max(z - 1, 0):z + 2, max(y - 1, 0):y + 2, max(v - 1, 0):v + 2] = True
    got = conv()
    assert lib.mi_last_kernel().decode().startswith("conv3_pipe_k ")
    exp = np.broadcast_to(exp.reshape(N, 1, -1), got.shape)
    assert np.array_equal(~np.isfinite(got), exp) and np.array_equal(got[~exp], clean[~exp])

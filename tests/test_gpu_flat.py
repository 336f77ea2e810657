"""The flat conv kernel (tiles of 128 consecutive voxels x 64 channels, the taps split over eight wavefronts): exact operands equal the oracle byte for byte in
every output type at the edges of its tiles, rows and slots, statistics are the oracle's and identical run to run, split inputs and z-slabs included."""
import numpy as np
import pytest

from ufsm_amd import lib
import orc
from test_gpu_conv import exact_case, rand_case, gpu_conv
from test_gpu_thin import conv_in_slabs

pytestmark = pytest.mark.gpu


@pytest.fixture
def flat():
    lib.mi_conv_flat(1)
    yield
    lib.mi_conv_flat(-1)


# (bits, N, Ci, Co, D, H, W): one voxel; one, two and more pairs of blocks than LDS slots; a last tile of one voxel and of a whole run; odd numbers of channel
# tiles; rows of one voxel, of a run, the widest the kernel takes; two samples
SHAPES = [(8, 1, 64, 64, 1, 1, 1), (8, 1, 64, 64, 3, 43, 1), (8, 2, 128, 96, 3, 5, 7), (8, 1, 256, 40, 2, 4, 32), (8, 1, 64, 128, 3, 7, 41), (8, 2, 384, 64, 5, 6, 13),
          (8, 1, 128, 128, 4, 8, 16), (4, 1, 64, 64, 1, 43, 3), (4, 1, 64, 64, 1, 3, 41), (4, 2, 192, 192, 4, 9, 16), (4, 1, 448, 64, 3, 5, 26), (4, 1, 704, 72, 2, 4, 17)]


@pytest.mark.parametrize("bits,N,Ci,Co,D,H,W", SHAPES)
def test_flat_tiles(gpu, flat, bits, N, Ci, Co, D, H, W):
    rng = np.random.default_rng(Ci * 3 + Co + D * 7 + W)
    S = D * H * W
    xdt = 3 if bits == 8 else 4
    x, w, b = exact_case(rng, N, Ci, Co, S)
    xq = orc.f32_to_mx(bits, x, N, Ci, S)
    for ydt in (0, 2, xdt):
        want, _ = orc.conv3(xq, xdt, N, Ci, D, H, W, w, b, Co, ydt, cbits=bits, acc64=1)
        got, _ = gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, ydt, cbits=bits)
        assert "conv3_flat_k" in lib.mi_last_kernel().decode(), lib.mi_last_kernel().decode()
        assert np.array_equal(got, want), ydt
    x, w, b = rand_case(rng, N, Ci, Co, S)
    xq = orc.f32_to_mx(bits, x, N, Ci, S)
    G = 8 if Co % 32 == 0 else 2
    want, ws = orc.conv3(xq, xdt, N, Ci, D, H, W, w, b, Co, 0, cbits=bits, Go=G, want_stats=True)
    got, gs = gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, 0, cbits=bits, Go=G, stats=True)
    assert "conv3_flat_k" in lib.mi_last_kernel().decode()
    assert np.abs(got - want).max() / np.abs(want).max() < 2e-4   # (the conv tolerance of the other kernels' tests: fp32 sums in another order)
    # (the sums of many voxels average the outputs' differences away; those of a few carry them: the bound above)
    assert np.abs(gs - ws).max() / np.abs(ws).max() < (1e-5 if S >= 64 else 2e-4)
    got2, gs2 = gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, 0, cbits=bits, Go=G, stats=True)
    assert np.array_equal(got, got2) and np.array_equal(gs, gs2)


def test_taps_outside_the_volume_read_zeros(gpu, flat):
    """NaN blocks on the last voxel of a sample's first channel block reach only the voxels whose taps meet them: not the next row, plane, block or sample"""
    rng = np.random.default_rng(5)
    N, Ci, Co, D, H, W = 2, 64, 64, 4, 4, 8
    S = D * H * W
    x, w, b = rand_case(rng, N, Ci, Co, S)
    x[0, 3, S - 1] = np.nan
    got, _ = gpu_conv(orc.f32_to_mx(8, x, N, Ci, S), 3, N, Ci, D, H, W, w, b, Co, 0)
    assert "conv3_flat_k" in lib.mi_last_kernel().decode()
    exp = np.zeros((N, Co, D, H, W), bool); exp[0, :, D - 2:, H - 2:, W - 2:] = True
    assert np.array_equal(~np.isfinite(got.reshape(N, Co, D, H, W)), exp)


@pytest.mark.parametrize("bits,N,Ci,Co,D,H,W,slab,up", [(8, 1, 64, 64, 16, 16, 16, 4, 0), (8, 2, 128, 64, 12, 6, 14, 4, 1), (4, 1, 128, 64, 8, 11, 13, 4, 0)])
def test_slabs_give_the_whole_tensors_bytes(gpu, flat, bits, N, Ci, Co, D, H, W, slab, up):
    (whole, ws, k0), (parts, ps, k1) = conv_in_slabs(bits, N, Ci, Co, D, H, W, slab, up)
    assert "conv3_flat_k" in k0 and "conv3_flat_k" in k1
    assert np.array_equal(whole, parts) and np.array_equal(ws, ps)

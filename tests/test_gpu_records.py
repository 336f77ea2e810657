"""A network's convs keep the kernels their GroupNorm statistics were added on (mi_conv_keep_records): a statistic that moves by its last bit can move a code of the next layer's rows."""
import numpy as np
import pytest

from ufsm_amd import lib
import orc
from ufsm_amd.lp import DevBuf
from test_gpu_conv import exact_case, rand_case, gpu_conv

pytestmark = pytest.mark.gpu

# (bits, N, Ci, Co, D, H, W, a conv by itself, the same inside a network)
CASES = [(8, 1, 32, 32, 16, 32, 32, "conv3_small_k", "conv3_row1_k"), (8, 1, 96, 32, 32, 32, 32, "conv3_thin_k", "conv3_row_k"),
         (8, 1, 64, 64, 32, 32, 32, "conv3_flat_k", "conv3_row_k"), (8, 1, 128, 192, 6, 23, 21, "conv3_flat_k", "conv3_"), (4, 1, 128, 64, 16, 32, 32, "conv3_flat_k", "conv3_")]


@pytest.mark.parametrize("bits,N,Ci,Co,D,H,W,alone,inside", CASES)
def test_kernel_alone_and_inside_a_network(gpu, bits, N, Ci, Co, D, H, W, alone, inside):
    rng = np.random.default_rng(Ci + Co + D)
    x, w, b = exact_case(rng, N, Ci, Co, D * H * W)
    xdt = 3 if bits == 8 else 4
    xq = orc.f32_to_mx(bits, x, N, Ci, D * H * W)
    out = []
    for keep in (0, 1):
        was = lib.mi_conv_keep_records(keep)
        try:
            out.append(gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, xdt, cbits=bits, Go=8, stats=True))
            name = lib.mi_last_kernel().decode()
        finally:
            lib.mi_conv_keep_records(was)
        assert (alone if not keep else inside) in name and (not keep or alone not in name), name
    assert np.array_equal(out[0][0], out[1][0])                                  # the codes do not depend on it
    assert np.abs(out[0][1] - out[1][1]).max() <= 1e-6 * np.abs(out[1][1]).max()


def test_forward_takes_none_of_the_regrouping_kernels(gpu):
    from ufsm_amd.unet import UNet, make_cfg
    N, D, W, cout = 2, 56, 64, 8
    net = UNet(make_cfg(4, [32, 64, 128, 256], G=8, head_out=cout, act_dt=8, prec=0), N, D, W, W, seed=5)
    ct = DevBuf.from_numpy(np.random.default_rng(1).integers(1, 255, (N, D, W, W), dtype=np.uint8))
    off = DevBuf.from_numpy(np.full(N * D, 9.0, np.float32))
    y = []
    for mode in (-1, 0):                                                         # by size, and the flat kernel nowhere: the same bits
        lib.mi_conv_flat(mode)
        lg = DevBuf(N * cout * D * W * W * 4)
        try:
            assert net.forward_ct(ct.ptr, 120.0, 0.02, off.ptr, off.ptr, 0, lg.ptr) == 0
        finally:
            lib.mi_conv_flat(-1)
        lib.mi_sync()
        y.append(lg.to_numpy(np.uint32))
    assert np.array_equal(y[0], y[1])
    assert lib.mi_conv_keep_records(0) == 0                                      # the setting is the forward's, not the thread's afterwards


def test_short_walks_keep_the_precision_of_the_row_kernels_sums(gpu):
    """One block into one channel tile on the small-channel kernel, where the one-block row kernel ran: a record per wavefront of 128 voxels there too, so that no more
    is summed in fp32. The errors of the sums of squares against 64 bits have the row kernel's size: their root mean squares over 128 groups differ by 9 % by chance (1 / sqrt 128);
    a record per tile of 512 voxels gives 1.7 times."""
    err = {}
    for seed in range(4):
        rng = np.random.default_rng(40 + seed)
        N, C, D, H, W, G = 4, 32, 16, 32, 64, 8
        x, w, b = rand_case(rng, N, C, C, D * H * W)
        xq = orc.f32_to_mx(8, x, N, C, D * H * W)
        for thin, kern in ((-1, "conv3_small_k"), (0, "conv3_row1_k")):
            lib.mi_conv_thin(thin)
            try:
                y, s = gpu_conv(xq, 3, N, C, D, H, W, w, b, C, 0, Go=G, stats=True)
            finally:
                lib.mi_conv_thin(-1)
            assert kern in lib.mi_last_kernel().decode()
            ref = (y.astype(np.float64) ** 2).reshape(N, G, -1).sum(-1)
            err.setdefault(kern, []).append((s[..., 1] - ref) / ref)
    rms = {k: np.sqrt(np.mean(np.square(v))) for k, v in err.items()}
    assert rms["conv3_small_k"] < 1.35 * rms["conv3_row1_k"], rms

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
    assert np.array_equal(out[0][0], out[1][0])                                  # exact operands: the codes do not depend on it
    assert np.abs(out[0][1] - out[1][1]).max() <= 1e-6 * np.abs(out[1][1]).max()


@pytest.mark.parametrize("bits,N,Ci,Co,D,H,W,alone,inside", CASES)
def test_what_separates_the_two(gpu, bits, N, Ci, Co, D, H, W, alone, inside):
    """The kernels add the products in another order, too, not only the statistics: on operands of several magnitudes the fp32 outputs themselves differ in their
    last bits with e4m3 (an order-free sum of the statistics alone would not bring such a network's bits together), and the statistics by as little. (e2m1 products, of
    four significant bits at most, add up without a rounding here: what separates those two is the statistics' records.)"""
    rng = np.random.default_rng(2 * Ci + Co + D)
    x, w, b = rand_case(rng, N, Ci, Co, D * H * W)
    x *= np.exp(2 * rng.standard_normal(x.shape)).astype(np.float32)
    xdt = 3 if bits == 8 else 4
    xq = orc.f32_to_mx(bits, x, N, Ci, D * H * W)
    out = []
    for keep in (0, 1):
        was = lib.mi_conv_keep_records(keep)
        try:
            out.append(gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, 0, cbits=bits, Go=8, stats=True))
        finally:
            lib.mi_conv_keep_records(was)
        assert (inside if keep else alone) in lib.mi_last_kernel().decode()
    d = np.abs(out[0][0] - out[1][0])
    assert (d.any() or bits == 4) and d.max() <= 2e-4 * np.abs(out[1][0]).max()                 # (the conv tolerance of the other kernels' tests)
    assert np.abs(out[0][1] - out[1][1]).max() <= 1e-5 * np.abs(out[1][1]).max()


@pytest.mark.parametrize("xdt", [3, 4])
@pytest.mark.parametrize("Ci,Co,N", [(192, 192, 6), (64, 96, 12)])
def test_a_slice_of_three_channel_tiles_in_one_workgroup_or_three(gpu, xdt, Ci, Co, N):
    """96 and 192 output channels in e2m1: few tiles run a channel tile per workgroup, more run three. A sample's codes and sums are the same bits either way (operands of
    several magnitudes; the squares' sums are what a differently compiled epilogue would move)."""
    rng = np.random.default_rng(Ci + Co + xdt)
    D, H, W = 8, 16, 24                                                         # 16 tiles of 2 x 8 x 16 per sample and slice; past the K-split kernel's launches
    if Co == 96:
        D = 16
    S = D * H * W
    x, w, b = rand_case(rng, N, Ci, Co, S)
    x *= np.exp(2 * rng.standard_normal(x.shape)).astype(np.float32)
    was = lib.mi_conv_keep_records(1)
    try:
        xq = orc.f32_to_mx(8 if xdt == 3 else 4, x, N, Ci, S)
        y, gs = gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, 0, cbits=4, Go=8, stats=True)
        assert "MT 3" in lib.mi_last_kernel().decode(), lib.mi_last_kernel().decode()
        for n in (0, N - 1):
            q1 = orc.f32_to_mx(8 if xdt == 3 else 4, x[n:n + 1], 1, Ci, S)
            y1, g1 = gpu_conv(q1, xdt, 1, Ci, D, H, W, w, b, Co, 0, cbits=4, Go=8, stats=True)
            assert "MT 1" in lib.mi_last_kernel().decode(), lib.mi_last_kernel().decode()
            assert np.array_equal(np.asarray(y1).reshape(-1), np.asarray(y).reshape(N, -1)[n]) and np.array_equal(np.asarray(g1).reshape(-1), np.asarray(gs).reshape(N, -1)[n])
    finally:
        lib.mi_conv_keep_records(was)


def kernels_of(run):
    """The conv kernels of what run() launches, in order."""
    import ctypes as C
    lib.mi_kernel_timing(1)
    try:
        run()
        name = C.create_string_buffer(96)
        n = lib.mi_kernel_timing_launch(-1, None, None, None, 0)
        out = []
        for i in range(n):
            lib.mi_kernel_timing_launch(i, None, None, name, 96)
            out.append(name.value.decode())
    finally:
        lib.mi_kernel_timing(0)
    return out


# windows whose 32 -> 32, 96 -> 32 and deep convs the three rules would take
@pytest.mark.parametrize("N,D,W", [(1, 32, 32), (2, 56, 64)])
def test_forward_takes_none_of_the_regrouping_kernels(gpu, N, D, W):
    from ufsm_amd.unet import UNet, make_cfg
    cout = 8
    net = UNet(make_cfg(4, [32, 64, 128, 256], G=8, head_out=cout, act_dt=8, prec=0), N, D, W, W, seed=5)
    ct = DevBuf.from_numpy(np.random.default_rng(1).integers(1, 255, (N, D, W, W), dtype=np.uint8))
    off = DevBuf.from_numpy(np.full(N * D, 9.0, np.float32))
    y, names = [], []
    for mode in (-1, 0):                                                         # by size, and the flat kernel nowhere: the same bits
        lib.mi_conv_flat(mode)
        lg = DevBuf(N * cout * D * W * W * 4)
        try:
            names.append(kernels_of(lambda: net.forward_ct(ct.ptr, 120.0, 0.02, off.ptr, off.ptr, 0, lg.ptr)))
        finally:
            lib.mi_conv_flat(-1)
        lib.mi_sync()
        y.append(lg.to_numpy(np.uint32))
    assert np.array_equal(y[0], y[1]) and names[0] == names[1]
    # one block into one channel tile: the two 32 -> 32 convs of level 0 on the one-block row kernel; 96 -> 32 on the row kernel; no flat tiles anywhere
    assert not any("conv3_flat_k" in k or "conv3_small_k" in k for k in names[0]), names[0]
    assert sum("conv3_row1_k" in k for k in names[0]) >= 2 and any("conv3_row_k" in k and "blocks 3" in k for k in names[0]), names[0]
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

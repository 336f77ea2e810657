"""Which kernel a conv's default rule takes at the edges of the rules that choose by size, and that it gives the oracle's bytes there (exact operands)."""
import numpy as np
import pytest

from ufsm_amd import lib, LP, DevBuf, shape5, gnp_t, split_t
import orc
from gpuutil import code_mismatch_fraction
from test_gpu_conv import exact_case, rand_case, gpu_conv

pytestmark = pytest.mark.gpu

# (bits, N, Ci, Co, D, H, W, kernel): one block into one channel tile around 16 384 voxels, around 1 024 row tiles, with rows that runs of 32 fit worse than 16;
# three blocks into one channel tile around 128, 512 and (e2m1) 256 tiles of the K-split kernel; the flat kernel behind that kernel's 256 (more than 128 output
# channels) or 512 tiles, at rows of 41 and 42 voxels, at 256 and 512 workgroups, with odd block counts and at the e2m1 limits of blocks and runs
CASES = [(8, 1, 32, 32, 16, 32, 32, "conv3_small_k"), (8, 1, 32, 32, 15, 32, 32, "conv3_row1_k"), (4, 2, 32, 24, 16, 16, 32, "conv3_small_k"),
         (8, 4, 32, 32, 32, 32, 255, "conv3_row1_k"), (8, 4, 32, 32, 28, 32, 255, "conv3_small_k"), (4, 4, 32, 32, 32, 32, 240, "conv3_small_k"),
         (8, 1, 96, 32, 9, 30, 31, "conv3_thin_k"), (8, 1, 96, 32, 8, 32, 32, "conv3_row_k"), (8, 1, 96, 32, 32, 32, 32, "conv3_thin_k"), (8, 1, 96, 32, 33, 32, 32, "conv3_row_k"),
         (4, 1, 96, 32, 16, 32, 32, "conv3_thin_k"), (4, 1, 96, 32, 17, 32, 32, "conv3_row_k"),
         (8, 1, 128, 192, 6, 23, 21, "conv3_flat_k"), (8, 1, 128, 192, 6, 21, 21, "conv3_thin_k"), (8, 1, 64, 64, 10, 23, 41, "conv3_flat_k"), (8, 1, 64, 64, 10, 23, 42, "conv3_row_k"),
         (8, 1, 64, 64, 32, 32, 32, "conv3_flat_k"), (8, 1, 64, 64, 33, 32, 32, "conv3_row_k"), (8, 1, 96, 96, 16, 16, 24, "conv3_mx_k"),
         (4, 1, 64, 64, 16, 32, 32, "conv3_row_k"), (4, 1, 128, 64, 16, 32, 32, "conv3_flat_k"), (4, 1, 128, 64, 17, 32, 32, "conv3_wide_k")]


@pytest.mark.parametrize("bits,N,Ci,Co,D,H,W,kern", CASES)
def test_default_rule_at_its_edges(gpu, bits, N, Ci, Co, D, H, W, kern):
    rng = np.random.default_rng(Ci + 3 * Co + D + W)
    x, w, b = exact_case(rng, N, Ci, Co, D * H * W)
    xdt = 3 if bits == 8 else 4
    xq = orc.f32_to_mx(bits, x, N, Ci, D * H * W)
    got, _ = gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, xdt, cbits=bits)
    assert kern in lib.mi_last_kernel().decode(), lib.mi_last_kernel().decode()
    want, _ = orc.conv3(xq, xdt, N, Ci, D, H, W, w, b, Co, xdt, cbits=bits, acc64=1)
    assert np.array_equal(got, want)


# (bits, input channels): three blocks; four of e4m3 and seven of e2m1, whose halo chunk would not fit LDS in one piece on the general kernel
@pytest.mark.parametrize("bits,Ci", [(8, 96), (8, 128), (4, 96), (4, 224)])
@pytest.mark.parametrize("call", ["act", "split"])
def test_few_tiles_that_the_k_split_kernel_does_not_take(gpu, bits, Ci, call):
    """three blocks and more into one channel tile of 129 tiles and more go to the K-split kernel by default; a call it cannot run stays on the row kernel"""
    rng = np.random.default_rng(Ci + bits)
    N, Co, D, H, W, G, xdt = 1, 32, 9, 30, 31, 8, 3 if bits == 8 else 4
    x, w, b = (rand_case if call == "act" else exact_case)(rng, N, Ci, Co, D * H * W)
    xq = orc.f32_to_mx(bits, x, N, Ci, D * H * W)
    if call == "act":
        got = []
        for thin in (-1, 0):
            lib.mi_conv_thin(thin)
            try:
                got.append(gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, xdt, cbits=bits, fused=(1, None, None))[0])
            finally:
                lib.mi_conv_thin(-1)
            assert "conv3_row_k" in lib.mi_last_kernel().decode(), lib.mi_last_kernel().decode()
        assert np.array_equal(got[0], got[1])
        want, _ = orc.conv3(xq, xdt, N, Ci, D, H, W, w, b, Co, xdt, cbits=bits, fused_act=1)
        assert code_mismatch_fraction(bits, got[0], want, N, Co, D * H * W)[1]
        return
    lib.mi_conv_split(0)
    try:
        got, gs = gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, xdt, cbits=bits, Go=G, stats=True)
    finally:
        lib.mi_conv_split(-1)
    assert "conv3_row_k" in lib.mi_last_kernel().decode(), lib.mi_last_kernel().decode()
    want, ws = orc.conv3(xq, xdt, N, Ci, D, H, W, w, b, Co, xdt, cbits=bits, acc64=1, Go=G, want_stats=True)
    assert np.array_equal(got, want) and np.allclose(gs, ws, rtol=1e-6)


# few output voxels (runs of 32 that meet several planes, or part of one), three blocks into one channel tile, flat tiles of whole and of ragged rows, and the staged kernels beside them
@pytest.mark.parametrize("bits,N,Ci,Co,D,H,W,kern", [(8, 2, 64, 64, 7, 3, 5, "conv3_thin_k"), (4, 1, 96, 64, 6, 6, 7, "conv3_thin_k"), (8, 1, 96, 32, 9, 30, 31, "conv3_thin_k"),
                                                     (8, 1, 64, 64, 10, 23, 41, "conv3_flat_k"), (4, 1, 128, 64, 16, 32, 32, "conv3_flat_k"), (8, 1, 96, 32, 8, 32, 32, "conv3_row_k"),
                                                     (8, 1, 32, 32, 16, 32, 32, "conv3_small_k"), (8, 1, 96, 96, 16, 16, 24, "conv3_mx_k")])
def test_statistics_of_a_range_of_planes(gpu, bits, N, Ci, Co, D, H, W, kern):
    """A conv whose statistics leave planes at its ends out (zlo, zhi) runs on the kernel of the whole call: the same fp32 outputs on operands of several
    magnitudes, whose sums depend on their order, and the sums over the planes that are left (none, too)."""
    rng = np.random.default_rng(Ci + Co + D + W)
    S, G, xdt = D * H * W, 8, 3 if bits == 8 else 4
    x, w, b = rand_case(rng, N, Ci, Co, S)
    x *= np.exp(2 * rng.standard_normal(x.shape)).astype(np.float32)
    xq = orc.f32_to_mx(bits, x, N, Ci, S)
    y, _ = gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, 0, cbits=bits, Go=G, stats=True)
    assert kern in lib.mi_last_kernel().decode(), lib.mi_last_kernel().decode()
    v = y.reshape(N, G, Co // G, D, H * W).astype(np.float64)
    for lo, hi in ((1, 2), (0, D - 1), (4, 0), (D, 0), (1 << 28, 0), (0, 1 << 28)):
        got, gs = gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, 0, cbits=bits, Go=G, stats=True, zrange=(lo, hi))
        assert kern in lib.mi_last_kernel().decode(), lib.mi_last_kernel().decode()
        assert np.array_equal(got, y), (lo, hi)
        u = v[:, :, :, lo:max(lo, D - hi)]
        want = np.stack([u.sum((2, 3, 4)), (u * u).sum((2, 3, 4))], -1)
        # (sums in fp32 within a record of at most 512 voxels x 4 channels, in double between them: 2^-24 per addition, a random walk of them, against the sum of magnitudes)
        assert np.abs(gs - want).max() <= 1e-5 * max(np.abs(u).sum((2, 3, 4)).max(), (u * u).sum((2, 3, 4)).max(), 1e-30), (lo, hi)


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_the_stride_2_choice_leaves_stride_1_alone(gpu, mode):
    """mi_conv_s2_direct is about stride-2 convs: with it set, stride-1 convs run on the kernels of the default"""
    for bits, N, Ci, Co, D, H, W, kern in [(8, 1, 64, 64, 4, 5, 7, "conv3_thin_k"), (8, 1, 128, 32, 9, 30, 31, "conv3_thin_k"), (8, 1, 64, 64, 10, 23, 41, "conv3_flat_k")]:
        rng = np.random.default_rng(Ci + D)
        x, w, b = exact_case(rng, N, Ci, Co, D * H * W)
        xq = orc.f32_to_mx(bits, x, N, Ci, D * H * W)
        lib.mi_conv_s2_direct(mode)
        try:
            got, _ = gpu_conv(xq, 3, N, Ci, D, H, W, w, b, Co, 3)
        finally:
            lib.mi_conv_s2_direct(-1)
        assert kern in lib.mi_last_kernel().decode(), lib.mi_last_kernel().decode()
        assert np.array_equal(got, orc.conv3(xq, 3, N, Ci, D, H, W, w, b, Co, 3, acc64=1)[0])


@pytest.mark.parametrize("bits,Ci,Co,D,H,W,kern", [(8, 64, 64, 13, 5, 7, "conv3_thin_k"), (4, 96, 64, 12, 6, 7, "conv3_thin_k"), (8, 96, 32, 14, 28, 31, "conv3_thin_k"), (8, 128, 64, 15, 21, 33, "conv3_flat_k"),
                                                   (4, 128, 64, 17, 29, 31, "conv3_flat_k")])
def test_overlapping_slabs_that_count_their_own_planes(gpu, bits, Ci, Co, D, H, W, kern):
    """A tensor in slabs of four planes that compute one more plane on either side and leave it out of their statistics: the whole call's outputs, plane by plane,
    and its sums (planes of odd voxel counts: a slab's runs start inside a run of the whole tensor's)."""
    rng = np.random.default_rng(Ci + D + W)
    S, G, xdt = D * H * W, 8, 3 if bits == 8 else 4
    x, w, b = rand_case(rng, 1, Ci, Co, S)
    x *= np.exp(2 * rng.standard_normal(x.shape)).astype(np.float32)
    xq = orc.f32_to_mx(bits, x, 1, Ci, S)
    y, ws = gpu_conv(xq, xdt, 1, Ci, D, H, W, w, b, Co, 0, cbits=bits, Go=G, stats=True)
    assert kern in lib.mi_last_kernel().decode(), lib.mi_last_kernel().decode()
    dx, dw, db = DevBuf.from_numpy(xq), DevBuf.from_numpy(w), DevBuf.from_numpy(b)
    sums, out = DevBuf(G * 2 * 24), DevBuf(G * 2 * 8)
    lib.mi_gn_sums_zero(sums.ptr, 2 * G)
    for z in range(0, D, 4):
        z0, z1, own = max(z - 1, 0), min(z + 5, D), min(z + 4, D)
        sp = split_t(); sp.zi0, sp.Di, sp.zlo, sp.zhi = z0, D, z - z0, z1 - own
        dy = DevBuf(Co * (z1 - z0) * H * W * 4)
        f = lib.lp_conv_fwd_f8 if bits == 8 else lib.lp_conv_fwd_f4
        assert f(dx.ptr, xdt, shape5(1, Ci, z1 - z0, H, W), dw.ptr, db.ptr, Co, dy.ptr, 0, gnp_t(), sums.ptr, G, sp) == 0
        assert kern in lib.mi_last_kernel().decode(), lib.mi_last_kernel().decode()
        assert np.array_equal(dy.to_numpy(np.float32, (Co, z1 - z0, H * W)), y.reshape(Co, D, H * W)[:, z0:z1]), z
    lib.mi_gn_sums_get(sums.ptr, 2 * G, out.ptr)
    LP.check()
    v = np.abs(y.astype(np.float64)).reshape(G, -1)
    # (fp32 within records of 32 voxels x 4 channels, cut elsewhere in the slabs)
    assert np.abs(out.to_numpy(np.float64, (G, 2)) - ws[0]).max() <= 1e-5 * max(v.sum(1).max(), (v * v).sum(1).max())


def first_word():
    """The kernel that ran. (A name goes on with the form whose products and records the kernel has, which may be another kernel's: `in` does not tell the two apart.)"""
    return lib.mi_last_kernel().decode().split("<")[0].split(" ")[0]


# the calls that other tests look for conv3_mx_k in, with what runs there: few tiles by the staged kernels' rule (thin 0), the general kernel's three-tile slices, a last chunk of fewer blocks, more tiles than the pipelined form takes
@pytest.mark.parametrize("bits,N,Ci,Co,D,H,W,thin,kern", [
    (8, 1, 96, 128, 5, 9, 18, 0, "conv3_pipe_k"), (8, 1, 32, 128, 3, 8, 16, 0, "conv3_pipe_k"), (8, 2, 128, 256, 6, 10, 33, 0, "conv3_pipe_k"), (4, 1, 160, 128, 7, 8, 16, 0, "conv3_mx_k"),
    (4, 2, 64, 256, 4, 16, 16, 0, "conv3_pipe_k"), (8, 1, 384, 128, 4, 8, 16, 0, "conv3_pipe_k"), (8, 1, 96, 96, 16, 16, 24, -1, "conv3_mx_k"), (8, 1, 64, 128, 18, 32, 32, -1, "conv3_pipe_k"),
    (8, 1, 416, 128, 16, 64, 128, -1, "conv3_mx_k"), (8, 1, 64, 40, 3, 96, 96, 0, "conv3_pipe_k"), (8, 1, 64, 40, 4, 128, 128, 0, "conv3_mx_k"), (8, 2, 64, 40, 3, 96, 96, 0, "conv3_mx_k")])
def test_the_kernel_that_ran_is_the_first_word(gpu, bits, N, Ci, Co, D, H, W, thin, kern):
    rng = np.random.default_rng(Ci + Co + W)
    S, xdt = D * H * W, 3 if bits == 8 else 4
    dx, dw = DevBuf.from_numpy(orc.f32_to_mx(bits, rng.standard_normal((N, Ci, S)).astype(np.float32), N, Ci, S)), DevBuf.from_numpy(rng.standard_normal((Co, Ci, 27)).astype(np.float32))
    dy, sums = DevBuf((lib.lp_mx8_bytes if bits == 8 else lib.lp_mx4_bytes)(N, Co, S)), DevBuf(N * Co * 2 * 24)
    f, G = lib.lp_conv_fwd_f8 if bits == 8 else lib.lp_conv_fwd_f4, 8 if Co % 32 == 0 else Co
    lib.mi_conv_thin(thin)
    try:
        assert f(dx.ptr, xdt, shape5(N, Ci, D, H, W), dw.ptr, None, Co, dy.ptr, xdt, gnp_t(), sums.ptr, G, split_t()) == 0
    finally:
        lib.mi_conv_thin(-1)
    LP.check()
    assert first_word() == kern, lib.mi_last_kernel().decode()

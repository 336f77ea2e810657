"""The K-split kernel of conv launches with few output voxels: exact operands equal the oracle byte for byte in every output type at the edges of its
tiles (64 voxels x 32 channels, eight wavefronts over the K pairs), statistics are the oracle's and identical run to run, split inputs and z-slabs included, and
launches on both sides of its range's edges give the bytes of the staged kernels."""
import numpy as np
import pytest

from ufsm_amd import lib, LP, DevBuf, shape5, gnp_t, split_t
import orc
from gpuutil import to_mx, mx_bytes, dev_gn
from test_gpu_conv import exact_case, rand_case, gpu_conv

pytestmark = pytest.mark.gpu

# (bits, N, Ci, Co, D, H, W, stride): one voxel, fewer pairs than wavefronts have sets (one block), odd block counts (the last pair is half empty), a run
# that ends inside a tile, partial channel tiles, two samples, the largest launches of the range, stride 2 on odd dims
SHAPES = [(8, 1, 64, 64, 1, 1, 1, 1), (8, 2, 32, 48, 3, 5, 7, 1), (8, 1, 96, 33, 2, 4, 8, 1), (8, 3, 160, 64, 5, 3, 13, 1), (8, 1, 256, 256, 8, 8, 16, 1), (8, 2, 64, 64, 16, 16, 16, 1),
          (4, 1, 64, 64, 4, 4, 4, 1), (4, 2, 96, 40, 3, 7, 9, 1), (4, 1, 288, 128, 5, 13, 13, 1),
          (8, 1, 64, 64, 8, 8, 8, 2), (8, 2, 96, 128, 7, 9, 5, 2), (4, 1, 32, 32, 8, 12, 16, 2)]


@pytest.mark.parametrize("bits,N,Ci,Co,D,H,W,stride", SHAPES)
def test_few_voxels(gpu, bits, N, Ci, Co, D, H, W, stride):
    rng = np.random.default_rng(Ci * 3 + Co + D * 7 + W)
    S = D * H * W
    xdt = 3 if bits == 8 else 4
    x, w, b = exact_case(rng, N, Ci, Co, S)
    xq = orc.f32_to_mx(bits, x, N, Ci, S)
    for ydt in (0, 2, xdt):
        want, _ = orc.conv3(xq, xdt, N, Ci, D, H, W, w, b, Co, ydt, cbits=bits, stride=stride, acc64=1)
        lib.mi_conv_thin(512)                                     # (the kernel is right for shapes the default rule leaves to others, too)
        try:
            got, _ = gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, ydt, cbits=bits, stride=stride)
        finally:
            lib.mi_conv_thin(-1)
        assert "conv3_thin_k" in lib.mi_last_kernel().decode(), lib.mi_last_kernel().decode()
        assert np.array_equal(got, want), ydt
    if stride == 2:
        return
    x, w, b = rand_case(rng, N, Ci, Co, S)
    xq = orc.f32_to_mx(bits, x, N, Ci, S)
    G = 8 if Co % 32 == 0 else 2 if Co % 8 == 0 else 1
    if (Co // G) % 4:                                             # (per-channel statistics leave this kernel)
        return
    want, ws = orc.conv3(xq, xdt, N, Ci, D, H, W, w, b, Co, 0, cbits=bits, Go=G, want_stats=True)
    got, gs = gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, 0, cbits=bits, Go=G, stats=True)
    assert "conv3_thin_k" in lib.mi_last_kernel().decode()
    assert np.abs(got - want).max() / np.abs(want).max() < 2e-4   # (the conv tolerance of the other kernels' tests: fp32 sums in another order)
    # (the sums of many voxels average the outputs' differences away; those of a few carry them: the bound above)
    assert np.abs(gs - ws).max() / np.abs(ws).max() < (1e-5 if S >= 64 else 2e-4)
    got2, gs2 = gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, 0, cbits=bits, Go=G, stats=True)
    assert np.array_equal(got, got2) and np.array_equal(gs, gs2)


def test_border_rows_stay_out_of_other_planes(gpu):
    """A tap outside the volume reads nothing: NaN blocks on the last plane of one channel block and of the sample before reach only the voxels whose taps
    meet them (the rows that follow a plane in memory are the next block's)."""
    rng = np.random.default_rng(5)
    N, Ci, Co, D, H, W = 2, 64, 64, 4, 4, 8
    S = D * H * W
    x, w, b = rand_case(rng, N, Ci, Co, S)
    x[0, 3, S - 1] = np.nan                                       # sample 0, block 0, last voxel
    xq = orc.f32_to_mx(8, x, N, Ci, S)
    got, _ = gpu_conv(xq, 3, N, Ci, D, H, W, w, b, Co, 0)
    assert "conv3_thin_k" in lib.mi_last_kernel().decode()
    bad = ~np.isfinite(got.reshape(N, Co, D, H, W))
    exp = np.zeros((N, Co, D, H, W), bool); exp[0, :, D - 2:, H - 2:, W - 2:] = True
    assert np.array_equal(bad, exp)


def conv_in_slabs(bits, N, Ci, Co, D, H, W, slab, up=0):
    """One conv over the whole tensor and slab by slab into the planes of a second one (stored statistics): [(MX bytes, sums, kernel of the last call)]."""
    rng = np.random.default_rng(Ci + Co + D * 3 + W)
    S, G, dt = D * H * W, 8, 3 if bits == 8 else 4
    Cu = Ci // 2 if up else 0
    w = (rng.standard_normal((Co, Ci, 27)) * np.sqrt(2.0 / (Ci * 27))).astype(np.float32)
    dw, db = DevBuf.from_numpy(w), DevBuf.from_numpy((rng.standard_normal(Co) * 0.1).astype(np.float32))
    sp = split_t()
    if up:
        dx = to_mx(bits, rng.standard_normal((N, Cu, S // 8)).astype(np.float32)); dx2 = to_mx(bits, rng.standard_normal((N, Ci - Cu, S)).astype(np.float32))
        sp.x2, sp.c_split, sp.up = dx2.ptr, Cu, 1
    else:
        dx = to_mx(bits, rng.standard_normal((N, Ci, S)).astype(np.float32))
    sp.stored_stats = 1
    f, res = (lib.lp_conv_fwd_f8 if bits == 8 else lib.lp_conv_fwd_f4), []
    for planes in (D, slab):
        y, sums, out = DevBuf(mx_bytes(bits, N, Co, S)), DevBuf(N * G * 2 * 24), DevBuf(N * G * 2 * 8)
        lib.mi_gn_sums_zero(sums.ptr, 2 * N * G)
        for z0 in range(0, D, planes):
            sk = min(planes, D - z0)
            if planes < D:
                sp.zi0, sp.Di, sp.yzo, sp.yD = z0, D, z0, D
            assert f(dx.ptr, dt, shape5(N, Ci, sk, H, W), dw.ptr, db.ptr, Co, y.ptr, dt, gnp_t(), sums.ptr, G, sp) == 0
        lib.mi_gn_sums_get(sums.ptr, 2 * N * G, out.ptr)
        LP.check()
        res.append((y.to_numpy(np.uint8), out.to_numpy(np.float64), lib.mi_last_kernel().decode()))
    return res


# whole tensors past the kernel's range whose slabs are inside it, and whole tensors inside it on planes of an odd voxel count, of one that is no
# multiple of 32 voxels in four planes, and of so few that a run of 32 voxels holds several multiples of four planes
@pytest.mark.parametrize("bits,N,Ci,Co,D,H,W,slab,up,thin", [(8, 1, 192, 64, 32, 32, 32, 4, 0, False), (8, 1, 192, 64, 32, 32, 32, 8, 1, False), (8, 2, 192, 64, 24, 24, 24, 4, 0, False),
                                                             (4, 1, 96, 96, 24, 24, 24, 4, 0, False), (8, 1, 64, 64, 12, 5, 7, 4, 0, True), (8, 2, 64, 128, 12, 10, 6, 4, 1, True),
                                                             (8, 1, 256, 64, 10, 9, 5, 4, 0, True), (4, 1, 96, 64, 16, 6, 7, 8, 0, True),
                                                             (8, 1, 64, 64, 13, 1, 3, 4, 0, True), (8, 2, 64, 64, 18, 2, 1, 8, 0, True), (4, 3, 64, 64, 9, 3, 3, 4, 0, True)])
def test_slabs_equal_whole(gpu, bits, N, Ci, Co, D, H, W, slab, up, thin):
    """A conv run in z-slabs takes the kernel of the whole tensor's conv and its statistics over the same voxels: the same bytes, and sums that differ
    only by the order in which doubles are added."""
    (y, s, k), (yz, sz, kz) = conv_in_slabs(bits, N, Ci, Co, D, H, W, slab, up)
    assert ("conv3_thin_k" in k) == thin and ("conv3_thin_k" in kz) == thin, (k, kz)
    assert np.array_equal(y, yz)
    assert np.allclose(s, sz, rtol=1e-12, atol=1e-9)


# 128 channels and more: slices of 64 or 128 channels, or the coarse form, by the tiles of the whole tensor (thirteen input blocks: the general kernel's
# slices); last slabs of one to three planes
@pytest.mark.parametrize("bits,N,Ci,Co,D,H,W,slab,kern", [(8, 1, 128, 128, 32, 32, 32, 4, "conv3_wide_k"), (8, 1, 256, 256, 32, 32, 32, 8, "conv3_wide_k"), (8, 2, 64, 128, 32, 64, 64, 4, "conv3_wide_k"),
                                                          (8, 1, 64, 128, 18, 32, 32, 8, "conv3_mx_k"), (8, 1, 64, 64, 10, 16, 32, 4, "conv3_row_k"), (8, 2, 32, 32, 9, 16, 48, 4, "conv3_row1_k"),
                                                          (8, 1, 96, 32, 11, 16, 32, 4, "conv3_row_k"), (8, 1, 32, 32, 6, 8, 8, 4, "conv3_small_k"), (8, 1, 64, 128, 21, 32, 64, 4, "conv3_wide_k"),
                                                          (8, 1, 416, 128, 16, 64, 128, 4, "conv3_mx_k"), (4, 1, 192, 64, 25, 32, 32, 8, "conv3_wide_k"), (8, 1, 32, 128, 29, 24, 40, 4, "conv3_row1_k")])
def test_slabs_take_the_whole_tensors_kernel(gpu, bits, N, Ci, Co, D, H, W, slab, kern):
    (y, s, k), (yz, sz, kz) = conv_in_slabs(bits, N, Ci, Co, D, H, W, slab)
    assert kern + "<" in k and kern + "<" in kz, (k, kz)
    assert np.array_equal(y, yz)
    assert np.allclose(s, sz, rtol=1e-12, atol=1e-9)


@pytest.mark.parametrize("bits,dims,slab", [(8, (64, 64, 64), 8), (8, (24, 20, 12), 4), (4, (32, 20, 28), 4)])
def test_network_in_slabs(gpu, bits, dims, slab):
    """Three levels, one window: level 1 of 64^3 is past the kernel's range and its slabs would be inside it; the other windows' levels are inside it on
    planes of 60 and 70 voxels. Logits and every statistic are those of the forward over whole tensors."""
    from ufsm_amd.unet import UNet, make_cfg, load_host
    host = load_host()
    S = dims[0] * dims[1] * dims[2]
    net = UNet(make_cfg(4, [32, 64, 128], G=8, head_out=3, act_dt=bits), 1, *dims, seed=3)
    dx = to_mx(bits, np.random.default_rng(1).standard_normal((1, 4, S)).astype(np.float32))
    got = []
    for planes in (0, slab):
        host.unet_set_infer_slab(planes)
        try:
            out = DevBuf(3 * S * 4)
            assert net.forward_x(dx.ptr, out.ptr) == 0
            LP.check()
            st = []
            for k, (name, _, _) in enumerate(net.layer_outs()):
                g, mp, rp = net.layer_stats(k)
                for p in (mp, rp) if g else ():
                    a = np.empty(g, np.float32); lib.mi_d2h(a.ctypes.data, p, a.nbytes); st.append((name, a))
            got.append((out.to_numpy(np.float32), st))
        finally:
            host.unet_set_infer_slab(0)
    net.close()
    assert np.array_equal(got[0][0], got[1][0])
    assert [n for n, _ in got[0][1]] == [n for n, _ in got[1][1]]
    for (name, a), (_, b) in zip(got[0][1], got[1][1]):
        assert np.array_equal(a, b), name


@pytest.mark.parametrize("bits,Cu,Cs,Co", [(8, 64, 96, 64), (4, 96, 32, 128), (8, 256, 128, 128)])
def test_split_inputs(gpu, bits, Cu, Cs, Co):
    """[x | x2] read as stored (exact operands: the oracle's bytes), and [2x upsampled coarse | skip] with both GroupNorms (the staged
    kernels' result but for the order of sums)."""
    rng = np.random.default_rng(Cu + Cs)
    N, D, H, W, G, dt = 2, 6, 4, 10, 8, 3 if bits == 8 else 4
    S = D * H * W
    x, w, b = exact_case(rng, N, Cu + Cs, Co, S)
    qu, qs = orc.f32_to_mx(bits, np.ascontiguousarray(x[:, :Cu]), N, Cu, S), orc.f32_to_mx(bits, np.ascontiguousarray(x[:, Cu:]), N, Cs, S)
    want, _ = orc.conv3(qu, dt, N, Cu + Cs, D, H, W, w, b, Co, dt, cbits=bits, x2=qs, c_split=Cu, acc64=1)
    got, _ = gpu_conv(qu, dt, N, Cu + Cs, D, H, W, w, b, Co, dt, cbits=bits, x2=qs, c_split=Cu)
    assert "conv3_thin_k" in lib.mi_last_kernel().decode() and np.array_equal(got, want)
    xu = rng.standard_normal((N, Cu, S // 8)).astype(np.float32)
    _, w, b = rand_case(rng, N, Cu + Cs, Co, S)
    qu = orc.f32_to_mx(bits, xu, N, Cu, S // 8)
    g = [[rng.uniform(0.5, 1.5, c).astype(np.float32), rng.uniform(-0.3, 0.3, c).astype(np.float32), rng.uniform(-0.2, 0.2, N * G).astype(np.float32), rng.uniform(0.7, 1.4, N * G).astype(np.float32)] for c in (Cu, Cs)]
    res = []
    for thin in (-1, 0):
        lib.mi_conv_thin(thin)
        try:
            res.append(gpu_conv(qu, dt, N, Cu + Cs, D, H, W, w, b, Co, 0, cbits=bits, x2=qs, c_split=Cu, up=1, gp=dev_gn(*g[0], G), gp2=dev_gn(*g[1], G))[0])
        finally:
            lib.mi_conv_thin(-1)
        assert ("conv3_thin_k" in lib.mi_last_kernel().decode()) == (thin < 0)
    assert np.abs(res[0] - res[1]).max() / np.abs(res[1]).max() < 2e-4      # (the same staged operands: fp32 sums in another order)


def test_one_memo_id_on_both_kernels(gpu):
    """Prepared weights are kept per id and layout: one id alternating between a launch of this kernel, a staged one and a thread's other choice gives the
    bytes of weights prepared per call."""
    rng = np.random.default_rng(3)
    Ci, Co = 128, 64
    w = (rng.standard_normal((Co, Ci, 27)) * 0.03).astype(np.float32)
    dw, db = DevBuf.from_numpy(w), DevBuf.from_numpy(rng.standard_normal(Co).astype(np.float32))
    dims = [(8, 8, 8), (24, 24, 24)]
    xs = [to_mx(8, rng.standard_normal((1, Ci, D * H * W)).astype(np.float32)) for D, H, W in dims]

    def conv(i, wkey, thin):
        D, H, W = dims[i]
        sp, y = split_t(), DevBuf(mx_bytes(8, 1, Co, D * H * W))
        sp.wkey = wkey
        lib.mi_conv_thin(thin)
        try:
            assert lib.lp_conv_fwd_f8(xs[i].ptr, 3, shape5(1, Ci, D, H, W), dw.ptr, db.ptr, Co, y.ptr, 3, gnp_t(), None, 0, sp) == 0
        finally:
            lib.mi_conv_thin(-1)
        LP.check()
        return y.to_numpy(np.uint8), lib.mi_last_kernel().decode().split("<")[0]
    ref = {(i, t): conv(i, 0, t) for i in (0, 1) for t in (-1, 0)}
    assert ref[0, -1][1] == "conv3_thin_k" and all(ref[k][1] != "conv3_thin_k" for k in ((0, 0), (1, -1), (1, 0)))
    for k in [(0, -1), (1, -1), (0, 0), (0, -1), (1, 0), (1, -1), (0, -1)]:
        y, name = conv(k[0], 77001, k[1])
        assert name == ref[k][1] and np.array_equal(y, ref[k][0]), k
    lib.lp_wmemo_clear()

# (bits, Ci, Co, stride, [(N, D, H, W, the kernel takes it)]): the last launch of a limit and the one of a plane more
EDGES = [(8, 64, 64, 1, [(1, 32, 16, 16, True), (1, 33, 16, 16, False)]), (8, 256, 128, 1, [(1, 32, 16, 16, True), (1, 33, 16, 16, False)]),
         (4, 64, 128, 1, [(1, 8, 8, 16, True), (1, 9, 8, 16, False)]), (8, 32, 128, 1, [(1, 8, 8, 16, True), (1, 9, 8, 16, False)]), (4, 256, 128, 1, [(1, 16, 16, 16, True), (1, 17, 16, 16, False)]),
         (4, 32, 64, 1, [(2, 16, 16, 16, True), (1, 33, 16, 16, False)]), (4, 32, 128, 1, [(1, 4, 4, 4, False), (1, 11, 13, 13, False)]),
         (4, 32, 32, 2, [(1, 16, 16, 16, False), (2, 8, 12, 16, False)]), (8, 64, 64, 2, [(2, 32, 32, 32, True), (2, 33, 32, 32, False)]),
         (8, 256, 256, 2, [(1, 16, 32, 32, True), (2, 24, 24, 24, True), (1, 32, 32, 32, False)])]


@pytest.mark.parametrize("bits,Ci,Co,stride,launches", EDGES)
def test_edges_of_the_range(gpu, bits, Ci, Co, stride, launches):
    """The default choice at its limits, and exact operands: both kernels give the same bytes."""
    rng = np.random.default_rng(Ci + Co + stride)
    dt = 3 if bits == 8 else 4
    for N, D, H, W, thin in launches:
        x, w, b = exact_case(rng, N, Ci, Co, D * H * W)
        xq = orc.f32_to_mx(bits, x, N, Ci, D * H * W)
        got, name = [], []
        for limit in (-1, 0, 4096):
            lib.mi_conv_thin(limit)
            try:
                got.append(gpu_conv(xq, dt, N, Ci, D, H, W, w, b, Co, dt, cbits=bits, stride=stride)[0])
            finally:
                lib.mi_conv_thin(-1)
            name.append("conv3_thin_k" in lib.mi_last_kernel().decode())
        assert name == [thin, False, True], (N, D, H, W, name)
        assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])


@pytest.mark.parametrize("bits,N,Ci,Co,dims", [(8, 1, 64, 64, (16, 16, 16)), (8, 1, 64, 64, (17, 16, 16)), (4, 1, 96, 160, (5, 13, 25)), (8, 1, 96, 160, (5, 13, 26)), (8, 1, 33, 17, (1, 1, 1)),
                                               (8, 1, 1280, 32, (3, 5, 7)), (4, 2, 1216, 32, (4, 4, 5)), (8, 1, 128, 64, (2, 3, 5))])
def test_one_run_or_two_per_workgroup(gpu, bits, N, Ci, Co, dims):
    """128 tiles of 64 voxels (a run of 32 per workgroup) and 136, an odd number of runs, one voxel, every length of the walk's tail, and more input blocks than the table of 64 units holds."""
    rng = np.random.default_rng(Ci + Co + dims[2])
    D, H, W = dims
    x, w, b = exact_case(rng, N, Ci, Co, D * H * W)
    xdt = 3 if bits == 8 else 4
    xq = orc.f32_to_mx(bits, x, N, Ci, D * H * W)
    G = 8 if Co % 32 == 0 else 1
    stats = (Co // G) % 4 == 0
    got, gs = gpu_conv(xq, xdt, N, Ci, D, H, W, w, b, Co, xdt, cbits=bits, Go=G if stats else 0, stats=stats)
    assert "conv3_thin_k" in lib.mi_last_kernel().decode(), lib.mi_last_kernel().decode()
    want, ws = orc.conv3(xq, xdt, N, Ci, D, H, W, w, b, Co, xdt, cbits=bits, acc64=1, Go=G if stats else 0, want_stats=stats)
    assert np.array_equal(got, want)
    assert not stats or np.allclose(gs, ws, rtol=1e-6)


@pytest.mark.parametrize("bits,Ci,Co,dims,stride", [(8, 64, 64, (4, 4, 8), 1), (8, 256, 96, (3, 5, 7), 1), (4, 96, 64, (4, 4, 8), 1), (4, 384, 64, (3, 5, 9), 1), (8, 128, 64, (6, 7, 9), 2), (4, 96, 64, (8, 8, 8), 2)])
def test_one_run_or_two_per_workgroup_give_the_same_bits(gpu, bits, Ci, Co, dims, stride):
    """Up to 128 tiles of 64 voxels a workgroup takes one run of 32, beyond that two: a sample's fp32 outputs and statistics are the same bits, on operands of several magnitudes, whose sums
    depend on their order."""
    rng = np.random.default_rng(Ci + Co + stride)
    N, G, xdt = 70, 8, 3 if bits == 8 else 4
    D, H, W = dims
    x, w, b = rand_case(rng, N, Ci, Co, D * H * W)
    x *= np.exp(2 * rng.standard_normal(x.shape)).astype(np.float32)
    out = []
    for n in (N, 9, 1):
        lib.mi_conv_thin(4096)
        try:
            y, g = gpu_conv(orc.f32_to_mx(bits, x[:n], n, Ci, D * H * W), xdt, n, Ci, D, H, W, w, b, Co, 0, cbits=bits, stride=stride, **(dict(Go=G, stats=True) if stride == 1 else {}))
        finally:
            lib.mi_conv_thin(-1)
        name = lib.mi_last_kernel().decode()
        assert name.startswith("conv3_thin_k<") and (int(name.split("tiles ")[1]) > 128) == (n == N), name
        out.append((y, g))
    for n, (y, g) in zip((9, 1), out[1:]):
        assert np.array_equal(y.view(np.uint32), out[0][0][:n].view(np.uint32)) and (g is None or np.array_equal(g, out[0][1][:n]))

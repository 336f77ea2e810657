"""GPU parity of the 2x2x2 stride-2 conv and transposed conv (mi_conv_down2_fwd, mi_convt_up2_fwd) against the oracle's restatement, through the C ABI.
The reference has neither layer (src/lp_s2.cu:4-9, src/lp_mx_gn.cu:32-33); the oracle is pinned by fp64 closed forms in tests/test_oracle_conv2.py."""
import numpy as np
import pytest

from ufsm_amd import lib, LP, shape5, gnp_t, DevBuf
from gpuutil import dev_gn, mx_bytes
import orc
import refnp

pytestmark = pytest.mark.gpu


def gpu_conv2(up, xq, xdt, N, Ci, D, H, W, w, b, Co, ydt, cbits, gp=None):
    So = 8 * D * H * W if up else (D // 2) * (H // 2) * (W // 2)
    dx, dw = DevBuf.from_numpy(xq), DevBuf.from_numpy(w.astype(np.float32))
    db = DevBuf.from_numpy(b.astype(np.float32)) if b is not None else None
    if ydt >= 3:
        nbytes, dtype = mx_bytes(8 if ydt == 3 else 4, N, Co, So), np.uint8
    else:
        nbytes, dtype = N * Co * So * (2 if ydt == 2 else 4), (np.uint16 if ydt == 2 else np.float32)
    dy = DevBuf(nbytes)
    f = lib.mi_convt_up2_fwd if up else lib.mi_conv_down2_fwd
    rc = f(cbits, dx.ptr, xdt, shape5(N, Ci, D, H, W), dw.ptr, db.ptr if db is not None else None, Co, dy.ptr, ydt, gp if gp is not None else gnp_t())
    LP.check()
    assert rc == 0 and "conv2_mx_k" in lib.mi_last_kernel().decode()
    y = dy.to_numpy(dtype)
    return y.reshape(N, Co, So) if ydt < 3 else y


SHAPES = [(32, 32, (4, 8, 16)), (64, 48, (6, 10, 14)), (128, 256, (8, 8, 8)), (40, 16, (2, 6, 10)), (16, 64, (4, 4, 6)), (256, 128, (4, 4, 8)), (96, 8, (2, 2, 18))]


@pytest.mark.parametrize("up", [0, 1])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("Ci,Co,dims", SHAPES)
def test_exact_operands_equal_the_oracle(gpu, up, bits, Ci, Co, dims):
    """Operands exact in the formats: fp32 planes equal the oracle's fp64 accumulation bit for bit, MX-fp8 / MX-fp4 outputs byte for byte (every row
    width 8 / 16 / 32 of the output, ragged channel blocks, column counts that are no multiple of the 64-column wavefront tile, N 2)."""
    rng = np.random.default_rng(1000 * up + 100 * bits + Ci + Co)
    D, H, W = dims
    N, S = 2, D * H * W
    x = refnp.gen_exact(rng, (N, Ci, S))
    w = refnp.gen_exact(rng, (Ci, Co, 8), block_axis=0) if up else refnp.gen_exact(rng, (Co, Ci, 8))
    b = rng.integers(-8, 9, Co).astype(np.float32) * 0.25
    xdt = 3 if bits == 8 else 4
    xq = orc.f32_to_mx(bits, x, N, Ci, S)
    for ydt in (0, 3, 4):
        want = orc.conv2(xq, xdt, N, Ci, D, H, W, w, b, Co, ydt, up, cbits=bits, acc64=1)
        got = gpu_conv2(up, xq, xdt, N, Ci, D, H, W, w, b, Co, ydt, bits)
        assert np.array_equal(got, want), (ydt, np.abs(got.astype(np.float64) - want.astype(np.float64)).max())


@pytest.mark.parametrize("up", [0, 1])
@pytest.mark.parametrize("bits,xbits,gn", [(8, 8, False), (4, 4, False), (4, 8, False), (8, 4, False), (8, 8, True), (4, 8, True)])
def test_random_operands_within_tolerance(gpu, up, bits, xbits, gn):
    """N(0,1) data and Kaiming weights, a stored format that differs from the compute format, GroupNorm + SiLU on the input: conv outputs within 1e-3
    max-abs-rel of the fp64-accumulated oracle under e4m3 compute; under e2m1 compute the matrix cores add the products exactly, so without the
    device's SiLU in the way the bound is 1e-5 (one differing staged code would show as ~1e-2)."""
    rng = np.random.default_rng(50 + 10 * up + bits + xbits + gn)
    N, Ci, Co, D, H, W, G = 1, 96, 64, 4, 6, 8, 8
    S = D * H * W
    x = rng.standard_normal((N, Ci, S)).astype(np.float32)
    w = (rng.standard_normal((Ci, Co, 8) if up else (Co, Ci, 8)) * np.sqrt(2.0 / (Ci * (1 if up else 8)))).astype(np.float32)
    b = (rng.standard_normal(Co) * 0.1).astype(np.float32)
    xdt = 3 if xbits == 8 else 4
    xq = orc.f32_to_mx(xbits, x, N, Ci, S)
    p = [rng.uniform(.5, 1.5, Ci).astype(np.float32), rng.uniform(-.3, .3, Ci).astype(np.float32), rng.uniform(-.2, .2, N * G).astype(np.float32), rng.uniform(.7, 1.4, N * G).astype(np.float32)]
    want = orc.conv2(xq, xdt, N, Ci, D, H, W, w, b, Co, 0, up, cbits=bits, gp=orc.gn(*p, G) if gn else None, acc64=1)
    got = gpu_conv2(up, xq, xdt, N, Ci, D, H, W, w, b, Co, 0, bits, gp=dev_gn(*p, G) if gn else None)
    err = np.abs(got - want).max() / np.abs(want).max()
    assert err < (3e-2 if gn and bits == 4 else 1e-3 if bits == 8 else 1e-5), err


@pytest.mark.parametrize("up", [0, 1])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("Ci,Co,dims,kind", [
    (96, 160, (2, 6, 22), 1), (224, 40, (4, 2, 8), 1), (160, 96, (2, 10, 26), 1),      # odd block counts (a K pair without its second block), channel tiles that no slice of 2 or 4 fills, columns past a multiple of 256
    (256, 32, (2, 2, 2), 1), (64, 256, (8, 8, 16), 1),                                  # the smallest launch; every channel tile a chunk of its own
    (288, 32, (2, 4, 6), 0), (64, 16, (4, 4, 6), 0)])                                   # past the pairs that the transposed conv holds; 16-channel rows: the general kernel
def test_row_kernels_at_their_edges(gpu, up, bits, Ci, Co, dims, kind):
    """The kernels that write MX rows of 32 channels (one wavefront per 32 columns): equal to the oracle byte for byte on exact operands, and not taken outside their range."""
    rng = np.random.default_rng(7 * Ci + Co + up)
    D, H, W = dims
    N, S = 2, D * H * W
    x = refnp.gen_exact(rng, (N, Ci, S))
    w = refnp.gen_exact(rng, (Ci, Co, 8), block_axis=0) if up else refnp.gen_exact(rng, (Co, Ci, 8))
    b = rng.integers(-8, 9, Co).astype(np.float32) * 0.25
    xdt = 3 if bits == 8 else 4
    xq = orc.f32_to_mx(bits, x, N, Ci, S)
    for ydt in (3, 4):
        want = orc.conv2(xq, xdt, N, Ci, D, H, W, w, b, Co, ydt, up, cbits=bits, acc64=1)
        got = gpu_conv2(up, xq, xdt, N, Ci, D, H, W, w, b, Co, ydt, bits)
        assert np.array_equal(got, want), ydt
        rows = ("conv2_up_k" if up else "conv2_down_k") in lib.mi_last_kernel().decode()
        assert rows == (kind == 1 or (not up and Co > 16))


def test_config2_layers_at_full_size(gpu):
    """BASELINE configs[2]'s stride-2 layers in MX-fp4: the 2x2x2 down conv 128 -> 256 on 64^3 (N 2) and the 2x2x2 transposed conv 256 -> 128 on
    32^3 (N 2), inputs uniform[-3, 3], Kaiming weights, MX-fp4 in and out, against the oracle (fp64 accumulation of the same e2m1 operands: fp32
    planes within 1e-5, and the stored MX-fp4 codes byte for byte up to rows whose pre-rounding value sits on a code boundary: < 1e-4 of them)."""
    rng = np.random.default_rng(2)
    for up, Ci, Co, D in ((0, 128, 256, 64), (1, 256, 128, 32)):
        N, S = 2, D ** 3
        x = rng.uniform(-3, 3, (N, Ci, S)).astype(np.float32)
        w = (rng.standard_normal((Ci, Co, 8) if up else (Co, Ci, 8)) * np.sqrt(2.0 / (Ci * (1 if up else 8)))).astype(np.float32)
        xq = orc.f32_to_mx(4, x, N, Ci, S)
        want = orc.conv2(xq, 4, N, Ci, D, D, D, w, None, Co, 0, up, cbits=4, acc64=1)
        got = gpu_conv2(up, xq, 4, N, Ci, D, D, D, w, None, Co, 0, 4)
        err = np.abs(got - want).max() / np.abs(want).max()
        assert err < 1e-5, (up, err)
        wq = orc.conv2(xq, 4, N, Ci, D, D, D, w, None, Co, 4, up, cbits=4, acc64=1)
        gq = gpu_conv2(up, xq, 4, N, Ci, D, D, D, w, None, Co, 4, 4)
        assert (gq != wq).mean() < 1e-4, (up, (gq != wq).mean())


@pytest.mark.parametrize("up", [0, 1])
def test_weight_memo(gpu, up):
    """mi_conv_s2_wkey: the prepared weights are kept under the caller's id (no second preparation, no further allocation), give the bytes of the
    per-call preparation, are told apart by direction, and are dropped by a new weight step."""
    rng = np.random.default_rng(81 + up)
    N, Ci, Co, D, H, W = 1, 64, 64, 4, 4, 8
    S = D * H * W
    x = rng.standard_normal((N, Ci, S)).astype(np.float32)
    w = (rng.standard_normal((Ci, Co, 8) if up else (Co, Ci, 8)) * 0.1).astype(np.float32)
    xq = orc.f32_to_mx(8, x, N, Ci, S)
    So = 8 * S if up else S // 8
    dx, dw, dy = DevBuf.from_numpy(xq), DevBuf.from_numpy(w), DevBuf(mx_bytes(8, N, Co, So))
    f = lib.mi_convt_up2_fwd if up else lib.mi_conv_down2_fwd

    def run(key):
        if key:
            lib.mi_conv_s2_wkey(key)
        assert f(8, dx.ptr, 3, shape5(N, Ci, D, H, W), dw.ptr, None, Co, dy.ptr, 3, gnp_t()) == 0
        LP.check()
        return dy.to_numpy(np.uint8).copy()

    lib.lp_wmemo_clear()
    plain = run(0)
    first = run(777)
    allocs = lib.mi_alloc_count()
    second = run(777)
    assert lib.mi_alloc_count() == allocs
    assert np.array_equal(plain, first) and np.array_equal(plain, second)
    w2 = np.ascontiguousarray(-2 * w)
    lib.mi_h2d(dw.ptr, w2.ctypes.data, w2.nbytes)
    assert np.array_equal(run(777), plain)                        # (the kept image: the caller said the weights are constant)
    assert np.array_equal(run(0), run(0)) and not np.array_equal(run(0), plain)      # the id was consumed by its call: these prepare per call
    lib.lp_wmemo_step(12345)                                      # weights changed: a new step drops the memo (src/nn_lp.h:56)
    assert np.array_equal(run(777), run(0))
    lib.lp_wmemo_clear(); lib.lp_wmemo_step(0)


def test_refusals(gpu):
    x = DevBuf(1 << 16); w = DevBuf(1 << 16); y = DevBuf(1 << 20)
    assert lib.mi_conv_down2_fwd(8, x.ptr, 3, shape5(1, 32, 3, 4, 4), w.ptr, None, 32, y.ptr, 3, gnp_t()) == -1      # odd depth
    assert lib.mi_conv_down2_fwd(6, x.ptr, 3, shape5(1, 32, 4, 4, 4), w.ptr, None, 32, y.ptr, 3, gnp_t()) == -1      # compute format
    assert lib.mi_convt_up2_fwd(8, x.ptr, 0, shape5(1, 32, 4, 4, 4), w.ptr, None, 32, y.ptr, 3, gnp_t()) == -1       # fp32 planes in
    LP.check()


def cancelling_case(rng, up, N, Ci, Co, S):
    """Operands whose fp32 sums are mostly rounding: the second half of the input blocks repeats the first with the weights negated, at row scales of many powers of two, so that
    another order of the same products gives other codes nearly everywhere."""
    half = Ci // 64 * 32
    x = rng.standard_normal((N, Ci // 32, 32, S)) * np.exp2(rng.integers(-9, 10, (N, Ci // 32, 1, S)))
    x = x.reshape(N, Ci, S).astype(np.float32)
    w = (rng.standard_normal((Ci, Co, 8)) * 0.1).astype(np.float32)
    x[:, half:2 * half] = x[:, :half]
    w[half:2 * half] = -w[:half]
    return x, w if up else np.ascontiguousarray(w.transpose(1, 0, 2))


def both_kernels(up, xq, xdt, N, Ci, dims, w, b, Co, ydt, bits):
    """The bytes of the kernel for MX rows and of the general one, and the former's name."""
    out = []
    for mode in (-1, 0):
        lib.mi_conv2_rows(mode)
        try:
            y = gpu_conv2(up, xq, xdt, N, Ci, *dims, w, b, Co, ydt, bits)
        finally:
            lib.mi_conv2_rows(-1)
        out.append((y, lib.mi_last_kernel().decode()))
    assert out[0][1].startswith("conv2_up_k<" if up and Ci <= 256 else "conv2_mx_k<" if up else "conv2_down_k<") and out[1][1].startswith("conv2_mx_k<fmt %d, out %d, up %d" % (bits, 8 if ydt == 3 else 4, up)), out
    return out[0][0], out[1][0], out[0][1]


@pytest.mark.parametrize("up", [0, 1])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("N,Ci,Co,dims", [(1, 128, 64, (8, 12, 20)), (2, 224, 96, (6, 6, 18)), (1, 256, 256, (8, 8, 16)), (1, 64, 40, (12, 20, 14)), (3, 96, 160, (4, 6, 10)), (1, 640, 64, (4, 4, 10))])
def test_the_row_kernels_keep_the_general_ones_products_and_order(gpu, up, bits, N, Ci, Co, dims):
    """The same bytes as the general kernel where every sum shows its order: one, two and four channel tiles a workgroup, odd block counts, a partial channel tile."""
    rng = np.random.default_rng(Ci + 3 * Co + up)
    S, xdt = int(np.prod(dims)), 3 if bits == 8 else 4
    x, w = cancelling_case(rng, up, N, Ci, Co, S)
    xq = orc.f32_to_mx(bits, x, N, Ci, S)
    for ydt in (3, 4):
        got, ref, _ = both_kernels(up, xq, xdt, N, Ci, dims, w, None, Co, ydt, bits)
        assert np.array_equal(got, ref), (ydt, (got != ref).mean())
        if bits == 8 and Ci % 128 == 0:                                        # (with 64 channels the two halves meet inside one product, which is exact)
            assert (got != orc.conv2(xq, xdt, N, Ci, *dims, w, None, Co, ydt, up, cbits=bits, acc64=1)).mean() > 0.1      # (the operands do what they are for)


@pytest.mark.parametrize("up", [0, 1])
@pytest.mark.parametrize("bits", [8, 4])
def test_rows_that_are_not_finite(gpu, up, bits):
    """NaN and infinite inputs and biases, and sums past the largest fp32 number: the row kernels' own epilogue writes what the general one does."""
    rng = np.random.default_rng(60 + up + bits)
    N, Ci, Co, dims, xdt = 2, 128, 96, (4, 6, 18), 3 if bits == 8 else 4
    S = int(np.prod(dims))
    x = rng.standard_normal((N, Ci, S)).astype(np.float32)
    w = (rng.standard_normal((Ci, Co, 8) if up else (Co, Ci, 8)) * 0.1).astype(np.float32)
    b = rng.standard_normal(Co).astype(np.float32)
    clean = orc.f32_to_mx(bits, x, N, Ci, S)
    x[0, 3, 17], x[0, 40, 200], x[1, 127, S - 1], x[1, :, 100] = np.nan, np.inf, -np.inf, 3e38
    w[..., 0] *= 64                                                           # (tap 0: products of 3e38 and more)
    xq = orc.f32_to_mx(bits, x, N, Ci, S)
    for ydt in (3, 4):
        fin, _, _ = both_kernels(up, clean, xdt, N, Ci, dims, w, b, Co, ydt, bits)
        for q, bad in ((xq, None), (xq, np.inf), (clean, np.inf), (clean, np.nan)):      # (not a NaN bias on a NaN sum: the sign of what that gives is nobody's)
            bias = b.copy()
            if bad is not None:
                bias[5], bias[40] = bad, -bad
            got, ref, _ = both_kernels(up, q, xdt, N, Ci, dims, w, bias, Co, ydt, bits)
            assert np.array_equal(got, ref), (ydt, bad)
            assert not np.array_equal(got, fin)


# (Ci, Co, N, dims, chunks of a workgroup): one to four K pairs, odd block counts, chunk counts that divide neither the channel tiles nor the chunks there are (walks that start between
# two tap pairs, a shorter last one), up to every chunk in one workgroup
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("Ci,Co,N,dims,cpw", [(32, 96, 180, (2, 2, 3), 4), (96, 160, 180, (2, 2, 3), 7), (160, 160, 130, (1, 3, 5), 5), (224, 136, 260, (1, 2, 3), 10), (256, 96, 520, (1, 1, 2), 12),
                                              (64, 160, 60, (3, 5, 45), 7), (160, 96, 20, (7, 11, 41), 6)])
def test_long_walks_of_the_transposed_conv(gpu, bits, Ci, Co, N, dims, cpw):
    """conv2_up_k's walk over its two weight slots, three chunks and more per workgroup: the oracle's bytes on exact operands in the first and the last sample, and every sample the same
    bytes where the inputs are."""
    rng = np.random.default_rng(Ci + Co + N)
    S, xdt, ydt = int(np.prod(dims)), 3 if bits == 8 else 4, 3 if bits == 8 else 4
    one = refnp.gen_exact(rng, (2, Ci, S))
    x = np.concatenate([one[:1]] * (N - 1) + [one[1:]])
    w = refnp.gen_exact(rng, (Ci, Co, 8), block_axis=0)
    b = rng.integers(-8, 9, Co).astype(np.float32) * 0.25
    got, ref, name = both_kernels(1, orc.f32_to_mx(bits, x, N, Ci, S), xdt, N, Ci, dims, w, b, Co, ydt, bits)
    assert "chunks %d " % cpw in name, name
    assert np.array_equal(got, ref)
    want = orc.mx_to_f32(bits, orc.conv2(orc.f32_to_mx(bits, one, 2, Ci, S), xdt, 2, Ci, *dims, w, b, Co, ydt, 1, cbits=bits, acc64=1), 2, Co, 8 * S)
    dec = orc.mx_to_f32(bits, got, N, Co, 8 * S).reshape(N, Co, 8 * S)
    assert np.array_equal(dec[:-1], np.broadcast_to(want.reshape(2, Co, 8 * S)[0], dec[:-1].shape)) and np.array_equal(dec[-1], want.reshape(2, Co, 8 * S)[1])


@pytest.mark.parametrize("up", [0, 1])
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("Ci,Co,dims", [(96, 32, (4, 6, 10)), (64, 48, (6, 10, 14)), (128, 256, (8, 8, 8))])
def test_the_general_kernel_still_writes_rows(gpu, up, bits, Ci, Co, dims):
    """conv2_mx_k into MX rows of 32 channels, which tensors of 2^27 voxels a sample and more run on: one, two and four channel tiles, the oracle's bytes."""
    rng = np.random.default_rng(Ci + Co + up)
    N, S, xdt = 2, int(np.prod(dims)), 3 if bits == 8 else 4
    x = refnp.gen_exact(rng, (N, Ci, S))
    w = refnp.gen_exact(rng, (Ci, Co, 8), block_axis=0) if up else refnp.gen_exact(rng, (Co, Ci, 8))
    xq = orc.f32_to_mx(bits, x, N, Ci, S)
    for ydt in (3, 4):
        got, ref, _ = both_kernels(up, xq, xdt, N, Ci, dims, w, None, Co, ydt, bits)
        want = orc.conv2(xq, xdt, N, Ci, *dims, w, None, Co, ydt, up, cbits=bits, acc64=1)
        assert np.array_equal(ref, want) and np.array_equal(got, want)


@pytest.mark.parametrize("bits,Ci,Co,W,rows", [(8, 32, 96, 48, False), (8, 32, 96, 36, True), (8, 64, 96, 48, False), (8, 32, 192, 48, False), (8, 64, 192, 48, True), (8, 96, 96, 48, True), (4, 32, 96, 48, True),
                                               (8, 32, 64, 64, True), (8, 32, 128, 64, True)])
def test_short_sums_into_many_slices(gpu, bits, Ci, Co, W, rows):
    """e4m3 down convs of one and two blocks into three and more slices of their channel tiles, past one round of CUs, run on the general kernel; beside the line, and either side of it: the
    oracle's bytes on exact operands."""
    rng = np.random.default_rng(Ci + Co + W)
    N, D, H, xdt = 2, 48, 48, 3 if bits == 8 else 4                            # (54 workgroups of 256 columns per sample and slice at W 48, 41 at 36)
    S = D * H * W
    one = refnp.gen_exact(rng, (1, Ci, S))
    w = refnp.gen_exact(rng, (Co, Ci, 8))
    xq = orc.f32_to_mx(bits, np.concatenate([one, one]), N, Ci, S)
    got = gpu_conv2(0, xq, xdt, N, Ci, D, H, W, w, None, Co, xdt, bits)
    assert lib.mi_last_kernel().decode().startswith("conv2_down_k<" if rows else "conv2_mx_k<")
    want = orc.mx_to_f32(bits, orc.conv2(orc.f32_to_mx(bits, one, 1, Ci, S), xdt, 1, Ci, D, H, W, w, None, Co, xdt, 0, cbits=bits, acc64=1), 1, Co, S // 8).reshape(Co, -1)
    dec = orc.mx_to_f32(bits, got, N, Co, S // 8).reshape(N, Co, -1)
    assert np.array_equal(dec[0], want) and np.array_equal(dec[1], want)

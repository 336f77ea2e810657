"""The graph's conv on operand rows: mi_conv_fwd_gn_stage (conv, statistics and the next reader's GroupNorm + SiLU rows in one call) and mi_conv_up_staged against the
separate calls they stand for."""
import numpy as np
import pytest

from gpuutil import DevBuf, LP, lib, to_mx
from ufsm_amd import gnp_t, shape5, split_t

pytestmark = pytest.mark.gpu


def _bytes(bits, n, c, s):
    return (lib.lp_mx8_bytes if bits == 8 else lib.lp_mx4_bytes)(n, c, s)


def _conv_operands(rng, bits, n, ci, co, dims):
    s = int(np.prod(dims))
    x = to_mx(bits, rng.standard_normal((n, ci, s)).astype(np.float32))
    w = DevBuf.from_numpy((rng.standard_normal((co, ci, 27)) * np.sqrt(2.0 / (ci * 27))).astype(np.float32)); b = DevBuf.from_numpy((0.1 * rng.standard_normal(co)).astype(np.float32))
    return x, w, b, s


# channels per group 4 and 8; 12 and 24 (groups across blocks of 32 channels); 32; 64 (a group of two blocks); 128 (too wide for the pass: the separate reduction); 1 (per-channel
# records: likewise); odd volumes; more than 512 records per sample (likewise); three samples; one voxel
CASES = [(8, 1, 32, 32, (8, 8, 8), 8), (8, 2, 64, 64, (9, 11, 13), 8), (8, 1, 32, 96, (8, 8, 16), 8), (8, 1, 64, 192, (5, 7, 9), 8), (8, 3, 64, 256, (8, 8, 8), 8), (8, 1, 32, 128, (8, 9, 10), 2),
         (8, 1, 32, 128, (8, 8, 8), 1), (8, 1, 32, 32, (8, 8, 8), 32), (8, 1, 32, 32, (33, 64, 64), 8), (8, 1, 32, 32, (1, 1, 1), 8), (4, 2, 64, 64, (9, 11, 13), 8), (4, 1, 32, 32, (16, 24, 40), 8), (4, 1, 64, 192, (5, 7, 9), 8)]


@pytest.mark.parametrize("bits,n,ci,co,dims,G", CASES)
def test_conv_with_rows_equals_the_separate_calls(gpu, bits, n, ci, co, dims, G):
    rng = np.random.default_rng(co + dims[0] + G)
    x, w, b, s = _conv_operands(rng, bits, n, ci, co, dims)
    dt = 3 if bits == 8 else 4
    gamma, beta = DevBuf.from_numpy(rng.uniform(0.7, 1.3, co).astype(np.float32)), DevBuf.from_numpy((0.2 * rng.standard_normal(co)).astype(np.float32))
    sums = DevBuf(n * G * 2 * 24)
    xs, ys = shape5(n, ci, *dims), shape5(n, co, *dims)
    y0, m0, r0 = DevBuf(_bytes(bits, n, co, s)), DevBuf(n * G * 4), DevBuf(n * G * 4)
    assert lib.mi_conv_fwd_gn(bits, x.ptr, dt, xs, w.ptr, b.ptr, co, y0.ptr, dt, gnp_t(), sums.ptr, G, split_t(), 1e-5, m0.ptr, r0.ptr) == 0
    for f8, f4 in ((1, 0), (0, 1), (1, 1)):
        y, m, r = DevBuf(_bytes(bits, n, co, s)), DevBuf.from_numpy(np.full(n * G, np.nan, np.float32)), DevBuf.from_numpy(np.full(n * G, np.nan, np.float32))
        st8, st4 = DevBuf(_bytes(8, n, co, s)), DevBuf(_bytes(4, n, co, s))
        assert lib.mi_conv_fwd_gn_stage(bits, x.ptr, dt, xs, w.ptr, b.ptr, co, y.ptr, dt, gnp_t(), sums.ptr, G, split_t(), 1e-5, m.ptr, r.ptr, gamma.ptr, beta.ptr,
                                        st8.ptr if f8 else None, st4.ptr if f4 else None) == 0
        LP.check()
        assert np.array_equal(y.to_numpy(np.uint8), y0.to_numpy(np.uint8))
        assert np.array_equal(m.to_numpy(np.float32), m0.to_numpy(np.float32)) and np.array_equal(r.to_numpy(np.float32), r0.to_numpy(np.float32))      # (added in one order)
        g = gnp_t(gamma.ptr, beta.ptr, m.ptr, r.ptr, G)
        for st, sb, on in ((st8, 8, f8), (st4, 4, f4)):      # the rows are those of the pre-pass under the statistics returned
            if on:
                want = DevBuf(_bytes(sb, n, co, s))
                assert lib.mi_conv_prestage(y.ptr, dt, ys, g, want.ptr, sb) == 0
                assert np.array_equal(st.to_numpy(np.uint8), want.to_numpy(np.uint8))


@pytest.mark.parametrize("bits,ci,co,dims", [(8, 64, 64, (64, 64, 64)), (4, 64, 64, (64, 64, 64))])
def test_statistics_do_not_depend_on_the_batch(gpu, bits, ci, co, dims):
    """A sample's mean, rstd and rows alone and as the first of two, on both sides of the size where the pre-pass stops adding the records itself (16 MB of records read over the
    launch: 1 x 64 channels at 64^3 is the last, 2 the first past it). The input's second half in y is the first one's negative except near the halves' edges, large further in, and
    there is no bias: the large tiles' records cancel exactly, and what is left of the small ones, some ten bits, shows in which order they were added."""
    rng = np.random.default_rng(co)
    H, h, s, G = dims[1], dims[1] // 2, int(np.prod(dims)), 8
    a = 2.0 ** -22 * rng.standard_normal((ci, dims[0], h, dims[2])).astype(np.float32)
    a[:, :, 10:h - 10] *= 2.0 ** 40                               # (output rows 8 .. h - 9, whole tiles, are the other half's negative, and every large one among them)
    x1 = np.concatenate([a, -a], 2)
    small = np.r_[0:6, h - 6:h + 6, H - 6:H]
    x1[:, :, small] = 2.0 ** -22 * rng.standard_normal((ci, dims[0], len(small), dims[2]))
    x2 = np.stack([x1, rng.standard_normal(x1.shape).astype(np.float32)]).reshape(2, ci, s)
    w = DevBuf.from_numpy((rng.standard_normal((co, ci, 27)) * np.sqrt(2.0 / (ci * 27))).astype(np.float32)); b = DevBuf(co * 4)
    gamma, beta = DevBuf.from_numpy(rng.uniform(0.7, 1.3, co).astype(np.float32)), DevBuf.from_numpy((0.2 * rng.standard_normal(co)).astype(np.float32))
    dt, got = (3 if bits == 8 else 4), []
    for n in (1, 2):
        x = to_mx(bits, x2[:n])
        for staged in (True, False):
            y, st, sums, m, r = DevBuf(_bytes(bits, n, co, s)), DevBuf(_bytes(bits, n, co, s)), DevBuf(n * G * 48), DevBuf(n * G * 4), DevBuf(n * G * 4)
            args = (bits, x.ptr, dt, shape5(n, ci, *dims), w.ptr, b.ptr, co, y.ptr, dt, gnp_t(), sums.ptr, G, split_t(), 1e-5, m.ptr, r.ptr)
            if staged:
                assert lib.mi_conv_fwd_gn_stage(*args, gamma.ptr, beta.ptr, st.ptr if bits == 8 else None, st.ptr if bits == 4 else None) == 0
            else:
                assert lib.mi_conv_fwd_gn(*args) == 0
                assert lib.mi_conv_prestage(y.ptr, dt, shape5(n, co, *dims), gnp_t(gamma.ptr, beta.ptr, m.ptr, r.ptr, G), st.ptr, bits) == 0
            LP.check()
            nb, rb = co // 32, 32 if bits == 8 else 16
            rows = st.to_numpy(np.uint8)
            codes, scales = rows[:n * nb * s * rb].reshape(n, -1), rows[n * nb * s * rb:n * nb * s * (rb + 1)].reshape(n, -1)
            got.append((m.to_numpy(np.float32)[:G], r.to_numpy(np.float32)[:G], codes[0], scales[0]))
    assert np.abs(got[0][0]).max() > 0
    for other in got[1:]:
        for p, q in zip(got[0], other):
            assert np.array_equal(p, q)


def test_conv_with_rows_refuses(gpu):
    z = split_t(); z.Di, z.zi0 = 8, 0
    one = DevBuf(1 << 16)
    p = one.ptr
    xs = shape5(1, 32, 4, 4, 4)
    assert lib.mi_conv_fwd_gn_stage(8, p, 3, xs, p, p, 48, p, 3, gnp_t(), p, 8, split_t(), 1e-5, p, p, p, p, p, None) == -1      # a partial block of channels
    assert lib.mi_conv_fwd_gn_stage(8, p, 3, xs, p, p, 32, p, 0, gnp_t(), p, 8, split_t(), 1e-5, p, p, p, p, p, None) == -1      # planes out
    assert lib.mi_conv_fwd_gn_stage(8, p, 3, xs, p, p, 32, p, 3, gnp_t(), p, 8, z, 1e-5, p, p, p, p, p, None) == -1              # a z-range
    assert lib.mi_conv_fwd_gn_stage(8, p, 3, xs, p, p, 32, p, 3, gnp_t(), p, 8, split_t(), 1e-5, p, p, p, p, None, None) == -1   # nothing to write


@pytest.mark.parametrize("bits,n,cc,cs,dims", [(8, 1, 64, 32, (8, 8, 16)), (8, 2, 32, 32, (4, 6, 10)), (4, 1, 64, 64, (8, 8, 8))])
def test_upsampled_segment_as_rows(gpu, bits, n, cc, cs, dims):
    """The coarse segment as the e4m3 rows of its pre-pass (whatever the conv computes in) gives the bytes of the conv that transforms it itself."""
    rng = np.random.default_rng(cc + cs)
    dt, s, sc, co, G = (3 if bits == 8 else 4), int(np.prod(dims)), int(np.prod(dims)) // 8, 32, 8
    coarse, skip = to_mx(bits, rng.standard_normal((n, cc, sc)).astype(np.float32)), to_mx(bits, rng.standard_normal((n, cs, s)).astype(np.float32))
    w = DevBuf.from_numpy((rng.standard_normal((co, cc + cs, 27)) * 0.05).astype(np.float32)); b = DevBuf.from_numpy((0.1 * rng.standard_normal(co)).astype(np.float32))
    v = [DevBuf.from_numpy(a.astype(np.float32)) for a in (rng.uniform(0.7, 1.3, cc), 0.2 * rng.standard_normal(cc), 0.1 * rng.standard_normal(n * G), rng.uniform(0.8, 1.2, n * G))]
    g = gnp_t(v[0].ptr, v[1].ptr, v[2].ptr, v[3].ptr, G)
    conv = lib.lp_conv_fwd_f8 if bits == 8 else lib.lp_conv_fwd_f4
    sp = split_t(); sp.x2, sp.c_split, sp.up = skip.ptr, cc, 1
    sp.gp2.G = -1
    y0, y1, rows = DevBuf(_bytes(bits, n, co, s)), DevBuf(_bytes(bits, n, co, s)), DevBuf(_bytes(8, n, cc, sc))
    conv(coarse.ptr, dt, shape5(n, cc + cs, *dims), w.ptr, b.ptr, co, y0.ptr, dt, g, None, 0, sp)
    assert lib.mi_conv_prestage(coarse.ptr, dt, shape5(n, cc, *[d // 2 for d in dims]), g, rows.ptr, 8) == 0
    lib.mi_conv_up_staged(1)
    if bits == 4:
        lib.mi_conv_x2_dt(4)
    conv(rows.ptr, 3, shape5(n, cc + cs, *dims), w.ptr, b.ptr, co, y1.ptr, dt, gnp_t(), None, 0, sp)
    LP.check()
    assert np.array_equal(y0.to_numpy(np.uint8), y1.to_numpy(np.uint8)) and y0.to_numpy(np.uint8).any()


@pytest.mark.parametrize("how", ["empty", "refused", "static"])
def test_words_for_one_call_end_with_it(gpu, how):
    """mi_conv_up_staged and mi_conv_x2_dt belong to the next call: one that has nothing to do or is refused takes them, and the conv after it reads its operands as they are."""
    rng = np.random.default_rng(5)
    n, cc, cs, dims, co, G = 1, 32, 32, (4, 8, 8), 32, 8
    s = int(np.prod(dims))
    coarse, skip = to_mx(8, rng.standard_normal((n, cc, s // 8)).astype(np.float32)), to_mx(8, rng.standard_normal((n, cs, s)).astype(np.float32))
    w = DevBuf.from_numpy((rng.standard_normal((co, cc + cs, 27)) * 0.05).astype(np.float32)); b = DevBuf.from_numpy((0.1 * rng.standard_normal(co)).astype(np.float32))
    v = [DevBuf.from_numpy(a.astype(np.float32)) for a in (rng.uniform(0.7, 1.3, cc), 0.2 * rng.standard_normal(cc), 0.1 * rng.standard_normal(n * G), rng.uniform(0.8, 1.2, n * G))]
    g = gnp_t(v[0].ptr, v[1].ptr, v[2].ptr, v[3].ptr, G)
    sp = split_t(); sp.x2, sp.c_split, sp.up = skip.ptr, cc, 1
    sp.gp2.G = -1
    ys = [DevBuf(_bytes(8, n, co, s)) for _ in range(2)]
    for y, words in zip(ys, (False, True)):
        if words:
            lib.mi_conv_up_staged(1); lib.mi_conv_x2_dt(4)
            p = w.ptr
            if how == "empty":
                assert lib.lp_conv_fwd_f8(p, 3, shape5(0, 32, 4, 4, 4), p, p, 32, y.ptr, 3, gnp_t(), None, 0, split_t()) == 0
            elif how == "refused":
                assert lib.mi_conv_fwd_gn_stage(8, p, 3, shape5(1, 32, 4, 4, 4), p, p, 48, y.ptr, 3, gnp_t(), p, 8, split_t(), 1e-5, p, p, p, p, y.ptr, None) == -1
            else:
                assert lib.mi_conv_fwd_static(8, p, 3, shape5(1, 512, 64, 64, 64), p, p, 512, y.ptr, 3, g, None, 0, split_t()) == -1      # (more than the fixed scratch)
        lib.lp_conv_fwd_f8(coarse.ptr, 3, shape5(n, cc + cs, *dims), w.ptr, b.ptr, co, y.ptr, 3, g, None, 0, sp)
    LP.check()
    assert np.array_equal(ys[0].to_numpy(np.uint8), ys[1].to_numpy(np.uint8)) and ys[0].to_numpy(np.uint8).any()

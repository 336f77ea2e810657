#!/usr/bin/env python3
"""Benchmark of the MX U-Net forward path on one MI355X. Prints one JSON line.

value / ms_per_step (the metric's "U-Net infer voxels/s (128^3 patch, MX fp8)"): one forward of the reference-style
U-Net (cin 4, widths 32/64/128/256, two 3x3x3 convs + GroupNorm + SiLU per level, 3x3x3 stride-2 downs, trilinear 2x fused into the decoder
convs, skip concat, 1x1x1 head of 8 logits) over N 2 x 128^3 voxels, MX-fp8 storage and compute. A step = unet_forward_ct on the two uint8 CT
windows resident in HBM: the network input is built on the device inside the timed region (lp_pred_input_mx), then the graph runs; the prepared (quantised, re-laid-out) weights are memoised across forwards as an inference loop keeps them - the reference's
fp8 path re-quantises them per call (src/lp_f8fwd.cu:54-71; about 15 us per layer here). `roofline`: the forward's dominant kernel (most
total time among its conv launches, HIP events around every launch on its stream).
conv_stack (configs[1], the metric's "3x3x3 conv % of MFMA peak"): four 3x3x3 convs 128 -> 128, N 2, 64^3, MX-fp8, bias + GroupNorm(8)
statistics fused, the previous layer's GroupNorm + SiLU on the input; its own `roofline` is the conv kernel alone."""
import argparse
import ctypes as C
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.join(ROOT, "tests"))

METRIC = "U-Net infer voxels/s (128^3 patch, MX fp8) + 3x3x3 conv % of MFMA peak"
MFMA_PEAK_FP8_TFLOPS = 5033.0          # MI355X dense MXFP8 (2.5 PFLOP/s bf16 x 2)
MFMA_PEAK_FP4_TFLOPS = 10066.0         # dense MXFP4
# HBM bytes per launch of a kernel cannot be measured from inside the process: they come from the committed rocprofv3 --pmc runs of this very
# command (FETCH_SIZE, then WRITE_SIZE, scaled by a copy of known size), each summary carrying one line "traffic_bytes_per_launch: <bytes>"
TRAFFIC_PROFILES = {"dec0.c1": "profiles/conv3_row_f8_unet_dec0c1_hbm_traffic.txt", "conv_stack": "profiles/conv3_mx_f8_c128_64cube_hbm_traffic.txt"}


def profile_traffic(key):
    """(bytes per launch, source file) from the committed counter summary of a kernel, or (None, None) when there is none."""
    import re
    rel = TRAFFIC_PROFILES.get(key)
    path = os.path.join(ROOT, rel) if rel else None
    if not path or not os.path.exists(path):
        return None, None
    m = re.search(r"^traffic_bytes_per_launch:\s*([0-9.eE+]+)", open(path).read(), re.M)
    return (float(m.group(1)), rel) if m else (None, None)


def unet_leg(np, lib, LP, DevBuf, steps, warmup):
    """the reference-style U-Net forward (cin 4, widths 32/64/128/256, two 3x3x3 convs + GroupNorm + SiLU per level, 3x3x3 stride-2
    downs, trilinear 2x fused into the decoder convs, skip concat, 1x1x1 head of 8 logits), N 2 x 128^3, MX-fp8 storage and compute, random
    init, CT-like synthetic uint8 windows resident in HBM, the 4-channel MX input built on the device by every forward (unet_forward_ct, as the
    reference's predict does per window). Two timed passes: the forwards alone (wall clock: `value`), then the same number of forwards with an
    event pair around every conv launch (per-kernel times for the roofline; the events cost a little)."""
    from ufsm_amd.unet import UNet, make_cfg
    N, D, widths = 2, 128, [32, 64, 128, 256]
    S = D ** 3
    net = UNet(make_cfg(4, widths, G=8, head_out=8, act_dt=8), N, D, D, D, seed=1)
    rng = np.random.default_rng(3)
    f = rng.standard_normal((N, D, D, D)).astype(np.float32)
    for ax in (1, 2, 3):
        f = (np.roll(f, 1, ax) + f + np.roll(f, -1, ax)) / 3                      # smoothed field -> sheet structure
    sheet = np.sin(6 * f / f.std() + np.linspace(0, 8, D, dtype=np.float32)[None, None, None, :]) > 0
    ct = np.clip(np.where(sheet, rng.normal(170, 20, f.shape), rng.normal(60, 20, f.shape)), 0, 255).astype(np.uint8)
    mean, isd = float(ct.mean()), float(1.0 / ct.std())
    dct = DevBuf.from_numpy(ct)                                                       # [N][D][H][W] uint8, the two windows back to back
    # per window plane the row / column offset from the scroll axis (an axis outside the window, as in a scroll volume)
    dyo = DevBuf.from_numpy(np.full(N * D, -300.0, np.float32)); dxo = DevBuf.from_numpy(np.full(N * D, 200.0, np.float32))
    H_ = net.L
    xs5 = net.shape

    def fwd():
        net._mode()
        p = H_.unet_forward_ct(net.h, dct.ptr, mean, isd, dyo.ptr, dxo.ptr, 1, xs5, 2)
        net._unmode()
        return p
    for _ in range(warmup):
        assert fwd()
    lib.mi_sync(); LP.check()
    t0 = time.perf_counter()
    for _ in range(steps):
        fwd()                                                                       # (the logits stay in the net's own device buffer)
    lib.mi_sync(); LP.check()
    dt = (time.perf_counter() - t0) / steps
    # per-kernel: every conv launch of `steps` more forwards, grouped by kernel variant and layer position within the forward
    lib.mi_kernel_timing(1)
    for _ in range(steps):
        fwd()
    lib.mi_sync()
    nlog = lib.mi_kernel_timing_launch(-1, None, None, None, 0)
    per_fwd = nlog // steps
    layers = {}
    name = C.create_string_buffer(128); ms = C.c_float(0); fl = C.c_double(0)
    for i in range(nlog):
        lib.mi_kernel_timing_launch(i, C.byref(ms), C.byref(fl), name, 128)
        k = i % per_fwd
        e = layers.setdefault(k, {"kernel": name.value.decode(), "flops": fl.value, "ms": 0.0, "n": 0})
        e["ms"] += ms.value; e["n"] += 1
    lib.mi_kernel_timing(0); LP.check()
    order = ["enc0.c1", "enc0.c2", "down0", "enc1.c1", "enc1.c2", "down1", "enc2.c1", "enc2.c2", "down2", "enc3.c1", "enc3.c2",
             "dec2.c1", "dec2.c2", "dec1.c1", "dec1.c2", "dec0.c1", "dec0.c2"]
    convs = []
    for k in sorted(layers):
        e = layers[k]; avg = e["ms"] / e["n"]
        convs.append({"layer": order[k] if per_fwd == len(order) else "conv%d" % k, "kernel": e["kernel"], "avg_launch_ms": avg, "tflops": e["flops"] / avg / 1e9,
                      "frac_of_mxfp8_peak": e["flops"] / avg / 1e9 / MFMA_PEAK_FP8_TFLOPS, "flops_per_launch": e["flops"]})
    # conv FLOPs of one forward, logical channels, all taps (tests/bench_lp.c:46)
    fl, lv = 0.0, [(D >> i) ** 3 for i in range(len(widths))]
    for i, wd in enumerate(widths):
        fl += 2 * 27 * ((4 if i == 0 else widths[i - 1]) * wd + wd * wd) * lv[i]      # encoder block
        if i + 1 < len(widths):
            fl += 2 * 27 * wd * wd * lv[i + 1]                                    # stride-2 down conv, width kept (src/unet.c:2970)
            fl += 2 * 27 * ((widths[i + 1] + wd) * wd + wd * wd) * lv[i]          # decoder block on [up | skip]
    fl += 2 * widths[0] * 8 * lv[0]
    fl *= N
    net.close()
    dom = max(convs, key=lambda c: c["avg_launch_ms"])
    return {"workload": "configs[3]: U-Net forward from two uint8 CT windows in HBM (unet_forward_ct: input rows built on the device, then the graph), N 2 x 128^3, widths 32/64/128/256, MX-fp8", "value": N * S / dt, "unit": "voxels/s", "ms_per_forward": dt * 1e3,
            "steps": steps, "gflop_per_forward": fl / 1e9, "tflops": fl / dt / 1e12, "conv_launches": convs,
            "conv_ms_per_forward": sum(c["avg_launch_ms"] for c in convs)}, dom


def _time_calls(lib, LP, call, steps, warmup):
    """(wall ms per call, HIP-event ms per conv launch, kernel name) of `call` repeated back to back."""
    for _ in range(warmup):
        call()
    lib.mi_sync(); LP.check()
    lib.mi_kernel_timing(1)
    t0 = time.perf_counter()
    for _ in range(steps):
        call()
    lib.mi_sync()
    wall = (time.perf_counter() - t0) * 1e3 / steps
    nl = C.c_long(0)
    kms = lib.mi_kernel_timing_read(C.byref(nl)) / max(nl.value, 1)
    lib.mi_kernel_timing(0); LP.check()
    return wall, kms, lib.mi_last_kernel().decode(), int(nl.value)


def c0_leg(np, lib, LP, DevBuf, shape5, gnp_t, split_t, steps, warmup):
    """one 3x3x3 conv 32 -> 32, N 1, 64^3, seed 0: activations N(0,1) as fp32 planes quantised to MX-fp8 while staging (bit for bit
    lp_f32_to_mx8), Kaiming weights in MX-fp8 blocks of 32 input channels, fp32 accumulate, fp16 planes out, through lp_conv_fwd_f8. The
    case sits at the ridge, so it reports both the MFMA fraction of the conv kernel and the HBM rate of the whole call (quantising
    pre-pass + conv; algorithmic bytes: the fp32 planes in, the fp16 planes out, the prepared weights)."""
    N, Cc, D = 1, 32, 64
    S = D ** 3
    rng = np.random.default_rng(0)
    dx = DevBuf.from_numpy(rng.standard_normal((N, Cc, S)).astype(np.float32))
    dw = DevBuf.from_numpy((rng.standard_normal((Cc, Cc, 27)) * np.sqrt(2.0 / (Cc * 27))).astype(np.float32))
    dy = DevBuf(N * Cc * S * 2)
    sp = split_t(); sp.wkey = 300
    xs = shape5(N, Cc, D, D, D)
    wall, kms, kernel, nl = _time_calls(lib, LP, lambda: lib.lp_conv_fwd_f8(dx.ptr, 0, xs, dw.ptr, None, Cc, dy.ptr, 2, gnp_t(), None, 0, sp), steps, warmup)
    fl = 2.0 * 27 * Cc * Cc * N * S
    nbytes = N * Cc * S * 4 + N * Cc * S * 2 + 28 * Cc * Cc * 33 // 32
    lib.lp_wmemo_clear()
    return {"workload": "configs[0]: 3x3x3 conv 32 -> 32, N 1, 64^3, fp32 planes in (quantised to MX-fp8 E4M3 per 32 channels while staging), fp16 planes out, seed 0",
            "entry": "lp_conv_fwd_f8(x dtype 0, y dtype 2)", "kernel": kernel, "ms_per_call": wall, "conv_kernel_ms": kms, "gflop": fl / 1e9,
            "tflops_conv_kernel": fl / kms / 1e9, "frac_of_mxfp8_peak": fl / kms / 1e9 / MFMA_PEAK_FP8_TFLOPS,
            "algorithmic_bytes": nbytes, "GBps_whole_call": nbytes / wall / 1e6, "frac_of_hbm_peak": nbytes / wall / 1e6 / 8000.0}


def c2a_leg(np, lib, LP, DevBuf, shape5, gnp_t, split_t, steps, warmup):
    """configs[2], the 3x3x3 part: MX-fp4 E2M1 conv 256 -> 256, N 2, 32^3, inputs uniform[-3, 3], Kaiming weights, 32-element E8M0 blocks, fp32
    accumulate, MX-fp4 in and out, fused GroupNorm(8) statistics, through lp_conv_fwd_f4; roofline against the dense MXFP4 peak."""
    N, Cc, D, G = 2, 256, 32, 8
    S = D ** 3
    rng = np.random.default_rng(0)
    dx = DevBuf.from_numpy(rng.uniform(-3, 3, (N, Cc, S)).astype(np.float32))
    dxq = DevBuf(lib.lp_mx4_bytes(N, Cc, S)); lib.lp_f32_to_mx4(dx.ptr, N, Cc, S, dxq.ptr)
    dw = DevBuf.from_numpy((rng.standard_normal((Cc, Cc, 27)) * np.sqrt(2.0 / (Cc * 27))).astype(np.float32))
    db = DevBuf.from_numpy((rng.standard_normal(Cc) * 0.1).astype(np.float32))
    dy = DevBuf(lib.lp_mx4_bytes(N, Cc, S)); dsum = DevBuf(N * G * 2 * 24)
    sp = split_t(); sp.wkey = 301
    xs = shape5(N, Cc, D, D, D)
    wall, kms, kernel, nl = _time_calls(lib, LP, lambda: lib.lp_conv_fwd_f4(dxq.ptr, 4, xs, dw.ptr, db.ptr, Cc, dy.ptr, 4, gnp_t(), dsum.ptr, G, sp), steps, warmup)
    fl = 2.0 * 27 * Cc * Cc * N * S
    lib.lp_wmemo_clear()
    return {"workload": "configs[2]: MX-fp4 E2M1 3x3x3 conv 256 -> 256, N 2, 32^3, MX-fp4 in / out, GroupNorm(8) statistics fused, inputs uniform[-3, 3]",
            "entry": "lp_conv_fwd_f4", "ms_per_call": wall,
            "roofline": {"bound": "mfma", "kernel": kernel, "achieved": fl / kms / 1e9, "peak": MFMA_PEAK_FP4_TFLOPS, "unit": "TFLOP/s", "frac": fl / kms / 1e9 / MFMA_PEAK_FP4_TFLOPS,
                         "launches": nl, "avg_launch_ms": kms, "flops_per_launch": fl, "algorithmic_bytes": 2 * N * (Cc // 32) * S * 17 + 28 * Cc * Cc * 17 // 32, "traffic": None}}


def stack_fused_leg(np, lib, LP, DevBuf, shape5, gnp_t, split_t, steps, warmup):
    """configs[1] to the letter: 4 x (3x3x3 conv 128 -> 128, N 2, 64^3, MX-fp8 in / out) with bias + GroupNorm(8) affine + GELU + MX-fp8
    re-quantisation fused into each conv's epilogue (mi_conv_fwd_fused). A GroupNorm inside the producer's epilogue needs its statistics before
    the conv has run, so they are frozen (per (sample, group) mean / rstd fixed beforehand, as the reference's unet_gn_freeze inference mode)
    and enter as the per-channel affine a = rstd gamma, b = beta - mean a."""
    N, Cc, D, L = 2, 128, 64, 4
    S = D * D * D
    rng = np.random.default_rng(0)
    dx = DevBuf.from_numpy(rng.standard_normal((N, Cc, S)).astype(np.float32))
    x0 = DevBuf(lib.lp_mx8_bytes(N, Cc, S)); lib.lp_f32_to_mx8(dx.ptr, N, Cc, S, x0.ptr)
    act = [DevBuf(lib.lp_mx8_bytes(N, Cc, S)) for _ in range(2)]
    ws = [DevBuf.from_numpy((rng.standard_normal((Cc, Cc, 27)) * np.sqrt(2.0 / (Cc * 27))).astype(np.float32)) for _ in range(L)]
    bs = [DevBuf.from_numpy((rng.standard_normal(Cc) * 0.1).astype(np.float32)) for _ in range(L)]
    ea = [DevBuf.from_numpy(rng.uniform(0.8, 1.25, Cc).astype(np.float32)) for _ in range(L)]        # rstd[g] gamma[c] of the frozen statistics
    eb = [DevBuf.from_numpy(rng.uniform(-0.1, 0.1, Cc).astype(np.float32)) for _ in range(L)]
    xs = shape5(N, Cc, D, D, D)

    def step():
        src = x0
        for l in range(L):
            dst = act[l & 1]
            sp = split_t(); sp.wkey = 310 + l
            lib.mi_conv_fwd_fused(8, src.ptr, 3, xs, ws[l].ptr, bs[l].ptr, Cc, dst.ptr, 3, ea[l].ptr, eb[l].ptr, 2, gnp_t(), None, 0, sp)
            src = dst
    wall, kms, kernel, nl = _time_calls(lib, LP, step, steps, warmup)
    fl = 2.0 * 27 * Cc * Cc * N * S
    lib.lp_wmemo_clear()
    return {"workload": "configs[1] to the letter: 4 x (3x3x3 conv 128->128, N 2, 64^3, MX-fp8) with bias + frozen-statistics GroupNorm(8) affine + GELU + MX-fp8 requant in the conv epilogue",
            "entry": "mi_conv_fwd_fused(act 2)", "value": N * S / (wall * 1e-3), "unit": "voxels/s", "ms_per_step": wall, "tflops": L * fl / wall / 1e9,
            "roofline": {"bound": "mfma", "kernel": kernel, "achieved": fl / kms / 1e9, "peak": MFMA_PEAK_FP8_TFLOPS, "unit": "TFLOP/s", "frac": fl / kms / 1e9 / MFMA_PEAK_FP8_TFLOPS,
                         "launches": nl, "avg_launch_ms": kms, "flops_per_launch": fl, "algorithmic_bytes": 2 * N * (Cc // 32) * S * 33 + 28 * Cc * Cc * 33 // 32, "traffic": None}}


def hbm_leg(np, lib, LP, DevBuf):
    """The HBM-bound kernels of the path at the level-0 shapes of configs[3] (N 2, 32 channels, 128^3; the upsample from 64 channels at 64^3;
    the stem 4 -> 32): algorithmic bytes (each tensor read or written once: 33 / 32 B per MX-fp8 element) over the time of one call, averaged
    over 10 back-to-back calls between two device synchronisations, against the 8 TB/s HBM peak."""
    from ufsm_amd import shape5, gnp_t, split_t
    N, C, D = 2, 32, 128
    S = D ** 3
    rng = np.random.default_rng(5)
    mx = lambda c, s: N * ((c + 31) // 32) * s * 33 if c > 8 else N * s * 9
    x = rng.standard_normal((N, C, S)).astype(np.float32)
    dx = DevBuf.from_numpy(x); del x
    q = DevBuf(lib.lp_mx8_bytes(N, C, S)); q2 = DevBuf(lib.lp_mx8_bytes(N, C, S))
    lib.lp_f32_to_mx8(dx.ptr, N, C, S, q.ptr)
    G = 8
    gam = DevBuf.from_numpy(rng.uniform(0.5, 1.5, C).astype(np.float32)); bet = DevBuf.from_numpy(rng.uniform(-.5, .5, C).astype(np.float32))
    mean = DevBuf.from_numpy(rng.uniform(-.2, .2, N * G).astype(np.float32)); rstd = DevBuf.from_numpy(rng.uniform(.8, 1.2, N * G).astype(np.float32))
    gp = gnp_t(gam.ptr, bet.ptr, mean.ptr, rstd.ptr, G)
    s5 = shape5(N, C, D, D, D)
    sums = DevBuf(N * G * 2 * 24)
    w1 = DevBuf.from_numpy((rng.standard_normal((8, C)) * 0.1).astype(np.float32)); b1 = DevBuf.from_numpy(np.zeros(8, np.float32))
    logits = DevBuf(N * 8 * S * 4)
    Cc, Sc = 64, (D // 2) ** 3
    xc = DevBuf.from_numpy(rng.standard_normal((N, Cc, Sc)).astype(np.float32)); qc = DevBuf(lib.lp_mx8_bytes(N, Cc, Sc)); lib.lp_f32_to_mx8(xc.ptr, N, Cc, Sc, qc.ptr)
    qu = DevBuf(lib.lp_mx8_bytes(N, Cc, S))
    x4 = DevBuf.from_numpy(rng.standard_normal((N, 4, S)).astype(np.float32)); q4 = DevBuf(lib.lp_mx8_bytes(N, 4, S)); lib.lp_f32_to_mx8(x4.ptr, N, 4, S, q4.ptr)
    ws = DevBuf.from_numpy((rng.standard_normal((C, 4, 27)) * 0.1).astype(np.float32)); bs = DevBuf.from_numpy(np.zeros(C, np.float32))
    sp = split_t(); sp.wkey = 901
    cases = [
        ("f32_to_mx_k (lp_f32_to_mx8, 32 ch)", N * C * S * 4 + mx(C, S), lambda: lib.lp_f32_to_mx8(dx.ptr, N, C, S, q2.ptr)),
        ("mx_to_f32_k (lp_mx8_to_f32, 32 ch)", N * C * S * 4 + mx(C, S), lambda: lib.lp_mx8_to_f32(q.ptr, N, C, S, dx.ptr)),
        ("gn_silu_apply_mx_k (GN + SiLU + requant, 32 ch; the conv pre-pass restage32_k is the same arithmetic)", 2 * mx(C, S), lambda: lib.lp_gn_silu_apply_mx(q.ptr, 3, s5, G, gam.ptr, bet.ptr, mean.ptr, rstd.ptr, q2.ptr, 3)),
        ("gn_sums_mx_k (lp_gn_sums_mx, 32 ch)", mx(C, S), lambda: lib.lp_gn_sums_mx(q.ptr, 3, N, C, G, S, sums.ptr, 0, S)),
        ("add_mx_k (lp_add_mx, 32 ch)", 3 * mx(C, S), lambda: lib.lp_add_mx(q2.ptr, q.ptr, s5, 3, 0)),
        ("conv1_mx_k (1x1x1 head 32 -> 8 with GN + SiLU, fp32 logits)", mx(C, S) + N * 8 * S * 4, lambda: lib.lp_conv1_fwd_mx(q.ptr, 3, s5, w1.ptr, b1.ptr, 8, logits.ptr, gp)),
        ("up2_mx_k (trilinear 2x, 64 ch, 64^3 -> 128^3)", mx(Cc, Sc) + mx(Cc, S), lambda: lib.lp_up2_fwd_mx(qc.ptr, 3, shape5(N, Cc, D // 2, D // 2, D // 2), qu.ptr, 3, gnp_t())),
        ("conv3_stem_k (3x3x3 stem 4 -> 32, MX-fp8 in / out)", mx(4, S) + mx(C, S), lambda: lib.lp_conv_fwd_f8(q4.ptr, 3, shape5(N, 4, D, D, D), ws.ptr, bs.ptr, C, q2.ptr, 3, gnp_t(), None, 0, sp)),
    ]
    # configs[2]'s stride-2 layers in MX-fp4 (N 2): 2x2x2 down conv 128 -> 256 from 64^3 and 2x2x2 transposed conv 256 -> 128 from 32^3 (weights prepared once
    # under a memo id, as an inference loop keeps them: mi_conv_s2_wkey)
    mx4 = lambda c, s: N * ((c + 31) // 32) * s * 17
    xd = DevBuf.from_numpy(rng.uniform(-3, 3, (N, 128, 64 ** 3)).astype(np.float32)); qd = DevBuf(lib.lp_mx4_bytes(N, 128, 64 ** 3)); lib.lp_f32_to_mx4(xd.ptr, N, 128, 64 ** 3, qd.ptr)
    yd = DevBuf(lib.lp_mx4_bytes(N, 256, 32 ** 3)); yu = DevBuf(lib.lp_mx4_bytes(N, 128, 64 ** 3))
    wd = DevBuf.from_numpy((rng.standard_normal((256, 128, 8)) * 0.04).astype(np.float32))
    cases += [
        ("conv2_down_k (2x2x2 stride-2 down conv 128 -> 256, 64^3 in, MX-fp4)", mx4(128, 64 ** 3) + mx4(256, 32 ** 3), lambda: (lib.mi_conv_s2_wkey(902), lib.mi_conv_down2_fwd(4, qd.ptr, 4, shape5(N, 128, 64, 64, 64), wd.ptr, None, 256, yd.ptr, 4, gnp_t()))),
        ("conv2_up_k (2x2x2 stride-2 transposed conv 256 -> 128, 32^3 in, MX-fp4)", mx4(256, 32 ** 3) + mx4(128, 64 ** 3), lambda: (lib.mi_conv_s2_wkey(903), lib.mi_convt_up2_fwd(4, yd.ptr, 4, shape5(N, 256, 32, 32, 32), wd.ptr, None, 128, yu.ptr, 4, gnp_t()))),
    ]
    rows = []
    for name, nbytes, call in cases:
        for _ in range(3):
            call()
        lib.mi_sync(); LP.check()
        t0 = time.perf_counter()
        for _ in range(10):
            call()
        lib.mi_sync(); LP.check()
        dt = (time.perf_counter() - t0) / 10
        rows.append({"kernel": name, "bytes": nbytes, "us": dt * 1e6, "GBps": nbytes / dt / 1e9, "frac_of_hbm_peak": nbytes / dt / 8e12})
    lib.lp_wmemo_clear()
    return rows


def sliding_leg(np, lib, LP, DevBuf, nbatch=64, radial=False):
    """a 512 x 1024 x 1024 uint8 volume resident in HBM, 128^3 windows with 16 voxels of halo (stride 96), per window a U-Net of
    widths 32/64/128/192 with MX-fp4 weights over MX-fp8 activations (prec 3) and two transformer blocks (MX-fp8 attention core, MX-fp8
    linears, 4 heads of 48, axial RoPE, 4 register tokens) on the 16^3 = 4096 bottleneck tokens, one head channel, sigmoid -> uint8
    placement and the 16-voxel feather blend of the window borders; end-to-end output voxels per second including gather, placement and blend.
    radial: the attention of the reference's production fine-tune instead (attn_axis 1, attn_pe 3: each block attends along the rays of the scroll
    coordinates, rotary embedding on (r, arc, z), no register tokens; the driver plans every forward's rays from its windows' axis records)."""
    from ufsm_amd.unet import UNet, make_cfg
    dims, W, halo, B = (512, 1024, 1024), 128, 16, 16
    rng = np.random.default_rng(7)
    z = np.arange(dims[0], dtype=np.float32)[:, None, None]; y = np.arange(dims[1], dtype=np.float32)[None, :, None]; x = np.arange(dims[2], dtype=np.float32)[None, None, :]
    r = np.sqrt((y - 400.0) ** 2 + (x + 300.0) ** 2)                                 # sheets wound around an axis outside the volume
    vol = (115 + 55 * np.sin(r * 0.35 + 0.02 * z)).astype(np.float32)
    vol += rng.integers(-20, 21, (1, dims[1], dims[2])).astype(np.float32) + rng.integers(-10, 11, (dims[0], 1, 1)).astype(np.float32)
    vol = np.clip(vol, 1, 255).astype(np.uint8)
    akw = dict(attn_pe=3, attn_axis=1, attn_reg=0) if radial else dict(attn_pe=1, attn_reg=4)
    net = UNet(make_cfg(4, [32, 64, 128, 192], G=8, head_out=1, act_dt=8, prec=3, attn_blocks=2, **akw), nbatch, W, W, W, seed=1)  # nbatch windows per forward
    dv = DevBuf.from_numpy(vol); dout = DevBuf(vol.size, zero=False)
    small = (W, W, W)                                                                 # warm-up: one window (weights prepared, scratch grown)
    rc, _, _ = net.predict_volume(dv.ptr, small, halo, B, 115.0, 1 / 40.0, 1, 400.0, -300.0, dout.ptr)
    assert rc == 0
    lib.mi_sync(); LP.check()
    t0 = time.perf_counter()
    rc, nw, ndone = net.predict_volume(dv.ptr, dims, halo, B, 115.0, 1 / 40.0, 1, 400.0, -300.0, dout.ptr)
    lib.mi_sync(); LP.check()
    dt_first = time.perf_counter() - t0
    assert rc == 0
    # the driver evens the windows out over its forwards, so the first prediction of a volume builds the graph for that sample count (activation
    # buffers, scratch): the second prediction of the same volume is the steady state the other legs' warm-up steps give them
    t0 = time.perf_counter()
    rc, nw, ndone = net.predict_volume(dv.ptr, dims, halo, B, 115.0, 1 / 40.0, 1, 400.0, -300.0, dout.ptr)
    lib.mi_sync(); LP.check()
    dt = time.perf_counter() - t0
    assert rc == 0
    head = dout.to_numpy(np.uint8)[:1 << 20]
    net.close()
    nvox = float(dims[0]) * dims[1] * dims[2]
    return {"workload": "configs[4]: 512x1024x1024 uint8 in HBM, 128^3 windows, halo 16, feather 16, U-Net 32/64/128/192, MX-fp4 weights over MX-fp8 activations, 2 attention blocks on 16^3 tokens (%s), up to %d windows per forward" % ("radial: 512 rays of 24 slots per window, fp16 core, scroll RoPE" if radial else "MX-fp8 core", nbatch),
            "value": nvox / dt, "unit": "voxels/s", "seconds": dt, "seconds_first_call": dt_first, "windows": int(nw), "windows_computed": int(ndone), "output_mean_first_mib": float(head.mean())}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=30)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--cpu-seconds", type=float, default=15.0, help="target seconds of CPU work for the cpu_baseline sample")
    ap.add_argument("--no-stack", action="store_true", help="skip the configs[1] conv-stack leg")
    ap.add_argument("--no-sliding", action="store_true", help="skip the configs[4]-geometry sliding-window leg")
    ap.add_argument("--no-hbm", action="store_true", help="skip the HBM-bound kernels leg")
    ap.add_argument("--no-single", action="store_true", help="skip the single-conv legs (configs[0], the MX-fp4 3x3x3 conv of configs[2])")
    ap.add_argument("--unet-only", action="store_true", help="the U-Net leg alone (what the rocprofv3 runs of the forward's kernels use)")
    ap.add_argument("--sliding-radial", action="store_true", help="also run the sliding-window leg with radial attention and scroll RoPE (sub-record sliding_window_radial)")
    ap.add_argument("--windows-per-forward", type=int, default=64, help="sliding-window leg: the most windows batched into one forward (the driver evens them out over its forwards)")
    ap.add_argument("--copy-probe", action="store_true", help="run 5 device-to-device copies of 1 GiB and exit: the known-size kernel that scales "
                    "rocprofv3's FETCH_SIZE / WRITE_SIZE counters")
    ap.add_argument("--conv-probe", default="", metavar="Ci,Co,N,D,bits", help="time one 3x3x3 conv shape (MX in / out of the compute format, fused statistics) "
                    "over --steps launches after --warmup, print one JSON line and exit: the command rocprofv3 counter runs of the other conv kernels use")
    a = ap.parse_args()
    if a.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py: this build runs on one GPU; --gpus %d is not supported (the path would shard by whole windows, or by z-slabs of one window with a one-plane halo exchange per layer)" % a.gpus, file=sys.stderr)
        sys.exit(2)
    import numpy as np
    from ufsm_amd import lib, LP, shape5, gnp_t, split_t, DevBuf
    if lib.mi_init(0) != 0:
        print("bench.py: no gfx950 GPU: the HIP path cannot run (there is no CPU fallback)", file=sys.stderr)
        sys.exit(3)
    if a.copy_probe:
        nb = 1 << 30
        src, dst = DevBuf(nb), DevBuf(nb)
        lib.mi_zero(src.ptr, nb)
        for _ in range(5):
            lib.mi_d2d(dst.ptr, src.ptr, nb)
        lib.mi_sync(); LP.check()
        print(json.dumps({"copy_probe_bytes": nb, "copies": 5}))
        return
    if a.conv_probe:
        Ci, Co, N, D, bits = [int(v) for v in a.conv_probe.split(",")]
        S = D * D * D
        rng = np.random.default_rng(0)
        dx = DevBuf.from_numpy(rng.standard_normal((N, Ci, S)).astype(np.float32))
        mxb, cvt, conv, dt = (lib.lp_mx8_bytes, lib.lp_f32_to_mx8, lib.lp_conv_fwd_f8, 3) if bits == 8 else (lib.lp_mx4_bytes, lib.lp_f32_to_mx4, lib.lp_conv_fwd_f4, 4)
        dxq = DevBuf(mxb(N, Ci, S)); cvt(dx.ptr, N, Ci, S, dxq.ptr)
        dw = DevBuf.from_numpy((rng.standard_normal((Co, Ci, 27)) * np.sqrt(2.0 / (Ci * 27))).astype(np.float32))
        db = DevBuf.from_numpy((rng.standard_normal(Co) * 0.1).astype(np.float32))
        dy = DevBuf(mxb(N, Co, S)); dsum = DevBuf(N * 8 * 2 * 24)
        sp = split_t(); sp.wkey = 7; xs = shape5(N, Ci, D, D, D)
        for _ in range(a.warmup):
            conv(dxq.ptr, dt, xs, dw.ptr, db.ptr, Co, dy.ptr, dt, gnp_t(), dsum.ptr, 8, sp)
        lib.mi_kernel_timing(1)
        for _ in range(a.steps):
            conv(dxq.ptr, dt, xs, dw.ptr, db.ptr, Co, dy.ptr, dt, gnp_t(), dsum.ptr, 8, sp)
        nl = C.c_long(0)
        ms = lib.mi_kernel_timing_read(C.byref(nl)) / max(nl.value, 1)
        lib.mi_kernel_timing(0); LP.check()
        fl = 2.0 * 27 * Ci * Co * N * S
        peak = 5033.0 if bits == 8 else 10066.0
        print(json.dumps({"conv_probe": a.conv_probe, "kernel": lib.mi_last_kernel().decode(), "launches": int(nl.value), "avg_launch_ms": ms,
                          "tflops": fl / ms / 1e9, "frac_of_mfma_peak": fl / ms / 1e9 / peak,
                          "algorithmic_bytes": int(mxb(N, Ci, S) + mxb(N, Co, S)), "GBps": (mxb(N, Ci, S) + mxb(N, Co, S)) / ms / 1e6}))
        return
    if a.unet_only:
        a.no_stack = a.no_sliding = a.no_hbm = a.no_single = a.no_cpu_baseline = True
    out = {"metric": METRIC, "unit": "voxels/s", "n_gpus": 1, "steps": a.steps, "warmup": a.warmup, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
           "dtype": "mxfp8 (e4m3 x e4m3 block-scaled, fp32 accumulate)", "data": "synthetic",
           "weights": "prepared (quantised, re-laid-out) once and memoised across the timed forwards, as an inference loop keeps them"}
    u, dom = unet_leg(np, lib, LP, DevBuf, a.steps, a.warmup)
    out["value"] = u["value"]; out["ms_per_step"] = u["ms_per_forward"]; out["tflops"] = u["tflops"]
    out["config"] = {"workload": u["workload"], "batch": 2, "dims": [128, 128, 128], "widths": [32, 64, 128, 256], "cin": 4, "head_out": 8, "gflop_per_forward": u["gflop_per_forward"]}
    prof = profile_traffic(dom["layer"])
    out["roofline"] = {"bound": "mfma", "kernel": "%s (%s)" % (dom["kernel"], dom["layer"]), "achieved": dom["tflops"], "peak": MFMA_PEAK_FP8_TFLOPS, "unit": "TFLOP/s",
                       "frac": dom["frac_of_mxfp8_peak"], "avg_launch_ms": dom["avg_launch_ms"], "launches": a.steps, "flops_per_launch": dom["flops_per_launch"],
                       "traffic": prof[0], "traffic_source": prof[1]}
    out["unet"] = u
    stack = None
    if not a.no_stack:
        # (the part's clock takes some tens of launches of this kernel to settle: the stack legs run at least 10 warm-up and 30 timed steps of four
        # launches each, whatever the U-Net leg was asked for; their sub-records carry their own counts)
        stack, xq0, w_host_l0 = stack_leg(np, lib, LP, DevBuf, shape5, gnp_t, split_t, max(a.steps, 30), max(a.warmup, 10))
        out["conv_stack"] = stack
        out["conv_stack_fused"] = stack_fused_leg(np, lib, LP, DevBuf, shape5, gnp_t, split_t, max(a.steps, 30), max(a.warmup, 10))
    if not a.no_single:
        out["c0"] = c0_leg(np, lib, LP, DevBuf, shape5, gnp_t, split_t, max(a.steps, 20) * 5, max(a.warmup, 5) * 2)
        out["c2a"] = c2a_leg(np, lib, LP, DevBuf, shape5, gnp_t, split_t, max(a.steps, 20) * 5, max(a.warmup, 5) * 2)
    if not a.no_sliding:
        out["sliding_window"] = sliding_leg(np, lib, LP, DevBuf, a.windows_per_forward)
        if a.sliding_radial:
            out["sliding_window_radial"] = sliding_leg(np, lib, LP, DevBuf, a.windows_per_forward, radial=True)
    if not a.no_hbm:
        out["hbm_kernels"] = hbm_leg(np, lib, LP, DevBuf)
    if not a.no_cpu_baseline:
        import orc
        # the oracle (a port: the reference has no CPU MX conv) on a bounded z-slab of the forward's heaviest layer shape class: one 128 -> 128 conv
        # at N 2 x 64^3, scaled by the forward's FLOPs to voxels/s of the whole U-Net
        N, Cc, D = 2, 128, 64
        S = D ** 3
        rng = np.random.default_rng(0)
        if stack is None:
            xq0 = orc.f32_to_mx(8, rng.standard_normal((N, Cc, S)).astype(np.float32), N, Cc, S)
            w_host_l0 = (rng.standard_normal((Cc, Cc, 27)) * np.sqrt(2.0 / (Cc * 27))).astype(np.float32)
        nthreads = orc.lib().orc_threads()
        t = time.perf_counter(); orc.conv3(xq0, 3, N, Cc, D, D, D, w_host_l0, None, Cc, 3, z0=0, z1=1); dt1 = time.perf_counter() - t
        nz = int(max(1, min(D, a.cpu_seconds / max(dt1, 1e-3))))
        t = time.perf_counter(); orc.conv3(xq0, 3, N, Cc, D, D, D, w_host_l0, None, Cc, 3, z0=D // 2 - nz // 2, z1=D // 2 - nz // 2 + nz); dt = time.perf_counter() - t
        gflops = 2.0 * 27 * Cc * Cc * N * S * nz / D / dt / 1e9
        out["cpu_baseline"] = {"value": 2 * 128 ** 3 / (u["gflop_per_forward"] / gflops), "unit": "voxels/s", "cores": nthreads, "kind": "port",
                               "sample": "oracle orc_conv3 (the reference has no CPU MX conv) on %d of %d output z planes of a 128 -> 128 conv at N 2 x 64^3: %.1f GFLOP/s, "
                                         "scaled by the forward's %.0f GFLOP to U-Net voxels/s" % (nz, D, gflops, u["gflop_per_forward"]),
                               "gflops": gflops}
    print(json.dumps(out))


def stack_leg(np, lib, LP, DevBuf, shape5, gnp_t, split_t, steps, warmup):
    """4 x (3x3x3 conv 128 -> 128, N 2, 64^3, MX-fp8 in / out, bias + GroupNorm(8) statistics, GN + SiLU on the input)."""
    N, Cc, D, L, G = 2, 128, 64, 4, 8
    S = D * D * D
    rng = np.random.default_rng(0)
    x = rng.standard_normal((N, Cc, S)).astype(np.float32)
    dx = DevBuf.from_numpy(x)
    act = [DevBuf(lib.lp_mx8_bytes(N, Cc, S)) for _ in range(2)]
    x0 = DevBuf(lib.lp_mx8_bytes(N, Cc, S))
    lib.lp_f32_to_mx8(dx.ptr, N, Cc, S, x0.ptr)
    ws, bs, gam, bet, mean, rstd, sums = [], [], [], [], [], [], []
    for l in range(L):
        w = (rng.standard_normal((Cc, Cc, 27)) * np.sqrt(2.0 / (Cc * 27))).astype(np.float32)
        ws.append(DevBuf.from_numpy(w)); bs.append(DevBuf.from_numpy((rng.standard_normal(Cc) * 0.1).astype(np.float32)))
        gam.append(DevBuf.from_numpy(np.ones(Cc, np.float32))); bet.append(DevBuf.from_numpy(np.zeros(Cc, np.float32)))
        mean.append(DevBuf(N * G * 4)); rstd.append(DevBuf(N * G * 4)); sums.append(DevBuf(N * G * 2 * 24))
    xs = shape5(N, Cc, D, D, D)

    def step():
        src = x0
        for l in range(L):
            dst = act[l & 1]
            gp = gnp_t() if l == 0 else LP.gn(gam[l - 1], bet[l - 1], mean[l - 1], rstd[l - 1], G)
            sp = split_t(); sp.wkey = 100 + l            # weights are constant across steps: prepared once (inference)
            # the op layer's call (host/nn_host.c): conv with fused statistics whose reduction sets the sum slots and finalises mean / rstd
            lib.mi_conv_fwd_gn(8, src.ptr, 3, xs, ws[l].ptr, bs[l].ptr, Cc, dst.ptr, 3, gp, sums[l].ptr, G, sp, 1e-5, mean[l].ptr, rstd[l].ptr)
            src = dst

    for _ in range(warmup):
        step()
    LP.check()
    lib.mi_kernel_timing(1)
    lib.mi_sync()
    t0 = time.perf_counter()
    for _ in range(steps):
        step()
    lib.mi_sync()
    t1 = time.perf_counter()
    LP.check()
    nl = C.c_long(0)
    kms = lib.mi_kernel_timing_read(C.byref(nl))
    lib.mi_kernel_timing(0)
    kernel = lib.mi_last_kernel().decode()
    ms_step = (t1 - t0) * 1e3 / steps
    flops_layer = 2.0 * 27 * Cc * Cc * N * S               # logical channels, all 27 taps (tests/bench_lp.c:46)
    k_ms = kms / max(nl.value, 1)
    achieved = flops_layer / (k_ms * 1e-3) / 1e12
    rec = {"workload": "configs[1]: 4 x (3x3x3 conv 128->128, N 2, 64^3, MX-fp8 in/out, bias + GroupNorm(8) stats, GN+SiLU on the input)",
           "value": N * S / (ms_step * 1e-3), "unit": "voxels/s", "ms_per_step": ms_step, "steps": steps, "warmup": warmup, "tflops": L * flops_layer / (ms_step * 1e-3) / 1e12,
           "roofline": {"bound": "mfma", "kernel": kernel, "achieved": achieved, "peak": MFMA_PEAK_FP8_TFLOPS, "unit": "TFLOP/s", "frac": achieved / MFMA_PEAK_FP8_TFLOPS,
                        "launches": nl.value, "avg_launch_ms": k_ms, "flops_per_launch": flops_layer,
                        "traffic": profile_traffic("conv_stack")[0], "traffic_source": profile_traffic("conv_stack")[1],
                        "algorithmic_bytes": 2 * N * (Cc // 32) * S * 33 + 28 * Cc * Cc * 33 // 32}}
    return rec, x0.to_numpy(np.uint8), w


if __name__ == "__main__":
    main()

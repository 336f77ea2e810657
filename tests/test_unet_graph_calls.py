"""What a U-Net forward asks of the kernels' library, without a GPU: the host layer (nn_host.c, unet.c, predict.c) linked with stand-ins that write down every allocation
and every call that reads or writes a tensor. No operand rows are made that nothing reads, and no buffer is held that nothing uses, whatever the configuration."""
import ctypes as C
import os
import re
import subprocess

import pytest

from ufsm_amd import shape5
from ufsm_amd.unet import unet_cfg

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# the calls that matter, with their own prototypes; every other entry is a function that does nothing
STUB = r"""
#include "mi_unet.h"
#include "mi_lp.h"
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
static char *buf; static size_t len, cap;
static void put(const char *fmt, ...) {
    va_list a; va_start(a, fmt);
    if (len + 512 > cap) { cap = 2 * cap + 4096; buf = realloc(buf, cap); }
    len += (size_t)vsnprintf(buf + len, 512, fmt, a); va_end(a);
}
const char *stub_log(void) { return buf ? buf : ""; }
void stub_clear(void) { len = 0; if (buf) buf[0] = 0; }
static int staged;
void *mi_malloc(size_t n) { void *p = malloc(n + 64); put("alloc %zu %zu\n", (size_t)p, n); return p; }
void mi_free(void *p) { if (p) put("free %zu\n", (size_t)p); }                   /* (the address stays taken: every buffer of a run has its own) */
void *mi_host_alloc(size_t n) { return calloc(1, n + 1); }
size_t lp_mx8_bytes(int n, int c, size_t s) { const int bw = c <= 8 ? 8 : c <= 16 ? 16 : 32; return (size_t)n * ((c + bw - 1) / bw) * s * (bw + 1); }
size_t lp_mx4_bytes(int n, int c, size_t s) { const int bw = c <= 8 ? 8 : c <= 16 ? 16 : 32; return (size_t)n * ((c + bw - 1) / bw) * s * (bw / 2 + 1); }
gnp_t gnp_mk(const float *g, const float *b, const float *m, const float *r, int G) { gnp_t p; memset(&p, 0, sizeof p); p.gamma = g; p.beta = b; p.mean = m; p.rstd = r; p.G = G; return p; }
void mi_conv_up_staged(int on) { staged = on; }
static int conv(const void *x, const void *x2, gnp_t gp, shape5 xs, int cout, void *y, void *st8, void *st4) {
    const size_t s = (size_t)xs.d * xs.h * xs.w;
    if (staged && gp.G) put("bad GroupNorm on staged rows\n");
    put("read %zu\n", (size_t)x); if (x2) put("read %zu\n", (size_t)x2);
    put("write %zu\n", (size_t)y);
    if (st8) put("rows %zu %zu\n", (size_t)st8, lp_mx8_bytes(xs.n, cout, s));
    if (st4) put("rows %zu %zu\n", (size_t)st4, lp_mx4_bytes(xs.n, cout, s));
    staged = 0;
    return 0;
}
int lp_conv_fwd_f8(const void *x, int xbf, shape5 xs, const float *w, const float *b, int cout, void *y, int ybf, gnp_t gp, double *o, int G, split_t sp) { return conv(x, sp.x2, gp, xs, cout, y, 0, 0); }
int lp_conv_fwd_f4(const void *x, int xbf, shape5 xs, const float *w, const float *b, int cout, void *y, int ybf, gnp_t gp, double *o, int G, split_t sp) { return conv(x, sp.x2, gp, xs, cout, y, 0, 0); }
int mi_conv_fwd_gn(int bits, const void *x, int xbf, shape5 xs, const float *w, const float *b, int cout, void *y, int ybf, gnp_t gp, double *o, int G, split_t sp, float e, float *m, float *r) {
    return conv(x, sp.x2, gp, xs, cout, y, 0, 0);
}
int mi_conv_fwd_gn_stage(int bits, const void *x, int xbf, shape5 xs, const float *w, const float *b, int cout, void *y, int ybf, gnp_t gp, double *o, int G, split_t sp, float e, float *m, float *r,
                         const float *ga, const float *be, void *st8, void *st4) {
    if (cout % 32) return -1;
    return conv(x, sp.x2, gp, xs, cout, y, st8, st4);
}
int lp_conv_fwd_s2_f8(const void *x, int xbf, shape5 xs, const float *w, const float *b, int cout, void *y, int ybf, shape5 ys, gnp_t gp) { put("read %zu\nwrite %zu\n", (size_t)x, (size_t)y); return 0; }
int mi_conv_prestage(const void *x, int xdt, shape5 s, gnp_t gp, void *y, int bits) {
    put("read %zu\npass %zu\nrows %zu %zu\n", (size_t)x, (size_t)x, (size_t)y, (bits == 8 ? lp_mx8_bytes : lp_mx4_bytes)(s.n, s.c, (size_t)s.d * s.h * s.w)); return 0;
}
int mi_conv_prestage2(const void *x, shape5 s, gnp_t gp, void *y8, void *y4) {
    const size_t v = (size_t)s.d * s.h * s.w;
    put("read %zu\npass %zu\nrows %zu %zu\nrows %zu %zu\n", (size_t)x, (size_t)x, (size_t)y8, lp_mx8_bytes(s.n, s.c, v), (size_t)y4, lp_mx4_bytes(s.n, s.c, v)); return 0;
}
void lp_conv1_fwd_mx(const void *x, int xdt, shape5 xs, const float *w, const float *b, int cout, float *y, gnp_t gp) { put("read %zu\nwrite %zu\n", (size_t)x, (size_t)y); }
void mi_d2d_rows(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t r) { put("read %zu\nwrite %zu\n", (size_t)s, (size_t)d); }
int lp_gn_sums_mx(const void *x, int xdt, int n, int c, int G, size_t S, double *sums, size_t v0, size_t vn) { return 0; }
"""


@pytest.fixture(scope="module")
def graph(tmp_path_factory):
    return link(tmp_path_factory.mktemp("graph"))


def link(d):
    host = [os.path.join(ROOT, "ufsm_amd", "host", f) for f in ("nn_host.c", "unet.c", "predict.c")]
    (d / "stub.c").write_text("#include <stdarg.h>\n" + STUB)
    def cc(out, src, *more):
        subprocess.run(["gcc", "-std=c2x", "-w", "-O1", "-fPIC", "-I" + os.path.join(ROOT, "include"), *more, "-o", str(d / out)] + [str(f) for f in src] + ["-lm"], check=True)
    cc("a.so", host + [d / "stub.c"], "-shared")
    undefined = subprocess.run(["nm", "-D", "--undefined-only", str(d / "a.so")], check=True, capture_output=True, text=True).stdout
    names = [n for n in re.findall(r" U (\w+)\n", undefined) if re.match(r"(mi|lp|nn|at)_", n)]
    (d / "other.c").write_text("\n".join("long %s(void) { return 0; }" % n for n in names))
    cc("graph.so", host + [d / "stub.c", d / "other.c"], "-shared", "-Wl,--no-undefined")
    L = C.CDLL(str(d / "graph.so"))
    L.stub_log.restype = C.c_char_p
    L.unet_create.restype = C.c_void_p; L.unet_create.argtypes = [C.POINTER(unet_cfg)]
    L.unet_free.argtypes = [C.c_void_p]
    L.mi_unet_forward_mx.restype = C.c_void_p; L.mi_unet_forward_mx.argtypes = [C.c_void_p, C.c_void_p, shape5]
    return L


def run(L, dims=(32, 32, 32), n=1, widths=(32, 64, 128), mx4=0, prec=0, slab=0, direct=1, forwards=1, **cfg):
    c = unet_cfg()
    c.nlev, c.cin, c.cout, c.G = len(widths), 4, 8, 8
    for i, w in enumerate(widths):
        c.widths[i] = w
    for k, v in cfg.items():
        if isinstance(v, tuple):
            for i, e in enumerate(v):
                getattr(c, k)[i] = e
        else:
            setattr(c, k, v)
    L.unet_set_act_mx4(mx4); L.nn_set_prec(prec); L.unet_set_infer_slab(slab); L.unet_set_slab_direct(direct)
    L.stub_clear()
    u = L.unet_create(C.byref(c))
    assert u
    params = [int(l.split()[1]) for l in L.stub_log().decode().splitlines() if l.startswith("alloc")]
    L.stub_clear()
    xin = C.create_string_buffer(64)
    try:
        for _ in range(forwards):
            assert L.mi_unet_forward_mx(u, C.addressof(xin), shape5(n, 4, *dims))
        return [(l.split()[0],) + tuple(int(v) if v.isdigit() else v for v in l.split()[1:]) for l in L.stub_log().decode().splitlines()], params
    finally:
        L.unet_free(u)
        L.unet_set_act_mx4(0); L.nn_set_prec(0); L.unet_set_infer_slab(0); L.unet_set_slab_direct(1)


CONFIGS = {
    "plain": dict(), "two samples": dict(n=2), "precision 3": dict(prec=3), "mx4": dict(mx4=1), "one level": dict(widths=(32,)), "two levels": dict(widths=(32, 64)),
    "narrow level 0": dict(widths=(16, 32, 64)), "48 channels": dict(widths=(32, 48, 64)), "dec_widths": dict(widths=(32, 64, 128), dec_widths=(0, 32, 0)),
    "l0_norm 1": dict(l0_norm=1), "l0_norm 3": dict(l0_norm=3), "l0_norm 4": dict(l0_norm=4, l0_slab=16), "l0_norm 1, mx4": dict(l0_norm=1, mx4=1),
    "dec_convs 1 at level 0": dict(dec_convs=(1, 2, 2)), "dec_convs 1": dict(dec_convs=(1, 1, 1)), "dec_convs 1, mx4": dict(dec_convs=(1, 1, 1), mx4=1),
    "enc_blocks": dict(enc_blocks=(0, 1, 1)), "enc_blocks, mx4": dict(enc_blocks=(0, 1, 1), mx4=1), "slabs": dict(slab=8), "slabs, mx4": dict(slab=8, mx4=1),
    "slabs, precision 3": dict(slab=8, prec=3), "slabs in place": dict(slab=8, direct=0), "slabs in place, mx4": dict(slab=8, direct=0, mx4=1),
    "slabs, two levels": dict(slab=8, widths=(32, 64)), "slabs of the whole depth": dict(slab=32), "four levels, slabs": dict(slab=8, widths=(32, 64, 128, 256)), "down_norm": dict(down_norm=1),
}


@pytest.mark.parametrize("name", CONFIGS)
def test_no_rows_are_made_that_nothing_reads(graph, name):
    """Every set of operand rows written behind a conv, or by a pass of its own, is read by a later call before its buffer is written again."""
    log, _ = run(graph, forwards=2, **CONFIGS[name])
    assert not [e for e in log if e[0] == "bad"]
    open_rows = {}
    for k, e in enumerate(log):
        if e[0] == "rows":
            assert e[1] not in open_rows, "rows at event %d overwrite rows of event %d that nothing read" % (k, open_rows[e[1]])
            open_rows[e[1]] = k
        elif e[0] == "read":
            open_rows.pop(e[1], None)
    assert not open_rows


@pytest.mark.parametrize("name", CONFIGS)
def test_a_skip_has_one_pass_of_its_own_at_most(graph, name):
    """A skip that no conv's pass has transformed gets one pass for both readers or, under MX-fp4 storage, none and no buffers: each reader transforms it."""
    log, _ = run(graph, **CONFIGS[name])
    passes = [e[1] for e in log if e[0] == "pass"]
    assert len(passes) == len(set(passes)) and not (passes and "mx4" in name)


@pytest.mark.parametrize("name,skips", [("mx4", 0), ("precision 3", 0), ("plain", 2)])
def test_skip_knob(tmp_path, monkeypatch, name, skips):
    """MI_UNET_SKIP2=0: where a skip's readers compute in different formats each transforms it itself; nothing is held or made for both (MX-fp8 alone shares its skips as ever)."""
    monkeypatch.setenv("MI_UNET_SKIP2", "0")
    L = link(tmp_path)
    log, _ = run(L, **CONFIGS[name])
    assert len([e for e in log if e[0] == "rows"]) == (2 * 3 - 1) + 2 + skips and not [e for e in log if e[0] == "pass"]      # (five blocks' conv1, two coarse segments, the skips)


@pytest.mark.parametrize("name", ["plain", "mx4", "precision 3", "dec_convs 1 at level 0", "dec_convs 1", "two levels"])
def test_rows_are_handed_on_where_they_can_be(graph, name):
    """... and outside slabs, constant statistics and residual blocks every block's conv2 reads rows, and every decoder block takes its coarse segment as rows."""
    log, _ = run(graph, **CONFIGS[name])
    rows, blocks = [e for e in log if e[0] == "rows"], len(CONFIGS[name].get("widths", (32, 64, 128)))
    singles = sum(v == 1 for v in CONFIGS[name].get("dec_convs", ())[:blocks - 1])
    skips = (2 if "mx4" in name or "precision" in name else 1) * (blocks - 1) - ("mx4" in name)      # (MX-fp4: level 0 of 32 channels has one form for both readers)
    assert len(rows) == (2 * blocks - 1 - singles) + skips + (blocks - 1)
    assert not [e for e in log if e[0] == "pass"]


@pytest.mark.parametrize("name", CONFIGS)
def test_every_buffer_of_a_forward_is_used(graph, name):
    """The graph holds no tensor that its forwards neither read nor write, and no buffer of operand rows larger than the rows it is given. (Of the buffers that are allocated:
    the statistics and the sum slots are reached through pointers that the stand-ins do not follow, so only those of tensor size count.)"""
    log, _ = run(graph, forwards=2, **CONFIGS[name])
    dims, n = CONFIGS[name].get("dims", (32, 32, 32)), CONFIGS[name].get("n", 1)
    small = 1 << 13                                                # (statistics of the widest level and two samples: 8 KB; the smallest tensor, 128 channels at 8^3 in e2m1: 34 KB)
    held = {e[1]: e[2] for e in log if e[0] == "alloc" and e[2] > small}
    freed = {e[1] for e in log if e[0] == "free"}
    used = {e[1] for e in log if e[0] in ("read", "write", "rows")}
    unused = {p: b for p, b in held.items() if p not in used and p not in freed}
    # the net's own input tensor (MX, one block of 8 channels) takes another forward entry's rows
    s = dims[0] * dims[1] * dims[2]
    own_input = {n * s * 9, n * s * 5}
    assert all(b in own_input for b in unused.values()) and len(unused) <= 1, unused
    written = {}
    for e in log:
        if e[0] == "rows":
            written[e[1]] = max(written.get(e[1], 0), e[2])
    assert all(b <= held[p] for p, b in written.items())          # they fit
    assert not [(held[p], b) for p, b in written.items() if held[p] > b]      # (a skip's buffer is filled by the skip itself, the blocks' own one by their widest rows)
    assert len(freed) == 0                                         # (two forwards of one kind: nothing is given back or grown)


@pytest.mark.parametrize("mx4,prec", [(0, 0), (0, 3), (1, 0)])
def test_slabs_switched_between_forwards(graph, mx4, prec):
    """A net built in the direct slab form and then run whole makes its rows in buffers that hold them, and goes back to slabs: no rebuild, no rows that nothing reads."""
    c = unet_cfg()
    c.nlev, c.cin, c.cout, c.G = 3, 4, 8, 8
    c.widths[0], c.widths[1], c.widths[2] = 16, 48, 64
    c.dec_widths[1] = 32
    graph.unet_set_act_mx4(mx4); graph.nn_set_prec(prec)
    graph.stub_clear()
    u = graph.unet_create(C.byref(c))
    xin = C.create_string_buffer(64)
    counts = []
    try:
        for slab in (8, 0, 8, 0):
            graph.unet_set_infer_slab(slab)
            before = len(graph.stub_log())
            assert graph.mi_unet_forward_mx(u, C.addressof(xin), shape5(1, 4, 32, 32, 32))
            counts.append(graph.stub_log()[before:].count(b"rows"))
        log = [(l.split()[0],) + tuple(int(v) for v in l.split()[1:]) for l in graph.stub_log().decode().splitlines()]
    finally:
        graph.unet_free(u)
        graph.unet_set_act_mx4(0); graph.nn_set_prec(0); graph.unet_set_infer_slab(0)
    assert counts[1] == counts[3] > counts[0] == counts[2]
    held, open_rows = {}, set()
    for e in log:
        if e[0] == "alloc":
            held[e[1]] = e[2]
        elif e[0] == "free":
            del held[e[1]]
        elif e[0] == "rows":
            assert e[1] not in open_rows and e[2] <= held[e[1]]
            open_rows.add(e[1])
        elif e[0] == "read":
            open_rows.discard(e[1])
    assert not open_rows
